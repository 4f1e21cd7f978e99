"""Lanes of folds whose rows are few (no GPU): rows without a CU of their own take no more than 256,
but in 16-bit merge folds, whose lanes start at a few."""
import pytest
import torch

import neptune_codegen as CG
from neptune_codegen import template as T
from neptune_codegen.autotune import default_config


def _variant(name, rows, ncols, dtype):
    kernel = CG.compile_skeleton(name, {**CG.param_defaults(name),
                                        **({"eps": 1e-6} if name == "rmsnorm_max" else {})})
    x = torch.empty((rows, ncols), dtype=dtype, device="meta")
    return T._serial_variant(kernel, x, rows, ncols, *default_config(rows, ncols, dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", ["logsumexp", "softcap_lse", "stable_l2", "rmsnorm_max"])
def test_lanes_of_rows_without_a_cu_of_their_own(name, dtype):
    for ncols in (8192, 32000, 65536, 185024):
        var = _variant(name, T.CUS + 1, ncols, dtype)
        if dtype == torch.float32 or name in ("logsumexp", "softcap_lse"):
            assert var.tpr <= 256, (name, dtype, ncols)
        assert _variant(name, T.CUS, ncols, dtype).tpr >= var.tpr


def test_lanes_that_do_not_pay():
    """1024 lanes want 32 slots each of 512 and half a CU; 512 want 12 each of 256."""
    f32 = torch.float32
    assert _variant("logsumexp", 64, 65536, f32).tpr == 1024
    assert _variant("logsumexp", 64, 32000, f32).tpr == 512
    assert _variant("logsumexp", 200, 65536, f32).tpr == 512
    assert _variant("softcap_lse", 64, 8192, f32).tpr == 256
    assert _variant("stable_l2", 800, 4096, f32).tpr == 128
    assert _variant("stable_l2", 400, 32000, torch.bfloat16).tpr == 512
