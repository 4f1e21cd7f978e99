"""Row access of small folds (no GPU): narrow rows that are few in all take one element per load."""
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


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", ["logsumexp", "softcap_lse", "stable_l2", "rmsnorm_max", "variance"])
def test_narrow_rows_that_are_few(name, dtype):
    for ncols in (33, 77, 301, 1001):
        most = (T.FEW_ELEMENTS - 1) // ncols
        assert _variant(name, 1, ncols, dtype).access == "nep::kStrided"
        assert _variant(name, most, ncols, dtype).access == "nep::kStrided"
        assert _variant(name, most + 1, ncols, dtype).access == "nep::kRagged"
    assert _variant(name, 1, 1025, dtype).access == "nep::kRagged"
    assert _variant(name, 1, 64, dtype).access == "nep::kAligned"
