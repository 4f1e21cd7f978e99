"""A launch configuration other than the shape's default keeps its lanes per row also where the rows
are few (no GPU)."""
import torch

import neptune_codegen as CG
from neptune_codegen import template as T
from neptune_codegen.autotune import CANDIDATES, default_config


def test_requested_configurations_are_launched():
    kernel = CG.compile_skeleton("logsumexp", {"tiny": 0.0})
    for rows, ncols, dtype in ((4, 262144, torch.float32), (64, 32000, torch.bfloat16), (8, 4096, torch.float16)):
        x = torch.empty((rows, ncols), dtype=dtype, device="meta")
        default = default_config(rows, ncols, dtype)
        for cfg in CANDIDATES:
            if cfg != default:
                assert T._serial_variant(kernel, x, rows, ncols, *cfg) == T._fold_variant(x, ncols, *cfg)
        assert (T._serial_variant(kernel, x, rows, ncols, *default)
                == T._few_rows(T._fold_variant(x, ncols, *default), rows, ncols))
    # a sweep at few rows measures different launches
    x = torch.empty((4, 262144), dtype=torch.float32, device="meta")
    shapes = {T._serial_variant(kernel, x, 4, 262144, *cfg) for cfg in CANDIDATES}
    assert len(shapes) == len({T._fold_variant(x, 262144, *cfg) for cfg in CANDIDATES})


def test_spread_rows_keep_their_registers():
    """No fold of few wide rows gets a launch shape whose kernel spills: 16-bit exponential folds,
    which hold unpacked values beside two tiles of raw words, stop at 512 lanes."""
    for name in ("logsumexp", "softcap_lse", "lse_scaled"):
        kernel = CG.compile_skeleton(name, CG.param_defaults(name))
        for dtype in (torch.bfloat16, torch.float16, torch.float32):
            for rows, ncols in ((1, 262144), (22, 235968), (4, 100001), (200, 250000)):
                x = torch.empty((rows, ncols), dtype=dtype, device="meta")
                var = T._serial_variant(kernel, x, rows, ncols, *default_config(rows, ncols, dtype))
                assert var.tpr <= (1024 if dtype == torch.float32 else 512), (name, dtype, ncols)
