"""Launch shapes of serial folds with few rows (no GPU): a shape the kernels take, with lanes added
only while they are short and every lane keeps at least 4 slots."""
import pytest
import torch

from neptune_codegen import template as T
from neptune_codegen.autotune import MAX_TPR, best_config, vec_of


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_few_rows_lanes(dtype):
    for rows in (1, 7, 64, 300, 5000, 100000):
        for ncols in (33, 1000, 1001, 4096, 20011, 65536, 262144):
            x = torch.empty((rows, ncols), dtype=dtype, device="meta")
            for heavy in (False, True):
                var = T._fold_variant(x, ncols, *best_config(rows, ncols, dtype, None), merge_heavy=heavy)
                few = T._few_rows(var, rows, ncols)
                slots = -(-ncols // (vec_of(dtype) if few.vector else 1))
                assert few.tpr & (few.tpr - 1) == 0 and var.tpr <= few.tpr <= MAX_TPR
                assert 1 <= few.unroll <= var.unroll and few.wg % 64 == 0 and few.wg >= few.tpr
                assert few.wg % few.tpr == 0
                if few.tpr > var.tpr:
                    assert slots >= 4 * few.tpr and rows * few.tpr // 2 < T.FEW_ROWS_LANES
                else:
                    assert few == var


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_short_row_shapes_hold_their_row(dtype):
    """Norms, readouts and two-pass folds of short rows: one tile holds the row, lanes are a power
    of two, and no slot is wholly past the row's end."""
    vec = vec_of(dtype)
    for ncols in list(range(vec, 300)) + [512, 1000, 1001, 1024, 2047, 2048]:
        x = torch.empty((500, ncols), dtype=dtype, device="meta")
        slots = -(-ncols // vec)
        cfg = best_config(500, ncols, dtype, None)
        shapes = [T._fold_variant(x, ncols, *cfg, resident=True),
                  T._fold_variant(x, ncols, *cfg, resident=True, readout=True)]
        for var in shapes:
            assert var.vector and var.tpr & (var.tpr - 1) == 0 and var.wg % var.tpr == 0
            assert var.tpr * var.unroll >= slots > var.tpr * (var.unroll - 1)
        row = T._row_variant(x, None, ncols)
        assert row.vector and row.tpr & (row.tpr - 1) == 0 and row.wg % row.tpr == 0
        assert row.tpr * row.nv >= slots > row.tpr * (row.nv - 1)
        heavy = T._fold_variant(x, ncols, *cfg, merge_heavy=True)
        assert heavy.tpr & (heavy.tpr - 1) == 0 and 1 <= heavy.unroll <= 8
