"""Launch shapes of fp32 norms and readouts at the sizes where a launch just fills the chip (no GPU):
half the lanes, each with twice the slots, hold the same row there, and nowhere else."""
import pytest
import torch

from neptune_codegen import template as T
from neptune_codegen.autotune import best_config

FULL = 1 << 19      # lanes that the chip holds at once


def _norm(rows, ncols):
    var = T._row_variant(torch.empty((rows, ncols), device="meta"), None, ncols)
    return var.tpr, var.nv


def _readout(rows, ncols):
    x = torch.empty((rows, ncols), device="meta")
    var = T._fold_variant(x, ncols, *best_config(rows, ncols, x.dtype, None), resident=True, readout=True)
    return var.tpr, var.unroll


@pytest.mark.parametrize("shape", [_norm, _readout])
@pytest.mark.parametrize("ncols,lanes", [(128, 16), (256, 32), (512, 64)])
def test_rows_of_a_just_full_launch(shape, ncols, lanes):
    for rows in (FULL // lanes * 7 // 8, FULL // lanes + 1):
        assert shape(rows, ncols) == (lanes, 2)
    for rows in (FULL // lanes * 7 // 8 + 1, FULL // lanes):
        assert shape(rows, ncols) == (lanes // 2, 4)


def test_ragged_rows_of_eight_waves():
    assert _norm(100, 3001) == (512, 2) and _norm(20000, 2999) == (512, 2)
    assert _norm(1000, 3001) == (256, 3) and _norm(700, 4001) == (256, 4)
