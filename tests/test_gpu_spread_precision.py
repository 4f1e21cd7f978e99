"""Folds of few rows on more lanes: no further from 64 bits than the same rows on the lanes that many
rows get, and the same special values (empty waves, a wave of zeros, NaN and infinities)."""
import pytest
import torch

import neptune_codegen as CG
from neptune_codegen import hip
from neptune_codegen import template as T
from neptune_codegen.skeleton import param_defaults

pytestmark = pytest.mark.gpu


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    return torch.device("cuda:0")


def _kernel(name):
    return CG.compile_skeleton(name, {**param_defaults(name), **({"eps": 1e-6} if name == "rmsnorm_max" else {})})


def _both(name, x):
    """(result on spread lanes, result on the default lanes)."""
    kernel, (rows, ncols) = _kernel(name), x.shape
    cfg = CG.best_config(rows, ncols, x.dtype, x.device)
    spread = T._serial_variant(kernel, x, rows, ncols, *cfg)
    plain = T._fold_variant(x, ncols, *cfg, merge_heavy=True)
    assert spread.spread and spread.tpr > max(64, plain.tpr)
    out = []
    for var in (spread, plain):
        print(f"{name} {rows} x {ncols} {x.dtype} {var.tag()}", flush=True)
        y = torch.empty(rows, dtype=x.dtype, device=x.device)
        kernel.kernel(var, "", 0).launch((-(-rows // max(1, var.wg // var.tpr)),),
                                         (x.data_ptr(), y.data_ptr(), rows, ncols, x.stride(0), x.stride(1)),
                                         hip.current_stream(x.device))
        out.append(y)
    return out


def _exact(name, x):
    x = x.double()
    if name == "stable_l2":
        return x.norm(dim=1)
    return x.amax(1) * torch.rsqrt(x.square().mean(1) + 1e-6)


@pytest.mark.parametrize("name", ["stable_l2", "rmsnorm_max"])
@pytest.mark.parametrize("rows,ncols", [(100, 4096), (20, 40000), (20, 40001), (4, 200000), (500, 16384)])
def test_spread_rows_are_as_exact(name, rows, ncols):
    dev = _dev()
    g = torch.Generator(device=dev).manual_seed(ncols)
    errors = torch.zeros(2, dtype=torch.float64)
    count = 0
    while count < 3000:
        x = 3 * torch.randn(rows, ncols, generator=g, device=dev)
        want = _exact(name, x)
        for i, got in enumerate(_both(name, x)):
            errors[i] += ((got.double() - want) / want).square().sum().item()
        count += rows
    # 2-norms over 3000 rows are known to 1/sqrt(2 * 3000) = 1.3% each
    assert errors[0].sqrt() <= 1.04 * errors[1].sqrt(), errors.div(count).sqrt()


@pytest.mark.parametrize("name", ["stable_l2", "rmsnorm_max"])
def test_spread_rows_special_values(name):
    dev = _dev()
    x = torch.randn(12, 20000, generator=torch.Generator().manual_seed(1)).to(dev)
    x[1] = 0.0
    x[2, :15000] = 0.0
    x[3, 777] = float("nan")
    x[4, 19999] = float("inf")
    x[5, 0] = float("-inf")
    x[6] = -x[6].abs()
    x[7] *= 1e-30
    x[8] *= 1e30
    x[9, ::2], x[9, 1::2] = float("inf"), float("-inf")
    spread, plain = _both(name, x)
    assert torch.equal(torch.isnan(spread), torch.isnan(plain)) and torch.equal(torch.isinf(spread), torch.isinf(plain))
    torch.testing.assert_close(spread, plain, rtol=3e-6, atol=0, equal_nan=True)
