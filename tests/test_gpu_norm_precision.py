"""fp32 row norms are as exact as sums of one element per load on up to 16 elements per lane (the
general strided path's order), whatever the launch shape: L2-normalize's error against 64 bits, in
the 2-norm over many rows, is held to that order's error of the same rows, emulated in fp32."""
import pytest
import torch

import neptune_codegen as CG

pytestmark = pytest.mark.gpu
ROWS = 6000


def _butterfly(t):
    while t.shape[1] > 1:
        t = t[:, 0::2] + t[:, 1::2]
    return t[:, 0]


def _strided_order(x):
    """Row sums of squares: lane t adds the elements t, t + lanes, ... ; 64 lanes meet in a
    butterfly, the waves one after the other."""
    rows, n = x.shape
    lanes = 1 << max(0, (-(-n // 16) - 1).bit_length())
    per = -(-n // lanes)
    sq = torch.zeros(rows, per * lanes).index_copy_(1, torch.arange(n), x * x).view(rows, per, lanes)
    t = torch.zeros(rows, lanes)
    for u in range(per):
        t += sq[:, u]
    waves = [_butterfly(t[:, i:i + 64]) for i in range(0, lanes, 64)]
    total = waves[0]
    for w in waves[1:]:
        total = total + w
    return total


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("ncols", [333, 2999, 3000, 4096, 4099, 5001, 8191])
def test_norms_are_as_exact_as_the_strided_order(ncols, offset):
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    g = torch.Generator().manual_seed(ncols)
    x = torch.randn(ROWS, ncols, generator=g)
    wide = torch.zeros(ROWS, ncols + offset, device="cuda")
    view = wide[:, offset:]
    view.copy_(x)
    print(f"l2_normalize fp32 {ROWS} x {ncols} +{offset}", flush=True)
    got = CG.run_l2_normalize(view, eps=1e-6).cpu().double()
    exact = x.double() / x.double().square().sum(1, keepdim=True).sqrt()

    def error(y):
        return ((y - exact).norm() / exact.norm()).item()

    base = error((x / _strided_order(x).sqrt()[:, None]).double())
    # the norms' errors of 6000 rows have a 2-norm known to 1/sqrt(2 * 6000) = 0.9%
    assert error(got) <= 1.02 * base, (error(got), base)
