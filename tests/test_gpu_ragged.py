"""GPU parity of the ragged row access (unit column stride, any alignment and width) against the
CPU oracle: widths around whole vectors and tiles, every offset of the row start inside a 16-byte
vector, rows whose stride is no multiple of the vector, and the extreme values at the row's ends,
where the vector and single-element parts meet."""
import pytest
import torch

import neptune_codegen as CG
from neptune_codegen import template as T
from oracle import references as R

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]
TOL = {torch.float32: (1e-5, 1e-6), torch.bfloat16: (1.6e-2, 1e-3), torch.float16: (1.6e-2, 1e-3)}


def _say(*a):
    print(*a, flush=True)


def _rows(rows, width, dtype, offset, pad, seed=3):
    """[rows, width] on the CPU and the same values on the device, `offset` elements into its
    storage with row stride width + pad.  Each row's largest values are its first and last."""
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    x = 2 * torch.randn(rows, width, generator=torch.Generator().manual_seed(seed))
    x[:, 0] = 9.0
    x[:, -1] = -9.5
    x = x.to(dtype)
    store = torch.full((offset + rows * (width + pad),), float("nan"), dtype=dtype, device="cuda:0")
    dev = store[offset:].view(rows, width + pad)[:, :width]
    dev.copy_(x)
    return x, dev


SHAPES = [(9, 1, 0), (17, 0, 0), (31, 3, 1), (64, 0, 5), (127, 5, 0), (130, 7, 6), (1000, 0, 3),
          (1001, 0, 0), (2049, 2, 0), (4095, 6, 7), (12301, 4, 0)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["logsumexp", "softcap_lse", "stable_l2", "rmsnorm_max", "variance"])
def test_ragged_folds(name, dtype):
    params = {"rmsnorm_max": {"eps": 1e-6}, "softcap_lse": {"beta": 0.5}}.get(name, {})
    for width, offset, pad in SHAPES:
        x, dev = _rows(21, width, dtype, offset, pad)
        _say(f"ragged {name} {dtype} width={width} offset={offset} pad={pad}")
        got = CG.run(name, dev, **params).cpu().float()
        want = R.reference(name, x, **params)
        rtol, atol = TOL[dtype]
        torch.testing.assert_close(got, want, rtol=rtol, atol=atol)
        if dtype != torch.float32:   # one rounding of an fp32 result: within one ulp
            torch.testing.assert_close(got, want, rtol=torch.finfo(dtype).eps, atol=1e-6)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["logsumexp", "stable_l2"])
def test_ragged_split(name, dtype):
    for width, offset, pad in ((1025, 0, 0), (8191, 3, 0), (5000, 1, 2)):
        x, dev = _rows(5, width, dtype, offset, pad)
        _say(f"ragged split {name} {dtype} width={width} offset={offset} pad={pad}")
        got = CG.run(name, dev, plan="split").cpu().float()
        rtol, atol = TOL[dtype]
        torch.testing.assert_close(got, R.reference(name, x), rtol=rtol, atol=atol)


@pytest.mark.parametrize("dtype", DTYPES)
def test_ragged_non_finite_rows(dtype):
    """NaN, +inf and all -inf rows, the special element in the leading, vector and trailing part."""
    width = 1003
    for offset in (0, 1, 3):
        x, dev = _rows(9, width, dtype, offset, 0)
        for i, col in enumerate((0, 500, width - 1)):
            x[i, col] = float("nan")
            x[3 + i, col] = float("inf")
        x[6] = float("-inf")
        x[7] = float("-inf")
        x[7, width - 1] = 1.0
        dev.copy_(x)
        _say(f"ragged non-finite {dtype} offset={offset}")
        got = CG.run("logsumexp", dev).cpu().float()
        want = torch.logsumexp(x.float(), -1)
        rtol, atol = TOL[dtype]
        torch.testing.assert_close(got, want, rtol=rtol, atol=atol, equal_nan=True)
        out = CG.run_log_softmax(dev).cpu().float()
        assert torch.isnan(out[:7]).all()      # NaN rows, +inf rows, and -inf - (-inf)
        torch.testing.assert_close(out[7:], torch.log_softmax(x[7:].float(), -1), rtol=rtol, atol=atol)


@pytest.mark.parametrize("dtype", DTYPES)
def test_ragged_log_softmax(dtype):
    """Rows held in registers, and (65536 + 9 columns, 70001 in 16 bits) rows read twice."""
    for width, offset, pad in SHAPES + [(65545, 1, 0), (140001, 0, 0)]:
        rows = 21 if width < 20000 else 3
        x, dev = _rows(rows, width, dtype, offset, pad)
        _say(f"ragged log_softmax {dtype} width={width} offset={offset} pad={pad}")
        got = CG.run_log_softmax(dev).cpu().float()
        rtol, atol = TOL[dtype]
        torch.testing.assert_close(got, torch.log_softmax(x.float(), -1), rtol=rtol, atol=atol)


def test_ragged_rule():
    """Only unit-stride rows of at least one vector take the ragged access, and only where the
    aligned one does not hold."""
    def access(x):
        return T._fold_variant(x, x.shape[1], 1024, 4).access.split("::k")[1]

    x = torch.empty(64, 1024, dtype=torch.bfloat16, device="cuda:0")
    assert access(x) == "Aligned"
    assert access(x[:, :1001]) == "Ragged" and access(x[:, 1:1001]) == "Ragged"
    assert access(x[:, :7]) == "Strided" and access(x[:, ::2]) == "Strided"


def _ulps(got, want, dtype):
    """Largest distance in units of the last place (as ordered integers) over finite values."""
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    a, b = got.view(bits).long(), want.view(bits).long()
    low = torch.iinfo(bits).min
    a, b = torch.where(a < 0, low - a, a), torch.where(b < 0, low - b, b)
    return int((a - b).abs().max())


@pytest.mark.parametrize("dtype", DTYPES)
def test_ragged_norms(dtype):
    """RMSNorm and L2-normalize at ragged rows, gamma at another alignment than its rows, against
    fp64 statistics with the same rounding stages: the fp32 sum's order moves the scale by at most
    a few fp32 units (4 here), which in 16 bits can flip one rounding at each of two stages."""
    for width, offset, pad in SHAPES + [(16383, 1, 0), (32767, 0, 1)]:
        x, dev = _rows(21, width, dtype, offset, pad)
        gamma = (1 + 0.1 * torch.randn(width + 3, generator=torch.Generator().manual_seed(4))).to(dtype)
        g_dev = gamma.cuda()[3:]
        gamma = gamma[3:]
        _say(f"ragged norms {dtype} width={width} offset={offset} pad={pad}")
        xd = x.double()
        scale = torch.rsqrt(xd.square().mean(-1, True) + 1e-6).float()
        want = ((x.float() * scale).to(dtype).float() * gamma.float()).to(dtype)
        got = CG.run_rms_norm(dev, g_dev, eps=1e-6).cpu()
        assert _ulps(got, want, dtype) <= (8 if dtype == torch.float32 else 2)
        want = (x.float() / xd.square().sum(-1, True).sqrt().float()).to(dtype)
        got = CG.run_l2_normalize(dev, eps=1e-6).cpu()
        assert _ulps(got, want, dtype) <= (8 if dtype == torch.float32 else 1)


def test_ragged_l2_exact_division_of_tiny_and_huge_norms():
    """Rows whose norm is not a normal number, or that hold denormal quotients, take the exact
    division in the vector part too; a zero row divides by eps."""
    width = 1001
    x, dev = _rows(5, width, torch.float32, 1, 0)
    x[0] = 0.0
    x[1] *= 2.0 ** 66           # the sum of squares overflows: x / inf = 0
    x[2] *= 2.0 ** -80          # the sum of squares underflows to a denormal or 0
    x[3, 1:-1] *= 2.0 ** -120   # quotients in the denormal range beside ordinary ones
    dev.copy_(x)
    got = CG.run_l2_normalize(dev, eps=1e-6).cpu()
    norm = x.square().sum(-1, True).sqrt().clamp_min(1e-6)
    assert torch.equal(got[1], torch.zeros(width)) and torch.equal(got[0], torch.zeros(width))
    assert _ulps(got[2:], (x / norm)[2:], torch.float32) <= 8


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", ["logsumexp", "softcap_lse", "stable_l2", "rmsnorm_max", "linear_attn"])
def test_few_long_rows(name, dtype):
    """Few rows over up to 1024 lanes and 16 wavefronts each, aligned and ragged."""
    params = {"rmsnorm_max": {"eps": 1e-6}, "softcap_lse": {"beta": 0.5}}.get(name, {})
    for rows, width, offset in ((1, 65536, 0), (3, 65537, 1), (16, 8192, 0), (2, 262144, 0)):
        x, dev = _rows(rows, width, dtype, offset, 0)
        if name == "linear_attn":
            x = x.abs()          # a signed sum cancels: its relative error is not bounded
            dev.copy_(x)
        print(f"few rows {name} {dtype} {rows}x{width}+{offset}", flush=True)
        got = CG.run(name, dev, **params).cpu().float()
        rtol, atol = TOL[dtype]
        torch.testing.assert_close(got, R.reference(name, x, **params), rtol=rtol, atol=atol)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["variance", "std"])
def test_two_pass_rows_held_and_read_twice(name, dtype):
    """Rows around the widest that 1024 lanes hold (8 and 16 slots each), and wider ones."""
    top = 65536 if dtype == torch.float32 else 131072
    for width, offset in ((top // 2, 0), (top // 2 + 1, 1), (top, 0), (top - 1, 3), (top + 8, 0),
                          (2 * top + 5, 0)):
        x, dev = _rows(3, width, dtype, offset, 0)
        _say(f"two-pass {name} {dtype} width={width} offset={offset}")
        got = CG.run(name, dev).cpu().float()
        rtol, atol = TOL[dtype]
        torch.testing.assert_close(got, R.reference(name, x), rtol=rtol, atol=atol)


@pytest.mark.parametrize("dtype", DTYPES)
def test_log_softmax_rows_of_16_slots(dtype):
    """Rows that 1024 lanes hold with up to 16 slots each, with NaN and +inf rows among them."""
    top = 65536 if dtype == torch.float32 else 131072
    for width, offset in ((top // 2 + 8, 0), (top, 0), (top - 3, 1)):
        x, dev = _rows(4, width, dtype, offset, 0)
        x[1, width // 3] = float("inf")
        x[2, width - 1] = float("nan")
        dev.copy_(x)
        _say(f"log_softmax 16 slots {dtype} width={width} offset={offset}")
        got = CG.run_log_softmax(dev).cpu().float()
        rtol, atol = TOL[dtype]
        torch.testing.assert_close(got[::3], torch.log_softmax(x[::3].float(), -1), rtol=rtol, atol=atol)
        assert torch.isnan(got[1:3]).all()
