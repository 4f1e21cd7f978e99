"""GPU parity of the attention fold with its keys in parts and 128-query workgroups, against the
fp32 closed form: parts of one to all tiles, a short last part, causal blocks with different part
counts and parts beyond a wave's diagonal, the exact fp32 path inside a part."""
import math

import pytest
import torch

from neptune_codegen import attention as A
from oracle import references as R

pytestmark = pytest.mark.gpu

SHAPES = [(1, 2, 100, 1000), (2, 1, 300, 257), (1, 3, 513, 513), (1, 1, 129, 65)]


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    return torch.device("cuda:0")


def _qkv(B, H, Sq, Sk, D, dtype):
    g = torch.Generator().manual_seed(9)
    return [torch.randn(B, H, s, D, generator=g).to(dtype) for s in (Sq, Sk, Sk)]


def _lse(q, k, causal):
    s = torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous()) / math.sqrt(q.shape[3])
    if causal:
        s = s.masked_fill(~torch.ones(q.shape[2], k.shape[2], dtype=torch.bool).tril(0), float("-inf"))
    return torch.logsumexp(s, -1)


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_parts_parity(dtype, causal, dim):
    dev = _dev()
    for B, H, Sq, Sk in SHAPES:
        q, k, v = _qkv(B, H, Sq, Sk, dim, dtype)
        want, lse_want = R.attention_reference(q, k, v, causal=causal), _lse(q, k, causal)
        for per, e_max in ((None, 13), (1, 13), (2, 13), (3, 13), (2, -1)):
            print(f"attention parts {B}x{H} {Sq}x{Sk} d={dim} {dtype} causal={causal} per={per} "
                  f"e_max={e_max}", flush=True)
            got, lse, _ = A._launch(q.to(dev), k.to(dev), v.to(dev), None, causal, True, e_max,
                                    w64=False, waves=4, per=per)
            torch.testing.assert_close(got.cpu().float(), want.float(), rtol=1.6e-2, atol=1e-3)
            torch.testing.assert_close(lse.cpu(), lse_want, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("causal", [True, False])
def test_four_waves_equal_eight_bit_for_bit(causal):
    """The waves of a workgroup share tiles, not arithmetic."""
    dev = _dev()
    for dim in (64, 128):
        q, k, v = (t.to(dev) for t in _qkv(1, 3, 600, 600, dim, torch.bfloat16))
        four, eight = (A._launch(q, k, v, None, causal, True, 13, w64=False, waves=w) for w in (4, 8))
        assert torch.equal(four[0], eight[0]) and torch.equal(four[1], eight[1])


def test_a_part_with_non_finite_v_is_exact_beside_ordinary_parts():
    """inf in one part's V: only the rows that see it, and the rest keep the MFMA path's values."""
    dev = _dev()
    q, k, v = _qkv(1, 1, 400, 400, 128, torch.bfloat16)
    v[0, 0, 200, 3] = float("inf")
    got, _, exps = A._launch(q.to(dev), k.to(dev), v.to(dev), None, True, False, 13, w64=False,
                             waves=4, per=2)
    assert A.exact_path_taken(exps)
    got = got.cpu().float()
    clean = v.clone()
    clean[0, 0, 200, 3] = 0.0
    want = R.attention_reference(q, k, clean, causal=True).float()
    want[0, 0, 200:, 3] = float("inf")
    torch.testing.assert_close(got, want, rtol=1.6e-2, atol=1e-3)
