"""GPU parity of the short-query attention kernels (few queries over keys split into chunks)
against the fp32 closed form, at the edges of their 16-query blocks, 32-key tiles, 4 waves and
chunks.  Tolerances are the attention fold's: rtol 1.6e-2 / atol 1e-3 for O, fp32 rtol 1e-5 /
atol 1e-6 for the logsumexp."""
import math

import pytest
import torch

import neptune_codegen as CG
from neptune_codegen import attention as A
from oracle import references as R

pytestmark = pytest.mark.gpu


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    return torch.device("cuda:0")


def _say(*a):
    print(*a, flush=True)


def _qkv(B, H, Sq, Sk, D, dtype, seed=5):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(B, H, s, D, generator=g).to(dtype) for s in (Sq, Sk, Sk)]


def _scores(q, k, causal, scale=None):
    s = torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous())
    s = s * (1.0 / math.sqrt(q.shape[3]) if scale is None else scale)
    if causal:
        s = s.masked_fill(~torch.ones(q.shape[2], k.shape[2], dtype=torch.bool).tril(0), float("-inf"))
    return s


SHAPES = [(1, 1, 1, 1), (2, 3, 1, 31), (1, 2, 16, 32), (2, 1, 15, 33), (1, 5, 2, 127), (1, 2, 8, 129),
          (3, 1, 4, 700), (1, 1, 1, 5000), (9, 31, 1, 300), (1, 1, 16, 4097)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("causal", [False, True])
def test_short_parity(causal, dim, dtype):
    dev = _dev()
    for B, H, Sq, Sk in SHAPES:
        q, k, v = _qkv(B, H, Sq, Sk, dim, dtype)
        _say(f"short attention {B}x{H} sq={Sq} sk={Sk} d={dim} {dtype} causal={causal} "
             f"chunks={A.short_chunks(B * H, Sk)}")
        got, lse = CG.run_attention(q.to(dev), k.to(dev), v.to(dev), causal=causal, return_lse=True)
        want = R.attention_reference(q, k, v, causal=causal)
        torch.testing.assert_close(got.cpu().float(), want.float(), rtol=1.6e-2, atol=1e-3)
        torch.testing.assert_close(lse.cpu(), torch.logsumexp(_scores(q, k, causal), -1),
                                   rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("chunks", [1, 2, 3, 7, 40])
def test_short_chunk_counts(chunks, monkeypatch):
    """Any split of the keys gives the result (several lane groups of the merge, a short last chunk)."""
    dev = _dev()
    q, k, v = _qkv(1, 3, 5, 1250, 128, torch.bfloat16)
    tiles = -(-1250 // 32)
    per = -(-tiles // chunks)
    monkeypatch.setattr(A, "short_chunks", lambda units, sk: (-(-tiles // per), per))
    _say(f"short attention in {-(-tiles // per)} chunks of {per} tiles")
    got, lse = CG.run_attention(q.to(dev), k.to(dev), v.to(dev), causal=False, return_lse=True)
    want = R.attention_reference(q, k, v, causal=False)
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=1.6e-2, atol=1e-3)
    torch.testing.assert_close(lse.cpu(), torch.logsumexp(_scores(q, k, False), -1), rtol=1e-5, atol=1e-6)


def test_short_layouts():
    """Projection layout, broadcast keys (stride 0) and a misaligned view give the same bits."""
    dev = _dev()
    q, k, v = (t.to(dev) for t in _qkv(2, 4, 3, 333, 128, torch.bfloat16))
    k[:, 1:] = k[:, :1]
    want = CG.run_attention(q, k, v, causal=False)
    swap = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]
    assert torch.equal(CG.run_attention(*swap, causal=False), want)
    assert torch.equal(CG.run_attention(q, k[:, :1].expand(2, 4, 333, 128), v, causal=False), want)
    odd = torch.empty(v.numel() + 1, dtype=v.dtype, device=dev)[1:].view(v.shape).copy_(v)
    assert torch.equal(CG.run_attention(q, k, odd, causal=False), want)


@pytest.mark.parametrize("sk", [70, 2000])
def test_short_values_out_of_the_ordinary(sk):
    """Huge, infinite and NaN V, an infinite key and a query whose scores are all -inf: what IEEE
    arithmetic on the visible keys gives.  sk=70: inf sits beside the zero-filled rows past the end."""
    dev = _dev()
    q, k, v = _qkv(1, 6, 2, sk, 128, torch.bfloat16)
    v[0, 0, 3] = 3e38       # one such key: |sum| <= 3e38 in any order of the fp32 sums
    v[0, 1, sk - 1, 7] = float("inf")
    v[0, 2, 0, 9] = float("nan")
    k[0, 3, 5] = 0.0
    k[0, 3, 5, 0] = float("-inf")
    q[0, 3, :, 0] = 1.0
    q[0, 4, 1, 0] = float("inf")
    k[0, 4, :, 0] = -1.0
    v[0, 5] *= 2.0 ** 40
    _say(f"short attention, unusual values, sk={sk}")
    got, lse = (t.cpu() for t in CG.run_attention(q.to(dev), k.to(dev), v.to(dev), causal=False,
                                                  return_lse=True))
    p = torch.softmax(_scores(q, k, False), -1)
    want = torch.matmul(p[0, 1], v[0, 1].float().nan_to_num(posinf=0.0))
    want[:, 7] = float("inf")
    torch.testing.assert_close(got[0, 1].float(), want, rtol=1.6e-2, atol=1e-3)
    assert torch.isnan(got[0, 2, :, 9]).all() and torch.isfinite(got[0, 2, :, 10:]).all()
    for h in (3, 5):
        want = torch.matmul(p[0, h], v[0, h].float())
        torch.testing.assert_close(got[0, h].float(), want, rtol=1.6e-2, atol=1e-3 * want.abs().max())
    assert torch.isnan(got[0, 4, 1]).all() and lse[0, 4, 1] == float("-inf")
    torch.testing.assert_close(got[0, 4, 0].float(), torch.matmul(p[0, 4, 0], v[0, 4].float()),
                               rtol=1.6e-2, atol=1e-3)
    torch.testing.assert_close(got[0, 0].float(), p[0, 0, :, 3:4] * v[0, 0, 3].float(),
                               rtol=1.6e-2, atol=0)


def test_short_under_graph_capture():
    """Captured with its split and merge, replayed on changed inputs."""
    dev = _dev()
    q, k, v = (t.to(dev) for t in _qkv(1, 2, 1, 3000, 128, torch.float16))
    CG.run_attention(q, k, v, causal=False)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = CG.run_attention(q, k, v, causal=False)
    for seed in (6, 7, 8):
        for t, new in zip((q, k, v), _qkv(1, 2, 1, 3000, 128, torch.float16, seed)):
            t.copy_(new)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, CG.run_attention(q, k, v, causal=False)), seed
