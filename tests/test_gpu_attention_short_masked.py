"""Causal calls on the short-query attention kernels: a V value reaches only the queries that see
its key.  Against the fp32 closed form of the visible keys, at blocks of one to 16 queries, keys
behind the last query, several query blocks, and a head's keys in several chunks (some wholly past
a block's diagonal).  Tolerances are the attention fold's: rtol 1.6e-2 / atol 1e-3 for O, fp32
rtol 1e-5 / atol 1e-6 for the logsumexp."""
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


def _qkv(B, H, Sq, Sk, D, dtype):
    g = torch.Generator().manual_seed(31)
    return [torch.randn(B, H, s, D, generator=g).to(dtype) for s in (Sq, Sk, Sk)]


def _lse(q, k):
    s = torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous()) / math.sqrt(q.shape[3])
    hidden = ~torch.ones(q.shape[2], k.shape[2], dtype=torch.bool).tril(0)
    return torch.logsumexp(s.masked_fill(hidden, float("-inf")), -1)


def _chunks(B, H, Sq, Sk, D):
    """Chunks of a causal call; the call takes the short-query kernels."""
    assert A._short_wins(B * H, Sq, Sk, D, True)
    return A.short_chunks(B * H * -(-Sq // A.ATTN_SHORT_BLOCK_M), min(Sq, Sk))[0]


# (heads, queries, keys, head dim, key of the value, chunks)
CASES = [(2, 1, 64, 128, 20, 1), (2, 5, 64, 128, 3, 1), (2, 5, 64, 128, 20, 1), (2, 16, 40, 64, 9, 1),
         (2, 16, 64, 128, 40, 1), (2, 16, 64, 256, 15, 1), (1, 16, 7, 128, 6, 1),
         (8, 512, 512, 128, 300, 1), (8, 512, 512, 256, 511, 1), (1, 700, 700, 256, 333, 5),
         (1, 512, 512, 256, 0, 4), (2, 300, 512, 256, 131, 1)]


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_masked_v_reaches_only_the_rows_that_see_it(case, dtype, value):
    dev = _dev()
    H, Sq, Sk, D, key, chunks = case
    assert _chunks(1, H, Sq, Sk, D) == chunks
    q, k, v = _qkv(1, H, Sq, Sk, D, dtype)
    col = D - 7
    v[0, 0, key, col] = value
    print(f"short attention, masked V {value} at key {key} of {H}x{Sq}x{Sk} d={D} {dtype}", flush=True)
    got, lse = (t.cpu().float() for t in CG.run_attention(q.to(dev), k.to(dev), v.to(dev),
                                                          causal=True, return_lse=True))
    clean = v.clone()
    clean[0, 0, key, col] = 0.0
    want = R.attention_reference(q, k, clean, causal=True).float()
    bad = got[0, 0, key:, col]
    assert torch.isnan(bad).all() if math.isnan(value) else (bad == value).all()
    keep = torch.ones_like(got, dtype=torch.bool)
    keep[0, 0, key:, col] = False
    torch.testing.assert_close(got[keep], want[keep], rtol=1.6e-2, atol=1e-3)
    torch.testing.assert_close(lse, _lse(q, k), rtol=1e-5, atol=1e-6)


def test_unwritten_future_keys_and_values():
    """A cache filled up to the queries: what lies behind them is NaN in K and V alike."""
    dev = _dev()
    q, k, v = _qkv(2, 3, 4, 200, 128, torch.bfloat16)
    want = R.attention_reference(q, k, v, causal=True).float()
    k[:, :, 4:], v[:, :, 4:] = float("nan"), float("nan")
    print("short attention, NaN behind the last query", flush=True)
    got = CG.run_attention(q.to(dev), k.to(dev), v.to(dev), causal=True).cpu().float()
    torch.testing.assert_close(got, want, rtol=1.6e-2, atol=1e-3)


@pytest.mark.parametrize("shape", [(1, 1, 512, 512), (1, 1, 700, 700), (1, 1, 700, 600), (1, 1, 300, 700)])
@pytest.mark.parametrize("causal", [True, False])
def test_several_blocks_in_several_chunks(shape, causal):
    """Query blocks whose diagonal ends before a chunk merge it as an empty state."""
    dev = _dev()
    B, H, Sq, Sk = shape
    assert A._short_wins(B * H, Sq, Sk, 256, causal)
    chunks = A.short_chunks(B * H * -(-Sq // A.ATTN_SHORT_BLOCK_M), min(Sq, Sk) if causal else Sk)[0]
    assert chunks > 1 or (causal and Sq == 300)
    q, k, v = _qkv(B, H, Sq, Sk, 256, torch.bfloat16)
    print(f"short attention {shape} d=256 causal={causal} in {chunks} chunks", flush=True)
    got, lse = (t.cpu().float() for t in CG.run_attention(q.to(dev), k.to(dev), v.to(dev),
                                                          causal=causal, return_lse=True))
    want = R.attention_reference(q, k, v, causal=causal).float()
    s = torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous()) / 16.0
    if causal:
        s = s.masked_fill(~torch.ones(Sq, Sk, dtype=torch.bool).tril(0), float("-inf"))
    torch.testing.assert_close(got, want, rtol=1.6e-2, atol=1e-3)
    torch.testing.assert_close(lse, torch.logsumexp(s, -1), rtol=1e-5, atol=1e-6)
