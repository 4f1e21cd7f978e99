"""Segment pooling over every channel chunking, bit-exact against the ordered oracle: chunk widths
of 1, 2 and 4 words, a last chunk that overlaps its neighbour, rows at odd alignments, segments
around whole steps (0, 1, 15..17, 31..33 tokens), few and many segments."""
import pytest
import torch

import neptune_codegen as CG
from neptune_codegen import torch_op as TO
from oracle import references as R

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 15, 16, 17, 0, 31, 32, 33, 64, 2]


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    return torch.device("cuda:0")


def _same(got, want):
    bits = torch.int32 if want.dtype == torch.float32 else torch.int16
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    assert torch.equal(torch.where(nan, 0, got.view(bits)), torch.where(nan, 0, want.view(bits)))


# (channels, repeats of LENGTHS): few lanes; rows of whole wavefronts; wide and two-word chunks
CASES = [(1, 1), (2, 1), (3, 1), (7, 1), (33, 1), (64, 1), (246, 1), (128, 300), (33, 2000), (100, 300),
         (300, 100), (50, 400), (36, 900)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("reduce", ["sum", "mean"])
def test_segment_chunks_bit_exact(reduce, dtype):
    dev = _dev()
    seen = set()
    for channels, repeats in CASES:
        lengths = torch.tensor(LENGTHS * repeats, dtype=torch.int32)
        rows = int(lengths.sum())
        data = torch.randn(rows, channels, generator=torch.Generator().manual_seed(channels)).to(dtype)
        want = R.segment_reference(data, lengths, reduce)
        for offset, pad in ((0, 0), (1, 3)):
            store = torch.zeros(offset + rows * (channels + pad), dtype=dtype, device=dev)
            view = store[offset:].view(rows, channels + pad)[:, :channels]
            view.copy_(data)
            var = TO._segment_variant(view, torch.empty(len(lengths) + 1, dtype=torch.int64), channels)
            seen.add((var.words, var.unroll, var.aligned))
            print(f"segment {reduce} {dtype} channels={channels} x{repeats} +{offset}/{pad} {var.tag()}", flush=True)
            _same(CG.run_segment_pool(view, lengths.to(dev), reduce=reduce).cpu(), want)
    assert {w for w, _, _ in seen} >= {1, 2, 4} and {a for _, _, a in seen} == {True, False}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_segment_long_and_few(dtype):
    """Few long segments (32 rows per step), their lengths around whole steps."""
    dev = _dev()
    lengths = torch.tensor([1000, 991, 0, 992, 993, 1023], dtype=torch.int64)
    for channels in (64, 77, 1024):
        data = torch.randn(int(lengths.sum()), channels, generator=torch.Generator().manual_seed(1)).to(dtype)
        var = TO._segment_variant(data, torch.empty(7, dtype=torch.int64), channels)
        assert var.unroll == 32 and var.words == 1
        print(f"segment long {dtype} channels={channels} {var.tag()}", flush=True)
        got = CG.run_segment_pool(data.to(dev), lengths.to(dev), reduce="sum").cpu()
        _same(got, R.segment_reference(data, lengths, "sum"))


def test_segment_data_beyond_4_gib():
    """Rows past the 32-bit byte range take 64-bit addresses; the last rows are at 4.3 GiB."""
    dev = _dev()
    channels, rows = 256, (1 << 23) + (1 << 19)
    data = torch.zeros(rows, channels, dtype=torch.float16, device=dev)
    data[-40:] = torch.randn(40, channels, generator=torch.Generator().manual_seed(2)).half().to(dev)
    offsets = torch.tensor([rows - 40, rows - 37, rows - 20, rows], dtype=torch.int64)
    assert not TO._segment_variant(data, offsets, channels).near
    got = CG.run_segment_pool(data, offsets.to(dev), reduce="sum", offsets=True).cpu()
    tail = data[-40:].cpu()
    want = R.segment_reference(tail, torch.tensor([3, 17, 20]), "sum")
    _same(got, want)
