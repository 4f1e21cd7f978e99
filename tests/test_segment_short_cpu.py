"""Channel chunks of segments shorter than one step of token rows (no GPU): wide on a full chip, two
words in bf16; segments of whole steps keep theirs."""
import pytest
import torch

from neptune_codegen import torch_op as TO


def _words(dtype, segments, tokens, channels):
    flat = torch.empty((segments * tokens, channels), dtype=dtype, device="meta")
    var = TO._segment_variant(flat, torch.empty(segments + 1, dtype=torch.int64, device="meta"), channels)
    assert var.vector
    return var.words


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_words_of_short_segments(dtype):
    small = 2 if dtype == torch.bfloat16 else 1
    for channels in (128, 256, 512):
        assert _words(dtype, 60000, 2, channels) == 4
        assert _words(dtype, 60000, 5, channels) == 4
        assert _words(dtype, 60000, 6, channels) == 2
        assert _words(dtype, 60000, 15, channels) == 2
        assert _words(dtype, 60000, 16, channels) == 1
        assert _words(dtype, 60000, 26, channels) == small
        assert _words(dtype, 60000, 32, channels) == 1
        assert _words(dtype, 300, 4, channels) == small
        assert _words(dtype, 300, 40, channels) == 1
    assert _words(dtype, 300, 11, 300) == small
    assert _words(dtype, 25000, 11, 300) == 4
    assert _words(torch.float32, 1500, 100, 100) == 1 and _words(torch.float32, 1500, 20, 100) == 2
