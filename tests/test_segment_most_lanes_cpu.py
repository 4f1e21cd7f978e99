"""Segment counts near the most lanes of a launch (no GPU): channel counts that fit it with 16-byte
chunks run the vector kernel, whose lanes then number fewer than 2^32."""
import pytest
import torch

from neptune_codegen import torch_op as TO


@pytest.mark.parametrize("dtype,channels", [(torch.float16, 128), (torch.bfloat16, 512), (torch.float32, 64),
                                            (torch.float32, 256), (torch.float16, 8), (torch.bfloat16, 300)])
def test_many_segments(dtype, channels):
    size = torch.empty(0, dtype=dtype).element_size()
    flat = torch.empty((1000, channels), dtype=dtype, device="meta")
    lanes = -(-channels * size // 16)       # with 16-byte chunks
    for nseg in (1000, TO.MOST_LANES // (4 * lanes) + 1, TO.MOST_LANES // (2 * lanes) + 1,
                 TO.MOST_LANES // lanes, TO.MOST_LANES // lanes + 1):
        spans = torch.empty(nseg + 1, dtype=torch.int32, device="meta")
        var = TO._segment_variant(flat, spans, channels)
        assert var.vector == (nseg * lanes <= TO.MOST_LANES)
        if var.vector:
            assert nseg * -(-channels * size // (4 * var.words)) <= TO.MOST_LANES
            assert channels * size >= 4 * var.words
    # the ordinary choice is untouched
    few = torch.empty(3001, dtype=torch.int32, device="meta")
    assert TO._segment_variant(torch.empty((60000, 128), dtype=torch.float16, device="meta"), few, 128).words == 1
