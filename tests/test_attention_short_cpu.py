"""The split of a head's keys into chunks (no GPU): every tile belongs to exactly one chunk, no
chunk is empty, and short key ranges stay whole."""
from neptune_codegen import attention as A
from neptune_codegen.emitters import ATTN_SHORT_TILE


def test_short_chunks_cover_the_keys_once():
    for units in (1, 2, 7, 64, 136, 255, 256, 257, 512, 5000, 70000):
        for sk in (1, 31, 32, 33, 128, 129, 500, 3000, 8192, 32768, 1 << 20):
            chunks, per = A.short_chunks(units, sk)
            tiles = -(-sk // ATTN_SHORT_TILE)
            assert 1 <= chunks <= A.SHORT_MAX_CHUNKS
            assert (chunks - 1) * per < tiles <= chunks * per
            assert chunks == 1 or per >= 1
    assert A.short_chunks(1, 128) == (1, 4)
    assert A.short_chunks(512, 3000)[0] == 1          # the heads fill the chip
    assert A.short_chunks(1, 1 << 20)[0] == A.SHORT_MAX_CHUNKS
