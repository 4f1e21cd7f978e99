"""Query blocks of attention over more K and V^T than the last cache holds (no GPU): every block reads
them from HBM again, so the larger blocks are taken there."""
from neptune_codegen import attention as A


def test_blocks_beyond_the_cache():
    def waves(bh, sq, sk, dim, causal=False):
        return A._fold_choice(bh, sq, sk, dim, causal)[1][1]

    assert waves(640, 601, 1184, 128) == 8 and waves(1120, 601, 601, 128) == 8
    # the same blocks within the cache
    assert waves(640, 601, 601, 128) == 4 and waves(160, 784, 784, 128) == 4
    for bh, sk in ((640, 1184), (600, 1100), (64, 600)):
        kv = bh * -(-sk // 64) * 64 * 128 * 4
        blocks = A._fold_blocks(640, -(-sk // 64) * 64, False, 128)
        cost = A._fold_cost(bh, 640, 128, False, 128, blocks, 1.15, 999)
        assert kv <= A.CACHE_BYTES or cost >= 5 * kv / A.CACHE_BYTES_PER_US
