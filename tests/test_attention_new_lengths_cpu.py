"""Launch choices of attention calls whose lengths were not seen before (no GPU): the searches
equal their definition, and their work does not grow with the lengths -- a decode or a stream of
prompts has new ones in every call."""
import random
import sys

import pytest

from neptune_codegen import attention as A


def _steps(fn):
    """Lines (and loop steps) executed by fn()."""
    count = 0

    def trace(frame, event, arg):
        nonlocal count
        count += 1
        return trace

    sys.settrace(trace)
    try:
        fn()
    finally:
        sys.settrace(None)
    return count


def _chunks_by_definition(units, sk):
    tiles = -(-sk // A.ATTN_SHORT_TILE)

    def cost(chunks):
        rounds = -(-units * chunks // A.CUS)
        return (rounds * -(-tiles // chunks) * A.SHORT_TILE_US
                + (A.SHORT_MERGE_US + chunks * A.SHORT_CHUNK_US if chunks > 1 else 0.0))

    most = max(1, min(A.SHORT_MAX_CHUNKS, tiles // A.ATTN_SHORT_WAVES, A.SHORT_MAX_WORKGROUPS // units))
    chunks = min(range(1, most + 1), key=cost)
    per = -(-tiles // chunks)
    return -(-tiles // per), per


def test_chunks_are_the_cheapest():
    rng = random.Random(3)
    for _ in range(3000):
        units, sk = int(2 ** rng.uniform(0, 16)), int(2 ** rng.uniform(0, 20))
        assert A.short_chunks(units, sk) == _chunks_by_definition(units, sk), (units, sk)


@pytest.mark.parametrize("causal", [True, False])
def test_block_sums(causal):
    """Tiles and workgroups of a head, block by block."""
    rng = random.Random(4)
    for _ in range(3000):
        sq, sk = int(2 ** rng.uniform(0, 13)), int(2 ** rng.uniform(0, 14))
        bm, per = rng.choice([128, 256]), rng.randint(1, 70)
        tiles = [-(-(min(sk, (i + 1) * bm) if causal else sk) // A.BLOCK_N) for i in range(-(-sq // bm))]
        blocks = A._fold_blocks(sq, sk, causal, bm)
        assert (blocks[0], blocks[2], blocks[3]) == (len(tiles), tiles[-1], sum(tiles))
        assert A._fold_items(blocks, per, bm // A.BLOCK_N) == sum(-(-t // per) for t in tiles)


def test_the_choice_ends_its_search_only_past_the_best():
    """Every part count that fits, against the one chosen."""
    rng = random.Random(5)
    for _ in range(1000):
        bh, dim, causal = int(2 ** rng.uniform(0, 10)), rng.choice([64, 128, 256]), rng.random() < 0.5
        sq, sk = A.BLOCK_N * int(2 ** rng.uniform(0, 8)), A.BLOCK_N * int(2 ** rng.uniform(0, 9))
        blocks = A._fold_blocks(sq, sk, causal, 128)
        most = -(-(min(sk, sq) if causal else sk) // A.BLOCK_N)
        us = A._fold_choice(bh, sq, sk, dim, causal)[0]
        for parts in (1, 2, 3, 4, 6, 8, 12, 16):
            per = -(-most // parts)
            if parts > 1 and (per < 2 or parts * bh * sq * (dim + 2) * 4 > A.MAX_STATE_BYTES):
                break
            assert us <= A._fold_cost(bh, sq, dim, causal, 128, blocks, A.TILE_128_US[dim],
                                      per if parts > 1 else most + 4)


def test_searches_do_not_grow_with_the_lengths():
    for causal in (True, False):
        steps = [_steps(lambda: A._short_wins(32, n, n, 128, causal)) for n in (1021, 100_003)]
        assert max(steps) < 500, steps
    assert _steps(lambda: A.short_chunks(3, 999_983)) < 500


def test_growing_by_a_token_rarely_searches():
    A._tile_chunks.cache_clear()
    for sk in range(5000, 5320):
        A.short_chunks(32, sk)
    assert A._tile_chunks.cache_info().misses <= 11      # 32-key tiles
    A._tile_choice.cache_clear()
    for sk in range(5000, 5320):
        A._fold_choice(4, sk, sk, 64, True)
    assert A._tile_choice.cache_info().misses <= 6       # 64-key tiles
    A._short_cheaper.cache_clear()
    for sk in range(5000, 5320):
        A._short_wins(4, sk, sk, 64, True)
    assert A._short_cheaper.cache_info().misses <= 21    # 16-query blocks
