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


def test_fold_choice_is_launchable():
    """Every choice is a kernel that exists, with parts that cover the keys and fit the scratch."""
    for dim in (64, 128, 256):
        for causal in (True, False):
            for bh in (1, 8, 36, 128, 1000):
                for sq, sk in ((17, 17), (100, 4000), (300, 300), (4096, 4096), (5000, 90)):
                    cost, (w64, waves, per) = A._fold_choice(bh, sq, sk, dim, causal)
                    assert cost > 0 and waves in ((8, 4) if dim <= 128 else (4,))
                    assert not w64 or (dim == 128 and A.use_w64(dim, causal, sq, sk))
                    if per is not None:
                        most = -(-(min(sq, sk) if causal else sk) // A.BLOCK_N)
                        assert waves == 4 and 2 <= per < most
                        assert -(-most // per) * bh * sq * (dim + 2) * 4 <= A.MAX_STATE_BYTES
    # a full chip keeps whole keys and the largest blocks; few heads over long keys are split
    assert A._fold_choice(128, 4096, 4096, 128, True)[1] == (True, 8, None)
    assert A._fold_choice(36, 100, 4000, 128, False)[1][2] is not None
    assert A._short_wins(1, 16, 1 << 15, 128, False) and not A._short_wins(128, 4096, 4096, 128, True)


def test_metadata_calls_choose_no_launch():
    """Meta and fake tensors, symbolic sizes among them, return shapes only."""
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.symbolic_shapes import ShapeEnv

    q = torch.empty(2, 3, 5, 64, dtype=torch.bfloat16, device="meta")
    out, lse = A.run_attention(q, q, q, causal=False, return_lse=True)
    assert out.shape == q.shape and lse.shape == q.shape[:3] and lse.dtype == torch.float32
    mode = FakeTensorMode(shape_env=ShapeEnv())
    real = torch.empty(2, 3, 40, 64, dtype=torch.bfloat16)
    fake = mode.from_tensor(real)
    with mode:
        assert A.run_attention(fake, fake, fake).shape == real.shape


def test_short_chunks_bound_the_scratch():
    for units in (1, 100, 257, 480, 4096, 4097, 100000):
        chunks, _ = A.short_chunks(units, 1 << 20)
        assert chunks == 1 or chunks * units <= A.SHORT_MAX_WORKGROUPS
