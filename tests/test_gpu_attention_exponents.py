"""The tile exponents that `launch_attention` returns are a tensor of their own: a caller that keeps
them keeps no workspace (V^T images, the states of split keys) alive."""
import pytest
import torch

import neptune_codegen as CG
from neptune_codegen import attention as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,causal,split", [((1, 2, 300, 128), True, False),
                                                ((1, 8, 2048, 64), True, True),
                                                ((1, 4, 700, 128), False, True)])
def test_exponents_hold_no_workspace(shape, causal, split):
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    B, H, S, D = shape
    assert (A._fold_plan(B * H, S, S, D, causal)[2] is not None) == split
    g = torch.Generator().manual_seed(7)
    q, k, v = (torch.randn(shape, generator=g).bfloat16().cuda() for _ in range(3))
    v[0, 1, 70, 5] = 2.0 ** 20       # a tile with an exponent
    print(f"launch_attention {shape} causal={causal}", flush=True)
    out, _, exps = CG.launch_attention(q, k, v, causal=causal)
    tiles = -(-S // A.BLOCK_N)
    assert exps.dtype == torch.int32 and exps.shape == (B * H * tiles,)
    held = exps.untyped_storage().nbytes()
    assert held == 4 * exps.numel()
    want = torch.zeros(B * H, tiles, dtype=torch.int32)
    want[1, 70 // A.BLOCK_N] = 6     # 2^(14 + e) <= 2^20
    assert torch.equal(exps.cpu().view(B * H, tiles), want)
    assert torch.equal(out, A._launch(q, k, v, None, causal, False, A.V_EXPONENT_MAX)[0])
