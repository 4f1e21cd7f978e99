"""GPU parity of narrow rows of any width and alignment on both accesses that the number of elements
chooses between (one element per load, vectors).  Tolerances are the folds': rtol 1e-5 / atol 1e-6
in fp32, 1.6e-2 / 1e-3 in 16 bits."""
import pytest
import torch

import neptune_codegen as CG
from neptune_codegen import template as T
from oracle import references as R

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]
TOL = {torch.float32: (1e-5, 1e-6), torch.bfloat16: (1.6e-2, 1e-3), torch.float16: (1.6e-2, 1e-3)}


def _rows(rows, width, dtype, offset):
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")
    x = 2 * torch.randn(rows, width, generator=torch.Generator().manual_seed(width))
    x[:, 0], x[:, -1] = 9.0, -9.5
    x = x.to(dtype)
    store = torch.full((offset + rows * width,), float("nan"), dtype=dtype, device="cuda:0")
    dev = store[offset:].view(rows, width)
    dev.copy_(x)
    return x, dev


@pytest.mark.parametrize("few", [0, T.FEW_ELEMENTS])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["logsumexp", "softcap_lse", "stable_l2", "rmsnorm_max", "variance", "log_softmax"])
def test_narrow_rows(name, dtype, few, monkeypatch):
    monkeypatch.setattr(T, "FEW_ELEMENTS", few)
    monkeypatch.setattr(T, "_RUN_SEEN", {})
    params = {"rmsnorm_max": {"eps": 1e-6}, "softcap_lse": {"beta": 0.5}}.get(name, {})
    for width, offset in ((9, 1), (17, 0), (31, 3), (64, 5), (127, 0), (257, 7), (1001, 0)):
        x, dev = _rows(21, width, dtype, offset)
        print(f"narrow {name} {dtype} width={width} offset={offset} few={few}", flush=True)
        if name == "log_softmax":
            got, want = CG.run_log_softmax(dev), torch.log_softmax(x.float(), -1)
        else:
            got, want = CG.run(name, dev, **params), R.reference(name, x, **params)
        rtol, atol = TOL[dtype]
        torch.testing.assert_close(got.cpu().float(), want.float(), rtol=rtol, atol=atol)
