"""GPU parity of two-pass rows around the widths from which only a lane's last slot may lie past the
row's end, aligned and not.  Tolerances are the folds': rtol 1e-5 / atol 1e-6 in fp32, 1.6e-2 / 1e-3
in 16 bits."""
import pytest
import torch

import neptune_codegen as CG
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


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["variance", "std"])
def test_two_pass_rows_but_for_the_last_slot(name, dtype):
    vec = 4 if dtype == torch.float32 else 8
    for lanes, slots in ((64, 1), (64, 3), (512, 8), (1024, 8)):
        whole = lanes * (slots - 1) * vec
        for width in {max(vec, whole - 1), max(vec, whole), whole + 1, whole + vec, whole + 3 * vec + 1,
                      lanes * slots * vec - 1, lanes * slots * vec}:
            for offset in (0, 1):
                x, dev = _rows(3, width, dtype, offset)
                print(f"two-pass {name} {dtype} width={width} offset={offset}", flush=True)
                rtol, atol = TOL[dtype]
                torch.testing.assert_close(CG.run(name, dev).cpu().float(), R.reference(name, x),
                                           rtol=rtol, atol=atol)
