"""The key under which a fold call's launch is kept holds the exact value of every parameter, of
any number type (no GPU)."""
import numpy as np
import pytest
import torch

from neptune_codegen import template as T


@pytest.fixture()
def key_of(monkeypatch):
    x = torch.empty(4, 8)

    class Plain:
        is_cuda, layout, dtype, device, shape = True, torch.strided, x.dtype, x.device, x.shape
        stride, data_ptr = x.stride, x.data_ptr

    monkeypatch.setattr(torch, "Tensor", Plain)
    return lambda **params: T._fold_seen(Plain(), ("rmsnorm_max", "serial", None, None, False), params)[0]


def test_numbers_of_any_type_have_a_key(key_of):
    for value in (1e-6, 1, True, np.float64(1e-6), np.float32(1e-6), np.int64(3), np.float16(0.5)):
        assert key_of(eps=value) is not None, type(value)
        assert key_of(eps=value) == key_of(eps=value)


def test_keys_tell_values_apart(key_of):
    values = [1e-6, np.float64(1e-6), np.float64(1.0000000000000002e-06), np.float32(1e-6), 0.0, -0.0,
              np.float64(0.0), np.float64(-0.0), 1, 1.0, True]
    assert len({key_of(eps=v) for v in values}) == len(values)
    # a printed form that is not the value
    a, b = torch.tensor(0.1, dtype=torch.float64), torch.tensor(0.1 + 1e-12, dtype=torch.float64)
    assert repr(a) == repr(b) and key_of(eps=a) != key_of(eps=b)
    assert key_of(eps="x") is None
    assert key_of(eps=None) is None and key_of(eps=[1.0]) is None
