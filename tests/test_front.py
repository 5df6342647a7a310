"""The package where the native front (hexmi/_front.so) is absent or was built for another torch: the operators keep their route
through ctypes. No GPU."""
import sys
import types
import warnings

import pytest
import torch

import hexmi
from hexmi import ops


@pytest.mark.parametrize("native", [None, types.SimpleNamespace(torch_version="1.0", set_check=None, softmax=None)])
def test_without_a_native_front_that_loads(monkeypatch, native):
    monkeypatch.setitem(sys.modules, "hexmi._front", native)
    monkeypatch.delattr(hexmi, "_front", raising=False)
    if native is not None:
        monkeypatch.setattr(hexmi, "_front", native, raising=False)
    front = ops._Front()
    monkeypatch.setattr(ops, "_front", front)
    x = torch.zeros(4, 8)
    with pytest.warns(RuntimeWarning, match="_front.so"):
        assert front.softmax(x) is None
    with warnings.catch_warnings():                       # once
        warnings.simplefilter("error")
        assert front.layer_norm(x, None, None, 1e-5) is None and front.binary(0, x, x) is None and front.softmax(x) is None
        with pytest.raises(ValueError):                   # the operators go on to what ops.py does and refuses
            hexmi.matmul(x, x)
        if not torch.cuda.is_available():
            with pytest.raises(RuntimeError, match="needs a GPU"):
                hexmi.softmax(x)
        else:
            assert torch.equal(hexmi.softmax(x), torch.full((4, 8), 0.125))


def test_the_native_front_is_the_one_that_is_built():
    front = ops._Front()
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert front.softmax(torch.zeros(4, 8)) is None   # a host tensor is not of the plain form
    assert type(front.softmax).__name__ == "builtin_function_or_method"
    with pytest.raises(AttributeError):
        front.no_such_operator
