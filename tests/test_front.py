"""The package where the native front (hexmi/_front.so) is absent or was built for another torch: the operators keep their route
through ctypes. No GPU."""
import importlib.util
import os
import subprocess
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
    assert type(front.softmax).__name__ == "Operator"
    with pytest.raises(AttributeError):
        front.no_such_operator
    with pytest.raises(TypeError):
        front.softmax(x=torch.zeros(4, 8))


def test_the_front_is_built_again_for_another_torch(monkeypatch, tmp_path):
    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(hexmi.__file__))), "build.py")
    spec = importlib.util.spec_from_file_location("hexmi_build_under_test", path)
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    ran = []

    def run(cmd, **kw):
        ran.append(cmd)
        open(cmd[cmd.index("-o") + 1], "w").close()
        return subprocess.CompletedProcess(cmd, 0, "", "")
    monkeypatch.setattr(build.subprocess, "run", run)
    monkeypatch.setattr(build, "OUT_FRONT", str(tmp_path / "_front.so"))
    monkeypatch.setattr(build, "FRONT_STAMP", str(tmp_path / "torch_front.cmd"))
    build.build_front()
    build.build_front()
    assert len(ran) == 1                                  # up to date
    monkeypatch.setattr(torch, "__version__", "99.0")
    build.build_front()
    assert len(ran) == 2 and '-DHEXMI_TORCH_VERSION="99.0"' in ran[1]
    monkeypatch.setattr(build, "HIPCC", "hipcc")          # found on PATH, or the usual place
    build.build_front()
    assert all(os.path.isdir(d) for c in ran for flag, d in zip(c, c[1:]) if flag == "-I")
    before = len(ran)
    monkeypatch.setitem(sys.modules, "torch", None)       # the C ABI's users need none
    build.build_front(force=True)
    assert len(ran) == before
