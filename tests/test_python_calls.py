"""The native module that carries the forward paths' calls (csrc/hipq_python.cpp): conversions and errors, without a GPU.  A call
without a context returns the library's error before it looks at anything else."""
import types

import numpy as np
import pytest
import torch


@pytest.fixture()
def native(hipq):
    return hipq._load_native()


def _linear(native, x, w=None, bias=None, m=2, ctx=0):
    native.hipq_linear_static_f32(ctx, x, 0.5, w, None, bias, m, 3, 4, 0, None)


def test_the_library_status_becomes_an_exception(hipq, native):
    for x in (None, 0, 4096, torch.zeros(2, 4), torch.nn.Parameter(torch.zeros(2, 4)), torch.zeros(0, 4)):
        for m in (2, np.int64(2), True, -1):
            with pytest.raises(hipq.HipqError) as e:
                _linear(native, x, m=m)
            assert e.value.code == hipq.INVALID_ARGUMENT and "'ctx'" in str(e.value)


def test_what_is_no_argument_is_refused(native):
    with pytest.raises(ValueError, match="dense row-major"):
        _linear(native, torch.zeros(4, 2).t())
    with pytest.raises(TypeError):
        _linear(native, torch.zeros(2, 4), m=2.0)
    with pytest.raises(TypeError):
        native.hipq_linear_static_f32(0, None, "0.5", None, None, None, 2, 3, 4, 0, None)
    with pytest.raises(TypeError):
        native.hipq_linear_static_f32(0)
    with pytest.raises(AttributeError):
        _linear(native, "x")
    with pytest.raises(TypeError):
        native.empty([2, 3], torch.float32, 0)
    with pytest.raises(TypeError):
        native.empty((2, 3), "float32", 0)


def test_a_tensor_without_data_raises(hipq, native):
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda x: _linear(native, x))(torch.zeros(2, 2, 4))
    with pytest.raises(Exception) as e:
        _linear(native, torch.sparse_coo_tensor(size=(2, 4)))
    assert not isinstance(e.value, hipq.HipqError)


def test_a_subclass_answers_for_itself(hipq, native):
    class Strided(torch.Tensor):
        def is_contiguous(self):
            return False

    with pytest.raises(ValueError, match="dense row-major"):
        _linear(native, torch.zeros(2, 4).as_subclass(Strided))


def test_addresses_of_blocks(native):
    a, b = torch.zeros(3), torch.zeros(4, 4).t()
    blocks = [{"a": a, "b": b}, types.MappingProxyType({"a": None, "c": a})]
    got = np.frombuffer(native.pointers(blocks, ("a", "b", "c")), dtype=np.uint64)
    assert got.tolist() == [a.data_ptr(), b.data_ptr(), 0, 0, 0, a.data_ptr()]
    assert native.pointers([], ("a",)) == b""
    with pytest.raises(TypeError):
        native.pointers(3, ("a",))
    with pytest.raises(AttributeError):
        native.pointers([{"a": "text"}], ("a",))


def test_the_module_is_built_again_for_another_torch(monkeypatch, tmp_path):
    """An incremental build leaves the module alone only where it was built against the python and the torch that are there."""
    from torsh_amd import build

    runs = []
    monkeypatch.setattr(build, "PYTHON_PATH", str(tmp_path / "_hipq_python.so"))
    monkeypatch.setattr(build, "PYTHON_STAMP", str(tmp_path / "_hipq_python.stamp"))

    def run(cmd, **kwargs):
        runs.append(cmd)
        open(cmd[cmd.index("-o") + 1], "w").close()
        return types.SimpleNamespace(returncode=0, stdout="", stderr="")

    monkeypatch.setattr(build.subprocess, "run", run)
    for expected in (1, 1):  # nothing there; all there
        build._build_python(False)
        assert len(runs) == expected
    monkeypatch.setattr(torch, "__version__", "0.0.1")
    for expected in (2, 2):
        build._build_python(False)
        assert len(runs) == expected
    build._build_python(True)
    assert len(runs) == 3
