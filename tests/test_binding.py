"""The native half of the Python binding converts what its wrappers documented
and refuses what ctypes refused (CPU: calls over no rows launch nothing)."""
import ctypes
import os
import subprocess
import sys

import pytest

import l2c


class Tensor:
    """What a wrapper needs of a GPU tensor."""

    def __init__(self, address, is_cuda=True):
        self.address, self.is_cuda = address, is_cuda

    def data_ptr(self):
        return self.address


class Stream:
    cuda_stream = 0


class Index(int):
    pass


T = Tensor(0x1000)


@pytest.mark.parametrize("stream", [0, Stream()])
@pytest.mark.parametrize("size", [16, Index(16)])
def test_accepted(stream, size):
    l2c.rmsnorm(T, T, T, size, 0, 1e-5, stream)
    l2c.rmsnorm(T, None, T, size, batch=0, eps=1, stream=stream)
    l2c.matmul_bf16(T, T, T, 0, 32, 1, stream=stream)
    l2c.to_bf16(T, T, 0, stream)
    l2c.to_bf16_x4(T, T, 0, stream)


def test_refused_by_the_library():
    with pytest.raises(l2c.L2CError):
        l2c.rmsnorm(T, T, T, 0, 1, stream=0)
    with pytest.raises(l2c.L2CError):
        l2c.rmsnorm(None, T, T, 4, 1, stream=0)
    with pytest.raises(l2c.L2CError):
        l2c.to_bf16_x4(T, T, 3, stream=0)


def test_refused_by_the_binding():
    with pytest.raises(ValueError):
        l2c.rmsnorm(T, Tensor(0x1000, is_cuda=False), T, 4, 0, stream=0)
    with pytest.raises(AttributeError):
        l2c.rmsnorm(T, 5, T, 4, 0, stream=0)
    with pytest.raises(AttributeError):
        l2c.rmsnorm(T, T, T, 4, 0, stream="default")
    with pytest.raises(ctypes.ArgumentError):
        l2c.rmsnorm(T, T, T, 4.0, 0, stream=0)
    with pytest.raises(ctypes.ArgumentError):
        l2c.rmsnorm(T, T, T, 4, 0, eps="small", stream=0)


def test_integers_past_the_c_type_wrap_as_in_ctypes():
    l2c.rmsnorm(T, T, T, (1 << 32) + 16, 1 << 32, stream=0)
    with pytest.raises(l2c.L2CError):
        l2c.rmsnorm(T, T, T, 16, (1 << 32) - 1, stream=0)


def test_every_entry_point_has_a_native_function():
    l2c.load()
    assert set(l2c._native) == set(l2c._ENTRIES)
    assert all("l2c_" + name in l2c.KERNEL_SYMBOLS for name in l2c._ENTRIES)


@pytest.mark.parametrize("python,built", [(sys.executable, True), ("/bin/false", False)])
def test_the_build_needs_no_python_headers(python, built):
    """Without Python.h the native half is left out, not the build refused."""
    recipes = subprocess.run(["make", "-n", "-B", "-C", l2c.PKG_DIR, f"PYTHON={python}"], capture_output=True, text=True,
                             check=True, timeout=120).stdout
    assert "lib/libl2c.so" in recipes
    assert ("host/python_binding.cpp" in recipes) == built
    assert (os.path.basename(l2c.NATIVE_PATH) in recipes) == built


def test_wrappers_without_the_native_half():
    """The same calls through ctypes, where l2c_native was not built for this Python."""
    code = """if True:
        import l2c
        l2c.NATIVE_PATH += ".absent"
        import test_binding as t
        l2c.load()
        assert not any("built-in" in repr(f) for f in l2c._native.values())
        for stream in (0, t.Stream()):
            for size in (16, t.Index(16)):
                t.test_accepted(stream, size)
        t.test_refused_by_the_library()
        t.test_refused_by_the_binding()
        t.test_integers_past_the_c_type_wrap_as_in_ctypes()
        t.test_every_entry_point_has_a_native_function()
        print("done")
    """
    path = os.pathsep.join([l2c.PKG_DIR, os.path.dirname(os.path.abspath(__file__))])
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300,
                         env=dict(os.environ, PYTHONPATH=path))
    assert run.returncode == 0 and run.stdout.endswith("done\n"), run.stderr[-2000:]
