"""The Python extension of the linears (csrc/fast_linear.cpp) as a library."""

import os
import struct
import subprocess
import warnings

import pytest
import torch

from cider_amd import _lib

PT_TLS = 7


def test_no_thread_local_storage():
    # thread-local storage in a library loaded late slows every other library's
    # thread-local access (see the Makefile's -DNDEBUG)
    if not os.path.exists(_lib.FAST_PATH):
        pytest.skip("extension not built")
    with open(_lib.FAST_PATH, "rb") as f:
        elf = f.read()
    assert elf[:5] == b"\x7fELF\x02"
    phoff, = struct.unpack_from("<Q", elf, 32)
    size, count = struct.unpack_from("<HH", elf, 54)
    kinds = [struct.unpack_from("<I", elf, phoff + i * size)[0] for i in range(count)]
    assert PT_TLS not in kinds


@pytest.mark.parametrize("there", [False, True])
def test_linears_run_without_the_extension(monkeypatch, tmp_path, there):
    path = tmp_path / "_cider_fast.so"
    if there:
        path.write_bytes(b"built against another torch")
    monkeypatch.setattr(_lib, "FAST_PATH", str(path))
    monkeypatch.setattr(_lib, "_fast_linear", None)
    with pytest.warns(RuntimeWarning, match="make -C cider_amd/csrc"):
        f = _lib.fast_linear()
    assert f(0, None, None, None, None, 0, True) is None  # the general path
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _lib.fast_linear() is f  # said once


def test_build_follows_torch(tmp_path):
    # the extension's build: the C++ ABI of the torch that will load it, and built
    # again where torch, Python or a flag differs from the last build
    make = ["make", "-n", "-C", os.path.join(os.path.dirname(_lib.LIB_DIR), "csrc"),
            f"STAMP={tmp_path}/stamp", f"OUT={tmp_path}"]

    def planned(*more):
        out = subprocess.run([*make, *more], capture_output=True, text=True, check=True).stdout
        return [line for line in out.splitlines() if "fast_linear.cpp" in line]

    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    first, = planned()
    assert f"-D_GLIBCXX_USE_CXX11_ABI={abi} " in first
    assert torch.__version__ in (tmp_path / "stamp").read_text()
    for name in ("libcider_hip.so", "libcider_probe.so", "_cider_fast.so"):
        (tmp_path / name).touch()
    objects = ["-o", "libcider_hip.so", "-o", f"{tmp_path}/libcider_hip.so"]
    assert not planned(*objects)
    assert planned(*objects, "TORCH_VERSION=0.0")
    os.utime(tmp_path / "_cider_fast.so")
    assert planned(*objects, "PYINC=/elsewhere")
