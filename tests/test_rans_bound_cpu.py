"""The scratch of a reference rANS segment holds whatever the encoder sheds,
also where the entries do not fit the symbols (ref_rans.h compiled for the
host): the kernel then stores inside the segment's area by construction."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rans") / "rans_bound.so")
    subprocess.run([CLANG, "-x", "hip", "--offload-host-only", "--rocm-path=/opt/rocm", "-std=c++17", "-O1", "-shared",
                    "-fPIC", "-I", os.path.join(HERE, "..", "ptwm_amd", "csrc"),
                    os.path.join(HERE, "host", "rans_bound.hip"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.rans_bound.restype = ctypes.c_uint64
    lib.rans_bound.argtypes = [ctypes.c_uint64, ctypes.c_uint32, ctypes.c_uint32]
    lib.rans_identity.argtypes = [ctypes.c_uint32]
    return lib


@pytest.mark.parametrize("n", [0, 1, 31, 32, 33, 1000])
@pytest.mark.parametrize("tail", [0, 1, 31, 500])
def test_scratch(model, n, tail):
    assert model.rans_bound(n, tail, 7 * n + tail) == 0


def test_identity(model):
    assert all(model.rans_identity(x) for x in (0, 1 << 11, 1 << 23, (1 << 31) - 1))
