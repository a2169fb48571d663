"""The device's Huffman table build: the wavefronts of a workgroup take the
steps of the merge between two barriers each for itself, and one may be any
number of steps behind another.  The step (huffman_merge.h, compiled for the
host) must be the same whatever a wavefront ahead has stored already: in every
schedule the wavefronts meet at the same barriers, and the code lengths are
the host construction's."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from ptwm_amd import _native

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("merge") / "merge_lag.so")
    subprocess.run([CLANG, "-x", "hip", "--offload-host-only", "--rocm-path=/opt/rocm", "-std=c++17", "-O1", "-shared",
                    "-fPIC", "-I", os.path.join(HERE, "..", "ptwm_amd", "csrc"),
                    os.path.join(HERE, "host", "merge_lag.hip"), "-o", so], check=True)
    return ctypes.CDLL(so)


def depths(model, counts, lag, fill):
    c = np.sort(np.asarray(counts, np.uint32))
    d = np.zeros(256, np.uint32)
    p = ctypes.POINTER(ctypes.c_uint32)
    rc = model.merge_lag(c.ctypes.data_as(p), len(c), lag, ctypes.c_uint32(fill), d.ctypes.data_as(p))
    return d[:len(c)] if rc == 0 else None


def want(counts):
    """Code lengths by the host construction, sorted as the counts are."""
    f = np.zeros(256, np.uint32)
    f[:len(counts)] = np.sort(np.asarray(counts, np.uint32))
    n = np.zeros(256, np.uint8)
    _native.lib().ptwm_mi355x_huffman_code_lengths(f.ctypes.data_as(ctypes.c_void_p), n.ctypes.data_as(ctypes.c_void_p))
    return n[:len(counts)]


def histograms():
    for n in range(2, 257):
        yield [37] * n
    rng = np.random.default_rng(1)
    for k in range(300):
        n = int(rng.integers(2, 257))
        yield (rng.pareto(0.7 + 0.01 * k, n) * 50).astype(np.int64).clip(0, 1 << 20) + 1
        yield rng.integers(900, 1100, n)
        yield rng.integers(1, 4, n)
    yield [(1 << 24) - 1] * 256          # 2^32 - 256 in all
    yield [1 << 30, 1 << 30, 1 << 30, (1 << 30) - 1]  # 2^32 - 1


@pytest.mark.parametrize("fill", [0xFFFFFFFF, 0, 40])
def test_any_lag(model, fill):
    for counts in histograms():
        first = None
        for lag in (0, 1, 2):
            d = depths(model, counts, lag, fill)
            assert d is not None, (len(counts), lag, "the wavefronts part")
            assert first is None or np.array_equal(d, first)
            first = d
        if first.max() <= 11:
            assert np.array_equal(first, want(counts)), len(counts)
