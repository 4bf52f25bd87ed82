"""Pages of output arrays that are mapped ahead of the threads that write them:
all of a small array; of a large one, where one thread would map slower than the
writing threads do, as many as fit behind the device's work, and the rest by all
threads where they read before they write."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import zisafvm_amd as z
from zisafvm_amd import workloads as W

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "zisafvm_amd", "csrc")
PAGE, PIECE = 4096, 64 * 4096


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pages") / "pages.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-fopenmp", "-w", "-shared", "-o", out,
                    os.path.join(HERE, "cpp", "pages.cpp"), os.path.join(CSRC, "setup.cpp"),
                    os.path.join(CSRC, "mesh.cpp")], check=True)
    lib = ctypes.CDLL(out)
    lib.map_whole_bytes.restype = ctypes.c_int64
    return lib


def _mapped(lib, n, skip=0, keep=0, all_=False, polls=0):
    got = (ctypes.c_ubyte * (n * 8 // PAGE + 16))()
    pages = lib.pages_mapped(ctypes.c_int64(n), ctypes.c_int64(skip), ctypes.c_int64(keep), int(all_), polls, got)
    assert pages > 0  # (-1: a value changed)
    return np.array(got[:pages], dtype=bool), skip * 8 // PAGE, (skip + n) * 8 // PAGE


@pytest.mark.parametrize("skip", [0, 2, 300, 511])
@pytest.mark.parametrize("pages", [40, 200, 700])
def test_small_arrays_are_mapped_whole(lib, pages, skip):
    n = pages * 512 - 100
    assert n * 8 < lib.map_whole_bytes()
    got, first, last = _mapped(lib, n, skip, keep=3)
    assert got[first:last].all()


@pytest.mark.parametrize("polls", [0, 1, 5, 10 ** 6])
@pytest.mark.parametrize("skip", [0, 300])
def test_large_arrays_are_mapped_while_the_device_is_busy(lib, skip, polls):
    n = (lib.map_whole_bytes() + 10 * PIECE) // 8
    got, first, last = _mapped(lib, n, skip, polls=polls)
    pieces = got[first:last].sum() * PAGE / PIECE
    assert got[first:last].all() if polls > 100 else polls <= pieces <= polls + 1
    assert np.diff(got[first:last].astype(int)).sum() <= 0  # from the front


@pytest.mark.parametrize("polls", [0, 3])
@pytest.mark.parametrize("skip", [0, 2, 300])
@pytest.mark.parametrize("more", [0, 1, PAGE // 8, 5 * PIECE // 8 + 17])
def test_large_arrays_that_are_read_first_are_mapped_whole(lib, more, skip, polls):
    got, first, last = _mapped(lib, 2 * lib.map_whole_bytes() // 8 + 512 + more, skip, keep=2, all_=True, polls=polls)
    assert got[first:last].all()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [200, 215, 290, 300])  # 3.2, 3.7, 6.7 and 7.2 MB
def test_large_states_and_tendencies(gpu, n):
    wl = W.vortex_2d(n=n, order=2)
    s = z.Solver(wl.mesh, wl.params)
    s.set_state(wl.u0)
    s.snapshot_begin()
    new = s.rate(wl.u0)
    np.testing.assert_array_equal(s.get_state(), wl.u0)
    np.testing.assert_array_equal(s.snapshot_end(), wl.u0)
    np.testing.assert_array_equal(s.rate(wl.u0, dudt=np.zeros_like(wl.u0)), new)
    base = np.random.default_rng(n).normal(size=wl.u0.shape)
    np.testing.assert_array_equal(s.rate(wl.u0, dudt=base.copy()), base + new)
