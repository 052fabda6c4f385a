"""The native packing of raw batches (host code, no GPU) against numpy: bytes of
coordinates and element indices, extents, elements outside the list, and batches
large enough to be split over threads."""
import ctypes
import os
import subprocess
import sys
from ctypes import POINTER, byref, c_int, c_int64, c_void_p

import numpy as np
import pytest

from emsim_amd import atoms as atm
from emsim_amd.backend import hip_ext
from emsim_amd.batch import centred_thickness, element_indices

ELEMS = [1, 6, 7, 8, 16]


def _pack(mols, threads):
    off = np.zeros(len(mols) + 1, np.int64)
    np.cumsum([len(m) for m in mols], out=off[1:])
    lut = np.full(max(ELEMS) + 1, 255, np.uint8)
    lut[ELEMS] = np.arange(len(ELEMS))
    c = np.full((off[-1] + 1, 3), 7, np.float32)     # one row more: not written
    e = np.full(off[-1] + 1, 77, np.uint8)
    ext = np.full(len(mols), -1, np.float32)
    ptrs = c_void_p * len(mols)
    zs = [np.ascontiguousarray(m.elements, np.int64) for m in mols]
    bad = c_int(5)
    hip_ext.call("emsim_hip_pack_raw", len(mols), ptrs(*[m.coordinates.ctypes.data for m in mols]),
                 ptrs(*[z.ctypes.data for z in zs]), off.ctypes.data_as(POINTER(c_int64)),
                 lut.ctypes.data, lut.size, c.ctypes.data, e.ctypes.data, ext.ctypes.data, threads,
                 byref(bad))
    assert (c[-1] == 7).all() and e[-1] == 77
    return c[:-1], e[:-1], ext, bad.value


@pytest.mark.parametrize("sizes,threads", [([1], 1), ([0, 5, 0], 4), ([3, 100, 7000], 16),
                                           ([90000] * 5, 4), ([400000, 1], 16)])
def test_equals_numpy(sizes, threads):
    rng = np.random.default_rng(len(sizes))
    mols = [atm.AtomList(rng.choice(ELEMS, n), rng.normal(0, 30, (n, 3))) for n in sizes]
    c, e, ext, bad = _pack(mols, threads)
    assert bad == -1
    np.testing.assert_array_equal(c, np.concatenate([m.coordinates for m in mols]))
    np.testing.assert_array_equal(e, np.concatenate([element_indices(m, ELEMS) for m in mols]))
    assert [float(x) for x in ext] == [centred_thickness(m) for m in mols]


def test_outside_elements_and_nan():
    rng = np.random.default_rng(1)
    mols = [atm.AtomList(rng.choice(ELEMS, 50), rng.normal(0, 9, (50, 3))) for _ in range(4)]
    mols[2].elements[7] = 26
    mols[3].elements[0] = -1
    mols[1].coordinates[4, 0] = np.nan
    _, e, ext, bad = _pack(mols, 2)
    assert bad == 2 and e[107] == 255 and e[150] == 255
    assert np.isnan(ext[1]) and np.isfinite(ext[[0, 2, 3]]).all()


def test_bad_arguments():
    bad = c_int()
    raw = hip_ext.raw("emsim_hip_pack_raw")
    off = (c_int64 * 2)(0, 3)
    none = (c_void_p * 1)(None)
    lut = (ctypes.c_uint8 * 2)()
    assert raw(0, none, none, off, lut, 2, None, None, None, 1, byref(bad)) == hip_ext.EINVAL
    assert raw(1, none, none, off, lut, 2, None, None, None, 1, byref(bad)) == hip_ext.EINVAL


def test_bounds_and_runs_equal_numpy():
    """The bounds and element runs of atom lists equal numpy's reductions."""
    rng = np.random.default_rng(3)
    for n in (1, 2, 999):
        m = atm.AtomList(rng.choice(ELEMS, n), rng.normal(0, 30, (n, 3)))
        np.testing.assert_array_equal(m.r_min, m.coordinates.min(axis=0))
        np.testing.assert_array_equal(m.r_max, m.coordinates.max(axis=0))
        np.testing.assert_array_equal(m.space, m.r_max - m.r_min)
        s, zs, counts = atm.sort_elements_and_count(m)
        ref = np.unique(m.elements, return_counts=True)
        np.testing.assert_array_equal(zs, ref[0])
        np.testing.assert_array_equal(counts, ref[1])
        assert counts.dtype == ref[1].dtype and zs.dtype == ref[0].dtype
    with pytest.raises(ValueError):
        atm.AtomList(np.zeros(0, int), np.zeros((0, 3))).space


NEW = r"""
#include <cstdlib>
#include <new>
static bool failing = false;
extern "C" void fail_new(int on) { failing = on; }
void* operator new(std::size_t n) {
    void* p = failing ? nullptr : std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
"""
PACK = """
import ctypes
import numpy as np
from emsim_amd import atoms as atm
from tests.test_pack_raw import ELEMS, _pack
mols = [atm.AtomList(np.full(150000, 6), np.full((150000, 3), k, np.float32)) for k in range(4)]
fail = ctypes.CDLL(None).fail_new
call = __import__("emsim_amd.backend.hip_ext", fromlist=["call"])
real = call.call
def failing(*args):
    fail(1)
    try:
        return real(*args)
    finally:
        fail(0)
call.call = failing
c, e, ext, bad = _pack(mols, 4)
assert bad == -1 and (e == ELEMS.index(6)).all()
assert (c == np.repeat(np.arange(4), 150000)[:, None]).all()
print("packed")
"""


def test_no_memory_for_a_thread(tmp_path):
    """A thread that cannot be had for want of memory is no error: the call's own
    thread packs everything."""
    src, lib = tmp_path / "new.cpp", tmp_path / "libnew.so"
    src.write_text(NEW)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", str(src), "-o", str(lib)], check=True)
    env = dict(os.environ, LD_PRELOAD=" ".join([str(lib), os.environ.get("LD_PRELOAD", "")]).strip())
    out = subprocess.run([sys.executable, "-c", PACK], env=env, capture_output=True, text=True,
                         timeout=100, cwd=os.path.dirname(os.path.dirname(__file__)))
    assert out.returncode == 0 and "packed" in out.stdout, out.stderr[-500:]
