"""Host side of the readout: the pool of large arrays and the stepper's replay start."""
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

from pypybox2d_amd import layout as L
from pypybox2d_amd._native import host_copy
from pypybox2d_amd.stepper import Stepper


def test_pool_never_hands_out_memory_that_is_still_referred_to():
    pool = L.ArrayPool()
    shape = (2000, 28)
    a = pool.get("x", shape, np.float64)
    a[:] = 1.0
    row = a[5]  # a view keeps the memory
    addr = a.ctypes.data
    del a
    b = pool.get("x", shape, np.float64)
    b[:] = 2.0
    assert b.ctypes.data != addr and np.all(row == 1.0)
    del row
    c = pool.get("x", (1999, 28), np.float64)  # free again, and large enough
    assert c.ctypes.data == addr and c.shape == (1999, 28)
    held = [pool.get("x", shape, np.float64) for _ in range(4)]
    assert len({h.ctypes.data for h in held} | {b.ctypes.data, c.ctypes.data}) == 6
    assert len(pool._blocks["x"]) == 2  # bounded
    assert pool.get("x", shape, np.int32).dtype == np.int32
    y = pool.get("y", shape, np.float64)
    y[:] = 3.0
    z = pool.get("y", (1900, 28), np.float64, over=y)  # the caller gives y up for it
    assert z.ctypes.data == y.ctypes.data and np.all(z == 3.0)
    assert pool.get("y", (5000, 28), np.float64, over=z).ctypes.data != z.ctypes.data


def test_threaded_copy_copies_every_byte():
    for n in (0, 1, 100, (4 << 20) // 8 - 1, (4 << 20) // 8, 3_000_001):
        src = np.arange(n, dtype=np.float64)
        assert np.array_equal(host_copy(src, np.zeros(n)), src)
    src = np.arange(24.0).reshape(4, 6)
    assert np.array_equal(host_copy(src[:, ::2], np.zeros((4, 3))), src[:, ::2])


NEW_FAILS = r"""
#include <cstdlib>
#include <new>
extern "C" { long new_fails_at = -1; }
void* operator new(std::size_t n) {
  if (new_fails_at >= 0 && new_fails_at-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
"""

COPY = r"""
import ctypes, sys
import numpy as np
from pypybox2d_amd._native import host_copy, load
load()
fails = ctypes.c_long.in_dll(ctypes.CDLL(sys.argv[1]), "new_fails_at")
src = np.arange(4_000_001, dtype=np.float64)
for at in range(12):
    fails.value = at
    out = host_copy(src, np.zeros_like(src))
    fails.value = -1
    assert np.array_equal(out, src), at
print("copied")
"""


def test_threaded_copy_without_memory_for_its_threads(tmp_path):
    """An allocation that fails while the copying threads start: no exception leaves the C entry and no
    running thread is dropped (either would end the process)."""
    if not shutil.which("g++"):
        pytest.skip("no C++ compiler")
    (tmp_path / "n.cpp").write_text(NEW_FAILS)
    lib = str(tmp_path / "libn.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", lib, str(tmp_path / "n.cpp")], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, LD_PRELOAD=" ".join(filter(None, [lib, os.environ.get("LD_PRELOAD")])))
    r = subprocess.run([sys.executable, "-c", COPY, lib], cwd=root, env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "copied" in r.stdout, (r.returncode, r.stderr[-500:])


class _Engine:
    def __init__(self, *a, **k):
        self.n = 0

    def upload(self, b):
        pass

    def download(self):
        self.n += 1
        b = L.BatchArrays.empty_world()
        b.body_d = np.full((3, L.BODY_ND), float(self.n))
        b.body_i = np.zeros((3, L.BODY_NI), np.int32)
        b.fix_d = np.full((2, L.FIX_ND), 7.0)
        b.fix_d[:, L.FD_FAT_LX:L.FD_FAT_LX + 4] = self.n
        b.con_d = np.full((self.n, L.CON_ND), float(self.n))
        b.con_i = np.full((self.n, L.CON_NI), self.n, np.int32)
        return b

    def close(self):
        pass


def test_replay_start_is_apart_from_the_state_given_out():
    s = Stepper("fp32", 0, engine_factory=_Engine)
    start = _Engine().download()
    s.upload(start)
    for n in range(1, 5):
        st = s.download()
        want = {f: getattr(st, f).copy() for f in L.ALL_FIELDS}
        for f in L.ALL_FIELDS:
            getattr(st, f)[...] = -5
        for f in L.ALL_FIELDS:
            assert np.array_equal(getattr(s._ckpt, f), want[f]), (n, f)


def test_replay_start_survives_a_readout_without_memory_for_its_own():
    s = Stepper("fp32", 0, engine_factory=_Engine)
    s.upload(_Engine().download())
    s.download()
    want = {f: getattr(s._ckpt, f).copy() for f in L.ALL_FIELDS}
    s._log.append(("pairs",))

    class Pool:
        def get(self, name, shape, dtype, over=None):
            if name == "con_i":
                raise MemoryError(name)
            return np.empty(shape, dtype)
    s._pool = Pool()
    with pytest.raises(MemoryError):
        s.download()
    for f in L.ALL_FIELDS:
        assert np.array_equal(getattr(s._ckpt, f), want[f]), f
    assert s._log == [("pairs",)]
