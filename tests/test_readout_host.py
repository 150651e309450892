"""Host side of the readout: the pool of large arrays and the stepper's replay start."""
import numpy as np

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


def test_threaded_copy_copies_every_byte():
    for n in (0, 1, 100, (4 << 20) // 8 - 1, (4 << 20) // 8, 3_000_001):
        src = np.arange(n, dtype=np.float64)
        assert np.array_equal(host_copy(src, np.zeros(n)), src)
    src = np.arange(24.0).reshape(4, 6)
    assert np.array_equal(host_copy(src[:, ::2], np.zeros((4, 3))), src[:, ::2])


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
