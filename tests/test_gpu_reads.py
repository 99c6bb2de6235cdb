"""Blocking reads of a field: the same values whatever memory the caller gives
(plain, pinned or device memory) and whatever route the size takes."""
import ctypes
import threading

import numpy as np
import pytest

import smokesim

pytestmark = pytest.mark.gpu

# 56 KB and just below 4 MB (once the pinned slots are there, one copy into them);
# just above, where a thread takes each 2 MB slot (four of them), all eight with
# pieces of under 2 MB, and several pieces each
DIMS = [(29, 23, 21), (128, 128, 63), (128, 128, 65), (160, 151, 149), (187, 165, 160)]


class Memory:
    """Memory of the HIP runtime: pinned host memory or device memory."""

    def __init__(self, kind, nbytes):
        self.hip = ctypes.CDLL("libamdhip64.so")
        vp = ctypes.c_void_p
        self.hip.hipMemcpy.argtypes = [vp, vp, ctypes.c_size_t, ctypes.c_int]
        self.hip.hipFree.argtypes = self.hip.hipHostFree.argtypes = [vp]
        self.kind, self.n, self.p = kind, nbytes, vp()
        if kind == "pinned":
            assert self.hip.hipHostMalloc(ctypes.byref(self.p), ctypes.c_size_t(nbytes), 0) == 0
        else:
            assert self.hip.hipMalloc(ctypes.byref(self.p), ctypes.c_size_t(nbytes)) == 0

    def floats(self):
        out = np.empty(self.n // 4, np.float32)
        assert self.hip.hipMemcpy(out.ctypes.data, self.p, self.n, 4) == 0  # hipMemcpyDefault
        return out

    def free(self):
        assert (self.hip.hipHostFree if self.kind == "pinned" else self.hip.hipFree)(self.p) == 0


@pytest.mark.parametrize("dims", DIMS, ids=str)
@pytest.mark.parametrize("kind", ["pinned", "device"])
def test_read_targets(dims, kind):
    x = np.random.default_rng(3).standard_normal(dims[::-1]).astype(np.float32)
    with smokesim.Simulation(*dims, density=x) as g, smokesim.Simulation(187, 165, 160) as other:
        for _ in range(3):
            assert np.array_equal(g.get_density(0), x)
        other.get_density(0)  # 19 MB: the slots are there now
        assert np.array_equal(g.get_density(0), x)
        m = Memory(kind, x.nbytes)
        smokesim._check(g.lib.smoke_get_density(g.h, 0, ctypes.cast(m.p, ctypes.POINTER(ctypes.c_float))))
        assert np.array_equal(m.floats(), x.ravel())
        m.free()
        assert np.array_equal(g.get_density(0), x)


def test_readers_at_once():
    # One reader has the slots, the others copy the plain way.
    rng = np.random.default_rng(4)
    sims = [(smokesim.Simulation(*d), rng.standard_normal(d[::-1]).astype(np.float32))
            for d in [DIMS[4], DIMS[2], DIMS[4], DIMS[3]]]
    wrong = []

    def work(g, x):
        for k in range(8):
            y = x * np.float32(k + 1)
            g.set_density(0, y)
            if not np.array_equal(g.get_density(0), y):
                wrong.append((g.cell_shape, k))

    threads = [threading.Thread(target=work, args=p) for p in sims]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    for g, _ in sims:
        g.close()


def test_lives_of_one_read():
    # Simulations that are created, read and destroyed, below and above the
    # size at which the slots are built.
    x = np.random.default_rng(5).standard_normal(DIMS[4][::-1]).astype(np.float32)
    for k, n in enumerate([70, 160, 30, 160, 160]):
        y = x[:n]
        with smokesim.Simulation(187, 165, n, density=y) as g:
            assert np.array_equal(g.get_density(0), y), k
