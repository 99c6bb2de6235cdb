"""Blocking reads of a field: the same values whatever memory the caller gives
(plain, pinned or device memory) and whatever route the size takes."""
import ctypes

import numpy as np
import pytest

import smokesim

pytestmark = pytest.mark.gpu

# 56 KB and just below 4 MB; just above, where pinned slots of 2 MB begin (four
# threads), all eight threads with pieces of under 2 MB, and several each
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
    with smokesim.Simulation(*dims, density=x) as g:
        for _ in range(3):
            assert np.array_equal(g.get_density(0), x)
        m = Memory(kind, x.nbytes)
        smokesim._check(g.lib.smoke_get_density(g.h, 0, ctypes.cast(m.p, ctypes.POINTER(ctypes.c_float))))
        assert np.array_equal(m.floats(), x.ravel())
        m.free()
        assert np.array_equal(g.get_density(0), x)
