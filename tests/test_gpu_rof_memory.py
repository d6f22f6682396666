"""GPU: the ROF denoiser where its two states do not fit: a memory pool of limited size makes the larger workspace fail,
and the iterations run on one state.  The same bits as with two states, and no error is left behind."""
import ctypes
import re

import numpy as np
import pytest

import tigre_amd
from tigre_amd import _native

pytestmark = pytest.mark.gpu


class _Props(ctypes.Structure):  # hipMemPoolProps
    _fields_ = [("allocType", ctypes.c_int), ("handleTypes", ctypes.c_int), ("locationType", ctypes.c_int),
                ("locationId", ctypes.c_int), ("security", ctypes.c_void_p), ("maxSize", ctypes.c_size_t),
                ("reserved", ctypes.c_ubyte * 56)]


def _hip():
    """The HIP runtime that is loaded."""
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(re.search(r"(/\S*libamdhip64\.so\S*)", f.read()).group(1))


class _SmallPool:
    """hipMallocAsync takes its blocks from a pool of `size` bytes."""

    def __init__(self, size):
        self.hip, self.pool, self.old = _hip(), ctypes.c_void_p(), ctypes.c_void_p()
        props = _Props(1, 0, 1, 0, None, size)  # pinned device memory, no handles, device 0
        assert self.hip.hipMemPoolCreate(ctypes.byref(self.pool), ctypes.byref(props)) == 0

    def __enter__(self):
        assert self.hip.hipDeviceGetMemPool(ctypes.byref(self.old), 0) == 0
        assert self.hip.hipDeviceSetMemPool(0, self.pool) == 0
        return self

    def fits(self, size):
        p = ctypes.c_void_p()
        st = self.hip.hipMallocAsync(ctypes.byref(p), ctypes.c_size_t(size), None)
        if st == 0:
            assert self.hip.hipFreeAsync(p, None) == 0
        self.hip.hipGetLastError()
        return st == 0

    def __exit__(self, *args):
        import torch

        torch.cuda.synchronize()
        assert self.hip.hipDeviceSetMemPool(0, self.old) == 0
        assert self.hip.hipMemPoolDestroy(self.pool) == 0


@pytest.mark.parametrize("iterations", [4, 7, 10])
@pytest.mark.parametrize("spacing", [(1.0, 1.0, 1.0), (0.7, 1.3, 2.0)])
def test_one_state(cuda, iterations, spacing):
    import torch

    shape = (61, 250, 301)
    voxels = (shape[0] + 2) * shape[1] * shape[2]
    img = np.random.default_rng(iterations).random(shape, dtype=np.float32)
    x = torch.from_numpy(img).to(cuda)
    want = tigre_amd.tvdenoise(x, iterations, 4.0, spacing=spacing)
    torch.cuda.synchronize()
    with _SmallPool(24 * voxels) as pool:  # one state of 16 bytes a voxel and a copy of the image, not two states
        if pool.fits(32 * voxels):
            pytest.skip("this runtime does not limit a pool")
        got = [tigre_amd.tvdenoise(x, iterations, 4.0, spacing=spacing) for _ in range(3)]  # one after the other
        assert all(torch.equal(g, want) for g in got)
        st = _native.lib().tigre_tvdenoising_device(
            ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(x.data_ptr()), 4.0, (ctypes.c_float * 3)(*spacing),
            (ctypes.c_long * 3)(*shape[::-1]), iterations, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        _native.check(st, "tvdenoise in place")
        assert torch.equal(x, want)
