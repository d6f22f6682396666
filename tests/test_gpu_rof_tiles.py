"""GPU: the ROF denoiser at the edges of its tiles, chunks and passes, against the FP64 oracle.

Tolerance: the iteration is non-expansive in p and one iteration rounds u and p about ten times at 2^-24 of the
image's range, so after at most 10 iterations the error is below 10 * 10 * 6e-8 = 6e-6 of it: 1e-5 in L2."""
import ctypes

import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd import _native

pytestmark = pytest.mark.gpu

# one voxel; one slice (no mirror); a tile of 58 x 10 voxels exactly and one more; several chunks along z
SHAPES = [(1, 1, 1), (1, 7, 5), (2, 10, 58), (3, 11, 59), (45, 9, 64), (17, 31, 117)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("iterations", [0, 1, 2, 3, 4, 7, 9])
def test_rof_tiles(cuda, shape, iterations):
    import torch

    rng = np.random.default_rng(sum(shape))
    img = rng.random(shape).astype(np.float32)
    spacing = (1.0, 1.0, 1.0) if iterations % 2 else (0.7, 1.3, 2.0)
    x = torch.from_numpy(img).to(cuda)
    got = tigre_amd.tvdenoise(x, iterations, 4.0, spacing=spacing)
    ref = oracle.tvdenoise(img, 4.0, iterations, spacing)
    err = oracle.rel_l2(got.cpu().numpy(), ref)
    print("ROF %s, %d iterations rel-L2 %.3e" % (shape, iterations, err))
    assert err <= 1e-5
    assert torch.equal(x, torch.from_numpy(img).to(cuda))
    # in place
    st = _native.lib().tigre_tvdenoising_device(
        ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(x.data_ptr()), 4.0, (ctypes.c_float * 3)(*spacing),
        (ctypes.c_long * 3)(*shape[::-1]), iterations, None)
    _native.check(st, "tvdenoise")
    torch.cuda.synchronize()
    assert torch.equal(x, got)
