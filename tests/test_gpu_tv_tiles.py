"""GPU: the TV steps at the edges of their tiles and chunks, against the FP64 oracle.

Tolerance: a step moves a voxel by at most alpha and rounds it some twenty times at 2^-24 of the image's range, and
the normalised differences are 1-Lipschitz up to 1 / |difference|, kept above 0.01 by the images' noise: after at most
4 steps the error is below 4 x 20 x 6e-8 = 5e-6 of the range, 1e-5 in L2 as for the other TV tests."""
import ctypes

import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd import _native

pytestmark = pytest.mark.gpu

# one voxel, one plane, one column; a tile of 63 columns exactly, one more, and of 123; tiles of two rows and one more;
# the last one takes tiles of eight rows, with a ragged tile on every side
SHAPES = [(1, 1, 1), (1, 5, 3), (4, 1, 1), (2, 2, 63), (3, 3, 64), (7, 4, 123), (5, 3, 124), (61, 133, 190)]


def _run(kind, img, prior, alpha, iterations):
    if kind == "tv":
        return tigre_amd.minTV(img, alpha, iterations)
    if kind == "awtv":
        return tigre_amd.AwminTV(img, alpha, iterations, delta=-0.3)
    return tigre_amd.minPICCS(img, prior, alpha, iterations, ratio=0.6)


def _ref(kind, img, prior, alpha, iterations):
    if kind == "tv":
        return oracle.pocs_tv(img, alpha, iterations)
    if kind == "awtv":
        return oracle.aw_pocs_tv(img, alpha, iterations, -0.3)
    return oracle.piccs_tv(img, prior, alpha, 0.6, iterations)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", ["tv", "awtv", "piccs"])
def test_tv_tiles(cuda, shape, kind):
    import torch

    rng = np.random.default_rng(sum(shape))
    img, prior = rng.random(shape).astype(np.float32), rng.random(shape).astype(np.float32)
    x, p = torch.from_numpy(img).to(cuda), torch.from_numpy(prior).to(cuda)
    for iterations in (0, 1, 2, 4):
        got = _run(kind, x, p, 0.05, iterations)
        ref = _ref(kind, img, prior, 0.05, iterations)
        # without a padding slice one voxel has no differences: 0 / 0 in both (PICCS)
        assert np.array_equal(np.isnan(got.cpu().numpy()), np.isnan(ref))
        err = oracle.rel_l2(np.nan_to_num(got.cpu().numpy()), np.nan_to_num(ref)) if np.any(ref == ref) else 0.0
        print("%s %s, %d iterations rel-L2 %.3e" % (kind, shape, iterations, err))
        assert err <= 1e-5
        assert torch.equal(got.nan_to_num(), _run(kind, x, p, 0.05, iterations).nan_to_num())
    if kind == "tv":  # in place
        want = tigre_amd.minTV(x, 0.05, 3)
        st = _native.lib().tigre_pocs_tv_device(ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(x.data_ptr()), 0.05,
                                                (ctypes.c_long * 3)(*shape[::-1]), 3, None)
        _native.check(st, "minTV")
        torch.cuda.synchronize()
        assert torch.equal(x, want)
