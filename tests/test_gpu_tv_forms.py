"""GPU: the TV steps in each of their forms (one pass an iteration, two, LDS tiles) on volumes at the edges of the rule
between them, ragged ones among them, against the FP64 oracle, in place as well.

Tolerance as in the other TV tests: a step moves a voxel by at most alpha and rounds it some twenty times at 2^-24 of
the image's range, and the normalised differences are 1-Lipschitz up to 1 / |difference|, kept above 0.01 by the
images' noise: after 2 steps the error is below 5e-6 of the range, 1e-5 in L2."""
import ctypes

import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd import _native

pytestmark = pytest.mark.gpu

# TV: 2^24 voxels and a plane more; nine planes, eight; LDS tiles of 128 columns filled and not, a second chunk of one plane
CASES = [("tv", (256, 256, 256)), ("tv", (257, 256, 256)), ("tv", (8, 1450, 1450)), ("tv", (9, 1400, 1400)),
         ("tv", (17, 1024, 1023)), ("awtv", (2, 1000, 1000)), ("awtv", (4, 1000, 1000)), ("awtv", (17, 513, 1025)),
         ("awtv", (250, 250, 250)), ("awtv", (90, 260, 254)), ("piccs", (8, 1024, 1024)), ("piccs", (7, 1024, 1024)),
         ("piccs", (17, 700, 1025))]


@pytest.mark.parametrize("kind,shape", CASES)
def test_tv_forms(cuda, kind, shape):
    import torch

    rng = np.random.default_rng(sum(shape))
    img, prior = rng.random(shape, dtype=np.float32), rng.random(shape, dtype=np.float32)
    x, p = torch.from_numpy(img).to(cuda), torch.from_numpy(prior).to(cuda)
    alpha, steps = 2.0, 2
    size = (ctypes.c_long * 3)(*shape[::-1])
    at = ctypes.c_void_p(x.data_ptr())
    lib = _native.lib()
    if kind == "tv":
        got, ref = tigre_amd.minTV(x, alpha, steps), oracle.pocs_tv(img, alpha, steps)
        st = lib.tigre_pocs_tv_device(at, at, alpha, size, steps, None)
    elif kind == "awtv":
        got, ref = tigre_amd.AwminTV(x, alpha, steps, delta=-0.3), oracle.aw_pocs_tv(img, alpha, steps, -0.3)
        st = lib.tigre_aw_pocs_tv_device(at, at, alpha, size, steps, -0.3, None)
    else:
        got, ref = tigre_amd.minPICCS(x, p, alpha, steps, ratio=0.6), oracle.piccs_tv(img, prior, alpha, 0.6, steps)
        st = lib.tigre_piccs_tv_device(at, ctypes.c_void_p(p.data_ptr()), at, alpha, 0.6, size, steps, None)
    _native.check(st, kind)
    torch.cuda.synchronize()
    err = oracle.rel_l2(got.cpu().numpy(), ref)
    print("%s %s rel-L2 %.3e" % (kind, shape, err), flush=True)
    assert err <= 1e-5
    assert torch.equal(x, got)
