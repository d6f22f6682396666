"""GPU: the TV steps on volumes just beyond the sizes up to which a step takes the norm in a pass of its own, and just
below them, against the FP64 oracle.

Tolerance: as for the other TV tests.  A step moves a voxel by at most alpha and rounds it some twenty times at 2^-24
of the image's range, and the normalised differences are 1-Lipschitz up to 1 / |difference|, kept above 0.01 by the
images' noise: after 2 steps the error is below 5e-6 of the range, 1e-5 in L2."""
import numpy as np
import pytest

import oracle
import tigre_amd

pytestmark = pytest.mark.gpu

# 2^23 voxels, one row of planes more; 2^25, one plane more
CASES = [("tv", (128, 256, 256)), ("tv", (129, 256, 256)), ("awtv", (129, 256, 256)),
         ("piccs", (128, 512, 512)), ("piccs", (129, 512, 512))]


@pytest.mark.parametrize("kind,shape", CASES)
def test_tv_passes(cuda, kind, shape):
    import torch

    rng = np.random.default_rng(sum(shape))
    img, prior = rng.random(shape, dtype=np.float32), rng.random(shape, dtype=np.float32)
    x, p = torch.from_numpy(img).to(cuda), torch.from_numpy(prior).to(cuda)
    alpha, steps = 2.0, 2
    if kind == "tv":
        got, ref = tigre_amd.minTV(x, alpha, steps), oracle.pocs_tv(img, alpha, steps)
    elif kind == "awtv":
        got, ref = tigre_amd.AwminTV(x, alpha, steps, delta=-0.3), oracle.aw_pocs_tv(img, alpha, steps, -0.3)
    else:
        got, ref = tigre_amd.minPICCS(x, p, alpha, steps, ratio=0.6), oracle.piccs_tv(img, prior, alpha, 0.6, steps)
    err = oracle.rel_l2(got.cpu().numpy(), ref)
    print("%s %s rel-L2 %.3e" % (kind, shape, err))
    assert err <= 1e-5
