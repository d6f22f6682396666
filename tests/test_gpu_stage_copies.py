"""GPU: the projectors' staging copies at the edges of their 64 x 32 tiles, with views along x, along y and both,
against the FP64 oracle.

Tolerance: FP32 sums of at most 130 segments, 1e-5 in relative L2 as for the other projector tests; bfloat16 results
are rounded to 8 bits, 2^-9 at most, from volumes that bfloat16 holds exactly: 4e-3."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd.geometry import cone_geometry, prepared

pytestmark = pytest.mark.gpu

# (z, y, x): one voxel; copies that fill one tile exactly (56 + 8 by 24 + 8), one more either way, and several
SHAPES = [(1, 1, 1), (3, 24, 56), (2, 25, 57), (2, 57, 25), (1, 60, 121), (4, 33, 64)]
VIEWS = {"x": [0.05], "y": [np.pi / 2 + 0.05], "both": [0.3, 2.0, 4.1]}


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("views", sorted(VIEWS))
@pytest.mark.parametrize("kind", ["Siddon", "interpolated"])
def test_stage_copies(cuda, shape, views, kind):
    import torch

    geo = cone_geometry(shape, tuple(float(n) for n in shape), (9, 80), (1.1, 2.3), 400.0, 600.0)
    angles = np.array(VIEWS[views])
    img = torch.from_numpy(np.random.default_rng(sum(shape)).random(shape).astype(np.float32)).bfloat16()
    ref = oracle.ax(img.float().numpy(), prepared(geo, angles), kind)
    for dtype, tol in ((torch.float32, 1e-5), (torch.bfloat16, 4e-3)):
        got = tigre_amd.Ax(img.to(dtype).to(cuda), geo, angles, kind).float().cpu().numpy()
        err = oracle.rel_l2(got, ref)
        print("%s %s %s %s rel-L2 %.3e" % (kind, shape, views, dtype, err))
        assert err <= tol
