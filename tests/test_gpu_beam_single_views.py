"""GPU: forward projections of views too far apart to share a workgroup, whose detector tile is 32 x 16 pixels or, with
pixels well below a voxel, 32 x 32: both kinds, on either side of the rule and on detectors that no tile divides, against
the FP64 oracle and, to the bit, against each view projected alone (in tiles of another shape).

Tolerances as in the other projector tests: 1e-5 in L2 and 1e-4 of the largest value at a pixel."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd.geometry import cone_geometry, prepared
from tigre_amd.phantom import ellipsoid_phantom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["Siddon", "interpolated"])
@pytest.mark.parametrize("ratio", [1.0, 0.75, 0.7, 0.3, 0.1])  # a pixel's width on the axis over a voxel's
@pytest.mark.parametrize("detector", [(257, 289), (256, 256)])
def test_single_view_groups(cuda, kind, ratio, detector):
    import torch

    shape = (44, 57, 51)
    angles = np.array([0.1, 0.9, 1.7, 3.0, 4.1, 5.3])
    geo = cone_geometry(shape, tuple(float(n) for n in shape), detector, (1.536 * ratio,) * 2, 1000.0, 1536.0)
    img = (ellipsoid_phantom(shape, geo.sVoxel, 5, seed=4) + 0.2 * np.random.default_rng(3).random(shape)).astype(np.float32)
    x = torch.from_numpy(img).to(cuda)
    got = tigre_amd.Ax(x, geo, angles, kind)
    ref = oracle.ax(img, prepared(geo, angles), kind)
    err = oracle.rel_l2(got.cpu().numpy(), ref)
    worst = float(np.max(np.abs(got.cpu().numpy() - ref))) / float(np.max(np.abs(ref)))
    print("%s %g rel-L2 %.3e max %.3e" % (kind, ratio, err, worst), flush=True)
    assert err <= 1e-5 and worst <= 1e-4
    for i in range(len(angles)):
        assert torch.equal(tigre_amd.Ax(x, geo, angles[i : i + 1], kind), got[i : i + 1]), i
