"""GPU: Siddon projections in which rays parallel to an axis pass beside the volume, on either side of it, in the same
wavefront as rays that hit it: parallel beams onto detectors larger than the volume, and cone beams whose central row or
column passes 0.3 voxels above, below or beside it.  Against the FP64 oracle; tolerances as in the other projector tests:
1e-5 in L2 and 1e-4 of the largest value at a pixel, and 0 at pixels whose rays stay a voxel away from the volume."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd.geometry import cone_geometry, prepared

pytestmark = pytest.mark.gpu
SHAPE = (30, 34, 38)
ANGLES = np.array([0.0, 0.4, np.pi / 2, 2.2, np.pi, 4.0, 1.5 * np.pi])


def _geometry(case):
    detector, pixel, offset = (49, 57), 1.6, (0.0, 0.0, 0.0)
    if case == "parallel":
        detector, pixel = (48, 56), 1.1
    else:
        half = {"above": (-15.3, 0, 0), "below": (15.3, 0, 0), "left": (0, 17.3, 0), "right": (0, -17.3, 0),
                "front": (0, 0, 19.3), "back": (0, 0, -19.3)}
        offset = half[case]
    geo = cone_geometry(SHAPE, tuple(float(n) for n in SHAPE), detector, (pixel, pixel), 1000.0, 1536.0)
    geo.offOrigin = np.array(offset, dtype=np.float64)
    if case == "parallel":
        geo.mode = "parallel"
    return geo


@pytest.mark.parametrize("case", ["parallel", "above", "below", "left", "right", "front", "back"])
def test_rays_beside_the_volume(cuda, case):
    import torch

    geo = _geometry(case)
    img = (0.5 + np.random.default_rng(8).random(SHAPE)).astype(np.float32)
    x = torch.from_numpy(img).to(cuda)
    got = tigre_amd.Ax(x, geo, ANGLES, "Siddon").cpu().numpy()
    ref = oracle.ax(img, prepared(geo, ANGLES), "Siddon")
    err = oracle.rel_l2(got, ref)
    worst = float(np.max(np.abs(got - ref))) / float(np.max(np.abs(ref)))
    print("%s rel-L2 %.3e max %.3e" % (case, err, worst), flush=True)
    assert err <= 1e-5 and worst <= 1e-4
    if case == "parallel":
        v = 1.1 * np.abs(np.arange(48) - 23.5)
        assert np.all(got[:, v > SHAPE[0] / 2 + 1] == 0.0)
    for i in (0, 1, 4):  # the same bits alone as in company
        assert np.array_equal(tigre_amd.Ax(x, geo, ANGLES[i : i + 1], "Siddon").cpu().numpy(), got[i : i + 1])
