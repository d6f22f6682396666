"""GPU: backprojection of volumes that reach around the source, where columns of a workgroup lie on both sides of it and
their corners do not bound their detector positions, against the FP64 oracle; detectors narrow enough for a window.

Tolerance: no voxel is nearer than 0.05 voxels to the source's plane.  There the distance along the axis (FP32, of
numbers near 20: 2e-6) is good to 4e-5, so a position below 40 pixels is to 1.6e-3 and a sample of values below 1 to as
much; the weight is then one of the largest.  4e-3 of the largest value a view can add."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd.geometry import cone_geometry, prepared

pytestmark = pytest.mark.gpu

# n, DSO, DSD, detector (v, u), pixels (v, u)
CASES = [(20, 7.11, 9.1, (36, 20), (0.84, 2.75)), (48, 12.96, 38.62, (36, 30), (3.52, 4.24)),
         (32, 10.01, 13.61, (36, 20), (2.16, 2.34)), (20, 11.72, 14.88, (60, 3), (4.94, 2.84))]


def _clear_angles(n, DSO, count):
    """Angles at which no voxel is within 0.05 of the plane through the source across the central ray."""
    c = np.arange(n) - (n - 1) / 2
    x, y = np.meshgrid(c, c)
    found = [a for a in np.random.default_rng(n).uniform(0, 2 * np.pi, 20000)
             if np.abs(DSO - x * np.cos(a) - y * np.sin(a)).min() > 0.05]
    return np.array(found[:count])


@pytest.mark.parametrize("kind", ["matched", "FDK"])
@pytest.mark.parametrize("n,DSO,DSD,detector,pixel", CASES)
def test_source_inside(cuda, kind, n, DSO, DSD, detector, pixel):
    import torch

    geo = cone_geometry((n, n, n), (float(n),) * 3, detector, pixel, DSO, DSD)
    angles = _clear_angles(n, DSO, 6)
    assert len(angles) == 6
    proj = np.random.default_rng(3).random((6,) + detector).astype(np.float32)
    got = tigre_amd.Atb(torch.from_numpy(proj).to(cuda), geo, angles, kind).cpu().numpy()
    ref = oracle.atb(proj, prepared(geo, angles), kind)
    most = max(np.abs(oracle.atb(np.ones_like(proj[i:i + 1]), prepared(geo, angles[i:i + 1]), kind)).max() for i in range(6))
    off = float(np.abs(got - ref).max() / most)
    print("%s n %d: off by %.2e of %.2e" % (kind, n, off, most), flush=True)
    assert off <= 4e-3
