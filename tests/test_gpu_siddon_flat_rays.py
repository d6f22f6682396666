"""GPU: Siddon rays nearly parallel to a principal axis that cross one voxel plane inside the volume, against the FP64
oracle: slopes from 1e-6 (just above those taken as zero) to 3e-3, in the detector's u and in v.

Tolerance, of the ray's own value: 64 cells of random voxels (sum 32, neighbours differ by at most 1).  The plane walk's
position is off by at most (1 + 64 / 2) 2^-32 voxel, which at its smallest slope of 2^-12 moves the crossing by 3.2e-5
cells: 1e-6.  The crossing walk below that slope rounds 64 crossing times, each by up to 64 2^-25 cells, with random
signs: rms 0.5 * 8 * 64 2^-25 / 32 * 0.4 = 1e-7.  FP32 sums add 64 terms: 64 2^-25 = 2e-6 at most.  4e-6."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd.geometry import cone_geometry, prepared

pytestmark = pytest.mark.gpu

SLOPES = [1e-6, 3e-6, 1e-5, 3e-5, 1e-4, 2e-4, 3e-4, 1e-3, 3e-3]


@pytest.mark.parametrize("angle", [0.0, np.pi / 2, np.pi, 3 * np.pi / 2])
@pytest.mark.parametrize("axis", ["u", "v"])
def test_flat_rays(cuda, axis, angle):
    import torch

    DSO, DSD = 1000.0, 1500.0
    geo = cone_geometry((64, 64, 64), (64.0, 64.0, 64.0), (4, 16), (1e-6, 1e-6), DSO, DSD)
    n = len(SLOPES)
    s = np.array(SLOPES)
    offs, det = np.zeros((n, 3)), np.zeros((n, 2))
    # the line leaves the voxel plane through the volume's middle behind at about its middle; the other axis half a
    # voxel off a plane
    if axis == "u":
        det[:, 1] = s * DSD
        offs[:, 1], offs[:, 2] = np.cos(angle) * s * DSO, -np.sin(angle) * s * DSO
        offs[:, 0] = 0.5
    else:
        det[:, 0] = s * DSD
        offs[:, 0] = s * DSO
        offs[:, 1], offs[:, 2] = 0.5 * np.cos(angle), -0.5 * np.sin(angle)
    geo.offOrigin, geo.offDetector = offs, det
    views = np.full(n, angle)
    img = np.random.default_rng(8).random((64, 64, 64)).astype(np.float32)
    ref = oracle.ax(img, prepared(geo, views))
    got = tigre_amd.Ax(torch.from_numpy(img).to(cuda), geo, views).cpu().numpy()
    assert ref.min() > 20
    err = np.abs(got / ref - 1).reshape(n, -1).max(axis=1)
    print(axis, angle, " ".join("%.0e: %.1e" % p for p in zip(SLOPES, err)), flush=True)
    assert err.max() <= 4e-6
