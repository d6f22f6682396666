"""GPU: Siddon line integrals of volumes with infinite and undefined voxels.

A ray is infinite or NaN by the voxels it has a segment in, and no other ray is touched: the rays of each such voxel
are those where the FP64 oracle's projection of that voxel alone is not zero (rays with less than 1e-3 of its largest
segment, or that a shift of the detector by 1e-3 mm takes off the voxel or onto it, are left out: a rounding decides).  All other rays agree with the oracle's projection of the finite voxels:
1e-4 of the largest value, as in the other projector tests."""
import copy

import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd.geometry import cone_geometry, prepared
from tigre_amd.plan import Plan

pytestmark = pytest.mark.gpu

VOXELS = [((9, 11, 13), np.inf), ((20, 7, 4), -np.inf), ((3, 25, 30), np.nan), ((9, 12, 13), np.inf)]
BLOCKS = [((2, 1, 1), np.inf), ((4, 3, 1), -np.inf), ((1, 2, 3), np.nan), ((2, 2, 1), np.inf)]  # of 20 voxels: rays are sparse


def _case(name):
    if name == "cone":  # odd detector: rays inside one row of voxels, tilted rays, both principal axes
        return cone_geometry((24, 30, 36), (24.0, 30.0, 36.0), (21, 57), (1.7, 1.3), 120.0, 190.0), \
            np.concatenate([np.arange(4) * np.pi / 2, np.linspace(0.1, 6.2, 9)])
    if name == "diagonal":  # slopes on either side of 1
        return cone_geometry((24, 30, 36), (24.0, 30.0, 36.0), (20, 100), (1.6, 0.9), 90.0, 140.0), \
            np.pi / 4 + np.linspace(-0.2, 0.2, 5)
    # "coarse": the box of a tile does not fit LDS
    return cone_geometry((120, 120, 120), (120.0, 120.0, 120.0), (9, 9), (24.0, 24.0), 1000.0, 1536.0), \
        np.array([0.1, 1.8, 3.3, 4.9])


@pytest.mark.parametrize("name", ["cone", "diagonal", "coarse"])
def test_nonfinite_voxels(cuda, name):
    import torch

    geo, views = _case(name)
    gp = prepared(geo, views)
    img = np.random.default_rng(2).random(tuple(geo.nVoxel)).astype(np.float32)
    want, aside = np.zeros((len(views),) + tuple(geo.nDetector)), np.zeros((len(views),) + tuple(geo.nDetector), bool)
    scale, bad = (20, BLOCKS) if name == "coarse" else (1, VOXELS)
    finite = img.copy()
    for at, value in bad:
        block = tuple(slice(scale * k, scale * k + scale) for k in at)
        alone = np.zeros_like(img)
        alone[block] = 1.0
        finite[block] = 0.0
        img[block] = value
        length = oracle.ax(alone, gp)
        with np.errstate(invalid="ignore"):
            want += np.where(length > 0, value, 0.0)
        aside |= (length > 0) & (length < 1e-3 * length.max())
        for shift in ((1e-3, 1e-3), (-1e-3, 1e-3), (1e-3, -1e-3), (-1e-3, -1e-3)):
            near = copy.deepcopy(geo)
            near.offDetector = np.array(shift)
            aside |= (length > 0) != (oracle.ax(alone, prepared(near, views)) > 0)
    x = torch.from_numpy(img).to(cuda)
    got = tigre_amd.Ax(x, geo, views).cpu().numpy()
    ref = oracle.ax(finite, gp)
    assert np.isinf(want).sum() >= 12 and np.isnan(want).sum() >= 6
    assert aside.mean() < 0.05  # the central column and row of a detector with an odd count
    keep = ~aside
    assert np.array_equal(np.isnan(got)[keep], np.isnan(want)[keep])
    inf = np.isinf(want) & keep
    assert np.array_equal(got[inf], want[inf])
    plain = (want == 0) & keep
    assert np.abs(got - ref)[plain].max() <= 1e-4 * np.abs(ref).max()
    for per_group, planes in ((1, 8), (4, 2)):
        p = Plan(geo, views, per_group, planes, 16)
        out = torch.zeros(got.shape, dtype=torch.float32, device=cuda)
        p.ax(x, out, p.workspace())
        assert np.array_equal(out.cpu().numpy(), got, equal_nan=True), (per_group, planes)
        p.close()
