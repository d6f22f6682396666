"""GPU: the Siddon projector's plane walk where it can go wrong, against the FP64 oracle, and the same bits for
every grouping of views and every slab depth.

Tolerance: positions are within 1e-7 voxel of the line and every ray is an FP32 sum of at most 1.8e3 segments, so
the relative error is below u sqrt(1.8e3) = 2.5e-6 for a ray of one sign; 1e-5 in L2 as for the other projector
tests, and 1e-4 of the largest value at a pixel (a crossing position's rounding moves the weight of one voxel)."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd.geometry import cone_geometry, prepared
from tigre_amd.phantom import ellipsoid_phantom
from tigre_amd.plan import Plan

pytestmark = pytest.mark.gpu


def _case(name):
    views = np.linspace(0.0, 2 * np.pi, 16, endpoint=False)
    if name == "diagonal":  # slopes on either side of 1 inside a detector tile: both walks in one workgroup
        geo = cone_geometry((20, 40, 40), (20.0, 40.0, 40.0), (24, 100), (1.0, 0.6), 90.0, 140.0)
        views = np.pi / 4 + np.concatenate([np.linspace(-0.2, 0.2, 9), np.pi / 2 + np.linspace(-0.1, 0.1, 4)])
    elif name == "axis":  # odd detector: central rays lie in voxel planes
        geo = cone_geometry((16, 18, 20), (16.0, 18.0, 20.0), (17, 33), (1.0, 1.0), 100.0, 150.0)
        views = np.arange(4) * np.pi / 2
    elif name == "thin":
        geo = cone_geometry((1, 9, 2), (1.0, 9.0, 2.0), (5, 19), (1.0, 1.0), 100.0, 150.0)
    elif name == "aside":  # most beams miss part of the volume, some all of it
        geo = cone_geometry((24, 30, 17), (24.0, 30.0, 17.0), (40, 70), (1.0, 1.1), 200.0, 300.0)
        geo.offOrigin = np.array([9.0, -14.0, 11.0])
        geo.offDetector = np.array([-6.0, 8.0])
    elif name == "anisotropic":
        geo = cone_geometry((33, 40, 21), (40.0, 20.0, 30.0), (37, 41), (1.7, 1.3), 150.0, 240.0)
    elif name == "coarse":  # a tile's box does not fit LDS: walked from the staging copy
        geo = cone_geometry((70, 70, 70), (70.0, 70.0, 70.0), (9, 9), (24.0, 24.0), 1000.0, 1536.0)
    else:  # "parted": the beams of a group part around the axis, leaving a slab outside the volume between two inside
        geo = cone_geometry((170, 230, 201), (170 * 256 / 230, 256.0, 201 * 256 / 230), (190, 243),
                            (409.6 / 243, 409.6 / 243), 1000.0, 1536.0)
        geo.offDetector = np.array([-3.1, 7.3])
        views = np.linspace(0, 2 * np.pi, 97, endpoint=False)[:8]
    return geo, views


@pytest.mark.parametrize("name", ["diagonal", "axis", "thin", "aside", "anisotropic", "coarse", "parted"])
def test_plane_walk(cuda, name):
    import torch

    geo, views = _case(name)
    g = np.random.default_rng(11)
    img = ellipsoid_phantom(geo.nVoxel, geo.sVoxel, 5, seed=3) + 0.2 * g.random(tuple(geo.nVoxel)).astype(np.float32)
    x = torch.from_numpy(img.astype(np.float32)).to(cuda)
    got = tigre_amd.Ax(x, geo, views)
    ref = oracle.ax(x.cpu().numpy(), prepared(geo, views))
    err = oracle.rel_l2(got.cpu().numpy(), ref)
    worst = float(np.max(np.abs(got.cpu().numpy() - ref))) / float(np.max(np.abs(ref)))
    print("Siddon %s rel-L2 %.3e max %.3e" % (name, err, worst))
    assert err <= 1e-5 and worst <= 1e-4
    for per_group in (1, 2, 4):
        for planes in (1, 2, 3, 4, 8):
            p = Plan(geo, views, per_group, planes, 16)
            out = torch.full_like(got, float("nan"))
            p.ax(x, out, p.workspace())
            assert torch.equal(out, got), (per_group, planes)
            p.close()
