"""GPU: forward projections whose slab boxes exceed the LDS buffer even at one plane, so that rays read the staging copy
in global memory: both Siddon walks (views along the axes and across the diagonals) and the interpolated projector, in
both sweep directions of both principal axes, against the FP64 oracle and the same bits for every plan.

Tolerances as in the other projector tests: 1e-5 in L2 and 1e-4 of the largest value at a pixel."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd import _native
from tigre_amd.geometry import cone_geometry, prepared
from tigre_amd.phantom import ellipsoid_phantom
from tigre_amd.plan import Plan

pytestmark = pytest.mark.gpu

SLAB_FLOATS = 9216  # the beam kernel's LDS buffer for a slab
DSO, DSD = 1000.0, 1536.0


def _middle_box(shape, detector, pixel, angle):
    """Floats of the box that the beam of the whole detector crosses in the volume's middle plane, clipped to the volume."""
    nz, ny, nx = shape
    c, s = np.cos(angle), np.sin(angle)
    n_a = ny if abs(c) >= abs(s) else nx
    a, z = [], []
    for u in (-1, 1):
        for v in (-1, 1):
            du, dv = u * pixel * (detector[1] - 1) / 2, v * pixel * (detector[0] - 1) / 2
            src = np.array([DSO * c, DSO * s, 0.0])
            pix = np.array([-(DSD - DSO) * c - du * s, -(DSD - DSO) * s + du * c, dv])
            p = 0 if abs(c) >= abs(s) else 1
            t = -src[p] / (pix[p] - src[p])
            at = src + t * (pix - src)
            a.append(at[1 - p])
            z.append(at[2])
    width = min(max(a), n_a / 2) - max(min(a), -n_a / 2)
    height = min(max(z), nz / 2) - max(min(z), -nz / 2)
    return width * height


@pytest.mark.parametrize("kind", ["Siddon", "interpolated"])
@pytest.mark.parametrize("views", ["axes", "diagonals"])
def test_unstaged(cuda, kind, views):
    import torch

    shape, detector, pixel = (103, 118, 126), (8, 29), 24.0
    angles = np.array([0.05, 1.62, 3.2, 4.75]) if views == "axes" else np.pi / 4 + np.arange(4) * np.pi / 2 + 0.01
    for angle in angles:
        assert _middle_box(shape, detector, pixel, angle) > SLAB_FLOATS
    geo = cone_geometry(shape, tuple(float(n) for n in shape), detector, (pixel, pixel), DSO, DSD)
    img = (ellipsoid_phantom(shape, geo.sVoxel, 5, seed=4) + 0.2 * np.random.default_rng(3).random(shape)).astype(np.float32)
    x = torch.from_numpy(img).to(cuda)
    got = tigre_amd.Ax(x, geo, angles, kind)
    ref = oracle.ax(img, prepared(geo, angles), kind)
    err = oracle.rel_l2(got.cpu().numpy(), ref)
    worst = float(np.max(np.abs(got.cpu().numpy() - ref))) / float(np.max(np.abs(ref)))
    print("%s %s rel-L2 %.3e max %.3e" % (kind, views, err, worst), flush=True)
    assert err <= 1e-5 and worst <= 1e-4
    for per_group, planes in ((1, 1), (1, 8), (4, 4)):
        p = Plan(geo, angles, per_group, planes, 16)
        out = torch.full_like(got, float("nan"))
        p.ax(x, out, p.workspace(), _native.PROJ_SIDDON if kind == "Siddon" else _native.PROJ_INTERPOLATED)
        assert torch.equal(out, got), (per_group, planes)
        p.close()


@pytest.mark.parametrize("accuracy", [0.5, 1.5])
def test_unstaged_interpolated_large_planes(cuda, accuracy):
    """Planes of more than 2^24 floats: four of 4200 x 4200, seen by a detector that covers 1400 x 1400 of them.  FP32
    positions near 2900 are good to 2^-12 voxel, samples of random voxels change by as much and twelve or fewer are
    added: 3e-4 of the largest value; by the nearest voxel (accuracy 1.5) a sample within 2^-12 of a face takes
    another one, in at most 4 x 3 x 2^-11 = 0.6 % of the rays."""
    import torch

    shape, detector, pixel = (4200, 4200, 4), (8, 30), 60.0
    geo = cone_geometry(shape, tuple(float(n) for n in shape), detector, (pixel, pixel), 8000.0, 9000.0, accuracy=accuracy)
    angles = np.array([0.0])
    img = np.random.default_rng(6).random(shape, dtype=np.float32)
    got = tigre_amd.Ax(torch.from_numpy(img).to(cuda), geo, angles, "interpolated").cpu().numpy()
    ref = oracle.ax(img, prepared(geo, angles), "interpolated")
    off = np.abs(got - ref) / np.abs(ref).max()
    print("accuracy %g: max %.3e, over 3e-4: %d of %d" % (accuracy, off.max(), (off > 3e-4).sum(), off.size), flush=True)
    assert (off > 3e-4).mean() <= (0.0 if accuracy < 1 else 0.02)
