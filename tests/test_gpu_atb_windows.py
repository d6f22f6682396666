"""GPU: the staged backprojector at the edges of its windows, against the FP64 oracle: view counts around the 64
whose windows are computed together, columns and layers that fill no workgroup or XCD, windows at and beyond the
detector's border and beyond the staged size, and every number of slices per lane.

Tolerance: detector positions carry a few FP32 roundings, below 2e-5 pixel on these detectors, and the projections
change by less than their mean from pixel to pixel, so 1e-5 in relative L2 as for the other backprojection tests.  The
same bits for 4, 8 and 16 slices per lane, and 2e-6 between 32 and these, whose row positions are rounded differently
(4e-6 pixel at 40 rows)."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd import _native
from tigre_amd.geometry import cone_geometry, prepared
from tigre_amd.phantom import ellipsoid_phantom
from tigre_amd.plan import Plan

pytestmark = pytest.mark.gpu


def _case(name):
    if name == "odd":  # 10 x 4 columns of workgroups: a strip of 8 and one of 2, and a last layer of one slice
        return cone_geometry((33, 50, 150), (33.0, 50.0, 150.0), (47, 90), (1.3, 2.4), 400.0, 600.0)
    if name == "one":  # less than a workgroup, on a detector narrower than a staged row
        return cone_geometry((1, 3, 5), (1.0, 3.0, 5.0), (1, 2), (2.0, 3.0), 100.0, 150.0)
    if name == "border":  # the volume projects beyond the detector on every side
        geo = cone_geometry((50, 40, 44), (50.0, 40.0, 44.0), (21, 23), (1.1, 1.2), 150.0, 240.0)
        geo.offDetector = np.array([3.0, -7.0])
        return geo
    # "coarse": 2.4 rows a slice, so windows of 16 slices fit at some views and corners and not at others
    geo = cone_geometry((70, 64, 64), (140.0, 64.0, 64.0), (200, 90), (1.3, 1.3), 300.0, 460.0)
    return geo


@pytest.mark.parametrize("kind", ["FDK", "matched"])
@pytest.mark.parametrize("name,views", [("odd", 65), ("one", 130), ("border", 64), ("coarse", 63), ("odd", 1)])
def test_atb_windows(cuda, name, views, kind):
    import torch

    geo = _case(name)
    angles = np.linspace(0.2, 2 * np.pi + 0.2, views, endpoint=False)
    proj = oracle.ax(ellipsoid_phantom(geo.nVoxel, geo.sVoxel, 5, seed=views) + 0.1, prepared(geo, angles))
    proj = proj.astype(np.float32)
    ref = oracle.atb(proj, prepared(geo, angles), kind)
    btype = _native.BACKPROJ_FDK if kind == "FDK" else _native.BACKPROJ_MATCHED
    first = None
    for slices in (4, 8, 16):
        p = Plan(geo, angles, 4, 8, slices)
        got = torch.full(p.vol_shape, float("nan"), device="cuda")
        p.atb(torch.from_numpy(proj).to(cuda), got, p.workspace(), btype)
        err = oracle.rel_l2(got.cpu().numpy(), ref)
        print("Atb %s %s %d views %d slices rel-L2 %.3e" % (kind, name, views, slices, err))
        first = got if first is None else first
        assert err <= 1e-5 and torch.equal(got, first)
        p.close()


@pytest.mark.parametrize("kind", ["FDK", "matched"])
def test_atb_many_slices(cuda, kind):
    """A volume of 2048 workgroups with 32 slices each, the last layer of eight."""
    import torch

    geo = cone_geometry((40, 512, 507), (40.0, 512.0, 507.0), (60, 300), (1.3, 3.0), 2000.0, 2500.0)
    angles = np.array([0.3, 2.2, 4.0])
    proj = torch.rand((3, 60, 300), generator=torch.Generator(device="cuda").manual_seed(5), device="cuda")
    got = tigre_amd.Atb(proj, geo, angles, kind)
    p = Plan(geo, angles, 4, 8, 8)
    ref = torch.empty(p.vol_shape, device="cuda")
    p.atb(proj, ref, p.workspace(), _native.BACKPROJ_FDK if kind == "FDK" else _native.BACKPROJ_MATCHED)
    p.close()
    err = oracle.rel_l2(got.cpu().numpy(), ref.cpu().numpy())
    print("Atb %s 32 against 8 slices rel-L2 %.3e" % (kind, err))
    assert err <= 2e-6
