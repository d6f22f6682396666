"""GPU: backprojection into volumes of few slices and many columns (one slice of a fan beam up to a workgroup's sixteen
and one more), against the FP64 oracle, and the same bits as with four slices a lane up to sixteen slices."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd import _native
from tigre_amd.geometry import cone_geometry, prepared
from tigre_amd.plan import Plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["FDK", "matched"])
@pytest.mark.parametrize("slices", [1, 4, 5, 8, 9, 16, 17])
def test_few_slices(cuda, slices, kind):
    import torch

    geo = cone_geometry((slices, 768, 750), (float(slices), 768.0, 750.0), (slices + 2, 400), (1.5, 3.0), 2000.0, 2500.0)
    angles = np.array([0.3, 2.2, 4.0])
    proj = np.random.default_rng(slices).random((3, slices + 2, 400)).astype(np.float32)
    p_dev = torch.from_numpy(proj).to(cuda)
    got = tigre_amd.Atb(p_dev, geo, angles, kind)
    err = oracle.rel_l2(got.cpu().numpy(), oracle.atb(proj, prepared(geo, angles), kind))
    print("Atb %s %d slices rel-L2 %.3e" % (kind, slices, err), flush=True)
    assert err <= 1e-5
    plan = Plan(geo, angles, 4, 8, 4)
    four = torch.full_like(got, float("nan"))
    plan.atb(p_dev, four, plan.workspace(), _native.BACKPROJ_FDK if kind == "FDK" else _native.BACKPROJ_MATCHED)
    plan.close()
    assert torch.equal(got, four) if slices <= 16 else oracle.rel_l2(got.cpu().numpy(), four.cpu().numpy()) <= 2e-6
