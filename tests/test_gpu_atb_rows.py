"""GPU: row positions of the staged backprojector in views that are gathered (3.3 detector rows a slice: no window
fits).  A parallel beam has no weight, so with projections that hold their row number the result is the row position.

Tolerance, rows below 1760 (half an ulp is 6.1e-5): the position's two roundings (3.0e-5, 6.1e-5), the slice's (6.1e-5),
the sample's (6.1e-5), and the FP32 step (5.1e-5 over 853 rows) and origin (3.0e-5): 3e-4 rows.  Positions added up slice
by slice are off by 7e-4."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd.geometry import geometry, prepared

pytestmark = pytest.mark.gpu


def test_rows_of_gathered_views(cuda):
    import torch

    geo = geometry(mode="parallel", nVoxel=np.array([512, 20, 24]))
    geo.dVoxel = np.ones(3)
    geo.sVoxel = geo.nVoxel * geo.dVoxel
    geo.nDetector = np.array([1760, 40])
    geo.dDetector = np.array([0.3, 1.0])
    geo.sDetector = geo.nDetector * geo.dDetector
    angles = np.array([0.4])
    proj = np.broadcast_to(np.arange(1760, dtype=np.float32)[:, None], (1, 1760, 40)).copy()
    got = tigre_amd.Atb(torch.from_numpy(proj).to(cuda), geo, angles, "FDK")
    ref = oracle.atb(proj, prepared(geo, angles), "FDK")
    off = float(np.abs(got.cpu().numpy() - ref).max())
    print("rows off by %.2e" % off, flush=True)
    assert ref.max() > 1700 and off <= 3e-4
