"""GPU: Siddon line integrals across 1024 planes of one constant value, against the FP64 oracle.

Tolerance: adding the same value again and again rounds the same way each time.  One FP32 sum of 1024 values of 0.7
or 0.1 is off by 1.0e-5 of itself, sums of eights added up by 9.7e-7 (both in plain FP32 arithmetic); the rays' other
roundings (segment lengths, the scale) are a few 2^-24 and average out: 3e-6 on every ray that crosses the volume."""
import numpy as np
import pytest

import oracle
import tigre_amd
from tigre_amd.geometry import cone_geometry, prepared

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [0.7, 0.1])
@pytest.mark.parametrize("angle", [0.05, np.pi / 2 + 0.05, 0.3, np.pi + 0.6])
def test_constant_volume(cuda, value, angle):
    import torch

    shape = (4, 1024, 1024)
    geo = cone_geometry(shape, tuple(float(n) for n in shape), (3, 70), (0.9, 17.0), 4000.0, 6000.0)
    angles = np.array([angle])
    img = np.full(shape, value, np.float32)
    ref = oracle.ax(img, prepared(geo, angles), "Siddon")
    got = tigre_amd.Ax(torch.from_numpy(img).to(cuda), geo, angles, "Siddon").cpu().numpy()
    long = ref > 900 * value
    assert long.sum() > 60
    err = np.abs(got - ref)[long].max() / ref.max()
    print("value %g angle %.2f: %.3e" % (value, angle, err))
    assert err <= 3e-6
    assert oracle.rel_l2(got, ref) <= 3e-6
