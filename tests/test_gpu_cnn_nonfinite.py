"""GPU: weight gradients with one infinite input voxel: the taps that pair it with a voxel of the gradient are infinite
in its input channel, with that voxel's signs, and all others are those of the finite input (1e-5 in L2, as in the
other weight-gradient tests)."""
import numpy as np
import pytest

import oracle.cnn as ocnn
from tigre_amd import _native

from .test_gpu_cnn import _dev, _rand_bf16, _rel, _wgrad

pytestmark = pytest.mark.gpu

# segments that end in the volume or not, tiles of 8 rows that are full or not, chunks of planes
SHAPES = [(1, 3, 8, 32), (1, 5, 9, 33), (2, 4, 7, 47), (1, 21, 16, 40), (1, 1, 1, 1)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("modes", [(32, 32), (1, 32), (32, 1)])
def test_infinite_input(cuda, shape, modes):
    import torch

    rng = np.random.default_rng(sum(shape))
    cin, cout = modes
    n, D, H, W = shape
    x = _rand_bf16(rng, shape + (cin,))
    g = _rand_bf16(rng, shape + (cout,))
    g[g == 0] = 1.0
    dev = lambda a: _dev(a, torch.bfloat16) if a.shape[-1] == 32 else _dev(a[..., 0])  # noqa: E731
    mode = {32: _native.CNN_IN_BF16X32, 1: _native.CNN_IN_F32X1}
    edges = {(z, y, u) for z in (0, D - 1) for y in (0, H - 1) for u in (0, W - 1)} | {(D // 2, H // 2, W // 2)}
    for at in sorted(edges):
        i0 = int(rng.integers(cin))
        finite = x.copy()
        finite[(n - 1,) + at + (i0,)] = 0.0
        bad = finite.copy()
        bad[(n - 1,) + at + (i0,)] = np.inf
        out = _wgrad(dev(bad), mode[cin], dev(g), mode[cout], shape).cpu().numpy()
        ref = ocnn.conv3d_weight_grad(finite, g)
        plain = np.ones((27, cout, cin), bool)
        for tap in range(27):
            v = (at[0] - (tap // 9 - 1), at[1] - (tap // 3 % 3 - 1), at[2] - (tap % 3 - 1))
            if all(0 <= c < m for c, m in zip(v, (D, H, W))):
                plain[tap, :, i0] = False
                assert np.array_equal(out[tap, :cout, i0], np.inf * g[(n - 1,) + v]), (at, tap)
        got = out[:27, :cout, :cin]
        assert np.isfinite(got[plain]).all(), at
        assert _rel(got[plain], ref[plain]) <= 1e-5 and np.isfinite(out[27]).all()
