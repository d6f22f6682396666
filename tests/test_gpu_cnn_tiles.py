"""GPU: the network's kernels at the edges of their tiles, against the FP64 oracle on bf16-representable inputs.

Tolerances: FP32 sums of K products; K is at most 27 x 32 for a convolution and N D H W < 7e3 for a weight
gradient, so the relative error is about u sqrt(K) = 6e-8 * 83 = 5e-6: 1e-5 (the 32-channel convolutions are
then rounded to bf16, 2^-9 at most: 2e-3)."""
import numpy as np
import pytest

import oracle.cnn as ocnn
from tigre_amd import _native

from .test_gpu_cnn import _conv, _dev, _rand_bf16, _rel, _wgrad

pytestmark = pytest.mark.gpu

# one voxel; a full tile of the weight gradient and one more or less on each axis; several chunks along z,
# the last one ragged, several batches
SHAPES = [(1, 1, 1, 1), (1, 4, 8, 32), (1, 5, 9, 33), (2, 3, 7, 31), (1, 37, 2, 5), (3, 9, 17, 8), (1, 2, 24, 66)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("modes", [(32, 32), (1, 32), (32, 1)])
def test_weight_gradient_tiles(cuda, shape, modes):
    import torch

    rng = np.random.default_rng(sum(shape))
    cin, cout = modes
    x = _rand_bf16(rng, shape + (cin,))
    g = _rand_bf16(rng, shape + (cout,))
    dev = lambda a: _dev(a, torch.bfloat16) if a.shape[-1] == 32 else _dev(a[..., 0])  # noqa: E731
    mode = {32: _native.CNN_IN_BF16X32, 1: _native.CNN_IN_F32X1}
    out = _wgrad(dev(x), mode[cin], dev(g), mode[cout], shape).cpu().numpy()
    err = _rel(out[:27, :cout, :cin], ocnn.conv3d_weight_grad(x, g))
    berr = _rel(out[27, :cout, 0], g.reshape(-1, cout).sum(axis=0))
    print("weight gradient %s %s rel-L2 %.3e, bias %.3e" % (shape, modes, err, berr))
    assert err <= 1e-5 and berr <= 1e-5
    # the padding channels hold zeros
    assert not np.any(out[:27, :, cin:]) and not np.any(out[:, cout:]) and not np.any(out[27, :, 1:])


@pytest.mark.parametrize("shape", [(1, 1, 3, 5), (1, 4, 5, 33), (2, 5, 4, 16), (1, 33, 6, 40), (1, 17, 4, 65)])
@pytest.mark.parametrize("epilogue", ["bias", "mask", "residual"])
def test_convolution_chunks(cuda, shape, epilogue):
    import torch

    rng = np.random.default_rng(sum(shape) + 1)
    x = _rand_bf16(rng, shape + (32,))
    cout = 1 if epilogue == "residual" else 32
    w = _rand_bf16(rng, (27, cout, 32), 0.2)
    b = rng.standard_normal(32).astype(np.float32) * 0.1
    wk = np.zeros((27, 32, 32))
    wk[:, :cout] = w
    xd, wd = _dev(x, torch.bfloat16), _dev(wk, torch.bfloat16)
    ref = ocnn.conv3d(x, w)
    if epilogue == "residual":
        img = rng.standard_normal(shape).astype(np.float32)
        y = torch.empty(shape, device="cuda")
        _conv(xd, _native.CNN_IN_BF16X32, wd, _dev(b), _dev(img), y, _native.CNN_EPI_RESIDUAL, shape)
        assert _rel(y.cpu().numpy(), img + ref[..., 0] + b[0]) <= 1e-5
        return
    y = torch.empty(shape + (32,), dtype=torch.bfloat16, device="cuda")
    if epilogue == "bias":
        _conv(xd, _native.CNN_IN_BF16X32, wd, _dev(b), None, y, _native.CNN_EPI_BIAS_RELU, shape)
        ref = np.maximum(ref + b, 0.0)
    else:
        h = np.maximum(_rand_bf16(rng, shape + (32,)), 0.0)
        _conv(xd, _native.CNN_IN_BF16X32, wd, None, _dev(h, torch.bfloat16), y, _native.CNN_EPI_RELU_MASK, shape)
        ref = ref * (h > 0)
    assert _rel(y.float().cpu().numpy(), ref) <= 2e-3
