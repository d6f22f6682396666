"""GPU: the network's image layers (one channel to 32, and 32 to one) at the edges of their tiles and chunks and with
operands that only allow two-byte accesses, against the FP64 oracle on bf16-representable inputs.

Tolerances: FP32 sums of at most 27 x 32 products, relative error about u sqrt(864) = 1.8e-6: 1e-5; the 32-channel
results are then rounded to bf16, 2^-9 at most: 2e-3."""
import numpy as np
import pytest

import oracle.cnn as ocnn
from tigre_amd import _native

from .test_gpu_cnn import _conv, _dev, _rand_bf16, _rel

pytestmark = pytest.mark.gpu

# chunks of 4 and more planes with remainders, tiles of 128 x 4 (64 x 8) and one more or less
SHAPES = [(1, 1, 1, 1), (1, 3, 4, 16), (2, 4, 5, 17), (1, 5, 8, 127), (1, 17, 9, 129), (3, 9, 7, 64), (1, 33, 17, 65)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("layer", ["bias", "mask", "out"])
def test_image_layers(cuda, shape, layer):
    import torch

    rng = np.random.default_rng(sum(shape))
    b = rng.standard_normal(32).astype(np.float32) * 0.1
    if layer == "out":
        x, w = _rand_bf16(rng, shape + (32,)), np.zeros((27, 32, 32))
        w[:, :1] = _rand_bf16(rng, (27, 1, 32), 0.2)
        img = rng.standard_normal(shape).astype(np.float32)
        y = torch.empty(shape, device="cuda")
        _conv(_dev(x, torch.bfloat16), _native.CNN_IN_BF16X32, _dev(w, torch.bfloat16), _dev(b), _dev(img), y,
              _native.CNN_EPI_RESIDUAL, shape)
        assert _rel(y.cpu().numpy(), img + ocnn.conv3d(x, w[:, :1])[..., 0] + b[0]) <= 1e-5
        return
    x, w = _rand_bf16(rng, shape + (1,)), np.zeros((27, 32, 32))
    w[:, :, :1] = _rand_bf16(rng, (27, 32, 1), 0.2)
    h = np.maximum(_rand_bf16(rng, shape + (32,)), 0.0)
    ref = ocnn.conv3d(x, w[:, :, :1])
    ref = np.maximum(ref + b, 0.0) if layer == "bias" else ref * (h > 0)
    first = None
    for shift in (0, 1):  # elements: 16-byte aligned, and two bytes further
        n = int(np.prod(shape)) * 32
        y = torch.empty(n + shift, dtype=torch.bfloat16, device="cuda")[shift:].view(shape + (32,))
        mask = torch.empty(n + shift, dtype=torch.bfloat16, device="cuda")[shift:].view(shape + (32,))
        mask.copy_(_dev(h, torch.bfloat16))
        _conv(_dev(x[..., 0]), _native.CNN_IN_F32X1, _dev(w, torch.bfloat16), _dev(b) if layer == "bias" else None,
              None if layer == "bias" else mask, y,
              _native.CNN_EPI_BIAS_RELU if layer == "bias" else _native.CNN_EPI_RELU_MASK, shape)
        assert _rel(y.float().cpu().numpy(), ref) <= 2e-3
        first = y.clone() if first is None else first
        assert torch.equal(y, first)
