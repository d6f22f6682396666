"""The analytic reconstructions' row filter: the response of the short transform against the padded one in 64 bits
(here), and the kernel at the sizes where its passes change (GPU).

Tolerance of the kernel: two FP32 transforms of M <= 4096 elements, each of at most 12 roundings of 2^-24 relative to
its input's norm, and responses whose mean square is above 0.3 of their largest: 2 x 12 x 6e-8 / sqrt(0.3) < 3e-6 in
relative L2 on white rows."""
import importlib

import numpy as np
import pytest

from tigre_amd.geometry import cone_geometry
F = importlib.import_module("tigre_amd.utilities.filtering")

SIZES = [1, 5, 31, 32, 33, 64, 65, 128, 129, 200, 256, 257, 512, 513, 1024, 1025, 2048]


def _padded(rows, n_u, name):
    """The padded rows' filter in 64 bits, unscaled."""
    filt, length = F.ramp_filter(n_u, name)
    pad = (length - n_u) // 2
    buf = np.zeros(rows.shape[:-1] + (length,))
    buf[..., pad:pad + n_u] = rows
    spec = np.fft.rfft(buf) * filt[: length // 2 + 1].astype(np.float64)
    return np.fft.irfft(spec, length)[..., pad:pad + n_u]


@pytest.mark.parametrize("n_u", SIZES)
@pytest.mark.parametrize("name", [None, "shepp_logan", "hann"])
def test_row_response(n_u, name):
    """One complex transform of a row's two quarters gives the padded filter's pixels: exact but for the response's
    single rounding, 6e-8 of each value."""
    filt, _ = F.ramp_filter(n_u, name)
    length = max(64, 1 << (2 * n_u - 1).bit_length())
    resp = F.row_response(filt, length, 1.0).astype(np.float64) * length
    rows = np.random.default_rng(n_u).standard_normal((3, n_u))
    quarter = length // 4
    z = np.zeros((3, length), dtype=complex)
    z[:, : min(quarter, n_u)] += rows[:, :quarter]
    z[:, : max(n_u - quarter, 0)] += 1j * rows[:, quarter:]
    c = np.fft.ifft(np.fft.fft(z) * np.concatenate([resp, resp[1:-1][::-1]]))
    got = c.real[:, :n_u] + np.roll(c.imag, quarter, axis=1)[:, :n_u]
    ref = _padded(rows, n_u, name)
    assert np.linalg.norm(got - ref) <= 2e-7 * np.linalg.norm(ref)


def _geo(n_u, name):
    geo = cone_geometry((4, 4, 4), (4.0, 4.0, 4.0), (3, n_u), (1.0, 0.7), 300.0, 450.0)
    geo.filter = name
    return geo


@pytest.mark.gpu
@pytest.mark.parametrize("n_u", SIZES + [2049])
def test_filter_kernel(cuda, n_u):
    import torch

    views = 7
    angles = np.linspace(0, 2 * np.pi, views, endpoint=False)
    rng = np.random.default_rng(n_u)
    rows = rng.standard_normal((views, 3, n_u)).astype(np.float32)
    weight = rng.uniform(0.5, 1.0, (3, n_u)).astype(np.float32)
    geo = _geo(n_u, "hann" if n_u % 2 else None)
    scale = 450.0 / 300.0 * (2 * np.pi / views) / (4 * 0.7)
    x, w = torch.from_numpy(rows).to(cuda), torch.from_numpy(weight).to(cuda)
    strided = torch.empty((views, n_u, 3), device=cuda).transpose(1, 2).copy_(x)
    for got, ref in ((F.filtering(strided, geo, angles), rows), (F.weighted_filtering(x, w, geo, angles), rows * weight)):
        ref = _padded(ref.astype(np.float64), n_u, geo.filter) * scale
        err = np.linalg.norm(got.cpu().numpy() - ref) / np.linalg.norm(ref)
        print("row filter %d rel-L2 %.3e" % (n_u, err))
        assert got.is_contiguous() and err <= 3e-6
    # rows do not mix, and tensors that autograd records keep their gradient
    x[2, 1, n_u // 2] = float("inf")
    bad = ~torch.isfinite(F.filtering(x, geo, angles)).all(dim=2)
    assert bad.sum() == 1 and bool(bad[2, 1])
    y = w.expand(2, 3, n_u).clone().requires_grad_()
    F.filtering(y, geo, angles).sum().backward()
    assert y.grad is not None and bool(torch.isfinite(y.grad).all())


@pytest.mark.gpu
@pytest.mark.parametrize("shape,pixel", [((1, 1), (0.8, 0.8)), ((3, 257), (1.3, 0.7)), ((129, 64), (1 / 3, 2.1))])
def test_cosine_weight(cuda, shape, pixel):
    """The bits of the FP64 expression, rounded once."""
    import ctypes

    import torch

    from tigre_amd import _native

    dsd = 1536.1
    w = torch.empty(shape, device=cuda)
    _native.check(_native.lib().tigre_cosine_weight_device(ctypes.c_void_p(w.data_ptr()), *shape, *pixel, dsd, None), "w")
    torch.cuda.synchronize()
    yy, xx = ((np.arange(n) - n / 2 + 0.5) * d for n, d in zip(shape, pixel))
    ref = (dsd / np.sqrt(dsd ** 2 + xx[None, :] ** 2 + yy[:, None] ** 2)).astype(np.float32)
    assert np.array_equal(w.cpu().numpy(), ref)
