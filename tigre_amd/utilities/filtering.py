"""FDK pre-processing filter, Python/tigre/utilities/filtering.py:15-87.

The filter's frequency response is built exactly as the reference builds it
(spatial ramp kernel h[0] = 1/4, h[odd n] = -1/(pi n)^2, |FFT| * 2, optional
window, zero above the Nyquist band, mirrored), then applied to the detector
rows on the device, scaled by (DSD/DSO) (2 pi / nangles) / (4 dU): by one kernel
that weights, transforms, multiplies and transforms back (csrc/filter.hip), or,
for tensors it does not take, with a real FFT of the zero-padded rows.
"""
from __future__ import annotations

import ctypes

import numpy as np

from .. import _native
from ..operators import _on, _stream_handle

LONGEST = 4096  # elements of the row kernel's longest transform


def _nextpow2(n):
    i = 1
    while 2 ** i <= n:
        i += 1
    return i


def ramp_filter(n_u, filter_name=None):
    """(filter, padded length) for detectors n_u pixels wide."""
    filt_len = max(64, 2 ** _nextpow2(2 * int(n_u)))
    nn = np.arange(-filt_len / 2, filt_len / 2)
    h = np.zeros(nn.shape, dtype=np.float32)
    h[int(filt_len / 2)] = 1 / 4
    odd = nn % 2 == 1
    h[odd] = -1 / (np.pi * nn[odd]) ** 2
    resp = np.abs(np.fft.fft(h)) * 2
    filt = resp[: int(filt_len / 2 + 1)]
    w = 2 * np.pi * np.arange(len(filt)) / filt_len
    d = 1
    if filter_name in ("ram_lak", None):
        pass
    elif filter_name == "shepp_logan":
        filt[1:] *= np.sin(w[1:] / (2 * d)) / (w[1:] / (2 * d))
    elif filter_name == "cosine":
        filt[1:] *= np.cos(w[1:] / (2 * d))
    elif filter_name == "hamming":
        filt[1:] *= 0.54 + 0.46 * np.cos(w[1:] / d)
    elif filter_name == "hann":
        filt[1:] *= (1 + np.cos(w[1:] / d)) / 2
    else:
        raise ValueError("filter not recognized: " + str(filter_name))
    filt[w > np.pi * d] = 0
    return np.hstack((filt, filt[1:-1][::-1])).astype(np.float32), filt_len


def filtering(proj, geo, angles, parker=False, verbose=False):
    """Filter cosine-weighted projections (torch tensor on the GPU, (n, nV, nU))."""
    import torch

    if parker:
        # as the reference: weights applied to the (views, u, v) transpose
        from .parkerweight import parkerweight

        proj = parkerweight(proj.transpose(1, 2).contiguous(), geo, angles, parker).transpose(1, 2).contiguous()
    return weighted_filtering(proj, None, geo, angles)


def _unwatched(t):
    """A plain strided tensor that nothing follows: no recorded gradient, forward-mode tangent, torch.func transform,
    trace, compilation or dispatch mode, all of which would miss a kernel that is not a torch operation."""
    import torch

    if type(t) is not torch.Tensor or t.layout != torch.strided or (torch.is_grad_enabled() and t.requires_grad):
        return False
    if torch.jit.is_tracing() or torch.compiler.is_compiling():
        return False
    # private to torch: where one is missing, the general path is taken
    wrapped = getattr(getattr(torch._C, "_functorch", None), "is_functorch_wrapped_tensor", None)
    modes = getattr(torch._C, "_len_torch_dispatch_stack", None)
    if wrapped is None or modes is None or wrapped(t) or modes() > 0:
        return False
    return torch.autograd.forward_ad.unpack_dual(t).tangent is None and not t.is_neg()


def _plain(t):
    """A tensor whose memory a kernel may read behind torch's back."""
    return t.is_cuda and _unwatched(t)


def weighted_filtering(proj, weight, geo, angles):
    """filtering(proj * weight): weight an (nV, nU) image or None."""
    import torch

    n_u = int(geo.nDetector[1])
    filt, filt_len = ramp_filter(n_u, getattr(geo, "filter", None))
    DSD0 = float(np.asarray(geo.DSD).reshape(-1)[0])
    DSO0 = float(np.asarray(geo.DSO).reshape(-1)[0])
    scale = (DSD0 / DSO0) * (2 * np.pi / len(angles)) / (4 * float(geo.dDetector[1]))
    length = max(64, 1 << (2 * n_u - 1).bit_length())
    if (_plain(proj) and proj.dtype == torch.float32 and proj.dim() == 3 and proj.shape[2] == n_u and proj.numel() > 0
            and length <= LONGEST and (weight is None or (_plain(weight) and weight.dtype == torch.float32
                                                          and weight.shape == proj.shape[1:]
                                                          and weight.device == proj.device))):
        return _filter_rows(proj, weight, filt, length, scale)
    if weight is not None:
        proj = proj * weight
    pad = int((filt_len - n_u) // 2)
    # the mirrored response is real and even: the half spectrum drives an rfft/irfft pair
    half = torch.as_tensor(filt[: filt_len // 2 + 1], device=proj.device)
    buf = torch.zeros(proj.shape[0], proj.shape[1], filt_len, dtype=torch.float32, device=proj.device)
    buf[:, :, pad:pad + n_u] = proj
    spec = torch.fft.rfft(buf, dim=2)
    spec *= half
    out = torch.fft.irfft(spec, n=filt_len, dim=2)[:, :, pad:pad + n_u]
    return (out * scale).contiguous()


def row_response(filt, length, scale):
    """Spectrum over ``length`` elements of the kernel whose mirrored response is ``filt``, cut to the lags below
    length / 2 that rows of at most length / 2 pixels meet; scaled, with the inverse transform's 1 / length."""
    full = len(filt)
    half = np.asarray(filt[: full // 2 + 1], dtype=np.float64)
    if full != length:
        h = np.fft.irfft(half, full)
        cut = np.zeros(length)
        cut[: length // 2] = h[: length // 2]
        cut[length // 2 + 1:] = h[full - length // 2 + 1:]
        half = np.fft.rfft(cut).real
    return (half * (scale / length)).astype(np.float32)


def _filter_rows(proj, weight, filt, length, scale):
    import torch

    x = proj.contiguous()
    w = None if weight is None else weight.contiguous()
    response = torch.as_tensor(row_response(filt, length, scale), device=x.device)
    out = torch.empty_like(x)
    with _on(x.device):
        st = _native.lib().tigre_filter_rows_device(
            ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(w.data_ptr() if w is not None else None),
            ctypes.c_void_p(response.data_ptr()), ctypes.c_void_p(out.data_ptr()), x.shape[0] * x.shape[1], x.shape[1],
            x.shape[2], length.bit_length() - 1, _stream_handle())
    _native.check(st, "TIGRE: row filter failed")
    return out
