"""Matrix Fourier transforms on the HIP device (lentil fourier.py).

``dft2`` and ``idft2`` keep lentil's signatures and semantics; the work runs
in ``mftx_dft2`` (two complex GEMMs against twiddle tables on MFMA).

Returned types follow the input: a NumPy input gives a complex128 NumPy
result (the drop-in contract), a device tensor gives a complex64 device
tensor.  ``out`` may be either kind and is returned.

The extra keyword-only ``precision`` selects 'fp32' (default) or 'bf16x3'.
"""
import math

import numpy as np
import torch

from . import _lib
from ._arrays import is_dev, to_dev, write_back

_default_precision = 'fp32'


def set_precision(precision):
    """Set the default precision of dft2/idft2/propagate_dft ('fp32' or 'bf16x3')."""
    global _default_precision
    _lib.precision_code(precision)
    _default_precision = precision


def get_precision():
    return _default_precision


def _mft(f, alpha, shape, shift, offset, scale, conj, out, precision):
    alpha_r, alpha_c = _lib.pair(alpha)
    host_input = not is_dev(f)
    if host_input:
        f = np.asarray(f)
    if f.ndim != 2:
        raise ValueError(f'f must be 2-dimensional, got shape {tuple(f.shape)}')
    m, n = f.shape
    if shape is None:
        M, N = m, n
    elif type(shape) is tuple and len(shape) == 2:
        M, N = int(shape[0]), int(shape[1])
    else:
        M, N = (int(v) for v in np.broadcast_to(shape, (2,)))
    shift_r, shift_c = _lib.pair(shift)
    off_r, off_c = _lib.pair(offset)
    if out is not None:
        odt = out.dtype
        ok = odt.is_complex if isinstance(out, torch.Tensor) else np.can_cast(complex, odt)
        if not ok:
            raise TypeError(f"Cannot cast complex output to dtype('{odt}')")
    prec = _lib.precision_code(precision or _default_precision)
    src = f if not host_input else to_dev(f)
    if src.dtype not in _lib.DTYPE_CODE:
        src = src.to(torch.complex128 if src.is_complex() else torch.float64)
    src = src.contiguous()
    if out is not None and is_dev(out) and out.dtype == torch.complex64 and out.dim() == 2 and out.stride(1) == 1 \
            and tuple(out.shape) == (M, N) and out.data_ptr() != src.data_ptr():
        F = out
    else:
        F = torch.empty((M, N), dtype=torch.complex64, device=src.device)
    ctx = _lib.context()
    rc = _lib.load().mftx_dft2(ctx, src.data_ptr(), _lib.DTYPE_CODE[src.dtype], m, n, src.stride(0), F.data_ptr(), M, N,
                               F.stride(0), alpha_r, alpha_c, shift_r, shift_c, off_r, off_c, float(scale),
                               1 if conj else 0, prec)
    if rc != _lib.OK:
        _lib.check(rc, ctx, 'mftx_dft2')
    if out is None:
        return F.cpu().numpy().astype(complex) if host_input else F
    if F is out:
        return out
    if is_dev(out):
        out.copy_(F)
    else:
        write_back(out, F)
    return out


def dft2(f, alpha, shape=None, shift=(0, 0), offset=(0, 0), unitary=True, out=None, *, precision=None):
    """2-D DFT by matrix triple product (fourier.py:5-103).

    F[u, v] = c * sum_{r, s} f[r, s] exp(-2 pi i (ar (R_r + or)(U_u - sr) + ac (S_s + oc)(V_v - sc)))
    with centred coordinates R = arange(m) - floor(m/2) (fourier.py:113-121)
    and c = sqrt(|ar ac|) when ``unitary``.
    """
    ar, ac = _lib.pair(alpha)
    scale = math.sqrt(abs(ar * ac)) if unitary else 1.0
    return _mft(f, (ar, ac), shape, shift, offset, scale, False, out, precision)


# dft2_list puts transforms into one grouped call while they are small: up to
# this many samples (input and output) each and this many together, so the
# operands of a group stay below 128 MiB.  A transform of 1024^2 fills the chip
# by itself and gains nothing; six of 100^2 -> 303^2 take 160 us of launches one
# by one (24 launches on quarter-filled chips) and 55 us as a group.
_LIST_ONE = 1 << 20
_LIST_ALL = 1 << 22


def dft2_list(jobs, *, precision=None):
    """Unitary ``dft2`` of every (f, alpha, shape, shift, offset); ``f`` are 2-D
    device arrays, ``shape`` a pair of ints.  Neighbouring small transforms run
    as one mftx_dft2_many call."""
    if len(jobs) == 1:
        f, alpha, shape, shift, offset = jobs[0]
        return [dft2(f, alpha, shape, shift, offset, precision=precision)]
    out = [None] * len(jobs)
    sizes = [f.shape[0] * f.shape[1] + shape[0] * shape[1] for f, _, shape, _, _ in jobs]
    grouped = bool(jobs) and not torch.cuda.is_current_stream_capturing()   # a group uploads its descriptors
    b = 0
    while b < len(jobs):
        e, total = b, 0
        while grouped and e < len(jobs) and sizes[e] <= _LIST_ONE and total + sizes[e] <= _LIST_ALL:
            total += sizes[e]
            e += 1
        if e - b > 1:
            out[b:e] = _mft_group(jobs[b:e], precision)
        else:
            e = b + 1
            f, alpha, shape, shift, offset = jobs[b]
            out[b] = dft2(f, alpha, shape, shift, offset, precision=precision)
        b = e
    return out


def _mft_group(jobs, precision):
    prec = _lib.precision_code(precision or _default_precision)
    entries, out, keep = [], [], []
    for f, alpha, (M, N), shift, offset in jobs:
        ar, ac = _lib.pair(alpha)
        sr, sc = _lib.pair(shift)
        orr, oc = _lib.pair(offset)
        if f.dtype not in _lib.DTYPE_CODE:
            f = f.to(torch.complex128 if f.is_complex() else torch.float64)
        f = f.contiguous()
        keep.append(f)
        F = torch.empty((M, N), dtype=torch.complex64, device=f.device)
        out.append(F)
        entries.append((f.data_ptr(), None, None, _lib.DTYPE_CODE[f.dtype], 0, 0, 0, f.shape[0], f.shape[1], f.stride(0),
                        0, 0, 0.0, F.data_ptr(), M, N, N, ar, ac, sr, sc, orr, oc, math.sqrt(abs(ar * ac))))
    ctx = _lib.context()
    rc = _lib.load().mftx_dft2_many(ctx, (_lib.MftxMft * len(entries))(*entries), len(entries), prec)
    if rc != _lib.OK:
        _lib.check(rc, ctx, 'mftx_dft2_many')
    return out


def idft2(F, alpha, shape=None, shift=(0, 0), unitary=True, out=None, *, precision=None):
    """Inverse DFT (fourier.py:124-198): conj(dft2(conj(F))) / F.size.

    The division is by the size of the *input* ``F`` whatever ``shape`` is,
    as in the reference.  Implemented as conjugated twiddles on F directly.
    """
    size = int(F.numel()) if is_dev(F) else int(np.size(F))
    ar, ac = _lib.pair(alpha)
    scale = (np.sqrt(abs(ar * ac)) if unitary else 1.0) / size
    return _mft(F, (ar, ac), shape, shift, (0, 0), scale, True, out, precision)


def dft2_adjoint(G, alpha, in_shape, shift=(0, 0), offset=(0, 0), unitary=True, *, precision=None):
    """Adjoint of f -> dft2(f, alpha, G.shape, shift, offset, unitary).

    E1^H . G . E2^H is an MFT from the output grid back to the input grid with
    conjugated twiddles, the output coordinates' shift acting as the input
    offset and vice versa.  No counterpart in the reference (it has no
    gradients); used by the autograd path.
    """
    ar, ac = np.broadcast_to(alpha, (2,))
    scale = np.sqrt(np.abs(ar * ac)) if unitary else 1.0
    sr, sc = np.broadcast_to(shift, (2,))
    orr, oc = np.broadcast_to(offset, (2,))
    m, n = in_shape
    M, N = tuple(G.shape)
    # input coords of the adjoint: U - s = (u - floor(M/2)) - s  -> offset -s
    # output coords:               R + o = (r - floor(m/2)) + o  -> shift  -o
    return _mft(G, alpha, (m, n), (-orr, -oc), (-sr, -sc), scale, True, None, precision)
