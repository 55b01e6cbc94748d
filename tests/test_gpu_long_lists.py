"""Lists of long, thin transforms, whose twiddle tables (2 bytes per input
sample and output pixel of the axis) are far larger than their arrays: they run
one by one with tables made in pieces.  Against single transforms, and against
the complex128 oracle on windows of the output at the fields' gates."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import mft
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = {'fp32': 2e-6, 'bf16x3': 2e-5}


def _window_err(got, f, alpha, shift, axis, at, n=150):
    """Relative error of ``got`` on n outputs from ``at`` on along ``axis``: the
    oracle's transform of that window is one of a shifted grid."""
    shape, sh = list(got.shape), list(shift)
    sh[axis] += shape[axis] // 2 - at - n // 2
    shape[axis] = n
    ref = mft.dft2(f, alpha, tuple(shape), tuple(sh), unitary=False)
    part = got[:, at:at + n] if axis else got[at:at + n]
    return rel_l2(part.cpu().numpy(), ref)


@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
def test_tables_past_a_launch(precision):
    """A list of transforms of half a million samples each, a table of 90 GB:
    the bits of single transforms."""
    from lentil_amd import fourier
    rng = np.random.default_rng(1)
    n, N = 500000, 90000
    f = [(rng.standard_normal((1, n)) + 1j * rng.standard_normal((1, n))).astype(np.complex64) for _ in range(2)]
    jobs = [(torch.from_numpy(x).cuda(), (1.0, 1 / n), (1, N), (0, 1.25), (0, 0)) for x in f]
    for job, got in zip(jobs, fourier.dft2_list(jobs, precision=precision)):
        assert torch.equal(got, fourier.dft2(*job, precision=precision))


def test_plan_tables_past_a_launch():
    """A persistent plan holds its table whole: 90 GB, three launches."""
    from lentil_amd import _lib, fourier
    lib, ctx = _lib.load(), _lib.context()
    n, N = 500000, 90000
    f = torch.from_numpy(np.random.default_rng(3).standard_normal((1, n)).astype(np.float32)).cuda()
    F = torch.full((1, N), float('nan'), dtype=torch.complex64, device='cuda')
    q = (_lib.MftxMft * 1)()
    q[0].f, q[0].f_dtype, q[0].m, q[0].n, q[0].ldf = f.data_ptr(), _lib.DT_F32, 1, n, n
    q[0].F, q[0].M, q[0].N, q[0].ldF = F.data_ptr(), 1, N, N
    q[0].alpha_r, q[0].alpha_c, q[0].shift_c, q[0].scale = 1.0, 1 / n, 1.25, 1.0
    plan = ctypes.c_void_p()
    _lib.check(lib.mftx_mft_plan_create(ctx, q, 1, 1, ctypes.byref(plan)), ctx, 'mftx_mft_plan_create')
    try:
        _lib.check(lib.mftx_mft_plan_execute(plan), ctx, 'mftx_mft_plan_execute')
        want = fourier.dft2(f, (1.0, 1 / n), (1, N), (0, 1.25), unitary=False, precision='bf16x3')
        assert rel_l2(F.cpu().numpy(), want.cpu().numpy()) < 1e-5
    finally:
        lib.mftx_mft_plan_destroy(plan)


@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
def test_every_kind_of_entry(precision):
    """Complex and phasor sources, weight maps, conjugate twiddles and both
    orientations beside a small entry, in a list whose tables exceed 1 GiB."""
    from lentil_amd import _lib
    rng = np.random.default_rng(2)
    n, ctx = 24000, _lib.context()
    small = (rng.standard_normal((30, 20)) + 1j * rng.standard_normal((30, 20))).astype(np.complex64)
    amp, opd = rng.uniform(0.5, 1, (3, n)), rng.normal(0, 1e-7, (3, n))
    arr = (rng.standard_normal((n, 3)) + 1j * rng.standard_normal((n, 3))).astype(np.complex64)
    src = [small, amp * np.exp(2j * np.pi * opd / 6e-7), np.conj(arr)]
    alpha = [(0.03, 0.02), (0.1, 0.9 / n), (0.8 / n, 0.1)]
    shift = [(0.5, -1.0), (0.25, -3.5), (2.0, 0.0)]
    shape = [(25, 31), (2, n), (n, 2)]
    dev = [torch.from_numpy(a).cuda() for a in (small, amp, opd, arr)]
    w = torch.rand(shape[1], dtype=torch.float64, device='cuda')
    out = [torch.full(s, float('nan'), dtype=torch.complex64, device='cuda') for s in shape]
    q = (_lib.MftxMft * 3)()
    for k in range(3):
        q[k].m, q[k].n = src[k].shape
        q[k].M, q[k].N = shape[k]
        q[k].F, q[k].ldF, q[k].scale = out[k].data_ptr(), shape[k][1], 1.0
        q[k].alpha_r, q[k].alpha_c = alpha[k]
        q[k].shift_r, q[k].shift_c = shift[k]
    for k, t in ((0, dev[0]), (2, dev[3])):
        q[k].f, q[k].f_dtype, q[k].ldf = t.data_ptr(), _lib.DT_C64, t.shape[1]
    q[1].amp, q[1].opd, q[1].amp_dtype, q[1].opd_dtype = dev[1].data_ptr(), dev[2].data_ptr(), _lib.DT_F64, _lib.DT_F64
    q[1].ld_amp = q[1].ld_opd = n
    q[1].inv_wl = 1 / 6e-7
    q[1].w, q[1].w_dtype, q[1].ldw = w.data_ptr(), _lib.DT_F64, n
    q[2].conj = 1   # F = conj of the plain transform of the conjugate source
    _lib.check(_lib.load().mftx_dft2_many(ctx, q, 3, _lib.precision_code(precision)), ctx, 'mftx_dft2_many')
    tol = TOL[precision]
    assert rel_l2(out[0].cpu().numpy(), mft.dft2(small.astype(complex), alpha[0], shape[0], shift[0], unitary=False)) < tol
    for at in (0, n // 2 - 75, n - 150):
        assert _window_err(out[1] / w, src[1], alpha[1], shift[1], 1, at) < tol, at
        assert _window_err(out[2].conj(), src[2].astype(complex), alpha[2], shift[2], 0, at) < tol, at
