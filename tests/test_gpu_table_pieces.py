"""Transforms whose twiddle table is larger than its space (what the operands
leave of the no-allocation array, 64 MiB to 1 GiB of the context workspace): the
table is made and used in pieces of whole tile columns, the last of them a
remainder.  Against the complex128 oracle at the fields' gates, and against each
other."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import mft
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = [2e-6, 2e-5]


def _call(name, f, F, alpha, shift, prec):
    from lentil_amd import _lib
    ctx = _lib.context()
    _lib.check(getattr(_lib.load(), name)(
        ctx, ctypes.c_void_p(f.data_ptr()), 0, *f.shape, f.stride(0), ctypes.c_void_p(F.data_ptr()), *F.shape,
        F.stride(0), *alpha, *shift, 0.0, 0.0, 1.0, 0, prec), ctx, name)


@pytest.mark.parametrize('prec', [0, 1])
@pytest.mark.parametrize('flip', [False, True])
@pytest.mark.parametrize('names, shape_in, shape_out', [
    (('mftx_dft2_noalloc', 'mftx_dft2'), (64, 1024), (16, 20001)),   # stage 2, a table of 41 MB
    (('mftx_dft2_noalloc', 'mftx_dft2'), (16, 1024), (64, 20001)),   # the same in stage 1
    (('mftx_dft2_noalloc', 'mftx_dft2'), (2, 9000), (3, 7001)),      # 126 MB: 3 pieces on the array, 1 on the context
    (('mftx_dft2_noalloc', 'mftx_dft2'), (3, 9000), (2, 7001)),      # the same in stage 2
    (('mftx_dft2',), (5, 1200), (3, 30001))])                        # 73 MB
def test_tables_in_pieces(names, shape_in, shape_out, flip, prec):
    rng = np.random.default_rng(shape_in[0])
    x = (rng.standard_normal(shape_in) + 1j * rng.standard_normal(shape_in)).astype(np.complex64)
    alpha, shift = (1 / 70, 1 / 20011), (0.25, -3.5)
    print(f'{names} {shape_in} -> {shape_out}, transposed {flip}, precision {prec}', flush=True)
    ref = mft.dft2(x.astype(complex), alpha, shape_out, shift, unitary=False)
    if flip:
        x, ref, alpha, shift = np.ascontiguousarray(x.T), ref.T, alpha[::-1], shift[::-1]
    f = torch.from_numpy(x).cuda()
    got = []
    for name in names:
        F = torch.full(ref.shape, float('nan'), dtype=torch.complex64, device='cuda')
        _call(name, f, F, alpha, shift, prec)
        assert rel_l2(F.cpu().numpy(), ref) < TOL[prec], name
        got.append(F)
    assert torch.equal(got[0], got[-1])
