"""The FP32 form over long axes: f16 pairs are scaled for sums over every
sample, and a source of few bright ones among very many must keep its bits.
Against the complex128 oracle on windows of the output.

A source of few samples adds few terms: the fields' gate, 2e-6.  A dense one
rounds an FP32 running sum three times per 16 pairs, 2^-24 sqrt(3 K / 32) of
it in all where that is more."""
import numpy as np
import pytest
import torch

from oracle import mft
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


def _source(kind, shape, rng):
    f = np.zeros(shape, dtype=np.complex64)
    if kind == 'few':      # of very different sizes
        f.flat[rng.integers(0, f.size, 5)] = [1, 1e-3j, 2e-2, 0.5 + 1j, -1e-5]
    elif kind == 'dense':
        f[:] = 1 + rng.standard_normal(shape)
    elif kind == 'largest':    # every sample as bright as the brightest: sums at their bound
        f[:] = 3e4
    else:
        f.flat[f.size // 3] = 1e-20
    return f


@pytest.mark.parametrize('kind', ['one', 'few', 'dense', 'largest'])
@pytest.mark.parametrize('shape_in, shape_out', [
    ((1, 500000), (1, 3001)), ((40001, 2), (700, 5)), ((3, 32768), (4, 900)), ((3, 32770), (4, 900))])
@pytest.mark.parametrize('listed', [False, True])
def test_long_axes(kind, shape_in, shape_out, listed):
    from lentil_amd import fourier
    K, axis = max(shape_in), int(np.argmax(shape_in))
    f = _source(kind, shape_in, np.random.default_rng(K))
    alpha, shift = [0.05, 0.05], [0.0, 0.0]
    alpha[axis], shift[axis] = 1 / K, 1.25
    t = torch.from_numpy(f).cuda()
    if listed:
        got = fourier.dft2_list([(t, alpha, shape_out, shift, (0, 0))] * 2, precision='fp32')[1]
    else:
        got = fourier.dft2(t, alpha, shape_out, shift, precision='fp32')
    tol = max(2e-6, 2 ** -24 * (3 * K / 32) ** 0.5) if kind in ('dense', 'largest') else 2e-6
    n, N = 100, shape_out[axis]
    for at in (0, N // 2 - n // 2, N - n):
        size, sh = list(shape_out), list(shift)
        size[axis] = n
        sh[axis] += N // 2 - at - n // 2
        ref = mft.dft2(f.astype(complex), alpha, tuple(size), tuple(sh))
        part = got[:, at:at + n] if axis else got[at:at + n]
        full = np.linalg.norm(ref) if kind != 'largest' else max(np.linalg.norm(ref), np.abs(f).sum() * (alpha[0] * alpha[1]) ** 0.5)
        assert np.linalg.norm(part.cpu().numpy() - ref) < tol * full, at
