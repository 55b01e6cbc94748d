"""The complex-field store: pieces of two samples traded between neighbouring lanes, cut to the window and the row
stride, and work items that run several fields of one shape.

Tolerances: an f16 pair carries 22 bits (fields below 2e-6), a bf16 pair 16 (2e-5)."""
import numpy as np
import pytest
import torch

from oracle import mft
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = {'fp32': 2e-6, 'bf16x3': 2e-5}


# one wavelength: small tiles; 50: runs of two fields per work item.  Windows of one row or column, odd and even,
# clipped by the tilt; strides that put every other row off 16-byte alignment
@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
@pytest.mark.parametrize('wdtype', [None, torch.float32, torch.float64])
@pytest.mark.parametrize('shape_in, npix, nwave, tile_n, pad', [
    ((40, 41), (1, 7), 1, 0, 1), ((65, 40), (7, 1), 2, 64, 3), ((96, 90), (101, 130), 1, 0, 1),
    ((64, 96), (321, 290), 50, 128, 1), ((96, 64), (289, 322), 50, 64, 2)])
def test_fields_into_strided_arrays(precision, wdtype, shape_in, npix, nwave, tile_n, pad):
    import lentil_amd as L
    m, n = shape_in
    rng = np.random.default_rng(m + npix[0])
    amp, opd = rng.uniform(0.5, 1, (m, n)), rng.normal(0, 5e-8, (m, n))
    wl = np.linspace(5e-7, 7e-7, nwave) if nwave > 1 else np.array([6e-7])
    # a few pixels, which clip the window; a part of one where it is one pixel wide
    tilt = L.Tilt(1.7e-6, -1.2e-6) if min(npix) > 1 else L.Tilt(0.4e-6, -0.3e-6)
    plan = L.PSFPlan(L.Pupil(amplitude=amp, opd=opd, mask=np.ones((m, n)), pixelscale=1 / 64, focal_length=10), wl, None,
                     pixelscale=5e-6, shape=npix, oversample=1, tilts=[tilt], precision=precision,
                     tile_n=tile_n)
    M, N = plan.problems[0]['M'], plan.problems[0]['N']
    buf = torch.full((len(plan.problems), M + 1, N + pad), float('nan'), dtype=torch.complex64, device='cuda')
    F = [b[:M, :N] for b in buf]
    w = None if wdtype is None else torch.rand((M, N + 1), dtype=wdtype, device='cuda')[:, :N]
    scale = list(1.0 + 0.25 * np.arange(len(F)))
    plan()
    plan.set_fields(F, scale, weights=None if w is None else [w] * len(F))
    plan.fields()
    plan.fields()
    # nothing outside the window is written
    assert bool(buf[:, :M, N:].isnan().all() and buf[:, M:].isnan().all())
    wn = 1.0 if w is None else w.double().cpu().numpy()
    for i in sorted({0, 1 % len(F), len(F) // 2, len(F) - 1}):
        p = plan.problems[i]
        ref = scale[i] * wn * mft.dft2(amp * np.exp(2j * np.pi * opd / wl[p['wave']]), p['alpha'], (M, N), p['shift'],
                                       p['offset'], unitary=False)
        assert rel_l2(F[i].cpu().numpy(), ref) < TOL[precision]
