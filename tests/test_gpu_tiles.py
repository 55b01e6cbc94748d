"""The GEMM's workgroup tiles at their edges: transforms and plans whose row,
slot and K counts sit on, one below and one above the 32-wide blocks and the
64- and 128-wide tiles, against the complex128 oracle.

Tolerances follow from the formats: an f16 pair carries 22 bits and the three
products drop 2^-22 per term, so fields stay below 2e-6 (the FP32 form's gate);
a bf16 pair carries 16 bits and drops 2^-16, gate 2e-5; intensities 1e-5."""
import numpy as np
import pytest
import torch

from oracle import mft, optics
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = {'fp32': 2e-6, 'bf16x3': 2e-5}


@pytest.fixture(scope='module')
def L():
    import lentil_amd
    assert torch.cuda.is_available()
    return lentil_amd


@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
@pytest.mark.parametrize('shape_in, shape_out', [
    ((1, 1), (1, 1)), ((1, 40), (3, 1)), ((31, 33), (63, 65)), ((32, 32), (64, 64)), ((63, 95), (127, 130)),
    ((97, 64), (260, 31)), ((129, 257), (129, 500)), ((512, 640), (900, 1030)), ((1030, 700), (1100, 1500))])
def test_single_transforms(L, precision, shape_in, shape_out):
    """Every single-transform tile choice, both contraction orders, even and odd."""
    rng = np.random.default_rng(sum(shape_in) + sum(shape_out))
    f = rng.standard_normal(shape_in) + 1j * rng.standard_normal(shape_in)
    alpha, shift, offset = (0.9 / max(shape_in[0], 8), -0.6 / max(shape_in[1], 8)), (1.3, -0.4), (-3, 2)
    print(f'{precision} {shape_in} -> {shape_out}', flush=True)
    got = L.fourier.dft2(torch.from_numpy(f).cuda(), alpha, shape_out, shift, offset, precision=precision)
    ref = mft.dft2(f, alpha, shape_out, shift, offset)
    assert rel_l2(got.cpu().numpy(), ref) < TOL[precision]


@pytest.mark.parametrize('scale', [1e-30, 1e-4, 1.0, 1e9, 1e30])
def test_f16_form_scales_any_magnitude(L, scale):
    """The f16 form's power-of-two scaling: sources far outside f16's range,
    with a bright sample 1e4 above the rest, small and large arrays."""
    rng = np.random.default_rng(3)
    for n, M in ((40, 48), (150, 100)):
        f = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))).astype(np.complex64)
        f[n // 3, n // 5] *= 1e4
        f = (f * np.float32(scale)).astype(np.complex64)
        got = L.fourier.dft2(torch.from_numpy(f).cuda(), 1 / (2 * n), (M, M), (0.3, 1.7))
        ref = mft.dft2(f.astype(np.complex128), 1 / (2 * n), (M, M), (0.3, 1.7))
        assert rel_l2(got.cpu().numpy(), ref) < TOL['fp32']


def test_f16_form_zero_and_nonfinite(L):
    f = torch.zeros((64, 64), dtype=torch.complex64, device='cuda')
    assert torch.equal(L.fourier.dft2(f, 0.01, (70, 70)), torch.zeros((70, 70), dtype=torch.complex64, device='cuda'))
    for bad in (float('nan'), float('inf')):
        for n in (64, 200):
            f = torch.ones((n, n), dtype=torch.complex64, device='cuda')
            f[5, 7] = bad
            assert not torch.isfinite(torch.view_as_real(L.fourier.dft2(f, 0.01, (70, 70)))).any()


@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
@pytest.mark.parametrize('tile_n', [0, 64, 128])
@pytest.mark.parametrize('n, npix, nwave', [(33, 31, 3), (64, 64, 1), (130, 129, 5), (257, 200, 9)])
def test_plans(L, precision, tile_n, n, npix, nwave):
    amp = L.normalize_power(L.circle((n, n), n // 2))
    yy, xx = np.mgrid[:n, :n] / n - 0.5
    opd = 2e-7 * (yy * xx + yy ** 2) + 1e-7 * xx
    wl = np.linspace(5e-7, 8e-7, nwave)
    wt = np.linspace(0.5, 1.5, nwave) / nwave
    plan = L.PSFPlan(L.Pupil(amplitude=amp, opd=opd, pixelscale=1 / n, focal_length=10), wl, wt, pixelscale=5e-6,
                     shape=npix, oversample=2, precision=precision, tile_n=tile_n, lambda_group=4)
    ref = optics.broadband_image(optics.Pupil(amp, opd, 1 / n, 10), wl, wt, 5e-6, npix, 2)
    a = plan()
    assert rel_l2(a.double().cpu().numpy(), ref) < 1e-5
    assert torch.equal(plan(), a)


@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
@pytest.mark.parametrize('tile_n', [0, 64, 128])
def test_several_segments_along_k(L, precision, tile_n):
    """Separated tiles on one output grid (no merging): their segments follow
    each other along K with a turn between, and the field output applies the
    phase of the last one."""
    n = 150
    masks = np.zeros((3, n, n))
    masks[0, 5:46, 10:43] = 1
    masks[1, 80:121, 60:127] = 1
    masks[2, 30:61, 100:142] = 1
    amp = masks.sum(axis=0)
    yy, xx = np.mgrid[:n, :n] / n - 0.5
    opd = 3e-7 * (yy ** 2 - yy * xx)
    wl, wt = np.array([5.5e-7, 7e-7]), np.array([0.4, 0.6])
    plan = L.PSFPlan(L.Pupil(amplitude=amp, opd=opd, mask=masks, pixelscale=1 / n, focal_length=10), wl, wt,
                     pixelscale=5e-6, shape=70, oversample=2, tilts=[L.Tilt(1e-6, -2e-6)], precision=precision,
                     tile_n=tile_n, contraction='per_tile')
    assert plan.info['coherent_fast'] == 1
    ref = optics.broadband_image(optics.Pupil(amp, opd, 1 / n, 10, mask=masks), wl, wt, 5e-6, 70, 2,
                                 tilts=[optics.Tilt(1e-6, -2e-6)])
    assert rel_l2(plan().double().cpu().numpy(), ref) < 1e-5


@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
@pytest.mark.parametrize('shape_in', [(21, 34), (64, 64)])
def test_fields_of_a_single_segment(L, precision, shape_in):
    """fields() of a plan whose stage 1 leaves the midpoint phases out."""
    m, n = shape_in
    rng = np.random.default_rng(m)
    amp = rng.uniform(0.5, 1, (m, n))
    opd = rng.normal(0, 5e-8, (m, n))
    wl = np.array([5e-7, 6.5e-7])
    plan = L.PSFPlan(L.Pupil(amplitude=amp, opd=opd, mask=np.ones((m, n)), pixelscale=1 / 64, focal_length=10), wl, None,
                     pixelscale=5e-6, shape=(40, 33), oversample=2, tilts=[L.Tilt(3e-7, 2e-7)], precision=precision)
    F = [torch.empty((p['M'], p['N']), dtype=torch.complex64, device='cuda') for p in plan.problems]
    w = torch.rand(F[0].shape, device='cuda')  # the window, clipped by the tilt
    plan()
    plan.set_fields(F, [2.0, 0.5], weights=[w, w])
    plan.fields()
    for p, f, sc in zip(plan.problems, F, (2.0, 0.5)):
        ref = sc * w.double().cpu().numpy() * mft.dft2(amp * np.exp(2j * np.pi * opd / wl[p['wave']]), p['alpha'],
                                                       (p['M'], p['N']), p['shift'], p['offset'], unitary=False)
        assert rel_l2(f.cpu().numpy(), ref) < TOL[precision]


@pytest.mark.parametrize('precision, tol', [('fp32', 2e-6), ('bf16x3', 2e-5)])
@pytest.mark.parametrize('shape', [(1, 1), (2, 3), (31, 64), (97, 65), (200, 131)])
def test_filter_grids(L, precision, tol, shape):
    """The FFT filter's centred transforms: even, odd and ragged grids, a kernel
    that is symmetric in neither axis, negative pixels, against numpy's FFT.
    Two transforms at the fields' gates, relative to the filtered image."""
    rng = np.random.default_rng(shape[0])
    img = rng.standard_normal(shape)
    k = rng.uniform(-1, 1, shape)
    ref = np.abs(np.fft.ifft2(np.fft.fft2(img) * k))
    t = torch.from_numpy(img).cuda()
    got = L.detector.fft_filter(t, torch.from_numpy(k).cuda(), False, precision)
    assert rel_l2(got.cpu().numpy(), ref) < 3 * tol
    got = L.detector.fft_filter(t.float(), torch.from_numpy(k).cuda().float(), True, precision)
    assert rel_l2(got.cpu().numpy(), ref * img.sum() / ref.sum()) < 5 * tol * max(1, abs(np.abs(img).sum() / img.sum()))
