"""Values far from 1, and far from each other: the FP32 form's operands are f16
pairs scaled by powers of two, and its results keep FP32's range.  Against the
complex128 oracle at the gates of the forms (fields 2e-6, images 1e-5)."""
import numpy as np
import pytest
import torch

from oracle import mft, optics
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def L():
    import lentil_amd
    assert torch.cuda.is_available()
    return lentil_amd


# an image of (1e-18)^2 times unit weights is still a normal float32 in the
# core; 1e9 squared is far from float32's end
@pytest.mark.parametrize('nseg, tile_n', [(1, 0), (1, 64), (1, 128), (3, 0), (3, 64)])
@pytest.mark.parametrize('level', [1e-18, 1e-16, 1e-13, 1.0, 1e9])
def test_plan_images_of_any_amplitude(L, nseg, tile_n, level):
    """Every tile's intensity epilogue (one segment, several along K)."""
    n, os, du, z = 72, 2, 5e-6, 10.0
    masks = np.zeros((nseg, n, n))
    for k in range(nseg):
        masks[k, 3 + 24 * k:21 + 24 * k, 5:60] = 1
    yy, xx = np.mgrid[:n, :n] / n - 0.5
    amp, opd = masks.sum(axis=0) * (1 + xx * yy), 3e-7 * (yy ** 2 - yy * xx)
    wl, wt = np.array([5.2e-7, 6e-7, 7e-7]), np.array([0.5, 0.2, 0.3])
    mask = masks if nseg > 1 else None
    plan = L.PSFPlan(L.Pupil(amplitude=amp * level, opd=opd, mask=mask, pixelscale=1 / n, focal_length=z), wl, wt,
                     pixelscale=du, shape=(60, 45), oversample=os, precision='fp32', tile_n=tile_n,
                     contraction='per_tile')
    ref = optics.broadband_image(optics.Pupil(amp, opd, 1 / n, z, mask=mask), wl, wt, du, (60, 45), os)
    img = plan(out=torch.empty(plan.shape_out, dtype=torch.float64, device='cuda'))
    assert rel_l2(img.cpu().numpy() / level / level, ref) < 1e-5


@pytest.mark.parametrize('tilt', [1.0, 9.0])
def test_fields_of_unequal_segments(L, tilt):
    """Segments of one coherent group on grids of their own (windows of one
    grid, and Fields far apart): a dim one keeps its own 22 bits.  Two segments
    share a grid and a class."""
    n, os, du, z = 64, 2, 5e-6, 10.0
    level = np.array([1.0, 1e-7, 1e-12, 1e3, 0.5])
    masks = np.zeros((5, n, n))
    for k in range(5):
        masks[k, 1 + 20 * (k // 2):20 + 20 * (k // 2), 2 + 31 * (k % 2):30 + 31 * (k % 2)] = 1
    yy, xx = np.mgrid[:n, :n] / n - 0.5
    amp, opd = (masks * level[:, None, None]).sum(axis=0), 3e-7 * (yy ** 2 - yy * xx)
    wl = np.array([5e-7, 6.5e-7])
    px = np.random.default_rng(1).uniform(-tilt, tilt, (5, 2))
    px[4] = px[0]
    pupil = L.Pupil(amplitude=amp, opd=opd, mask=masks, pixelscale=1 / n, focal_length=z)
    pupil.tilt.extend(L.Tilt(*a) for a in px * du / os / z)
    plan = L.PSFPlan(pupil, wl, None, pixelscale=du, shape=(30, 47), prop_shape=(20, 20), oversample=os,
                     precision='fp32', contraction='per_tile')
    assert plan.info['coherent_fast'] == 0 and plan.info['n_stage2'] == 8
    F = [torch.zeros((p['M'], p['N']), dtype=torch.complex64, device='cuda') for p in plan.problems]
    plan()
    plan.set_fields(F, [1.0] * len(F))
    plan.fields()
    tiles = list(pupil.phasor_tiles())
    field = {}
    for p in plan.problems:
        _, _, a, o = tiles[p['tile']]
        field[p['tile'], p['wave']] = mft.dft2(a * np.exp(2j * np.pi * o / wl[p['wave']]), p['alpha'],
                                               (p['M'], p['N']), p['shift'], p['offset'], unitary=False)
    for p, f in zip(plan.problems, F):
        if p['tile'] == 4:
            continue    # written with its class's first segment
        ref = field[p['tile'], p['wave']] + (field[4, p['wave']] if p['tile'] == 0 else 0)
        assert rel_l2(f.cpu().numpy(), ref) < 2e-6, p['tile']


@pytest.mark.parametrize('n', [16, 120])
@pytest.mark.parametrize('sample', [2e38 + 2e38j, 3.4028234e38 - 3.4028234e38j, 3.4e38j])
def test_samples_at_the_ends_of_float32(L, n, sample):
    """One sample whose parts are finite and whose |re| + |im| may not be."""
    f = torch.zeros((n, n), dtype=torch.complex64, device='cuda')
    f[n // 2, n // 2] = sample
    got = L.fourier.dft2(f, 1 / (2 * n), (20, 30)).cpu().numpy().astype(complex)
    ref = mft.dft2(f.cpu().numpy().astype(complex), 1 / (2 * n), (20, 30))
    assert rel_l2(got / abs(sample), ref / abs(sample)) < 2e-6


@pytest.mark.parametrize('n', [40, 130])
@pytest.mark.parametrize('level', [1e-36, 1e-38, 1e-40, 3e-43])
def test_sources_at_the_lower_end_of_float32(L, n, level):
    """Sources near FP32's smallest normal number and among the denormals, as
    one transform and in a list; results are rounded to steps of 1.4e-45."""
    rng = np.random.default_rng(n)
    f = ((1 + rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) * level).astype(np.complex64)
    t = torch.from_numpy(f).cuda()
    jobs = [(t, (1 / (2 * n),) * 2, (31, 44), (0.3, 1.7), (0, 0))] * 2
    for got, unitary in [(L.fourier.dft2(t, 1 / (2 * n), (31, 44), (0.3, 1.7), unitary=False), False)] + [
            (g, True) for g in L.fourier.dft2_list(jobs, precision='fp32')]:
        ref = mft.dft2(f.astype(complex), 1 / (2 * n), (31, 44), (0.3, 1.7), unitary=unitary)
        err = np.linalg.norm((got.cpu().numpy().astype(complex) - ref) / level)
        assert err < 2e-6 * np.linalg.norm(ref / level) + 1.5e-45 / level * ref.size ** 0.5
