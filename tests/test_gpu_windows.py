"""Coherent groups whose Fields are windows of one output grid: summed in registers where the windows nearly
coincide, stored as Fields and summed where they lie apart; both against the 64-bit oracle."""
import numpy as np
import pytest
import torch

from oracle import mft, optics

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def L():
    import lentil_amd
    return lentil_amd


def rel_l2(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def segments(nseg, n):
    """nseg disjoint rectangles of different odd and even sizes in an n x n grid."""
    masks = np.zeros((nseg, n, n))
    side = int(np.ceil(np.sqrt(nseg)))
    cell = n // side
    for k in range(nseg):
        r, c = (k // side) * cell, (k % side) * cell
        masks[k, r + 1:r + cell - k % 3, c:c + cell - 1 - k % 2] = 1
    return masks


# number of segments around the four waves that share a group; tilts in output pixels: sub-pixel, a few pixels,
# far apart; windows smaller than the detector, clipped by it, of other shape than the pupil
@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
@pytest.mark.parametrize('nseg, n, shape, prop, tilt, same', [
    (2, 40, (32, 32), None, 0.4, 0), (3, 61, (33, 90), None, 2.5, 0), (4, 64, (70, 41), (40, 30), 3.0, 2),
    (5, 100, (64, 64), (31, 33), 6.0, 0), (9, 131, (50, 60), None, 30.0, 3), (6, 90, (64, 64), (16, 16), 25.0, 0),
    (17, 140, (48, 48), None, 1.5, 5)])
def test_windows(L, precision, nseg, n, shape, prop, tilt, same):
    rng = np.random.default_rng(nseg + n)
    masks = segments(nseg, n)
    amp = masks.sum(axis=0) * rng.uniform(0.5, 1, (n, n))
    yy, xx = np.mgrid[:n, :n] / n - 0.5
    opd = 3e-7 * (yy ** 2 - yy * xx)
    wl, wt = np.array([5.2e-7, 6e-7, 7e-7]), np.array([0.5, 0.2, 0.3])
    os, du, z = 2, 5e-6, 10.0
    px = rng.uniform(-tilt, tilt, (nseg, 2))
    px[:same] = px[:1] if same else px[:0]      # these share one grid: one class of several members
    ang = px * du / os / z
    pupil = L.Pupil(amplitude=amp, opd=opd, mask=masks, pixelscale=1 / n, focal_length=z)
    pupil.tilt.extend(L.Tilt(*a) for a in ang)
    plan = L.PSFPlan(pupil, wl, wt, pixelscale=du, shape=shape, prop_shape=prop, oversample=os, precision=precision,
                     contraction='per_tile')
    assert plan.info['coherent_fast'] == 0
    ref = optics.broadband_image(optics.Pupil(amp, opd, 1 / n, z, mask=masks, tilt=[optics.Tilt(*a) for a in ang]),
                                 wl, wt, du, shape, os, prop_shape=prop)
    img = plan()
    assert rel_l2(img.double().cpu().numpy(), ref) < 1e-5
    # written everywhere, added to where asked, the same on a replay
    out = torch.full(plan.shape_out, float('nan'), dtype=torch.float64, device='cuda')
    plan(out=out)
    assert rel_l2(out.cpu().numpy(), ref) < 1e-5
    plan(out=out, accumulate=True)
    assert rel_l2(out.cpu().numpy(), 2 * ref) < 1e-5
    assert torch.equal(plan(), img)


@pytest.mark.parametrize('precision, tol', [('fp32', 2e-6), ('bf16x3', 2e-5)])
@pytest.mark.parametrize('shape, tilt', [((30, 47), 2.0), ((47, 30), 5.0)])
def test_fields_of_windows(L, precision, tol, shape, tilt):
    """fields() writes each problem's own window of the shared grid, with its weight map."""
    n, nseg, os, du, z = 64, 4, 2, 5e-6, 10.0
    rng = np.random.default_rng(7)
    masks = segments(nseg, n)
    amp = masks.sum(axis=0)
    opd = rng.normal(0, 5e-8, (n, n))
    wl = np.array([5e-7, 6.5e-7])
    pupil = L.Pupil(amplitude=amp, opd=opd, mask=masks, pixelscale=1 / n, focal_length=z)
    pupil.tilt.extend(L.Tilt(*a) for a in rng.uniform(-tilt, tilt, (nseg, 2)) * du / os / z)
    plan = L.PSFPlan(pupil, wl, None, pixelscale=du, shape=shape, prop_shape=(20, 20), oversample=os,
                     precision=precision, contraction='per_tile')
    shapes = {(p['M'], p['N']) for p in plan.problems}
    assert shapes == {(40, 40)}
    F = [torch.full((40, 43), float('nan'), dtype=torch.complex64, device='cuda')[:, :40] for _ in plan.problems]
    w = torch.rand((40, 40), device='cuda')
    scale = rng.uniform(0.5, 2, len(F))
    plan()
    plan.set_fields(F, scale, weights=[w] * len(F))
    plan.fields()
    tiles = [t for t in pupil.phasor_tiles()]
    for p, f, sc in zip(plan.problems, F, scale):
        _, _, a, o = tiles[p['tile']]
        ref = sc * w.double().cpu().numpy() * mft.dft2(a * np.exp(2j * np.pi * o / wl[p['wave']]), p['alpha'], (40, 40),
                                                       p['shift'], p['offset'], unitary=False)
        assert rel_l2(f.cpu().numpy(), ref) < tol
