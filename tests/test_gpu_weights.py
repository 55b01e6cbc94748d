"""Wavelength weights of any magnitude: an image is linear in them while its
values are ordinary float32 numbers.  Against the complex128 oracle at the
image gate (1e-5), through every path of a class to the image."""
import numpy as np
import pytest
import torch

from oracle import optics
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('precision', ['fp32', 'bf16x3'])
@pytest.mark.parametrize('kind', ['single', 'along_k', 'windows', 'fields'])
@pytest.mark.parametrize('level', [1e-38, 1e-36, 1e-33, 1e-25, 1e-18, 1.0, 1e30])
def test_weights_of_any_magnitude(precision, kind, level):
    import lentil_amd as L
    n, os, du, z = 72, 2, 5e-6, 10.0
    masks = np.zeros((3, n, n))
    for k in range(3):
        masks[k, 3 + 24 * k:21 + 24 * k, 5:60] = 1
    yy, xx = np.mgrid[:n, :n] / n - 0.5
    amp, opd = masks.sum(axis=0) * (1 + xx * yy), 3e-7 * (yy ** 2 - yy * xx)
    amp *= 1e3      # a peak of 1e6: the image of the least weight is 1e-32
    wl, wt = np.array([5.2e-7, 6e-7, 7e-7]), np.array([0.5, -0.2, 0.3])
    mask = None if kind == 'single' else masks
    tilt = {'windows': 1.0, 'fields': 9.0}.get(kind)
    px = np.random.default_rng(1).uniform(-1, 1, (3, 2)) * (tilt or 0)
    angles = px * du / os / z if tilt else []
    pupil = L.Pupil(amplitude=amp, opd=opd, pixelscale=1 / n, focal_length=z, mask=mask)
    pupil.tilt.extend(L.Tilt(*a) for a in angles)
    exact = optics.Pupil(amp, opd, 1 / n, z, mask=mask, tilt=[optics.Tilt(*a) for a in angles] or None)
    plan = L.PSFPlan(pupil, wl, wt * level, pixelscale=du, shape=(30, 47), prop_shape=(20, 20) if tilt else None,
                     oversample=os, precision=precision, contraction='per_tile')
    assert plan.info['coherent_fast'] == (0 if tilt else 1)
    ref = optics.broadband_image(exact, wl, wt, du, (30, 47), os, **(dict(prop_shape=(20, 20)) if tilt else {}))
    img = torch.zeros(plan.shape_out, dtype=torch.float64, device='cuda')
    plan(img)
    assert rel_l2(img.cpu().numpy() / level, ref) < 1e-5
    plan(img, accumulate=True)
    assert rel_l2(img.cpu().numpy() / level, 2 * ref) < 1e-5
