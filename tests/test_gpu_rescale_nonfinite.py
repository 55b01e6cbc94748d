"""Samples that are not finite reach the outputs whose spline taps lie on them
and no others: taps past the line count as zero in mode 'grid-constant',
whatever the image holds.  Against scipy's map_coordinates (the oracle), at
its 1e-11, and against 0 beyond the padded line."""
import numpy as np
import pytest
import torch

from oracle import detector as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('order', [0, 1])
@pytest.mark.parametrize('bad', [np.nan, np.inf, complex(1, np.nan)])
def test_columns_past_the_line_ignore_column_0(order, bad):
    """Orders without a prefilter, real and complex: the oracle's values and its non-finite places."""
    import lentil_amd as L
    rng = np.random.default_rng(order)
    img = rng.uniform(1, 2, (21, 26)) + (1j * rng.uniform(1, 2, (21, 26)) if np.iscomplexobj(bad) else 0)
    img[3:6, 0] = bad
    for scale, shape in ((1.3, (40, 60)), (0.7, (30, 33))):
        ref = D.rescale(img, scale, shape=shape, order=order, mode='grid-constant', unitary=False)
        got = L.rescale(img, scale, shape=shape, order=order, mode='grid-constant', unitary=False)
        finite = np.isfinite(ref)
        assert not finite.all() and finite[:, shape[1] // 2:].all()
        assert np.array_equal(np.isfinite(got), finite)
        assert np.abs(got[finite] - ref[finite]).max() <= 1e-11 * np.abs(ref[finite]).max()


@pytest.mark.parametrize('order', range(6))
def test_zero_beyond_the_padded_line(order):
    """Every order: outputs more than the padding and the taps past the line are 0."""
    import lentil_amd as L
    img = np.random.default_rng(order).uniform(1, 2, (20, 24))
    img[7, 0] = np.nan
    got = L.rescale(torch.from_numpy(img).cuda(), 1.0, shape=(20, 100), order=order, mode='grid-constant', unitary=False)
    assert torch.equal(got[:, 80:], torch.zeros_like(got[:, 80:]))
