"""The reach of a sample that is not finite through the spline prefilter: that
of every tap of the explicit algorithm (48 to either side), whatever taps a
finite image needs.  Places and values against the oracle's explicit algorithm,
at the detector operators' 1e-11."""
import numpy as np
import pytest
import torch

from oracle import detector as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('order', [2, 3, 4, 5])
@pytest.mark.parametrize('mode', ['nearest', 'mirror', 'grid-wrap', 'constant', 'grid-constant'])
@pytest.mark.parametrize('bad, at', [(np.nan, (30, 100)), (np.inf, (0, 3)), (-np.inf, (111, 259))])
def test_reach(order, mode, bad, at):
    import lentil_amd as L
    img = np.random.default_rng(order).uniform(1, 2, (112, 260))
    img[at] = bad
    shape, scale = (21, 48), 0.1875
    xx, yy = D.rescale_coords(img.shape, scale, shape)
    with np.errstate(invalid='ignore'):
        ref = D.map_coordinates_explicit(img, yy, xx, order, mode)
    got = L.rescale(torch.from_numpy(img).cuda(), scale, shape=(shape[0] / scale, shape[1] / scale), mask=np.ones(img.shape),
                    order=order, mode=mode, unitary=False).cpu().numpy()
    assert got.shape == shape
    finite = np.isfinite(ref)
    assert 0 < finite.sum() < finite.size
    assert np.array_equal(np.isfinite(got), finite)
    assert np.abs(got[finite] - ref[finite]).max() <= 1e-11 * np.abs(ref[finite]).max()


@pytest.mark.parametrize('mode', ['nearest', 'reflect', 'grid-wrap', 'constant'])
@pytest.mark.parametrize('order', [2, 3, 4, 5])
def test_unitary_has_the_same_reach(order, mode):
    """The sums of a unitary result are not finite either, so nothing of it is; an
    infinite sample of both signs in different places must not cancel in them."""
    import lentil_amd as L
    img = np.random.default_rng(order).uniform(1, 2, (64, 150))
    img[3, 5], img[60, 140] = np.inf, -np.inf
    got = L.rescale(torch.from_numpy(img).cuda(), 0.5, mask=np.ones(img.shape), order=order, mode=mode, unitary=True)
    assert not torch.isfinite(got).any()


@pytest.mark.parametrize('where', ['re', 'im'])
def test_components_apart(where):
    """A bad imaginary part leaves the real parts' reach alone, and the other way round."""
    import lentil_amd as L
    rng = np.random.default_rng(7)
    re, im = rng.uniform(1, 2, (90, 120)), rng.uniform(1, 2, (90, 120))
    (re if where == 're' else im)[44, 60] = np.nan
    got = L.rescale(torch.complex(torch.from_numpy(re), torch.from_numpy(im)).cuda(), 0.5, mask=np.ones(re.shape), unitary=False)
    for part, ref in ((got.real, re), (got.imag, im)):
        alone = L.rescale(torch.from_numpy(ref).cuda(), 0.5, mask=np.ones(re.shape), unitary=False)
        assert torch.equal(torch.nan_to_num(part, nan=-1.0), torch.nan_to_num(alone, nan=-1.0))
