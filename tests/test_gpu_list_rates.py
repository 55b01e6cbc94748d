"""Transforms of one list share twiddle tables where their rates agree, and only
there: an entry whose rate is not a number leaves the others alone."""
import numpy as np
import pytest
import torch

from oracle import mft
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('precision, tol', [('fp32', 2e-6), ('bf16x3', 2e-5)])
@pytest.mark.parametrize('bad', [0, 1, 2])
def test_a_rate_that_is_not_a_number(precision, tol, bad):
    """Whichever entry it is; the fields' gates of the two forms."""
    from lentil_amd import fourier
    rng = np.random.default_rng(bad)
    f = (rng.standard_normal((40, 33)) + 1j * rng.standard_normal((40, 33))).astype(np.complex64)
    t = torch.from_numpy(f).cuda()
    rates = [0.01, 0.02, 0.01]
    rates[bad] = float('nan')
    got = fourier.dft2_list([(t, (a, a), (50, 61), (0, 0), (0, 0)) for a in rates], precision=precision)
    for k, (a, g) in enumerate(zip(rates, got)):
        if k == bad:
            assert torch.isnan(torch.view_as_real(g)).all()
        else:
            assert rel_l2(g.cpu().numpy(), mft.dft2(f.astype(complex), a, (50, 61))) < tol
