"""Phase retrieval with an OPD, diversities and gradients of every shape that
broadcasts to the pupil, leading axes of length 1 among them."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
N = 33


def _model(lead=0):
    from lentil_amd.autograd import BroadbandPSFModel
    yy, xx = np.mgrid[:N, :N] / N - 0.5
    div = [2e-7 * k * (xx ** 2 + yy ** 2).reshape((1,) * lead + (N, N)) for k in range(2)]
    return BroadbandPSFModel(np.hypot(xx, yy) < 0.5, div, [5e-7, 6e-7], 0.5, 1 / N, 5e-6, 10.0, 16)


def _opd():
    yy, xx = np.mgrid[:N, :N] / N - 0.5
    return torch.from_numpy(1e-7 * xx * yy).cuda()


@pytest.mark.parametrize('lead', [0, 1, 2])
@pytest.mark.parametrize('dtype', [torch.float64, torch.float32])
def test_leading_axes(lead, dtype):
    plain, model, o = _model(), _model(lead), _opd().to(dtype)
    a, b = o.clone().requires_grad_(), o.reshape((1,) * lead + (N, N)).clone().requires_grad_()
    ia, ib = plain(a), model(b)
    assert torch.equal(ia, ib)
    g = torch.rand_like(ia)
    ia.backward(g)
    ib.backward(g)
    assert b.grad.shape == b.shape and torch.equal(a.grad, b.grad.reshape(N, N))


@pytest.mark.parametrize('shape', [(1, N), (N,), (N, 1), ()])
def test_broadcast(shape):
    """An OPD of fewer rows, columns or dimensions is the full one it broadcasts to."""
    o = _opd()
    o = (o[:1] if shape == (1, N) else o[0] if shape == (N,) else o[:, :1] if shape == (N, 1) else o[0, 1]).clone()
    model = _model()
    assert torch.equal(model(o), model(o.expand(N, N).contiguous()))


@pytest.mark.parametrize('shape', [(2, N, N), (1, 2, N, N), (N, N + 1), (0, N, N)])
def test_other_shapes_are_refused(shape):
    model = _model()
    with pytest.raises((ValueError, RuntimeError)):
        model(torch.zeros(shape, dtype=torch.float64, device='cuda'))
    assert torch.isfinite(model(_opd())).all()
