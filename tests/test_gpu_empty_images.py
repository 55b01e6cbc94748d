"""Images without pixels take a coherent group as they take a single Field: nothing is added."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape', [(0, 5), (7, 0), (0, 0)])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('count', [1, 2, 3])
def test_insert_into_an_empty_image(shape, dtype, count):
    import lentil_amd as L
    w = L.Wavefront(6e-7)
    w.data = [L.Field(torch.ones((6, 7 + k), dtype=torch.complex64, device='cuda')) for k in range(count)]
    out = torch.zeros(shape, dtype=dtype, device='cuda')
    assert w.insert(out) is out and out.shape == shape
    w.shape = shape
    assert w.intensity_tensor(dtype).shape == shape
