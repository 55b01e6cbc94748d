"""Plans whose small windows lie in an image of more than 2^32 pixels: a launch
holds fewer threads than that, and every pixel is written."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
SIDE = 65600    # 17 GB of float32


@pytest.mark.parametrize('segments', [False, True])
def test_windows_in_a_giant_image(segments):
    """The window at the image's end against the same plan on a small image; all
    else zero, and left alone when adding.  Segments far apart store Fields."""
    import lentil_amd as L
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        torch.cuda.empty_cache()
    n, du, z = 32, 5e-6, 10.0
    masks = np.zeros((2, n, n))
    masks[0, 2:15, 3:29] = masks[1, 17:30, 3:29] = 1
    yy, xx = np.mgrid[:n, :n] / n - 0.5
    wl = [5e-7, 6e-7]

    def plan(side):
        p = L.Pupil(amplitude=masks.sum(0), opd=2e-7 * xx * yy, mask=masks if segments else None, pixelscale=1 / n,
                    focal_length=z)
        if segments:
            p.tilt.extend(L.Tilt(x=k * 20 * du / z, y=0) for k in (-0.5, 0.5))
        # 40 pixels from the end on both axes, and a quarter so that rounding leaves the whole pixels alone
        shift = (side // 2 - 39.75) * du / z
        return L.PSFPlan(p, wl, None, pixelscale=du, shape=side, prop_shape=24, oversample=1, tilts=[L.Tilt(shift, -shift)],
                         precision='fp32')

    small = plan(200)()
    assert float(small[100:, 100:].sum(dtype=torch.float64)) == float(small.sum(dtype=torch.float64))
    big, end, eps = plan(SIDE), slice(SIDE - 200, None), 1e-5 * float(small.max())
    out = torch.full((SIDE, SIDE), float('nan'), device='cuda')
    big(out)
    assert float((out[end, end] - small).abs().max()) < eps
    assert int((out == 0).sum()) == SIDE * SIDE - int((out[end, end] != 0).sum())
    out.fill_(1.0)
    big(out, accumulate=True)
    assert float((out[end, end] - 1 - small).abs().max()) < eps + 2 ** -23 * float(small.max())
    assert int((out == 1).sum()) == SIDE * SIDE - int((out[end, end] != 1).sum())
