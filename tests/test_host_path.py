"""Scalar shortcuts of the per-call path against the general NumPy forms they stand for (CPU)."""
import numpy as np
import pytest

from lentil_amd import _lib, extent as ext
from lentil_amd._arrays import two
from lentil_amd.helper import slice_offset
from lentil_amd.propagate import field_geometry


@pytest.mark.parametrize('value', [0.25, 3, True, np.float64(0.5), np.float32(0.1), (1, 2.5), [1, 2], (np.int64(3), 4),
                                   np.array([0.5, -2.0]), np.array(7), [4], (np.float32(0.3), 1)])
def test_pair_is_broadcast(value):
    want = tuple(float(v) for v in np.broadcast_to(value, (2,)))
    got = _lib.pair(value)
    assert got == want and all(type(v) is float for v in got)
    assert np.array_equal(two(value), np.broadcast_to(value, (2,))) and not two(value).flags.writeable


@pytest.mark.parametrize('value', [(1, 2, 3), [], np.zeros((2, 2))])
def test_pair_refuses_other_shapes(value):
    with pytest.raises(ValueError):
        _lib.pair(value)


@pytest.mark.parametrize('shape', [(8, 8), (9, 8), (301, 300)])
@pytest.mark.parametrize('box', [(0, 8, 0, 8), (1, 4, 2, 8), (3, 4, 0, 1), (2, 7, 5, 8)])
def test_slice_offset(shape, box):
    r0, r1, c0, c1 = box
    size = np.array((r1 - r0, c1 - c0))
    want = np.array((r0 + size[0] // 2, c0 + size[1] // 2)) - np.asarray(shape) // 2
    assert tuple(slice_offset(np.s_[r0:r1, c0:c1], shape)) == tuple(want)


class _Field:
    offset = (3, -2)

    def __init__(self, sh):
        self.sh = sh

    def shift(self, **kwargs):
        return self.sh


@pytest.mark.parametrize('sh', [(0.0, -0.0), (0.3, -0.7), (-1.0, 2.0), (12.5, -40.25), (-0.999, 63.5), (200.0, 0.0)])
@pytest.mark.parametrize('prop,out', [((64, 64), (64, 64)), ((31, 40), (64, 65)), ((100, 90), (51, 64))])
def test_field_geometry_scalars_match_arrays(sh, prop, out):
    out_ext = ext.array_extent(out, (0, 0))
    args = (5e-7, (1e-2, 1e-2), (5e-6, 5e-6), 10.0, np.array(prop), out_ext, 2)
    scalar = field_geometry(_Field(tuple(np.float64(v) for v in sh)), *args)
    general = field_geometry(_Field(tuple(np.array(v) for v in sh)), *args)     # 0-d arrays take the array branch
    assert (scalar is None) == (general is None)
    if scalar is not None:
        assert scalar.keys() == general.keys()
        for k in scalar:
            assert np.array_equal(np.asarray(scalar[k], float), np.asarray(general[k], float)), k
