"""Which pixelscales Fields of one group may have (CPU): equal by value, and one that is not a number equals none."""
import numpy as np
import pytest

from lentil_amd.field import _check_pixelscales

NAN = float('nan')
ARRAY, NAN_ARRAY = np.array([1.0, 2.0]), np.array([1.0, NAN])


class _Field:
    def __init__(self, pixelscale):
        self.pixelscale = pixelscale


@pytest.mark.parametrize('values', [(None, None), (1, 1.0), (2.5,), (ARRAY, ARRAY), (ARRAY, ARRAY.copy(), ARRAY), ((1, 2), (1, 2))])
def test_equal(values):
    _check_pixelscales([_Field(v) for v in values])


@pytest.mark.parametrize('values', [(None, 1), (1, 2), (ARRAY, 2 * ARRAY), (NAN, NAN), (NAN_ARRAY, NAN_ARRAY), ((1, 2), (1, 3))])
def test_unequal(values):
    with pytest.raises(ValueError):
        _check_pixelscales([_Field(v) for v in values])
