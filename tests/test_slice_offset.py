"""helper.slice_offset for every form of shape and index that numpy takes (CPU)."""
import numpy as np
import pytest

from lentil_amd.helper import slice_offset

BOX = np.s_[2:7, 3:9]


@pytest.mark.parametrize('shape', [(8, 8), [9, 8], 8, (8,), np.array([8, 9]), np.array(9), (9.0, 8.0)])
def test_shapes_broadcast(shape):
    centre = np.broadcast_to(shape, (2,)) // 2
    assert tuple(slice_offset(BOX, shape)) == (4 - centre[0], 6 - centre[1])


@pytest.mark.parametrize('shape', [(3, 8, 8), (), (1, 2, 3, 4)])
def test_other_shapes_are_refused(shape):
    with pytest.raises(ValueError):
        slice_offset(BOX, shape)


@pytest.mark.parametrize('kind', [int, np.int64, np.int8, np.uint8, np.uint64, float])
def test_indices_of_any_kind(kind):
    """Offsets left of the centre are negative, whatever type the indices have."""
    box = (slice(kind(1), kind(4)), slice(kind(0), kind(2)))
    assert tuple(slice_offset(box, (20, 600))) == (2 - 10, 1 - 300)
