"""Shapes of the tensor backend's operations (born_amd/backend.py), without a GPU."""
import pytest


def test_a_shape_may_be_a_list():
    """A program may set a tensor's shape to a list; what is kept for tuples is not kept for it."""
    from born_amd import backend as BK
    shape = [2, 3, 4]
    assert list(BK._shape_arr(shape)) == shape and list(BK._shape_arr(tuple(shape))) == shape
    shape[0] = 5
    assert list(BK._shape_arr(shape)) == [5, 3, 4] and list(BK._shape_arr((2, 3, 4))) == [2, 3, 4]
    assert BK._broadcast([2, 1], (2, 3)) == (2, 3) and BK._broadcast([2, 3], [4, 3]) is None and BK._broadcast([3], [2, 3]) is None
    with pytest.raises(TypeError):
        BK._shape_arr(("a",))
