"""Meta-data that a program sets on an image after making it, in any sequence of numbers (host
only): the descriptor takes it, and an image made like it does not share it."""
import numpy as np
import pytest
import torch


@pytest.mark.parametrize("kind", [tuple, list, np.array, torch.tensor])
def test_metadata_set_later(kind):
    from rtk_amd.filters import Image
    image = Image(torch.zeros(4, 3, 2))
    image.origin, image.spacing, image.index = kind([-1.5, 2., 3.]), kind([1., 2., 0.5]), kind([1, 0, 7])
    d = image.descriptor()
    assert list(d.size) == [2, 3, 4] and list(d.index) == [1, 0, 7]
    assert list(d.origin) == [-1.5, 2., 3.] and list(d.spacing) == [1., 2., 0.5]
    other = image.like(torch.zeros(1, 1, 1))
    if kind is not tuple:
        image.origin[0] = 9.
    assert (other.origin, other.spacing, other.index) == ((-1.5, 2., 3.), (1., 2., 0.5), (1, 0, 7))
    assert all(type(x) is float for x in other.origin + other.spacing) and all(type(x) is int for x in other.index)
