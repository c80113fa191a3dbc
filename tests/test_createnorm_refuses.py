"""What createnorm takes at the small end: two vertices are one segment, one
vertex is none, no vertex is an error."""
import numpy as np
import pytest

from fribois2d_amd.cases import createnorm


def test_number_of_vertices():
    assert createnorm([[0.0, 0.0], [1.0, 1.0]]).shape == (1, 2)
    assert createnorm(np.zeros((1, 2))).shape == (0, 2)
    for v in (np.zeros((0, 2)), np.zeros(0)):
        with pytest.raises(ValueError):
            createnorm(v)
