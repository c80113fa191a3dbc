"""The vectorised normals against the segment formulas."""
import math

import numpy as np

from fribois2d_amd.cases import createnorm


def test_createnorm_equals_the_segment_formulas():
    """All segments at once give the bits of rigid.F90:468-495 taken segment
    by segment (cross product of the segment with the vector to its lifted
    midpoint, divided by its length)."""
    rng = np.random.default_rng(4)
    for n in (1, 2, 5, 377):
        v = 20.0 * rng.standard_normal((n + 1, 2))
        for orient in (-1.0, 1.0):
            ref = np.zeros((n, 2))
            for i in range(n):
                t1, t2 = np.array([0.0, *v[i]]), np.array([0.0, *v[i + 1]])
                a, b = t2 - t1, np.array([orient, *((v[i] + v[i + 1]) * 0.5)]) - t1
                cr = np.array([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])
                ref[i] = (cr / math.sqrt(float(np.sum(cr ** 2))))[1:]
            assert np.array_equal(createnorm(v, orient), ref)
