"""Fixed-radius search on the device against the oracle's lists (integers:
exact), at the sizes where its waves and LDS rows end: rows of 0, 1, 63 to 65,
512 and 513 entries and beyond (an LDS row holds 512 before it is flushed in
pieces), cells of more than 64 points, one to three cells along an axis."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

PLANE = np.array([[0.0, 1.0, 0.0, -1.0, 0.4, -1.0, 1.0, 0.0, 0.0, 1.5, 3.0],
                  [1.0, 0.0, 0.0, 0.7, -1.0, -1.0, 0.0, 1.0, 0.0, 3.0, 3.0]])


@pytest.mark.parametrize("planes", [None, PLANE])
@pytest.mark.parametrize("n,radius", [(1, 0.1), (2, 2.0), (5, 0.02), (64, 2.0), (65, 2.0),
                                      (66, 2.0), (513, 2.0), (514, 2.0), (515, 2.0), (1500, 0.6),
                                      (1500, 2.0), (3000, 0.15), (2000, 0.34)])
def test_radius_search_rows(n, radius, planes):
    from peridigm_amd.discretization import radius_search
    x = np.random.default_rng(n).random((n, 3))
    nl = O.radius_search(x, radius)
    if planes is not None:
        nl = O.filter_planes(x, nl, planes)
    assert np.array_equal(radius_search(x, radius, planes), nl)


def test_coincident_points():
    from peridigm_amd.discretization import radius_search
    x = np.zeros((700, 3))
    x[650:] = 1.0
    assert np.array_equal(radius_search(x, 0.5), O.radius_search(x, 0.5))
