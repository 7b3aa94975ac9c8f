"""Search rows above the LDS row's 512 entries, which a kernel of their own sorts
in pieces of 4,096: one id more and less than a piece and two, rows that planes
shorten, rows of very different lengths in one list. Integers: exact."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4096, 4097, 4098, 8193, 8194])
def test_everything_in_reach(n):
    from peridigm_amd.discretization import radius_search
    x = np.random.default_rng(n).random((n, 3))
    rows = radius_search(x, 2.0).reshape(n, n)
    assert (rows[:, 0] == n - 1).all()
    want = np.arange(n - 1, dtype=np.int32)
    for i in range(n):
        assert np.array_equal(rows[i, 1:], want + (want >= i)), i


PLANE = np.array([[0.0, 1.0, 0.0, -1.0, 0.4, -1.0, 1.0, 0.0, 0.0, 1.5, 3.0]])


@pytest.mark.parametrize("planes", [None, PLANE])
@pytest.mark.parametrize("n,radius", [(4500, 0.45), (6000, 1.0), (5000, 0.25)])
def test_rows_of_many_lengths(n, radius, planes):
    from peridigm_amd.discretization import radius_search
    x = np.random.default_rng(n).random((n, 3)) ** 2  # dense towards a corner
    nl = O.radius_search(x, radius)
    if planes is not None:
        nl = O.filter_planes(x, nl, planes)
    assert np.array_equal(radius_search(x, radius, planes), nl)
