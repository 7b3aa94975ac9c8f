"""Contact lists where the search's waves and rows end, against the oracle's
(integers: exact): fewer points than a wave, buckets of more than 64 points,
bond rows of 0, 256 and more bonds (a row of up to 256 is searched in LDS),
rows of hundreds of contacts, cells that share a bucket."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bond,radius,shift", [(1, 0.1, 0.3, 0.0), (3, 0.01, 2.0, 0.3),
                                                 (257, 2.0, 0.7, 0.4), (258, 2.0, 0.5, 0.4),
                                                 (400, 0.9, 0.6, 0.5), (700, 0.05, 0.9, 0.2),
                                                 (900, 0.3, 0.12, 0.3), (1200, 0.2, 0.2, 5.0)])
def test_contact_rows(n, bond, radius, shift):
    from peridigm_amd import Context
    from peridigm_amd.core import csr_to_list
    rng = np.random.default_rng(n)
    x = rng.random((n, 3))
    nl = O.radius_search(x, bond)
    # some bonds of each point removed (both ends), so that near points are contacts
    rp, col = O.list_to_csr(nl, n)
    i = np.repeat(np.arange(n), np.diff(rp))
    key = rng.random(n)
    keep = (key[np.minimum(i, col)] + key[np.maximum(i, col)]) % 1.0 > 0.1
    if n in (257, 258):
        keep[:] = True  # rows of exactly 256 and 257 bonds
    nl = csr_to_list(np.concatenate([[0], np.cumsum(np.bincount(i[keep], minlength=n))]), col[keep])
    y = x + shift * (rng.random((n, 3)) - 0.5)
    with Context(0) as ctx:
        ctx.set_topology(nl, n)
        ctx.set_constants(x, np.full(n, 1e-3), 140e9, 48e9, bond, 0, 0.0)
        ctx.set_contact(radius, 10, 0.5 * radius, 1e12, 0.0)
        got = ctx.contact_search(y)
    assert np.array_equal(got, O.contact_search(y, radius, nl))
