"""More than 2^26 points: kernels that give a wave to each point then need more
than 2^32 threads, more than one axis of a launch holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_radius_search_of_more_points_than_waves_on_an_axis():
    from peridigm_amd.discretization import radius_search
    n = (1 << 26) + 5
    x = np.zeros((n, 3))
    x[:, 0] = np.arange(n)
    print("search of", n, "points", flush=True)
    nl = radius_search(x, 1.0)
    assert nl.size == 3 * n - 2
    # rows 0 and n - 1 hold one neighbour, the others two
    assert nl[:2].tolist() == [1, 1] and nl[-2:].tolist() == [1, n - 2]
    rows = nl[2:-2].reshape(-1, 3)
    i = np.arange(1, n - 1, dtype=np.int32)
    assert (rows[:, 0] == 2).all() and (rows[:, 1] == i - 1).all() and (rows[:, 2] == i + 1).all()


def test_bond_fields_and_contacts_of_points_on_the_second_axis():
    """Just above the 2^22 waves of a launch's first axis: a chain whose points
    are bonded to the next ones and in contact with those after them."""
    from peridigm_amd import Context
    n = (1 << 22) + 7
    x = np.zeros((n, 3))
    x[:, 0] = np.arange(n)
    i = np.arange(n, dtype=np.int32)
    nl = np.empty(3 * n - 2, np.int32)
    nl[:2], nl[-2:] = (1, 1), (1, n - 2)
    nl[2:-2].reshape(-1, 3)[:] = np.stack([np.full(n - 2, 2, np.int32), i[:-2], i[2:]], axis=1)
    print("context of", n, "points", flush=True)
    with Context(0) as ctx:
        ctx.set_topology(nl, n)
        ctx.set_constants(x, np.ones(n), 130e9, 60e9, 1.1, 0, 1e-2)
        # bond k joins points k and k + 1: list entries 2 k and 2 k + 1
        bd = np.repeat((np.random.default_rng(3).random(n - 1) < 0.3).astype(float), 2)
        ctx.upload_state(bond_damage=bd)
        assert np.array_equal(ctx.download_state()["bond_damage"], bd)
        ctx.set_contact(2.5, 10, 0.9, 1.0)
        got = ctx.contact_search(x)
    want = [np.r_[1, 2], np.r_[1, 3], *(np.r_[2, k - 2, k + 2] for k in range(2, 100))]
    assert np.array_equal(got[:4 + 3 * 98], np.concatenate(want))
    rows = got[4:-4].reshape(-1, 3)
    assert (rows[:, 0] == 2).all()
    assert np.array_equal(np.sort(rows[:, 1:], axis=1), np.stack([i[2:-2] - 2, i[2:-2] + 2], axis=1))
    assert got[-4:].tolist() == [1, n - 4, 1, n - 3]
