"""Bond fields up and back where their route has an edge: the last word of the
bits (a field of 64 k, and one bond more or less), fields that one, four and
eight threads pack, rows whose neighbours do and do not ascend (the index map is
then computed or copied), untiled meshes with rows past 128, and the values a
field may and may not hold, anywhere in it. Exact throughout."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pairs(nl, n):
    from peridigm_amd.core import list_to_csr
    rp, col = list_to_csr(nl, n)
    i = np.repeat(np.arange(n), np.diff(rp))
    lo, hi = np.minimum(i, col), np.maximum(i, col)
    _, pair = np.unique(lo.astype(np.int64) * n + hi, return_inverse=True)
    return rp, col, pair  # pair: the same number at both ends of a bond


def _shuffled(nl, rp, col, rng):
    """The list with every row in another order, and the order."""
    key = np.repeat(np.arange(len(rp) - 1), np.diff(rp)) + rng.random(len(col))
    order = np.argsort(key)
    out = nl.copy()
    mask = np.ones(len(nl), bool)
    mask[rp[:-1] + np.arange(len(rp) - 1)] = False
    out[mask] = col[order]
    return out, order


CASES = [((33, 1, 1), 1.1), ((32, 1, 1), 1.1), ((34, 1, 1), 1.1), ((12, 11, 3), 3.015),
         ((24, 20, 20), 3.015), ((52, 30, 30), 3.015), ((9, 9, 9), 4.6)]


@pytest.mark.parametrize("ascending", [True, False])
@pytest.mark.parametrize("n,horizon", CASES)
def test_round_trip_and_refusals(n, horizon, ascending):
    from peridigm_amd import Context
    from peridigm_amd._lib import PdgError
    from peridigm_amd.discretization import lattice_centres, radius_search
    rng = np.random.default_rng(9)
    x, vol = lattice_centres(n, [0, 0, 0], list(n))
    x = x[rng.permutation(len(vol))]
    N = len(vol)
    nl = radius_search(x, horizon)
    rp, col, pair = _pairs(nl, N)
    if not ascending:
        nl, order = _shuffled(nl, rp, col, rng)
        col, pair = col[order], pair[order]
    B = len(col)
    u = 1e-4 * x
    with Context(0) as ctx:
        ctx.set_topology(nl, N)
        ctx.set_constants(x, vol, 130e9, 78e9, horizon, 0, 1e-2)
        f = []
        for share in (0.0, 0.02, 0.5, 1.0):
            broken = rng.random(pair.max() + 1) < share
            bd = broken[pair].astype(float)
            bd[bd == 0.0] = rng.choice([0.0, -0.0], size=int((bd == 0.0).sum()))
            ctx.upload_state(bond_damage=bd)
            assert np.array_equal(ctx.download_state()["bond_damage"], bd)
            f.append(ctx.compute_force(x + u, bd)[1])
            out, dmg, _ = ctx.compute_damage(x + u, bd)
            assert np.array_equal(out, bd)
            at = np.add.reduceat(np.r_[bd, 0.0], np.minimum(rp[:-1], B))
            deg = np.diff(rp)
            assert np.array_equal(dmg, np.where(deg > 0, at, 0.0) / np.maximum(deg, 1))
        # a field of ones is no force; a field of zeros is that of no field
        assert not f[3].any() and np.array_equal(f[0], ctx.compute_force(x + u)[1])
        for k in (0, B // 2, B - 1):
            ctx.upload_state(bond_damage=bd)  # a call without a field leaves every bond intact
            for value in (0.5, np.nan, np.inf, -1.0, 5e-324, 2.0, 1.0 - bd[k]):
                wrong = bd.copy()
                wrong[k] = value
                with pytest.raises(PdgError) as e:
                    ctx.upload_state(bond_damage=wrong)
                assert e.value.code == -3
                assert np.array_equal(ctx.download_state()["bond_damage"], bd)
            # intact but for one end of one bond
            one = np.zeros(B)
            one[k] = 1.0
            with pytest.raises(PdgError) as e:
                ctx.compute_force(x + u, one)
            assert e.value.code == -3
