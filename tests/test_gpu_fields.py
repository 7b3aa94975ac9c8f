"""Node fields across the boundary: what goes up in reference order comes back
in it, bit for bit, at sizes on both sides of the transfer rules (vectors of up
to 2 MB go up through the staging buffer; results of 2 MB and of 32 MB take
more threads)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1, 1, 1), (3, 3, 3), (21, 20, 20), (44, 44, 45), (44, 44, 46),
                               (100, 60, 52)])
def test_state_round_trip(n):
    from peridigm_amd import Context
    from peridigm_amd.discretization import lattice_centres, radius_search
    h = 1e-3
    x, vol = lattice_centres(n, [0, 0, 0], [k * h for k in n])
    rng = np.random.default_rng(1)
    order = rng.permutation(len(vol))  # a numbering far from the internal one
    x = x[order]
    nl = radius_search(x, 1.1 * h)
    with Context(0) as ctx:
        ctx.set_topology(nl, len(vol))
        ctx.set_constants(x, vol, 130e9, 78e9, 1.1 * h, 0, 1e-2)
        ctx.set_density(7800.0)
        for k in range(2):
            u, v, a = (rng.standard_normal(x.shape) * 1e-5 for _ in range(3))
            ctx.upload_state(u=u, v=v, a=None if k else a)
            st = ctx.download_state()
            assert np.array_equal(st["u"], u) and np.array_equal(st["v"], v)
            assert np.array_equal(st["a"], np.zeros_like(a) if k else a)
        ctx.upload_state()
        assert not ctx.download_state()["u"].any()
        # per-node results come back in the same numbering: a uniform stretch
        # gives theta = 3 strain at the nodes with a full, symmetric stencil
        th, f = ctx.compute_force((1.0 + 1e-4) * x)
        inner = np.all((x > 1.01 * h) & (x < (np.array(n) - 1.01) * h), axis=1)
        assert np.abs(th[inner] - 3e-4).max(initial=0.0) <= 1e-8
        bd, dmg, _ = ctx.compute_damage((1.0 + 2e-2 * (x[:, :1] < 0.3 * n[0] * h)) * x)
        deg = np.array([nl[p] for p in _heads(nl, len(vol))])
        at = np.concatenate([[0], np.cumsum(deg)])
        want = [bd[at[i]:at[i + 1]].sum() / max(deg[i], 1) for i in range(0, len(vol), 97)]
        assert np.array_equal(dmg[::97], want)


def _heads(nl, n):
    p, out = 0, []
    for _ in range(n):
        out.append(p)
        p += nl[p] + 1
    return out


# 24 nodes (rows of up to 23 bonds), rows past 64 bonds, and 5.3M bonds (two
# chunks of the bond field, several threads)
@pytest.mark.parametrize("n", [(4, 3, 2), (9, 8, 7), (60, 30, 30)])
def test_bond_field_round_trip(n):
    from peridigm_amd import Context
    from peridigm_amd._lib import PdgError
    from peridigm_amd.core import list_to_csr
    from peridigm_amd.discretization import lattice_centres, radius_search
    h = 1e-3
    x, vol = lattice_centres(n, [0, 0, 0], [k * h for k in n])
    rng = np.random.default_rng(2)
    x = x[rng.permutation(len(vol))]
    N = len(vol)
    nl = radius_search(x, 3.015 * h)
    rp, col = list_to_csr(nl, N)
    i = np.repeat(np.arange(N), np.diff(rp))
    key = rng.random(N)
    with Context(0) as ctx:
        ctx.set_topology(nl, N)
        ctx.set_constants(x, vol, 130e9, 78e9, 3.015 * h, 0, 1e-2)
        for share in (0.0, 0.3, 1.0):
            bd = ((key[np.minimum(i, col)] + key[np.maximum(i, col)]) % 1.0 < share).astype(float)
            ctx.upload_state(bond_damage=bd)
            assert np.array_equal(ctx.download_state()["bond_damage"], bd)
        # a rejected field (one value, or one end only, in the last chunk) leaves
        # the state as it was
        for value in (0.5, np.nan, 1.0 - bd[-1]):
            wrong = bd.copy()
            wrong[-1] = value
            with pytest.raises(PdgError) as e:
                ctx.upload_state(bond_damage=wrong)
            assert e.value.code == -3
            assert np.array_equal(ctx.download_state()["bond_damage"], bd)
