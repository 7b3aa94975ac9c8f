"""One tangent product on both sides of the size (4,500 nodes) from which it
takes the tiled passes, and the tiled passes themselves in every form they have:
influence functions, linearized model, thermal strains, volumes that differ
(1,024 threads a tile), 4, 8 and 16 lanes a node, damage, prescribed DOFs. Against
the untiled kernels in FP64, which the oracle checks elsewhere: sums of up to
122 terms without cancellation in another order, 1e-12 of the largest."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

LARGE = (24, 17, 16)  # 6,528 nodes


def _problem(n, uniform, rng):
    h = 1e-3
    x, vol, nl = O.quickgrid(*n, [0, 0, 0], [k * h for k in n], 3.015 * h)
    if not uniform:
        vol = vol * rng.uniform(0.8, 1.2, size=len(vol))
    return x, vol, nl, 3.015 * h


def _broken(nl, n, rng):
    from peridigm_amd.core import list_to_csr
    rp, col = list_to_csr(nl, n)
    i = np.repeat(np.arange(n), np.diff(rp))
    key = rng.random(n)
    return ((key[np.minimum(i, col)] + key[np.maximum(i, col)]) % 1.0 < 0.2).astype(float)


def _both(ctx, f):
    out = []
    for variant in (0, 1):
        ctx.set_kernel_variant(variant)
        out.append(f())
    return out


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("influence", [0, 1, 2])
@pytest.mark.parametrize("model", ["Elastic", "Linear LPS", "thermal"])
@pytest.mark.parametrize("uniform,tile,lanes", [(True, 0, 4), (False, 32, 16), (True, 64, 8),
                                                (False, 64, 8), (False, 128, 4), (True, 128, 4)])
def test_tiled_product(influence, model, uniform, tile, lanes):
    from peridigm_amd import Context
    from peridigm_amd import quasistatic as Q
    rng = np.random.default_rng(23)
    x, vol, nl, hz = _problem(LARGE, uniform, rng)
    N = len(vol)
    u = 1e-3 * x[:, ::-1] + 2e-7 * rng.standard_normal(x.shape)
    w = rng.standard_normal(x.shape)
    fixed = np.unique(rng.integers(0, 3 * N, size=N // 4))
    with Context(0, lanes=lanes, tile_nodes=tile) as ctx:
        ctx.set_topology(nl, N)
        ctx.set_material_model("Elastic" if model == "thermal" else model)
        ctx.set_constants(x, vol, 130e9, 60e9, hz, influence, 1e-2)
        if model == "thermal":
            ctx.set_thermal_expansion(1e-5)
            ctx.set_temperature_change(rng.uniform(0.0, 50.0, size=N))
        assert ctx.tiling()[0] > 0
        for bd in (None, _broken(nl, N, rng)):
            ctx.upload_state(bond_damage=bd)
            Q.set_fixed(ctx, fixed)
            k0, k1 = _both(ctx, lambda: Q.tangent_apply(ctx, u, w))
            # another route, not the same one twice: the sums' order differs
            assert not np.array_equal(k0, k1) and _rel(k0, k1) <= 1e-12
            assert np.array_equal(k0.ravel()[fixed], w.ravel()[fixed])


@pytest.mark.parametrize("n,tiled", [((20, 15, 15), False), ((4501, 1, 1), True), ((30, 15, 10), False),
                                     ((4500, 1, 1), False), ((43, 35, 3), True)])
def test_size_from_which_one_product_is_tiled(n, tiled):
    from peridigm_amd import Context
    from peridigm_amd import quasistatic as Q
    rng = np.random.default_rng(5)
    x, vol, nl, hz = _problem(n, True, rng)
    u = 1e-3 * x + 2e-7 * rng.standard_normal(x.shape)
    w = rng.standard_normal(x.shape)
    assert (len(vol) > 4500) == tiled
    with Context(0) as ctx:
        ctx.set_topology(nl, len(vol))
        ctx.set_constants(x, vol, 130e9, 60e9, hz, 0, 0.0)
        assert ctx.tiling()[0] > 0
        k0, k1 = _both(ctx, lambda: Q.tangent_apply(ctx, u, w))
    assert np.array_equal(k0, k1) == (not tiled) and _rel(k0, k1) <= 1e-12


def test_coincident_points_in_a_tiled_product():
    from peridigm_amd import Context
    from peridigm_amd import quasistatic as Q
    rng = np.random.default_rng(3)
    x, vol, nl, hz = _problem(LARGE, True, rng)
    x = x.copy()
    x[1] = x[0]
    u = 1e-3 * x + 1e-6 * rng.standard_normal(x.shape)
    w = rng.standard_normal(x.shape)
    with Context(0) as ctx:
        ctx.set_topology(nl, len(vol))
        ctx.set_constants(x, vol, 130e9, 60e9, hz, 0, 0.0)
        k0, k1 = _both(ctx, lambda: Q.tangent_apply(ctx, u, w))
    assert np.isfinite(k1).all() and not np.array_equal(k0, k1) and _rel(k0, k1) <= 1e-11


@pytest.mark.parametrize("n,uniform,model,tile,lanes", [
    ((111, 59, 1), False, "Elastic", 32, 16), (LARGE, True, "Elastic", 64, 8),
    (LARGE, False, "Linear LPS", 32, 16), (LARGE, False, "Elastic", 128, 4)])
def test_stale_lds_does_not_reach_a_product(n, uniform, model, tile, lanes):
    """As for the solves and the set-up of the two-level preconditioner: what an
    earlier kernel left in LDS, NaN, in slots that masked-out bonds address."""
    from peridigm_amd import Context
    from peridigm_amd import quasistatic as Q
    rng = np.random.default_rng(7)
    x, vol, nl, hz = _problem(n, uniform, rng)
    xb, vb, nb, hb = _problem((60, 34, 34), False, rng)
    u = 1e-3 * x[:, ::-1]
    w = rng.standard_normal(x.shape)
    nan = np.full(xb.shape, np.nan)
    with Context(0, lanes=lanes, tile_nodes=tile) as ctx, Context(0) as big:
        for c, (p, v, l, z, m) in ((ctx, (x, vol, nl, hz, model)), (big, (xb, vb, nb, hb, "Elastic"))):
            c.set_topology(l, len(v))
            c.set_material_model(m)
            c.set_constants(p, v, 130e9, 60e9, z, 0, 0.0)
        clean = Q.tangent_apply(ctx, u, w)
        assert np.isfinite(clean).all()
        Q.tangent_apply(big, nan, nan)
        assert np.array_equal(Q.tangent_apply(ctx, u, w), clean)
