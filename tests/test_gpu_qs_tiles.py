"""The LDS-tiled FP64 quasi-static passes against the untiled kernels, which
the oracle checks elsewhere.

Both evaluate the same formulas in FP64. A bond's extension is known to about
2 eps of its length, so at strains of 1e-3 a force term is good to 2 eps / 1e-3
= 4e-13 of itself; with up to 128 terms of mixed sign the sums are held to
1e-11 of the largest (residual, dilatation) and the tangent, whose terms carry
no such cancellation, to 1e-12.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _mesh(n, rng, uniform):
    h = 1e-3
    x, vol, nl = O.quickgrid(*n, [0, 0, 0], [k * h for k in n], 3.015 * h)
    if not uniform:
        vol = vol * rng.uniform(0.8, 1.2, size=len(vol))
    return x, vol, nl, 3.015 * h


def _broken(nl, n, rng):
    """A symmetric bond-damage field with a fifth of the bonds broken."""
    from peridigm_amd.core import list_to_csr
    rp, col = list_to_csr(nl, n)
    i = np.repeat(np.arange(n), np.diff(rp))
    pair = rng.random(n)[np.minimum(i, col)] + rng.random(n)[np.maximum(i, col)]
    return (pair % 1.0 < 0.2).astype(float)


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


# sizes: fewer nodes than a tile, one past a tile, several tiles with a short last one
CASES = [(influence, model, uniform, tile, lanes, n)
         for influence in (0, 1, 2) for model in ("Elastic", "Linear LPS", "thermal")
         for uniform, tile, lanes, n in ((True, 0, 4, (4, 3, 2)), (False, 32, 8, (11, 3, 1)),
                                         (True, 128, 4, (13, 9, 7)), (False, 128, 4, (13, 9, 7)),
                                         (True, 64, 8, (21, 6, 5)), (False, 0, 64, (12, 8, 8)))]


@pytest.mark.parametrize("influence,model,uniform,tile,lanes,n", CASES)
def test_tiled_passes_match_untiled(influence, model, uniform, tile, lanes, n):
    from peridigm_amd import Context
    from peridigm_amd import quasistatic as Q
    rng = np.random.default_rng(17)
    x, vol, nl, hz = _mesh(n, rng, uniform)
    N = len(vol)
    bd = _broken(nl, N, rng)
    u = 1e-3 * x[:, ::-1] + 2e-7 * rng.standard_normal(x.shape)
    w = rng.standard_normal(x.shape)
    fixed = np.unique(rng.integers(0, 3 * N, size=N // 4 + 1))
    out = {}
    with Context(0, lanes=lanes, tile_nodes=tile) as ctx:
        ctx.set_topology(nl, N)
        ctx.set_material_model("Elastic" if model == "thermal" else model)
        ctx.set_constants(x, vol, 130e9, 60e9, hz, influence, 1e-2)
        if model == "thermal":
            ctx.set_thermal_expansion(1e-5)
            ctx.set_temperature_change(rng.uniform(0.0, 50.0, size=N))
        ctx.upload_state(bond_damage=bd)
        Q.set_fixed(ctx, fixed)
        assert ctx.tiling()[0] > 0
        for variant in (0, 1):
            ctx.set_kernel_variant(variant)
            f, th = Q.force_and_dilatation(ctx, u)
            out[variant] = (f, th, Q.residual(ctx, u)[0], Q.tangent_apply(ctx, u, w))
    (f0, t0, r0, k0), (f1, t1, r1, k1) = out[0], out[1]
    assert _rel(f0, f1) <= 1e-11 and _rel(t0, t1) <= 1e-11 and _rel(r0, r1) <= 1e-11
    assert np.array_equal(r0.ravel()[fixed], np.zeros(len(fixed)))
    assert _rel(k0, k1) <= 1e-12
    assert np.array_equal(k0.ravel()[fixed], w.ravel()[fixed])


def test_coincident_points():
    """Two bonded points with one reference position: the untiled kernels give
    such a bond no dilatation term but a finite force, and so do the tiled."""
    from peridigm_amd import Context
    from peridigm_amd import quasistatic as Q
    rng = np.random.default_rng(3)
    x, vol, nl, hz = _mesh((6, 4, 4), rng, True)
    x = x.copy()
    x[1] = x[0]
    u = 1e-3 * x + 1e-6 * rng.standard_normal(x.shape)
    w = rng.standard_normal(x.shape)
    out = {}
    with Context(0) as ctx:
        ctx.set_topology(nl, len(vol))
        ctx.set_constants(x, vol, 130e9, 60e9, hz, 0, 0.0)
        for variant in (0, 1):
            ctx.set_kernel_variant(variant)
            out[variant] = (Q.residual(ctx, u)[0], Q.tangent_apply(ctx, u, w))
    for a, b in zip(out[0], out[1]):
        assert np.isfinite(b).all() and _rel(a, b) <= 1e-11


def _bar(n):
    from peridigm_amd import Context, discretization
    from peridigm_amd import quasistatic as Q
    h = 1e-3
    x, vol = discretization.lattice_centres(n, [0, 0, 0], [k * h for k in n])
    nl = discretization.radius_search(x, 3.015 * h)
    i = np.rint(x[:, 0] / h - 0.5).astype(int)
    ctx = Context(0)
    ctx.set_topology(nl, len(vol))
    ctx.set_constants(x, vol, 130e9, 78e9, 3.015 * h, 0, 0.0)
    fixed = Q.end_dofs(np.nonzero(i <= 1)[0], np.nonzero(i >= n[0] - 2)[0])
    Q.set_fixed(ctx, fixed)
    return ctx, x, fixed


# 120 nodes (one workgroup of the update), 1,920, and 67,200 (wide workgroups)
@pytest.mark.parametrize("n", [(8, 5, 3), (20, 12, 8), (42, 40, 40)])
@pytest.mark.parametrize("precond", ["none", "block_jacobi", "two_level"])
def test_solve_from_a_guess(n, precond):
    """Solves from a non-zero guess on tiled and untiled kernels: the residual
    by the tangent itself is the reported one (1e-8, plus the drift of the
    recursive residual, far below a tenth of it)."""
    from peridigm_amd import quasistatic as Q
    ctx, x, fixed = _bar(n)
    with ctx:
        rng = np.random.default_rng(5)
        u = 2e-4 * x
        b = rng.standard_normal(x.shape)
        b.reshape(-1)[fixed] = 0.0
        x0 = rng.standard_normal(x.shape) * 1e-9
        x0.reshape(-1)[fixed] = 0.0
        for variant in (0, 1):
            ctx.set_kernel_variant(variant)
            xs, it, rel = Q.solve(ctx, u, b, x0=x0, precond=precond, rel_tol=1e-8)
            r = np.linalg.norm(b - Q.tangent_apply(ctx, u, xs)) / np.linalg.norm(b)
            assert it > 0 and rel <= 1e-8 and r <= 1.1e-8


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("precond", ["none", "block_jacobi"])
def test_iteration_limit(precond, graphs):
    """A solve cut off after k iterations reports it and leaves the k-th
    iterate: the same on tiled, untiled and replayed launches (FP64 sums in
    another order over at most 13 iterations: 1e-10)."""
    from peridigm_amd import quasistatic as Q
    from peridigm_amd.learned import _iterate
    from peridigm_amd._lib import PdgError
    ctx, x, fixed = _bar((20, 8, 6))
    with ctx:
        Q.set_graphs(ctx, graphs)
        rng = np.random.default_rng(6)
        u = 2e-4 * x
        b = rng.standard_normal(x.shape)
        b.reshape(-1)[fixed] = 0.0
        with pytest.raises(PdgError) as e:
            Q.solve(ctx, u, b, precond=precond, max_iter=6)
        assert e.value.code == -5
        if precond == "block_jacobi":
            for k in (0, 1, 4, 7, 9, 13):
                it = []
                for variant in (0, 1):
                    ctx.set_kernel_variant(variant)
                    it.append(_iterate(ctx, u, b, k, 1e-12))
                assert np.abs(it[0] - it[1]).max() <= 1e-10 * max(np.abs(it[1]).max(), 1e-300)
