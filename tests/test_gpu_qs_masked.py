"""Bonds past a row's end address LDS slots that the tile does not fill: what an
earlier kernel left there, NaN among it, must not reach a result. The
two-level set-up and every tiled quasi-static pass after passes whose halos
were all NaN, against the same before them, bit for bit."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _bar(ctx, n, uniform, model):
    h = 1e-3
    x, vol, nl = O.quickgrid(*n, [0, 0, 0], [k * h for k in n], 3.015 * h)
    if not uniform:
        vol = vol * np.random.default_rng(2).uniform(0.8, 1.2, size=len(vol))
    ctx.set_topology(nl, len(vol))
    ctx.set_material_model(model)
    ctx.set_constants(x, vol, 130e9, 60e9, 3.015 * h, 0, 0.0)
    return x, np.flatnonzero(np.repeat(x[:, 0] < x[:, 0].min() + 1.5 * h, 3))


@pytest.mark.parametrize("n,uniform,model,tile,lanes", [
    ((24, 9, 1), False, "Elastic", 32, 16), ((24, 9, 1), True, "Elastic", 64, 8),
    ((9, 5, 4), False, "Linear LPS", 32, 16), ((30, 10, 10), True, "Elastic", 128, 4)])
def test_stale_lds_does_not_reach_results(n, uniform, model, tile, lanes):
    from peridigm_amd import Context
    from peridigm_amd import quasistatic as Q
    rng = np.random.default_rng(7)
    with Context(0, lanes=lanes, tile_nodes=tile) as ctx, Context(0) as big:
        x, fixed = _bar(ctx, n, uniform, model)
        xb, fb = _bar(big, (60, 34, 34), False, "Elastic")
        if n[2] == 1:
            fixed = np.union1d(fixed, 3 * np.arange(len(x)) + 2)
        Q.set_fixed(big, fb)
        nan = np.full(xb.shape, np.nan)
        u = 1e-3 * x[:, ::-1] * (x[:, 2:] != x[0, 2] if n[2] > 1 else np.array([1.0, 1.0, 0.0]))
        b = rng.standard_normal(x.shape)
        b.ravel()[fixed] = 0.0
        w = rng.standard_normal(x.shape)
        got = []
        for poison in (False, True):
            Q.set_fixed(ctx, fixed)  # the coarse matrix is set up anew
            if poison:
                Q.tangent_apply(big, nan, nan)
            t = Q.tangent_apply(ctx, u, w)
            if poison:
                Q.tangent_apply(big, nan, nan)
            got.append((t, Q.solve(ctx, u, b, precond="two_level", max_iter=400)[0]))
    for a, c in zip(*got):
        assert np.all(np.isfinite(c)) and np.array_equal(a, c)
