"""A bond whose two points the deformation brings to one place. Its extension is
-|xi|, so the dilatation stays finite everywhere; its force has no direction,
so the force of its two ends is undefined, and that of every other point is
not. Tiled passes against the untiled kernels, FP64 in another order (1e-11 of
the largest, as for other states)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("influence", [0, 1, 2])
@pytest.mark.parametrize("uniform,thermal,n", [(True, False, (13, 9, 7)), (False, True, (13, 9, 7)),
                                               (True, True, (3, 2, 1)), (False, False, (24, 17, 16))])
def test_collapsed_bond(influence, uniform, thermal, n):
    from peridigm_amd import Context
    from peridigm_amd import quasistatic as Q
    h = 1e-3
    rng = np.random.default_rng(11)
    x, vol, nl = O.quickgrid(*n, [0, 0, 0], [k * h for k in n], 3.015 * h)
    if not uniform:
        vol = vol * rng.uniform(0.8, 1.2, size=len(vol))
    N = len(vol)
    u = 1e-3 * x[:, ::-1] + 2e-7 * rng.standard_normal(x.shape)
    a, b = N // 2, N // 2 + 1  # neighbours along x, or around a corner: bonded
    u[a] = 0.0
    u[b] = x[a] - x[b]
    out = {}
    with Context(0) as ctx:
        ctx.set_topology(nl, N)
        ctx.set_constants(x, vol, 130e9, 60e9, 3.015 * h, influence, 0.0)
        if thermal:
            ctx.set_thermal_expansion(1e-5)
            ctx.set_temperature_change(rng.uniform(0.0, 50.0, size=N))
        assert ctx.tiling()[0] > 0
        for variant in (0, 1):
            ctx.set_kernel_variant(variant)
            out[variant] = (*Q.force_and_dilatation(ctx, u), Q.residual(ctx, u)[0])
    (f0, t0, r0), (f1, t1, r1) = out[0], out[1]
    assert np.isfinite(t1).all() and np.abs(t0 - t1).max() <= 1e-11 * np.abs(t1).max()
    others = np.setdiff1d(np.arange(N), [a, b])
    for v0, v1 in ((f0, f1), (r0, r1)):
        assert np.isnan(v1[[a, b]]).all() and np.isnan(v0[[a, b]]).all()
        assert np.isfinite(v1[others]).all()
        assert np.abs(v0 - v1)[others].max() <= 1e-11 * np.abs(v1[others]).max()
