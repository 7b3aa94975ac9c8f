"""The two-level preconditioner on small jittered meshes, where coarse functions
depend on one another: it has to stay symmetric positive, so PCG converges, in no
more iterations than with block Jacobi alone and a few, to the same solution
(both residuals are 1e-8 of the right-hand side; at the condition numbers below
1e4 of these meshes the solutions agree to 1e-4)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(rng):
    h = 1e-3
    while True:
        n = rng.integers(2, 11, size=3)
        if 24 <= np.prod(n) <= 700:
            break
    g = np.stack(np.meshgrid(*[np.arange(k) for k in n], indexing="ij"), -1).reshape(-1, 3)
    return (g + rng.uniform(-0.2, 0.2, size=g.shape)) * h, h * rng.uniform(2.2, 3.1)


@pytest.mark.parametrize("model", ["Elastic", "Linear LPS"])
@pytest.mark.parametrize("tile", [0, 64])
def test_small_meshes_converge(model, tile):
    from peridigm_amd import Context
    from peridigm_amd import quasistatic as Q
    for seed in range(40):
        rng = np.random.default_rng(seed)
        x, R = _mesh(rng)
        N = len(x)
        near = np.linalg.norm(x[None] - x[:, None], axis=2) <= R
        np.fill_diagonal(near, False)
        nl = np.concatenate([np.r_[len(j), j] for j in map(np.flatnonzero, near)]).astype(np.int32)
        held = np.flatnonzero(x[:, 0] < 1.5e-3)
        fixed = (3 * held[:, None] + np.arange(3)).ravel()
        if len(held) == N:
            continue
        b = rng.standard_normal((N, 3))
        b.ravel()[fixed] = 0.0
        with Context(0, tile_nodes=tile) as ctx:
            ctx.set_topology(nl, N)
            ctx.set_material_model(model)
            ctx.set_constants(x, np.full(N, 1e-9), 130e9, 78e9, R, 0, 0.0)
            ctx.upload_state(bond_damage=None)
            Q.set_fixed(ctx, fixed)
            u = np.zeros((N, 3))
            xj, itj, _ = Q.solve(ctx, u, b, precond="block_jacobi", rel_tol=1e-8, max_iter=3000)
            xt, itt, _ = Q.solve(ctx, u, b, precond="two_level", rel_tol=1e-8, max_iter=3000)
            assert itt <= itj + 5, (seed, N, itj, itt)
            assert np.abs(xt - xj).max() <= 1e-4 * np.abs(xj).max(), (seed, N)
