"""The two-level preconditioner's set-up and application: one iteration of
conjugate gradients from zero gives a multiple of z = D^-1 b + P A_c^-1 P^T b,
here against the same in numpy, with A_c = P^T K P from tangent products of
the coarse functions one at a time.

A tangent product is good to 1e-12 of its largest entry (see the tiled
passes' tests), so A_c is to about that and z to cond(A_c) times it.
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _coarse_functions(x, fixed):
    """P: hat functions of the coarse grid's points times unit vectors, zero on
    prescribed DOFs (3n x nc)."""
    lo, e = x.min(0), np.ptp(x, axis=0)
    cap = max(64, min(160, len(x) // 500))
    for div in range(1, 65):
        h1 = e.max() / div
        d1 = np.maximum(2, np.ceil(e / h1 - 1e-9).astype(int) + 1)
        if d1.prod() > cap:
            break
        h, d = h1, d1
    f = (x - (lo - 0.5 * ((d - 1) * h - e))) / h
    c = np.clip(np.floor(f).astype(int), 0, d - 2)
    t = f - c
    P = np.zeros((3 * len(x), 3 * d.prod()))
    for q in range(8):
        o = np.array([q & 1, q >> 1 & 1, q >> 2 & 1])
        w = np.where(o, t, 1.0 - t).prod(1)
        g = c + o
        pt = g[:, 0] + d[0] * (g[:, 1] + d[1] * g[:, 2])
        for k in range(3):
            P[3 * np.arange(len(x)) + k, 3 * pt + k] += w
    P[fixed] = 0.0
    return P


# meshes: fewer nodes than a tile; a sheet, whose two layers of grid points
# carry the same functions (one of each pair is dropped); a coarse matrix that
# is no multiple of the inversion's blocks; tile sizes and lanes; untiled
@pytest.mark.parametrize("n,uniform,influence,model,tile,lanes,variant", [
    ((4, 3, 2), True, 0, "Elastic", 0, 4, 0), ((24, 9, 1), False, 0, "Elastic", 32, 16, 0),
    ((21, 6, 5), True, 1, "Elastic", 64, 8, 0), ((13, 9, 7), False, 2, "Elastic", 128, 4, 0),
    ((36, 10, 10), True, 0, "Elastic", 128, 4, 0), ((12, 8, 8), False, 0, "Linear LPS", 32, 16, 0),
    ((21, 6, 5), True, 2, "Linear LPS", 64, 8, 0), ((13, 9, 7), True, 0, "Elastic", 0, 4, 1)])
def test_first_iteration_is_the_two_level_correction(n, uniform, influence, model, tile, lanes, variant):
    from peridigm_amd import Context
    from peridigm_amd import quasistatic as Q
    from peridigm_amd.core import list_to_csr
    rng = np.random.default_rng(5)
    h = 1e-3
    x, vol, nl = O.quickgrid(*n, [0, 0, 0], [k * h for k in n], 3.015 * h)
    N = len(vol)
    if not uniform:
        vol = vol * rng.uniform(0.8, 1.2, size=N)
    rp, col = list_to_csr(nl, N)
    i = np.repeat(np.arange(N), np.diff(rp))
    pair = rng.random(N)[np.minimum(i, col)] + rng.random(N)[np.maximum(i, col)]
    bd = (pair % 1.0 < 0.05).astype(float)  # symmetric, a few bonds broken
    u = 1e-3 * x[:, ::-1] + 2e-7 * rng.standard_normal(x.shape)
    fixed = np.flatnonzero(np.repeat(x[:, 0] < x[:, 0].min() + 1.5 * h, 3))
    fixed = np.union1d(fixed, rng.integers(0, 3 * N, size=5))
    if n[2] == 1:  # a sheet has no stiffness out of its plane
        fixed = np.union1d(fixed, 3 * np.arange(N) + 2)
        u[:, 2] = 0.0
    b = rng.standard_normal(x.shape)
    b.ravel()[fixed] = 0.0
    with Context(0, lanes=lanes, tile_nodes=tile) as ctx:
        ctx.set_topology(nl, N)
        ctx.set_material_model(model)
        ctx.set_constants(x, vol, 130e9, 60e9, 3.015 * h, influence, 1e-2)
        ctx.upload_state(bond_damage=bd)
        Q.set_fixed(ctx, fixed)
        ctx.set_kernel_variant(variant)
        x1 = np.zeros((N, 3))
        it, rel = C.c_int(), C.c_double()
        p = lambda a: a.ctypes.data_as(C.c_void_p)
        ctx.lib.pdg_qs_solve(ctx.h, p(u), p(b), p(x1), Q.PRECOND["two_level"], 0.0, 1,
                             C.byref(it), C.byref(rel))
        assert it.value == 1
        D = Q.block_diagonal_inverse(ctx, u).reshape(N, 3, 3)
        P = _coarse_functions(x, fixed)
        KP = np.stack([Q.tangent_apply(ctx, u, P[:, j].reshape(N, 3)).ravel() for j in range(P.shape[1])], 1)
        A = P.T @ KP
        A = 0.5 * (A + A.T)
        ev, V = np.linalg.eigh(A)
        keep = ev > 1e-10 * ev[-1]
        cond = ev[-1] / ev[keep][0]
        z = np.einsum("nij,nj->ni", D, b).ravel()
        z += P @ (V[:, keep] @ ((V[:, keep].T @ (P.T @ b.ravel())) / ev[keep]))
        Kz = Q.tangent_apply(ctx, u, z.reshape(N, 3)).ravel()
    assert cond < 1e7
    ref = z * (b.ravel() @ z) / (z @ Kz)
    assert np.abs(x1.ravel() - ref).max() <= 1e-12 * cond * np.abs(ref).max()
