"""The network's kernels at the edges of their tiles and of their groups of
neighbours (sums go four neighbours at a time, eight groups in flight): node
counts around 32 and 64, rows of 0 to 122 bonds. Against the FP64 CPU network
with the tolerances that the BF16 multiplications need there (outputs within
3e-2 of their scale, gradients within 5e-2 in norm), and the forward pass
alone bit for bit against the one before a backward pass."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,horizon", [((1, 1, 1), 1.1), ((2, 1, 1), 1.1), ((31, 1, 1), 2.1),
                                       ((32, 1, 1), 3.1), ((33, 1, 1), 3.1), ((65, 1, 1), 4.1),
                                       ((9, 8, 1), 3.015), ((13, 9, 7), 3.015)])
def test_network_edges(n, horizon):
    from peridigm_amd import Context
    from peridigm_amd import learned as Lr
    x, vol, nl = O.quickgrid(*n, [0, 0, 0], list(n), horizon)
    rp, col = O.list_to_csr(nl, len(vol))
    N = len(vol)
    rng = np.random.default_rng(N)
    with Context(0) as ctx:
        ctx.set_topology(nl, N)
        ctx.set_constants(x, vol, 130e9, 60e9, horizon, 0, 0.0)
        Lr.init(ctx, 3)
        p = (0.3 * rng.standard_normal(Lr.num_params(ctx))).astype(np.float32)
        Lr.set_params(ctx, p)
        feat = rng.standard_normal((N, 8)).astype(np.float32)
        gout = rng.standard_normal((N, 3)).astype(np.float32)
        alone, none = Lr.forward_backward(ctx, feat)
        out, dp = Lr.forward_backward(ctx, feat, gout)
        again, dp2 = Lr.forward_backward(ctx, feat, gout)
    assert none is None
    assert np.array_equal(alone, out) and np.array_equal(again, out) and np.array_equal(dp, dp2)
    deg = np.diff(rp).astype(float)
    ew = np.repeat(1.0 / np.maximum(deg, 1.0), np.diff(rp))
    p64, f64 = p.astype(np.float64), feat.astype(np.float64)
    outo, acts = O.gnn_forward(rp, col, ew, list(Lr.DIMS), p64, f64)
    dpo = O.gnn_backward(rp, col, ew, list(Lr.DIMS), p64, acts, gout.astype(np.float64))
    assert np.abs(out - outo).max() <= 3e-2 * np.abs(outo).max()
    assert np.linalg.norm(dp - dpo) <= 5e-2 * np.linalg.norm(dpo)
