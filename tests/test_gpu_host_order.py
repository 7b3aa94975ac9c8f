"""Node vectors on both sides of the size from which kernels, not the host,
reorder them (32,768 nodes): round trips are exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1, 1, 1), (32, 32, 32), (32769, 1, 1), (33, 32, 32)])
def test_vectors_round_trip(n):
    from peridigm_amd import Context
    from peridigm_amd.discretization import radius_search
    x = np.stack(np.meshgrid(*[np.arange(k, dtype=float) for k in n], indexing="ij"), -1).reshape(-1, 3)
    N = len(x)
    rng = np.random.default_rng(N)
    v, a = rng.standard_normal((2, N, 3))
    u = np.ldexp(rng.integers(-1000, 1000, size=(N, 3)).astype(float), -20)  # exact in any unit
    with Context(0) as ctx:
        ctx.set_topology(radius_search(x, 1.1), N)
        ctx.set_constants(x, np.ones(N), 130e9, 60e9, 1.1, 0, 0.0)
        ctx.set_density(7800.0)
        ctx.upload_state(u=u, v=v, a=a)
        st = ctx.download_state()
        theta, f = ctx.compute_force(x + u)
        ctx.upload_state(u=u)
        ctx.verlet_run(0, 1e-9)
        run = ctx.download_state()
    for k, ref in (("u", u), ("v", v), ("a", a)):
        assert np.array_equal(st[k], ref), k
    # x + u and its difference with x are exact here, so the same displacement
    assert np.array_equal(theta, run["theta"]) and np.array_equal(f, run["force"])
