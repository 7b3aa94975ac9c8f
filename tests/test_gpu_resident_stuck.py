"""Resident explicit runs whose waits end in vain, at either of a step's two
waits and after any number of steps: every workgroup leaves, and the run
repeated with launches gives every field bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 4 to 313 tiles; waits from none to about as long as an exchange takes, so that
# some end at the first displacement, some at a dilatation term, some not at all
@pytest.mark.parametrize("n", [(20, 6, 1), (40, 10, 4), (50, 50, 4)])
@pytest.mark.parametrize("wait", [0.0, 2e-8, 2e-6, 4e-6, 1e-5])
def test_run_with_short_waits(n, wait):
    from peridigm_amd import Context, problems
    p = problems.plate(nx=n[0], ny=n[1], nz=n[2], notch_cells=max(2, n[0] // 4), pull=20.0)
    u0 = 2e-4 * p["x"] * np.sin(40.0 * p["x"][:, ::-1])
    v0 = np.random.default_rng(4).standard_normal(p["x"].shape)
    out = []
    with Context(0) as ctx:
        ctx.set_topology(problems.neighbours(p), len(p["volume"]))
        ctx.set_constants(p["x"], p["volume"], p["K"], p["mu"], p["horizon"], 0, 5e-4)
        ctx.set_density(p["density"])
        for timed in (False, True):
            ctx.set_per_pass_timing(timed)
            ctx.set_resident_wait(wait)
            ctx.upload_state(u=u0, v=v0)
            ctx.verlet_run(40, p["dt"])
            out.append((ctx.download_state(), ctx.near_critical_count()))
    for k, v in out[0][0].items():
        assert np.array_equal(v, out[1][0][k]), k
    assert out[0][1] == out[1][1]
