"""Explicit runs of small meshes, which keep every tile on the GPU for the whole
run, against the same runs with two launches a step (which per-pass timing
asks for): every field bit for bit, the near-critical count too."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "a", "bond_damage", "damage", "theta", "force")


def _run(ctx, p, steps, timed):
    ctx.set_per_pass_timing(timed)
    ctx.upload_state(u=p["u0"], v=p["v0"])
    ctx.verlet_run(steps[0], p["dt"])
    near = [ctx.near_critical_count()]
    first = ctx.download_state()
    ctx.verlet_run(steps[1], p["dt"], t0=steps[0] * p["dt"], initial_eval=False)
    near.append(ctx.near_critical_count())
    return first, ctx.download_state(), near


# one tile, a short last tile, 313 tiles; no damage, damage with prescribed
# displacements; the pair models and influence functions
CASES = [((4, 3, 2), 0, 0, 0.0), ((11, 3, 1), 1, 0, 5e-4), ((100, 10, 10), 0, 0, 0.0),
         ((40, 40, 4), 0, 0, 5e-4), ((40, 40, 4), 1, 0, 5e-4), ((33, 20, 4), 2, 0, 5e-4),
         ((40, 40, 4), 0, 1, 5e-4), ((64, 64, 4), 0, 0, 2e-4)]


@pytest.mark.parametrize("n,influence,model,sc", CASES)
def test_resident_run_is_bitwise_the_launched_one(n, influence, model, sc):
    from peridigm_amd import Context, problems
    p = problems.plate(nx=n[0], ny=n[1], nz=n[2], notch_cells=max(2, n[0] // 4), pull=20.0)
    nl = problems.neighbours(p)
    rng = np.random.default_rng(4)
    p["u0"] = 2e-4 * p["x"] * np.sin(40.0 * p["x"][:, ::-1]) + 1e-9 * rng.standard_normal(p["x"].shape)
    p["v0"] = rng.standard_normal(p["x"].shape)
    with Context(0) as ctx:
        ctx.set_topology(nl, len(p["volume"]))
        ctx.set_material_model(("Elastic", "Elastic Bond Based")[model])
        ctx.set_constants(p["x"], p["volume"], p["K"], p["mu"], p["horizon"], influence, sc)
        ctx.set_density(p["density"])
        if n[1] > 6:
            ctx.set_bcs(p["bcs"])
        assert ctx.tile_config() == (32, 16)
        got = _run(ctx, p, (16, 37), False)
        ref = _run(ctx, p, (16, 37), True)
    for g, r in zip(got[:2], ref[:2]):
        for k in FIELDS:
            assert np.array_equal(g[k], r[k]), k
    assert got[2] == ref[2]
    if sc > 0.0 and n[0] >= 40:
        assert 0 < ref[1]["bond_damage"].sum() < ref[1]["bond_damage"].size


@pytest.mark.parametrize("initial_eval", [True, False])
def test_run_whose_waits_end_at_once_is_repeated_with_launches(initial_eval):
    from peridigm_amd import Context, problems
    p = problems.plate(nx=40, ny=40, nz=4, notch_cells=10, pull=20.0)
    p["u0"] = 2e-4 * p["x"] * np.sin(40.0 * p["x"][:, ::-1])
    p["v0"] = np.random.default_rng(4).standard_normal(p["x"].shape)
    out = []
    with Context(0) as ctx:
        ctx.set_topology(problems.neighbours(p), len(p["volume"]))
        ctx.set_constants(p["x"], p["volume"], p["K"], p["mu"], p["horizon"], 0, 5e-4)
        ctx.set_density(p["density"])
        ctx.set_bcs(p["bcs"])
        for wait in (0.2, 0.0):
            ctx.upload_state(u=p["u0"], v=p["v0"], bond_damage=np.zeros_like(ctx.download_state()["bond_damage"]))
            if not initial_eval:
                ctx.verlet_run(0, p["dt"])
            ctx.set_resident_wait(wait)
            ctx.verlet_run(40, p["dt"], initial_eval=initial_eval)
            out.append((ctx.download_state(), ctx.near_critical_count()))
    for k in FIELDS:
        assert np.array_equal(out[0][0][k], out[1][0][k]), k
    assert out[0][1] == out[1][1] and out[0][0]["bond_damage"].sum() > 0


def test_non_finite_force_is_reported():
    from peridigm_amd import Context, problems
    from peridigm_amd._lib import PdgError
    p = problems.bar(nx=20, ny=5, nz=5)
    with Context(0) as ctx:
        ctx.set_topology(problems.neighbours(p), len(p["volume"]))
        ctx.set_constants(p["x"], p["volume"], p["K"], p["mu"], p["horizon"])
        ctx.set_density(p["density"])
        v = p["v0"].copy()
        v[7, 0] = np.inf
        ctx.upload_state(v=v)
        with pytest.raises(PdgError) as e:
            ctx.verlet_run(20, p["dt"])
        assert e.value.code == -4
