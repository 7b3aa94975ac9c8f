"""Explicit runs with contact, whose contact force goes with the first pass's
launch, against the same runs with a launch of its own (which per-pass timing
asks for): every field bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "a", "bond_damage", "damage", "theta", "force")


# lanes and tile sizes; pair models, influence functions, with and without
# damage and friction; few points with contacts, and more than a workgroup
# (32) takes; a mesh of one tile
@pytest.mark.parametrize("n,tile,lanes,influence,model,sc,mu", [
    ((6, 4, 2), 0, 4, 0, 0, 0.0, 0.0), ((20, 12, 3), 32, 16, 0, 0, 5e-4, 0.3),
    ((40, 40, 4), 32, 16, 1, 0, 5e-4, 0.0), ((40, 40, 4), 64, 8, 2, 0, 5e-4, 0.3),
    ((40, 40, 4), 64, 8, 0, 1, 0.0, 0.0), ((60, 40, 4), 128, 4, 0, 0, 5e-4, 0.0),
    ((60, 40, 4), 128, 4, 1, 0, 0.0, 0.3), ((60, 40, 4), 128, 4, 0, 1, 5e-4, 0.0)])
def test_joint_contact_force_is_bitwise_the_separate_one(n, tile, lanes, influence, model, sc, mu):
    from peridigm_amd import Context, problems
    p = problems.plate(nx=n[0], ny=n[1], nz=n[2], notch_cells=max(2, n[0] // 2), pull=5.0)
    x, h = p["x"], p["horizon"] / 3.015
    rng = np.random.default_rng(3)
    u0 = 1e-6 * h * rng.standard_normal(x.shape)
    v0 = np.zeros_like(x)
    v0[:, 1] = np.where(x[:, 1] > x[:, 1].mean(), -20.0, 20.0)  # the notch closes
    # contact radius over the spacing: the notch faces touch at rest
    out = []
    with Context(0, lanes=lanes, tile_nodes=tile) as ctx:
        ctx.set_topology(problems.neighbours(p), len(x))
        ctx.set_material_model(("Elastic", "Elastic Bond Based")[model])
        ctx.set_constants(x, p["volume"], p["K"], p["mu"], p["horizon"], influence, sc)
        ctx.set_density(p["density"])
        ctx.set_contact(p["horizon"], 7, 1.05 * h, 15.0 * p["K"], mu)
        for timed in (False, True):
            ctx.set_per_pass_timing(timed)
            ctx.upload_state(u=u0, v=v0)
            force = []
            for steps, t0, initial in ((0, 0, True), (17, 0, False), (40, 17, False)):
                ctx.verlet_run(steps, p["dt"], t0=t0 * p["dt"], initial_eval=initial)
                force.append(ctx.contact_force_density())
            out.append((ctx.download_state(), force))
    for k in FIELDS:
        assert np.array_equal(out[0][0][k], out[1][0][k]), k
    for a, b in zip(out[0][1], out[1][1]):
        assert np.array_equal(a, b)
    points = int(np.any(out[0][1][0] != 0.0, axis=1).sum())  # at rest
    assert points > (32 if n[0] >= 40 else 0)
