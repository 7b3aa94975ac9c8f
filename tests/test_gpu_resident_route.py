"""The route of explicit runs is the one their rule says: resident on small
tiled meshes, and then to its end; launched where something asks for it;
repeated, and launched from then on, once a wait has ended in vain."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _context(n, influence=0, model="Elastic", sc=5e-4, **kw):
    from peridigm_amd import Context, problems
    p = problems.plate(nx=n[0], ny=n[1], nz=n[2], notch_cells=max(2, n[0] // 4), pull=20.0)
    ctx = Context(0, **kw)
    ctx.set_topology(problems.neighbours(p), len(p["volume"]))
    ctx.set_material_model(model)
    ctx.set_constants(p["x"], p["volume"], p["K"], p["mu"], p["horizon"], influence, sc)
    ctx.set_density(p["density"])
    return ctx, p


# the meshes, models and influence functions of the bitwise comparison with
# launched runs, so that it compares two routes
@pytest.mark.parametrize("n,influence,model,sc", [
    ((4, 3, 2), 0, 0, 0.0), ((11, 3, 1), 1, 0, 5e-4), ((100, 10, 10), 0, 0, 0.0),
    ((40, 40, 4), 0, 0, 5e-4), ((40, 40, 4), 1, 0, 5e-4), ((33, 20, 4), 2, 0, 5e-4),
    ((40, 40, 4), 0, 1, 5e-4), ((64, 64, 4), 0, 0, 2e-4)])
@pytest.mark.parametrize("initial_eval", [True, False])
def test_small_meshes_run_resident(n, influence, model, sc, initial_eval):
    ctx, p = _context(n, influence, ("Elastic", "Elastic Bond Based")[model], sc)
    with ctx:
        ctx.upload_state()
        ctx.verlet_run(0, p["dt"])
        assert ctx.last_run_route() == "launched"
        ctx.verlet_run(37, p["dt"], initial_eval=initial_eval)
        assert ctx.last_run_route() == "resident"
        ctx.set_per_pass_timing(True)
        ctx.verlet_run(37, p["dt"])
        assert ctx.last_run_route() == "launched"


def test_few_steps_large_meshes_and_other_kernels_are_launched():
    ctx, p = _context((40, 40, 4))
    with ctx:
        ctx.upload_state()
        for steps, route in ((15, "launched"), (16, "resident")):
            ctx.verlet_run(steps, p["dt"])
            assert ctx.last_run_route() == route
        ctx.set_critical_stretch_function([0.0, 1.0], [5e-4, 5e-4])
        ctx.verlet_run(40, p["dt"])
        assert ctx.last_run_route() == "launched"
    for n, kw in (((80, 80, 4), {}), ((40, 40, 4), dict(variant=1)), ((40, 40, 4), dict(variant=2))):
        ctx, p = _context(n, **kw)
        with ctx:
            ctx.upload_state()
            ctx.verlet_run(40, p["dt"])
            assert ctx.last_run_route() == "launched", (n, kw)


def test_a_wait_in_vain_is_reported():
    ctx, p = _context((50, 50, 4))  # 313 tiles: none finds every word at its first look
    with ctx:
        ctx.upload_state()
        ctx.set_resident_wait(0.0)
        for route in ("repeated", "launched"):
            ctx.verlet_run(40, p["dt"])
            assert ctx.last_run_route() == route
        ctx.set_resident_wait(0.2)
        ctx.verlet_run(40, p["dt"])
        assert ctx.last_run_route() == "resident"


def test_runs_on_several_threads_are_launched():
    """A run that another accompanies shares the GPU in launches; the fields are
    those of the run alone, bit for bit."""
    import threading
    import time
    (long, p), (other, _) = _context((50, 50, 4)), _context((50, 50, 4))
    with long, other:
        for c in (long, other):
            c.upload_state()
            c.verlet_run(40, p["dt"])
            assert c.last_run_route() == "resident"
        alone = other.download_state()
        thread = threading.Thread(target=lambda: long.verlet_run(40000, p["dt"]))  # 0.3 s
        thread.start()
        time.sleep(0.05)
        other.upload_state()
        other.verlet_run(40, p["dt"])
        route, under_way = other.last_run_route(), thread.is_alive()
        together = other.download_state()
        thread.join()
        assert route == "launched" or not under_way
        for k, v in alone.items():
            assert np.array_equal(v, together[k]), k
        time.sleep(0.2)  # runs that met are remembered for a tenth of a second
        other.verlet_run(40, p["dt"])
        assert other.last_run_route() == "resident"


def test_a_run_beside_a_persistent_one_is_launched():
    """A persistent run's workgroups wait for each other without a limit, so no
    resident run takes places from it."""
    import threading
    import time
    (long, p), (other, _) = _context((50, 50, 4)), _context((50, 50, 4))
    with long, other:
        for c in (long, other):
            c.upload_state()
        other.verlet_run(40, p["dt"])
        alone = other.download_state()
        thread = threading.Thread(target=lambda: long.verlet_run_persistent(20000, p["dt"]))
        thread.start()
        time.sleep(0.05)
        other.upload_state()
        other.verlet_run(40, p["dt"])
        route, under_way = other.last_run_route(), thread.is_alive()
        together = other.download_state()
        thread.join()
        assert route == "launched" or not under_way
        for k, v in alone.items():
            assert np.array_equal(v, together[k]), k
