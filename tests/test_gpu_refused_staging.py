"""A system that refuses the pinned staging buffer: every call then copies from
and to the caller's memory, with the same results. In a process of its own,
where hipHostMalloc is replaced by one that refuses buffers above a page, after
an invalid call that leaves the error which a refusal leaves behind."""
import subprocess
import sys
import textwrap

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static int refuse;
static size_t pinned;
extern "C" long long pinned_bytes() { return (long long)pinned; }
extern "C" void set_refuse(int on) { refuse = on; }
extern "C" int hipHostMalloc(void** p, size_t n, unsigned flags) {
  typedef int (*fn)(void**, size_t, unsigned);
  static fn real = (fn)dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), "hipHostMalloc");
  if (refuse && n > 4096) {
    *p = nullptr;
    real(nullptr, n, flags);
    return 2;  // hipErrorOutOfMemory
  }
  pinned += n;
  return real(p, n, flags);
}
"""

PROGRAM = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np
from peridigm_amd import Context, learned, problems
from peridigm_amd import quasistatic as Q
p = problems.plate(nx=int(sys.argv[3]), ny=20, nz=4, notch_cells=5, pull=20.0)
nl = problems.neighbours(p)
x, N = p["x"], len(p["volume"])
rng = np.random.default_rng(1)
u = 1e-4 * x[:, ::-1]
v = rng.standard_normal(x.shape)
def calls():
    out = []
    with Context(0) as c:
        c.set_topology(nl, N)
        c.set_constants(x, p["volume"], p["K"], p["mu"], p["horizon"], 0, 5e-4)
        c.set_density(p["density"])
        bd, dmg, near = c.compute_damage(x + 20 * u)
        out += [bd, dmg, *c.compute_force(x + u), *c.compute_force(x + u, bd)]
        c.upload_state(u=u, v=v, bond_damage=bd)
        c.verlet_run(20, 1e-9)
        out += list(c.download_state().values())
        out += [Q.residual(c, u)[0], Q.tangent_apply(c, u, v), *Q.force_and_dilatation(c, u)]
        learned.init(c, 1)
        out.append(learned.forward_backward(c, np.float32(rng.standard_normal((N, 8)) * 0 + 1))[0])
    return out
ref = calls()
shim.set_refuse(1)
got = calls()
assert len(ref) == len(got)
for k, (a, b) in enumerate(zip(ref, got)):
    assert np.array_equal(a, b), k
print("same", flush=True)
"""


LARGE = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
shim.pinned_bytes.restype = ctypes.c_longlong
sys.path.insert(0, sys.argv[2])
import numpy as np
from peridigm_amd import Context
n = int(sys.argv[3])
x = np.zeros((n, 3))
x[:, 0] = np.arange(n)
i = np.arange(n, dtype=np.int32)
nl = np.empty(3 * n - 2, np.int32)
nl[:2], nl[-2:] = (1, 1), (1, n - 2)
nl[2:-2].reshape(-1, 3)[:] = np.stack([np.full(n - 2, 2, np.int32), i[:-2], i[2:]], axis=1)
with Context(0) as c:
    c.set_topology(nl, n)
    c.set_constants(x, np.ones(n), 130e9, 60e9, 1.1, 0, 1e-2)
    ahead = shim.pinned_bytes()
    assert ahead <= 128 << 20, ahead
    assert (ahead > 100 * n) == (112 * n + 384 <= 128 << 20), ahead
    c.set_density(7800.0)
    v = np.random.default_rng(1).standard_normal(x.shape)
    c.upload_state(v=v)
    out = np.zeros((n, 3))
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    c.check(c.lib.pdg_state_download(c.h, None, p(out), None, None, None, None, None))
    assert np.array_equal(out, v)
    # what the download needed: its one field
    assert shim.pinned_bytes() - ahead <= 24 * n + 4096, shim.pinned_bytes()
print("same", flush=True)
"""


def _run(tmp_path, program, *args):
    import os
    src, so, prog = tmp_path / "shim.cpp", tmp_path / "shim.so", tmp_path / "prog.py"
    src.write_text(SHIM)
    prog.write_text(textwrap.dedent(program))
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(so), str(src), "-ldl"], check=True, timeout=60)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, str(prog), str(so), root, *map(str, args)], timeout=100,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0 and r.stdout.strip().endswith("same"), r.stdout[-2000:]


@pytest.mark.parametrize("nx", [20, 450])  # 1,600 and 36,000 nodes
def test_calls_without_the_staging_buffer(tmp_path, nx):
    _run(tmp_path, PROGRAM, nx)


@pytest.mark.parametrize("n", [100000, 1300000])
def test_set_up_pins_a_bounded_buffer(tmp_path, n):
    """Set-up pins a whole state's buffer up to 128 MB; larger contexts pin what
    their calls need."""
    _run(tmp_path, LARGE, n)
