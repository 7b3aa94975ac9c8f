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
extern "C" void set_refuse(int on) { refuse = on; }
extern "C" int hipHostMalloc(void** p, size_t n, unsigned flags) {
  typedef int (*fn)(void**, size_t, unsigned);
  static fn real = (fn)dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), "hipHostMalloc");
  if (refuse && n > 4096) {
    *p = nullptr;
    real(nullptr, n, flags);
    return 2;  // hipErrorOutOfMemory
  }
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


@pytest.mark.parametrize("nx", [20, 450])  # 1,600 and 36,000 nodes
def test_calls_without_the_staging_buffer(tmp_path, nx):
    import os
    src, so, prog = tmp_path / "shim.cpp", tmp_path / "shim.so", tmp_path / "prog.py"
    src.write_text(SHIM)
    prog.write_text(textwrap.dedent(PROGRAM))
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(so), str(src), "-ldl"], check=True, timeout=60)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, str(prog), str(so), root, str(nx)], timeout=100,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0 and r.stdout.strip().endswith("same"), r.stdout[-2000:]
