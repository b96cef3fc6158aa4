"""A coarse matrix that does not fit the device: the context and the parameter batch fall back to
the patches alone, as they did without a coarse grid.  The allocation of the coarse matrix is
made to fail by a hipMalloc of the test's own, in a process of its own, that refuses one
size and passes every other on to the runtime."""
import os
import subprocess
import sys

import numpy as np
import pytest

from test_gpu_coarse import background_grid

from cardiomechanics_amd import mesh as M

pytestmark = pytest.mark.gpu

REFUSE = r"""
#include <dlfcn.h>
#include <cstddef>
static size_t refused;
static int count;
extern "C" void refuse(size_t n) { refused = n; }
extern "C" int refusals() { return count; }
extern "C" int hipMalloc(void** p, size_t n) {
    static auto f = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so", RTLD_NOW | RTLD_LOCAL), "hipMalloc");
    if (n == refused) return ++count, 2;   // hipErrorOutOfMemory
    return f(p, n);
}
"""

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # found before the runtime's
shim.refuse.argtypes = [ctypes.c_size_t]
sys.path[:0] = sys.argv[2:4]
import numpy as np
from test_gpu_batch_breakdown import pcg, schwarz
from test_gpu_coarse import gmres_count
from cardiomechanics_amd import materials as MT
from cardiomechanics_amd import mesh as M
from cardiomechanics_amd.context import MechanicsContext, ParameterBatch

bytes_of_one = int(sys.argv[4])
mesh, mat = M.cube_mesh(4), MT.guccione(500.0, 8.0, 4.0, 8.0, 1e5)
b = np.random.default_rng(3).normal(size=3 * mesh.n_nodes)


def count():
    with MechanicsContext(mesh, [mat], krylov_method=0, krylov_restart=400, krylov_maxit=400) as ctx:
        vals = ctx.tangent(mesh.coords.ravel(), 0.0)
        K = ctx.bsr(vals).tocsr()
        x, st = ctx.linear_solve(vals, K @ b, rtol=1e-6)
        return K, st.iterations


def batch_count(sets):
    opts = dict(pressure_tangent=0, newton_maxit=1)
    with MechanicsContext(mesh, [mat], **opts) as ctx:
        ctx.set_pressures([100.0])
        with ParameterBatch(ctx, [[mat]] * sets, spmv_lanes=8, element_variant=6) as batch:
            _, st = batch.static_step(0.0, 1.0)
            assert batch.info()["preconditioner"] == "vertex-patch Schwarz"
            x = mesh.coords.ravel()
            return ctx.bsr(ctx.tangent(x, 0.0)).tocsr(), -ctx.residual(x, 0.0), [s.krylov_iterations for s in st]


K, with_grid = count()
shim.refuse(bytes_of_one)
K, without = count()
assert shim.refusals() == 1, shim.refusals()
one, two, _ = schwarz(mesh, K)
want = [gmres_count(K, p, K @ b, 1e-6) for p in (two, one)]
print("context: GMRES", with_grid, without, "numpy", want, flush=True)
assert abs(with_grid - want[0]) <= 1 and abs(without - want[1]) <= 1 and want[1] > want[0] + 2
shim.refuse(0)
A, f, with_grid = batch_count(3)
shim.refuse(3 * bytes_of_one)
A, f, without = batch_count(3)
assert shim.refusals() == 2, shim.refusals()
want = [pcg(A, p, f, 0.1)[1] for p in (two, one)]
print("batch: CG", with_grid, without, "numpy", want, flush=True)
assert with_grid == [want[0]] * 3 and without == [want[1]] * 3 and want[1] > want[0]
"""


def test_refused_coarse_matrix_leaves_the_patches(tmp_path):
    src, shim = tmp_path / "refuse.cpp", tmp_path / "librefuse.so"
    src.write_text(REFUSE)
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", str(src), "-ldl", "-o", str(shim)])
    mesh = M.cube_mesh(4)
    vertices = len(np.unique(mesh.elements[:, :4]))
    nodes = background_grid(mesh.coords, mesh.elements, min(340, vertices // 4)).shape[1]
    ld = (3 * nodes + 31) // 32 * 32
    here = os.path.dirname(os.path.abspath(__file__))
    out = subprocess.run([sys.executable, "-c", CHILD, str(shim), here, os.path.dirname(here), str(8 * ld * ld)],
                         capture_output=True, text=True, timeout=110)
    print(out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
