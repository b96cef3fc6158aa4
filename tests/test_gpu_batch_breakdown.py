"""Conjugate gradients of the parameter batch that break down: sets whose tangent is not
positive definite (Guccione with a negative penalty) beside sets that converge.  The first
Newton update of each set is compared, through its norm, with the iterate of the same
recurrence in numpy where it breaks down.  It must not depend on the order in which a
launch's workgroups find the breakdown, so the same step also gives the same bits twice."""
import numpy as np
import pytest

from cardiomechanics_amd import materials as MT
from cardiomechanics_amd import mesh as M
from cardiomechanics_amd.context import MechanicsContext, ParameterBatch

pytestmark = pytest.mark.gpu

CONVERGED, BREAKDOWN = 1, 2
OPTS = dict(pressure_tangent=0, newton_maxit=1)
PENALTIES = (1e5, -900.0, 2e4, -1000.0)   # of four sets; C 500 Pa, bf 8, bt 4, bfs 8


def block_jacobi(A):
    D = A.tobsr((3, 3))
    n = len(D.indptr) - 1
    d = np.linalg.inv(np.array([D.data[D.indptr[r]:D.indptr[r + 1]][D.indices[D.indptr[r]:D.indptr[r + 1]] == r][0]
                                for r in range(n)]))
    return lambda r: (d.astype(r.dtype) * r.reshape(-1, 1, 3)).sum(2).ravel()


def pcg(A, pre, b, rtol, dtype=np.float64, maxit=20_000):
    """x, iterations and the end of a preconditioned conjugate gradient from zero"""
    data, b = A.data.astype(dtype), b.astype(dtype)

    def mul(v):
        return np.add.reduceat(data * v[A.indices], A.indptr[:-1])
    x, r = np.zeros_like(b), b.copy()
    z = pre(r)
    p, rz, target = z.copy(), (r * z).sum(), rtol ** 2 * (r * r).sum()
    if not rz > 0:
        return x, 0, BREAKDOWN
    for it in range(maxit):
        q = mul(p)
        pq = (p * q).sum()
        if not pq > 0:
            return x, it, BREAKDOWN
        x, r = x + rz / pq * p, r - rz / pq * q
        z = pre(r)
        if (r * r).sum() <= target:
            return x, it + 1, CONVERGED
        rz, old = (r * z).sum(), rz
        p = z + rz / old * p
    return x, maxit, 0


def first_step(mesh, sets, **opts):
    """stats and nodes of one Newton iteration of every set, the matrices and right-hand sides"""
    systems = []
    for m in sets:
        with MechanicsContext(mesh, [m], **opts) as one:
            one.set_pressures([100.0])
            x = mesh.coords.ravel()
            systems.append((one.bsr(one.tangent(x, 0.0)).tocsr(), -one.residual(x, 0.0)))
    runs = []
    for _ in range(2):
        with MechanicsContext(mesh, [sets[0]], **opts) as ctx:
            ctx.set_pressures([100.0])
            with ParameterBatch(ctx, [[m] for m in sets], spmv_lanes=8, element_variant=6) as batch:
                _, st = batch.static_step(0.0, 1.0)
                runs.append(([(s.step_norm, s.krylov_iterations, s.residual_norm, s.converged_reason) for s in st],
                             batch.nodes()))
    assert runs[0][0] == runs[1][0] and runs[0][1].tobytes() == runs[1][1].tobytes()
    return runs[0][0], systems


# 729 nodes: three workgroups of the update
@pytest.mark.parametrize("order,n", [(10, 4), (4, 8)])
def test_update_of_a_broken_down_set_is_the_iterate_before_it(order, n):
    mesh = M.cube_mesh(n, order=order)
    sets = [MT.guccione(500.0, 8.0, 4.0, 8.0, K) for K in PENALTIES]
    stats, systems = first_step(mesh, sets, preconditioner=1, **OPTS)
    for (step, its, _, _), (A, b), K in zip(stats, systems, PENALTIES):
        pre = block_jacobi(A)
        ref, want, end = pcg(A, pre, b, 0.1, np.longdouble)
        plain, _, _ = pcg(A, pre, b, 0.1)
        norm = float(np.linalg.norm(ref.astype(float)))
        lost = float(np.linalg.norm((plain - ref).astype(float))) / norm
        print(f"K {K:g}: {its} iterations (numpy {want}, end {end}), |delta| {step:.15e} (numpy {norm:.15e}, "
              f"lost in double {lost:.1e})", flush=True)
        assert end == (CONVERGED if K > 0 else BREAKDOWN) and want > 0
        assert its == want
        # another order of the same sums may lose a hundred times what numpy's loses
        assert abs(step - norm) <= (100 * lost + 1e-13) * norm
