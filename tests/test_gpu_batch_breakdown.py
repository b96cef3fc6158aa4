"""Conjugate gradients of the parameter batch that break down: sets whose tangent is not
positive definite (Guccione with a negative penalty) beside sets that converge.  The first
Newton update of each set is compared, through its norm, with the iterate of the same
recurrence in numpy where it breaks down.  It must not depend on the order in which a
launch's workgroups find the breakdown, so the same step also gives the same bits twice."""
import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_coarse import background_grid, patches

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


def schwarz(mesh, A):
    """the vertex-patch preconditioner without and with the coarse correction; the smallest eigenvalue of
    the coarse matrix"""
    inv = []
    for nodes in patches(mesh.elements, np.unique(mesh.elements[:, :4])):
        d = (3 * nodes[:, None] + np.arange(3)).ravel()
        inv.append((d, np.linalg.inv(A[d][:, d].toarray())))
    free = np.ones(3 * mesh.n_nodes)
    for c in range(3):
        free[c::3][(mesh.bc >> c) & 1 == 1] = 0.0
    P = sp.diags(free) @ sp.kron(background_grid(mesh.coords, mesh.elements, min(340, len(inv) // 4)), sp.eye(3)).tocsr()
    Ac = (P.T @ A @ P).toarray()
    keep = np.diag(Ac) > 0
    P, Ac = P[:, keep], Ac[np.ix_(keep, keep)]
    Ai = np.linalg.inv(Ac)

    def one(r):
        z = np.zeros_like(r)
        for d, Ap in inv:
            z[d] += Ap @ r[d]
        return z
    return one, lambda r: one(r) + P @ (Ai @ (P.T @ r)), np.linalg.eigvalsh((Ac + Ac.T) / 2)[0]


def test_second_solve_without_the_correction_only_where_the_first_had_it():
    """Penalties for which the tangent is indefinite and the coarse matrix still positive (the
    correction is on, the set is solved again without it) or not (it is off from the start)."""
    mesh = M.cube_mesh(4)
    penalties = (1e5, -815.0, -870.0)
    sets = [MT.guccione(500.0, 8.0, 4.0, 8.0, K) for K in penalties]
    stats, systems = first_step(mesh, sets, **OPTS)
    for (step, its, _, _), (A, b), K in zip(stats, systems, penalties):
        one, two, least = schwarz(mesh, A)
        x, want, end = pcg(A, two if least > 0 else one, b, 0.1)
        if K < 0:
            assert end == BREAKDOWN and (least > 0) == (K == -815.0)
            if least > 0:
                x, more, end = pcg(A, one, b, 0.1)
                assert end == BREAKDOWN and more > want > 0
                want += more
        print(f"K {K:g}: {its} iterations (numpy {want}), |delta| {step:.12e} (numpy {np.linalg.norm(x):.12e})", flush=True)
        assert its == want
        # iterates of at most nine iterations; a converged one is known to the forcing tolerance
        assert abs(step - np.linalg.norm(x)) <= (1e-8 if K < 0 else 1e-2) * np.linalg.norm(x)
