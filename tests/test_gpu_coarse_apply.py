"""One application of the two-level Schwarz preconditioner against numpy, entry by entry.  A GMRES
of one iteration from zero returns a multiple of M^-1 b, so its solution, normalised, is that of
M^-1 b written out in numpy (patch inverses, trilinear hats, Galerkin matrix).  Coarse matrices
of fewer and of more than 1,024 unknowns (one and two launches per solve; up to 340 and 680 grid
nodes), and indefinite matrices, for which the correction is off until the next set-up."""
import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_coarse import EDGES, background_grid

from cardiomechanics_amd import materials as MT
from cardiomechanics_amd import mesh as M
from cardiomechanics_amd.context import MechanicsContext

pytestmark = pytest.mark.gpu


def one_level(mesh, K, b):
    """sum of the vertex patches' R^T A_p^-1 R b; and the number of patches"""
    el, N = mesh.elements.astype(np.int64), mesh.n_nodes
    v = np.unique(el[:, :4])
    pairs = np.concatenate([np.stack([v, v], 1)] + [np.stack([el[:, e], el[:, 4 + k]], 1)
                                                    for k, ends in enumerate(EDGES) for e in ends])
    pairs = np.unique(pairs, axis=0)
    start = np.searchsorted(pairs[:, 0], v)
    size = np.append(start[1:], len(pairs)) - start
    keys = np.repeat(np.arange(N), np.diff(K.indptr)) * N + K.indices
    z = np.zeros((N, 3))
    for s in np.unique(size):
        nodes = pairs[start[size == s][:, None] + np.arange(s), 1]
        want = nodes[:, :, None] * N + nodes[:, None, :]
        at = np.minimum(np.searchsorted(keys, want), len(keys) - 1)
        A = np.where((keys[at] == want)[..., None, None], K.data[at], 0.0)
        A = A.transpose(0, 1, 3, 2, 4).reshape(len(nodes), 3 * s, 3 * s)
        y = np.linalg.solve(A, b.reshape(-1, 3)[nodes].reshape(len(nodes), 3 * s, 1))
        np.add.at(z, nodes, y.reshape(len(nodes), s, 3))
    return z.ravel(), len(v)


def correction(mesh, K, b, patches):
    """P A_c^-1 P^T b, the number of grid nodes and the smallest eigenvalue of A_c"""
    free = np.ones(3 * mesh.n_nodes)
    for c in range(3):
        free[c::3][(mesh.bc >> c) & 1 == 1] = 0.0
    w = background_grid(mesh.coords, mesh.elements, min(680 if patches >= 20_000 else 340, patches // 4))
    P = (sp.diags(free) @ sp.kron(w, sp.eye(3))).tocsr()
    Ac = (P.T @ (K.tocsr() @ P)).toarray()
    keep = np.diag(Ac) > 0
    P, Ac = P[:, keep], Ac[np.ix_(keep, keep)]
    return P @ np.linalg.solve(Ac, P.T @ b), w.shape[1], np.linalg.eigvalsh((Ac + Ac.T) / 2)[0]


def unit(v):
    return v / np.linalg.norm(v)


def apply_once(ctx, vals, b):
    x, st = ctx.linear_solve(vals, b, rtol=1e-30)
    assert st.iterations == 1
    return unit(x)


def newmark(ctx, mesh, vals):
    """the matrix of a 1 ms Newmark step, its constrained columns cleared as the assembly leaves them"""
    M = ctx.mass_matrix().reshape(-1, 3, 3).copy()
    for c in range(3):
        M[((mesh.bc >> c) & 1 == 1)[ctx.colind], :, c] = 0.0
    return (vals + 4e6 * M.ravel()).astype(vals.dtype)


def matrix(ctx, vals):
    K = ctx.bsr(vals.astype(np.float64))
    K.sort_indices()
    return K


ONE = dict(krylov_method=0, krylov_maxit=1)
# largest difference between two correct applications: the patch inverses' and A_c's own rounding
# (condition about 1e4), in mixed precision FP32 inverses
TOL = {0: 1e-9, 1: 1e-3}


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("case", ["cube_4", "lv_2500", "lv_100k"])
def test_application_equals_numpy(case, precision):
    mesh, mat = {"cube_4": lambda: (M.cube_mesh(4), MT.cube_guccione()),
                 "lv_2500": lambda: (M.lv_mesh(2500), MT.lv_holzapfel()),
                 "lv_100k": lambda: (M.lv_mesh(100_000), MT.lv_holzapfel())}[case]()
    with MechanicsContext(mesh, [mat], precision=precision, **ONE) as ctx:
        vals = ctx.tangent(mesh.coords.ravel(), 0.0)
        if mesh.name.startswith("lv"):
            vals = newmark(ctx, mesh, vals)
        K = matrix(ctx, vals)
        b = K @ np.random.default_rng(7).normal(size=ctx.n_dofs)
        x = apply_once(ctx, vals, b)
    one, patches = one_level(mesh, K, b)
    two, nodes, _ = correction(mesh, K, b, patches)
    err, without = np.linalg.norm(x - unit(one + two)), np.linalg.norm(x - unit(one))
    print(f"{case}: {patches} patches, {nodes} grid nodes, error {err:.1e}, without the correction {without:.1e}", flush=True)
    assert (3 * nodes > 1024) == (case == "lv_100k") and (nodes > 340) == (case == "lv_100k")
    assert err <= TOL[precision] and without > 10 * TOL[precision]


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_indefinite_coarse_matrix_switches_the_correction_off_until_the_next_set_up(precision):
    mesh = M.cube_mesh(4)
    values, rhs = {}, {}
    for K in (-900.0, 1e5):   # a negative penalty makes the tangent indefinite
        with MechanicsContext(mesh, [MT.guccione(500.0, 8.0, 4.0, 8.0, K)], precision=precision) as ctx:
            values[K] = ctx.tangent(mesh.coords.ravel(), 0.0)
    with MechanicsContext(mesh, [MT.cube_guccione()], precision=precision, **ONE) as ctx:
        for K in (-900.0, 1e5, -900.0):
            A = matrix(ctx, values[K])
            b = A @ np.random.default_rng(7).normal(size=ctx.n_dofs)
            x = apply_once(ctx, values[K], b)
            one, patches = one_level(mesh, A, b)
            two, _, least = correction(mesh, A, b, patches)
            assert (least > 0) == (K > 0)
            err = np.linalg.norm(x - unit(one + two if K > 0 else one))
            print(f"K {K:g}: smallest eigenvalue of A_c {least:.2e}, error {err:.1e}", flush=True)
            assert err <= TOL[precision]
