"""The Schwarz preconditioner with its coarse-grid correction, pinned through GMRES: the
iterations that cmg_linear_solve needs equal those of a numpy GMRES with the same
preconditioner written out in numpy (patch inverses, trilinear hats of the background
grid, Galerkin matrix), to one iteration in FP64.  A wrong partial sum, grid neighbour or
pivot changes the preconditioner and with it the count."""
import numpy as np
import pytest
import scipy.sparse as sp
from scipy.spatial import ConvexHull

from cardiomechanics_amd import materials as MT
from cardiomechanics_amd import mesh as M
from cardiomechanics_amd.context import MechanicsContext

pytestmark = pytest.mark.gpu

EDGES = ((0, 1), (1, 2), (0, 2), (0, 3), (1, 3), (2, 3))


def patches(el, vertices):
    p = {int(v): set() for v in vertices}
    for k, (i, j) in enumerate(EDGES):
        for a, b, m in zip(el[:, i], el[:, j], el[:, 4 + k]):
            p[int(a)].add(int(m))
            p[int(b)].add(int(m))
    return [np.array([v] + sorted(p[v])) for v in p]


def background_grid(X, el, target):
    """weights [N, grid nodes] of the finest grid with at most `target` nodes next to the mesh"""
    lo, hi = X.min(0), X.max(0)
    L = hi - lo
    ext = (X[el].max(1) - X[el].min(1)).max(0)

    def lay(k):
        n = np.array([max(1, min(int(np.ceil(L[d] / (L.max() / k) - 1e-9)), int(np.floor(L[d] / ext[d] + 1e-9))))
                      for d in range(3)])
        u = (X - lo) / L * n
        q = np.clip(np.floor(u).astype(int), 0, n - 1)
        if (q[el].max(1) - q[el].min(1)).max() > 1:
            return None
        f = np.clip(u - q, 0, 1)
        ids, w = [], []
        for a in range(8):
            o = np.array([a & 1, (a >> 1) & 1, a >> 2])
            c = q + o
            ids.append((c[:, 2] * (n[1] + 1) + c[:, 1]) * (n[0] + 1) + c[:, 0])
            w.append(np.prod(np.where(o == 1, f, 1 - f), axis=1))
        return np.stack(ids, 1), np.stack(w, 1)
    best, k = None, 1
    while True:
        g = lay(k)
        if g is None or len(np.unique(g[0])) > target:
            break
        best, k = g, k + 1
        if k > 40:
            break
    ids, w = best
    u, inv = np.unique(ids, return_inverse=True)
    return sp.csr_matrix((w.ravel(), (np.repeat(np.arange(len(X)), 8), inv.ravel())), shape=(len(X), len(u)))


def preconditioner(mesh, K):
    X, el = mesh.coords, mesh.elements
    ps = patches(el, np.unique(el[:, :4]))
    inverses = []
    for nodes in ps:
        d = (3 * nodes[:, None] + np.arange(3)).ravel()
        inverses.append((d, np.linalg.inv(K[d][:, d].toarray())))
    free = np.ones(3 * len(X))
    for c in range(3):
        free[c::3][(mesh.bc >> c) & 1 == 1] = 0.0
    if len(ps) // 4 < 8:   # too few patches for a grid
        def apply(r):
            z = np.zeros_like(r)
            for d, Ap in inverses:
                z[d] += Ap @ r[d]
            return z
        return apply, 0
    P = sp.diags(free) @ sp.kron(background_grid(X, el, min(340, len(ps) // 4)), sp.eye(3)).tocsr()
    Ac = (P.T @ K @ P).toarray()
    keep = np.diag(Ac) > 0
    P, Ai = P[:, keep], np.linalg.pinv(Ac[np.ix_(keep, keep)], rcond=1e-13)

    def apply(r):
        z = P @ (Ai @ (P.T @ r))
        for d, Ap in inverses:
            z[d] += Ap @ r[d]
        return z
    return apply, int(keep.sum())


def gmres_count(K, pre, b, rtol, m=400):
    V, H = [b / np.linalg.norm(b)], np.zeros((m + 1, m))
    for j in range(m):
        w = K @ pre(V[j])
        for _ in range(2):
            for i in range(j + 1):
                h = V[i] @ w
                H[i, j] += h
                w = w - h * V[i]
        H[j + 1, j] = np.linalg.norm(w)
        V.append(w / H[j + 1, j])
        e = np.zeros(j + 2)
        e[0] = 1.0
        y, *_ = np.linalg.lstsq(H[: j + 2, : j + 1], e, rcond=None)
        if np.linalg.norm(H[: j + 2, : j + 1] @ y - e) <= rtol:
            return j + 1
    return m


def star(points):
    """tetrahedra between the origin and the hull of `points` points on a sphere: the origin's
    patch has 3 (points + 1) components"""
    k = np.arange(points) + 0.5
    z, phi = 1 - 2 * k / points, np.pi * (1 + 5 ** 0.5) * k
    v = 0.01 * np.stack([np.sqrt(1 - z * z) * np.cos(phi), np.sqrt(1 - z * z) * np.sin(phi), z], 1)
    tets = np.concatenate([ConvexHull(v).simplices, np.full((2 * points - 4, 1), points)], 1)
    X = np.concatenate([v, np.zeros((1, 3))])
    coords, el, _ = M.t4_to_t10(X, M.orient_t4(X, tets))
    E = len(el)
    return M.Mesh(coords=coords, elements=el.astype(np.int32), bases=np.tile(np.eye(3), (E, 5, 1, 1)),
                  bc=np.zeros(len(coords), np.uint8), material=np.zeros(E, np.int32), activation=np.zeros(E),
                  name=f"lv-like star {points}")


MESHES = {   # grid nodes: 8 (one padded panel), 27, a ventricle with constrained base, two panels and more
    "cube3": lambda: (M.cube_mesh(3), MT.cube_guccione()),
    "cube4": lambda: (M.cube_mesh(4), MT.cube_guccione()),
    "cube5": lambda: (M.cube_mesh(5), MT.cube_guccione()),
    "lv_900": lambda: (M.lv_mesh(900), MT.lv_holzapfel()),
    "lv_2500": lambda: (M.lv_mesh(2500), MT.lv_holzapfel()),
    # largest patch 24 to 72 components, the most that patches may have: the register inversion ends its
    # classes at 24, 30, ..
    # 60, and an application's lanes at 64
    **{f"star_{n}": (lambda n=n: (star(n), MT.lv_holzapfel()))
       for n in (7, 8, 9, 11, 12, 13, 15, 16, 17, 18, 19, 20, 21, 23)},
}


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("case", list(MESHES))
def test_gmres_needs_the_iterations_of_the_numpy_preconditioner(case, precision):
    mesh, mat = MESHES[case]()
    length = np.ptp(mesh.coords, axis=0).max()
    x = (mesh.coords + M.smooth_displacement(mesh.coords, length, 1e-3, 5)).ravel()
    rng = np.random.default_rng(7)
    rtol = 1e-6 if precision == 0 else 1e-4
    with MechanicsContext(mesh, [mat], krylov_method=0, krylov_restart=400, krylov_maxit=400,
                          precision=precision) as ctx:
        vals = ctx.tangent(x, 0.0)
        if mesh.name.startswith("lv"):   # the matrix of a 1 ms Newmark step
            vals = (vals + 4e6 * ctx.mass_matrix()).astype(vals.dtype)
        K = ctx.bsr(vals.astype(np.float64)).tocsr()
        b = K @ (rng.normal(size=ctx.n_dofs))
        _, st = ctx.linear_solve(vals, b, rtol=rtol)
    pre, dim = preconditioner(mesh, K)
    want = gmres_count(K, pre, b, rtol)
    print(f"{case} precision {precision}: {dim} coarse DOFs, GMRES {st.iterations}, numpy {want}", flush=True)
    assert st.converged
    # mixed: the patch inverses are rounded to FP32
    assert abs(st.iterations - want) <= (1 if precision == 0 else 2)
