"""Performance cases of the framework: what a program that uses it has it do, through its
public entry points, from the smallest calls to the largest.

The kinds of work:

    residual   element residuals + surface pressure, summed per node (cmg_residual_device):
               the line search and convergence check of a solver that keeps its vectors on
               the GPU
    assemble   residual and tangent in the block pattern (cmg_residual_tangent_device): one
               Newton assembly
    static     one quasi-static load step (static_step), state restored before, read after
    newmark    one Newmark step (newmark_step), state restored before, read after
    batch      one load step of several parameter sets on one mesh (ParameterBatch)
    forward    inference of the learned warm start (WarmStartNet.forward)
    train      loss, gradient and Adam update of the learned warm start

Meshes and materials are those of the repository's configurations and benchmark: the unit
cube (Guccione, clamped at x = 0, pressure on x = 1) and the truncated-ellipsoid left
ventricle (Holzapfel-Ogden with active tension, or Guccione for parameter fits).
"""
import functools
import math

import numpy as np
import torch

from cardiomechanics_amd import materials as MT
from cardiomechanics_amd import mesh as M
from cardiomechanics_amd.context import MechanicsContext, ParameterBatch
from cardiomechanics_amd.hip import DeviceArray
from cardiomechanics_amd.warmstart import WarmStartNet

T_EVAL = 0.12        # time of the element evaluations: inside the twitch
DT = 1e-3            # Newmark step
# Newton tolerances: the benchmark's for the beat and the sweep, the cube configuration's for static steps
BEAT_TOL = dict(newton_atol=1e-12, newton_rtol=1e-12, newton_stol=1e-14)
SWEEP_TOL = dict(newton_atol=1e-12, newton_rtol=1e-10, newton_stol=1e-14, krylov_maxit=20000, newton_maxit=100)
CUBE_TOL = dict(newton_atol=1e-10, newton_rtol=1e-10, newton_stol=1e-10, krylov_maxit=20000)


def _elem(kind, name=None, **kw):
    c = dict(kind=kind, mesh="lv", size=200_000, order=10, law="holzapfel", tension="sinus", precision="fp64")
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: the 1,296-element cube, where launches and the status read are what counts
        _elem("residual", "residual_cube_1296", mesh="cube", size=6, law="guccione", tension="none"),
        # the residual of the benchmark's ventricle: line search, convergence check, learned-guess check
        _elem("residual", "residual_lv_200k"),
        # linear tetrahedra, the other element type
        _elem("assemble", "assemble_cube_t4_24k", mesh="cube", size=16, order=4, law="guccione", tension="none"),
        # an ordinary ventricle (the size of the parameter fits) in mixed precision, stretch-dependent tension
        _elem("assemble", "assemble_lv_50k_mixed", size=50_000, tension="tanh", precision="mixed"),
        # one Newton assembly of the benchmark
        _elem("assemble", "assemble_lv_200k"),
        # a load step of the cube configuration: many short launches
        _elem("static", "static_cube_1296", mesh="cube", size=6, law="guccione", tension="none"),
        # a beat step of a coarse ventricle
        _elem("newmark", "newmark_lv_20k", size=20_000),
        # the benchmark's beat step, in both precisions
        _elem("newmark", "newmark_lv_200k"),
        _elem("newmark", "newmark_lv_200k_mixed", precision="mixed"),
        # a load step of a passive-parameter fit, all sets at once
        _elem("batch", "batch_lv_5k_8_sets", size=5_000, law="guccione", tension="none", sets=8),
        # the warm start of the benchmark's ventricle: bfloat16 inference over all nodes, and a training step
        dict(name="forward_bf16_291k", kind="forward", rows=290_927, bf16=True),
        dict(name="train_31k", kind="train", rows=31_000),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["residual", "assemble", "assemble", "static", "newmark", "newmark", "batch", "forward", "train"])
    if kind == "forward":
        return dict(kind=kind, rows=log_int(500, 290_927), bf16=rng.random() < 0.5)
    if kind == "train":
        return dict(kind=kind, rows=log_int(500, 31_000))
    precision = rng.choice(["fp64", "mixed"])
    if kind == "static":
        return _elem(kind, mesh="cube", size=rng.randint(2, 6), order=rng.choice([10, 10, 4]), law="guccione",
                     tension="none", precision=precision, load=rng.randint(50, 250))
    if kind == "newmark":
        return _elem(kind, size=log_int(1_500, 150_000), precision=precision)
    if kind == "batch":
        return _elem(kind, size=log_int(800, 5_000), law="guccione", tension="none", sets=rng.randint(2, 8),
                     precision=precision)
    if rng.random() < 0.35:
        order = rng.choice([10, 4])
        return _elem(kind, mesh="cube", size=rng.randint(3, 22 if order == 4 else 14), order=order, law="guccione",
                     tension=rng.choice(["none", "tanh"]), precision=precision, load=rng.randint(500, 3000))
    return _elem(kind, size=log_int(1_500, 200_000), order=rng.choice([10, 10, 4]),
                 law=rng.choice(["holzapfel", "guccione"]), tension=rng.choice(["none", "sinus", "tanh", "land17"]),
                 precision=precision)


# --------------------------------------------------------------------------- inputs

@functools.lru_cache(maxsize=8)
def _mesh(kind, size, order):
    return M.cube_mesh(size, order=order) if kind == "cube" else M.lv_mesh(size, order=order)


def _material(case, tension_scale=1.0):
    m = MT.lv_holzapfel() if case["law"] == "holzapfel" else MT.cube_guccione()
    sinus = MT.lv_holzapfel()
    if case["tension"] == "sinus":
        m.tension_max, m.tension_fn, m.fn = sinus.tension_max * tension_scale, sinus.tension_fn, list(sinus.fn)
    elif case["tension"] == "tanh":
        MT.with_tanh(m, PeakTension=60.0)
    elif case["tension"] == "land17":
        MT.with_land17(m)
    else:
        m.tension_fn, m.tension_max = MT.FN_NONE, 0.0
    return m


def _problem(case, seed):
    """mesh, material, pressure and coordinates of a case's inputs, from the seed alone"""
    base = _mesh(case["mesh"], case["size"], case["order"])
    rng = np.random.default_rng(seed)
    tension_scale, shift, load = rng.uniform(0.85, 1.15), rng.uniform(-2e-3, 0.0), rng.uniform(0.85, 1.15)
    mesh = M.Mesh(coords=base.coords, elements=base.elements, bases=base.bases, bc=base.bc, material=base.material,
                  activation=np.maximum(base.activation + shift, 0.0), surfaces=base.surfaces,
                  surface_id=base.surface_id, name=base.name)
    p = dict(mesh=mesh, material=_material(case, tension_scale))
    kind = case["kind"]
    if kind in ("residual", "assemble"):
        length = np.ptp(base.coords, axis=0).max()
        p["x"] = base.coords + M.smooth_displacement(base.coords, length, 0.02, seed)
        p["pressure"], p["time"] = case.get("load", 2000.0 if case["mesh"] == "cube" else -4000.0) * load, T_EVAL
    elif kind == "static":
        p["pressure"], p["time"], p["dt"] = case.get("load", 200.0) * load, 0.1, 0.1
    elif kind == "newmark":
        p["pressure"], p["time"], p["dt"] = -16000.0 * load * math.sin(math.pi * DT / 0.8) ** 2, DT, DT
    else:
        p["pressure"], p["time"], p["dt"] = -100.0 * load, 0.05, 0.05
        p["sets"] = MT.guccione_sweep(case["sets"], seed=seed)
    return p


def _net_inputs(case, seed):
    """features and targets with the scaled values of a beat: increments, pressure rate, phase"""
    g = torch.Generator().manual_seed(seed)
    X = torch.randn(case["rows"], 8, generator=g)
    X[:, 6] = 0.3 * X[0, 6]
    X[:, 7] = torch.rand(case["rows"], generator=g) * 2.0 - 1.0
    T = 0.8 * X[:, 0:3] + 0.1 * torch.sin(X[:, 3:6]) + 0.01 * torch.randn(case["rows"], 3, generator=g)
    w = []
    for fan_in, fan_out in ((8, 128), (128, 128), (128, 3)):
        a = math.sqrt(6.0 / (fan_in + fan_out))
        w += [(torch.rand(fan_in * fan_out, generator=g) * 2.0 - 1.0) * a,
              0.05 * torch.randn(fan_out, generator=g)]
    return X.numpy(), T.numpy(), torch.cat(w).numpy()


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("forward", "train"):
        X, T, w = _net_inputs(case, seed)
        ctx = MechanicsContext(_mesh("cube", 1, 10), [MT.cube_guccione()])
        net = WarmStartNet(ctx, seed=seed)
        net.set_weights(w)
        return dict(kind=kind, ctx=ctx, net=net, rows=case["rows"], bf16=case.get("bf16", False), X=DeviceArray(X),
                    T=DeviceArray(T), Y=torch.zeros(case["rows"], 3, device="cuda"))
    p = _problem(case, seed)
    mixed = dict(precision=1 if case["precision"] == "mixed" else 0)
    state = dict(kind=kind, time=p["time"], dt=p.get("dt"), pressure=[p["pressure"]])
    if kind in ("residual", "assemble"):
        ctx = MechanicsContext(p["mesh"], [p["material"]], **mixed)
        ctx.set_pressures(state["pressure"])
        state["x"] = torch.from_numpy(np.ascontiguousarray(p["x"].ravel())).cuda()
        state["f"] = torch.zeros(ctx.n_dofs, dtype=torch.float64, device="cuda")
        if kind == "assemble":
            state["values"] = torch.zeros(ctx.nnzb * 9, device="cuda",
                                          dtype=torch.float32 if ctx.fp32 else torch.float64)
        torch.cuda.synchronize()
    else:
        tol = dict(static=CUBE_TOL, newmark=BEAT_TOL, batch=SWEEP_TOL)[kind]
        first = p["sets"][0] if kind == "batch" else p["material"]
        ctx = MechanicsContext(p["mesh"], [first], **mixed, **tol)
        state["nodes"] = np.ascontiguousarray(p["mesh"].coords.ravel())
        state["zero"] = np.zeros(ctx.n_dofs)
        if kind == "batch":
            state["batch"] = ParameterBatch(ctx, [[m] for m in p["sets"]])
    state["ctx"] = ctx
    return state


def _ok(rc, what):
    if rc != 2:
        raise RuntimeError(f"{what} returned {rc}")


def run(s):
    ctx, kind = s["ctx"], s["kind"]
    if kind == "residual":
        _ok(ctx.L.cmg_residual_device(ctx.h, s["x"].data_ptr(), s["time"], 1, s["f"].data_ptr()), "residual")
        return s["f"]
    if kind == "assemble":
        _ok(ctx.L.cmg_residual_tangent_device(ctx.h, s["x"].data_ptr(), s["time"], 1, s["f"].data_ptr(),
                                              s["values"].data_ptr()), "residual + tangent")
        return s["f"], s["values"]
    if kind == "static":
        ctx.set_state(nodes=s["nodes"])
        ctx.set_pressures(s["pressure"])
        rc, _ = ctx.static_step(s["time"], s["dt"])
        _ok(rc, "static step")
        return ctx.get_state()["increment"]
    if kind == "newmark":
        ctx.set_state(s["nodes"], s["zero"], s["zero"])
        ctx.set_pressures(s["pressure"])
        rc, _ = ctx.newmark_step(s["time"], s["dt"])
        _ok(rc, "Newmark step")
        out = ctx.get_state()
        return out["increment"], out["velocity"], out["acceleration"]
    if kind == "batch":
        s["batch"].set_nodes(s["nodes"])
        ctx.set_pressures(s["pressure"])
        rc, _ = s["batch"].static_step(s["time"], s["dt"])
        _ok(rc, "batched step")
        return s["batch"].nodes() - s["nodes"]
    if kind == "forward":
        ctx._check(ctx.L.cmg_mlp_forward(s["net"].h, s["X"].ptr, s["rows"], int(s["bf16"]), s["Y"].data_ptr()),
                   "cmg_mlp_forward")
        return s["Y"]
    loss, grad = s["net"].loss_grad(s["X"], s["T"], s["rows"], want_grad=True)
    s["net"].adam_step(1e-3)
    return loss, grad, s["net"].weights()


# --------------------------------------------------------------------------- work and tolerance

def work(case):
    """One pass: every input once, every output once.  Element inputs: connectivity, fibre frames,
    material index, activation time; node inputs: reference and current coordinates.  A step
    counts one residual, one tangent and its state in and out; what its iterations read again
    is the method's, not the path's.  Blocks per node of the pattern: 27.3 (T10), 14 (T4)."""
    if case["kind"] in ("forward", "train"):
        rows, nw = case["rows"], 8 * 128 + 128 * 128 + 128 * 3
        if case["kind"] == "forward":
            return dict(bytes=44 * rows + 4 * nw, flops=2 * nw * rows)
        return dict(bytes=44 * rows + 24 * nw, flops=6 * nw * rows - 2 * 8 * 128 * rows)
    mesh = _mesh(case["mesh"], case["size"], case["order"])
    t10 = case["order"] == 10
    E, N = mesh.n_elements, mesh.n_nodes
    inputs = E * ((40 + 288 if t10 else 16 + 72) + 12) + 48 * N
    res = 3_160 if t10 else 600
    tan = 42_700 if t10 else 2_500
    block = 36 if case["precision"] == "mixed" else 72
    matrix = (27.3 if t10 else 14.0) * N * block
    if case["kind"] == "residual":
        return dict(bytes=inputs + 24 * N, flops=res * E)
    if case["kind"] == "assemble":
        return dict(bytes=inputs + 24 * N + matrix, flops=tan * E)
    one = dict(bytes=inputs + 24 * N * (4 if case["kind"] == "newmark" else 2), flops=(res + tan) * E)
    return {k: v * case.get("sets", 1) for k, v in one.items()}


def tolerance(case):
    kind, mixed = case["kind"], case.get("precision") == "mixed"
    if kind == "forward":
        # bfloat16 operands; float32 sums over 128 terms
        return {"rel": 1e-2, "max": 0.2} if case["bf16"] else {"rel": 4e-6, "max": 1e-4}
    if kind == "train":
        return {"rel": 2e-5, "max": 2e-2}
    # residuals and FP64 tangents: 2.7e-12 measured against the 64-bit values (cancellation in the sums)
    if kind == "residual" or (kind == "assemble" and not mixed):
        return {"rel": 1e-11, "max": 1e-9}
    if kind == "assemble":
        return {"rel": 4e-7, "max": 1e-4}
    # converged steps: what the Newton tolerances leave open, four times what runs with other
    # Krylov methods, preconditioners and summation orders differ by
    if kind == "static":
        return {"rel": 2e-6, "max": 1e-5}
    if kind == "newmark":
        return {"rel": 6e-6, "max": 4e-5}
    return {"rel": 4e-9, "max": 3e-8}


# --------------------------------------------------------------------------- 64-bit values

_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _barycentric_gradients(order, l4):
    """dN/dlambda_i [npe, 4] of the element at barycentric coordinates l4"""
    if order == 4:
        return np.eye(4)
    g = np.zeros((10, 4))
    for v in range(4):
        g[v, v] = 4 * l4[v] - 1
    for k, (i, j) in enumerate(((0, 1), (1, 2), (0, 2), (0, 3), (1, 3), (2, 3))):
        g[4 + k, i], g[4 + k, j] = 4 * l4[j], 4 * l4[i]
    return g


class _Exact:
    """the element model in 64-bit torch: residual, tangent (forward-mode derivative of the
    residual), mass, and their sums in the block pattern"""

    def __init__(self, case, p):
        mesh, m = p["mesh"], p["material"]
        self.m, self.time, self.pressure, self.order = m, p["time"], p["pressure"], case["order"]
        self.tension = case["tension"]

        def put(a, dt):
            return torch.from_numpy(np.ascontiguousarray(a)).to(_DEV, dt)
        self.X, self.el = put(mesh.coords, torch.float64), put(mesh.elements, torch.int64)
        self.N, self.npe = mesh.n_nodes, mesh.npe
        self.sur, self.bc = put(mesh.surfaces, torch.int64), put(mesh.bc, torch.int64)
        self.act = put(mesh.activation, torch.float64)
        nb = 5 if self.npe == 10 else 1
        bases = put(mesh.bases.reshape(-1, nb, 3, 3), torch.float64)
        self.B = bases[:, 1:] if nb == 5 else bases
        self.Binv = torch.linalg.inv(self.B)
        a, b = (5 + 3 * math.sqrt(5.0)) / 20, (5 - math.sqrt(5.0)) / 20
        qp = [[a if i == q else b for i in range(4)] for q in range(4)] if self.npe == 10 else [[0.25] * 4]
        Xe = self.X[self.el]
        grads = []
        for l4 in qp:
            g = put(_barycentric_gradients(self.order, l4), torch.float64)
            J = torch.einsum("nai,ak->nik", Xe, g[:, 1:] - g[:, :1])            # dX/dxi
            grads.append(torch.einsum("ak,nki->nai", g[:, 1:] - g[:, :1], torch.linalg.inv(J)))
        self.dN = torch.stack(grads, 1)                                          # [E, q, a, 3]
        gc = put(_barycentric_gradients(self.order, [0.25] * 4), torch.float64)
        self.detJ = torch.linalg.det(torch.einsum("nai,ak->nik", Xe, gc[:, 1:] - gc[:, :1]))
        self.w = self.detJ / (24.0 if self.npe == 10 else 6.0)
        self.free = torch.stack([((self.bc >> c) & 1) == 0 for c in range(3)], 1)   # [N, 3]

    def stress(self, F, act):
        m, P = self.m, self.m.params
        C = F.transpose(-1, -2) @ F
        eye = torch.eye(3, dtype=F.dtype, device=F.device)

        def det(A):
            return (A[..., 0, 0] * (A[..., 1, 1] * A[..., 2, 2] - A[..., 1, 2] * A[..., 2, 1])
                    - A[..., 0, 1] * (A[..., 1, 0] * A[..., 2, 2] - A[..., 1, 2] * A[..., 2, 0])
                    + A[..., 0, 2] * (A[..., 1, 0] * A[..., 2, 1] - A[..., 1, 1] * A[..., 2, 0]))
        J = det(F)
        c = [[C[..., i, j] for j in range(3)] for i in range(3)]
        rows = [torch.stack([c[(j + 1) % 3][(i + 1) % 3] * c[(j + 2) % 3][(i + 2) % 3]
                             - c[(j + 1) % 3][(i + 2) % 3] * c[(j + 2) % 3][(i + 1) % 3] for j in range(3)], -1)
                for i in range(3)]
        Z = torch.stack(rows, -2) / det(C)[..., None, None]
        if m.law == MT.LAW_GUCCIONE:
            Cg, bf, bt, bfs, K = P[:5]
            b = torch.tensor([[bf, bfs, bfs], [bfs, bt, bt], [bfs, bt, bt]], dtype=F.dtype, device=F.device)
            E = 0.5 * (C - eye)
            Q = (b * E * E).sum((-1, -2))
            S = Cg * torch.exp(Q)[..., None, None] * b * E + (K * (J - 1) * J)[..., None, None] * Z
        else:
            a, b, af, bf, as_, bs, afs, bfs, kappa, k = P[:10]
            I1 = c[0][0] + c[1][1] + c[2][2]
            If, Is, I8 = c[0][0], c[1][1], 0.5 * (c[0][1] + c[1][0])
            Hf, Hs = 1 / (1 + torch.exp(-k * (If - 1))), 1 / (1 + torch.exp(-k * (Is - 1)))
            S = (((kappa / 2) * (J - 1 / J) * J)[..., None, None] * Z
                 + (a * torch.exp(b * (I1 - 3)))[..., None, None] * (eye - I1[..., None, None] / 3 * Z))
            cf = 2 * af * Hf * (If - 1) * torch.exp(bf * (If - 1) ** 2)
            cs = 2 * as_ * Hs * (Is - 1) * torch.exp(bs * (Is - 1) ** 2)
            cfs = afs * I8 * torch.exp(bfs * I8 * I8)
            for (i, j), v in (((0, 0), cf), ((1, 1), cs), ((0, 1), cfs), ((1, 0), cfs)):
                e = torch.zeros(3, 3, dtype=F.dtype, device=F.device)
                e[i, j] = 1.0
                S = S + v[..., None, None] * e
        lam = torch.sqrt(F[..., 0, 0] ** 2 + F[..., 1, 0] ** 2 + F[..., 2, 0] ** 2)
        Sff = None
        if self.tension == "sinus":
            start, stop, _, omega, phi = m.fn[:5]
            t = self.time - act
            T = torch.where((t >= start) & (t <= stop), 0.5 - 0.5 * torch.cos(omega * (t - start) + phi),
                            torch.zeros_like(t)) * m.tension_max
            Sff = T[:, None] / lam
        elif self.tension == "tanh":
            cyc, l0, emd, peak, dur, tc0, ld, ldup, tr, kff, st = m.fn[:11]
            t = self.time % cyc if self.time > cyc else self.time
            ts = torch.clamp(t - (act + st) - emd, 0.0, dur)
            phi = torch.tanh(ld * (lam - l0))
            T = (m.tension_max * peak * torch.tanh((dur - ts) / tr) ** 2)[:, None] * phi \
                * torch.tanh(ts[:, None] / (tc0 + ldup * (1 - phi))) ** 2
            Sff = kff * torch.clamp(T, min=0.0) / lam
        if Sff is not None:
            e = torch.zeros(3, 3, dtype=F.dtype, device=F.device)
            e[0, 0] = 1.0
            S = S + Sff[..., None, None] * e
        return S

    def element_forces(self, xe, sl):
        dN, B, Binv = self.dN[sl], self.B[sl], self.Binv[sl]
        F = torch.einsum("nai,nqaj->nqij", xe, dN)
        Fl = B.transpose(-1, -2) @ F @ Binv.transpose(-1, -2)
        S = self.stress(Fl, self.act[sl])
        Pk = Binv.transpose(-1, -2) @ (Fl @ S).transpose(-1, -2) @ B.transpose(-1, -2)
        return self.w[sl][:, None, None] * torch.einsum("nqak,nqkc->nac", dN, Pk)

    def surface_forces(self, xs):
        n = torch.linalg.cross(xs[:, 0] - xs[:, 1], xs[:, 0] - xs[:, 2])
        return (-self.pressure / 6.0) * n[:, None, :].expand(-1, 3, -1)

    def chunks(self, n=50_000):
        E = self.el.shape[0]
        return [slice(i, min(i + n, E)) for i in range(0, E, n)]

    def residual(self, x):
        f = torch.zeros_like(x)
        for sl in self.chunks():
            f.index_add_(0, self.el[sl].reshape(-1), self.element_forces(x[self.el[sl]], sl).reshape(-1, 3))
        f.index_add_(0, self.sur.reshape(-1), self.surface_forces(x[self.sur]).reshape(-1, 3))
        return f * self.free

    def derivative(self, fn, xe):
        """d fn_ai / d x_bj as [n, a, b, i, j]"""
        n, k, _ = xe.shape
        out = torch.empty(n, k, k, 3, 3, dtype=xe.dtype, device=xe.device)
        for b in range(k):
            for j in range(3):
                t = torch.zeros_like(xe)
                t[:, b, j] = 1.0
                out[:, :, b, :, j] = torch.func.jvp(fn, (xe,), (t,))[1]
        return out

    def pattern(self):
        keys = []
        for sl in self.chunks():
            e = self.el[sl]
            keys.append(torch.unique((e[:, :, None] * self.N + e[:, None, :]).reshape(-1)))
        return torch.unique(torch.cat(keys))

    def tangent(self, x, keys, mass=0.0):
        """block values in the pattern `keys` (+ mass * consistent mass), identity on constrained DOFs"""
        V = torch.zeros(keys.numel(), 3, 3, dtype=x.dtype, device=x.device)

        def add(conn, K):
            at = torch.searchsorted(keys, (conn[:, :, None] * self.N + conn[:, None, :]).reshape(-1))
            V.index_add_(0, at, K.reshape(-1, 3, 3))
        for sl in self.chunks():
            K = self.derivative(lambda v: self.element_forces(v, sl), x[self.el[sl]])
            if mass:
                K += (mass * self.m.density) * self.detJ[sl][:, None, None, None, None] \
                    * self.mass_table()[None, :, :, None, None] * torch.eye(3, dtype=x.dtype, device=x.device)
            add(self.el[sl], K)
        add(self.sur, self.derivative(self.surface_forces, x[self.sur]))
        r, c = keys // self.N, keys % self.N
        V *= (self.free[r][:, :, None] & self.free[c][:, None, :])
        d = torch.nonzero(r == c).reshape(-1)
        V[d] += torch.diag_embed((~self.free[r[d]]).to(x.dtype))
        return V

    def mass_table(self):
        """integral of N_a N_b over the reference tetrahedron (density and det J factored out)"""
        def monomial(p):   # of L1^p0 .. L4^p3: product of factorials over (3 + sum)!
            return math.prod(math.factorial(v) for v in p) / math.factorial(3 + sum(p))
        polys = []
        for a in range(self.npe):
            if self.npe == 4:
                polys.append([(1.0, [a])])
            elif a < 4:
                polys.append([(2.0, [a, a]), (-1.0, [a])])
            else:
                i, j = ((0, 1), (1, 2), (0, 2), (0, 3), (1, 3), (2, 3))[a - 4]
                polys.append([(4.0, [i, j])])
        t = [[sum(ca * cb * monomial([(ia + ib).count(v) for v in range(4)]) for ca, ia in pa for cb, ib in pb)
              for pb in polys] for pa in polys]
        return torch.tensor(t, dtype=torch.float64, device=_DEV)

    def solve(self, mass):
        """Newton with a dense solve from the reference configuration at rest"""
        keys = self.pattern()
        r, c = keys // self.N, keys % self.N
        n = 3 * self.N
        rows = (3 * r[:, None] + torch.arange(3, device=_DEV))[:, :, None].expand(-1, 3, 3)
        cols = (3 * c[:, None] + torch.arange(3, device=_DEV))[:, None, :].expand(-1, 3, 3)
        d = torch.zeros_like(self.X)

        def residual(d):
            f = self.residual(self.X + d)
            if mass:
                for sl in self.chunks():
                    e = self.el[sl]
                    md = (mass * self.m.density) * self.detJ[sl][:, None, None] \
                        * torch.einsum("ab,nbi->nai", self.mass_table(), d[e])
                    f.index_add_(0, e.reshape(-1), md.reshape(-1, 3))
            return f * self.free
        best, scale = None, None
        for _ in range(30):
            f = residual(d)
            nf = float(f.norm())
            scale = scale or nf
            if best is not None and nf >= 0.5 * best and nf < 1e-9 * scale:
                break
            best = nf
            A = torch.zeros(n, n, dtype=torch.float64, device=_DEV)
            A[rows, cols] = self.tangent(self.X + d, keys, mass)
            step = torch.linalg.solve(A, -f.reshape(-1, 1)).reshape(-1, 3)
            size = 1.0
            while size > 1e-3 and not float(residual(d + size * step).norm()) < nf and nf > 1e-9 * scale:
                size *= 0.5
            d = d + size * step
        return d


def exact(case, seed):
    if case["kind"] in ("forward", "train"):
        X, T, w = (torch.from_numpy(a).to(_DEV, torch.float64) for a in _net_inputs(case, seed))
        w.requires_grad_(case["kind"] == "train")
        W1, b1, W2, b2, W3, b3 = torch.split(w, [1024, 128, 16384, 128, 384, 3])
        Y = torch.tanh(torch.tanh(X @ W1.view(8, 128) + b1) @ W2.view(128, 128) + b2) @ W3.view(128, 3) + b3
        if case["kind"] == "forward":
            return Y
        loss = ((Y - T) ** 2).mean()
        loss.backward()
        g = w.grad
        return float(loss), g, w.detach() - 1e-3 * g / (g.abs() + 1e-8)
    if case["tension"] == "land17" or case["kind"] == "batch":
        return None
    p = _problem(case, seed)
    if case["kind"] in ("static", "newmark"):
        if 3 * p["mesh"].n_nodes > 13_000:
            return None
        if case["kind"] == "static":
            return _Exact(case, p).solve(0.0).reshape(-1)
        d = _Exact(case, p).solve(4.0 / DT ** 2).reshape(-1)   # beta 1/4, gamma 1/2, from rest
        return d, d * (2.0 / DT), d * (4.0 / DT ** 2)
    e = _Exact(case, p)
    x = torch.from_numpy(p["x"]).to(_DEV)
    f = e.residual(x).reshape(-1)
    return f if case["kind"] == "residual" else (f, e.tangent(x, e.pattern()).reshape(-1))
