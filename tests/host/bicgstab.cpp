// The BiCGStab solver (bicgstab.hip) with block Jacobi on the CPU model of workgroups: solves
// that converge, that spend their iterations, whose sums overflow or whose alpha breaks down.
#include "bicgstab.hip"

#include <cstdio>

namespace cmg {
void set_error(const std::string&) {}
int fail(const std::string& m, int code) { return std::printf("%s\n", m.c_str()), code; }
int alloc(DevBuf& b, size_t n) { return b.alloc(n) ? CMG_SUCCESS : CMG_ERR_NOMEM; }
void launch_patch_apply(cmg_ctx*, const double*, double*, const PatchSets&) {}
void launch_patch_apply_s(cmg_ctx*, const BicgVec&, const double*, int, double*, const PatchSets&) {}

void launch_spmv(int64_t N, const int64_t* rp, const int32_t* ci, const void* vals, bool, const double* x, double* y,
                 hipStream_t, int, int) {
    const double* v = (const double*)vals;
    for (int64_t r = 0; r < N; r++)
        for (int i = 0; i < 3; i++) {
            double s = 0.0;
            for (int64_t k = rp[r]; k < rp[r + 1]; k++)
                for (int j = 0; j < 3; j++) s += v[9 * k + 3 * i + j] * x[3 * ci[k] + j];
            y[3 * r + i] = s;
        }
}
}  // namespace cmg

using namespace cmg;

// three block diagonals: `diag` I, and `up` / `down` I beside them; preconditioned by I / pre
struct System {
    cmg_ctx c;
    std::vector<double> vals;
    System(int64_t N, double diag, double up, double down, double pre) {
        std::vector<int64_t> rp(1, 0);
        std::vector<int32_t> ci;
        for (int64_t r = 0; r < N; r++) {
            for (int64_t k = std::max<int64_t>(0, r - 1); k <= std::min(N - 1, r + 1); k++) {
                ci.push_back((int32_t)k);
                for (int q = 0; q < 9; q++) vals.push_back(q % 4 ? 0.0 : k == r ? diag : k > r ? up : down);
            }
            rp.push_back((int64_t)ci.size());
        }
        c.N = N;
        c.n = 3 * N;
        c.nnzb = (int64_t)ci.size();
        auto put = [](DevBuf& b, const void* p, size_t n) {
            b.alloc(n);
            memcpy(b.p, p, n);
        };
        put(c.rowptr, rp.data(), rp.size() * sizeof(int64_t));
        put(c.colind, ci.data(), ci.size() * sizeof(int32_t));
        std::vector<double> dinv(9 * N, 0.0);
        for (int64_t r = 0; r < N; r++)
            for (int i = 0; i < 3; i++) dinv[9 * r + 4 * i] = 1.0 / pre;
        put(c.dinv, dinv.data(), dinv.size() * sizeof(double));
        c.gm_V.alloc((size_t)10 * (c.n + 1) * sizeof(double));
    }
    double residual(const std::vector<double>& b, const std::vector<double>& x) {
        std::vector<double> y(c.n);
        launch_spmv(c.N, c.rowptr.as<int64_t>(), c.colind.as<int32_t>(), vals.data(), false, x.data(), y.data(),
                    nullptr, 0, 0);
        double s = 0.0;
        for (int64_t i = 0; i < c.n; i++) s += (b[i] - y[i]) * (b[i] - y[i]);
        return std::sqrt(s);
    }
    cmg_solve_stats solve(const std::vector<double>& b, std::vector<double>& x, double rtol, int maxit) {
        cmg_solve_stats st = {};
        if (bicgstab(&c, vals.data(), b.data(), x.data(), true, rtol, maxit, &st) != CMG_SUCCESS) st.converged = -1;
        std::printf("%lld nodes: %d iterations, converged %d, residual %.3e of %.3e\n", (long long)c.N, st.iterations,
                    st.converged, st.final_residual, st.initial_residual);
        return st;
    }
};

std::vector<double> some(int64_t n, double scale) {
    std::vector<double> b(n);
    for (int64_t i = 0; i < n; i++) b[i] = scale * (1.0 + (i * i) % 7);
    return b;
}

int check(bool ok, const char* what) {
    if (!ok) std::printf("WRONG: %s\n", what);
    return !ok;
}

int main() {
    int wrong = 0;
    for (int64_t N : {1, 5, 100, 300}) {
        System a(N, 4.0, -1.0, -1.5, 4.0);
        std::vector<double> b = some(a.c.n, 1.0), x(a.c.n, 7.0);
        const cmg_solve_stats st = a.solve(b, x, 1e-9, 100);
        wrong += check(st.converged == 1 && a.residual(b, x) <= 1.000001e-9 * st.initial_residual, "a converged solve");
        const cmg_solve_stats two = a.solve(b, x, 1e-9, 2);
        wrong += check(two.iterations <= 2 && std::fabs(a.residual(b, x) - two.final_residual) <= 1e-9 * two.initial_residual,
                       "a solve of two iterations");
    }
    {   // r.r is finite, the products of the second half are not: x stays where it was, and once is enough
        System a(100, 4.0, -1e5, -1e5, 4.0);
        std::vector<double> b = some(a.c.n, 1e149), x(a.c.n, 0.0);
        const cmg_solve_stats st = a.solve(b, x, 1e-9, 100);
        wrong += check(st.converged == 0 && st.iterations == 0, "overflow is no convergence");
        bool zero = true;
        for (double v : x) zero = zero && v == 0.0;
        wrong += check(zero && st.final_residual == st.initial_residual, "x before the overflow");
    }
    {   // a skew matrix and whole numbers: (r^, v) is zero exactly, and would be after any restart
        System a(300, 0.0, 1.0, -1.0, 1.0);
        std::vector<double> b = some(a.c.n, 1.0), x(a.c.n, 0.0);
        const cmg_solve_stats st = a.solve(b, x, 1e-9, 100);
        wrong += check(st.converged == 0 && st.iterations == 0 && a.c.bicg_seq == 2, "a breakdown in alpha, one restart");
    }
    // alpha breaks down and one wave of a workgroup starts after workgroup 0 has ended: nothing is
    // written, and the flags are those of a breakdown from the next product on
    for (int wave = 0; wave < 4; wave++) {
        System a(600, 4.0, -1.0, -1.5, 4.0);
        const int nb = 75;
        std::vector<double> part(nb, 1.0), v(7 * a.c.n, 1.0);
        BicgScalars sc = {};
        BicgHost host = {};
        BicgVec k;
        k.r = &v[0], k.v = &v[a.c.n], k.sh = &v[2 * a.c.n], k.rh = &v[3 * a.c.n], k.t = &v[4 * a.c.n];
        k.sc = &sc, k.host = &host;
        sc.rho = 1.0;
        const unsigned blocks = 3;
        auto form = [&] {
            hipLaunchKernelGGL(k_bicg_s_bj, dim3(blocks), dim3(kThreads), 0, nullptr, k, a.c.N, a.c.dinv.as<double>(),
                               part.data(), nb);
        };
        form();   // leaves a positive sum in the LDS
        std::fill(v.begin() + 2 * a.c.n, v.begin() + 3 * a.c.n, 7.0);
        std::fill(part.begin(), part.end(), 0.0);
        model::plan.count = 0;
        model::plan.launch = 0;
        model::plan.late = dim3(1, 0);
        model::plan.late_wave = wave;
        form();
        model::plan.launch = -1;
        int moved = 0;
        for (int64_t i = 0; i < a.c.n; i++) moved += v[2 * a.c.n + i] != 7.0;
        hipLaunchKernelGGL((k_bicg_spmv<double, 16, kDots>), dim3((600 + 15) / 16), dim3(kThreads), 0, nullptr, k, a.c.N, 1,
                           a.c.rowptr.as<int64_t>(), a.c.colind.as<int32_t>(), a.vals.data(), k.sh, k.t, part.data());
        std::printf("late wave %d: entries written %d, done %d, fin %d\n", wave, moved, sc.done, sc.fin);
        wrong += check(moved == 0 && sc.done == 1 && sc.fin == kBicgBreakdown && (host.word & 0xff) == kBicgBreakdown,
                       "a breakdown in alpha seen late");
    }
    return wrong;
}
