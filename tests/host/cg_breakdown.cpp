// The parameter batch's conjugate gradient (batch_kernels.hip) where a set breaks down, on the
// CPU model of workgroups: in the update, where one wave of a workgroup reads the set's flag
// after the launch's first workgroup has set it, the others before; at the start and at
// the end of an iteration, by the flag that the set is left with.
#include "batch_kernels.hip"

#include <cstdio>

using namespace cmg;

int main() {
    // S = 2 sets of 600 nodes (three workgroups), diagonal blocks; set 0 is positive, set 1 negative
    const int S = 2;
    const int64_t N = 600, n = 3 * N;
    std::vector<int64_t> rowptr(N + 1);
    std::vector<int32_t> colind(N), active(S, 1), done(S), it(S);
    std::vector<double> vals(S * 9 * N, 0.0), dinv(S * 9 * N, 0.0), b(S * n), rtol(S, 1e-3);
    for (int64_t r = 0; r <= N; r++) rowptr[r] = r;
    for (int64_t r = 0; r < N; r++) colind[r] = (int32_t)r;
    for (int s = 0; s < S; s++)
        for (int64_t k = 0; k < N; k++)
            for (int c = 0; c < 3; c++) {
                vals[(s * N + k) * 9 + 4 * c] = (s ? -1.0 : 1.0) * (2.0 + (k + c) % 3);
                dinv[(s * N + k) * 9 + 4 * c] = 1.0;
                b[s * n + 3 * k + c] = 1.0 + (k % 7);
            }
    const int64_t ld = batch_spmv_blocks(N, 16) + 1, ld_rz = 2 * batch_node_blocks(N);
    std::vector<double> x(S * n), r(S * n), z(S * n), p(S * n), q(S * n), sc(6 * S), part(S * ld), part_rz(S * ld_rz);
    BatchCG cg;
    cg.S = S;
    cg.x = x.data(), cg.r = r.data(), cg.z = z.data(), cg.p = p.data(), cg.q = q.data();
    cg.rz = sc.data(), cg.rz_next = cg.rz + S, cg.rr = cg.rz + 2 * S, cg.rr0 = cg.rz + 3 * S, cg.alpha = cg.rz + 4 * S;
    cg.tol2 = cg.rz + 5 * S;
    cg.done = done.data(), cg.it = it.data();
    cg.part = part.data(), cg.part_ld = ld, cg.part_rz = part_rz.data(), cg.part_rz_ld = ld_rz;
    int wrong = 0;
    for (int wave = 0; wave < 4; wave++) {
        launch_bcg_init(cg, N, b.data(), dinv.data(), rtol.data(), active.data(), nullptr);
        model::plan.count = 0;
        model::plan.launch = 1;   // product, update, p
        model::plan.late = dim3(1, 1);
        model::plan.late_wave = wave;
        launch_bcg_iteration(cg, 8, N, rowptr.data(), colind.data(), vals.data(), false, 9 * N, dinv.data(), nullptr);
        model::plan.launch = -1;
        int moved = 0;
        for (int64_t i = 0; i < n; i++) moved += x[n + i] != 0.0 || r[n + i] != b[n + i];
        std::printf("late wave %d: set 0 iterations %d, set 1 flag %d, entries changed %d\n", wave, it[0], done[1], moved);
        wrong += it[0] != 1 || done[1] != 2 || moved != 0 || x[0] == 0.0;
    }
    // the start: solved (no right-hand side), turned round by the preconditioner, not finite
    auto start = [&](double rhs, double pre) {
        for (int64_t k = 0; k < N; k++)
            for (int c = 0; c < 3; c++) b[3 * k + c] = rhs, dinv[9 * k + 4 * c] = pre;
        launch_bcg_init(cg, N, b.data(), dinv.data(), rtol.data(), active.data(), nullptr);
        std::printf("right-hand side %g, preconditioner %g: flag %d\n", rhs, pre, done[0]);
        return done[0];
    };
    wrong += start(0.0, 1.0) != 1;
    wrong += start(1.0, 1.0) != 0;
    wrong += start(1.0, -1.0) != 2;
    wrong += start(1.0, 0.0) != 2;
    wrong += start(NAN, 1.0) != 2;
    wrong += start(1e200, 1.0) != 2;
    // the end of an iteration from the products r.z and r.r: converged, running, not finite
    auto end = [&](double rr) {
        start(1.0, 1.0);
        for (int k = 0; k < batch_node_blocks(N); k++) part_rz[2 * k] = 1.0, part_rz[2 * k + 1] = rr;
        model::launch(dim3(1, 1), dim3(kThreads), [&] { k_bcg_p(cg, n, batch_node_blocks(N)); });
        std::printf("r.r %g: flag %d\n", rr, done[0]);
        return done[0];
    };
    wrong += end(1e-12) != 1;
    wrong += end(1.0) != 0;
    wrong += end(INFINITY) != 2;
    wrong += end(NAN) != 2;
    return wrong;
}
