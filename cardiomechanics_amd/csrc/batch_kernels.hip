// Kernels of the parameter-set batch (gfx950): S independent systems on one mesh,
// laid out set-major ([S][n] vectors, [S][nnzb*9] block values, [S][N*9] block
// Jacobi inverses).  Every launch covers all sets (blockIdx.y = set); the scalar
// recurrences of the preconditioned conjugate gradient stay in device memory, so a
// run of iterations needs no host synchronisation and can be captured as one graph.
// The kernels that use a scalar sum its partials themselves, every workgroup in the same
// order: a launch of one workgroup per set took 3 to 4 us, and there were three such per
// iteration (eight sets of 5k elements: six launches and 38 us against nine and 46 us).  A scalar
// that the first workgroup stores is never one that the others read: r.z goes to rz_next, which
// the next product commits.  The exception is the set's flag, see set_done.
// Reductions are two-stage in a fixed order: results do not depend on timing.
#include "batch_kernels.h"

namespace cmg {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ double block_sum256(double v, double* sh) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int w = threadIdx.x / 64, l = threadIdx.x % 64;
    __syncthreads();
    if (l == 0) sh[w] = v;
    __syncthreads();
    return sh[0] + sh[1] + sh[2] + sh[3];
}

// The set's flag, for a kernel whose first workgroup may set it: one thread reads it for its
// whole workgroup, so that a flag set meanwhile stops all of its waves or none.  (Waves that
// each read it could part ways before a sum over the workgroup, which then lacks the share
// of those that left.)  The workgroups may differ: each finds the same verdict in its own
// sums and leaves the set's vectors alone.
__device__ __forceinline__ bool set_done(const int32_t* done, int64_t set) {
    __shared__ int32_t flag;
    if (threadIdx.x == 0) flag = done[set];
    __syncthreads();
    return flag != 0;
}

// q = A p for one set, LANES lanes per block row, plus the block's share of p . q
template <typename VT, int LANES>
__global__ __launch_bounds__(kThreads) void k_bcg_spmv_dot(int64_t N, const int64_t* rowptr, const int32_t* colind,
                                                           const VT* vals, int64_t set_vals, const double* p,
                                                           double* q, int64_t n, const int32_t* done,
                                                           double* partial, int nb, double* rz, const double* rz_next) {
    __shared__ double sh[4];
    const int64_t set = blockIdx.y;
    if (done[set]) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) rz[set] = rz_next[set];
    vals += set * set_vals;
    p += set * n;
    q += set * n;
    const int64_t gt = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int64_t r = gt / LANES;
    const int sub = (int)(gt % LANES);
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    if (r < N) {
        const int64_t end = rowptr[r + 1];
        for (int64_t k = rowptr[r] + sub; k < end; k += LANES) {
            const int64_t c = colind[k];
            const VT* a = vals + 9 * k;
            const double x0 = p[3 * c], x1 = p[3 * c + 1], x2 = p[3 * c + 2];
            s0 += (double)a[0] * x0 + (double)a[1] * x1 + (double)a[2] * x2;
            s1 += (double)a[3] * x0 + (double)a[4] * x1 + (double)a[5] * x2;
            s2 += (double)a[6] * x0 + (double)a[7] * x1 + (double)a[8] * x2;
        }
    }
#pragma unroll
    for (int o = LANES / 2; o > 0; o >>= 1) {
        s0 += __shfl_xor(s0, o, LANES);
        s1 += __shfl_xor(s1, o, LANES);
        s2 += __shfl_xor(s2, o, LANES);
    }
    double pq = 0.0;
    if (r < N && sub == 0) {
        q[3 * r] = s0;
        q[3 * r + 1] = s1;
        q[3 * r + 2] = s2;
        pq = p[3 * r] * s0 + p[3 * r + 1] * s1 + p[3 * r + 2] * s2;
    }
    const double tot = block_sum256(pq, sh);
    if (threadIdx.x == 0) partial[set * nb + blockIdx.x] = tot;
}

// sum of nb partials (stride `ld` between sets, `k` consecutive values per block);
// eight independent loads in flight per thread, summed in a fixed order
__device__ __forceinline__ double reduce_partials(const double* part, int nb, int k, int j, double* sh) {
    double v = 0.0;
#pragma unroll 8
    for (int b = threadIdx.x; b < nb; b += kThreads) v += part[(int64_t)b * k + j];
    return block_sum256(v, sh);
}

// the K sums of nb partials of K consecutive values each, in one pass over contiguous
// memory (thread t takes blocks t, t + 256, ... in order, then the fixed block tree)
template <int K>
__device__ __forceinline__ void reduce_partials_k(const double* part, int nb, double* sh, double* out) {
    double v[K];
#pragma unroll
    for (int j = 0; j < K; j++) v[j] = 0.0;
#pragma unroll 4
    for (int b = threadIdx.x; b < nb; b += kThreads)
#pragma unroll
        for (int j = 0; j < K; j++) v[j] += part[(int64_t)b * K + j];
#pragma unroll
    for (int j = 0; j < K; j++) out[j] = block_sum256(v[j], sh);
}

__global__ __launch_bounds__(kThreads) void k_bcg_alpha(BatchCG cg, int nb) {
    __shared__ double sh[4];
    const int set = blockIdx.x;
    if (cg.done[set]) return;
    const double pq = reduce_partials(cg.part + (int64_t)set * cg.part_ld, nb, 1, 0, sh);
    if (threadIdx.x == 0) {
        if (pq > 0.0 && isfinite(pq)) {
            cg.alpha[set] = cg.rz[set] / pq;
        } else {
            cg.alpha[set] = 0.0;
            cg.done[set] = 2;   // breakdown: the operator is not positive definite on p
        }
    }
}

// x += alpha p, r -= alpha q, z = D^-1 r; partial r.z and r.r (one node per thread).
// Without dinv only x and r (z and the partials then come from the preconditioner).
// alpha from the product's nb partials, or from k_bcg_alpha (nb = 0).
__global__ __launch_bounds__(kThreads) void k_bcg_update(BatchCG cg, int64_t N, const double* dinv, int nb) {
    __shared__ double sh[4];
    const int64_t set = blockIdx.y;
    if (set_done(cg.done, set)) return;
    const int64_t n = 3 * N;
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    double al;
    if (nb) {
        const double pq = reduce_partials(cg.part + set * cg.part_ld, nb, 1, 0, sh);
        if (!(pq > 0.0 && isfinite(pq))) {   // the operator is not positive definite on p
            if (blockIdx.x == 0 && threadIdx.x == 0) cg.done[set] = 2;
            return;
        }
        al = cg.rz[set] / pq;
    } else {
        al = cg.alpha[set];
    }
    if (!dinv) {
        if (i < N) {
            double* x = cg.x + set * n + 3 * i;
            double* r = cg.r + set * n + 3 * i;
            const double* p = cg.p + set * n + 3 * i;
            const double* q = cg.q + set * n + 3 * i;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                x[c] += al * p[c];
                r[c] = r[c] - al * q[c];
            }
        }
        return;
    }
    double rz = 0.0, rr = 0.0;
    if (i < N) {
        double* x = cg.x + set * n + 3 * i;
        double* r = cg.r + set * n + 3 * i;
        double* z = cg.z + set * n + 3 * i;
        const double* p = cg.p + set * n + 3 * i;
        const double* q = cg.q + set * n + 3 * i;
        const double* a = dinv + set * 9 * N + 9 * i;
        double rv[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            x[c] += al * p[c];
            rv[c] = r[c] - al * q[c];
            r[c] = rv[c];
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double zc = a[3 * c] * rv[0] + a[3 * c + 1] * rv[1] + a[3 * c + 2] * rv[2];
            z[c] = zc;
            rz += rv[c] * zc;
            rr += rv[c] * rv[c];
        }
    }
    const double trz = block_sum256(rz, sh);
    const double trr = block_sum256(rr, sh);
    if (threadIdx.x == 0) {
        double* part = cg.part_rz + set * cg.part_rz_ld + 2 * blockIdx.x;
        part[0] = trz;
        part[1] = trr;
    }
}

// p = z, partial r.z and r.r of the active sets after the preconditioner wrote z
__global__ __launch_bounds__(kThreads) void k_bcg_start(BatchCG cg, int64_t N, const int32_t* active) {
    __shared__ double sh[4];
    const int64_t set = blockIdx.y;
    if (!active[set]) return;
    const int64_t n = 3 * N;
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    double rz = 0.0, rr = 0.0;
    if (i < N) {
        const int64_t o = set * n + 3 * i;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double rv = cg.r[o + c], zc = cg.z[o + c];
            cg.p[o + c] = zc;
            rz += rv * zc;
            rr += rv * rv;
        }
    }
    const double trz = block_sum256(rz, sh);
    const double trr = block_sum256(rr, sh);
    if (threadIdx.x == 0) {
        double* part = cg.part_rz + set * cg.part_rz_ld + 2 * blockIdx.x;
        part[0] = trz;
        part[1] = trr;
    }
}

// beta from the nb partials of r.z and r.r, p = z + beta p unless the set has converged
__global__ __launch_bounds__(kThreads) void k_bcg_p(BatchCG cg, int64_t n, int nb) {
    __shared__ double sh[4];
    const int64_t set = blockIdx.y;
    if (set_done(cg.done, set)) return;
    double t2[2];
    reduce_partials_k<2>(cg.part_rz + set * cg.part_rz_ld, nb, sh, t2);
    const double rz = t2[0], rr = t2[1];
    const int fin = rr <= cg.tol2[set] ? 1 : !isfinite(rr) ? 2 : 0;
    const double b = rz / cg.rz[set];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        cg.it[set] += 1;
        cg.rr[set] = rr;
        if (fin)
            cg.done[set] = fin;
        else
            cg.rz_next[set] = rz;
    }
    if (fin) return;
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    double* p = cg.p + set * n;
    p[i] = cg.z[set * n + i] + b * p[i];
}

// start: x = 0, r = b, z = D^-1 r, p = z; partial r.z and r.r (without dinv: x and r only)
__global__ __launch_bounds__(kThreads) void k_bcg_init(BatchCG cg, int64_t N, const double* b, const double* dinv,
                                                       const int32_t* active) {
    __shared__ double sh[4];
    const int64_t set = blockIdx.y;
    if (!active[set]) return;
    const int64_t n = 3 * N;
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (!dinv) {
        if (i < N)
            for (int c = 0; c < 3; c++) {
                cg.x[set * n + 3 * i + c] = 0.0;
                cg.r[set * n + 3 * i + c] = b[set * n + 3 * i + c];
            }
        return;
    }
    double rz = 0.0, rr = 0.0;
    if (i < N) {
        const int64_t o = set * n + 3 * i;
        const double* a = dinv + set * 9 * N + 9 * i;
        const double rv[3] = {b[o], b[o + 1], b[o + 2]};
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double zc = a[3 * c] * rv[0] + a[3 * c + 1] * rv[1] + a[3 * c + 2] * rv[2];
            cg.x[o + c] = 0.0;
            cg.r[o + c] = rv[c];
            cg.z[o + c] = zc;
            cg.p[o + c] = zc;
            rz += rv[c] * zc;
            rr += rv[c] * rv[c];
        }
    }
    const double trz = block_sum256(rz, sh);
    const double trr = block_sum256(rr, sh);
    if (threadIdx.x == 0) {
        double* part = cg.part_rz + set * cg.part_rz_ld + 2 * blockIdx.x;
        part[0] = trz;
        part[1] = trr;
    }
}

__global__ __launch_bounds__(kThreads) void k_bcg_init_reduce(BatchCG cg, int nb, const double* rtol,
                                                              const int32_t* active) {
    __shared__ double sh[4];
    const int set = blockIdx.x;
    if (!active[set]) {
        if (threadIdx.x == 0) {
            cg.done[set] = 1;
            cg.it[set] = 0;
        }
        return;
    }
    const double* part = cg.part_rz + (int64_t)set * cg.part_rz_ld;
    double t2[2];
    reduce_partials_k<2>(part, nb, sh, t2);
    const double rz = t2[0], rr = t2[1];
    if (threadIdx.x == 0) {
        cg.rz_next[set] = rz;
        cg.rr[set] = rr;
        cg.rr0[set] = rr;
        cg.tol2[set] = rtol[set] * rtol[set] * rr;
        cg.it[set] = 0;
        // a right-hand side that the preconditioner turns round (or that is not finite) is no solution
        cg.done[set] = rr == 0.0 ? 1 : !(rz > 0.0) || !isfinite(rr) ? 2 : 0;
    }
}

// ---- per-set BLAS-1 and dots ----
__global__ __launch_bounds__(kThreads) void k_bdot(int64_t n, const double* x, const double* y, double* partial,
                                                   int nb, int64_t part_ld) {
    __shared__ double sh[4];
    const int64_t set = blockIdx.y;
    x += set * n;
    y += set * n;
    double v = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)nb * kThreads)
        v += x[i] * y[i];
    const double t = block_sum256(v, sh);
    if (threadIdx.x == 0) partial[set * part_ld + blockIdx.x] = t;
}

__global__ __launch_bounds__(kThreads) void k_breduce(const double* partial, int nb, int64_t part_ld, double* out) {
    __shared__ double sh[4];
    const int set = blockIdx.x;
    const double t = reduce_partials(partial + (int64_t)set * part_ld, nb, 1, 0, sh);
    if (threadIdx.x == 0) out[set] = t;
}

__global__ __launch_bounds__(kThreads) void k_baxpy(int64_t n, SetCoefs a, const double* x, double* y) {
    const int64_t set = blockIdx.y;
    const double c = a.c[set];
    if (c == 0.0) return;
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    y[set * n + i] += c * x[set * n + i];
}

__global__ __launch_bounds__(kThreads) void k_bscale(int64_t n, SetCoefs a, double* y) {
    const int64_t set = blockIdx.y;
    const double c = a.c[set];
    if (c == 1.0) return;
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    y[set * n + i] *= c;
}


}  // namespace

int batch_dot_blocks(int64_t n) {
    const int64_t b = (n + 8 * kThreads - 1) / (8 * kThreads);
    return (int)std::max<int64_t>(1, std::min<int64_t>(b, 1024));
}

int batch_spmv_blocks(int64_t N, int lanes) { return (int)((N * lanes + kThreads - 1) / kThreads); }

int batch_node_blocks(int64_t N) { return (int)((N + kThreads - 1) / kThreads); }

void launch_bcg_spmv_dot(const BatchCG& cg, int lanes, int64_t N, const int64_t* rowptr, const int32_t* colind,
                         const void* vals, bool fp32, int64_t set_vals, hipStream_t s) {
    const int nb = batch_spmv_blocks(N, lanes);
    const dim3 grid(nb, cg.S);
    const int64_t n = 3 * N;
#define CMG_SPMV(VT, L)                                                                                          \
    hipLaunchKernelGGL((k_bcg_spmv_dot<VT, L>), grid, dim3(kThreads), 0, s, N, rowptr, colind, (const VT*)vals, \
                       set_vals, cg.p, cg.q, n, cg.done, cg.part, (int)cg.part_ld, cg.rz, cg.rz_next)
    if (fp32) {
        if (lanes == 4) CMG_SPMV(float, 4);
        else if (lanes == 16) CMG_SPMV(float, 16);
        else CMG_SPMV(float, 8);
    } else {
        if (lanes == 4) CMG_SPMV(double, 4);
        else if (lanes == 16) CMG_SPMV(double, 16);
        else CMG_SPMV(double, 8);
    }
#undef CMG_SPMV
}

// The spmv writes one partial per block at stride part_ld: part_ld >= blocks (checked by the caller).
void launch_bcg_iteration(const BatchCG& cg, int lanes, int64_t N, const int64_t* rowptr, const int32_t* colind,
                          const void* vals, bool fp32, int64_t set_vals, const double* dinv, hipStream_t s,
                          PrecondApply apply, void* apply_ctx) {
    launch_bcg_spmv_dot(cg, lanes, N, rowptr, colind, vals, fp32, set_vals, s);
    // up to kSelfSummed partials every workgroup of the update sums them; beyond, that is more
    // traffic than a launch is worth
    constexpr int kSelfSummed = 1024;
    int nb = batch_spmv_blocks(N, lanes);
    if (nb > kSelfSummed) {
        hipLaunchKernelGGL(k_bcg_alpha, dim3(cg.S), dim3(kThreads), 0, s, cg, nb);
        nb = 0;
    }
    const int nbn = batch_node_blocks(N);
    hipLaunchKernelGGL(k_bcg_update, dim3(nbn, cg.S), dim3(kThreads), 0, s, cg, N, apply ? nullptr : dinv, nb);
    if (apply) apply(apply_ctx, cg.r, cg.z, cg.part_rz, cg.part_rz_ld);
    const int64_t n = 3 * N;
    hipLaunchKernelGGL(k_bcg_p, dim3((unsigned)((n + kThreads - 1) / kThreads), cg.S), dim3(kThreads), 0, s, cg, n,
                       nbn);
}

void launch_bcg_init(const BatchCG& cg, int64_t N, const double* b, const double* dinv, const double* rtol,
                     const int32_t* active, hipStream_t s, PrecondApply apply, void* apply_ctx) {
    const int nbn = batch_node_blocks(N);
    hipLaunchKernelGGL(k_bcg_init, dim3(nbn, cg.S), dim3(kThreads), 0, s, cg, N, b, apply ? nullptr : dinv, active);
    if (apply) {
        apply(apply_ctx, cg.r, cg.z, nullptr, 0);
        hipLaunchKernelGGL(k_bcg_start, dim3(nbn, cg.S), dim3(kThreads), 0, s, cg, N, active);
    }
    hipLaunchKernelGGL(k_bcg_init_reduce, dim3(cg.S), dim3(kThreads), 0, s, cg, nbn, rtol, active);
}

void launch_bdot(int S, int64_t n, const double* x, const double* y, double* partial, int64_t part_ld, double* out,
                 hipStream_t s) {
    const int nb = batch_dot_blocks(n);
    hipLaunchKernelGGL(k_bdot, dim3(nb, S), dim3(kThreads), 0, s, n, x, y, partial, nb, part_ld);
    hipLaunchKernelGGL(k_breduce, dim3(S), dim3(kThreads), 0, s, partial, nb, part_ld, out);
}

void launch_baxpy(int S, int64_t n, const SetCoefs& a, const double* x, double* y, hipStream_t s) {
    hipLaunchKernelGGL(k_baxpy, dim3((unsigned)((n + kThreads - 1) / kThreads), S), dim3(kThreads), 0, s, n, a, x, y);
}

void launch_bscale(int S, int64_t n, const SetCoefs& a, double* y, hipStream_t s) {
    hipLaunchKernelGGL(k_bscale, dim3((unsigned)((n + kThreads - 1) / kThreads), S), dim3(kThreads), 0, s, n, a, y);
}

}  // namespace cmg
