// BiCGStab with right preconditioning (van der Vorst 1992), scalars on the device.
//
// One iteration is nine launches with the Schwarz preconditioner (seven with block Jacobi)
// and no host synchronisation:
//   ph = P^-1 p                      patch apply + restriction, coarse solve, patch gather
//   v = A ph, partials of (r^, v)    k_bicg_spmv<1>
//   sh = P^-1 (r - alpha v)          the patch launch sums the partials, forms alpha and s
//   t = A sh, five partials          k_bicg_spmv<5>: (t,s) (t,t) (r^,t) (r^,s) (s,s)
//   x, r, p, scalars                 k_bicg_update sums the partials and decides
// s is never stored: every kernel that needs it reads r and v, which it needs anyway or
// which cost one vector instead of two.  A consumer sums the product's partials itself when
// there are at most kBicgPartials of them (four loads per thread); above that a small kernel
// leaves kReduceBlocks of them, because every workgroup of the consumer would read them all.
//
// kBicgChunk iterations are one HIP graph.  The host keeps one graph queued behind the
// running one and follows the iteration by the word that k_bicg_update stores in pinned
// memory, so the GPU does not wait for it; iterations queued behind the last one return at
// once (fin).  A finished recurrence is confirmed with the true residual b - A x and
// restarted from x where it has drifted.
// Measured against two host-side scalar exchanges and twelve launches per iteration (whole
// steps, ms): static step of the 1,296-element cube 13.3 / 18.5, Newmark step of the 20k LV
// 24.0 / 31.0, of the 200k LV 320 / 328 in FP64 and 211 / 257 with the FP32 matrix (there
// the product's time counts, see k_bicg_spmv).
// All sums have a fixed order: a context repeats a solve bit for bit (another one may have chosen
// another layout for the product of the true residual, unless spmv_choice fixes it).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "bicgstab.h"
#include "cmg_ctx.h"

namespace cmg {
namespace {

constexpr int kThreads = 256;
constexpr int kDots = 5;
constexpr int kReduceBlocks = 32;
constexpr int kBicgChunk = 4;     // iterations per graph launch

// y = A u and the partial dot products of each workgroup's rows.  DOTS = 1: (rh, y);
// DOTS = 5: the five sums with s = r - alpha v.
//
// Bound by the block values (572 MB on the 200k-element LV in FP64): the first product moves
// 744 MB at 5.2 TB/s, in FP32 453 MB at 5.6 TB/s, a large copy 5.9.  G lanes share a block
// row.  FP64: three lanes per 3x3 block, one per block row, so a wave's load instruction
// covers contiguous 24-byte pieces of 10 (G = 32) or 5 (G = 16) blocks per row; FP32: one
// lane per block.  The loads of kUnroll steps (all of an average row) are issued before
// the first product.  Measured on the 200k LV, against one block per lane and step:
// 131 / 145 us (FP64), 68 / 82 us (FP32, where three lanes per block take 92 us).  Giving
// each XCD a contiguous range of rows costs a factor of 1.9, nontemporal loads 1.3 to 1.9.
// Each workgroup takes `tiles` groups of rows, so that a large mesh leaves fewer partials.
template <typename VT, int G, int DOTS>
__global__ __launch_bounds__(kThreads) void k_bicg_spmv(BicgVec k, int64_t N, int tiles, const int64_t* rowptr,
                                                        const int32_t* colind, const VT* vals, const double* u,
                                                        double* y, double* part) {
    BicgScalars* sc = k.sc;
    if (DOTS == 1 && sc->fin) {
        if (blockIdx.x == 0 && threadIdx.x == 0) sc->done = 1;
        return;
    }
    if (DOTS != 1 && sc->done) {   // by the product before, or because alpha broke down
        if (blockIdx.x == 0 && threadIdx.x == 0 && !sc->fin) sc->fin = kBicgBreakdown;
        return;
    }
    if (DOTS == 1 && blockIdx.x == 0 && threadIdx.x == 0) {
        sc->rho = sc->rho_next;
        sc->it = sc->it_next;
    }
    constexpr int kRows = kThreads / G;
    constexpr bool SPLIT = sizeof(VT) == 8;        // three lanes per block
    constexpr int NB = SPLIT ? G / 3 : G;          // blocks per step
    constexpr int kUnroll = SPLIT ? 3 : 2;
    const int l = (int)(threadIdx.x % G), b = SPLIT ? l / 3 : l, i = SPLIT ? l - 3 * b : 0;
    const double alpha = DOTS == 1 ? 0.0 : sc->alpha;
    double d[DOTS];
#pragma unroll
    for (int j = 0; j < DOTS; j++) d[j] = 0.0;
    for (int t = 0; t < tiles; t++) {
        const int64_t r = ((int64_t)blockIdx.x * tiles + t) * kRows + threadIdx.x / G;
        if (r >= N) break;   // whole groups of G lanes: the shuffles below stay within one
        double yv;
        const int64_t beg = rowptr[r], end = rowptr[r + 1];
        if constexpr (SPLIT) {
            double s = 0.0;
            if (b < NB)
                for (int64_t k0 = beg + b; k0 < end; k0 += NB * kUnroll) {
                    int32_t c[kUnroll];
                    VT a[kUnroll][3];
                    double x[kUnroll][3];
#pragma unroll
                    for (int q = 0; q < kUnroll; q++) {
                        const int64_t kk = k0 + NB * q < end ? k0 + NB * q : k0;
                        c[q] = colind[kk];
#pragma unroll
                        for (int j = 0; j < 3; j++) a[q][j] = vals[9 * kk + 3 * i + j];
                    }
#pragma unroll
                    for (int q = 0; q < kUnroll; q++)
#pragma unroll
                        for (int j = 0; j < 3; j++) x[q][j] = u[3 * (int64_t)c[q] + j];
#pragma unroll
                    for (int q = 0; q < kUnroll; q++)
                        if (q == 0 || k0 + NB * q < end) s += a[q][0] * x[q][0] + a[q][1] * x[q][1] + a[q][2] * x[q][2];
                }
            // fold the NB blocks, fixed tree
#pragma unroll
            for (int o = NB > 8 ? 8 : 4; o > 0; o >>= 1) {
                const double v = __shfl_down(s, 3 * o, G);
                if (b < o && b + o < NB) s += v;
            }
            yv = s;   // lanes 0, 1, 2: the row's components
        } else {
            double s0 = 0.0, s1 = 0.0, s2 = 0.0;
            for (int64_t k0 = beg + b; k0 < end; k0 += NB * kUnroll) {
                int32_t c[kUnroll];
                VT a[kUnroll][9];
                double x[kUnroll][3];
#pragma unroll
                for (int q = 0; q < kUnroll; q++) {
                    const int64_t kk = k0 + NB * q < end ? k0 + NB * q : k0;
                    c[q] = colind[kk];
#pragma unroll
                    for (int j = 0; j < 9; j++) a[q][j] = vals[9 * kk + j];
                }
#pragma unroll
                for (int q = 0; q < kUnroll; q++)
#pragma unroll
                    for (int j = 0; j < 3; j++) x[q][j] = u[3 * (int64_t)c[q] + j];
#pragma unroll
                for (int q = 0; q < kUnroll; q++)
                    if (q == 0 || k0 + NB * q < end) {
                        s0 += (double)a[q][0] * x[q][0] + (double)a[q][1] * x[q][1] + (double)a[q][2] * x[q][2];
                        s1 += (double)a[q][3] * x[q][0] + (double)a[q][4] * x[q][1] + (double)a[q][5] * x[q][2];
                        s2 += (double)a[q][6] * x[q][0] + (double)a[q][7] * x[q][1] + (double)a[q][8] * x[q][2];
                    }
            }
#pragma unroll
            for (int o = G / 2; o > 0; o >>= 1) {
                s0 += __shfl_xor(s0, o, G);
                s1 += __shfl_xor(s1, o, G);
                s2 += __shfl_xor(s2, o, G);
            }
            yv = l == 0 ? s0 : l == 1 ? s1 : s2;
        }
        if (l < 3) {
            y[3 * r + l] = yv;
            const double hr = k.rh[3 * r + l];
            if (DOTS == 1) {
                d[0] += hr * yv;
            } else {
                const double s = k.r[3 * r + l] - alpha * k.v[3 * r + l];
                d[0] += yv * s;
                d[DOTS > 1 ? 1 : 0] += yv * yv;
                d[DOTS > 2 ? 2 : 0] += hr * yv;
                d[DOTS > 3 ? 3 : 0] += hr * s;
                d[DOTS > 4 ? 4 : 0] += s * s;
            }
        }
    }
    __shared__ double shm[DOTS][kThreads / 64];
#pragma unroll
    for (int j = 0; j < DOTS; j++)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) d[j] += __shfl_xor(d[j], o, 64);
    if (threadIdx.x % 64 == 0)
#pragma unroll
        for (int j = 0; j < DOTS; j++) shm[j][threadIdx.x / 64] = d[j];
    __syncthreads();
    if (threadIdx.x < DOTS)
        part[(int64_t)DOTS * blockIdx.x + threadIdx.x] =
            shm[threadIdx.x][0] + shm[threadIdx.x][1] + shm[threadIdx.x][2] + shm[threadIdx.x][3];
}

// workgroup g sums the g-th of kReduceBlocks ranges of the nb partials of K values each
template <int K>
__global__ __launch_bounds__(kThreads) void k_bicg_reduce(const BicgScalars* sc, const double* part, int nb,
                                                          double* out) {
    __shared__ double sh[K][4];
    if (sc->fin) return;
    const int per = (nb + kReduceBlocks - 1) / kReduceBlocks;
    const int lo = (int)blockIdx.x * per, hi = min(nb, lo + per);
    double v[K];
#pragma unroll
    for (int j = 0; j < K; j++) v[j] = 0.0;
#pragma unroll 2
    for (int b = lo + (int)threadIdx.x; b < hi; b += kThreads)
#pragma unroll
        for (int j = 0; j < K; j++) v[j] += part[(int64_t)b * K + j];
#pragma unroll
    for (int j = 0; j < K; j++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v[j] += __shfl_xor(v[j], o, 64);
        if (threadIdx.x % 64 == 0) sh[j][threadIdx.x / 64] = v[j];
    }
    __syncthreads();
    if (threadIdx.x < K)
        out[K * blockIdx.x + threadIdx.x] =
            sh[threadIdx.x][0] + sh[threadIdx.x][1] + sh[threadIdx.x][2] + sh[threadIdx.x][3];
}

// ph = D^-1 p (block Jacobi)
__global__ __launch_bounds__(kThreads) void k_bicg_p_bj(BicgVec k, int64_t N, const double* dinv) {
    if (k.sc->fin) return;
    const int64_t n = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (n >= N) return;
    const double* a = dinv + 9 * n;
    const double p0 = k.p[3 * n], p1 = k.p[3 * n + 1], p2 = k.p[3 * n + 2];
    k.ph[3 * n] = a[0] * p0 + a[1] * p1 + a[2] * p2;
    k.ph[3 * n + 1] = a[3] * p0 + a[4] * p1 + a[5] * p2;
    k.ph[3 * n + 2] = a[6] * p0 + a[7] * p1 + a[8] * p2;
}

// alpha, then sh = D^-1 (r - alpha v) (block Jacobi)
__global__ __launch_bounds__(kThreads) void k_bicg_s_bj(BicgVec k, int64_t N, const double* dinv, const double* part,
                                                        int nb) {
    __shared__ double sh[4];
    if (k.sc->fin) return;
    double alpha;
    if (!bicg_alpha(k, part, nb, sh, alpha)) return;
    const int64_t n = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (n >= N) return;
    const double* a = dinv + 9 * n;
    double s[3];
#pragma unroll
    for (int c = 0; c < 3; c++) s[c] = k.r[3 * n + c] - alpha * k.v[3 * n + c];
    k.sh[3 * n] = a[0] * s[0] + a[1] * s[1] + a[2] * s[2];
    k.sh[3 * n + 1] = a[3] * s[0] + a[4] * s[1] + a[5] * s[2];
    k.sh[3 * n + 2] = a[6] * s[0] + a[7] * s[1] + a[8] * s[2];
}

// x += alpha ph + omega sh; r = s - omega t; p = r + beta (p - omega v) unless the solve
// ends here.  Two entries per thread (the vectors are 16-byte aligned).  Every workgroup
// sums the partials and forms the scalars; workgroup 0 stores them in the *_next slots, so
// none of them reads what another one writes.
__global__ __launch_bounds__(kThreads) void k_bicg_update(BicgVec k, int64_t n, const double* part, int nb) {
    __shared__ double sh[kDots][4];
    BicgScalars* sc = k.sc;
    if (sc->done) return;
    double d[kDots];
#pragma unroll
    for (int j = 0; j < kDots; j++) {
        d[j] = 0.0;
#pragma unroll
        for (int b = 0; b < kBicgPartials; b += 256)
            d[j] += b + (int)threadIdx.x < nb ? part[(int64_t)(b + threadIdx.x) * kDots + j] : 0.0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) d[j] += __shfl_xor(d[j], o, 64);
        if (threadIdx.x % 64 == 0) sh[j][threadIdx.x / 64] = d[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kDots; j++) d[j] = sh[j][0] + sh[j][1] + sh[j][2] + sh[j][3];
    const double ts = d[0], tt = d[1], rht = d[2], rhs = d[3], ss = d[4];
    const double alpha = sc->alpha, rho = sc->rho;
    const double om = tt > 0.0 ? ts / tt : 0.0;
    const double rho_new = rhs - om * rht;
    const double rr = ss - 2.0 * om * ts + om * om * tt;
    // sums that are not finite: x stays where the iteration found it, which then does not count
    const bool lost = !isfinite(rr);
    const int it = sc->it + (lost ? 0 : 1);
    int fin = 0;
    if (lost)
        fin = kBicgBreakdown;
    else if (rr <= sc->tol2)
        fin = kBicgConverged;
    else if (om == 0.0 || !(fabs(rho_new) > 0.0) || !isfinite(rho_new))
        fin = kBicgBreakdown;
    else if (it >= sc->maxit)
        fin = kBicgMaxit;
    const double beta = fin ? 0.0 : (rho_new / rho) * (alpha / om);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->rho_next = rho_new;
        sc->it_next = it;
        sc->fin = fin;
        bicg_publish(sc, k.host, it, fin);
    }
    if (lost) return;
    const int64_t i = 2 * ((int64_t)blockIdx.x * kThreads + threadIdx.x);
    if (i + 1 < n) {
        const double2 v = *reinterpret_cast<const double2*>(k.v + i), t = *reinterpret_cast<const double2*>(k.t + i);
        const double2 ph = *reinterpret_cast<const double2*>(k.ph + i);
        const double2 s2 = *reinterpret_cast<const double2*>(k.sh + i);
        double2 x = *reinterpret_cast<const double2*>(k.x + i), r = *reinterpret_cast<const double2*>(k.r + i);
        double2 p = *reinterpret_cast<const double2*>(k.p + i);
        x.x += alpha * ph.x + om * s2.x;
        x.y += alpha * ph.y + om * s2.y;
        r.x = (r.x - alpha * v.x) - om * t.x;
        r.y = (r.y - alpha * v.y) - om * t.y;
        *reinterpret_cast<double2*>(k.x + i) = x;
        *reinterpret_cast<double2*>(k.r + i) = r;
        if (!fin) {
            p.x = r.x + beta * (p.x - om * v.x);
            p.y = r.y + beta * (p.y - om * v.y);
            *reinterpret_cast<double2*>(k.p + i) = p;
        }
    } else if (i < n) {
        k.x[i] += alpha * k.ph[i] + om * k.sh[i];
        const double r = (k.r[i] - alpha * k.v[i]) - om * k.t[i];
        k.r[i] = r;
        if (!fin) k.p[i] = r + beta * (k.p[i] - om * k.v[i]);
    }
}

// r = b - A x (A x in k.v; zero: x = 0 instead), r^ = p = r; partials of (r, r) and (b, b)
__global__ __launch_bounds__(kThreads) void k_bicg_init(BicgVec k, int64_t n, const double* b, int zero,
                                                        double* part) {
    __shared__ double sh[2][4];
    double rr = 0.0, bb = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
        const double bv = b[i];
        const double rv = zero ? bv : bv - k.v[i];
        if (zero) k.x[i] = 0.0;
        k.r[i] = rv;
        k.rh[i] = rv;
        k.p[i] = rv;
        rr += rv * rv;
        bb += bv * bv;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        rr += __shfl_xor(rr, o, 64);
        bb += __shfl_xor(bb, o, 64);
    }
    if (threadIdx.x % 64 == 0) {
        sh[0][threadIdx.x / 64] = rr;
        sh[1][threadIdx.x / 64] = bb;
    }
    __syncthreads();
    if (threadIdx.x < 2)
        part[2 * blockIdx.x + threadIdx.x] =
            sh[threadIdx.x][0] + sh[threadIdx.x][1] + sh[threadIdx.x][2] + sh[threadIdx.x][3];
}

// scalars of a (re)start from the partials of k_bicg_init (nb <= 256)
__global__ __launch_bounds__(kThreads) void k_bicg_start(BicgVec k, const double* part, int nb, double rtol, int maxit,
                                                         int first, unsigned seq) {
    __shared__ double sh[2][4];
    double d[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        d[j] = (int)threadIdx.x < nb ? part[2 * threadIdx.x + j] : 0.0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) d[j] += __shfl_xor(d[j], o, 64);
        if (threadIdx.x % 64 == 0) sh[j][threadIdx.x / 64] = d[j];
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    const double rr = sh[0][0] + sh[0][1] + sh[0][2] + sh[0][3];
    const double bb = sh[1][0] + sh[1][1] + sh[1][2] + sh[1][3];
    BicgScalars* sc = k.sc;
    sc->seq = seq;
    sc->maxit = maxit;
    if (first) {
        sc->it_next = 0;
        sc->tol2 = rtol * rtol * (bb > 0.0 ? bb : 1.0);
    }
    sc->rho_next = rr;
    const int fin = (rr <= sc->tol2 || rr == 0.0) ? kBicgConverged : !isfinite(rr) ? kBicgBreakdown
                    : sc->it_next >= maxit ? kBicgMaxit : 0;
    sc->fin = fin;
    sc->done = fin ? 1 : 0;
    k.host->rr = rr;
    k.host->tol2 = sc->tol2;
    __threadfence_system();
    bicg_publish(sc, k.host, sc->it_next, fin);
}

struct Launch {
    cmg_ctx* c;
    BicgVec k;
    const void* vals;
    double *part, *sums;
    int lanes, tiles, nb;   // lanes per block row, row groups per workgroup, partials of one product

    template <int DOTS>
    void product(const double* u, double* y) const {
        const dim3 grid((unsigned)nb);
        hipStream_t s = c->stream;
        const int64_t* rp = c->rowptr.as<int64_t>();
        const int32_t* ci = c->colind.as<int32_t>();
#define CMG_BICG(VT, G)                                                                                           \
    hipLaunchKernelGGL((k_bicg_spmv<VT, G, DOTS>), grid, dim3(kThreads), 0, s, k, c->N, tiles, rp, ci,            \
                       (const VT*)vals, u, y, part)
        if (c->fp32) {
            if (lanes == 16) CMG_BICG(float, 16);
            else CMG_BICG(float, 8);
        } else {
            if (lanes == 32) CMG_BICG(double, 32);
            else CMG_BICG(double, 16);
        }
#undef CMG_BICG
        if (nb > kBicgPartials)
            hipLaunchKernelGGL(k_bicg_reduce<DOTS>, dim3(kReduceBlocks), dim3(kThreads), 0, s, k.sc, part, nb, sums);
    }

    void iteration() const {
        hipStream_t s = c->stream;
        const bool summed = nb > kBicgPartials;
        const double* pt = summed ? sums : part;
        const int np = summed ? kReduceBlocks : nb;
        const unsigned node_blocks = (unsigned)((c->N + kThreads - 1) / kThreads);
        PatchSets ps;
        ps.flags = &k.sc->fin;
        if (c->schwarz)
            launch_patch_apply(c, k.p, k.ph, ps);
        else
            hipLaunchKernelGGL(k_bicg_p_bj, dim3(node_blocks), dim3(kThreads), 0, s, k, c->N, c->dinv.as<double>());
        product<1>(k.ph, k.v);
        if (c->schwarz)
            launch_patch_apply_s(c, k, pt, np, k.sh, ps);
        else
            hipLaunchKernelGGL(k_bicg_s_bj, dim3(node_blocks), dim3(kThreads), 0, s, k, c->N, c->dinv.as<double>(), pt,
                               np);
        product<kDots>(k.sh, k.t);
        hipLaunchKernelGGL(k_bicg_update, dim3((unsigned)((c->n + 2 * kThreads - 1) / (2 * kThreads))), dim3(kThreads),
                           0, s, k, c->n, pt, np);
    }
};

// waits until the solve `seq` has reached iteration `it` or ended; the word then
int wait_for(cmg_ctx* c, unsigned seq, int it, unsigned long long& word) {
    const unsigned long long* w = &c->bicg_host->word;
    auto reached = [&]() {
        word = __atomic_load_n(w, __ATOMIC_ACQUIRE);
        return (unsigned)(word >> 40) == seq && ((int)((word >> 8) & 0xffffffffu) >= it || (word & 0xff) != 0);
    };
    return wait_host(c, reached);
}

}  // namespace

int bicgstab(cmg_ctx* c, const void* vals, const double* b, double* x, bool zero_guess, double rtol, int maxit,
             cmg_solve_stats* st) {
    hipStream_t s = c->stream;
    const int64_t n = c->n, ld = (n + 1) / 2 * 2;   // even: 16-byte aligned vectors
    Launch L;
    L.c = c;
    L.vals = vals;
    // lanes per row by its average length (T10 about 27 blocks, T4 about 14): one unrolled step
    // holds 30 or 15 blocks in FP64, 32 or 16 in FP32
    L.lanes = (c->nnzb > 20 * c->N ? 2 : 1) * (c->fp32 ? 8 : 16);
    // row groups per workgroup: as few as leave kBicgPartials partials, up to four; meshes too
    // large for that have one or, where the chip is full anyway, four (20k-element LV, four
    // groups: two reductions of 4.6 us less, the first product 2.6 us and the update 1.5 us more).
    // Whole steps with one / four groups, iterations that move with the order of the sums among it
    // (ms): FP64 40k elements 44.2 / 39.5, 50k (75,744 nodes) 57.5 / 57.8, 75k 84.0 / 88.5; mixed
    // 31.8 / 31.7, 40.9 / 36.6, 54.3 / 56.2
    const int64_t groups = (c->N + kThreads / L.lanes - 1) / (kThreads / L.lanes);
    L.tiles = (int)((groups + kBicgPartials - 1) / kBicgPartials);
    if (L.tiles > 4) L.tiles = c->N > 65536 ? 4 : 1;
    const int64_t rows = (int64_t)L.tiles * (kThreads / L.lanes);
    L.nb = (int)((c->N + rows - 1) / rows);
    if (!c->bicg_host) {
        CMG_TRY(alloc(c->bicg_part, ((size_t)kDots * (L.nb + kReduceBlocks) + 2 * 256) * sizeof(double)));
        CMG_TRY(alloc(c->bicg_sc, sizeof(BicgScalars)));
        CMG_HIP_CHECK(hipHostMalloc((void**)&c->bicg_host, sizeof(BicgHost),
                                    hipHostMallocCoherent | hipHostMallocMapped));
        std::memset((void*)c->bicg_host, 0, sizeof(BicgHost));
    }
    double* W = c->gm_V.as<double>();   // (restart + 2) >= 10 vectors of n
    BicgVec& k = L.k;
    k.x = x;
    k.r = W;
    k.rh = W + ld;
    k.p = W + 2 * ld;
    k.v = W + 3 * ld;
    k.t = W + 4 * ld;
    k.ph = W + 5 * ld;
    k.sh = W + 6 * ld;
    k.sc = c->bicg_sc.as<BicgScalars>();
    k.host = c->bicg_host;
    L.part = c->bicg_part.as<double>();
    L.sums = L.part + (int64_t)kDots * L.nb + 2 * 256;
    double* ipart = L.part + (int64_t)kDots * L.nb;
    const int ni = (int)std::min<int64_t>(256, (n + 4 * kThreads - 1) / (4 * kThreads));
    auto start = [&](bool first, bool zero) {
        if (!zero)
            launch_spmv(c->N, c->rowptr.as<int64_t>(), c->colind.as<int32_t>(), vals, c->fp32, x, k.v, s, c->spmv_lanes,
                        c->spmv_layout);
        hipLaunchKernelGGL(k_bicg_init, dim3(ni), dim3(kThreads), 0, s, k, n, b, zero ? 1 : 0, ipart);
        c->bicg_seq = (c->bicg_seq + 1) & 0xffffff;
        hipLaunchKernelGGL(k_bicg_start, dim3(1), dim3(kThreads), 0, s, k, ipart, ni, rtol, maxit, first ? 1 : 0,
                           c->bicg_seq);
    };
    start(true, zero_guess);
    if (!c->bicg_graph || c->bicg_graph_x != x || c->bicg_graph_vals != vals) {
        if (c->bicg_graph) (void)hipGraphExecDestroy(c->bicg_graph);
        c->bicg_graph = nullptr;
        hipGraph_t g = nullptr;
        CMG_HIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        for (int i = 0; i < kBicgChunk; i++) L.iteration();
        CMG_HIP_CHECK(hipStreamEndCapture(s, &g));
        const hipError_t e = hipGraphInstantiate(&c->bicg_graph, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        CMG_HIP_CHECK(e);
        c->bicg_graph_x = x;
        c->bicg_graph_vals = vals;
    }
    unsigned long long word = 0;
    int it0 = 0;   // iterations before the last (re)start
    bool stuck = false;   // broken down in the first iteration after it: another one would do the same
    for (int restarts = 0;; restarts++) {
        CMG_TRY(wait_for(c, c->bicg_seq, 0, word));
        const double rn = std::sqrt(c->bicg_host->rr);
        if (restarts == 0) st->initial_residual = rn;
        st->iterations = it0;
        st->final_residual = rn;
        st->converged = (word & 0xff) == kBicgConverged && c->bicg_host->rr <= c->bicg_host->tol2;
        if (rn == 0.0) st->converged = 1;
        // the residual just computed is the true one: converged, out of restarts or iterations, or lost
        if ((word & 0xff) != 0 || stuck || restarts > 50) break;
        int queued = it0;
        auto queue = [&]() -> int {
            CMG_HIP_CHECK(hipGraphLaunch(c->bicg_graph, s));
            queued += kBicgChunk;
            return CMG_SUCCESS;
        };
        CMG_TRY(queue());
        do {
            CMG_TRY(queue());
            CMG_TRY(wait_for(c, c->bicg_seq, queued - kBicgChunk, word));
        } while ((word & 0xff) == 0);
        const int it = (int)((word >> 8) & 0xffffffffu);
        stuck = (word & 0xff) == kBicgBreakdown && it == it0;
        it0 = it;
        start(false, false);   // r = b - A x: confirms, or continues from x
    }
    CMG_HIP_CHECK(hipGetLastError());
    return CMG_SUCCESS;
}

}  // namespace cmg
