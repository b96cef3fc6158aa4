// Vertex-patch additive Schwarz preconditioner for T10 tangents (a replacement of the
// 3x3 nodal block Jacobi inside the Krylov solves; the reference factorises the whole
// matrix instead, CBSolverNewmarkBeta.cpp:176-192).
//
// Patch p belongs to element vertex v: the nodes {v} and the midside nodes of every edge
// incident to v (every midside node is in the patches of its two end vertices, every
// vertex in its own).  z = sum_p R_p^T A_p^{-1} R_p r with A_p the principal submatrix
// of the assembled tangent on the patch's DOFs.  On the near-incompressible wall the
// patches carry the locally divergence-free motions that point block Jacobi cannot
// (about 3x fewer BiCGStab iterations on the LV meshes).
//
// Device work per tangent: one wave per patch gathers A_p from the block values into
// LDS and inverts it by Gauss-Jordan elimination with partial pivoting (FP64), storing
// the inverse in groups of kGroup columns (FP64, or FP32 in mixed precision): a lane's
// entries of one row and group are 16 consecutive bytes.  Per application: one
// wave per patch forms y_p = A_p^{-1} r_p (lane i owns row i: coalesced group reads),
// then every node sums its one or two patch results in patch order (deterministic,
// no atomics) and the coarse-grid correction (coarse.hip).
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <vector>

#include "bicgstab.h"
#include "cmg_ctx.h"

namespace cmg {
namespace {

constexpr int kWave = 64;
template <typename IT>
constexpr int kGroup = 16 / sizeof(IT);   // columns of an inverse stored together: [group][row][kGroup]

// A_p^{-1} of the patches order[0, n) that k_patch_invert has no registers for, one wave per
// patch.  Dynamic LDS: nd_cap^2 + nd_cap doubles + nd_cap ints for the largest patch.  Gauss-Jordan with
// partial pivoting; in the elimination each lane owns columns j = lane, lane + 64 and
// walks the rows, so no index is divided and the pivot row stays in registers.
template <typename VT, typename IT>
__global__ __launch_bounds__(kWave) void k_patch_setup(int64_t n, const int32_t* order, const int32_t* pptr,
                                                       const int64_t* sptr, const int32_t* slots, const int64_t* iptr,
                                                       const VT* vals, IT* inv, int nd_cap, int64_t set_vals,
                                                       int64_t set_inv, const int32_t* active) {
    extern __shared__ double lds[];
    if ((int64_t)blockIdx.x >= n) return;
    const int64_t set = blockIdx.y;
    if (active && !active[set]) return;
    vals += set * set_vals;
    inv += set * set_inv;
    const int64_t p = order[blockIdx.x];
    const int lane = threadIdx.x;
    const int np = pptr[p + 1] - pptr[p];
    const int nd = 3 * np;
    double* A = lds;                                   // row-major nd x nd
    double* col = lds + (size_t)nd_cap * nd_cap;
    int* perm = reinterpret_cast<int*>(col + nd_cap);
    const int32_t* sl = slots + sptr[p];
    const int j0 = lane, j1 = lane + kWave;            // this lane's columns (j1 only when nd > 64)
    const int bj0 = j0 / 3, cj0 = j0 - 3 * bj0, bj1 = j1 / 3, cj1 = j1 - 3 * bj1;
    for (int I = 0; I < nd; I++) {
        const int bi = I / 3, ci = I - 3 * bi;
        if (j0 < nd) {
            const int s = sl[bi * np + bj0];
            A[I * nd + j0] = s >= 0 ? (double)vals[9 * (int64_t)s + 3 * ci + cj0] : 0.0;
        }
        if (j1 < nd) {
            const int s = sl[bi * np + bj1];
            A[I * nd + j1] = s >= 0 ? (double)vals[9 * (int64_t)s + 3 * ci + cj1] : 0.0;
        }
    }
    __syncthreads();
    for (int k = 0; k < nd; k++) {
        // pivot: the largest |A[i][k]|, i >= k (smallest i among equals)
        double best = -1.0;
        int bi = k;
        for (int i = k + lane; i < nd; i += kWave) {
            const double v = fabs(A[i * nd + k]);
            if (v > best) {
                best = v;
                bi = i;
            }
        }
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) {
            const double ob = __shfl_xor(best, off);
            const int oi = __shfl_xor(bi, off);
            if (ob > best || (ob == best && oi < bi)) {
                best = ob;
                bi = oi;
            }
        }
        if (lane == 0) perm[k] = bi;
        // swap rows k and bi, scale row k by 1 / pivot (the pivot entry becomes 1 / pivot);
        // the scaled pivot row stays in registers
        double rk0 = 0.0, rk1 = 0.0, a0 = 0.0, a1 = 0.0;
        if (j0 < nd) {
            a0 = A[bi * nd + j0];
            rk0 = A[k * nd + j0];
        }
        if (j1 < nd) {
            a1 = A[bi * nd + j1];
            rk1 = A[k * nd + j1];
        }
        const double piv = __shfl(k < kWave ? a0 : a1, k & (kWave - 1));   // A[bi][k]
        const double ip = 1.0 / piv;
        __syncthreads();
        if (bi != k) {
            if (j0 < nd) A[bi * nd + j0] = rk0;
            if (j1 < nd) A[bi * nd + j1] = rk1;
        }
        rk0 = (j0 == k) ? ip : a0 * ip;
        rk1 = (j1 == k) ? ip : a1 * ip;
        if (j0 < nd) A[k * nd + j0] = rk0;
        if (j1 < nd) A[k * nd + j1] = rk1;
        __syncthreads();
        // column k of the other rows, read before any of them changes
        for (int i = lane; i < nd; i += kWave) col[i] = A[i * nd + k];
        __syncthreads();
        for (int i = 0; i < nd; i++) {
            if (i == k) continue;
            const double f = col[i];
            if (j0 < nd) A[i * nd + j0] = (j0 == k) ? -f * ip : A[i * nd + j0] - f * rk0;
            if (j1 < nd) A[i * nd + j1] = (j1 == k) ? -f * ip : A[i * nd + j1] - f * rk1;
        }
        __syncthreads();
    }
    // row interchanges of the factorisation become column interchanges of the inverse
    for (int k = nd - 1; k >= 0; k--) {
        const int q = perm[k];
        if (q != k)
            for (int i = lane; i < nd; i += kWave) {
                const double t = A[i * nd + k];
                A[i * nd + k] = A[i * nd + q];
                A[i * nd + q] = t;
            }
        __syncthreads();
    }
    IT* out = inv + iptr[p];
    constexpr int G = kGroup<IT>;
    for (int j = 0; j < (nd + G - 1) / G * G; j++)   // columns past nd are zero
        for (int i = lane; i < nd; i += kWave)
            out[((int64_t)(j / G) * nd + i) * G + j % G] = j < nd ? (IT)A[i * nd + j] : (IT)0;
}

// restriction partials of one chunk of fine nodes (all of one grid cell): [corner][component],
// summed over the workgroup in a fixed order
template <typename F>
__device__ __forceinline__ void restrict_chunk(const CoarseGrid& g, int ch, const uint8_t* bcmask, F rhs, double* out,
                                               double* sh) {
    const int start = g.rchunk[3 * ch + 1], count = g.rchunk[3 * ch + 2];
    double s[24];
#pragma unroll
    for (int q = 0; q < 24; q++) s[q] = 0.0;
    for (int k = (int)threadIdx.x; k < count; k += 256) {
        const int64_t n = g.order[start + k];
        const int m = bcmask[n];
        const double fx = g.frac[3 * n], fy = g.frac[3 * n + 1], fz = g.frac[3 * n + 2];
        const double v[3] = {(m & 1) ? 0.0 : rhs(3 * n), (m & 2) ? 0.0 : rhs(3 * n + 1),
                             (m & 4) ? 0.0 : rhs(3 * n + 2)};
#pragma unroll
        for (int a = 0; a < 8; a++) {
            const double w = ((a & 1) ? fx : 1.0 - fx) * ((a & 2) ? fy : 1.0 - fy) * ((a & 4) ? fz : 1.0 - fz);
#pragma unroll
            for (int i = 0; i < 3; i++) s[3 * a + i] += w * v[i];
        }
    }
    // 24 sums over the wave: a halving exchange leaves each lane three of them in 21 exchanges
    // (x, y and z of corner lane / 8), three more steps finish them; one by one they are 144
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
#pragma unroll
    for (int o = 32, h = 12; o >= 8; o >>= 1, h /= 2) {
        const bool up = (lane & o) != 0;
#pragma unroll
        for (int q = 0; q < h; q++) {
            const double give = up ? s[q] : s[h + q], keep = up ? s[h + q] : s[q];
            s[q] = keep + __shfl_xor(give, o, 64);
        }
    }
#pragma unroll
    for (int o = 4; o > 0; o >>= 1)
#pragma unroll
        for (int i = 0; i < 3; i++) s[i] += __shfl_xor(s[i], o, 64);
    if (lane % 8 == 0)
#pragma unroll
        for (int i = 0; i < 3; i++) sh[24 * w + 3 * (lane / 8) + i] = s[i];
    __syncthreads();
    if (threadIdx.x < 24)
        out[3 * (int64_t)g.rslot[8 * ch + threadIdx.x / 3] + threadIdx.x % 3] =
            sh[threadIdx.x] + sh[24 + threadIdx.x] + sh[48 + threadIdx.x] + sh[72 + threadIdx.x];
}

__device__ __forceinline__ double read_lane(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// A_p^{-1} of patches of at most ND DOFs, in registers: lane i holds row i.  Gauss-Jordan with
// partial pivoting, rows left in place: step k picks the free lane with the largest entry of
// column k (by the upper 32 bits of its magnitude, the lowest lane among equals), broadcasts
// its row through scalar registers and subtracts multiples of it from every other row.  The
// pivot row is scaled at the end instead, so one fused multiply-add per entry and step
// remains.  Columns rotate by one register per step, which keeps every register index fixed
// in a loop that is not unrolled.  Bound by the vector ALUs: two lane reads and one
// multiply-add per entry (all
// patches of a setup: 200k LV 5.3 ms in LDS, 1.2 ms; 20k LV 1.0 / 0.54 ms; eight sets of 5k
// 0.83 / 0.30 ms; cube 0.26 / 0.14 ms).
template <typename VT, typename IT, int ND>
__global__ __launch_bounds__(256) void k_patch_invert(int64_t n, const int32_t* order, const int32_t* pptr,
                                                      const int64_t* sptr, const int32_t* slots, const int64_t* iptr,
                                                      const VT* vals, IT* inv, int64_t set_vals, int64_t set_inv,
                                                      const int32_t* active) {
    const int64_t set = blockIdx.y;
    if (active && !active[set]) return;
    const int64_t idx = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;
    if (idx >= n) return;   // whole waves
    vals += set * set_vals;
    inv += set * set_inv;
    const int64_t p = order[idx];
    const int lane = threadIdx.x % kWave;
    const int np = __builtin_amdgcn_readfirstlane(pptr[p + 1] - pptr[p]), nd = 3 * np;
    const int32_t* sl = slots + sptr[p];
    const int bi = lane / 3, ci = lane - 3 * bi;
    double a[ND];
#pragma unroll
    for (int bj = 0; bj < ND / 3; bj++) {
        if (bj < np) {
            const int s = lane < nd ? sl[bi * np + bj] : -1;
#pragma unroll
            for (int c = 0; c < 3; c++) a[3 * bj + c] = s >= 0 ? (double)vals[9 * (int64_t)s + 3 * ci + c] : 0.0;
        } else {
#pragma unroll
            for (int c = 0; c < 3; c++) a[3 * bj + c] = 3 * bj + c == lane ? 1.0 : 0.0;   // identity padding
        }
    }
    bool used = lane >= ND;
    int row = -1, perm = 0;      // the row of the inverse this lane ends with; lane k: the pivot lane of step k
    double scale = 1.0;
#pragma unroll 1
    for (int k = 0; k < ND; k++) {
        const unsigned key = used ? 0u : ((unsigned)(__double_as_longlong(a[0]) >> 32) & 0x7fffffffu) + 1u;
        unsigned best = key;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) best = max(best, (unsigned)__shfl_xor((int)best, o));
        const int piv_lane = __builtin_amdgcn_readfirstlane(__ffsll((long long)__ballot(key == best && !used)) - 1);
        const double ip = 1.0 / read_lane(a[0], piv_lane);
        const bool mine = lane == piv_lane;
        const double m = mine ? 0.0 : a[0] * ip;
        if (mine) {
            used = true;
            row = k;
            scale = ip;
        }
        if (lane == k) perm = piv_lane;
#pragma unroll
        for (int j = 1; j < ND; j++) a[j - 1] = fma(-m, read_lane(a[j], piv_lane), a[j]);
        a[ND - 1] = mine ? 1.0 : -m;
    }
    constexpr int G = kGroup<IT>;
    IT* out = inv + iptr[p];
#pragma unroll
    for (int j = 0; j < ND; j++) {
        const int c = __builtin_amdgcn_readlane(perm, j);
        if (j < nd && c < nd && row >= 0 && row < nd)
            out[((int64_t)(c / G) * nd + row) * G + c % G] = (IT)(a[j] * scale);
    }
    for (int c = nd; c < (nd + G - 1) / G * G; c++)   // columns past nd are zero
        if (lane < nd) out[((int64_t)(c / G) * nd + lane) * G + c % G] = (IT)0;
}

// y_p = A_p^{-1} r_p, one wave per patch, four patches per workgroup; bound by the inverses
// (548 MB on the 200k-element LV) or, on small meshes, by its chain of dependent loads.  Loads
// return in order, so they are issued as they are needed: the patch's nodes, the first
// U groups of the lane's row of the inverse (all of an average patch), the right-hand side
// at the nodes, and only then alpha is formed.  One column
// per load, requested after the right-hand side and behind alpha, took (us, plain / BICG): 200k
// LV 119 / 125 now 105 / 103, FP32 78 / 93 now 58 / 60, 20k LV 14.2 / 17.4 now 12.3 / 14.9,
// 1,296-element cube 8.0 / 9.0 now 4.1 / 4.8.
// The first g.n_rchunk workgroups restrict r to the coarse grid instead.  BICG: s = r - alpha v of a BiCGStab solve
// (one set) in place of r, with alpha from the partials of (r^, v)
template <typename IT, bool BICG>
__global__ __launch_bounds__(256) void k_patch_apply(BicgVec kv, const double* apart, int na, CoarseGrid g,
                                                     const uint8_t* bcmask, double* rpart, int64_t set_rpart,
                                                     int64_t P, const int32_t* pptr, const int32_t* pnodes,
                                                     const int64_t* iptr, const IT* inv, const double* r,
                                                     double* y, int nd_max, int64_t set_inv, int64_t set_vec,
                                                     int64_t set_y, const int32_t* skip) {
    extern __shared__ double lds[];
    const int64_t set = blockIdx.y;
    if (skip && skip[set]) return;   // uniform per workgroup
    inv += set * set_inv;
    r += set * set_vec;
    y += set * set_y;
    __shared__ double sh4[4];
    const double* bv = kv.v;
    if ((int)blockIdx.x < g.n_rchunk) {
        double alpha = 0.0;
        if (BICG && !bicg_alpha(kv, apart, na, sh4, alpha)) return;
        auto rhs = [&](int64_t i) { return BICG ? r[i] - alpha * bv[i] : r[i]; };
        restrict_chunk(g, (int)blockIdx.x, bcmask, rhs, rpart + set * set_rpart, lds);
        return;
    }
    // the wave's number as a scalar: the patch's sizes and offsets become scalar loads and branches
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int64_t p = ((int64_t)blockIdx.x - g.n_rchunk) * 4 + w;
    constexpr int G = kGroup<IT>;
    typedef IT VG __attribute__((ext_vector_type(G)));
    constexpr int U = sizeof(IT) == 8 ? 20 : 12;   // groups requested ahead
    double* rp = lds + (size_t)w * nd_max;
    int p0 = 0, nd = 0;
    const VG* a = nullptr;
    if (p < P) {
        p0 = pptr[p];
        nd = 3 * (pptr[p + 1] - p0);
        a = reinterpret_cast<const VG*>(inv + iptr[p]);
    }
    const int ng = (nd + G - 1) / G;
    VG pre[U];
    double rv = 0.0, vv = 0.0;
    if (lane < nd) {
        const int64_t at = 3 * (int64_t)pnodes[p0 + lane / 3] + lane % 3;
#pragma unroll
        for (int u = 0; u < U; u++) pre[u] = a[(u < ng ? u : 0) * nd + lane];
        rv = r[at];
        if (BICG) vv = bv[at];
    }
    double alpha = 0.0;
    if (BICG && !bicg_alpha(kv, apart, na, sh4, alpha)) return;
    if (nd == 0) return;   // past the last patch
    auto entry = [&](int l) {   // of a patch of more than 64 DOFs
        const int64_t at = 3 * (int64_t)pnodes[p0 + l / 3] + l % 3;
        return BICG ? r[at] - alpha * bv[at] : r[at];
    };
    if (lane < ng * G) rp[lane] = BICG ? rv - alpha * vv : rv;
    for (int l = lane + kWave; l < ng * G; l += kWave) rp[l] = l < nd ? entry(l) : 0.0;
    __builtin_amdgcn_wave_barrier();   // rp belongs to this wave; its LDS operations keep their order
    double* yo = y + 3 * (int64_t)p0;
    if (lane < nd) {
        double acc = 0.0;
#pragma unroll
        for (int u = 0; u < U; u++)
            if (u < ng) {
#pragma unroll
                for (int q = 0; q < G; q++) acc += (double)pre[u][q] * rp[G * u + q];
            }
        for (int gr = U; gr < ng; gr++) {
            const VG v = a[gr * nd + lane];
#pragma unroll
            for (int q = 0; q < G; q++) acc += (double)v[q] * rp[G * gr + q];
        }
        yo[lane] = acc;
    }
    for (int i = lane + kWave; i < nd; i += kWave) {   // the few patches of more than 64 DOFs
        double s = 0.0;
        for (int gr = 0; gr < ng; gr++) {
            const VG v = a[(int64_t)gr * nd + i];
#pragma unroll
            for (int q = 0; q < G; q++) s += (double)v[q] * rp[G * gr + q];
        }
        yo[i] = s;
    }
}

// z[3n + c] = sum over the patches holding node n of their y rows, in patch order, plus the
// coarse correction at the node (g.nodes > 0); DOTS: and the workgroup's share of r.z and r.r
template <bool DOTS>
__global__ __launch_bounds__(256) void k_patch_gather(CoarseGrid g, const uint8_t* bcmask, const double* zc, int64_t N,
                                                      const int32_t* cptr, const int32_t* cpos, const double* y,
                                                      double* z, int64_t set_y, int64_t set_vec, const int32_t* skip,
                                                      const double* r, double* dots, int64_t dots_ld) {
    const int64_t set = blockIdx.y;
    if (skip && skip[set]) return;
    y += set * set_y;
    z += set * set_vec;
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (!DOTS && n >= N) return;
    double rz = 0.0, rr = 0.0;
    if (n < N) {
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        for (int k = cptr[n]; k < cptr[n + 1]; k++) {
            const double* q = y + cpos[k];
            s0 += q[0];
            s1 += q[1];
            s2 += q[2];
        }
        if (g.nodes > 0) {
            const int32_t* ids = g.corner + 8 * (int64_t)g.cell[n];
            const double fx = g.frac[3 * n], fy = g.frac[3 * n + 1], fz = g.frac[3 * n + 2];
            const double* u = zc + set * (int64_t)g.ld;
            double c0 = 0.0, c1 = 0.0, c2 = 0.0;
#pragma unroll
            for (int a = 0; a < 8; a++) {
                const double w = ((a & 1) ? fx : 1.0 - fx) * ((a & 2) ? fy : 1.0 - fy) * ((a & 4) ? fz : 1.0 - fz);
                const double* q = u + 3 * ids[a];
                c0 += w * q[0];
                c1 += w * q[1];
                c2 += w * q[2];
            }
            const int m = bcmask[n];
            s0 += (m & 1) ? 0.0 : c0;
            s1 += (m & 2) ? 0.0 : c1;
            s2 += (m & 4) ? 0.0 : c2;
        }
        z[3 * n] = s0;
        z[3 * n + 1] = s1;
        z[3 * n + 2] = s2;
        if (DOTS) {
            const double* rv = r + set * set_vec + 3 * n;
            const double zv[3] = {s0, s1, s2};
#pragma unroll
            for (int c = 0; c < 3; c++) {
                rz += rv[c] * zv[c];
                rr += rv[c] * rv[c];
            }
        }
    }
    if (DOTS) {
        __shared__ double sh[2][4];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            rz += __shfl_xor(rz, o, 64);
            rr += __shfl_xor(rr, o, 64);
        }
        if (threadIdx.x % 64 == 0) {
            sh[0][threadIdx.x / 64] = rz;
            sh[1][threadIdx.x / 64] = rr;
        }
        __syncthreads();
        if (threadIdx.x < 2)
            dots[set * dots_ld + 2 * blockIdx.x + threadIdx.x] =
                sh[threadIdx.x][0] + sh[threadIdx.x][1] + sh[threadIdx.x][2] + sh[threadIdx.x][3];
    }
}

}  // namespace

int build_vertex_patches(cmg_ctx* c, const int32_t* elements) {
    c->schwarz = false;
    if (c->npe != 10) return CMG_SUCCESS;   // T4: every node is a vertex, patches would be block Jacobi
    const int64_t N = c->N, E = c->E;
    // patch of each vertex: itself and the midside nodes of its edges
    std::vector<int32_t> vid(N, -1);
    for (int64_t e = 0; e < E; e++)
        for (int a = 0; a < 4; a++) vid[elements[e * 10 + a]] = 0;
    int64_t P = 0;
    for (int64_t n = 0; n < N; n++)
        if (vid[n] == 0) vid[n] = (int32_t)P++;
    std::vector<std::vector<int32_t>> patch(P);
    for (int64_t n = 0; n < N; n++)
        if (vid[n] >= 0) patch[vid[n]].push_back((int32_t)n);
    static const int kEdge[6][2] = {{0, 1}, {1, 2}, {0, 2}, {0, 3}, {1, 3}, {2, 3}};   // T10 midside order
    for (int64_t e = 0; e < E; e++)
        for (int k = 0; k < 6; k++) {
            const int32_t m = elements[e * 10 + 4 + k];
            patch[vid[elements[e * 10 + kEdge[k][0]]]].push_back(m);
            patch[vid[elements[e * 10 + kEdge[k][1]]]].push_back(m);
        }
    int np_max = 0;
    for (auto& q : patch) {
        std::sort(q.begin() + 1, q.end());
        q.erase(std::unique(q.begin() + 1, q.end()), q.end());
        np_max = std::max(np_max, (int)q.size());
    }
    if (3 * np_max > kMaxPatchDofs) return CMG_SUCCESS;   // stays with block Jacobi
    // setup launches by size class: up to 24, 30, ... 60 DOFs in registers, the rest in LDS
    std::vector<int32_t> order;
    order.reserve(P);
    c->sw_cls[0] = 0;
    for (int k = 0; k < kPatchClasses; k++) {
        for (int64_t p = 0; p < P; p++) {
            const int nd = 3 * (int)patch[p].size();
            const int cls = nd <= 24 ? 0 : std::min(kPatchClasses - 1, (nd - 24 + 5) / 6);
            if (cls == k) order.push_back((int32_t)p);
        }
        c->sw_cls[k + 1] = (int64_t)order.size();
    }
    std::vector<int32_t> pptr(P + 1, 0), pnodes;
    std::vector<int64_t> sptr(P + 1, 0), iptr(P + 1, 0);
    std::vector<int32_t> slots;
    for (int64_t p = 0; p < P; p++) {
        const auto& q = patch[p];
        const int np = (int)q.size();
        pptr[p + 1] = pptr[p] + np;
        pnodes.insert(pnodes.end(), q.begin(), q.end());
        for (int i = 0; i < np; i++)
            for (int j = 0; j < np; j++) {
                const int32_t* b = c->h_colind.data() + c->h_rowptr[q[i]];
                const int32_t* e = c->h_colind.data() + c->h_rowptr[q[i] + 1];
                const int32_t* f = std::lower_bound(b, e, q[j]);
                slots.push_back((f != e && *f == q[j]) ? (int32_t)(c->h_rowptr[q[i]] + (f - b)) : -1);
            }
        sptr[p + 1] = (int64_t)slots.size();
        const int gc = c->fp32 ? kGroup<float> : kGroup<double>;
        iptr[p + 1] = iptr[p] + (int64_t)(3 * np) * ((3 * np + gc - 1) / gc * gc);
    }
    // node -> positions of its rows in y (y rows follow pnodes), in patch order
    std::vector<int32_t> cnt(N + 1, 0);
    for (int64_t k = 0; k < (int64_t)pnodes.size(); k++) cnt[pnodes[k] + 1]++;
    for (int64_t n = 0; n < N; n++) cnt[n + 1] += cnt[n];
    std::vector<int32_t> cpos(pnodes.size()), fill(cnt.begin(), cnt.end() - 1);
    for (int64_t k = 0; k < (int64_t)pnodes.size(); k++) cpos[fill[pnodes[k]]++] = (int32_t)(3 * k);
    for (int64_t n = 0; n < N; n++)
        if (cnt[n + 1] == cnt[n]) return CMG_SUCCESS;   // a node outside every patch: keep block Jacobi
    hipStream_t s = c->stream;
    CMG_TRY(upload(c->sw_pptr, pptr.data(), pptr.size(), s));
    CMG_TRY(upload(c->sw_pnodes, pnodes.data(), pnodes.size(), s));
    CMG_TRY(upload(c->sw_sptr, sptr.data(), sptr.size(), s));
    CMG_TRY(upload(c->sw_slots, slots.data(), slots.size(), s));
    CMG_TRY(upload(c->sw_iptr, iptr.data(), iptr.size(), s));
    CMG_TRY(upload(c->sw_cptr, cnt.data(), cnt.size(), s));
    CMG_TRY(upload(c->sw_cpos, cpos.data(), cpos.size(), s));
    CMG_TRY(upload(c->sw_order, order.data(), order.size(), s));
    CMG_TRY(alloc(c->sw_inv, (size_t)iptr[P] * (c->fp32 ? sizeof(float) : sizeof(double))));
    CMG_TRY(alloc(c->sw_y, (size_t)3 * pnodes.size() * sizeof(double)));
    CMG_HIP_CHECK(hipStreamSynchronize(s));
    c->sw_P = P;
    c->sw_nd_max = 3 * np_max;
    c->sw_inv_len = iptr[P];
    c->sw_y_len = 3 * (int64_t)pnodes.size();
    c->schwarz = true;
    return CMG_SUCCESS;
}

namespace {

template <typename VT, typename IT>
void patch_setup(cmg_ctx* c, const VT* vals, IT* inv, const PatchSets& ps) {
    for (int k = 0; k < kPatchClasses; k++) {
        const int64_t n = c->sw_cls[k + 1] - c->sw_cls[k];
        if (n == 0) continue;
        const int32_t* order = c->sw_order.as<int32_t>() + c->sw_cls[k];
        const int32_t* pptr = c->sw_pptr.as<int32_t>();
        const int64_t *sptr = c->sw_sptr.as<int64_t>(), *iptr = c->sw_iptr.as<int64_t>();
        const int32_t* slots = c->sw_slots.as<int32_t>();
        const dim3 grid((unsigned)((n + 3) / 4), ps.S);
#define CMG_PINV(ND)                                                                                                \
    hipLaunchKernelGGL((k_patch_invert<VT, IT, ND>), grid, dim3(256), 0, c->stream, n, order, pptr, sptr, slots, iptr, \
                       vals, inv, ps.set_vals, ps.set_inv, ps.flags)
        switch (k) {
        case 0: CMG_PINV(24); break;
        case 1: CMG_PINV(30); break;
        case 2: CMG_PINV(36); break;
        case 3: CMG_PINV(42); break;
        case 4: CMG_PINV(48); break;
        case 5: CMG_PINV(54); break;
        case 6: CMG_PINV(60); break;
        default: {
            const int nd = c->sw_nd_max;
            const size_t lds = (size_t)(nd * nd + nd) * sizeof(double) + (size_t)nd * sizeof(int);
            hipLaunchKernelGGL((k_patch_setup<VT, IT>), dim3((unsigned)n, ps.S), dim3(kWave), lds, c->stream, n, order,
                               pptr, sptr, slots, iptr, vals, inv, nd, ps.set_vals, ps.set_inv, ps.flags);
        }
        }
#undef CMG_PINV
    }
}

}  // namespace

void launch_patch_setup(cmg_ctx* c, const void* vals, const PatchSets& ps) {
    void* inv = ps.inv ? ps.inv : c->sw_inv.p;
    if (c->fp32)
        patch_setup(c, (const float*)vals, (float*)inv, ps);
    else
        patch_setup(c, (const double*)vals, (double*)inv, ps);
    if (c->coarse && ps.use_coarse) launch_coarse_setup(c, vals, ps);
}

namespace {

void patch_apply(cmg_ctx* c, const BicgVec* kv, const double* apart, int na, const double* r, double* z,
                 const PatchSets& ps) {
    const int ndm = (c->sw_nd_max + 3) / 4 * 4;   // whole groups
    const bool coarse = c->coarse && ps.use_coarse;
    const CoarseGrid g = coarse ? c->co : CoarseGrid();
    const CoarseBuf& cb = ps.coarse ? *ps.coarse : c->co_buf;
    const int64_t set_rpart = (int64_t)g.n_rchunk * 24;
    const uint8_t* bc = c->bcmask.as<uint8_t>();
    const dim3 grid((unsigned)((c->sw_P + 3) / 4) + (unsigned)g.n_rchunk, ps.S);
    const size_t lds = (size_t)std::max(4 * ndm, 96) * sizeof(double);
    const void* inv = ps.inv ? ps.inv : c->sw_inv.p;
    double* y = ps.y ? ps.y : c->sw_y.as<double>();
    const BicgVec k = kv ? *kv : BicgVec();
#define CMG_PAPPLY(IT, BICG)                                                                                        \
    hipLaunchKernelGGL((k_patch_apply<IT, BICG>), grid, dim3(256), lds, c->stream, k, apart, na, g, bc,             \
                       cb.rpart.as<double>(), set_rpart, c->sw_P, c->sw_pptr.as<int32_t>(),                         \
                       c->sw_pnodes.as<int32_t>(), c->sw_iptr.as<int64_t>(), (const IT*)inv, r, y, ndm, ps.set_inv, \
                       ps.set_vec, ps.set_y, ps.flags)
    if (c->fp32) {
        if (kv) CMG_PAPPLY(float, true);
        else CMG_PAPPLY(float, false);
    } else {
        if (kv) CMG_PAPPLY(double, true);
        else CMG_PAPPLY(double, false);
    }
#undef CMG_PAPPLY
    if (coarse) launch_coarse_solve(c, ps);
    const dim3 node_grid((unsigned)((c->N + 255) / 256), ps.S);
#define CMG_PGATHER(DOTS)                                                                                          \
    hipLaunchKernelGGL(k_patch_gather<DOTS>, node_grid, dim3(256), 0, c->stream, g, bc, cb.zc.as<double>(), c->N,  \
                       c->sw_cptr.as<int32_t>(), c->sw_cpos.as<int32_t>(), y, z, ps.set_y, ps.set_vec, ps.flags, r, \
                       ps.dots, ps.dots_ld)
    if (ps.dots)
        CMG_PGATHER(true);
    else
        CMG_PGATHER(false);
#undef CMG_PGATHER
}

}  // namespace

void launch_patch_apply(cmg_ctx* c, const double* r, double* z, const PatchSets& ps) {
    patch_apply(c, nullptr, nullptr, 0, r, z, ps);
}

void launch_patch_apply_s(cmg_ctx* c, const BicgVec& k, const double* part, int nb, double* z, const PatchSets& ps) {
    patch_apply(c, &k, part, nb, k.r, z, ps);
}

}  // namespace cmg
