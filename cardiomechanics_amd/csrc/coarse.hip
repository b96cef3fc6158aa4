// Coarse-grid correction of the vertex-patch Schwarz preconditioner (schwarz.hip):
// z = sum_p R_p^T A_p^{-1} R_p r + P A_c^{-1} P^T r with A_c = P^T A P.
//
// One-level Schwarz needs iterations in proportion to the number of patches across the
// mesh, because a patch moves information by one edge per iteration.  P spans the smooth
// motions instead: the trilinear hats of a regular background grid over the bounding box,
// times the three translations, zero on constrained DOFs.  The grid has at most a few
// hundred nodes near the mesh (build_coarse), so A_c is a small dense matrix and its
// inverse one matrix-vector product.  Iterations to a residual of 0.1 (the first Newton
// solves), without / with it: 75 / 18 on the 1,296-element cube under static load,
// 300 / 34 on the 5k-element LV under static load, 32 / 16 on the 20k-element LV in a
// 1 ms Newmark step, where the inertia term already bounds the smooth motions.
//
// Setup per preconditioner build:
//   k_coarse_galerkin  one workgroup per chunk of fine nodes of one grid cell; a wave takes
//                      one block row at a time, lane = one of the 4^3 grid nodes the row's
//                      columns can reach (every element spans at most two cells per axis).
//                      It sums t = sum_c A_rc hat(c) over the row and adds the outer
//                      product with the row's own 8 hats to 72 accumulators per lane.
//   k_coarse_assemble  one workgroup per grid node sums its chunks in chunk order.
//   k_coarse_panel / k_coarse_update   blocked Gauss-Jordan inversion in place, 32 columns
//                      per panel, without pivoting: A_c of a positive tangent is positive.
//                      A column whose pivot vanishes against its original diagonal is
//                      dropped from the space (zero row and column): a grid function that
//                      the mesh does not resolve.  A clearly negative pivot marks an
//                      indefinite tangent (soft parameter sets at an extrapolated guess):
//                      the correction is then off (bad) until the next setup, and the
//                      preconditioner is the one-level Schwarz, as it is where these
//                      buffers do not fit the device.
// Per application: the restriction runs as extra workgroups of the patch launch,
// k_coarse_solve sums the restriction partials and multiplies by the inverse, and the
// patch gather adds P z_c.  All sums have a fixed order (no atomics).
#include <algorithm>
#include <cmath>
#include <vector>

#include "cmg_ctx.h"

namespace cmg {
namespace {

constexpr int kFusedRhs = 1024;     // components of r_c that the product's workgroups sum themselves
constexpr int kCoarseRows = 2048;   // and at most
constexpr int kRhsAhead = 8;
constexpr int kTile = 32;            // columns per elimination panel
constexpr int kGalRows = 28;         // blocks of a row staged in LDS at a time
constexpr int kGalPart = 8 * 9 * 64; // partial sums of one chunk: [corner][entry][lane]
// pivots relative to the original diagonal: dropped up to the first, indefinite below minus
// the second; FP32 block values carry noise of about 1e-7 of the diagonal
constexpr double kDrop64 = 1e-10, kNegative64 = 1e-8, kDrop32 = 1e-6, kNegative32 = 1e-5;

__device__ __forceinline__ double hat(double u) { return fmax(0.0, 1.0 - fabs(u)); }

template <typename VT>
__global__ __launch_bounds__(256) void k_coarse_galerkin(CoarseGrid g, const int64_t* rowptr, const int32_t* colind,
                                                         const uint8_t* bcmask, const VT* vals, int64_t set_vals,
                                                         double* part, int64_t set_part, const int32_t* active) {
    __shared__ double sv[4][9 * kGalRows];
    __shared__ double su[4][3 * kGalRows];
    __shared__ double sacc[kGalPart];
    const int64_t set = blockIdx.y;
    if (active && !active[set]) return;
    vals += set * set_vals;
    part += set * set_part + (int64_t)blockIdx.x * kGalPart;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
    const int lx = (lane & 3) - 1, ly = ((lane >> 2) & 3) - 1, lz = (lane >> 4) - 1;
    const int start = g.chunk[3 * blockIdx.x + 1], count = g.chunk[3 * blockIdx.x + 2];
    double acc[72];
#pragma unroll
    for (int q = 0; q < 72; q++) acc[q] = 0.0;
    for (int it = w; it < count; it += 4) {
        const int64_t r = g.order[start + it];
        const int32_t cp = g.pos[r];
        const int cx = cp & 1023, cy = (cp >> 10) & 1023, cz = cp >> 20;
        const double fx = g.frac[3 * r], fy = g.frac[3 * r + 1], fz = g.frac[3 * r + 2];
        const int mask = bcmask[r];
        const int64_t k0 = rowptr[r];
        const int nb = (int)(rowptr[r + 1] - k0);
        double t[9];
#pragma unroll
        for (int q = 0; q < 9; q++) t[q] = 0.0;
        for (int base = 0; base < nb; base += kGalRows) {
            const int nt = min(kGalRows, nb - base);
            const VT* v = vals + 9 * (k0 + base);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int idx = lane + 64 * j;
                if (idx < 9 * nt) sv[w][idx] = (double)v[idx];
            }
            if (lane < nt) {
                const int64_t c = colind[k0 + base + lane];
                const int32_t p = g.pos[c];
                su[w][3 * lane] = g.frac[3 * c] + (double)((p & 1023) - cx);
                su[w][3 * lane + 1] = g.frac[3 * c + 1] + (double)(((p >> 10) & 1023) - cy);
                su[w][3 * lane + 2] = g.frac[3 * c + 2] + (double)((p >> 20) - cz);
            }
            __builtin_amdgcn_wave_barrier();   // one wave's LDS operations keep their order
            for (int k = 0; k < nt; k++) {
                const double wt = hat(su[w][3 * k] - lx) * hat(su[w][3 * k + 1] - ly) * hat(su[w][3 * k + 2] - lz);
#pragma unroll
                for (int q = 0; q < 9; q++) t[q] += wt * sv[w][9 * k + q];
            }
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int q = 0; q < 9; q++)
            if ((mask >> (q / 3)) & 1) t[q] = 0.0;   // constrained rows (the assembly leaves zero columns)
#pragma unroll
        for (int a = 0; a < 8; a++) {
            const double wr = ((a & 1) ? fx : 1.0 - fx) * ((a & 2) ? fy : 1.0 - fy) * ((a & 4) ? fz : 1.0 - fz);
#pragma unroll
            for (int q = 0; q < 9; q++) acc[9 * a + q] += wr * t[q];
        }
    }
    for (int ww = 0; ww < 4; ww++) {
        if (w == ww) {
#pragma unroll
            for (int q = 0; q < 72; q++) {
                const double s = ww == 0 ? acc[q] : sacc[64 * q + lane] + acc[q];
                if (ww < 3)
                    sacc[64 * q + lane] = s;
                else
                    part[64 * q + lane] = s;
            }
        }
        __syncthreads();
    }
}

// dense A_c [ld][ld]: the 5^3 grid neighbours of node I, three rows per workgroup; the last
// workgroup writes the identity padding
__global__ __launch_bounds__(128) void k_coarse_assemble(CoarseGrid g, const double* part, int64_t set_part, double* A,
                                                         double* diag, int32_t* bad, const int32_t* active) {
    const int64_t set = blockIdx.y;
    if (active && !active[set]) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) bad[set] = 0;
    part += set * set_part;
    A += set * g.set_A;
    diag += set * (int64_t)g.ld;
    const int I = (int)blockIdx.x, ld = g.ld;
    if (I == g.nodes) {
        for (int r = 3 * g.nodes; r < ld; r++) {
            for (int c = (int)threadIdx.x; c < ld; c += 128) A[(int64_t)r * ld + c] = (c == r) ? 1.0 : 0.0;
            if (threadIdx.x == 0) diag[r] = 1.0;
        }
        return;
    }
    double* rows = A + (int64_t)(3 * I) * ld;
    for (int c = (int)threadIdx.x; c < 3 * ld; c += 128) rows[c] = 0.0;
    __syncthreads();
    const int t = (int)threadIdx.x;
    if (t >= 125) return;
    const int ox = t % 5 - 2, oy = (t / 5) % 5 - 2, oz = t / 25 - 2;
    const int32_t ip = g.ijk[I];
    const int jx = (ip & 1023) + ox, jy = ((ip >> 10) & 1023) + oy, jz = (ip >> 20) + oz;
    if (jx < 0 || jy < 0 || jz < 0 || jx > g.nx || jy > g.ny || jz > g.nz) return;
    const int J = g.map[((int64_t)jz * (g.ny + 1) + jy) * (g.nx + 1) + jx];
    if (J < 0) return;
    double s[9];
#pragma unroll
    for (int q = 0; q < 9; q++) s[q] = 0.0;
    for (int e = g.gptr[I]; e < g.gptr[I + 1]; e++) {
        const int idx = g.gidx[e], a = idx & 7;
        // the chunk's cell is I minus its corner a; lanes count grid nodes from one below the cell
        const int mx = ox + (a & 1) + 1, my = oy + ((a >> 1) & 1) + 1, mz = oz + (a >> 2) + 1;
        if (mx < 0 || my < 0 || mz < 0 || mx > 3 || my > 3 || mz > 3) continue;
        const double* p = part + (int64_t)(idx >> 3) * kGalPart + (int64_t)a * 9 * 64 + (mz * 16 + my * 4 + mx);
#pragma unroll
        for (int q = 0; q < 9; q++) s[q] += p[64 * q];
    }
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) rows[(int64_t)i * ld + 3 * J + j] = s[3 * i + j];
    if (J == I)
#pragma unroll
        for (int i = 0; i < 3; i++) diag[3 * I + i] = s[4 * i];
}

// panel k: every workgroup inverts the diagonal tile, multiplies its tile of the row panel
// by the inverse (U) and saves its tile of the column panel (C)
__global__ __launch_bounds__(256) void k_coarse_panel(int ld, int k, const double* A, int64_t set_A, const double* diag,
                                                      double* U, double* C, double drop, double negative,
                                                      int32_t* bad, const int32_t* active) {
    // The inversion is a chain of 32 dependent steps, bound by latency: the tile stays in
    // registers (four rows per thread), each step publishes the next pivot row and column in
    // the other half of two LDS buffers, so there is one barrier per step, and selects replace
    // branches (13 us per launch; 21 us with the tile in LDS and two barriers, 54 us in one
    // wave without barriers).
    __shared__ double D[kTile][kTile + 1], R[kTile][kTile + 1];
    __shared__ double prow[2][kTile], pcol[2][kTile], dg[kTile];
    const int64_t set = blockIdx.y;
    if (active && !active[set]) return;
    A += set * set_A;
    diag += set * (int64_t)ld + kTile * k;
    U += set * (int64_t)kTile * ld;
    C += set * (int64_t)kTile * ld;
    const int j = (int)blockIdx.x, col = (int)(threadIdx.x & 31), r0 = (int)(threadIdx.x >> 5);
    double v[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const int row = r0 + 8 * m;
        v[m] = A[(int64_t)(kTile * k + row) * ld + kTile * k + col];
        R[row][col] = A[(int64_t)(kTile * k + row) * ld + kTile * j + col];
        C[(int64_t)(kTile * j + row) * kTile + col] = A[(int64_t)(kTile * j + row) * ld + kTile * k + col];
        if (col == 0) pcol[0][row] = v[m];
    }
    if (r0 == 0) {
        prow[0][col] = v[0];
        dg[col] = diag[col];
    }
    __syncthreads();
    bool neg = false;
    for (int p = 0; p < kTile; p++) {
        const int h = p & 1;
        const double piv = prow[h][p], d0 = dg[p], pr = prow[h][col];
        double f[4];
#pragma unroll
        for (int m = 0; m < 4; m++) f[m] = pcol[h][r0 + 8 * m];
        double ip = __builtin_amdgcn_rcp(piv);   // and two Newton steps: a preconditioner's reciprocal
        ip = fma(fma(-piv, ip, 1.0), ip, ip);
        ip = fma(fma(-piv, ip, 1.0), ip, ip);
        ip = piv > drop * d0 ? ip : 0.0;   // 0: the column is dropped
        neg = neg || !(piv >= -negative * fabs(d0));
        const bool pc = col == p;
        const double g = pc ? ip : pr * ip;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const double t = (pc ? 0.0 : v[m]) - f[m] * g;
            v[m] = r0 + 8 * m == p ? g : t;
        }
        const int q = p + 1;
        const double nr = (q >> 3) == 0 ? v[0] : (q >> 3) == 1 ? v[1] : (q >> 3) == 2 ? v[2] : v[3];
        if (r0 == (q & 7)) prow[h ^ 1][col] = nr;
        if (col == q) {
#pragma unroll
            for (int m = 0; m < 4; m++) pcol[h ^ 1][r0 + 8 * m] = v[m];
        }
        __syncthreads();
    }
    if (j == 0 && threadIdx.x == 0 && neg) bad[set] = 1;
#pragma unroll
    for (int m = 0; m < 4; m++) D[r0 + 8 * m][col] = v[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const int row = r0 + 8 * m;
        double s = 0.0;
        if (j == k)
            s = D[row][col];
        else
#pragma unroll 8
            for (int p = 0; p < kTile; p++) s += D[row][p] * R[p][col];
        U[(int64_t)row * ld + kTile * j + col] = s;
    }
}

__global__ __launch_bounds__(256) void k_coarse_update(int ld, int k, double* A, int64_t set_A, const double* U,
                                                       const double* C, const int32_t* active) {
    __shared__ double sc[kTile][kTile + 1], su[kTile][kTile + 1];
    const int64_t set = blockIdx.z;
    if (active && !active[set]) return;
    A += set * set_A;
    U += set * (int64_t)kTile * ld;
    C += set * (int64_t)kTile * ld;
    const int i = (int)blockIdx.y, j = (int)blockIdx.x, col = (int)(threadIdx.x & 31), r0 = (int)(threadIdx.x >> 5);
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const int row = r0 + 8 * m;
        su[row][col] = U[(int64_t)row * ld + kTile * j + col];
        sc[row][col] = C[(int64_t)(kTile * i + row) * kTile + col];
    }
    __syncthreads();
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (i != k)
#pragma unroll 8
        for (int p = 0; p < kTile; p++) {
            const double u = su[p][col];
#pragma unroll
            for (int m = 0; m < 4; m++) s[m] += sc[r0 + 8 * m][p] * u;
        }
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const int row = r0 + 8 * m;
        double* a = A + (int64_t)(kTile * i + row) * ld + kTile * j + col;
        *a = i == k ? su[row][col] : (j == k ? -s[m] : *a - s[m]);
    }
}

// r_c from the restriction partials, eight lanes per component
__global__ __launch_bounds__(256) void k_coarse_rhs(CoarseGrid g, const double* rpart, int64_t set_rpart, double* rc,
                                                    const int32_t* bad, const int32_t* skip) {
    const int64_t set = blockIdx.y;
    if ((skip && skip[set]) || bad[set]) return;
    rpart += set * set_rpart;
    const int d = (int)blockIdx.x * 32 + (int)(threadIdx.x >> 3), l = (int)(threadIdx.x & 7);
    double s = 0.0;
    if (d < 3 * g.nodes) {
        const int I = d / 3, i = d - 3 * I, e1 = g.rptr[I + 1];
        for (int e = g.rptr[I] + l; e < e1; e += 8) s += rpart[3 * (int64_t)e + i];
    }
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) s += __shfl_xor(s, o, 8);
    if (l == 0 && d < 3 * g.nodes) rc[set * (int64_t)g.ld + d] = s;
}

// z_c = A_c^{-1} r_c, one row per wave.  FUSED: every workgroup sums r_c itself, in chunk
// order.  With more than kFusedRhs components that serial sum costs more than a launch of
// its own: 990 components (20k-element LV) 5.9 us fused, 4.7 + 4.7 us with k_coarse_rhs;
// 2,040 (200k) 34 us fused, 9.0 + 4.7 us.  The inverse's row and eight partials at a time are
// requested ahead (7.8 us fused and 11.4 + 4.7 us without).
template <bool FUSED>
__global__ __launch_bounds__(256) void k_coarse_solve(CoarseGrid g, const double* A, const double* rpart,
                                                      int64_t set_rpart, const double* rcg, double* zc,
                                                      const int32_t* bad, const int32_t* skip) {
    extern __shared__ double rc[];   // [ld]
    const int64_t set = blockIdx.y;
    if (skip && skip[set]) return;
    if (bad[set]) {
        if ((int)threadIdx.x < 4 && 4 * blockIdx.x + threadIdx.x < (unsigned)g.ld)
            zc[set * (int64_t)g.ld + 4 * blockIdx.x + threadIdx.x] = 0.0;
        return;
    }
    A += set * g.set_A;
    zc += set * (int64_t)g.ld;
    const int n = 3 * g.nodes;
    // the row of the inverse is requested before r_c is summed
    constexpr int K = (FUSED ? kFusedRhs : kCoarseRows) / 64;
    const int row = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
    const double* a = A + (int64_t)min(row, n - 1) * g.ld;
    double ar[K];
#pragma unroll
    for (int u = 0; u < K; u++) ar[u] = lane + 64 * u < n ? a[lane + 64 * u] : 0.0;
    if (FUSED) {
        rpart += set * set_rpart;
        for (int d = (int)threadIdx.x; d < n; d += 256) {
            const int I = d / 3, i = d - 3 * I, e0 = g.rptr[I], e1 = g.rptr[I + 1];
            double s = 0.0;
            for (int e = e0; e < e1; e += kRhsAhead) {   // loaded together, summed in order
                double v[kRhsAhead];
#pragma unroll
                for (int u = 0; u < kRhsAhead; u++) v[u] = rpart[3 * (int64_t)min(e + u, e1 - 1) + i];
#pragma unroll
                for (int u = 0; u < kRhsAhead; u++)
                    if (e + u < e1) s += v[u];
            }
            rc[d] = s;
        }
    } else {
        for (int d = (int)threadIdx.x; d < n; d += 256) rc[d] = rcg[set * (int64_t)g.ld + d];
    }
    __syncthreads();
    if (row >= n) return;
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < K; u++)
        if (lane + 64 * u < n) s += ar[u] * rc[lane + 64 * u];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) zc[row] = s;
}

}  // namespace

// Background grid: cubic cells as far as the bounding box allows, as many as keep the grid
// nodes next to the mesh within the limit and a quarter of the vertex patches, and no
// smaller than any element's extent (a block row then reaches the grid nodes of its own and
// the adjacent cells only).
int build_coarse(cmg_ctx* c, const double* X, const int32_t* elements) {
    c->coarse = false;
    const int64_t N = c->N, E = c->E;
    const int npe = c->npe;
    // more grid nodes save iterations and cost inversion (2 n^3) and products (8 n^2 bytes):
    // twice as many pay from about 20,000 patches on (1 ms Newmark step, 340 / 680 nodes:
    // 20k-element LV, 4,400 patches, 29.9 / 32.0 ms; 200k-element LV, 39,375 patches,
    // 320.9 / 301.4 ms).  In between either side may be ahead by 5 % (FP64, mixed: 50k elements,
    // 10,610 patches, 58.4 / 57.1 and 36.5 / 38.5 ms; 75k 88.4 / 86.8 and 56.6 / 55.4; 100k, 21,175
    // patches, 129.4 / 115.6 and 77.9 / 81.6)
    const int64_t most = c->sw_P < 20000 ? kCoarseMaxNodes : 2 * kCoarseMaxNodes;
    const int64_t target = std::min(most, c->sw_P / 4);
    if (target < 8) return CMG_SUCCESS;
    double lo[3], hi[3], ext[3] = {0.0, 0.0, 0.0};
    for (int d = 0; d < 3; d++) lo[d] = INFINITY, hi[d] = -INFINITY;
    for (int64_t n = 0; n < N; n++)
        for (int d = 0; d < 3; d++) {
            lo[d] = std::min(lo[d], X[3 * n + d]);
            hi[d] = std::max(hi[d], X[3 * n + d]);
        }
    for (int64_t e = 0; e < E; e++)
        for (int d = 0; d < 3; d++) {
            double a = INFINITY, b = -INFINITY;
            for (int k = 0; k < npe; k++) {
                const double v = X[3 * (int64_t)elements[e * npe + k] + d];
                a = std::min(a, v);
                b = std::max(b, v);
            }
            ext[d] = std::max(ext[d], b - a);
        }
    double len = 0.0;
    for (int d = 0; d < 3; d++) {
        if (!(hi[d] > lo[d]) || !std::isfinite(hi[d] - lo[d]) || !(ext[d] > 0.0)) return CMG_SUCCESS;
        len = std::max(len, hi[d] - lo[d]);
    }
    int n[3] = {1, 1, 1};
    std::vector<int32_t> pos(N);
    std::vector<int32_t> map;
    int64_t nodes = 0;
    auto cell_of = [&](int64_t v, int d) {
        const double u = (X[3 * v + d] - lo[d]) / (hi[d] - lo[d]) * n[d];
        return std::max(0, std::min(n[d] - 1, (int)std::floor(u)));
    };
    // cells per axis for k cells along the longest one; the number of grid nodes next to the mesh
    auto lay = [&](int k) -> bool {
        for (int d = 0; d < 3; d++) {
            const int want = (int)std::ceil((hi[d] - lo[d]) / (len / k) - 1e-9);
            const int most = (int)std::floor((hi[d] - lo[d]) / ext[d] + 1e-9);
            n[d] = std::max(1, std::min({want, most, 1000}));
        }
        map.assign((size_t)(n[0] + 1) * (n[1] + 1) * (n[2] + 1), -1);
        for (int64_t v = 0; v < N; v++) {
            const int x = cell_of(v, 0), y = cell_of(v, 1), z = cell_of(v, 2);
            pos[v] = x | (y << 10) | (z << 20);
            map[((size_t)z * (n[1] + 1) + y) * (n[0] + 1) + x] = 0;   // marks the cell (its lower corner)
        }
        std::vector<int32_t> node(map.size(), -1);
        nodes = 0;
        for (int z = 0; z < n[2]; z++)
            for (int y = 0; y < n[1]; y++)
                for (int x = 0; x < n[0]; x++) {
                    if (map[((size_t)z * (n[1] + 1) + y) * (n[0] + 1) + x] < 0) continue;
                    for (int a = 0; a < 8; a++) {
                        int32_t& m = node[((size_t)(z + (a >> 2)) * (n[1] + 1) + y + ((a >> 1) & 1)) * (n[0] + 1) + x +
                                          (a & 1)];
                        if (m < 0) {
                            m = 0;
                            nodes++;
                        }
                    }
                }
        map.swap(node);
        if (nodes > target) return false;
        for (int64_t e = 0; e < E; e++) {
            int mn[3] = {1024, 1024, 1024}, mx[3] = {0, 0, 0};
            for (int q = 0; q < npe; q++) {
                const int32_t p = pos[elements[e * npe + q]];
                const int v[3] = {p & 1023, (p >> 10) & 1023, p >> 20};
                for (int d = 0; d < 3; d++) mn[d] = std::min(mn[d], v[d]), mx[d] = std::max(mx[d], v[d]);
            }
            for (int d = 0; d < 3; d++)
                if (mx[d] - mn[d] > 1) return false;
        }
        return true;
    };
    int good = 0, bad = 1;
    while (bad <= 512 && lay(bad)) {
        good = bad;
        bad *= 2;
    }
    if (good == 0) return CMG_SUCCESS;
    while (bad - good > 1) {
        const int mid = (good + bad) / 2;
        if (lay(mid))
            good = mid;
        else
            bad = mid;
    }
    if (!lay(good)) return CMG_SUCCESS;
    // grid node ids, cells and fine nodes sorted by cell
    std::vector<int32_t> ijk;
    for (int z = 0, at = 0; z <= n[2]; z++)
        for (int y = 0; y <= n[1]; y++)
            for (int x = 0; x <= n[0]; x++, at++)
                if (map[at] >= 0) {
                    map[at] = (int32_t)ijk.size();
                    ijk.push_back(x | (y << 10) | (z << 20));
                }
    const size_t n_cells_all = (size_t)n[0] * n[1] * n[2];
    auto flat = [&](int32_t p) { return ((size_t)(p >> 20) * n[1] + ((p >> 10) & 1023)) * n[0] + (p & 1023); };
    std::vector<int32_t> cptr(n_cells_all + 1, 0), order(N);
    for (int64_t v = 0; v < N; v++) cptr[flat(pos[v]) + 1]++;
    for (size_t k = 0; k < n_cells_all; k++) cptr[k + 1] += cptr[k];
    {
        std::vector<int32_t> fill(cptr.begin(), cptr.end() - 1);
        for (int64_t v = 0; v < N; v++) order[fill[flat(pos[v])]++] = (int32_t)v;
    }
    std::vector<double> frac((size_t)3 * N);
    for (int64_t v = 0; v < N; v++) {
        const int q[3] = {pos[v] & 1023, (pos[v] >> 10) & 1023, pos[v] >> 20};
        for (int d = 0; d < 3; d++) {
            const double u = (X[3 * v + d] - lo[d]) / (hi[d] - lo[d]) * n[d] - q[d];
            frac[3 * v + d] = std::min(1.0, std::max(0.0, u));
        }
    }
    std::vector<int32_t> cell(N), corner;
    std::vector<int32_t> chunk, rchunk;
    std::vector<std::vector<int32_t>> gin(ijk.size()), rin(ijk.size());
    // Galerkin chunks: about a thousand workgroups, 16 to 256 rows each; restriction chunks:
    // few enough that every workgroup of the coarse solve can sum them all
    const int gal = (int)std::min<int64_t>(256, std::max<int64_t>(16, (N / 1024 + 15) / 16 * 16));
    int32_t n_cells = 0;
    for (int z = 0; z < n[2]; z++)
        for (int y = 0; y < n[1]; y++)
            for (int x = 0; x < n[0]; x++) {
                const int32_t p = x | (y << 10) | (z << 20);
                const int32_t b = cptr[flat(p)], e = cptr[flat(p) + 1];
                if (b == e) continue;
                for (int32_t k = b; k < e; k++) cell[order[k]] = n_cells;
                int32_t ids[8];
                for (int a = 0; a < 8; a++) {
                    ids[a] = map[((size_t)(z + (a >> 2)) * (n[1] + 1) + y + ((a >> 1) & 1)) * (n[0] + 1) + x + (a & 1)];
                    corner.push_back(ids[a]);
                }
                auto split = [&](int rows, std::vector<int32_t>& ch, std::vector<std::vector<int32_t>>& in) {
                    for (int32_t k = b; k < e; k += rows) {
                        for (int a = 0; a < 8; a++) in[ids[a]].push_back((int32_t)(ch.size() / 3) * 8 + a);
                        ch.push_back(n_cells);
                        ch.push_back(k);
                        ch.push_back(std::min<int32_t>(rows, e - k));
                    }
                };
                split(gal, chunk, gin);
                split(1024, rchunk, rin);
                n_cells++;
            }
    auto csr = [](const std::vector<std::vector<int32_t>>& in, std::vector<int32_t>& ptr, std::vector<int32_t>& idx) {
        ptr.assign(1, 0);
        for (const auto& v : in) {
            idx.insert(idx.end(), v.begin(), v.end());
            ptr.push_back((int32_t)idx.size());
        }
    };
    std::vector<int32_t> gptr, gidx, rptr, ridx;
    csr(gin, gptr, gidx);
    csr(rin, rptr, ridx);
    // the restriction writes each partial at its place in its grid node's run
    std::vector<int32_t> rslot(ridx.size());
    for (size_t e = 0; e < ridx.size(); e++) rslot[ridx[e]] = (int32_t)e;
    hipStream_t s = c->stream;
    auto put = [&]() -> int {
        CMG_TRY(upload(c->co_pos, pos.data(), pos.size(), s));
        CMG_TRY(upload(c->co_frac, frac.data(), frac.size(), s));
        CMG_TRY(upload(c->co_order, order.data(), order.size(), s));
        CMG_TRY(upload(c->co_cell, cell.data(), cell.size(), s));
        CMG_TRY(upload(c->co_corner, corner.data(), corner.size(), s));
        CMG_TRY(upload(c->co_chunk, chunk.data(), chunk.size(), s));
        CMG_TRY(upload(c->co_rchunk, rchunk.data(), rchunk.size(), s));
        CMG_TRY(upload(c->co_map, map.data(), map.size(), s));
        CMG_TRY(upload(c->co_ijk, ijk.data(), ijk.size(), s));
        CMG_TRY(upload(c->co_gptr, gptr.data(), gptr.size(), s));
        CMG_TRY(upload(c->co_gidx, gidx.data(), gidx.size(), s));
        CMG_TRY(upload(c->co_rptr, rptr.data(), rptr.size(), s));
        CMG_TRY(upload(c->co_rslot, rslot.data(), rslot.size(), s));
        return CMG_SUCCESS;
    };
    int rc = put();
    CoarseGrid& g = c->co;
    g.nodes = (int)ijk.size();
    g.ld = (3 * g.nodes + kTile - 1) / kTile * kTile;
    g.nx = n[0];
    g.ny = n[1];
    g.nz = n[2];
    g.n_chunk = (int)(chunk.size() / 3);
    g.n_rchunk = (int)(rchunk.size() / 3);
    g.set_A = (int64_t)g.ld * g.ld;
    g.pos = c->co_pos.as<int32_t>();
    g.frac = c->co_frac.as<double>();
    g.order = c->co_order.as<int32_t>();
    g.cell = c->co_cell.as<int32_t>();
    g.corner = c->co_corner.as<int32_t>();
    g.chunk = c->co_chunk.as<int32_t>();
    g.rchunk = c->co_rchunk.as<int32_t>();
    g.map = c->co_map.as<int32_t>();
    g.ijk = c->co_ijk.as<int32_t>();
    g.gptr = c->co_gptr.as<int32_t>();
    g.gidx = c->co_gidx.as<int32_t>();
    g.rptr = c->co_rptr.as<int32_t>();
    g.rslot = c->co_rslot.as<int32_t>();
    if (rc == CMG_SUCCESS && !c->co_buf.alloc(g, 1)) rc = CMG_ERR_NOMEM;
    CMG_HIP_CHECK(hipStreamSynchronize(s));
    if (rc == CMG_ERR_NOMEM) {   // does not fit: the patches alone
        for (DevBuf* b : {&c->co_pos, &c->co_frac, &c->co_order, &c->co_cell, &c->co_corner, &c->co_chunk, &c->co_rchunk,
                          &c->co_map, &c->co_ijk, &c->co_gptr, &c->co_gidx, &c->co_rptr, &c->co_rslot})
            b->release();
        c->co_buf.release();
        (void)hipGetLastError();   // the failed allocation is not an error of the context
        return CMG_SUCCESS;
    }
    CMG_TRY(rc);
    c->coarse = true;
    return CMG_SUCCESS;
}

bool CoarseBuf::alloc(const CoarseGrid& g, int S) {
    return A.alloc((size_t)S * g.set_A * sizeof(double)) && diag.alloc((size_t)S * g.ld * sizeof(double)) &&
           U.alloc((size_t)S * kTile * g.ld * sizeof(double)) && C.alloc((size_t)S * kTile * g.ld * sizeof(double)) &&
           gpart.alloc((size_t)S * g.n_chunk * kGalPart * sizeof(double)) &&
           rpart.alloc((size_t)S * g.n_rchunk * 24 * sizeof(double)) && zc.alloc((size_t)S * g.ld * sizeof(double)) &&
           rc.alloc((size_t)S * g.ld * sizeof(double)) &&
           bad.alloc((size_t)S * sizeof(int32_t));
}

void CoarseBuf::release() {
    for (DevBuf* b : {&A, &diag, &U, &C, &gpart, &rpart, &rc, &zc, &bad}) b->release();
}

void launch_coarse_setup(cmg_ctx* c, const void* vals, const PatchSets& ps) {
    const CoarseGrid& g = c->co;
    CoarseBuf& b = ps.coarse ? *ps.coarse : c->co_buf;
    hipStream_t s = c->stream;
    const int64_t set_part = (int64_t)g.n_chunk * kGalPart;
    const dim3 gg((unsigned)g.n_chunk, ps.S);
    if (c->fp32)
        hipLaunchKernelGGL(k_coarse_galerkin<float>, gg, dim3(256), 0, s, g, c->rowptr.as<int64_t>(),
                           c->colind.as<int32_t>(), c->bcmask.as<uint8_t>(), (const float*)vals, ps.set_vals,
                           b.gpart.as<double>(), set_part, ps.flags);
    else
        hipLaunchKernelGGL(k_coarse_galerkin<double>, gg, dim3(256), 0, s, g, c->rowptr.as<int64_t>(),
                           c->colind.as<int32_t>(), c->bcmask.as<uint8_t>(), (const double*)vals, ps.set_vals,
                           b.gpart.as<double>(), set_part, ps.flags);
    hipLaunchKernelGGL(k_coarse_assemble, dim3((unsigned)g.nodes + 1, ps.S), dim3(128), 0, s, g, b.gpart.as<double>(),
                       set_part, b.A.as<double>(), b.diag.as<double>(), b.bad.as<int32_t>(), ps.flags);
    const unsigned nt = (unsigned)(g.ld / kTile);
    for (unsigned k = 0; k < nt; k++) {
        hipLaunchKernelGGL(k_coarse_panel, dim3(nt, ps.S), dim3(256), 0, s, g.ld, (int)k, b.A.as<double>(), g.set_A,
                           b.diag.as<double>(), b.U.as<double>(), b.C.as<double>(), c->fp32 ? kDrop32 : kDrop64,
                           c->fp32 ? kNegative32 : kNegative64, b.bad.as<int32_t>(), ps.flags);
        hipLaunchKernelGGL(k_coarse_update, dim3(nt, nt, ps.S), dim3(256), 0, s, g.ld, (int)k, b.A.as<double>(),
                           g.set_A, b.U.as<double>(), b.C.as<double>(), ps.flags);
    }
}

void launch_coarse_solve(cmg_ctx* c, const PatchSets& ps) {
    const CoarseGrid& g = c->co;
    CoarseBuf& b = ps.coarse ? *ps.coarse : c->co_buf;
    const bool fused = 3 * g.nodes <= kFusedRhs;
    const int64_t set_rpart = (int64_t)g.n_rchunk * 24;
    const int32_t* bad = b.bad.as<int32_t>();
    const dim3 grid((unsigned)((3 * g.nodes + 3) / 4), ps.S);
    const size_t lds = (size_t)g.ld * sizeof(double);
    if (fused) {
        hipLaunchKernelGGL(k_coarse_solve<true>, grid, dim3(256), lds, c->stream, g, b.A.as<double>(),
                           b.rpart.as<double>(), set_rpart, b.rc.as<double>(), b.zc.as<double>(), bad, ps.flags);
        return;
    }
    hipLaunchKernelGGL(k_coarse_rhs, dim3((unsigned)((3 * g.nodes + 31) / 32), ps.S), dim3(256), 0, c->stream, g,
                       b.rpart.as<double>(), set_rpart, b.rc.as<double>(), bad, ps.flags);
    hipLaunchKernelGGL(k_coarse_solve<false>, grid, dim3(256), lds, c->stream, g, b.A.as<double>(),
                       b.rpart.as<double>(), set_rpart, b.rc.as<double>(), b.zc.as<double>(), bad, ps.flags);
}

}  // namespace cmg
