// Device state of one BiCGStab solve (bicgstab.hip), shared with the patch kernel that
// forms s = r - alpha v on the fly (schwarz.hip).  Internal.
#pragma once

#include "cmg_internal.h"

namespace cmg {

constexpr int kBicgConverged = 1, kBicgBreakdown = 2, kBicgMaxit = 3;

// fin ends the iterations, done the updates that belong to the one at hand; *_next are what the
// next iteration starts from.  No launch reads a flag that it may set: the first product reads fin
// and sets done, the launch that forms alpha the same, the second product reads done
// and sets fin, and the update too.
struct BicgScalars {
    double rho, rho_next, alpha, tol2;
    int32_t fin, done, it, it_next, maxit;
    uint32_t seq;
};

// pinned host memory: solve number, iteration and fin in one word; the true residual's
// square and its target of the last (re)start
struct BicgHost {
    unsigned long long word;
    double rr, tol2;
};

struct BicgVec {
    double *x, *r, *rh, *p, *v, *t, *ph, *sh;
    BicgScalars* sc;
    BicgHost* host;
};

#ifdef __HIPCC__
__device__ __forceinline__ void bicg_publish(const BicgScalars* sc, BicgHost* host, int it, int fin) {
    const unsigned long long word =
        ((unsigned long long)sc->seq << 40) | ((unsigned long long)(unsigned)it << 8) | (unsigned)fin;
    __hip_atomic_store(&host->word, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr int kBicgPartials = 1024;   // partial sums that their consumers add up themselves

// alpha = rho / (r^, v) from nb <= kBicgPartials partials, in every workgroup of 256 threads; the
// first one stores it, or ends the solve when the product is zero or not finite (false everywhere)
__device__ __forceinline__ bool bicg_alpha(const BicgVec& k, const double* part, int nb, double* sh, double& alpha) {
    double d = 0.0;
#pragma unroll
    for (int j = 0; j < kBicgPartials; j += 256) d += j + (int)threadIdx.x < nb ? part[j + threadIdx.x] : 0.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) d += __shfl_xor(d, o, 64);
    if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = d;
    __syncthreads();
    d = sh[0] + sh[1] + sh[2] + sh[3];
    const bool ok = fabs(d) > 0.0 && isfinite(d);
    alpha = ok ? k.sc->rho / d : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (ok) {
            k.sc->alpha = alpha;
        } else {
            k.sc->done = 1;
            bicg_publish(k.sc, k.host, k.sc->it, kBicgBreakdown);
        }
    }
    return ok;
}
#endif

}  // namespace cmg
