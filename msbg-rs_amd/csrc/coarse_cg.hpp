// The coarsest multigrid level (<= kCoarseMax cells) by conjugate gradients in
// FP64 within one work-group.
#pragma once

#include "poisson.hpp"

namespace msbg {
namespace mg {

constexpr int kCoarseMax = 1024;  // cells of the coarsest level (one FP64 CG work-group)
constexpr int kCgMaxIter = 1000;
constexpr double kCgTol = 1e-6;  // relative; the V-cycle needs far less

// A cell list: n cells, their links ([n][6], -1 none) with coefficients, diagonals, and where
// a component is singular (n_sing > 0) each cell's component and which components are.
struct CoarseArgs {
    int n, n_comp, n_sing;
    const int32_t *nb;
    const float *cf, *diag;
    const int16_t *comp;
    const uint8_t *sing;
};

struct CoarseShared {
    double p[kCoarseMax], mean[kCoarseMax];
    double red[2][kCoarseMax / 64];
    int16_t comp[kCoarseMax];
};

// v + the value of the lane that a data-parallel move within 16 lanes names
template <int MOVE>
__device__ __forceinline__ double plus_moved(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, MOVE, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), MOVE, 0xf, 0xf, true);
    return v + __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ double of_lane(double v, int lane) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// Sum over the work-group's first `waves` waves (v is 0 in the others) in a
// fixed order (16 lanes by moves, which pass no LDS; the wave's four groups;
// the waves in order); every thread receives the same value.  One barrier: a
// caller's next sum goes through another s_red, and the one after that may use
// this one again.
__device__ __forceinline__ double wg_sum(double v, double *s_red, int waves) {
    v = plus_moved<0xb1>(v);   // lane ^ 1
    v = plus_moved<0x4e>(v);   // lane ^ 2
    v = plus_moved<0x141>(v);  // the other 4 of 8 (mirrored)
    v = plus_moved<0x140>(v);  // the other 8 of 16 (mirrored)
    const double sum = (of_lane(v, 0) + of_lane(v, 16)) + (of_lane(v, 32) + of_lane(v, 48));
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = sum;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < waves; ++w) t += s_red[w];
    return t;
}

// Removes, on each singular component (no Dirichlet coupling: the constants
// are its null space), the component's mean from v.  Thread c < n_comp sums
// component c in cell order (deterministic).
__device__ __forceinline__ void project_singular(double &v, bool in, int n, int n_comp, const int16_t *s_comp,
                                 const uint8_t *__restrict__ sing, double *s_val, double *s_mean) {
    const int t = threadIdx.x;
    s_val[t] = in ? v : 0.0;
    __syncthreads();
    if (t < n_comp) {
        double sum = 0.0;
        int cnt = 0;
        if (sing[t])
            for (int i = 0; i < n; ++i)
                if (s_comp[i] == t) {
                    sum += s_val[i];
                    ++cnt;
                }
        s_mean[t] = cnt ? sum / cnt : 0.0;
    }
    __syncthreads();
    if (in && sing[s_comp[t]]) v -= s_mean[s_comp[t]];
    __syncthreads();
}

// Conjugate gradients, one cell per thread (the group holds at least the
// cells), until ||r|| <= kCgTol ||b|| or kCgMaxIter iterations (the loop
// condition is the same on every thread, so every barrier is reached by the
// whole group); thread t < n receives x of cell t.  On a component without
// Dirichlet coupling the operator is singular: b is projected onto its range
// first and x onto the zero-mean space after, so an inconsistent right-hand
// side (or rounding) cannot drive x along the constants.  A chain of
// latencies: 3 barriers, 6 LDS reads and two sums an iteration; 20.2 us became
// 16.5 under a shell of 1,104 blocks with one barrier a sum, its adds by moves, and no branch
// around an absent link.
// A caller may hold the links in LDS (nb and cf there instead of in A).
__device__ __forceinline__ double coarse_cg(const CoarseArgs &A, const int32_t *nb, const float *cf, float b,
                                            CoarseShared &S) {
    const int t = threadIdx.x, n = A.n, waves = (n + 63) >> 6;
    const bool in = t < n;
    // an absent link reads the cell itself, times 0
    int32_t q[6] = {t, t, t, t, t, t};
    double c[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    double dg = 0.0, r = 0.0;
    if (in) {
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            const int32_t j = nb[t * 6 + f];
            q[f] = j >= 0 ? j : t;
            c[f] = j >= 0 ? (double)cf[t * 6 + f] : 0.0;
        }
        dg = (double)A.diag[t];
        r = (double)b;
    }
    if (A.n_sing > 0) {
        S.comp[t] = in ? A.comp[t] : (int16_t)0;
        project_singular(r, in, n, A.n_comp, S.comp, A.sing, S.p, S.mean);
    }
    double xi = 0.0, p = r;
    double rr = wg_sum(r * r, S.red[1], waves);
    const double stop = kCgTol * kCgTol * rr;
    for (int it = 0; it < kCgMaxIter && rr > stop; ++it) {
        S.p[t] = p;
        __syncthreads();
        double ap = dg * p;
#pragma unroll
        for (int f = 0; f < 6; ++f) ap -= c[f] * S.p[q[f]];
        const double pap = wg_sum(p * ap, S.red[0], waves);
        if (!(pap > 0.0)) break;
        const double alpha = rr / pap;
        xi += alpha * p;
        r -= alpha * ap;
        const double rr1 = wg_sum(r * r, S.red[1], waves);
        p = r + (rr1 / rr) * p;
        rr = rr1;
    }
    if (A.n_sing > 0) project_singular(xi, in, n, A.n_comp, S.comp, A.sing, S.p, S.mean);
    return xi;
}

}  // namespace mg
}  // namespace msbg
