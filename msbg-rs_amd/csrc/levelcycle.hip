// The structured levels of the multigrid V-cycle (8^3, 4^3 and 2^3 cells per
// listed block, FP32), one pass over memory per full red-black sweep, as on the
// band itself: a listed block's cells and two rings around them go into LDS,
// the first colour is relaxed on the block and on the ring cells that its
// second colour looks at, the second colour on the block.  The first sweep of a
// level starts from x = 0 and reads b alone; the first one after the coarse
// correction adds the interpolated correction as it loads (not on the 2^3
// level, whose second ring interpolates from cells two blocks away).
//
// Operator (unscaled): (A x)_c = dg x_c - the sum of the linked neighbours,
// dg = 1 per face towards a cell of the level, w per face towards an unlisted
// block (x = 0), 0 per face on the domain's bound.  Cells beyond the domain
// and blocks that are not listed hold 0 in every x field.
//
// 8^3 level of a 1024^3 shell (19 M cells), two sweeps before and after the
// correction: 113 us (first half sweep), 7 x 87 (half sweeps), 160 (residual and
// restriction) and 129 (prolongation) as passes of their own; 53 (first sweep),
// 71 (sweep), 63, 127 (prolongation and sweep) and 71 here.  A row of 8 cells
// has 32 bytes and 30 instructions a cell, so it is bound by both.  On bands of
// a few hundred blocks a pass takes its launch, 3 to 4 us, and a level has 5 of
// them instead of 10; there the 2^3 level and the coarsest one are one launch.
#include <algorithm>

#include "coarse_cg.hpp"
#include "poisson.hpp"

namespace msbg {
namespace mg {
namespace {

constexpr int kWg = 256;

// Rows of B cells: the block's B^2, those next to its y and z faces, those one
// further, the four edge rows; lanes per block, and blocks per work-group.
template <int B>
struct Rows {
    static constexpr int kOwn = B * B, kRing = kOwn + 4 * B, kAll = kRing + 4 * B + 4;
    static constexpr int kLanes = B == 8 ? 128 : (B == 4 ? 64 : 32);  // 132, 52, 24 rows
    static constexpr int kBlocks = kWg / kLanes;
    static constexpr int kHalf = B / 2;  // cells of one colour in a row
    // A row in LDS: its colour 0 cells, its colour 1 cells, the cells -2, -1,
    // B, B + 1 (48 bytes for B = 8: 16-byte reads of 8 neighbouring lanes fall
    // on all banks).
    static constexpr int kRow = B + 4;
    static constexpr int kSize = (B + 4) * (B + 4) * kRow;
    static __device__ __forceinline__ int at(int ry, int rz) { return ((rz + 2) * (B + 4) + ry + 2) * kRow; }
    static __device__ __forceinline__ void of(int i, int &ry, int &rz) {
        if (i < kOwn) {
            ry = i % B;
            rz = i / B;
        } else if (i < kAll - 4) {
            const int j = (i - kOwn) % (2 * B), f = (i - kOwn) / (2 * B);
            const int out = f < 2 ? (j < B ? -1 : B) : (j < B ? -2 : B + 1);
            ry = (f & 1) ? j % B : out;
            rz = (f & 1) ? out : j % B;
        } else {
            ry = (i & 1) ? B : -1;
            rz = (i & 2) ? B : -1;
        }
    }
};

template <int B>
__device__ __forceinline__ int side(int c) {
    return c < 0 ? 0 : (c < B ? 1 : 2);
}

struct LevelArgs {
    const PBlock *blocks;
    const int32_t *nb27;
    int n;                  // listed blocks
    int dx, dy, dz;         // the domain in cells of the level
    float w, omega;
    int first;              // colour of the first half
    const float *src, *b;   // x before (not from zero), right-hand side
    float *dst;             // x after
    const float *xc;        // the coarse correction
};

// a or b by value: a conditional on the elements of an array would keep the array in memory
__device__ __forceinline__ float sel(bool c, float a, float b) { return c ? a : b; }

enum { kFromZero = 0, kFromField = 1, kFromCoarse = 2 };

// A row's diagonals: of a middle cell, of cell 0, of the last one inside the
// domain or the block, and their reciprocals (0 for a cell without links).
struct Diag {
    float mid, head, tail, imid, ihead, itail;
};
__device__ __forceinline__ float inverse(float dg) { return dg > 0.0f ? 1.0f / dg : 0.0f; }

// x + omega t / dg, the quotient from the rounded reciprocal and one
// correction step (Markstein), which rounds it correctly.
__device__ __forceinline__ float relaxed(float x, float s, float b, float dg, float inv, float omega) {
    const float num = omega * (b + s - dg * x);
    const float q = num * inv;
    return x + __builtin_fmaf(__builtin_fmaf(-dg, q, num), inv, q);
}

// Everything a lane knows about its row.
template <int B>
struct LaneRow {
    int ry, rz, own, ym, yp, zm, zp;  // places in the tile
    int lim;                          // last x inside the domain
    bool in;                          // inside the domain and a listed block
    int nbl, nb, nbr;                 // the blocks at x - 1, here, x + 1
    Diag dg;
    i64 at;                           // cell 0 within its block

    // coefficient of a face towards block v, at cell `beyond` or not
    static __device__ __forceinline__ float coef(int v, bool beyond, float w) {
        return beyond ? 0.0f : (v >= 0 ? 1.0f : (v == -1 ? w : 0.0f));
    }
    // sum of the coefficients of the y and z faces in block column bx
    __device__ __forceinline__ float faces(const int32_t *N, int bx, int gy, int gz, const LevelArgs &A) const {
        const int by = side<B>(ry), bz = side<B>(rz);
        float f = coef(N[bx + 3 * side<B>(ry - 1) + 9 * bz], false, A.w);
        f += coef(N[bx + 3 * side<B>(ry + 1) + 9 * bz], gy + 1 >= A.dy, A.w);
        f += coef(N[bx + 3 * by + 9 * side<B>(rz - 1)], false, A.w);
        f += coef(N[bx + 3 * by + 9 * side<B>(rz + 1)], gz + 1 >= A.dz, A.w);
        return f;
    }
    __device__ __forceinline__ void set(int i, int k, const PBlock &Bk, const LevelArgs &A) {
        constexpr int h = 16 / B;
        Rows<B>::of(i, ry, rz);
        const int32_t *N = A.nb27 + (i64)k * 27;
        const int gx = Bk.ox / h, gy = Bk.oy / h + ry, gz = Bk.oz / h + rz;
        own = Rows<B>::at(ry, rz);
        ym = Rows<B>::at(ry - 1, rz);
        yp = Rows<B>::at(ry + 1, rz);
        zm = Rows<B>::at(ry, rz - 1);
        zp = Rows<B>::at(ry, rz + 1);
        lim = A.dx - 1 - gx;
        const int row = 3 * side<B>(ry) + 9 * side<B>(rz);
        nbl = N[row];
        nb = N[row + 1];
        nbr = N[row + 2];
        in = nb >= 0 && gy < A.dy && gz < A.dz;
        at = B * ((ry & (B - 1)) + B * (rz & (B - 1)));
    }
    __device__ __forceinline__ void diagonals(int k, const PBlock &Bk, const LevelArgs &A) {
        constexpr int h = 16 / B;
        const int32_t *N = A.nb27 + (i64)k * 27;
        const float yz = faces(N, 1, Bk.oy / h + ry, Bk.oz / h + rz, A);
        const int last = min(lim, B - 1);
        const float l = coef(nbl, false, A.w), r = coef(nbr, lim < B, A.w);
        dg.mid = yz + 2.0f;
        dg.head = yz + l + (last == 0 ? r : 1.0f);
        dg.tail = yz + (last == 0 ? l : 1.0f) + r;
        dg.imid = inverse(dg.mid);
        dg.ihead = inverse(dg.head);
        dg.itail = inverse(dg.tail);
    }
    __device__ __forceinline__ float diag(int x, float &inv) const {
        const bool tail = x == min(lim, B - 1);
        inv = x == 0 ? dg.ihead : sel(tail, dg.itail, dg.imid);
        return x == 0 ? dg.head : sel(tail, dg.tail, dg.mid);
    }
};

// Relaxes the cells 2 i + q of a row (colour `col`) from its other colour o,
// the cells left and right of the row, and the rows around it.
template <int B>
__device__ __forceinline__ void relax_half(float (&c)[B / 2], const float (&o)[B / 2], float left, float right,
                                           const float (&b)[B], const float *s_t, const LaneRow<B> &R, int col, int q,
                                           float omega) {
    constexpr int H = B / 2;
    const float *ym = s_t + R.ym + H * (col ^ 1), *yp = s_t + R.yp + H * (col ^ 1);
    const float *zm = s_t + R.zm + H * (col ^ 1), *zp = s_t + R.zp + H * (col ^ 1);
#pragma unroll
    for (int i = 0; i < H; ++i) {
        const float xl = sel(q, o[i], i ? o[i > 0 ? i - 1 : 0] : left);
        const float xr = sel(q, i < H - 1 ? o[i < H - 1 ? i + 1 : H - 1] : right, o[i]);
        float inv;
        const float dg = R.diag(2 * i + q, inv);
        const float s = ((((xl + xr) + ym[i]) + yp[i]) + zm[i]) + zp[i];
        const float v = relaxed(c[i], s, sel(q, b[2 * i + 1], b[2 * i]), dg, inv, omega);
        c[i] = 2 * i + q <= R.lim ? v : 0.0f;  // cells beyond the domain hold 0
    }
}

// The (B / 2 + 4)^3 cells of the coarser level around the block.
template <int B>
struct Coarse {
    static constexpr int C = B / 2, kEdge = C + 4, kSize = kEdge * kEdge * kEdge;
    static __device__ __forceinline__ void load(float *s_c, int t, int k, const LevelArgs &A) {
        constexpr int C3 = C * C * C;
        if (t >= kEdge * kEdge) return;
        const int y = t % kEdge - 2, z = t / kEdge - 2;
        const int32_t *N = A.nb27 + (i64)k * 27 + 3 * side<C>(y) + 9 * side<C>(z);
        const i64 at = C * ((y & (C - 1)) + C * (z & (C - 1)));
        const int n0 = N[0], n1 = N[1], n2 = N[2];
        float c[kEdge];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            c[x] = n0 >= 0 ? A.xc[(i64)n0 * C3 + at + C - 2 + x] : 0.0f;
            c[C + 2 + x] = n2 >= 0 ? A.xc[(i64)n2 * C3 + at + x] : 0.0f;
        }
#pragma unroll
        for (int x = 0; x < C; ++x) c[x + 2] = n1 >= 0 ? A.xc[(i64)n1 * C3 + at + x] : 0.0f;
#pragma unroll
        for (int x = 0; x < kEdge; ++x) s_c[t * kEdge + x] = c[x];
    }
    // Trilinear correction of the B + 4 cells of row (ry, rz); a partner beyond the domain is the cell itself.
    static __device__ __forceinline__ void row(const float *s_c, int ry, int rz, const PBlock &Bk, const LevelArgs &A,
                                               float (&v)[B + 4]) {
        constexpr int h = 16 / B;
        const int gy = Bk.oy / h, gz = Bk.oz / h, gx = Bk.ox / h;
        const int py = ry >> 1, pz = rz >> 1;
        int qy = py + ((ry & 1) ? 1 : -1), qz = pz + ((rz & 1) ? 1 : -1);
        if (gy + 2 * qy >= A.dy || gy + 2 * qy < 0) qy = py;
        if (gz + 2 * qz >= A.dz || gz + 2 * qz < 0) qz = pz;
#pragma unroll
        for (int yz = 0; yz < 4; ++yz) {
            const int y = (yz & 1) ? qy : py, z = (yz & 2) ? qz : pz;
            const float wyz = ((yz & 1) ? 0.25f : 0.75f) * ((yz & 2) ? 0.25f : 0.75f);
            const float *p = s_c + ((z + 2) * kEdge + y + 2) * kEdge;
            float c[kEdge];
#pragma unroll
            for (int x = 0; x < kEdge; ++x) c[x] = p[x];
#pragma unroll
            for (int i = 0; i < B + 4; ++i) {
                const int own = 1 + (i >> 1), other = (i & 1) ? own + 1 : own - 1;
                const int ox = gx + 2 * (other - 2);
                const float t = __builtin_fmaf(0.25f, sel(ox < 0 || ox >= A.dx, c[own], c[other]), 0.75f * c[own]);
                v[i] = yz ? __builtin_fmaf(wyz, t, v[i]) : wyz * t;
            }
        }
    }
};

template <int B, int FROM>
__global__ __launch_bounds__(kWg) void level_sweep_kernel(LevelArgs A) {
    using RW = Rows<B>;
    constexpr int H = B / 2, B3 = B * B * B, h = 16 / B;
    __shared__ __attribute__((aligned(16))) float s_all[RW::kBlocks * RW::kSize];
    const int sub = threadIdx.x / RW::kLanes, t = threadIdx.x % RW::kLanes;
    float *s_t = s_all + sub * RW::kSize;
    const int kk = xcd_remap(blockIdx.x, gridDim.x) * RW::kBlocks + sub;
    const bool there = kk < A.n;
    const int k = there ? kk : A.n - 1;
    const PBlock Bk = A.blocks[k];
    __shared__ __attribute__((aligned(16))) float s_cs[FROM == kFromCoarse ? RW::kBlocks * Coarse<B>::kSize : 4];
    float *s_c = FROM == kFromCoarse ? s_cs + sub * Coarse<B>::kSize : s_cs;
    if constexpr (FROM == kFromCoarse) Coarse<B>::load(s_c, t, k, A);
    LaneRow<B> R;
    R.set(min(t, RW::kAll - 1), k, Bk, A);
    const bool own = t < RW::kOwn, ring = t < RW::kRing;
    R.in = R.in && ring;
    const int par = (R.ry + R.rz) & 1, first = A.first, q = (par ^ first) & 1;
    float b[B], row[B], c[H], o[H];
    float left[2] = {0.0f, 0.0f}, right[2] = {0.0f, 0.0f};  // cells -2, -1 and B, B + 1
    float b_end = 0.0f, dg_end = 0.0f;
#pragma unroll
    for (int i = 0; i < B; ++i) b[i] = row[i] = 0.0f;
    if (R.nb >= 0 && ring)
#pragma unroll
        for (int i = 0; i < B; ++i) b[i] = A.b[(i64)R.nb * B3 + R.at + i];
    // the end cell of colour `first`: -1 (q = 1) or B (q = 0)
    const bool end_in = own && R.in && (q ? R.nbl >= 0 : R.nbr >= 0 && B <= R.lim);
    if (end_in) b_end = A.b[(i64)(q ? R.nbl : R.nbr) * B3 + R.at + (q ? B - 1 : 0)];
    if constexpr (FROM != kFromZero) {
        if (R.nb >= 0)
#pragma unroll
            for (int i = 0; i < B; ++i) row[i] = A.src[(i64)R.nb * B3 + R.at + i];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (R.nbl >= 0) left[i] = A.src[(i64)R.nbl * B3 + R.at + B - 2 + i];
            if (R.nbr >= 0) right[i] = A.src[(i64)R.nbr * B3 + R.at + i];
        }
        if constexpr (FROM == kFromCoarse) {
            __syncthreads();
            float v[B + 4];
            Coarse<B>::row(s_c, R.ry, R.rz, Bk, A, v);
            const bool inside = Bk.oy / h + R.ry < A.dy && Bk.oz / h + R.rz < A.dz;
#pragma unroll
            for (int i = 0; i < B; ++i)
                if (inside && R.nb >= 0 && i <= R.lim) row[i] += v[i + 2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (inside && R.nbl >= 0) left[i] += v[i];
                if (inside && R.nbr >= 0 && B + i <= R.lim) right[i] += v[B + 2 + i];
            }
        }
        // the edge rows of the 8^3 level, beyond its lanes
        if (RW::kAll > RW::kLanes && t < RW::kAll - RW::kLanes) {
            LaneRow<B> E;
            E.set(RW::kLanes + t, k, Bk, A);
            float x[B];
#pragma unroll
            for (int i = 0; i < B; ++i) x[i] = E.nb >= 0 ? A.src[(i64)E.nb * B3 + E.at + i] : 0.0f;
            if constexpr (FROM == kFromCoarse) {
                float v[B + 4];
                Coarse<B>::row(s_c, E.ry, E.rz, Bk, A, v);
                const bool inside = Bk.oy / h + E.ry < A.dy && Bk.oz / h + E.rz < A.dz;
#pragma unroll
                for (int i = 0; i < B; ++i)
                    if (inside && E.nb >= 0 && i <= E.lim) x[i] += v[i + 2];
            }
            const int pe = (E.ry + E.rz) & 1;
#pragma unroll
            for (int i = 0; i < B; ++i) s_t[E.own + H * ((pe + i) & 1) + i / 2] = x[i];
        }
    }
    if (R.in) {
        R.diagonals(k, Bk, A);
        if (end_in) {
            const int32_t *N = A.nb27 + (i64)k * 27;
            dg_end = R.faces(N, q ? 0 : 2, Bk.oy / h + R.ry, Bk.oz / h + R.rz, A) + (q || B < R.lim ? 2.0f : 1.0f);
        }
    }
    if constexpr (FROM == kFromZero) {
        // the first colour from x = 0
#pragma unroll
        for (int i = 0; i < H; ++i) {
            float inv;
            const float dg = R.in ? R.diag(2 * i + q, inv) : (inv = 0.0f);
            const float v = relaxed(0.0f, 0.0f, sel(q, b[2 * i + 1], b[2 * i]), dg, inv, A.omega);
            c[i] = R.in && 2 * i + q <= R.lim ? v : 0.0f;
            o[i] = 0.0f;
        }
        if (end_in) {
            const float v = relaxed(0.0f, 0.0f, b_end, dg_end, inverse(dg_end), A.omega);
            left[1] = q ? v : 0.0f;
            right[0] = q ? 0.0f : v;
        }
        if (ring || t < RW::kAll)
#pragma unroll
            for (int i = 0; i < H; ++i) s_t[R.own + H * first + i] = c[i];
        __syncthreads();
    } else {
#pragma unroll
        for (int i = 0; i < H; ++i) {
            c[i] = sel(q, row[2 * i + 1], row[2 * i]);
            o[i] = sel(q, row[2 * i], row[2 * i + 1]);
        }
        if (t < RW::kAll) {
#pragma unroll
            for (int i = 0; i < H; ++i) {
                s_t[R.own + H * first + i] = c[i];
                s_t[R.own + H * (first ^ 1) + i] = o[i];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                s_t[R.own + B + i] = left[i];
                s_t[R.own + B + 2 + i] = right[i];
            }
        }
        __syncthreads();
        if (R.in) {
            const float l = left[1], r = right[0];
            if (end_in) {
                const int e = B + (q ? 1 : 2);
                const float xl = sel(q, left[0], o[H - 1]), xr = sel(q, o[0], right[1]);
                const float s = ((((xl + xr) + s_t[R.ym + e]) + s_t[R.yp + e]) + s_t[R.zm + e]) + s_t[R.zp + e];
                const float v = relaxed(sel(q, left[1], right[0]), s, b_end, dg_end, inverse(dg_end), A.omega);
                left[1] = sel(q, v, left[1]);
                right[0] = sel(q, right[0], v);
            }
            relax_half<B>(c, o, l, r, b, s_t, R, first, q, A.omega);
            // other lanes look at this row's other colour only until the next barrier
#pragma unroll
            for (int i = 0; i < H; ++i) s_t[R.own + H * first + i] = c[i];
        }
        __syncthreads();
    }
    if (!own || !there) return;
    if (R.in) relax_half<B>(o, c, left[1], right[0], b, s_t, R, first ^ 1, q ^ 1, A.omega);
    float *out = A.dst + (i64)k * B3 + R.at;
#pragma unroll
    for (int i = 0; i < H; ++i) {
        out[2 * i] = R.in ? sel(q, o[i], c[i]) : 0.0f;
        out[2 * i + 1] = R.in ? sel(q, c[i], o[i]) : 0.0f;
    }
}

// bc = 0.5 * the sum of the 8 children's residuals b - A x (pairs along x, then
// y, then z), into the level of B / 2 cells per block edge.
template <int B>
__global__ __launch_bounds__(kWg) void level_restrict_kernel(LevelArgs A, float *__restrict__ bc) {
    using RW = Rows<B>;
    constexpr int H = B / 2, B3 = B * B * B, C3 = B3 / 8;
    constexpr int kStep = B + 4;  // floats per row: 48 bytes for B = 8
    __shared__ __attribute__((aligned(16))) float s_all[RW::kBlocks * RW::kSize];
    const int sub = threadIdx.x / RW::kLanes, t = threadIdx.x % RW::kLanes;
    float *s_t = s_all + sub * RW::kSize;
    const int kk = xcd_remap(blockIdx.x, gridDim.x) * RW::kBlocks + sub;
    const bool there = kk < A.n;
    const int k = there ? kk : A.n - 1;
    const PBlock Bk = A.blocks[k];
    LaneRow<B> R;
    R.set(min(t, RW::kRing - 1), k, Bk, A);
    const bool own = t < RW::kOwn;
    float x[B], b[B], left = 0.0f, right = 0.0f;
#pragma unroll
    for (int i = 0; i < B; ++i) {
        x[i] = R.nb >= 0 ? A.src[(i64)R.nb * B3 + R.at + i] : 0.0f;
        b[i] = 0.0f;
    }
    if (own) {
#pragma unroll
        for (int i = 0; i < B; ++i) b[i] = A.b[(i64)k * B3 + R.at + i];
        if (R.nbl >= 0) left = A.src[(i64)R.nbl * B3 + R.at + B - 1];
        if (R.nbr >= 0) right = A.src[(i64)R.nbr * B3 + R.at];
        if (R.in) R.diagonals(k, Bk, A);
    }
#pragma unroll
    for (int i = 0; i < B; ++i) s_t[R.own + i] = x[i];
    __syncthreads();
    float p[H];
#pragma unroll
    for (int i = 0; i < H; ++i) p[i] = 0.0f;
    if (own && R.in) {
        float r[B];
#pragma unroll
        for (int i = 0; i < B; ++i) {
            const float xl = i ? x[i > 0 ? i - 1 : 0] : left, xr = i < B - 1 ? x[i < B - 1 ? i + 1 : B - 1] : right;
            const float s = ((((xl + xr) + s_t[R.ym + i]) + s_t[R.yp + i]) + s_t[R.zm + i]) + s_t[R.zp + i];
            float inv;
            const float dg = R.diag(i, inv);
            r[i] = i <= R.lim ? b[i] + s - dg * x[i] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < H; ++i) p[i] = r[2 * i] + r[2 * i + 1];
    }
    __syncthreads();
    if (own)
#pragma unroll
        for (int i = 0; i < H; ++i) s_t[t * H + i] = p[i];
    __syncthreads();
    if (!there || t >= C3) return;
    const int ux = t % H, uy = (t / H) % H, uz = t / (H * H);
    const float *s = s_t + (2 * uy + B * 2 * uz) * H + ux;
    bc[(i64)k * C3 + t] = 0.5f * ((s[0] + s[H]) + (s[B * H] + s[(B + 1) * H]));
}

// The 2^3 level and the coarsest one (a cell per block) in one work-group, on
// bands of at most kCoarseMax blocks: nu sweeps from x = 0, the residual's sum,
// the coarsest level's solution, its interpolation and nu sweeps back.  A lane
// holds up to kTailRows rows of 2 cells (4 lanes to a block), one cell of each
// colour, in registers with everything that it knows of them; other lanes see x
// in LDS, so a half sweep is 5 LDS reads a row and one barrier.
// What bounds it is latency, barriers and the iterations of the coarsest level's
// solve, on one CU; seven launches (three sweeps of 4.3 us, 3.5, 2.9 and 4.6 us
// for the first sweep, the restriction and the interpolation, 13 to 27 us for
// the solve) took 37 us on 144 blocks, 41 on 450 and 51 on 704, it takes 20, 36
// and 45.  As many lanes as there are rows: with a lane per block, 300 blocks
// took 34 us instead of 31.
constexpr int kTailRows = 4, kTailLanes = kCoarseMax;
constexpr int kTailNone = 8 * kCoarseMax;  // two cells that hold 0

__global__ __launch_bounds__(kTailLanes) void level_tail_kernel(LevelArgs A, CoarseArgs C, int nu) {
    __shared__ float s_x[8 * kCoarseMax + 2];
    __shared__ float s_c[kCoarseMax];
    __shared__ int32_t s_nb[6 * kCoarseMax];  // the coarsest level's links, loaded with everything else
    __shared__ float s_cf[6 * kCoarseMax];
    __shared__ CoarseShared S;
    const int t = threadIdx.x, lanes = blockDim.x, rows = 4 * A.n;
    const int per = (rows + lanes - 1) / lanes;
    float x[kTailRows][2], b[kTailRows][2], dg[kTailRows][2], inv[kTailRows][2];
    int at[kTailRows], l[kTailRows], r[kTailRows], ym[kTailRows], yp[kTailRows], zm[kTailRows], zp[kTailRows];
    bool live[kTailRows][2];
    const int ry = t & 1, rz = (t >> 1) & 1, par = ry ^ rz;  // lanes is a multiple of 4
    for (int i = t; i < 8 * A.n; i += lanes) s_x[i] = 0.0f;
    if (t < 2) s_x[kTailNone + t] = 0.0f;
    for (int i = t; i < 6 * C.n; i += lanes) {
        s_nb[i] = C.nb[i];
        s_cf[i] = C.cf[i];
    }
#pragma unroll
    for (int j = 0; j < kTailRows; ++j) {
        const int i = t + j * lanes, k = i >> 2;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            x[j][e] = b[j][e] = dg[j][e] = inv[j][e] = 0.0f;
            live[j][e] = false;
        }
        at[j] = l[j] = r[j] = ym[j] = yp[j] = zm[j] = zp[j] = kTailNone;
        if (i >= rows) continue;
        const PBlock Bk = A.blocks[k];
        LaneRow<2> R;
        R.set(i & 3, k, Bk, A);
        const int32_t *N = A.nb27 + (i64)k * 27;
        const int vym = ry ? k : N[10], vyp = ry ? N[16] : k, vzm = rz ? k : N[4], vzp = rz ? N[22] : k;
        const int row = 2 * ry + 4 * rz;
        at[j] = 8 * k + row;
        if (R.nbl >= 0) l[j] = 8 * R.nbl + row + 1;
        if (R.nbr >= 0) r[j] = 8 * R.nbr + row;
        if (vym >= 0) ym[j] = 8 * vym + (row ^ 2);
        if (vyp >= 0) yp[j] = 8 * vyp + (row ^ 2);
        if (vzm >= 0) zm[j] = 8 * vzm + (row ^ 4);
        if (vzp >= 0) zp[j] = 8 * vzp + (row ^ 4);
        if (!R.in) continue;
        R.diagonals(k, Bk, A);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            b[j][e] = A.b[(i64)at[j] + e];
            dg[j][e] = R.diag(e, inv[j][e]);
            live[j][e] = e <= R.lim;
        }
    }
    __syncthreads();
    const auto neighbours = [&](int j, int e) {
        const float xl = sel(e, x[j][0], s_x[l[j]]), xr = sel(e, s_x[r[j]], x[j][1]);
        return ((((xl + xr) + s_x[ym[j] + e]) + s_x[yp[j] + e]) + s_x[zm[j] + e]) + s_x[zp[j] + e];
    };
    // the cells of one colour look at the other colour alone
    const auto half = [&](int colour) {
        const int e = par ^ colour;
#pragma unroll
        for (int j = 0; j < kTailRows; ++j) {
            if (j >= per || t + j * lanes >= rows) continue;
            const float v = relaxed(sel(e, x[j][1], x[j][0]), neighbours(j, e), sel(e, b[j][1], b[j][0]),
                                    sel(e, dg[j][1], dg[j][0]), sel(e, inv[j][1], inv[j][0]), A.omega);
            if (e ? live[j][1] : live[j][0]) {
                x[j][0] = sel(e, x[j][0], v);
                x[j][1] = sel(e, v, x[j][1]);
                s_x[at[j] + e] = v;
            }
        }
        __syncthreads();
    };
    for (int it = 0; it < nu; ++it) {
        half(0);
        half(1);
    }
#pragma unroll
    for (int j = 0; j < kTailRows; ++j) {
        const int i = t + j * lanes;
        float p = 0.0f;
        if (i < rows) {
            float res[2];
#pragma unroll
            for (int e = 0; e < 2; ++e)
                res[e] = live[j][e] ? b[j][e] + neighbours(j, e) - dg[j][e] * x[j][e] : 0.0f;
            p = res[0] + res[1];
        }
        p += __shfl_xor(p, 1);
        p += __shfl_xor(p, 2);
        if (i < rows && (i & 3) == 0) s_c[i >> 2] = 0.5f * p;
    }
    __syncthreads();
    const float xc = (float)coarse_cg(C, s_nb, s_cf, t < C.n ? s_c[t] : 0.0f, S);
    __syncthreads();
    if (t < C.n) s_c[t] = xc;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kTailRows; ++j) {
        const int i = t + j * lanes, k = i >> 2;
        if (i >= rows) continue;
        const int32_t *N = A.nb27 + (i64)k * 27;
        // towards the block on the cell's side; one beyond the domain is the cell itself
        int dy = ry ? 3 : -3, dz = rz ? 9 : -9;
        dy = N[13 + dy] == -2 ? 0 : dy;
        dz = N[13 + dz] == -2 ? 0 : dz;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            if (!live[j][e]) continue;
            const int dx = N[13 + (e ? 1 : -1)] == -2 ? 0 : (e ? 1 : -1);
            float v = 0.0f;
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) {
                const int nb = N[13 + ((kk & 1) ? dx : 0) + ((kk & 2) ? dy : 0) + ((kk & 4) ? dz : 0)];
                const float wt = ((kk & 1) ? 0.25f : 0.75f) * ((kk & 2) ? 0.25f : 0.75f) * ((kk & 4) ? 0.25f : 0.75f);
                if (nb >= 0) v += wt * s_c[nb];
            }
            x[j][e] += v;
            s_x[at[j] + e] = x[j][e];
        }
    }
    __syncthreads();
    for (int it = 0; it < nu; ++it) {
        half(1);
        half(0);
    }
#pragma unroll
    for (int j = 0; j < kTailRows; ++j)
        if (t + j * lanes < rows) {
            A.dst[(i64)at[j]] = x[j][0];
            A.dst[(i64)at[j] + 1] = x[j][1];
        }
}

template <int B>
void sweep(hipStream_t s, const LevelArgs &A, int from) {
    const int g = (A.n + Rows<B>::kBlocks - 1) / Rows<B>::kBlocks;
    if (from == kFromZero)
        level_sweep_kernel<B, kFromZero><<<g, kWg, 0, s>>>(A);
    else if (from == kFromField)
        level_sweep_kernel<B, kFromField><<<g, kWg, 0, s>>>(A);
    else if constexpr (B > 2)
        level_sweep_kernel<B, kFromCoarse><<<g, kWg, 0, s>>>(A);
}

void sweep(int B, hipStream_t s, const LevelArgs &A, int from) {
    if (B == 8)
        sweep<8>(s, A, from);
    else if (B == 4)
        sweep<4>(s, A, from);
    else
        sweep<2>(s, A, from);
}

LevelArgs args_of(const msbg_poisson *p, const int32_t *nb27, int B, float w, float omega, const float *b) {
    const int h = 16 / B;
    LevelArgs A{};
    A.blocks = p->d_blocks;
    A.nb27 = nb27;
    A.n = (int)p->n_active;
    A.dx = (p->dom.sx + h - 1) / h;
    A.dy = (p->dom.sy + h - 1) / h;
    A.dz = (p->dom.sz + h - 1) / h;
    A.w = w;
    A.omega = omega;
    A.b = b;
    return A;
}

}  // namespace

void level_before(const msbg_poisson *p, hipStream_t s, const int32_t *nb27, int B, float w, float omega, int nu,
                  float *x, float *y, const float *b, float *bc) {
    LevelArgs A = args_of(p, nb27, B, w, omega, b);
    A.first = 0;
    A.dst = x;
    sweep(B, s, A, kFromZero);
    for (int i = 1; i < nu; ++i) {
        A.src = A.dst;
        A.dst = A.src == x ? y : x;
        sweep(B, s, A, kFromField);
    }
    A.src = A.dst;
    const int per = B == 8 ? Rows<8>::kBlocks : (B == 4 ? Rows<4>::kBlocks : Rows<2>::kBlocks);
    const int g = (A.n + per - 1) / per;
    if (B == 8)
        level_restrict_kernel<8><<<g, kWg, 0, s>>>(A, bc);
    else if (B == 4)
        level_restrict_kernel<4><<<g, kWg, 0, s>>>(A, bc);
    else
        level_restrict_kernel<2><<<g, kWg, 0, s>>>(A, bc);
}

const float *level_after(const msbg_poisson *p, hipStream_t s, const int32_t *nb27, int B, float w, float omega, int nu,
                         float *x, float *y, const float *b, const float *xc) {
    LevelArgs A = args_of(p, nb27, B, w, omega, b);
    A.first = 1;
    A.xc = xc;
    A.src = level_field(x, y, nu);
    for (int i = 0; i < nu; ++i) {
        A.dst = A.src == x ? y : x;
        sweep(B, s, A, i == 0 && xc ? kFromCoarse : kFromField);
        A.src = A.dst;
    }
    return A.src;
}

void level_tail(const msbg_poisson *p, hipStream_t s, const int32_t *nb27, float w, float omega, int nu,
                const CoarseArgs &cg, const float *b, float *x) {
    LevelArgs A = args_of(p, nb27, 2, w, omega, b);
    A.dst = x;
    // a row a lane up to 256 blocks, whole waves
    const int lanes = std::min(kTailLanes, (4 * A.n + 63) / 64 * 64);
    level_tail_kernel<<<1, lanes, 0, s>>>(A, cg, nu);
}

}  // namespace mg
}  // namespace msbg
