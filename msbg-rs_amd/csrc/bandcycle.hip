// The band level of a multigrid V-cycle, one pass over memory per full
// red-black sweep.
//
// A half sweep reads the error e and its right-hand side rt and writes e, and
// does so at the rate of a copy on bands beyond the caches: what it costs is
// its bytes (on small bands its launch).  So a work-group takes one listed
// block with two rings of cells around it into LDS and runs both colours: the
// first colour on the block and the ring of cells its second colour looks at,
// the second on the block.  The ring is computed twice (768 cells beside the
// block's 4,096) from the same values in the same order as its own block
// computes it, so a sweep has the bits of two half sweeps in place.  It reads
// one field and writes another (e and the residual field take turns).
// Into the sweeps beside the transfers go the passes around them: the first
// sweep takes the scaled residual as its right-hand side and starts from e = 0,
// the first one after the coarse correction adds the interpolated correction
// as it loads, and the last one adds e to the iterate instead of storing it.
//
// 153 M cells of FP16 (a shell in 1024^3), two sweeps before and after the
// coarse correction, one cycle's band level: scaling 215 us, 7 half sweeps of
// 216, residual 330, restriction 130, prolongation 176 and update 262 as passes
// of their own; 284 (scaling and first sweep), 265 (sweep), 163 (residual and
// restriction), 405 (prolongation and sweep), 412 (sweep and update) here.  The
// last takes the time of its 14 bytes a cell, the restriction that of its 4.5;
// the others wait for their two dependent loads with 6 work-groups a CU.
#include "poisson.hpp"

namespace msbg {
namespace mg {
namespace {

// Two x-adjacent cells as stored.
template <int ST>
struct Duo {
    using T = uint32_t;
    using S = Sto<ST>;
    static __device__ __forceinline__ float lo(T w) { return S::lo(w); }
    static __device__ __forceinline__ float hi(T w) { return S::hi(w); }
    static __device__ __forceinline__ T make(float a, float b) { return (uint32_t)S::cv(a) | (uint32_t)S::cv(b) << 16; }
    static __device__ __forceinline__ T zero() { return 0u; }
};
template <>
struct Duo<MSBG_STORAGE_F32> {
    using T = float2;
    static __device__ __forceinline__ float lo(T w) { return w.x; }
    static __device__ __forceinline__ float hi(T w) { return w.y; }
    static __device__ __forceinline__ T make(float a, float b) { return make_float2(a, b); }
    static __device__ __forceinline__ T zero() { return make_float2(0.0f, 0.0f); }
};

// The 8 duos of a row, 16 bytes at a time.
template <int ST>
__device__ __forceinline__ void load8(const typename Duo<ST>::T *p, typename Duo<ST>::T (&w)[8]) {
    constexpr int K = 16 / (int)sizeof(w[0]);
#pragma unroll
    for (int i = 0; i < 8; i += K) {
        const uint4 q = *reinterpret_cast<const uint4 *>(p + i);
        __builtin_memcpy(&w[i], &q, 16);
    }
}
template <int ST>
__device__ __forceinline__ void store8(typename Duo<ST>::T *p, const typename Duo<ST>::T (&w)[8]) {
    constexpr int K = 16 / (int)sizeof(w[0]);
#pragma unroll
    for (int i = 0; i < 8; i += K) {
        uint4 q;
        __builtin_memcpy(&q, &w[i], 16);
        *reinterpret_cast<uint4 *>(p + i) = q;
    }
}

// The 8 cells of one colour of a row, x ascending.  par: parity of the row's
// cell 0, so colour c has the cells 2 i + (par ^ c).
template <int ST>
struct Half {
    uint32_t w[4];
    __device__ __forceinline__ float at(int i) const { return (i & 1) ? Sto<ST>::hi(w[i >> 1]) : Sto<ST>::lo(w[i >> 1]); }
    __device__ __forceinline__ void set2(int i, float a, float b) { w[i >> 1] = Duo<ST>::make(a, b); }  // cells i, i + 1
    __device__ __forceinline__ void set(int i, float v) {
        const uint32_t h = Sto<ST>::cv(v);
        w[i >> 1] = (i & 1) ? (w[i >> 1] & 0xffffu) | h << 16 : (w[i >> 1] & 0xffff0000u) | h;
    }
    // The odd (q = 1) or even cells of a row.
    static __device__ __forceinline__ Half of(const uint32_t (&d)[8], int q) {
        const uint32_t sel = q ? 0x07060302u : 0x05040100u;
        Half h;
#pragma unroll
        for (int j = 0; j < 4; ++j) h.w[j] = __builtin_amdgcn_perm(d[2 * j + 1], d[2 * j], sel);
        return h;
    }
    // The row whose odd (q = 1) or even cells are a, the others b.
    static __device__ __forceinline__ void row(const Half &a, const Half &b, int q, uint32_t (&d)[8]) {
        const uint32_t s0 = q ? 0x01000504u : 0x05040100u, s1 = q ? 0x03020706u : 0x07060302u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            d[2 * j] = __builtin_amdgcn_perm(b.w[j], a.w[j], s0);
            d[2 * j + 1] = __builtin_amdgcn_perm(b.w[j], a.w[j], s1);
        }
    }
    // The x neighbours of the cells 2 i + q, whose own half is the other one:
    // -x of cell i is entry i, +x entry i + 1.
    struct Sides {
        uint32_t w[5];
        __device__ __forceinline__ float at(int i) const { return (i & 1) ? Sto<ST>::hi(w[i >> 1]) : Sto<ST>::lo(w[i >> 1]); }
    };
    __device__ __forceinline__ Sides sides(uint32_t left, uint32_t right, int q) const {
        const uint32_t sel = q ? 0x07060504u : 0x05040302u;
        Sides s;
#pragma unroll
        for (int j = 0; j < 4; ++j) s.w[j] = __builtin_amdgcn_perm(w[j], j ? w[j > 0 ? j - 1 : 0] : left, sel);
        s.w[4] = __builtin_amdgcn_perm(right, w[3], q ? 0x0c0c0504u : 0x0c0c0302u);
        return s;
    }
};
template <>
struct Half<MSBG_STORAGE_F32> {
    float w[8];
    __device__ __forceinline__ float at(int i) const { return w[i]; }
    __device__ __forceinline__ void set2(int i, float a, float b) {
        w[i] = a;
        w[i + 1] = b;
    }
    __device__ __forceinline__ void set(int i, float v) { w[i] = v; }
    static __device__ __forceinline__ Half of(const float2 (&d)[8], int q) {
        Half h;
#pragma unroll
        for (int i = 0; i < 8; ++i) h.w[i] = q ? d[i].y : d[i].x;
        return h;
    }
    static __device__ __forceinline__ void row(const Half &a, const Half &b, int q, float2 (&d)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) d[i] = q ? make_float2(b.w[i], a.w[i]) : make_float2(a.w[i], b.w[i]);
    }
    struct Sides {
        float w[9];
        __device__ __forceinline__ float at(int i) const { return w[i]; }
    };
    __device__ __forceinline__ Sides sides(float2 left, float2 right, int q) const {
        Sides s;
#pragma unroll
        for (int i = 0; i < 9; ++i)
            s.w[i] = q ? (i < 8 ? w[i < 8 ? i : 7] : right.x) : (i ? w[i > 0 ? i - 1 : 0] : left.y);
        return s;
    }
};

// The tile: rows y, z = -2 .. 17 around the block.  A row holds its colour 0
// cells, its colour 1 cells, and the duos (-2, -1) and (16, 17): the
// neighbours of a row's cells of one colour along y and z are the other
// colour's of four rows, one 16-byte read each for the 16-bit types.  The row
// stride of 48 or 80 bytes spreads those reads of 8 neighbouring lanes over
// all banks.
template <int ST>
struct Tile {
    using T = typename Duo<ST>::T;
    static constexpr int kHalf = (int)sizeof(Half<ST>) / 16;               // in uint4
    static constexpr int kRow = 2 * kHalf + 1;
    static constexpr int kSize = 400 * kRow;
    static __device__ __forceinline__ int at(int ry, int rz) { return ((rz + 2) * 20 + ry + 2) * kRow; }
    static __device__ __forceinline__ Half<ST> get(const uint4 *s_t, int row, int colour) {
        Half<ST> h;
        __builtin_memcpy(&h, s_t + row + kHalf * colour, sizeof(h));
        return h;
    }
    static __device__ __forceinline__ void put(uint4 *s_t, int row, int colour, const Half<ST> &h) {
        __builtin_memcpy(s_t + row + kHalf * colour, &h, sizeof(h));
    }
    // the duo left (0) or right (1) of the row
    static __device__ __forceinline__ T &end(uint4 *s_t, int row, int right) {
        return reinterpret_cast<T *>(s_t + row + 2 * kHalf)[right];
    }
};

constexpr int kRowsOwn = 256, kRowsRing = 320, kRowsAll = 388;
constexpr int kSweepThreads = kRowsRing;  // a lane per row of the block and of the faces' first ring
constexpr int kCoarseThreads = 448;       // a lane per row of the tile

// Row i: the block's 256 rows (y fastest), the rows next to its y faces and
// to its z faces, the rows one further, the four edge rows.
__device__ __forceinline__ void row_of(int i, int &ry, int &rz) {
    if (i < kRowsOwn) {
        ry = i & 15;
        rz = i >> 4;
    } else if (i < 384) {
        const int j = i & 31, f = (i - kRowsOwn) >> 5;  // f: 0 y faces, 1 z faces, 2 / 3 one further
        const int out = f < 2 ? ((j & 16) ? 16 : -1) : ((j & 16) ? 17 : -2);
        ry = (f & 1) ? (j & 15) : out;
        rz = (f & 1) ? out : (j & 15);
    } else {
        ry = (i & 1) ? 16 : -1;
        rz = (i & 2) ? 16 : -1;
    }
}

// Index of a block in the 27 from in-tile cell coordinates.
__device__ __forceinline__ int side(int c) { return (c >> 4) + 1; }

// What a lane needs to relax its row: the four neighbour rows (a row beyond
// the domain is the row itself) and the last cell inside the domain.
struct RowAt {
    int ry, rz, own, ym, yp, zm, zp;  // each row's place in the tile
    int par;                          // parity of cell 0
    bool in;                          // the row is inside the domain
};
template <int ST>
__device__ __forceinline__ RowAt row_at(int i, const PBlock &B, const Dom &d) {
    RowAt R;
    row_of(i, R.ry, R.rz);
    const int gy = B.oy + R.ry, gz = B.oz + R.rz;
    R.own = Tile<ST>::at(R.ry, R.rz);
    R.ym = gy <= 0 ? R.own : Tile<ST>::at(R.ry - 1, R.rz);
    R.yp = gy + 1 >= d.sy ? R.own : Tile<ST>::at(R.ry + 1, R.rz);
    R.zm = gz <= 0 ? R.own : Tile<ST>::at(R.ry, R.rz - 1);
    R.zp = gz + 1 >= d.sz ? R.own : Tile<ST>::at(R.ry, R.rz + 1);
    R.par = (gy + gz) & 1;  // B.ox is a multiple of 16
    R.in = gy >= 0 && gy < d.sy && gz >= 0 && gz < d.sz ;
    return R;
}

// fmaf(w6, b - A x, x) of a cell from its neighbours, summed -x, +x, -y, +y, -z, +z.
__device__ __forceinline__ float relaxed(float c, float xl, float xr, float ym, float yp, float zm, float zp, float b,
                                         float w6) {
    const float s = ((((xl + xr) + ym) + yp) + zm) + zp;
    return __builtin_fmaf(w6, __builtin_fmaf(-6.0f, c, b + s), c);
}

// Relaxes colour `col` of a row, the cells 2 i + q, from the row's other
// colour and the four rows around it.  lim: the domain's last x; wall: x = 0
// is its first cell.  One path for all, and two cells at a time: with a second
// one without the bound's compares, or with every value widened at once, the
// kernel took 76 to 86 registers instead of 63, so 4 work-groups a CU instead
// of 6, and a sweep of 153 M cells 334 us instead of 265.
template <int ST>
__device__ __forceinline__ void relax_half(Half<ST> &c, const Half<ST> &other, typename Duo<ST>::T left,
                                           typename Duo<ST>::T right, const Half<ST> &b, const uint4 *s_t,
                                           const RowAt &R, int col, int q, int lim, bool wall, float w6) {
    const Half<ST> ym = Tile<ST>::get(s_t, R.ym, R.ym == R.own ? col : col ^ 1),
                   yp = Tile<ST>::get(s_t, R.yp, R.yp == R.own ? col : col ^ 1),
                   zm = Tile<ST>::get(s_t, R.zm, R.zm == R.own ? col : col ^ 1),
                   zp = Tile<ST>::get(s_t, R.zp, R.zp == R.own ? col : col ^ 1);
    const typename Half<ST>::Sides x = other.sides(left, right, q);
    auto cell = [&](int i) {
        const float ci = c.at(i);
        float xl = x.at(i), xr = x.at(i + 1);
        if (i == 0 && wall && !q) xl = ci;
        if (2 * i + q >= lim) xr = ci;
        return relaxed(ci, xl, xr, ym.at(i), yp.at(i), zm.at(i), zp.at(i), b.at(i), w6);
    };
    // (cells beyond the domain, never looked at, take a value too)
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const float v0 = cell(i), v1 = cell(i + 1);
        c.set2(i, v0, v1);
        __builtin_amdgcn_sched_barrier(0);
    }
}
// How a sweep begins and ends.
enum { kFromZero = 0, kFromField = 1, kFromCoarse = 2 };
enum { kToField = 0, kToIterate = 1, kToPair = 2 };

struct SweepArgs {
    const PBlock *blocks;
    const int32_t *nb27;    // the 27 blocks around each listed block: listed index,
    const int32_t *slot27;  // and slot; below 0 where not listed (its e is 0 and stays so)
    Dom d;
    int n;
    float w6;
    int first;           // colour of the first half
    const void *src;     // e, or the FP32 residual (kFromZero)
    void *rt;            // right-hand side (written by kFromZero)
    void *dst;           // e
    const float *scale;  // the refinement scale: [0] 2^k, [1] 2^-k
    float extra;
    const float *x1;     // the coarse correction (kFromCoarse)
    float *x, *lo;       // the iterate (kToIterate, kToPair)
};

// (hi, lo) + v, renormalised (error-free transformations).
__device__ __forceinline__ void pair_add_to(float &hi, float &lo, float v) {
    const float h = hi + v, hb = h - hi;
    const float t = (hi - (h - hb)) + (v - hb);
    const float u = lo + t;
    hi = h + u;
    const float ub = hi - h;
    lo = (h - (hi - ub)) + (u - ub);
}

template <int ST, int FROM, int TO>
__global__ __launch_bounds__(FROM == kFromCoarse ? kCoarseThreads : kSweepThreads) void band_sweep_kernel(SweepArgs A) {
    using D = Duo<ST>;
    using T = typename D::T;
    using E = typename Sto<ST>::T;
    using TL = Tile<ST>;
    using H = Half<ST>;
    __shared__ uint4 s_t[TL::kSize];
    const int k = xcd_remap(blockIdx.x, A.n), t = threadIdx.x;
    const PBlock B = A.blocks[k];
    const Dom d = A.d;
    const int lim = d.sx - 1 - B.ox;  // last cell inside the domain along x
    const bool wall = B.ox == 0;
    const int32_t *S = A.slot27 + (i64)k * 27;
    const float inv = FROM == kFromZero ? A.scale[1] * A.extra : 0.0f;
    // A lane's row of the tile, the duos left and right of it, and its
    // right-hand side.
    T w[8], left = D::zero(), right = D::zero(), b[8], b_end = D::zero();
    RowAt R = row_at<ST>(FROM == kFromCoarse ? min(t, kRowsAll - 1) : t, B, d);
    const int row_slots = 3 * side(R.ry) + 9 * side(R.rz);
    const int s0 = S[row_slots], s1 = S[1 + row_slots], s2 = S[2 + row_slots];
    const i64 in_row = ((R.rz & 15) << 8) | ((R.ry & 15) << 4);
    // rows to relax: in the domain and a listed block; the tile's outer rows are only looked at
    R.in = R.in && s1 >= 0 && (FROM != kFromCoarse || t < kRowsRing);
    // colour `first` of the row: the cells 2 i + q, and the end cell of the
    // block's rows: -1 (q = 1) or 16 (q = 0)
    const int first = A.first, q = (R.par ^ first) & 1;
    const bool own = t < kRowsOwn;
    const int s_end = q ? s0 : s2;
    const bool end_in = own && R.in && s_end >= 0 && (q ? !wall : 16 <= lim);
#pragma unroll
    for (int m = 0; m < 8; ++m) w[m] = b[m] = D::zero();
    H c, o, bc;  // the row's colours `first` and the other, and the right-hand side of one
    if constexpr (FROM == kFromZero) {
        const float *r = (const float *)A.src;
        if (s1 >= 0) {
            const float *p = r + ((i64)s1 << 12) + in_row;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const float4 v = *reinterpret_cast<const float4 *>(p + 4 * m);
                b[2 * m] = D::make(v.x * inv, v.y * inv);
                b[2 * m + 1] = D::make(v.z * inv, v.w * inv);
            }
        }
        float e_end = 0.0f;
        if (end_in) {
            const float v = r[((i64)s_end << 12) + in_row + (q ? 15 : 0)] * inv;
            e_end = relaxed(0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, D::lo(D::make(v, v)), A.w6);
        }
        left = D::make(0.0f, q ? e_end : 0.0f);
        right = D::make(q ? 0.0f : e_end, 0.0f);
        // a relaxation where every value is 0
        bc = H::of(b, q);
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
            const float v0 = relaxed(0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, bc.at(i), A.w6);
            const float v1 = relaxed(0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, bc.at(i + 1), A.w6);
            c.set2(i, R.in ? v0 : 0.0f, R.in ? v1 : 0.0f);
            o.set2(i, 0.0f, 0.0f);
        }
        TL::put(s_t, R.own, first, c);
        if (own) {
            TL::put(s_t, R.own, first ^ 1, o);  // a row at the domain's bound looks at itself
            // only the cells inside the domain take a right-hand side
            E *out = (E *)A.rt + ((i64)s1 << 12) + in_row;
            if (R.in && lim >= 15) {
                store8<ST>((T *)out, b);
            } else if (R.in) {
                const E *bits = reinterpret_cast<const E *>(b);
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (i <= lim) out[i] = bits[i];
            }
        }
        __syncthreads();
    } else {
        const E *e = (const E *)A.src, *rt = (const E *)A.rt;
        if (s1 >= 0) {
            load8<ST>((const T *)(e + ((i64)s1 << 12) + in_row), w);
            if (FROM != kFromCoarse || t < kRowsRing) load8<ST>((const T *)(rt + ((i64)s1 << 12) + in_row), b);
        }
        if (s0 >= 0) left = *reinterpret_cast<const T *>(e + ((i64)s0 << 12) + in_row + 14);
        if (s2 >= 0) right = *reinterpret_cast<const T *>(e + ((i64)s2 << 12) + in_row);
        if (end_in) b_end = *reinterpret_cast<const T *>(rt + ((i64)s_end << 12) + in_row + (q ? 14 : 0));
        if constexpr (FROM == kFromField) {
            // lanes 0 .. 67 fetch an outer row as well
            if (t < kRowsAll - kRowsRing) {
                int oy, oz;
                row_of(kRowsRing + t, oy, oz);
                const int os = S[1 + 3 * side(oy) + 9 * side(oz)], op = (B.oy + oy + B.oz + oz) & 1;
                T x[8];
#pragma unroll
                for (int m = 0; m < 8; ++m) x[m] = D::zero();
                if (os >= 0) load8<ST>((const T *)(e + ((i64)os << 12) + (((oz & 15) << 8) | ((oy & 15) << 4))), x);
                TL::put(s_t, TL::at(oy, oz), first ^ 1, H::of(x, op ^ first ^ 1));
            }
        } else {
            // The coarse correction interpolated along x: 12 x 12 rows of the
            // level-1 cells around the block, two lanes a row, each from 7
            // cells to the 10 band cells -2 .. 7 or 8 .. 17.  The rows lie
            // where the tile comes after them.
            static_assert(sizeof(s_t) >= 144 * 20 * sizeof(float), "room for the interpolated rows");
            float *s_x = reinterpret_cast<float *>(s_t);
            if (t < 288) {
                const int row = t >> 1, half = t & 1, cy = row % 12 - 2, cz = row / 12 - 2;
                const int32_t *N = A.nb27 + (i64)k * 27 + 3 * ((cy >> 3) + 1) + 9 * ((cz >> 3) + 1);
                const int n_own = N[1], n_side = N[2 * half];
                const i64 at = 8 * (cy & 7) + 64 * (cz & 7);
                float f[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                float2 g = make_float2(0.0f, 0.0f);
                if (n_own >= 0)
#pragma unroll
                    for (int i = 0; i < 5; ++i) f[i] = A.x1[(i64)n_own * 512 + at + 3 * half + i];
                if (n_side >= 0)
                    g = *reinterpret_cast<const float2 *>(A.x1 + (i64)n_side * 512 + at + 6 * (1 - half));
                const float c7[7] = {half ? f[0] : g.x, half ? f[1] : g.y, half ? f[2] : f[0], half ? f[3] : f[1],
                                     half ? f[4] : f[2], half ? g.x : f[3], half ? g.y : f[4]};
                // cells 2 p and 2 p + 1 lie between p and p - 1 / p + 1; a
                // partner beyond the domain is the cell itself
#pragma unroll
                for (int i = 0; i < 10; ++i) {
                    const int self = 1 + (i >> 1), other = (i & 1) ? self + 1 : self - 1;
                    const int gx = B.ox + 2 * (5 * half - 2 + other);
                    s_x[row * 20 + 10 * half + i] =
                        __builtin_fmaf(0.25f, gx < 0 || gx >= d.sx ? c7[self] : c7[other], 0.75f * c7[self]);
                }
            }
            __syncthreads();
            // and along y and z: the cells -2 .. 17 of a row
            const int py = R.ry >> 1, pz = R.rz >> 1;
            int qy = py + ((R.ry & 1) ? 1 : -1), qz = pz + ((R.rz & 1) ? 1 : -1);
            if (B.oy + 2 * qy >= d.sy || B.oy + 2 * qy < 0) qy = py;
            if (B.oz + 2 * qz >= d.sz || B.oz + 2 * qz < 0) qz = pz;
            const float *x4[4];
#pragma unroll
            for (int yz = 0; yz < 4; ++yz)
                x4[yz] = s_x + ((((yz & 2) ? qz : pz) + 2) * 12 + ((yz & 1) ? qy : py) + 2) * 20;
            auto plus = [](T &a, float x, float y) { a = D::make(D::lo(a) + x, D::hi(a) + y); };
#pragma unroll
            for (int j = 0; j < 5; ++j) {  // cells 4 j - 2 .. 4 j + 1
                float4 v;
#pragma unroll
                for (int yz = 0; yz < 4; ++yz) {
                    const float wyz = ((yz & 1) ? 0.25f : 0.75f) * ((yz & 2) ? 0.25f : 0.75f);
                    const float4 f = *reinterpret_cast<const float4 *>(x4[yz] + 4 * j);
                    v.x = yz ? __builtin_fmaf(wyz, f.x, v.x) : wyz * f.x;
                    v.y = yz ? __builtin_fmaf(wyz, f.y, v.y) : wyz * f.y;
                    v.z = yz ? __builtin_fmaf(wyz, f.z, v.z) : wyz * f.z;
                    v.w = yz ? __builtin_fmaf(wyz, f.w, v.w) : wyz * f.w;
                }
                if (j == 0 ? s0 >= 0 : s1 >= 0) plus(j == 0 ? left : w[2 * j - 1], v.x, v.y);
                if (j == 4 ? s2 >= 0 : s1 >= 0) plus(j == 4 ? right : w[2 * j], v.z, v.w);
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();
        }
        c = H::of(w, q);
        o = H::of(w, q ^ 1);
        TL::put(s_t, R.own, first ^ 1, o);
        if (FROM != kFromCoarse || t < kRowsRing) {
            TL::put(s_t, R.own, first, c);  // a row at the domain's bound looks at itself
            TL::end(s_t, R.own, 0) = left;
            TL::end(s_t, R.own, 1) = right;
        }
        __syncthreads();
        // First colour: the rows of the block with their end cell, and the ring's rows.
        if (R.in) {
            const T l = left, r = right;
            if (end_in) {
                const float xc = q ? D::hi(left) : D::lo(right);
                const float xl = q ? D::lo(left) : D::hi(w[7]);
                float xr = q ? D::lo(w[0]) : D::hi(right);
                if (!q && 16 >= lim) xr = xc;
                auto cell = [&](int row) {
                    const T v = TL::end(s_t, row, q ^ 1);
                    return q ? D::hi(v) : D::lo(v);
                };
                const float v = relaxed(xc, xl, xr, cell(R.ym), cell(R.yp), cell(R.zm), cell(R.zp),
                                        q ? D::hi(b_end) : D::lo(b_end), A.w6);
                if (q)
                    left = D::make(D::lo(left), v);
                else
                    right = D::make(v, D::hi(right));
            }
            bc = H::of(b, q);
            relax_half<ST>(c, o, l, r, bc, s_t, R, first, q, lim, wall, A.w6);
            // other lanes look at this row's other colour only until the next barrier
            TL::put(s_t, R.own, first, c);
        }
        __syncthreads();
    }
    // Second colour on the block.
    if (!own || !R.in) return;
    bc = H::of(b, q ^ 1);
    relax_half<ST>(o, c, left, right, bc, s_t, R, first ^ 1, q ^ 1, lim, wall, A.w6);
    H::row(c, o, q, w);
    const i64 at = ((i64)s1 << 12) + in_row;
    if constexpr (TO == kToField) {
        store8<ST>((T *)((E *)A.dst + at), w);
    } else {
        const float sc = A.scale[0] / A.extra;
        float *x = A.x + at, *lo = TO == kToPair ? A.lo + at : nullptr;
        if (lim >= 15) {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                float4 h = *reinterpret_cast<const float4 *>(x + 4 * m);
                const float e4[4] = {D::lo(w[2 * m]), D::hi(w[2 * m]), D::lo(w[2 * m + 1]), D::hi(w[2 * m + 1])};
                if constexpr (TO == kToIterate) {
                    h.x = __builtin_fmaf(sc, e4[0], h.x);
                    h.y = __builtin_fmaf(sc, e4[1], h.y);
                    h.z = __builtin_fmaf(sc, e4[2], h.z);
                    h.w = __builtin_fmaf(sc, e4[3], h.w);
                } else {
                    float4 l = *reinterpret_cast<const float4 *>(lo + 4 * m);
                    pair_add_to(h.x, l.x, sc * e4[0]);
                    pair_add_to(h.y, l.y, sc * e4[1]);
                    pair_add_to(h.z, l.z, sc * e4[2]);
                    pair_add_to(h.w, l.w, sc * e4[3]);
                    *reinterpret_cast<float4 *>(lo + 4 * m) = l;
                }
                *reinterpret_cast<float4 *>(x + 4 * m) = h;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (i <= lim) {
                    const float ei = (i & 1) ? D::hi(w[i >> 1]) : D::lo(w[i >> 1]);
                    if constexpr (TO == kToIterate)
                        x[i] = __builtin_fmaf(sc, ei, x[i]);
                    else
                        pair_add_to(x[i], lo[i], sc * ei);
                }
        }
    }
}

// b1 = 0.5 * the sum of the 8 children's residuals rt - A e, in the order x,
// y, z; children outside the domain count 0.  The residual never leaves the CU.
template <int ST>
__global__ __launch_bounds__(kSweepThreads) void band_restrict_kernel(SweepArgs A, float *__restrict__ b1) {
    using D = Duo<ST>;
    using T = typename D::T;
    using E = typename Sto<ST>::T;
    // the tile's rows, with their 16 cells as stored
    __shared__ uint4 s_m[Tile<ST>::kSize > kRowsOwn * 5 ? Tile<ST>::kSize : kRowsOwn * 5];
    auto row_in = [&](int at) { return reinterpret_cast<T *>(s_m + at); };
    const int k = xcd_remap(blockIdx.x, A.n), t = threadIdx.x;
    const PBlock B = A.blocks[k];
    const Dom d = A.d;
    const int lim = d.sx - 1 - B.ox;
    const bool wall = B.ox == 0;
    const int32_t *S = A.slot27 + (i64)k * 27;
    T w[8], left = D::zero(), right = D::zero(), b[8];
    const RowAt R = row_at<ST>(t, B, d);
    const int row_slots = 3 * side(R.ry) + 9 * side(R.rz);
    const int s0 = S[row_slots], s1 = S[1 + row_slots], s2 = S[2 + row_slots];
    const i64 in_row = ((R.rz & 15) << 8) | ((R.ry & 15) << 4);
    const bool own = t < kRowsOwn;
    const E *e = (const E *)A.src, *rt = (const E *)A.rt;
#pragma unroll
    for (int m = 0; m < 8; ++m) w[m] = b[m] = D::zero();
    if (s1 >= 0) {
        load8<ST>((const T *)(e + ((i64)s1 << 12) + in_row), w);
        if (own) {
            load8<ST>((const T *)(rt + ((i64)s1 << 12) + in_row), b);
            if (s0 >= 0) left = *reinterpret_cast<const T *>(e + ((i64)s0 << 12) + in_row + 14);
            if (s2 >= 0) right = *reinterpret_cast<const T *>(e + ((i64)s2 << 12) + in_row);
        }
    }
    store8<ST>(row_in(R.own), w);
    __syncthreads();
    float r[16];
    if (own) {
        T ym[8], yp[8], zm[8], zp[8];
        load8<ST>(row_in(R.ym), ym);
        load8<ST>(row_in(R.yp), yp);
        load8<ST>(row_in(R.zm), zm);
        load8<ST>(row_in(R.zp), zp);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int m = i >> 1, o = i & 1;
            auto cell = [&](T v) { return o ? D::hi(v) : D::lo(v); };
            const float c = cell(w[m]);
            float xl = o ? D::lo(w[m]) : D::hi(m == 0 ? left : w[m > 0 ? m - 1 : 0]);
            if (i == 0 && wall) xl = c;
            float xr = o ? D::lo(m == 7 ? right : w[m < 7 ? m + 1 : 7]) : D::hi(w[m]);
            if (i >= lim) xr = c;
            const float s = ((((xl + xr) + cell(ym[m])) + cell(yp[m])) + cell(zm[m])) + cell(zp[m]);
            r[i] = __builtin_fmaf(-6.0f, c, cell(b[m]) + s);
        }
    }
    __syncthreads();
    float *s_r = reinterpret_cast<float *>(s_m);  // the residuals of the block's rows, in the tile's place
    if (own) {
#pragma unroll
        for (int i = 0; i < 16; i += 4)
            *reinterpret_cast<float4 *>(s_r + (R.ry + 16 * R.rz) * 20 + i) = make_float4(r[i], r[i + 1], r[i + 2], r[i + 3]);
    }
    __syncthreads();
    for (int c = t; c < 512; c += kSweepThreads) {
        const int ux = c & 7, uy = (c >> 3) & 7, uz = c >> 6;
        float sum = 0.0f;
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            const int fy = 2 * uy + (o & 1), fz = 2 * uz + (o >> 1);
            const float2 v = *reinterpret_cast<const float2 *>(s_r + (fy + 16 * fz) * 20 + 2 * ux);
            const bool in = B.oy + fy < d.sy && B.oz + fz < d.sz;
            if (in && 2 * ux <= lim) sum += v.x;
            if (in && 2 * ux + 1 <= lim) sum += v.y;
        }
        b1[(i64)k * 512 + c] = 0.5f * sum;
    }
}

template <int ST>
void launch(hipStream_t s, const SweepArgs &A, int from, int to) {
    const dim3 g(A.n), b(from == kFromCoarse ? kCoarseThreads : kSweepThreads);
    if (from == kFromZero)
        band_sweep_kernel<ST, kFromZero, kToField><<<g, b, 0, s>>>(A);
    else if (from == kFromField && to == kToField)
        band_sweep_kernel<ST, kFromField, kToField><<<g, b, 0, s>>>(A);
    else if (from == kFromField && to == kToIterate)
        band_sweep_kernel<ST, kFromField, kToIterate><<<g, b, 0, s>>>(A);
    else if (from == kFromField)
        band_sweep_kernel<ST, kFromField, kToPair><<<g, b, 0, s>>>(A);
    else if (to == kToField)
        band_sweep_kernel<ST, kFromCoarse, kToField><<<g, b, 0, s>>>(A);
    else if (to == kToIterate)
        band_sweep_kernel<ST, kFromCoarse, kToIterate><<<g, b, 0, s>>>(A);
    else
        band_sweep_kernel<ST, kFromCoarse, kToPair><<<g, b, 0, s>>>(A);
}

template <int ST>
void before(msbg_poisson *p, hipStream_t s, SweepArgs A, int nu, float *b1) {
    // e in d_e, then in turn in d_r (whose residual the first sweep has consumed)
    A.first = 0;
    A.src = p->d_r;
    A.dst = p->d_e;
    launch<ST>(s, A, kFromZero, kToField);
    for (int i = 1; i < nu; ++i) {
        A.src = A.dst;
        A.dst = A.src == p->d_e ? (void *)p->d_r : p->d_e;
        launch<ST>(s, A, kFromField, kToField);
    }
    A.src = A.dst;
    band_restrict_kernel<ST><<<A.n, kSweepThreads, 0, s>>>(A, b1);
}

template <int ST>
void after(msbg_poisson *p, hipStream_t s, SweepArgs A, int nu) {
    A.first = 1;
    A.src = (nu & 1) ? p->d_e : (void *)p->d_r;  // where `before` left e
    for (int i = 0; i < nu; ++i) {
        A.dst = A.src == p->d_e ? (void *)p->d_r : p->d_e;
        launch<ST>(s, A, i == 0 ? kFromCoarse : kFromField, i + 1 < nu ? kToField : (A.lo ? kToPair : kToIterate));
        A.src = A.dst;
    }
}

SweepArgs args_of(const msbg_poisson *p, const int32_t *nb27, const int32_t *slot27, float omega, float extra) {
    SweepArgs A{};
    A.blocks = p->d_blocks;
    A.nb27 = nb27;
    A.slot27 = slot27;
    A.d = p->dom;
    A.n = (int)p->n_active;
    A.w6 = omega / 6.0f;
    A.rt = p->d_rt;
    A.scale = p->d_scale;
    A.extra = extra;
    return A;
}

}  // namespace

void band_before(msbg_poisson *p, hipStream_t s, int storage, const int32_t *nb27, const int32_t *slot27, float omega, int nu, float extra,
                 float *b1) {
    const SweepArgs A = args_of(p, nb27, slot27, omega, extra);
    if (storage == MSBG_STORAGE_F32)
        before<MSBG_STORAGE_F32>(p, s, A, nu, b1);
    else if (storage == MSBG_STORAGE_F16)
        before<MSBG_STORAGE_F16>(p, s, A, nu, b1);
    else
        before<MSBG_STORAGE_BF16>(p, s, A, nu, b1);
}

void band_after(msbg_poisson *p, hipStream_t s, int storage, const int32_t *nb27, const int32_t *slot27, float omega, int nu, float extra,
                const float *x1, float *x, float *lo) {
    SweepArgs A = args_of(p, nb27, slot27, omega, extra);
    A.x1 = x1;
    A.x = x;
    A.lo = lo;
    if (storage == MSBG_STORAGE_F32)
        after<MSBG_STORAGE_F32>(p, s, A, nu);
    else if (storage == MSBG_STORAGE_F16)
        after<MSBG_STORAGE_F16>(p, s, A, nu);
    else
        after<MSBG_STORAGE_BF16>(p, s, A, nu);
}

}  // namespace mg
}  // namespace msbg
