// Learned error correction for the Poisson band: a 4-layer 3^3 convolution
// network on 16^3 blocks with a 2-cell halo, BF16 operands on the MFMA
// matrix cores with FP32 accumulation, trained on the GPU by the kernels
// below (forward, backward-data, backward-weights, Adam).  No reference
// counterpart: the reference has no learned component.
//
// Network (per block): X0 = 20^3 x 2 (scaled residual, phase field),
//   L1 valid 20^3 x 2 -> 18^3 x 16, ReLU     L2 valid 18^3 -> 16^3 x 16, ReLU
//   L3 same 16^3 -> 16^3 x 16, ReLU          L4 same 16^3 -> 16^3 x 1
// out[p][o] = bias[o] + sum_t sum_c W[t][c][o] in[p + off + d_t][c], tap
// t = dx + 3 dy + 9 dz, off = 0 (valid) or -1 (same, zero padding).
// Parameters (FP32 master copy): per layer W[27][16][16] + bias[16], padded
// (layer 1 uses c < 2, layer 4 uses o < 1; the padding stays zero because
// its gradient is zero).  Tensors are channels-last [tile][z][y][x][c], BF16.
//
// Every convolution -- forward, and the data gradient (the same kernel with
// the flipped, channel-transposed weights and offset -off-2) -- is an implicit
// GEMM on the 16x16x32 BF16 MFMA: 16 output cells x 16 channels per MFMA
// chain of 14 tap pairs (K = 16 input channels x 2 taps), the input planes
// staged in LDS.  The weight gradient is a second GEMM with K running over
// cells.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "poisson.hpp"

namespace msbg {
namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr int kLP = 27 * 16 * 16 + 16;  // parameters per layer (padded)
constexpr int kParams = 4 * kLP;
constexpr int kTap = 27 * 16 * 16;

__device__ __forceinline__ uint16_t to_bf16(float v) {
    uint32_t u = __float_as_uint(v);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// ---------------------------------------------------------------------------
// Convolution as an implicit GEMM on gfx950's 16x16x32 BF16 MFMA.  A
// work-group (8 waves) computes kZS output z-planes of one tile: it stages the
// kZS + 2 input planes the 3^3 taps reach into LDS as SP x SP planes
// (SP = sout + 2, zero where the tap falls outside the input), so every tap
// read is in bounds and no lane tests a coordinate; then each wave takes kCG
// groups of 16 output cells at a time through the 14 tap pairs (K = 32 = 16
// input channels x 2 taps; the 27th tap pairs with zeros) or, for the
// 2-channel input layer, 2 MFMAs of 16 taps x 2 channels.  Lane layout of
// v_mfma_f32_16x16x32_bf16: A[m][k] and B[k][n] are held as 8 consecutive k by
// lane m (n) + 16 (k / 8), D[m][n] as element m % 4 of lane n + 16 (m / 4).  A
// is the weights (M = output channels), B the input cells (N = 16 cells), so
// lane c + 16 j ends with channels 4 j .. 4 j + 3 of cell c and stores them as
// one 8-byte vector (a wave writes 512 contiguous bytes).  The weight operands
// are arranged per lane by prep_wb_kernel and kept in registers for the whole
// work-group.  Each group's result is one MFMA chain in tap-pair order, so its
// bits do not depend on kZS, kCG or the work-group size.
// ---------------------------------------------------------------------------
// Tiles per inference pass: 512 tiles' activations (163 MB) stay in the
// 256 MB Infinity Cache from one layer to the next; 4096-tile passes stream
// them through HBM and measured 30% slower per tile.
constexpr int64_t kForwardChunk = 512;
constexpr int kZS = 4;   // output z-planes per work-group
// Two 16-cell groups per wave pass: with two MFMA chains the compiler keeps
// the next tap pair's B operands in flight (106 VGPRs, 4 waves per SIMD); with
// four it runs each LDS read and its MFMA back to back to stay within 128.
constexpr int kCG = 2;   // 16-cell groups per wave pass
constexpr int kConvThreads = 512;  // 8 waves share one work-group's staged planes
constexpr int kTP = 14;  // tap pairs of a 16-channel layer
constexpr int kWB = kTP * 64;  // A-operand vectors (16 B) per layer

// Tap of pair tp in lane half h (h = 0: k = 0..15, h = 1: k = 16..31) of a
// 16-channel layer; taps are t = dx + 3 dy + 9 dz, 27 is the zero tap.
// Pairs 0..8 are (dx, dy, 0) / (dx, dy, 1), pairs 9..11 (dx, 0, 2) / (dx, 1, 2),
// pair 12 (0, 2, 2) / (1, 2, 2), pair 13 (2, 2, 2) / zero: within each run of
// pairs the h = 1 tap is the h = 0 tap moved by one plane, one row or one
// cell, so a lane's address is a per-lane base plus a constant per pair.
__host__ __device__ constexpr int tap_of(int tp, int h) {
    return tp < 9 ? tp + 9 * h : tp < 12 ? 18 + (tp - 9) + 3 * h : tp == 12 ? 24 + h : (h ? 27 : 26);
}

struct Conv2Args {
    const uint16_t *in;
    const int32_t *idx;  // tile index into `in` per batch position, or null
    int sin, off;
    const u4v *wb;       // [kTP][64] A operands of this layer
    const float *bias;   // [16] or null
    int relu;
    const uint16_t *mask;  // [tile][sout^3][16]: output zeroed where mask <= 0, or null
    void *out;             // bf16 [tile][sout^3][16], or f32 [tile][sout^3] (channel 0)
    int slabs;             // ceil(sout / kZS)
};

// Two floats as bf16, rounded to nearest even (v_cvt_pk_bf16_f32: to_bf16's
// bits in one instruction instead of a dozen; NaNs stay NaNs).
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{lo, hi}), b2));
}

// Stages planes z0 + off .. z0 + off + zn + 1, rows and columns off .. off +
// SP - 1 of a tile (zero outside it).
template <int CIN, int SP>
__device__ __forceinline__ void stage_planes(const Conv2Args &a, u4v *lds, int64_t tin, int z0, int zn) {
    constexpr int VPC = CIN == 16 ? 2 : 1;  // staged words per cell: 2 x 16 B, or one 4-byte pair
    using W = std::conditional_t<CIN == 16, u4v, uint32_t>;
    const int sin = a.sin, off = a.off;
    const int nst = (zn + 2) * SP * SP * VPC;
    constexpr int kPer = ((kZS + 2) * SP * SP * VPC + kConvThreads - 1) / kConvThreads;
    const W *in = reinterpret_cast<const W *>(a.in) + tin * VPC;
    W w[kPer];
    // all of a lane's loads before its first LDS write: one round trip, not kPer
    // (2-channel layer, 512 tiles: 34 us, 41 with a round trip each and the
    // rounding of the results in integer instructions)
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = threadIdx.x + j * kConvThreads;
        const unsigned c = (unsigned)i / VPC, v = (unsigned)i - c * VPC;
        const int p = (int)(c / (SP * SP)), r = (int)(c - p * (SP * SP)), y = r / SP, x = r - y * SP;
        const int iz = z0 + off + p, iy = off + y, ix = off + x;
        const bool inside =
            i < nst && (unsigned)iz < (unsigned)sin && (unsigned)iy < (unsigned)sin && (unsigned)ix < (unsigned)sin;
        const int64_t g = (((int64_t)iz * sin + iy) * sin + ix) * VPC + v;
        if constexpr (CIN == 16) {
            // no branch (a cell outside reads the tile's first): branches around
            // 16-byte loads made the compiler spill hundreds of registers
            w[j] = in[inside ? g : 0];
            if (!inside) w[j] = W{};
        } else {
            w[j] = 0u;
            if (inside) w[j] = in[g];
        }
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = threadIdx.x + j * kConvThreads;
        if (i < nst) reinterpret_cast<W *>(lds)[i] = w[j];
    }
}

// Bias, ReLU, mask and store of one cell's channels 4 kb .. 4 kb + 3 at output cell o.
template <bool OUTF>
__device__ __forceinline__ void put_cell(const Conv2Args &a, const f4 &acc, const float *bias, int64_t o, int kb) {
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = acc[j] + bias[j];
        if (a.relu) v[j] = v[j] > 0.0f ? v[j] : 0.0f;
    }
    if (a.mask) {
        const uint2 mk = *reinterpret_cast<const uint2 *>(a.mask + o * 16 + 4 * kb);
        const uint16_t mh[4] = {(uint16_t)(mk.x & 0xffffu), (uint16_t)(mk.x >> 16), (uint16_t)(mk.y & 0xffffu),
                                (uint16_t)(mk.y >> 16)};
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (!(from_bf16(mh[j]) > 0.0f)) v[j] = 0.0f;
    }
    if (OUTF) {
        if (kb == 0) ((float *)a.out)[o] = v[0];
    } else {
        const uint2 w = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
        *reinterpret_cast<uint2 *>((uint16_t *)a.out + o * 16 + 4 * kb) = w;
    }
}

// The 16-channel layers of output edge 16: a wave takes 8 rows of 16 cells of
// one output plane, the row y + 0 .. 2 of an input plane pair serves three of
// them.  Per step the wave reads one input row at its three x offsets (planes z
// and z + 1 side by side along K) for the outputs y, y - 1 and y - 2, then the
// five operands of plane z + 2 that finish output y - 2: 70 LDS reads for 112
// matrix instructions, where a read for each took twice an instruction's time.
// 512 tiles: 42 us (the last layer 32), 47 (38) with a read for each; the rest
// is the staging's round trip and the bf16 stores, at two work-groups a CU.  Every output adds its tap pairs in the order of
// conv2_kernel, so the bits are the same.
template <bool OUTF>
__global__ __launch_bounds__(kConvThreads, 4) void conv16_kernel(Conv2Args a) {
    extern __shared__ u4v lds[];
    constexpr int SP = 18, PL = SP * SP, ROWS = 8;
    static_assert(kZS * 16 / ROWS == kConvThreads / 64, "a wave per 8 rows");
    const int tile = blockIdx.x / a.slabs, z0 = (blockIdx.x - tile * a.slabs) * kZS;
    stage_planes<16, SP>(a, lds, (int64_t)(a.idx ? a.idx[tile] : tile) * a.sin * a.sin * a.sin, z0, kZS);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u4v wv[kTP];
#pragma unroll
    for (int tp = 0; tp < kTP; ++tp) wv[tp] = a.wb[tp * 64 + lane];
    const int m = lane & 15, kb = lane >> 4, h = kb >> 1;
    float bias[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bias[j] = a.bias ? a.bias[4 * kb + j] : 0.0f;
    const int zl = wave >> 1, y0 = (wave & 1) * ROWS;
    const u4v *cell = lds + 2 * (zl * PL + y0 * SP + m) + (kb & 1);  // row y0, x = m of plane zl
    const u4v *pair = cell + 2 * h * PL;                              // planes zl, zl + 1
    const u4v *high = cell + 4 * PL;                                  // plane zl + 2
    __syncthreads();
    auto mma = [&](f4 &c, int tp, const u4v &v) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, wv[tp]), __builtin_bit_cast(bf8, v), c, 0, 0,
                                                    0);
    };
    f4 acc[3];  // output rows r, r - 1, r - 2 at r, r - 1, r - 2 modulo 3
    const int64_t o = ((int64_t)tile * 16 + z0 + zl) * 256 + y0 * 16 + m;
    u4v v[3];
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) v[dx] = pair[2 * dx];
#pragma unroll
    for (int r = 0; r < ROWS + 2; ++r) {
        const int y = r - 2;  // the output that this step finishes
        u4v next[3], top[5];
        if (r + 1 < ROWS + 2)
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) next[dx] = pair[2 * ((r + 1) * SP + dx)];
        if (y >= 0) {
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) top[dx] = high[2 * ((y + h) * SP + dx)];
            top[3] = high[2 * ((y + 2) * SP + h)];
            top[4] = high[2 * ((y + 2) * SP + 2)];
        }
        if (r < ROWS) acc[r % 3] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int dx = 0; dx < 3; ++dx)
#pragma unroll
            for (int dy = 0; dy < 3; ++dy)  // three outputs in turn; each one's dy, dx ascend
                if (r - dy >= 0 && r - dy < ROWS) mma(acc[(r - dy) % 3], 3 * dy + dx, v[dx]);
        if (y >= 0) {
            f4 &c = acc[y % 3];
#pragma unroll
            for (int i = 0; i < 5; ++i) mma(c, 9 + i, top[i]);
            put_cell<OUTF>(a, c, bias, o + 16 * y, kb);
        }
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) v[dx] = next[dx];
        // the next step's reads stay in the next step: all of them at once take 224 registers
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Output edge sout = SP - 2; input cell (off + x, off + y, off + z) of the
// tile's sin^3 input sits at staged (x, y, z - z0).
template <int CIN, int SP, bool OUTF>
__global__ __launch_bounds__(kConvThreads) void conv2_kernel(Conv2Args a) {
    extern __shared__ u4v lds[];
    constexpr int SOUT = SP - 2, S2 = SOUT * SOUT;
    constexpr int NTP = CIN == 16 ? kTP : 2;
    const int tile = blockIdx.x / a.slabs, slab = blockIdx.x - tile * a.slabs;
    const int z0 = slab * kZS, zn = min(kZS, SOUT - z0);
    const int sin = a.sin;
    const int64_t tin = (int64_t)(a.idx ? a.idx[tile] : tile) * sin * sin * sin;
    stage_planes<CIN, SP>(a, lds, tin, z0, zn);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u4v wv[NTP];
#pragma unroll
    for (int tp = 0; tp < NTP; ++tp) wv[tp] = a.wb[tp * 64 + lane];
    const int m = lane & 15, kb = lane >> 4, h = kb >> 1;
    // CIN 16: per-lane shifts of the three runs of tap pairs (16-byte words);
    // CIN 2: staged-cell offsets of this lane's 8 taps 16 tp + 4 kb + j (past 26: any in-bounds cell)
    const int dA = h * SP * SP * 2, dB = h * SP * 2, dC = h * 2;
    int toff[CIN == 16 ? 1 : 8];
    if constexpr (CIN != 16) {
#pragma unroll
        for (int tp = 0; tp < 2; ++tp)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int t = 16 * tp + 4 * kb + j;
                toff[tp * 4 + j] = t < 27 ? (t / 9) * SP * SP + ((t / 3) % 3) * SP + t % 3 : 0;
            }
    }
    __syncthreads();
    const int ncell = zn * S2, groups = (ncell + 15) / 16;
    float bias[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bias[j] = a.bias ? a.bias[4 * kb + j] : 0.0f;
    const uint32_t *L32 = reinterpret_cast<const uint32_t *>(lds);
    constexpr int kWaves = kConvThreads / 64;
    for (int g0 = wave * kCG; g0 < groups; g0 += kWaves * kCG) {
        int base[kCG];
#pragma unroll
        for (int g = 0; g < kCG; ++g) {
            const unsigned q = (unsigned)min((g0 + g) * 16 + m, ncell - 1);  // past the last cell: computed, not stored
            const unsigned cz = q / S2, r = q - cz * S2, cy = r / SOUT, cx = r - cy * SOUT;
            base[g] = (int)((cz * SP + cy) * SP + cx);  // staged cell of tap (0, 0, 0)
            if constexpr (CIN == 16) base[g] = base[g] * 2 + (kb & 1);
        }
        f4 acc[kCG];
#pragma unroll
        for (int g = 0; g < kCG; ++g) acc[g] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int tp = 0; tp < NTP; ++tp) {
            u4v av[kCG];
#pragma unroll
            for (int g = 0; g < kCG; ++g) {
                if constexpr (CIN == 16) {
                    const int t0 = tap_of(tp, 0);
                    const int c0 = 2 * ((t0 / 9) * SP * SP + ((t0 / 3) % 3) * SP + t0 % 3);
                    const int sh = tp < 9 ? dA : tp < 12 ? dB : tp == 12 ? dC : 0;
                    av[g] = lds[base[g] + sh + c0];
                } else {
                    u4v v;
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = L32[base[g] + toff[tp * 4 + j]];
                    av[g] = v;
                }
            }
#pragma unroll
            for (int g = 0; g < kCG; ++g)
                acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, wv[tp]),
                                                                 __builtin_bit_cast(bf8, av[g]), acc[g], 0, 0, 0);
        }
#pragma unroll
        for (int g = 0; g < kCG; ++g) {
            const int grp = g0 + g;
            const int cl = grp * 16 + m;  // this lane's cell; channels 4 kb .. 4 kb + 3
            if (grp >= groups || cl >= ncell) continue;
            const int64_t o = ((int64_t)tile * SOUT + z0) * S2 + cl;
            put_cell<OUTF>(a, acc[g], bias, o, kb);
        }
    }
}

// B operands of the four layers for conv2_kernel, forward (wb) and data
// gradient (wbf: layer l's flipped, channel-transposed weights, layers 1..3):
// lane (n, kb) of tap pair tp holds 8 bf16 at k = 8 kb .. 8 kb + 7.  16-channel
// layers: k = 16 (tap - 2 tp) + c, tap = 2 tp + (kb >> 1); the 2-channel layer
// 0: k = 2 (tap - 16 tp) + c, tap = 16 tp + 4 kb + (i >> 1).  Taps past 26 are 0.
__global__ void prep_wb_kernel(const float *__restrict__ params, u4v *wb, u4v *wbf) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 4 * kWB) return;
    const int l = i / kWB, r = i % kWB, tp = r / 64, lane = r % 64;
    const int n = lane & 15, kb = lane >> 4;
    const float *W = params + (int64_t)l * kLP;  // W[t][c][o]
    uint16_t f[8], b[8];
    for (int e = 0; e < 8; ++e) {
        int t, c;
        if (l == 0) {
            t = 16 * tp + 4 * kb + (e >> 1);
            c = e & 1;
            if (tp >= 2) t = 27;
        } else {
            t = tap_of(tp, kb >> 1);
            c = (kb & 1) * 8 + e;
        }
        f[e] = t < 27 ? to_bf16(W[(t * 16 + c) * 16 + n]) : (uint16_t)0;
        b[e] = (t < 27 && l > 0) ? to_bf16(W[((26 - t) * 16 + n) * 16 + c]) : (uint16_t)0;
    }
    u4v vf, vb;
    for (int e = 0; e < 4; ++e) {
        vf[e] = (uint32_t)f[2 * e] | (uint32_t)f[2 * e + 1] << 16;
        vb[e] = (uint32_t)b[2 * e] | (uint32_t)b[2 * e + 1] << 16;
    }
    wb[i] = vf;
    wbf[i] = vb;
}

// ---------------------------------------------------------------------------
// Weight gradients: dW[t][c][o] = sum over the cells p of X[p + off + d_t][c]
// G[p][o], a GEMM with K running over cells (16x16x32 BF16 MFMA, N = o).  Both
// operands need 8 cells of one channel per lane, and the tensors are
// channels-last, so a work-group stages a slab of z-planes of one tile in LDS
// channel-major (two x-neighbours packed per 32-bit word on the way in); K
// then runs along x in groups of 8 cells, one aligned 16-byte LDS read per
// operand.  The reads of single 2-byte values from global memory that this
// replaces bound the layer: 64 tiles took 499 us for a 16-channel layer and
// 288 us for the 2-channel one, plus 267 us a layer for one thread's serial
// sum over 1,024 partials.  Now 256 partials a layer at most (a work-group
// walks further tiles with its sums in registers), added by 8 waves per 64
// parameters in a fixed order.
// ---------------------------------------------------------------------------
constexpr int kWgTiles = 64;  // tile groups: 64 x 4 slabs = one 16-channel work-group per CU
constexpr int kWg16Slabs = 4, kWg16Waves = 9;          // 4 output planes each; one wave per (dy, dz)
constexpr int kWg2Planes = 3, kWg2Slabs = 6, kWg2Waves = 10;  // 3 of 18 output planes each
constexpr int kLP2 = 27 * 2 * 16 + 16;                 // partial of the 2-channel layer: W[27][2][16], bias[16]
// LDS, in 32-bit words (2 cells): X[16][6][18][24], G[16][4][16][16]; the
// channel strides are odd multiples of 16 bytes, so the 16 channels a wave
// reads side by side fall on different banks.
constexpr int kX16C = 6 * 18 * 12 + 4, kG16C = 4 * 16 * 8 + 4;
constexpr int kWg16Lds = 16 * (kX16C + kG16C) * 4;
// 2-channel layer: V[c][dx][5][20][24] with V[c][dx][..][x] = X[..][x + dx][c], G[16][3][18][24]
constexpr int kV2C = 5 * 20 * 12 + 4, kG2C = 3 * 18 * 12 + 4;
constexpr int kWg2Lds = (6 * kV2C + 16 * kG2C) * 4;

struct WgArgs {
    const uint16_t *X;
    const int32_t *idx;
    int sin, off;
    const uint16_t *G;  // [tile][sout^3][16]
    int n_tiles, groups;  // work-group (group g, slab) takes tiles g, g + groups, ...
    float *part;        // [work-group][kLP] (16 channels), [2 work-group][kLP2] (2 channels)
};

// Channel pairs of two x-neighbours (8 channels each) as 8 words, one per
// channel: low half the left cell.
__device__ __forceinline__ void pack_cells(const u4v &l, const u4v &r, uint32_t *w) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        w[2 * i] = (l[i] & 0xffffu) | (r[i] << 16);
        w[2 * i + 1] = (l[i] >> 16) | (r[i] & 0xffff0000u);
    }
}

__device__ __forceinline__ f4 mfma32(const u4v &a, const u4v &b, const f4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

// 16 -> 16 channels, 16^3 output cells.  Wave v takes the taps (dx, dy = v %
// 3, dz = v / 3), dx = 0..2: one 20-byte window of cells x .. x + 9 per group
// gives the three A operands (words 0..3, the words shifted by one cell,
// words 1..4), so the 27 taps cost 9 window reads.  Lane (m, kg) of a step
// holds channel m (A: input, B: output) of the 8 cells of group 4 step + kg:
// plane group >> 5, row (group >> 1) & 15, x = 8 (group & 1).
__global__ __launch_bounds__(kWg16Waves * 64) void wgrad16_kernel(WgArgs a) {
    extern __shared__ u4v lds[];
    uint32_t *Xs = reinterpret_cast<uint32_t *>(lds), *Gs = Xs + 16 * kX16C;
    constexpr int NT = kWg16Waves * 64;
    const int slab = blockIdx.x % kWg16Slabs, group = blockIdx.x / kWg16Slabs;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kg = lane >> 4, dy = wave % 3, dz = wave / 3;
    const u4v ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
    f4 acc[3], bsum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < 3; ++d) acc[d] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int tile = group; tile < a.n_tiles; tile += a.groups) {
        const int sin = a.sin;
        const int64_t tin = (int64_t)(a.idx ? a.idx[tile] : tile) * sin * sin * sin;
        const u4v *X = reinterpret_cast<const u4v *>(a.X) + tin * 2;
        const u4v *G = reinterpret_cast<const u4v *>(a.G) + ((int64_t)tile * 4096 + slab * 1024) * 2;
        if (tile != group) __syncthreads();  // the last tile's reads are done
        // X planes 4 slab + off .. + 5, rows and columns off .. off + 17, zero outside the input
        for (int i = threadIdx.x; i < 6 * 18 * 9 * 2; i += NT) {
            const int half = i & 1, c = i >> 1, p = c % 9, r = c / 9, y = r % 18, z = r / 18;
            const int iz = 4 * slab + a.off + z, iy = a.off + y, ix = a.off + 2 * p;
            const bool row = (unsigned)iz < (unsigned)sin && (unsigned)iy < (unsigned)sin;
            const int64_t g = ((int64_t)iz * sin + iy) * sin + ix;
            u4v l = {0u, 0u, 0u, 0u}, q = {0u, 0u, 0u, 0u};
            if (row && (unsigned)ix < (unsigned)sin) l = X[g * 2 + half];
            if (row && (unsigned)(ix + 1) < (unsigned)sin) q = X[g * 2 + 2 + half];
            uint32_t w[8];
            pack_cells(l, q, w);
            uint32_t *d = Xs + half * 8 * kX16C + r * 12 + p;
#pragma unroll
            for (int j = 0; j < 8; ++j) d[j * kX16C] = w[j];
        }
        for (int i = threadIdx.x; i < 512 * 2; i += NT) {  // 512 cell pairs of the slab's 4 planes
            const int half = i & 1, p = i >> 1;
            uint32_t w[8];
            pack_cells(G[p * 4 + half], G[p * 4 + 2 + half], w);
            uint32_t *d = Gs + half * 8 * kG16C + p;
#pragma unroll
            for (int j = 0; j < 8; ++j) d[j * kG16C] = w[j];
        }
        __syncthreads();
        const uint32_t *xr = Xs + m * kX16C + (dz * 18 + dy) * 12, *gr = Gs + m * kG16C;
#pragma unroll 4
        for (int st = 0; st < 32; ++st) {
            const int g = 4 * st + kg, z = g >> 5, y = (g >> 1) & 15, xh = (g & 1) * 4;
            const uint32_t *xp = xr + (z * 18 + y) * 12 + xh;
            const u4v w = *reinterpret_cast<const u4v *>(xp), b = *reinterpret_cast<const u4v *>(gr + g * 4);
            const uint32_t w4 = xp[4];
            const u4v s1 = {__builtin_amdgcn_alignbit(w[1], w[0], 16), __builtin_amdgcn_alignbit(w[2], w[1], 16),
                            __builtin_amdgcn_alignbit(w[3], w[2], 16), __builtin_amdgcn_alignbit(w4, w[3], 16)};
            const u4v s2 = {w[1], w[2], w[3], w4};
            acc[0] = mfma32(w, b, acc[0]);
            acc[1] = mfma32(s1, b, acc[1]);
            acc[2] = mfma32(s2, b, acc[2]);
            if (wave == 0) bsum = mfma32(ones, b, bsum);  // every row: the sum of G over the cells
        }
    }
    float *P = a.part + (int64_t)blockIdx.x * kLP;
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j) P[((9 * dz + 3 * dy + d) * 16 + 4 * kg + j) * 16 + m] = acc[d][j];
    if (wave == 0 && kg == 0) P[kTap + m] = bsum[0];
}

// 2 -> 16 channels, 18^3 output cells.  The 16 rows of an MFMA hold two (dy,
// dz) pairs x 3 dx x 2 channels: 5 MFMAs (waves) cover the 27 taps, each lane
// reading its own dx-shifted copy, and two sets of waves halve the steps.  A
// row of 18 cells is three groups of 8; the cells past its end are zero in
// both operands.
__global__ __launch_bounds__(kWg2Waves * 64) void wgrad2_kernel(WgArgs a) {
    extern __shared__ u4v lds[];
    uint32_t *Vs = reinterpret_cast<uint32_t *>(lds), *Gs = Vs + 6 * kV2C;
    constexpr int NT = kWg2Waves * 64, NG = kWg2Planes * 18 * 3, NS = (NG + 7) / 8;  // NS steps of 4 groups per wave set
    const int slab = blockIdx.x % kWg2Slabs, group = blockIdx.x / kWg2Slabs;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, set = wave / 5, j5 = wave % 5;
    const int m = lane & 15, kg = lane >> 4;
    // row m: channel m & 1, dx (m >> 1) & 3 (3: unused), pair 2 j5 + (m >> 3) (9: unused)
    const int pair = 2 * j5 + (m >> 3), dx = (m >> 1) & 3;
    const int pr = pair < 9 ? pair : 0, vr = (m & 1) * 3 + (dx < 3 ? dx : 0);
    const u4v ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
    f4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, bsum = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int tile = group; tile < a.n_tiles; tile += a.groups) {
        const int64_t tin = (int64_t)(a.idx ? a.idx[tile] : tile) * 8000;
        const uint32_t *X = reinterpret_cast<const uint32_t *>(a.X) + tin + slab * kWg2Planes * 400;
        const u4v *G = reinterpret_cast<const u4v *>(a.G) + ((int64_t)tile * 5832 + slab * kWg2Planes * 324) * 2;
        if (tile != group) __syncthreads();
        for (int i = threadIdx.x; i < 5 * 20 * 12; i += NT) {  // a pair of x positions: both channels, three dx
            const int p = i % 12, r = i / 12;
            uint32_t c[4];  // input cells 2 p .. 2 p + 3 of the row (positions 18 .. 23 of every copy are zero)
#pragma unroll
            for (int j = 0; j < 4; ++j) c[j] = p < 9 && 2 * p + j < 20 ? X[r * 20 + 2 * p + j] : 0u;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                Vs[d * kV2C + i] = (c[d] & 0xffffu) | (c[d + 1] << 16);
                Vs[(3 + d) * kV2C + i] = (c[d] >> 16) | (c[d + 1] & 0xffff0000u);
            }
        }
        for (int i = threadIdx.x; i < kWg2Planes * 18 * 12 * 2; i += NT) {
            const int half = i & 1, c = i >> 1, p = c % 12, r = c / 12;
            u4v l = {0u, 0u, 0u, 0u}, q = {0u, 0u, 0u, 0u};
            if (p < 9) {
                l = G[(r * 18 + 2 * p) * 2 + half];
                q = G[(r * 18 + 2 * p + 1) * 2 + half];
            }
            uint32_t w[8];
            pack_cells(l, q, w);
            uint32_t *d = Gs + half * 8 * kG2C + c;
#pragma unroll
            for (int j = 0; j < 8; ++j) d[j * kG2C] = w[j];
        }
        __syncthreads();
        const uint32_t *xr = Vs + vr * kV2C + ((pr / 3) * 20 + pr % 3) * 12, *gr = Gs + m * kG2C;
#pragma unroll 3
        for (int st = 0; st < NS; ++st) {
            const int g = 8 * st + 4 * set + kg;
            const bool in = g < NG;
            const int gg = in ? g : 0, z = gg / 54, y = (gg / 3) % 18, xh = (gg % 3) * 4;
            u4v w = *reinterpret_cast<const u4v *>(xr + (z * 20 + y) * 12 + xh);
            u4v b = *reinterpret_cast<const u4v *>(gr + gg * 4);
            if (!in) w = b = u4v{0u, 0u, 0u, 0u};
            acc = mfma32(w, b, acc);
            if (j5 == 0) bsum = mfma32(ones, b, bsum);
        }
    }
    float *P = a.part + ((int64_t)blockIdx.x * 2 + set) * kLP2;
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // row 4 kg + j of the result
        const int row = 4 * kg + j, q = 2 * j5 + (row >> 3), d = (row >> 1) & 3;
        if (q < 9 && d < 3) P[((9 * (q / 3) + 3 * (q % 3) + d) * 2 + (row & 1)) * 16 + m] = acc[j];
    }
    if (j5 == 0 && kg == 0) P[27 * 2 * 16 + m] = bsum[0];
}

// grad[l][k] = the sum of layer l's partials: blockIdx.y = l, 64 parameters
// per work-group, wave w adding the partials w, w + 8, ..., then the 8 waves
// in order (deterministic).  Layer 0's partials hold its two input channels
// only; the rest of its gradient is zero.
struct WgSum {
    const float *part[4];
    int n[4];
    float *grad;
};
__global__ __launch_bounds__(512) void reduce_partials_kernel(WgSum a) {
    __shared__ float s[8][64];
    const int l = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k = blockIdx.x * 64 + lane;
    const int c = (k >> 4) & 15;
    const int row = l ? kLP : kLP2;
    const int at = l || k >= kTap ? k - (kLP - row) : ((k >> 8) * 2 + c) * 16 + (k & 15);
    const bool in = k < kLP && (l || k >= kTap || c < 2);
    float v = 0.0f;
    if (in) {
        const float *p = a.part[l] + at;
#pragma unroll 8
        for (int w = wave; w < a.n[l]; w += 8) v += p[(int64_t)w * row];
    }
    s[wave][lane] = v;
    __syncthreads();
    if (wave == 0 && k < kLP) {
        float t = s[0][lane];
#pragma unroll
        for (int w = 1; w < 8; ++w) t += s[w][lane];
        a.grad[(int64_t)l * kLP + k] = t;
    }
}

// Loss (y - target)^2 / (2 n 4096): G4 = (y - target) / (n 4096) in channel 0,
// per-work-group partial sums of (y - target)^2.
__global__ __launch_bounds__(256) void loss_kernel(const float *__restrict__ y, const float *__restrict__ target,
                                                   const int32_t *idx, int n, float inv, uint16_t *g4,
                                                   double *part) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double d2 = 0.0;
    if (i < (int64_t)n * 4096) {
        const int b = (int)(i >> 12), c = (int)(i & 4095);
        const float d = y[i] - target[(int64_t)(idx ? idx[b] : b) * 4096 + c];
        d2 = (double)d * (double)d;
        uint16_t *g = g4 + i * 16;
        g[0] = to_bf16(d * inv);
        for (int k = 1; k < 16; ++k) g[k] = 0;
    }
    for (int o = 32; o > 0; o >>= 1) d2 += __shfl_xor(d2, o);
    __shared__ double s[4];
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = d2;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = ((s[0] + s[1]) + s[2]) + s[3];
}

// Sum of the n work-group partials: thread t takes t, t + 256, ..., then a fixed tree.
__global__ __launch_bounds__(256) void loss_reduce_kernel(const double *__restrict__ part, int n, double scale,
                                                          double *loss_out, float *loss_f) {
    __shared__ double s_a[256];
    double s = 0.0;
#pragma unroll 4
    for (int i = threadIdx.x; i < n; i += 256) s += part[i];
    s_a[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) s_a[threadIdx.x] += s_a[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    *loss_out = s_a[0] * scale;
    if (loss_f) *loss_f = (float)(s_a[0] * scale);
}

__global__ void adam_kernel(float *p, float *m, float *v, const float *__restrict__ g, int n, float lr, float b1,
                            float b2, float eps, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ---- band <-> tiles -------------------------------------------------------
__device__ __forceinline__ int mirror(int g, int s) { return g < 0 ? -g - 1 : (g >= s ? 2 * s - 1 - g : g); }

// X0[k] (20^3 x 2, bf16) of listed block k: channel 0 = r * inv_scale (0 in
// blocks that are not listed), channel 1 = phi; halo cells outside the domain
// mirror (Neumann).  inv_scale = scale[1] if scale is given, else inv_host.
__global__ __launch_bounds__(256) void net_input_kernel(const PBlock *__restrict__ blocks, Dom d, int nx, int ny,
                                                        const int32_t *__restrict__ b2s,
                                                        const uint8_t *__restrict__ listed, const float *r,
                                                        const float *scale, float inv_host, const float *phi_slab,
                                                        const int32_t *__restrict__ phi_b2s, uint16_t *x0, int n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)n * 8000) return;
    const int k = (int)(i / 8000), c = (int)(i % 8000);
    const PBlock B = blocks[k];
    const int gx = mirror(B.ox + c % 20 - 2, d.sx), gy = mirror(B.oy + (c / 20) % 20 - 2, d.sy),
              gz = mirror(B.oz + c / 400 - 2, d.sz);
    const int64_t bid = (gx >> 4) + (int64_t)(gy >> 4) * nx + (int64_t)(gz >> 4) * nx * ny;
    const int vid = (gx & 15) | (gy & 15) << 4 | (gz & 15) << 8;
    const float inv = scale ? scale[1] : inv_host;
    const float rv = listed[bid] ? r[((int64_t)b2s[bid] << 12) + vid] * inv : 0.0f;
    const float pv = phi_slab[((int64_t)phi_b2s[bid] << 12) + vid];
    x0[i * 2] = to_bf16(rv);
    x0[i * 2 + 1] = to_bf16(pv);
}

// target[k][vid] = (xs - x) * inv for the in-domain cells of listed block k, else 0.
__global__ __launch_bounds__(256) void error_target_kernel(const PBlock *__restrict__ blocks, Dom d, const float *x,
                                                           const float *xs, float inv, float *target, int n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)n * 4096) return;
    const int k = (int)(i >> 12), v = (int)(i & 4095);
    const PBlock B = blocks[k];
    const bool in = B.ox + (v & 15) < d.sx && B.oy + ((v >> 4) & 15) < d.sy && B.oz + (v >> 8) < d.sz;
    const int64_t c = ((int64_t)B.slot << 12) + v;
    target[i] = in ? (xs[c] - x[c]) * inv : 0.0f;
}

// delta[slot][vid] = y[k][vid] * out_scale * scale[0] on in-domain cells of listed blocks.
__global__ __launch_bounds__(256) void delta_kernel(const PBlock *__restrict__ blocks, Dom d, const float *y,
                                                    float out_scale, const float *scale, float *delta, int n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)n * 4096) return;
    const int k = (int)(i >> 12), v = (int)(i & 4095);
    const PBlock B = blocks[k];
    const bool in = B.ox + (v & 15) < d.sx && B.oy + ((v >> 4) & 15) < d.sy && B.oz + (v >> 8) < d.sz;
    if (in) delta[((int64_t)B.slot << 12) + v] = (y[i] * out_scale) * scale[0];
}

// q = A delta (delta is zero outside the listed cells); partials of r . q and q . q.
__global__ __launch_bounds__(kThreads) void dots_kernel(const PBlock *__restrict__ blocks, Dom d,
                                                        const float *delta, const float *r, double2 *partial) {
    const PBlock B = blocks[xcd_remap(blockIdx.x, gridDim.x) / kSlices];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int gx = B.ox + tx, gy = B.oy + ty;
    double rq = 0.0, qq = 0.0;
    if (gx < d.sx && gy < d.sy) {
        const int z0 = (xcd_remap(blockIdx.x, gridDim.x) % kSlices) * (16 / kSlices);
        for (int tz = z0; tz < z0 + 16 / kSlices; ++tz) {
            const int gz = B.oz + tz;
            if (gz >= d.sz) break;
            const int vid = tx | ty << 4 | tz << 8;
            const int64_t c = ((int64_t)B.slot << 12) + vid;
            const float xl = tx > 0 ? delta[c - 1] : (gx == 0 ? delta[c] : delta[((int64_t)B.nb[0] << 12) + (vid | 15)]);
            const float xr = gx + 1 >= d.sx ? delta[c]
                                            : (tx < 15 ? delta[c + 1] : delta[((int64_t)B.nb[1] << 12) + (vid & ~15)]);
            const float yd = ty > 0 ? delta[c - 16]
                                    : (gy == 0 ? delta[c] : delta[((int64_t)B.nb[2] << 12) + (vid | 0xf0)]);
            const float yu = gy + 1 >= d.sy
                                 ? delta[c]
                                 : (ty < 15 ? delta[c + 16] : delta[((int64_t)B.nb[3] << 12) + (vid & ~0xf0)]);
            const float zb = tz > 0 ? delta[c - 256]
                                    : (gz == 0 ? delta[c] : delta[((int64_t)B.nb[4] << 12) + (vid | 0xf00)]);
            const float zf = gz + 1 >= d.sz
                                 ? delta[c]
                                 : (tz < 15 ? delta[c + 256] : delta[((int64_t)B.nb[5] << 12) + (vid & ~0xf00)]);
            const float s = ((((xl + xr) + yd) + yu) + zb) + zf;
            const float q = __builtin_fmaf(6.0f, delta[c], -s);
            rq += (double)r[c] * (double)q;
            qq += (double)q * (double)q;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        rq += __shfl_xor(rq, o);
        qq += __shfl_xor(qq, o);
    }
    __shared__ double s_a[kThreads / 64], s_b[kThreads / 64];
    if ((threadIdx.x & 63) == 0) {
        s_a[threadIdx.x >> 6] = rq;
        s_b[threadIdx.x >> 6] = qq;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0.0, b = 0.0;
        for (int w = 0; w < kThreads / 64; ++w) {
            a += s_a[w];
            b += s_b[w];
        }
        partial[blockIdx.x] = make_double2(a, b);
    }
}

__global__ __launch_bounds__(256) void reduce_dots_kernel(const double2 *__restrict__ partial, int n, double *out) {
    __shared__ double s_a[256], s_b[256];
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) {
        a += partial[i].x;
        b += partial[i].y;
    }
    s_a[threadIdx.x] = a;
    s_b[threadIdx.x] = b;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            s_a[threadIdx.x] += s_a[threadIdx.x + o];
            s_b[threadIdx.x] += s_b[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = s_a[0];
        out[1] = s_b[0];
    }
}

// x_try = fmaf(alpha, delta, x) on the listed in-domain cells, alpha = (r.q)/(q.q)
// (0 when q = 0); commit = 1 copies x_try back into x instead.
__global__ __launch_bounds__(kThreads) void try_kernel(const PBlock *__restrict__ blocks, Dom d, const double *dots,
                                                       const float *delta, float *x, float *xt, int commit) {
    const PBlock B = blocks[xcd_remap(blockIdx.x, gridDim.x) / kSlices];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int gx = B.ox + tx, gy = B.oy + ty;
    if (gx >= d.sx || gy >= d.sy) return;
    const float alpha = dots[1] > 0.0 ? (float)(dots[0] / dots[1]) : 0.0f;
    const int z0 = (xcd_remap(blockIdx.x, gridDim.x) % kSlices) * (16 / kSlices);
    for (int tz = z0; tz < z0 + 16 / kSlices; ++tz) {
        if (B.oz + tz >= d.sz) break;
        const int64_t c = ((int64_t)B.slot << 12) + (tx | ty << 4 | tz << 8);
        if (commit)
            x[c] = xt[c];
        else
            xt[c] = __builtin_fmaf(alpha, delta[c], x[c]);
    }
}

__global__ void fill_zero_kernel(float *p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0.0f;
}

int blocks_for(int64_t threads) { return (int)((threads + 255) / 256); }

}  // namespace
}  // namespace msbg

using namespace msbg;

struct msbg_learned {
    float *d_params = nullptr, *d_m = nullptr, *d_v = nullptr, *d_grad = nullptr;
    msbg::u4v *d_wb = nullptr, *d_wbf = nullptr;  // MFMA B operands, forward and data gradient
    float out_scale = 1.0f;
    int adam_t = 0;
    // workspace for `cap` tiles
    int64_t cap = 0;
    uint16_t *A1 = nullptr, *A2 = nullptr, *A3 = nullptr, *G1 = nullptr, *G2 = nullptr, *G3 = nullptr, *G4 = nullptr;
    uint16_t *X0 = nullptr;  // network input assembled from a Poisson band
    float *Y = nullptr;
    float *wpart = nullptr;
    double *loss_part = nullptr, *d_loss = nullptr;
    int64_t cap_train = 0;
};

namespace msbg {
namespace {

void free_ws(msbg_learned *n) {
    for (uint16_t **p : {&n->A1, &n->A2, &n->A3, &n->G1, &n->G2, &n->G3, &n->G4, &n->X0}) {
        (void)hipFree(*p);
        *p = nullptr;
    }
    (void)hipFree(n->Y);
    (void)hipFree(n->wpart);
    (void)hipFree(n->loss_part);
    n->Y = nullptr;
    n->wpart = nullptr;
    n->loss_part = nullptr;
    n->cap = n->cap_train = 0;
}

// Workspace for `tiles` tiles; `train` adds the backward tensors.
int ensure_ws(msbg_learned *n, int64_t tiles, bool train) {
    if (tiles <= n->cap && (!train || tiles <= n->cap_train)) return MSBG_OK;
    free_ws(n);
    const size_t a18 = (size_t)tiles * 5832 * 16 * 2, a16 = (size_t)tiles * 4096 * 16 * 2;
    MSBG_HIP(hipMalloc(&n->A1, a18));
    MSBG_HIP(hipMalloc(&n->A2, a16));
    MSBG_HIP(hipMalloc(&n->A3, a16));
    MSBG_HIP(hipMalloc(&n->Y, (size_t)tiles * 4096 * 4));
    MSBG_HIP(hipMalloc(&n->X0, (size_t)tiles * 8000 * 2 * 2));
    n->cap = tiles;
    if (train) {
        MSBG_HIP(hipMalloc(&n->G1, a18));
        MSBG_HIP(hipMalloc(&n->G2, a16));
        MSBG_HIP(hipMalloc(&n->G3, a16));
        MSBG_HIP(hipMalloc(&n->G4, a16));
        const size_t wgs = std::min<int64_t>(tiles, kWgTiles);
        MSBG_HIP(hipMalloc(&n->wpart, wgs * (3 * kWg16Slabs * kLP + 2 * kWg2Slabs * kLP2) * 4));
        MSBG_HIP(hipMalloc(&n->loss_part, (size_t)tiles * 16 * sizeof(double)));
        n->cap_train = tiles;
    }
    return MSBG_OK;
}

// Output edge SOUT; the layer reads input cells off .. off + SOUT + 1 of each
// sin^3 tile along every axis (zero outside the tile).
template <int CIN, int SOUT, bool OUTF>
void conv(hipStream_t s, const uint16_t *in, const int32_t *idx, int sin, int off, const u4v *wb,
          const float *bias, int relu, const uint16_t *mask, void *out, int n) {
    Conv2Args a;
    a.in = in;
    a.idx = idx;
    a.sin = sin;
    a.off = off;
    a.wb = wb;
    a.bias = bias;
    a.relu = relu;
    a.mask = mask;
    a.out = out;
    a.slabs = (SOUT + kZS - 1) / kZS;
    constexpr int SP = SOUT + 2;
    const size_t lds = (size_t)(kZS + 2) * SP * SP * CIN * 2;
    if constexpr (CIN == 16 && SOUT == 16)
        conv16_kernel<OUTF><<<n * a.slabs, kConvThreads, lds, s>>>(a);
    else
        conv2_kernel<CIN, SP, OUTF><<<n * a.slabs, kConvThreads, lds, s>>>(a);
}

// The network's output of n tiles into y (f32 [tile][16^3]).
void forward(msbg_learned *net, hipStream_t s, const uint16_t *x0, const int32_t *idx, int n, float *y) {
    const u4v *W = net->d_wb;
    const float *P = net->d_params;
    conv<2, 18, false>(s, x0, idx, 20, 0, W, P + 0 * kLP + kTap, 1, nullptr, net->A1, n);
    conv<16, 16, false>(s, net->A1, nullptr, 18, 0, W + kWB, P + 1 * kLP + kTap, 1, nullptr, net->A2, n);
    conv<16, 16, false>(s, net->A2, nullptr, 16, -1, W + 2 * kWB, P + 2 * kLP + kTap, 1, nullptr, net->A3, n);
    conv<16, 16, true>(s, net->A3, nullptr, 16, -1, W + 3 * kWB, P + 3 * kLP + kTap, 0, nullptr, y, n);
}

// Partials of one layer's weight gradient in net->wpart: layers 1..3 one of
// kLP floats per work-group, then layer 0 two of kLP2.
WgArgs wgrad_args(msbg_learned *net, int l, const uint16_t *X, const int32_t *idx, int sin, int off,
                  const uint16_t *G, int n) {
    WgArgs a;
    a.X = X;
    a.idx = idx;
    a.sin = sin;
    a.off = off;
    a.G = G;
    a.n_tiles = n;
    a.groups = std::min(n, kWgTiles);
    a.part = net->wpart + (int64_t)(l ? l - 1 : 3) * a.groups * kWg16Slabs * kLP;
    return a;
}

const float *wgrad(msbg_learned *net, hipStream_t s, int l, const uint16_t *X, const int32_t *idx, int sin, int off,
                   const uint16_t *G, int n) {
    const WgArgs a = wgrad_args(net, l, X, idx, sin, off, G, n);
    if (l)
        wgrad16_kernel<<<a.groups * kWg16Slabs, kWg16Waves * 64, kWg16Lds, s>>>(a);
    else
        wgrad2_kernel<<<a.groups * kWg2Slabs, kWg2Waves * 64, kWg2Lds, s>>>(a);
    return a.part;
}

// Loss and gradients of n tiles into net->d_grad; loss into net->d_loss (and loss_f if given).
void loss_grad(msbg_learned *net, hipStream_t s, const uint16_t *x0, const float *target, const int32_t *idx, int n,
               float *loss_f) {
    forward(net, s, x0, idx, n, net->Y);
    const double inv = 1.0 / ((double)n * 4096.0);
    const int nb = n * 16;
    loss_kernel<<<nb, 256, 0, s>>>(net->Y, target, idx, n, (float)inv, net->G4, net->loss_part);
    loss_reduce_kernel<<<1, 256, 0, s>>>(net->loss_part, nb, 0.5 * inv, net->d_loss, loss_f);
    const u4v *Wf = net->d_wbf;
    const int groups = std::min(n, kWgTiles);
    WgSum sum;
    sum.n[0] = groups * kWg2Slabs * 2;
    sum.n[1] = sum.n[2] = sum.n[3] = groups * kWg16Slabs;
    sum.grad = net->d_grad;
    sum.part[3] = wgrad(net, s, 3, net->A3, nullptr, 16, -1, net->G4, n);
    conv<16, 16, false>(s, net->G4, nullptr, 16, -1, Wf + 3 * kWB, nullptr, 0, net->A3, net->G3, n);
    sum.part[2] = wgrad(net, s, 2, net->A2, nullptr, 16, -1, net->G3, n);
    conv<16, 16, false>(s, net->G3, nullptr, 16, -1, Wf + 2 * kWB, nullptr, 0, net->A2, net->G2, n);
    sum.part[1] = wgrad(net, s, 1, net->A1, nullptr, 18, 0, net->G2, n);
    conv<16, 18, false>(s, net->G2, nullptr, 16, -2, Wf + 1 * kWB, nullptr, 0, net->A1, net->G1, n);
    sum.part[0] = wgrad(net, s, 0, x0, idx, 20, 0, net->G1, n);
    reduce_partials_kernel<<<dim3((kLP + 63) / 64, 4), 512, 0, s>>>(sum);
}

void prep(msbg_learned *net, hipStream_t s) {
    prep_wb_kernel<<<blocks_for(4 * kWB), 256, 0, s>>>(net->d_params, net->d_wb, net->d_wbf);
}

}  // namespace

namespace learned {

int correct(msbg_poisson *p, msbg_learned *net, const msbg_grid *phi, float *x, const float *b, double r2_in,
            double *r2, double *b2, int *accepted) {
    hipStream_t s = stream();
    const size_t slab = (size_t)p->n_slots * 4096;
    if (!p->d_delta) {
        // all three buffers or none: a failed allocation leaves the band unchanged
        float *delta = nullptr, *xtry = nullptr;
        double *dots = nullptr;
        hipError_t e = hipMalloc(&delta, slab * 4);
        if (e == hipSuccess) e = hipMalloc(&xtry, slab * 4);
        if (e == hipSuccess) e = hipMalloc(&dots, 2 * sizeof(double));
        if (e != hipSuccess) {
            if (delta) (void)hipFree(delta);
            if (xtry) (void)hipFree(xtry);
            return hip_fail(e, "learned correction buffers");
        }
        fill_zero_kernel<<<1024, 256, 0, s>>>(delta, (int64_t)slab);
        p->d_delta = delta;
        p->d_xtry = xtry;
        p->d_dots = dots;
    }
    const int64_t chunk = std::min<int64_t>(p->n_active, kForwardChunk);
    int rc = ensure_ws(net, chunk, false);
    if (rc) return rc;
    uint16_t *x0 = net->X0;
    for (int64_t k0 = 0; k0 < p->n_active; k0 += chunk) {
        const int n = (int)std::min<int64_t>(chunk, p->n_active - k0);
        net_input_kernel<<<blocks_for((int64_t)n * 8000), 256, 0, s>>>(
            p->d_blocks + k0, p->dom, (int)p->nx, (int)p->ny, p->d_b2s, p->d_listed, p->d_r, p->d_scale, 0.0f,
            phi->d_slab, phi->d_b2s, x0, n);
        forward(net, s, x0, nullptr, n, net->Y);
        delta_kernel<<<blocks_for((int64_t)n * 4096), 256, 0, s>>>(p->d_blocks + k0, p->dom, net->Y, net->out_scale,
                                                                   p->d_scale, p->d_delta, n);
    }
    dots_kernel<<<p->n_wg, kThreads, 0, s>>>(p->d_blocks, p->dom, p->d_delta, p->d_r, p->d_partial);
    reduce_dots_kernel<<<1, 256, 0, s>>>(p->d_partial, p->n_wg, p->d_dots);
    MSBG_HIP(hipMemcpyAsync(p->d_xtry, x, slab * 4, hipMemcpyDeviceToDevice, s));
    try_kernel<<<p->n_wg, kThreads, 0, s>>>(p->d_blocks, p->dom, p->d_dots, p->d_delta, x, p->d_xtry, 0);
    pband::residual(p, s, MSBG_STORAGE_F32, p->d_xtry, b, p->d_r);
    MSBG_HIP(hipGetLastError());
    rc = pband::read_norms(p, r2, b2);
    if (rc) return rc;
    *accepted = *r2 < r2_in;
    if (*accepted) {
        try_kernel<<<p->n_wg, kThreads, 0, s>>>(p->d_blocks, p->dom, p->d_dots, p->d_delta, x, p->d_xtry, 1);
    } else {
        pband::residual(p, s, MSBG_STORAGE_F32, x, b, p->d_r);
        MSBG_HIP(hipGetLastError());
        rc = pband::read_norms(p, r2, b2);
        if (rc) return rc;
    }
    MSBG_HIP(hipGetLastError());
    return MSBG_OK;
}

}  // namespace learned
}  // namespace msbg

extern "C" {

int msbg_learned_param_count(int *n) {
    MSBG_CHECK(n, MSBG_EINVAL, "null argument");
    *n = kParams;
    return MSBG_OK;
}

int msbg_learned_new(msbg_learned **out) {
    MSBG_CHECK(out, MSBG_EINVAL, "null argument");
    msbg_learned *n = new msbg_learned();
    hipError_t e = hipMalloc(&n->d_params, kParams * 4);
    if (e == hipSuccess) e = hipMalloc(&n->d_m, kParams * 4);
    if (e == hipSuccess) e = hipMalloc(&n->d_v, kParams * 4);
    if (e == hipSuccess) e = hipMalloc(&n->d_grad, kParams * 4);
    if (e == hipSuccess) e = hipMalloc(&n->d_wb, 4 * kWB * sizeof(u4v));
    if (e == hipSuccess) e = hipMalloc(&n->d_wbf, 4 * kWB * sizeof(u4v));
    if (e == hipSuccess) e = hipMalloc(&n->d_loss, sizeof(double));
    if (e == hipSuccess) e = hipMemset(n->d_params, 0, kParams * 4);
    if (e == hipSuccess) e = hipMemset(n->d_m, 0, kParams * 4);
    if (e == hipSuccess) e = hipMemset(n->d_v, 0, kParams * 4);
    // the data gradient of layer 1 stages 6 planes of 20^2 x 16 channels (76.8 KB)
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)conv2_kernel<16, 20, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (kZS + 2) * 20 * 20 * 16 * 2);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)wgrad16_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kWg16Lds);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)wgrad2_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kWg2Lds);
    if (e != hipSuccess) {
        msbg_learned_free(n);
        return hip_fail(e, "msbg_learned_new");
    }
    prep(n, stream());
    *out = n;
    return MSBG_OK;
}

int msbg_learned_free(msbg_learned *n) {
    if (!n) return MSBG_OK;
    free_ws(n);
    (void)hipFree(n->d_params);
    (void)hipFree(n->d_m);
    (void)hipFree(n->d_v);
    (void)hipFree(n->d_grad);
    (void)hipFree(n->d_wb);
    (void)hipFree(n->d_wbf);
    (void)hipFree(n->d_loss);
    delete n;
    return MSBG_OK;
}

int msbg_learned_set_params(msbg_learned *n, const float *host_params, float out_scale) {
    MSBG_CHECK(n && host_params, MSBG_EINVAL, "null argument");
    MSBG_CHECK(std::isfinite(out_scale), MSBG_EINVAL, "out_scale must be finite");
    MSBG_HIP(hipMemcpyAsync(n->d_params, host_params, kParams * 4, hipMemcpyHostToDevice, stream()));
    MSBG_HIP(hipMemsetAsync(n->d_m, 0, kParams * 4, stream()));
    MSBG_HIP(hipMemsetAsync(n->d_v, 0, kParams * 4, stream()));
    n->adam_t = 0;
    n->out_scale = out_scale;
    prep(n, stream());
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}

int msbg_learned_get_params(const msbg_learned *n, float *host_params, float *out_scale) {
    MSBG_CHECK(n && host_params && out_scale, MSBG_EINVAL, "null argument");
    MSBG_HIP(hipMemcpyAsync(host_params, n->d_params, kParams * 4, hipMemcpyDeviceToHost, stream()));
    MSBG_HIP(hipStreamSynchronize(stream()));
    *out_scale = n->out_scale;
    return MSBG_OK;
}

int msbg_learned_forward(msbg_learned *n, const uint16_t *d_x0, int64_t count, float *d_y) {
    MSBG_CHECK(n && d_x0 && d_y && count >= 0, MSBG_EINVAL, "bad argument");
    const int64_t chunk = std::min<int64_t>(std::max<int64_t>(count, 1), kForwardChunk);
    int rc = ensure_ws(n, chunk, false);
    if (rc) return rc;
    for (int64_t k0 = 0; k0 < count; k0 += chunk) {
        const int c = (int)std::min<int64_t>(chunk, count - k0);
        forward(n, stream(), d_x0 + k0 * 16000, nullptr, c, d_y + k0 * 4096);
    }
    MSBG_HIP(hipGetLastError());
    return MSBG_OK;
}

int msbg_learned_loss_grad(msbg_learned *n, const uint16_t *d_x0, const float *d_target, int64_t count,
                           double *loss, float *host_grad) {
    MSBG_CHECK(n && d_x0 && d_target && loss && host_grad, MSBG_EINVAL, "null argument");
    MSBG_CHECK(count >= 1 && count <= 4096, MSBG_EINVAL, "1 <= count <= 4096 tiles");
    int rc = ensure_ws(n, count, true);
    if (rc) return rc;
    loss_grad(n, stream(), d_x0, d_target, nullptr, (int)count, nullptr);
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipMemcpyAsync(host_grad, n->d_grad, kParams * 4, hipMemcpyDeviceToHost, stream()));
    MSBG_HIP(hipMemcpyAsync(loss, n->d_loss, sizeof(double), hipMemcpyDeviceToHost, stream()));
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}

int msbg_learned_train(msbg_learned *n, const uint16_t *d_x0, const float *d_target, int64_t n_pairs, int steps,
                       int batch, float lr, uint64_t seed, float *host_losses) {
    MSBG_CHECK(n && d_x0 && d_target && host_losses, MSBG_EINVAL, "null argument");
    MSBG_CHECK(n_pairs >= 1 && n_pairs < ((int64_t)1 << 31), MSBG_EINVAL, "bad pair count");
    MSBG_CHECK(steps >= 0 && batch >= 1 && batch <= 1024, MSBG_EINVAL, "bad steps / batch");
    if (!steps) return MSBG_OK;
    int rc = ensure_ws(n, batch, true);
    if (rc) return rc;
    hipStream_t s = stream();
    // batch indices: SplitMix64 stream from `seed`, uniform over the pairs
    std::vector<int32_t> idx((size_t)steps * batch);
    uint64_t z = seed;
    for (int32_t &v : idx) {
        z += 0x9e3779b97f4a7c15ULL;
        uint64_t q = z;
        q = (q ^ (q >> 30)) * 0xbf58476d1ce4e5b9ULL;
        q = (q ^ (q >> 27)) * 0x94d049bb133111ebULL;
        q ^= q >> 31;
        v = (int32_t)(q % (uint64_t)n_pairs);
    }
    int32_t *d_idx = nullptr;
    float *d_losses = nullptr;
    MSBG_HIP(hipMalloc(&d_idx, idx.size() * 4));
    hipError_t e = hipMalloc(&d_losses, (size_t)steps * 4);
    if (e == hipSuccess) e = hipMemcpyAsync(d_idx, idx.data(), idx.size() * 4, hipMemcpyHostToDevice, s);
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int st = 0; st < steps && e == hipSuccess; ++st) {
        loss_grad(n, s, d_x0, d_target, d_idx + (size_t)st * batch, batch, d_losses + st);
        n->adam_t += 1;
        const float c1 = 1.0f - std::pow(b1, (float)n->adam_t), c2 = 1.0f - std::pow(b2, (float)n->adam_t);
        adam_kernel<<<blocks_for(kParams), 256, 0, s>>>(n->d_params, n->d_m, n->d_v, n->d_grad, kParams, lr, b1, b2,
                                                        eps, c1, c2);
        prep(n, s);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(host_losses, d_losses, (size_t)steps * 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFree(d_idx);
    (void)hipFree(d_losses);
    MSBG_HIP(e);
    return MSBG_OK;
}

int msbg_poisson_net_input(msbg_poisson *p, const msbg_grid *phi, const float *d_r, float inv_scale,
                           uint16_t *d_x0) {
    MSBG_CHECK(p && phi && d_r && d_x0, MSBG_EINVAL, "null argument");
    MSBG_CHECK(phi->L == 4 && phi->sx == p->dom.sx && phi->sy == p->dom.sy && phi->sz == p->dom.sz, MSBG_EINVAL,
               "phase field grid must have the layout's dimensions and 16^3 blocks");
    MSBG_CHECK(p->dom.sx >= 2 && p->dom.sy >= 2 && p->dom.sz >= 2, MSBG_EINVAL, "domain must be >= 2 cells per axis");
    if (!p->n_active) return MSBG_OK;
    net_input_kernel<<<blocks_for(p->n_active * 8000), 256, 0, stream()>>>(
        p->d_blocks, p->dom, (int)p->nx, (int)p->ny, p->d_b2s, p->d_listed, d_r, nullptr, inv_scale, phi->d_slab,
        phi->d_b2s, d_x0, (int)p->n_active);
    MSBG_HIP(hipGetLastError());
    return MSBG_OK;
}

int msbg_poisson_error_target(msbg_poisson *p, const float *d_x, const float *d_xstar, float inv_scale,
                              float *d_target) {
    MSBG_CHECK(p && d_x && d_xstar && d_target, MSBG_EINVAL, "null argument");
    if (!p->n_active) return MSBG_OK;
    error_target_kernel<<<blocks_for(p->n_active * 4096), 256, 0, stream()>>>(p->d_blocks, p->dom, d_x, d_xstar,
                                                                             inv_scale, d_target, (int)p->n_active);
    MSBG_HIP(hipGetLastError());
    return MSBG_OK;
}

int msbg_poisson_learned_correct(msbg_poisson *p, msbg_learned *net, const msbg_grid *phi, float *x, const float *b,
                                 double *r2_before, double *r2_after, int *accepted) {
    MSBG_CHECK(p && net && phi && x && b && r2_before && r2_after && accepted, MSBG_EINVAL, "null argument");
    MSBG_CHECK(phi->L == 4 && phi->sx == p->dom.sx && phi->sy == p->dom.sy && phi->sz == p->dom.sz, MSBG_EINVAL,
               "phase field grid must have the layout's dimensions and 16^3 blocks");
    MSBG_CHECK(p->dom.sx >= 2 && p->dom.sy >= 2 && p->dom.sz >= 2, MSBG_EINVAL, "domain must be >= 2 cells per axis");
    *accepted = 0;
    if (!p->n_active) return MSBG_OK;
    if (!p->d_r) MSBG_HIP(hipMalloc(&p->d_r, (size_t)p->n_slots * 4096 * 4));
    pband::residual(p, stream(), MSBG_STORAGE_F32, x, b, p->d_r);
    MSBG_HIP(hipGetLastError());
    double b2 = 0.0;
    int rc = pband::read_norms(p, r2_before, &b2);
    if (rc) return rc;
    return learned::correct(p, net, phi, x, b, *r2_before, r2_after, &b2, accepted);
}

}  // extern "C"
