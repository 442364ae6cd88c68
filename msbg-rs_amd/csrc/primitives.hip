// Device-wide exclusive scan and stable LSD radix sort (wave64 ballot ranking).
#include <algorithm>
#include <vector>

#include "primitives.hpp"

namespace msbg {

// ---------------------------------------------------------------------------
// Workspace.
// ---------------------------------------------------------------------------
static void *g_ws[25] = {nullptr};
static size_t g_ws_size[25] = {0};

void *workspace(int id, size_t bytes, int *rc) {
    *rc = MSBG_OK;
    if (bytes <= g_ws_size[id]) return g_ws[id];
    if (g_ws[id]) {
        (void)hipStreamSynchronize(stream());
        (void)hipFree(g_ws[id]);
        g_ws[id] = nullptr;
        g_ws_size[id] = 0;
    }
    size_t cap = std::max<size_t>(bytes, 1 << 20);
    hipError_t e = hipMalloc(&g_ws[id], cap);
    if (e != hipSuccess) {
        *rc = e == hipErrorOutOfMemory ? fail(MSBG_ENOMEM, "workspace: out of device memory")
                                       : hip_fail(e, "workspace");
        g_ws[id] = nullptr;
        return nullptr;
    }
    g_ws_size[id] = cap;
    return g_ws[id];
}

// ---------------------------------------------------------------------------
// Scan: tiles of 256 lanes x 8 items; tile sums, a one-workgroup scan of the
// sums, then the in-tile scan plus the tile's base.  Up to kScanSmall entries
// one workgroup holds them all.
// ---------------------------------------------------------------------------
constexpr int kScanThreads = 256, kScanItems = 8, kScanTile = kScanThreads * kScanItems;

// Inclusive scan of v across the workgroup (256 lanes, 4 waves); returns the
// inclusive prefix and writes the workgroup total to *total.
__device__ __forceinline__ uint32_t block_scan_inclusive(uint32_t v, uint32_t *s_wave, uint32_t *total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t o = __shfl_up(v, d, 64);
        if (lane >= d) v += o;
    }
    if (lane == 63) s_wave[wave] = v;
    __syncthreads();
    uint32_t add = 0;
    for (int w = 0; w < wave; ++w) add += s_wave[w];
    if (total) *total = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
    __syncthreads();
    return v + add;
}

__global__ __launch_bounds__(kScanThreads) void scan_tile_sums(const uint32_t *in, int64_t n, uint32_t *sums) {
    __shared__ uint32_t s_wave[4];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
        if (base + k < n) s += in[base + k];
    uint32_t total;
    block_scan_inclusive(s, s_wave, &total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// One workgroup, exclusive scan of `m` tile sums in place.
__global__ __launch_bounds__(kScanThreads) void scan_sums(uint32_t *sums, int64_t m, uint32_t *grand_total) {
    __shared__ uint32_t s_wave[4];
    __shared__ uint32_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int64_t off = 0; off < m; off += kScanThreads) {
        const int64_t i = off + threadIdx.x;
        const uint32_t v = i < m ? sums[i] : 0u;
        uint32_t total;
        const uint32_t inc = block_scan_inclusive(v, s_wave, &total);
        const uint32_t c = carry;
        if (i < m) sums[i] = c + inc - v;
        __syncthreads();
        if (threadIdx.x == 0) carry = c + total;
        __syncthreads();
    }
    if (threadIdx.x == 0 && grand_total) *grand_total = carry;
}

__global__ __launch_bounds__(kScanThreads) void scan_apply(const uint32_t *in, uint32_t *out, int64_t n,
                                                           const uint32_t *sums) {
    __shared__ uint32_t s_wave[4];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = base + k < n ? in[base + k] : 0u;
        s += v[k];
    }
    const uint32_t inc = block_scan_inclusive(s, s_wave, nullptr);
    uint32_t run = sums[blockIdx.x] + inc - s;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
    }
}

// All of a short array in one workgroup's registers: rounds of 4,096 entries, 4
// consecutive ones a lane, read at once; a scan within each wave and round, then
// one of the 128 wave sums.  A lane writes only what it has read, so out may be in.
// Latency and one CU's path to memory bound it: 7.0 us for 31,360 entries (the
// digit counts of 1 M keys), 2.9 for 512, against 4.1 + 3.2 + 1.8 and two more
// launches in three kernels; 128 KB each way are what its registers hold, and
// past that many CUs read faster than one.
constexpr int kSmallThreads = 1024, kSmallWaves = kSmallThreads / 64, kSmallRound = kSmallThreads * 4, kSmallRounds = 8;
constexpr int kScanSmall = kSmallRound * kSmallRounds;

template <int ROUNDS>
__global__ __launch_bounds__(kSmallThreads) void scan_small(const uint32_t *in, uint32_t *out, int n,
                                                            uint32_t *grand_total) {
    __shared__ uint32_t s_wave[ROUNDS * kSmallWaves];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const bool wide = (((uintptr_t)in | (uintptr_t)out) & 15) == 0;
    uint32_t v[ROUNDS][4], inc[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const int i = (r * kSmallThreads + t) * 4;
        v[r][0] = v[r][1] = v[r][2] = v[r][3] = 0u;
        if (wide && i + 4 <= n) {
            const uint4 q = *reinterpret_cast<const uint4 *>(in + i);
            v[r][0] = q.x;
            v[r][1] = q.y;
            v[r][2] = q.z;
            v[r][3] = q.w;
        } else if (i < n) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (i + k < n) v[r][k] = in[i + k];
        }
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) inc[r] = v[r][0] + v[r][1] + v[r][2] + v[r][3];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const uint32_t o = __shfl_up(inc[r], d, 64);
            if (lane >= d) inc[r] += o;
        }
    if (lane == 63)
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) s_wave[r * kSmallWaves + wave] = inc[r];
    __syncthreads();
    if (wave == 0) {  // exclusive scan of the wave sums, 2 a lane
        const bool sums = 2 * lane < ROUNDS * kSmallWaves;
        const uint32_t a = sums ? s_wave[2 * lane] : 0u, b = sums ? s_wave[2 * lane + 1] : 0u;
        uint32_t x = a + b;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(x, d, 64);
            if (lane >= d) x += o;
        }
        if (sums) {
            s_wave[2 * lane] = x - a - b;
            s_wave[2 * lane + 1] = x - b;
        }
        if (lane == 63) *grand_total = x;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const int i = (r * kSmallThreads + t) * 4;
        if (i >= n) continue;
        uint32_t run = s_wave[r * kSmallWaves + wave] + inc[r] - (v[r][0] + v[r][1] + v[r][2] + v[r][3]);
        uint32_t q[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            q[k] = run;
            run += v[r][k];
        }
        if (wide && i + 4 <= n) {
            *reinterpret_cast<uint4 *>(out + i) = make_uint4(q[0], q[1], q[2], q[3]);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (i + k < n) out[i + k] = q[k];
        }
    }
}

int64_t scan_sums_words(int64_t n) { return (n + kScanTile - 1) / kScanTile + 1; }

int scan_exclusive_u32(const uint32_t *in, uint32_t *out, int64_t n, uint32_t *total_host) {
    if (n <= 0) {
        if (total_host) *total_host = 0;
        return MSBG_OK;
    }
    int rc;
    uint32_t *sums = (uint32_t *)workspace(0, sizeof(uint32_t) * scan_sums_words(n), &rc);
    if (rc) return rc;
    return scan_exclusive_u32_with(in, out, n, sums, total_host);
}

int scan_exclusive_u32_with(const uint32_t *in, uint32_t *out, int64_t n, uint32_t *sums, uint32_t *total_host) {
    if (n <= 0) {
        if (total_host) *total_host = 0;
        return MSBG_OK;
    }
    const int64_t tiles = (n + kScanTile - 1) / kScanTile;
    if (n <= kSmallRound) {
        scan_small<1><<<1, kSmallThreads, 0, stream()>>>(in, out, (int)n, sums + tiles);
    } else if (n <= kScanSmall) {
        scan_small<kSmallRounds><<<1, kSmallThreads, 0, stream()>>>(in, out, (int)n, sums + tiles);
    } else {
        hipLaunchKernelGGL(scan_tile_sums, dim3((unsigned)tiles), dim3(kScanThreads), 0, stream(), in, n, sums);
        hipLaunchKernelGGL(scan_sums, dim3(1), dim3(kScanThreads), 0, stream(), sums, tiles, sums + tiles);
        hipLaunchKernelGGL(scan_apply, dim3((unsigned)tiles), dim3(kScanThreads), 0, stream(), in, out, n, sums);
    }
    MSBG_HIP(hipGetLastError());
    if (total_host) {
        MSBG_HIP(hipMemcpyAsync(total_host, sums + tiles, sizeof(uint32_t), hipMemcpyDeviceToHost, stream()));
        MSBG_HIP(hipStreamSynchronize(stream()));
    }
    return MSBG_OK;
}

// ---------------------------------------------------------------------------
// Radix sort: digits of 7 or 8 bits.  A tile is 256 lanes x 16 keys = 4096 keys; wave
// w of a tile owns the tile's keys [1024 w, 1024 w + 1024) as 16 chunks of 64.
// Pass = histogram (LDS atomics per tile, bin-major table), one exclusive scan
// of the table (so entry (d, tile) is the first output slot of digit d from
// that tile), then a stable scatter: inside a chunk a key's rank among equal
// digits comes from a ballot per bit (peer mask), across chunks and waves from LDS
// counters, so equal keys keep their input order.
// ---------------------------------------------------------------------------
constexpr int kRsThreads = 256, kRsChunks = 16, kRsTile = kRsThreads * kRsChunks;

template <int BITS>
__global__ __launch_bounds__(kRsThreads) void rs_histogram(const uint32_t *keys, int64_t n, int shift,
                                                           uint32_t *hist, int64_t ntiles) {
    constexpr int kBins = 1 << BITS;
    __shared__ uint32_t h[kBins];
    if (threadIdx.x < kBins) h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kRsTile;
#pragma unroll 4
    for (int i = threadIdx.x; i < kRsTile; i += kRsThreads)
        if (base + i < n) atomicAdd(&h[(keys[base + i] >> shift) & (kBins - 1)], 1u);
    __syncthreads();
    if (threadIdx.x < kBins) hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// (4 waves a SIMD, as its LDS allows: two registers more cost 13 us of 90)
template <int BITS>
__global__ __launch_bounds__(kRsThreads, 4) void rs_scatter(const uint32_t *__restrict__ kin,
                                                         const uint32_t *__restrict__ vin, uint32_t *__restrict__ kout,
                                                         uint32_t *__restrict__ vout, int64_t n, int shift,
                                                         const uint32_t *__restrict__ offsets, int64_t ntiles) {
    constexpr int kBins = 1 << BITS;
    constexpr uint32_t kMask = kBins - 1;
    __shared__ uint32_t cnt[4][kBins];
    __shared__ uint32_t base[kBins];   // first output slot of digit d from this tile
    __shared__ uint32_t lbase[kBins];  // first tile-local slot of digit d
    __shared__ uint32_t s_sum[4];
    __shared__ uint32_t sk[kRsTile], sv[kRsTile];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t < kBins) {
#pragma unroll
        for (int w = 0; w < 4; ++w) cnt[w][t] = 0;
        base[t] = offsets[(int64_t)t * ntiles + blockIdx.x];
    }
    __syncthreads();
    const int64_t tile0 = (int64_t)blockIdx.x * kRsTile;
    const int64_t wave0 = tile0 + (int64_t)wave * (kRsChunks * 64);
    const uint64_t lt = (1ull << lane) - 1ull;
    uint32_t k[kRsChunks], v[kRsChunks], off[kRsChunks];
#pragma unroll
    for (int c = 0; c < kRsChunks; ++c) {
        const int64_t idx = wave0 + c * 64 + lane;
        const bool valid = idx < n;
        k[c] = valid ? kin[idx] : 0u;
        v[c] = valid ? vin[idx] : 0u;
        const uint32_t d = (k[c] >> shift) & kMask;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < BITS; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        const uint32_t before = cnt[wave][d];
        off[c] = before + (uint32_t)__popcll(peers & lt);
        // The lowest lane of each peer group advances its digit's counter.
        if (valid && (peers & lt) == 0) cnt[wave][d] = before + (uint32_t)__popcll(peers);
    }
    __syncthreads();
    // exclusive scan over the 4 waves for digit t, then of the digits' totals
    // across the tile: lbase
    {
        uint32_t total = 0;
        if (t < kBins)
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint32_t x = cnt[w][t];
                cnt[w][t] = total;
                total += x;
            }
        uint32_t x = total;  // inclusive scan inside each wave, then wave sums
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (lane == 63) s_sum[wave] = x;
        __syncthreads();
        x -= total;
        for (int w = 0; w < wave; ++w) x += s_sum[w];
        if (t < kBins) lbase[t] = x;
    }
    __syncthreads();
    // Keys into LDS in output order: digit-major, stable within a digit.
#pragma unroll
    for (int c = 0; c < kRsChunks; ++c) {
        const int64_t idx = wave0 + c * 64 + lane;
        if (idx < n) {
            const uint32_t d = (k[c] >> shift) & kMask;
            const uint32_t l = lbase[d] + cnt[wave][d] + off[c];
            sk[l] = k[c];
            sv[l] = v[c];
        }
    }
    __syncthreads();
    // Consecutive lanes write consecutive slots of one digit's run.
    const int valid_n = (int)min((int64_t)kRsTile, n - tile0);
#pragma unroll
    for (int c = 0; c < kRsChunks; ++c) {
        const int l = c * kRsThreads + t;
        if (l < valid_n) {
            const uint32_t kk = sk[l];
            const uint32_t d = (kk >> shift) & kMask;
            const uint32_t pos = base[d] + (uint32_t)l - lbase[d];
            kout[pos] = kk;
            vout[pos] = sv[l];
        }
    }
}

int radix_sort_pairs(uint32_t *keys, uint32_t *vals, int64_t n, int key_bits) {
    MSBG_CHECK(key_bits >= 1 && key_bits <= 32, MSBG_EINVAL, "radix sort: key_bits must be 1..32");
    MSBG_CHECK(n >= 0 && n < ((int64_t)1 << 31), MSBG_EINVAL, "radix sort: n must be below 2^31");
    if (n <= 1) return MSBG_OK;
    // Passes of 8 bits, or 7 where as many of those do: 28 bits of keys take 4
    // passes of 7 (16.8 M pairs: 90 us a scatter, 23 a histogram; of 8: 102 and
    // 32), in less time than 3 of 9 (141 and 35).
    const int passes = (key_bits + 7) / 8;
    const int64_t ntiles = (n + kRsTile - 1) / kRsTile;
    int rc;
    uint32_t *tmp = (uint32_t *)workspace(1, sizeof(uint32_t) * 2 * n, &rc);
    if (rc) return rc;
    uint32_t *hist = (uint32_t *)workspace(2, sizeof(uint32_t) * 256 * ntiles, &rc);
    if (rc) return rc;
    uint32_t *ka = keys, *va = vals, *kb = tmp, *vb = tmp + n;
    int shift = 0;
    for (int p = 0; p < passes; ++p) {
        const int bits = key_bits - shift <= 7 * (passes - p) ? 7 : 8;
        const auto pass = [&](auto digit) -> int {
            constexpr int B = decltype(digit)::value;
            hipLaunchKernelGGL((rs_histogram<B>), dim3((unsigned)ntiles), dim3(kRsThreads), 0, stream(), ka, n, shift,
                               hist, ntiles);
            const int e = scan_exclusive_u32(hist, hist, ((int64_t)1 << B) * ntiles, nullptr);
            if (e) return e;
            hipLaunchKernelGGL((rs_scatter<B>), dim3((unsigned)ntiles), dim3(kRsThreads), 0, stream(), ka, va, kb, vb,
                               n, shift, hist, ntiles);
            return MSBG_OK;
        };
        rc = bits == 7 ? pass(std::integral_constant<int, 7>{}) : pass(std::integral_constant<int, 8>{});
        if (rc) return rc;
        MSBG_HIP(hipGetLastError());
        shift += bits;
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    if (ka != keys) {
        MSBG_HIP(hipMemcpyAsync(keys, ka, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, stream()));
        MSBG_HIP(hipMemcpyAsync(vals, va, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, stream()));
    }
    return MSBG_OK;
}

}  // namespace msbg
