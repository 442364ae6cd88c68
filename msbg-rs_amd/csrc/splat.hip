// Density min-splat: particles::splat (particles/splat.rs:92-319) for
// D = Density (u16, channel.rs:303-375) into a u16 slab over a grid layout.
//
// A block's particle bucket is cut into work items, one work-group each: it
// stages the item's (16 + 2m)^3 window (m = ceil(r_scan)) in LDS as the bits
// of the smallest squared distance so far, walks the item's particles in
// chunks (positions and footprint ranges staged in LDS), lowers every
// (particle, footprint row) pair's cells with an LDS atomic min, then
// quantises the window once and commits it to the blocks it covers with an
// atomic min.  Non-negative floats order as their bits do, and the quantised
// distance never decreases with the distance, so the smallest distance gives
// the smallest code.  min is associative and commutative, so neither the cut
// nor the order of the items changes the result, and all of them run in one
// launch: the 8 colour passes (block parity) that kept windows apart before
// left ~120 work-groups a pass (512^3, 64 instances of 8,171 points: 8 x 165
// us, 226 in one launch).
#include <algorithm>
#include <cmath>
#include <vector>

#include "internal.hpp"
#include "launch.hpp"
#include "primitives.hpp"

namespace msbg {
namespace {

struct SplatParams {
    int sx, sy, sz, nx, ny;
    int m, W;
    float r, dsq_max, inv;
};

constexpr int kMaxMargin = 6;   // window edge W <= 28: 88 KB of LDS
// Lanes per item: windows of up to 26^3 cells (70 KB) lie two to a CU, a larger one
// has it to itself (1 M particles in 512^3, r_scan = 6: 5.6 ms with 512 lanes, 3.9
// with 1,024).
constexpr int kSplatThreads = 512, kSplatThreadsWide = 1024, kSplatWide = 27;
constexpr int kChunk = 256;     // particles staged per pass

// A work item: particles p0 .. p1 - 1 (bucketed order) of occupied block blocks[k].
struct DItem {
    int32_t k, p0, p1;
};
// Particles per item: enough items to fill the chip four groups deep, but
// between a row of LDS atomics that outweighs the window's fill and commit,
// and a size past which splitting a dense block gains nothing.
constexpr int kItemMin = 128, kItemMax = 1024, kItemsWanted = 1024;

// Lowers the two 16-bit cells of a word to lo / hi, atomically.
__device__ __forceinline__ void atomic_min_2xu16(uint32_t *w, uint32_t lo, uint32_t hi) {
    uint32_t old = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (;;) {
        const uint32_t want = min(old & 0xffffu, lo) | min(old >> 16, hi) << 16;
        if (want == old) return;
        const uint32_t seen = atomicCAS(w, old, want);
        if (seen == old) return;
        old = seen;
    }
}

// Lowers one 16-bit cell, by its aligned word (in a slab that starts between
// words the pair of atomic_min_2xu16 is no aligned word).
__device__ __forceinline__ void atomic_min_u16(uint16_t *p, uint32_t v) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(p);
    const bool high = (a & 2) != 0;
    atomic_min_2xu16(reinterpret_cast<uint32_t *>(a & ~(uintptr_t)3), high ? 0xffffu : v, high ? v : 0xffffu);
}

// LDS atomics bound it: ~270 cells a particle at r_scan = 4.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void density_splat_kernel(SplatParams P, const int32_t *__restrict__ b2s,
                                                                      uint16_t *slab, const float *__restrict__ pos,
                                                                      const int32_t *__restrict__ blocks,
                                                                      const DItem *__restrict__ items) {
    extern __shared__ uint32_t st[];      // W^3 squared distances (float bits)
    __shared__ int rslot[27];
    __shared__ float s_p[kChunk][3];      // particle position - 0.5
    __shared__ int8_t s_r[kChunk][8];     // footprint: ix1, ix2, iy1, iy2, iz1, iz2 (window coordinates)
    __shared__ int s_ext[2];              // largest footprint extent of the chunk in y, in z
    const DItem item = items[blockIdx.x];
    const int bid = blocks[item.k];
    const int bx = bid % P.nx, by = (bid / P.nx) % P.ny, bz = bid / (P.nx * P.ny);
    const int W = P.W, m = P.m;
    const int cells = W * W * W;
    constexpr uint32_t kFar = 0x7f800000u;  // +inf
    for (int i = threadIdx.x; i < cells; i += THREADS) st[i] = kFar;
    const int b0x = bx * 16, b0y = by * 16, b0z = bz * 16, hi = 16 + m - 1;
    if (threadIdx.x < 27) {
        // region (rx, ry, rz): skipped when any voxel lies outside the domain
        // or the target block is not a value block (splat.rs:275-292)
        const int t = threadIdx.x, rx = t % 3 - 1, ry = (t / 3) % 3 - 1, rz = t / 9 - 1;
        const int gx0 = b0x + (rx < 0 ? -m : (rx == 0 ? 0 : 16)), gy0 = b0y + (ry < 0 ? -m : (ry == 0 ? 0 : 16)),
                  gz0 = b0z + (rz < 0 ? -m : (rz == 0 ? 0 : 16));
        const int wx = rx == 0 ? 16 : m, wy = ry == 0 ? 16 : m, wz = rz == 0 ? 16 : m;
        int slot = -1;
        if (gx0 >= 0 && gy0 >= 0 && gz0 >= 0 && gx0 + wx <= P.sx && gy0 + wy <= P.sy && gz0 + wz <= P.sz) {
            const int s = b2s[(gx0 >> 4) + (gy0 >> 4) * P.nx + (gz0 >> 4) * P.nx * P.ny];
            if (s >= 2) slot = s;
        }
        rslot[t] = slot;
    }
    // stage (splat.rs:179-225): footprint ceil(p - r - 0.5) .. floor(p + r - 0.5),
    // clipped to the window; d2 = dx*dx + (dz*dz + dy*dy)
    for (int c0 = item.p0; c0 < item.p1; c0 += kChunk) {
        if (threadIdx.x < 2) s_ext[threadIdx.x] = 0;
        __syncthreads();  // the last chunk's rows are done
        const int q = threadIdx.x, j = c0 + q;
        if (q < kChunk && j < item.p1) {
            const float px = pos[3 * j], py = pos[3 * j + 1], pz = pos[3 * j + 2];
            auto lo_of = [&](float p, int b0) { return min(max((int)ceilf((p - P.r) - 0.5f), b0 - m), b0 + hi) - (b0 - m); };
            auto hi_of = [&](float p, int b0) { return min(max((int)floorf((p + P.r) - 0.5f), b0 - m), b0 + hi) - (b0 - m); };
            const int y1 = lo_of(py, b0y), y2 = hi_of(py, b0y), z1 = lo_of(pz, b0z), z2 = hi_of(pz, b0z);
            s_p[q][0] = px - 0.5f;
            s_p[q][1] = py - 0.5f;
            s_p[q][2] = pz - 0.5f;
            s_r[q][0] = (int8_t)lo_of(px, b0x);
            s_r[q][1] = (int8_t)hi_of(px, b0x);
            s_r[q][2] = (int8_t)y1;
            s_r[q][3] = (int8_t)y2;
            s_r[q][4] = (int8_t)z1;
            s_r[q][5] = (int8_t)z2;
            atomicMax(&s_ext[0], y2 - y1 + 1);
            atomicMax(&s_ext[1], z2 - z1 + 1);
        }
        __syncthreads();
        const int n = min(kChunk, item.p1 - c0), ey = s_ext[0], rows = ey * s_ext[1];
        for (int i = threadIdx.x; i < n * rows; i += THREADS) {
            const int p = i / rows, rr = i - p * rows;
            const int cz = s_r[p][4] + rr / ey, cy = s_r[p][2] + rr % ey;
            if (cz > s_r[p][5] || cy > s_r[p][3]) continue;
            // window cell (cx, cy, cz) is grid voxel (b0 - m) + c
            const float dz = (float)(b0z - m + cz) - s_p[p][2], dy = (float)(b0y - m + cy) - s_p[p][1];
            const float dyz = dz * dz + dy * dy;
            if (dyz > P.dsq_max) continue;  // dx * dx >= 0: no cell of the row is in reach
            uint32_t *row = st + (cz * W + cy) * W;
            const int cx2 = s_r[p][1];
            const float x0 = s_p[p][0];
            for (int cx = s_r[p][0]; cx <= cx2; ++cx) {
                const float dx = (float)(b0x - m + cx) - x0;
                const float d2 = dx * dx + dyz;
                if (d2 <= P.dsq_max) atomicMin(row + cx, __float_as_uint(d2));
            }
        }
    }
    __syncthreads();  // the staging and the region table are complete
    // commit (splat.rs:227-313): a word of two x-neighbours at a time (blocks
    // and window regions start at even grid x, so both lie in one block and
    // region; with an odd margin the first and last word's outer cell is not
    // the window's), dst = min(dst, code)
    const int odd = m & 1, words = (W + 2 * odd) / 2;
    const bool words_apart = (reinterpret_cast<uintptr_t>(slab) & 2) != 0;
    auto code = [&](int cx, int row) -> uint32_t {
        if (cx < 0 || cx >= W) return 0xffffu;
        const uint32_t v = st[row + cx];
        return v == kFar ? 0xffffu : (uint32_t)(int)roundf((__uint_as_float(v) * P.inv) * 65535.0f);
    };
    for (int i = threadIdx.x; i < W * W * words; i += THREADS) {
        const int wd = i % words, r = i / words, cy = r % W, cz = r / W, cx = 2 * wd - odd;
        const uint32_t lo = code(cx, r * W), hi16 = code(cx + 1, r * W);
        if ((lo & hi16) == 0xffffu) continue;
        const int cr = cx < 0 ? 0 : cx;
        const int rx = cr < m ? 0 : (cr < m + 16 ? 1 : 2), ry = cy < m ? 0 : (cy < m + 16 ? 1 : 2),
                  rz = cz < m ? 0 : (cz < m + 16 ? 1 : 2);
        const int slot = rslot[rx + 3 * ry + 9 * rz];
        if (slot < 0) continue;
        const int gx = b0x + cx - m, gy = b0y + cy - m, gz = b0z + cz - m;
        uint16_t *d = slab + ((int64_t)slot << 12) + ((gx & 15) | ((gy & 15) << 4) | ((gz & 15) << 8));
        if (words_apart) {
            if (lo != 0xffffu) atomic_min_u16(d, lo);
            if (hi16 != 0xffffu) atomic_min_u16(d + 1, hi16);
        } else {
            atomic_min_2xu16(reinterpret_cast<uint32_t *>(d), lo, hi16);
        }
    }
}

__global__ void fill_u16_blocks_kernel(uint16_t *slab, const int32_t *__restrict__ b2s,
                                       const int32_t *__restrict__ bids, int64_t n, uint16_t v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n * 4096;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int s = b2s[bids[i >> 12]];
        if (s >= 2) slab[((int64_t)s << 12) + (i & 4095)] = v;
    }
}

__global__ void fill_u16_kernel(uint16_t *p, int64_t n, uint16_t v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

}  // namespace
}  // namespace msbg

using namespace msbg;

extern "C" {

int msbg_density_splat(msbg_grid *g, uint16_t *d_slab16, int64_t slab_slots, const float *d_pos, int64_t n,
                       float r_scan, int64_t *n_active) {
    MSBG_CHECK(g && d_slab16 && n_active, MSBG_EINVAL, "density splat: null argument");
    MSBG_CHECK(g->L == 4, MSBG_EINVAL, "density splat: 16^3-block grid required");
    MSBG_CHECK(r_scan > 0.0f && r_scan <= (float)kMaxMargin, MSBG_EINVAL, "density splat: need 0 < r_scan <= 6");
    MSBG_CHECK(n >= 0 && n < ((int64_t)1 << 31) && (n == 0 || d_pos), MSBG_EINVAL, "density splat: bad particles");
    MSBG_CHECK(g->n_blocks < ((int64_t)1 << 31), MSBG_EINVAL, "density splat: too many blocks");
    hipStream_t s = stream();
    // active blocks (active.rs:15-47) allocated in the layout and filled full
    int rc;
    int32_t *d_act = (int32_t *)workspace(10, sizeof(int32_t) * std::max<int64_t>(g->n_blocks, 1), &rc);
    if (rc) return rc;
    int64_t k = 0;
    if (n) {
        rc = msbg_active_blocks(g->sx, g->sy, g->sz, d_pos, n, r_scan, d_act, &k);
        if (rc) return rc;
    }
    std::vector<int32_t> h((size_t)k);
    if (k) MSBG_HIP(hipMemcpy(h.data(), d_act, sizeof(int32_t) * k, hipMemcpyDeviceToHost));
    std::vector<int64_t> bids(h.begin(), h.end());
    if (k) {
        rc = msbg_grid_ensure_blocks(g, bids.data(), k);
        if (rc) return rc;
    }
    MSBG_CHECK(g->n_slots <= slab_slots, MSBG_ENOMEM, "density splat: the u16 slab has fewer slots than the grid");
    *n_active = k;
    fill_u16_kernel<<<1, 256, 0, s>>>(d_slab16, 4096, 0);               // empty dummy: Density(0)
    fill_u16_kernel<<<1, 256, 0, s>>>(d_slab16 + 4096, 4096, 0xffff);  // full dummy: Density(u16::MAX)
    if (k)
        fill_u16_blocks_kernel<<<(int)std::min<int64_t>(4096, (k * 4096 + 255) / 256), 256, 0, s>>>(
            d_slab16, g->d_b2s, d_act, k, 0xffff);
    MSBG_HIP(hipGetLastError());
    if (!n) return MSBG_OK;
    // bucket the particles by block (particles/sort.rs:174-272) and gather them
    int32_t *d_bid = (int32_t *)workspace(11, sizeof(int32_t) * n, &rc);
    if (rc) return rc;
    int32_t *d_perm = (int32_t *)workspace(12, sizeof(int32_t) * n, &rc);
    if (rc) return rc;
    int32_t *d_blocks = (int32_t *)workspace(13, sizeof(int32_t) * (n + 1) * 2, &rc);
    if (rc) return rc;
    int32_t *d_starts = d_blocks + n + 1;
    float *d_sorted = (float *)workspace(14, sizeof(float) * 3 * n, &rc);
    if (rc) return rc;
    rc = msbg_particle_bids(g->sx, g->sy, g->sz, d_pos, n, d_bid);
    if (rc) return rc;
    int64_t nb = 0;
    rc = msbg_bucket_indices(d_bid, n, g->n_blocks, d_perm, d_blocks, d_starts, &nb);
    if (rc) return rc;
    rc = msbg_gather_rows(d_pos, (const uint32_t *)d_perm, n, 12, d_sorted);
    if (rc) return rc;
    SplatParams P;
    P.sx = (int)g->sx;
    P.sy = (int)g->sy;
    P.sz = (int)g->sz;
    P.nx = (int)g->nx;
    P.ny = (int)g->ny;
    P.m = (int)ceilf(r_scan);
    P.W = 16 + 2 * P.m;
    P.r = r_scan;
    P.dsq_max = r_scan * r_scan;
    P.inv = 1.0f / P.dsq_max;
    // work items: each block's particles, cut
    int64_t cut = kItemMin;
    while (cut < kItemMax && cut * kItemsWanted < n) cut *= 2;
    std::vector<int32_t> hs((size_t)nb + 1);
    MSBG_HIP(hipMemcpyAsync(hs.data(), d_starts, sizeof(int32_t) * (nb + 1), hipMemcpyDeviceToHost, s));
    MSBG_HIP(hipStreamSynchronize(s));
    std::vector<DItem> order;
    order.reserve((size_t)(nb + n / cut));
    for (int64_t i = 0; i < nb; ++i)
        for (int32_t q = hs[i]; q < hs[i + 1]; q += (int32_t)cut)
            order.push_back(DItem{(int32_t)i, q, (int32_t)std::min<int64_t>(hs[i + 1], q + cut)});
    DItem *d_items = (DItem *)workspace(23, sizeof(DItem) * std::max<size_t>(order.size(), 1), &rc);
    if (rc) return rc;
    MSBG_HIP(hipMemcpyAsync(d_items, order.data(), sizeof(DItem) * order.size(), hipMemcpyHostToDevice, s));
    const size_t lds = sizeof(uint32_t) * P.W * P.W * P.W;
    const bool wide = P.W >= kSplatWide;
    const auto kernel = wide ? density_splat_kernel<kSplatThreadsWide> : density_splat_kernel<kSplatThreads>;
    const int threads = wide ? kSplatThreadsWide : kSplatThreads;
    if (lds > 65536)
        MSBG_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    // (past 8.4 M items, which take a domain of 6 M occupied blocks, a second launch)
    const int64_t n_items = (int64_t)order.size(), most = max_groups(threads);
    for (int64_t i = 0; i < n_items; i += most)
        kernel<<<(unsigned)std::min(most, n_items - i), threads, lds, s>>>(P, g->d_b2s, d_slab16, d_sorted, d_blocks,
                                                                          d_items + i);
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipStreamSynchronize(s));
    return MSBG_OK;
}

}  // extern "C"
