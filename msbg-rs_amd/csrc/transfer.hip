// Particle <-> grid transfers.
//
//  * Sampler (G2P of the reference): Sample::sample (math/sample.rs:489-526)
//    with gather_map (math/gather.rs:54-158), per particle, plus the MAC
//    face sampler (fluid/g2p.rs:26-32) and the FLIP/PIC blend (g2p.rs:42-45).
//  * MAC P2G of the reference (fluid/p2g.rs:141-412): particles bucketed by
//    block; per face direction each workgroup stages a block's particles in
//    its (16+2m)^3 window in LDS (mass + momentum) and writes the window out,
//    then every cell adds the windows that cover it, in a fixed order, and
//    divides, u = P/M (mac.rs:106-132).
//  * B-spline P2G / G2P (trilinear, quadratic): particles sorted by block and
//    voxel for the P2G, where every cell gathers its 27 neighbour voxels in a
//    fixed order, so the result is deterministic and needs neither atomics nor
//    colouring, and visited along a Morton curve for the G2P.
#include <algorithm>
#include <climits>
#include <vector>

#include "launch.hpp"
#include "primitives.hpp"

namespace msbg {

unsigned grid_for(int64_t n, int threads);
int run_lengths(const uint32_t *keys, int64_t n, int32_t *blocks, int32_t *starts, int64_t *n_occ);

// ---------------------------------------------------------------------------
// Reference sampler.
// ---------------------------------------------------------------------------
__device__ __forceinline__ const float *block_ptr(const GridView &g, int64_t bid) {
    return g.slab + (int64_t)g.b2s[bid] * 4096;
}

// gather_map (math/gather.rs:54-158).
__device__ void gather_map_dev(const GridView &g, int ix0, int iy0, int iz0, int bc, int dmax, float *out) {
    const int span = dmax + 1;
    if (ix0 >= 0 && iy0 >= 0 && iz0 >= 0 && ix0 + dmax < g.sx && iy0 + dmax < g.sy && iz0 + dmax < g.sz) {
        const int vx0 = ix0 & 15, vy0 = iy0 & 15, vz0 = iz0 & 15;
        if (vx0 + dmax < 16 && vy0 + dmax < 16 && vz0 + dmax < 16) {
            const float *p = block_ptr(g, (ix0 >> 4) + (int64_t)(iy0 >> 4) * g.nx + (int64_t)(iz0 >> 4) * g.nx * g.ny);
            int s = 0;
            for (int k = 0; k < span; ++k)
                for (int j = 0; j < span; ++j)
                    for (int i = 0; i < span; ++i) out[s++] = p[(vx0 + i) | ((vy0 + j) << 4) | ((vz0 + k) << 8)];
            return;
        }
    }
    // gather.rs:104-121 reads the resolved voxel through a 2x2x2 table of
    // blocks anchored at the clamped window corner.  The voxel's own block is
    // looked up here instead: the same block whenever the table covers it, and
    // in bounds where it does not (a Neumann reflection across a partial last
    // block), where the reference's slot bounds check panics (gather.rs:143-146).
    const float empty = g.slab[0];
    if (dmax == 1) {
        // The 8 cells' slots and values are each loaded in one batch (a
        // window across a block face reads up to 8 blocks): every lookup is
        // issued before any is used.  Same cells, same values as below.
        int64_t bid[8];
        int vid[8];
        uint32_t ok = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            int rx, ry, rz;
            const bool in = resolve_axis(ix0 + (c & 1), g.sx - 1, bc, rx) &&
                            resolve_axis(iy0 + ((c >> 1) & 1), g.sy - 1, bc, ry) &&
                            resolve_axis(iz0 + (c >> 2), g.sz - 1, bc, rz);
            bid[c] = in ? (rx >> 4) + (int64_t)(ry >> 4) * g.nx + (int64_t)(rz >> 4) * g.nx * g.ny : 0;
            vid[c] = in ? (rx & 15) | ((ry & 15) << 4) | ((rz & 15) << 8) : 0;
            ok |= (uint32_t)in << c;
        }
        int slot[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) slot[c] = g.b2s[bid[c]];
#pragma unroll
        for (int c = 0; c < 8; ++c) out[c] = g.slab[(int64_t)slot[c] * 4096 + vid[c]];
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (!((ok >> c) & 1u)) out[c] = empty;
        return;
    }
    int s = 0;
    for (int k = 0; k < span; ++k) {
        int rz;
        const bool okz = resolve_axis(iz0 + k, g.sz - 1, bc, rz);
        for (int j = 0; j < span; ++j) {
            int ry;
            const bool oky = resolve_axis(iy0 + j, g.sy - 1, bc, ry);
            for (int i = 0; i < span; ++i) {
                int rx;
                const bool okx = resolve_axis(ix0 + i, g.sx - 1, bc, rx);
                if (okx && oky && okz) {
                    const float *p = block_ptr(g, (rx >> 4) + (int64_t)(ry >> 4) * g.nx + (int64_t)(rz >> 4) * g.nx * g.ny);
                    out[s] = p[(rx & 15) | ((ry & 15) << 4) | ((rz & 15) << 8)];
                } else {
                    out[s] = empty;
                }
                ++s;
            }
        }
    }
}

__device__ __forceinline__ float lerp_f(float a, float b, float t) { return __builtin_fmaf(b - a, t, a); }

__device__ __forceinline__ float dot4_seq(const float *f, const float *w) {  // f32x4 reduce_sum, sequential
    float s = -0.0f;
    s = s + f[0] * w[0];
    s = s + f[1] * w[1];
    s = s + f[2] * w[2];
    s = s + f[3] * w[3];
    return s;
}

__device__ __forceinline__ void cubic_weights_dev(float t, float *w) {  // math/bspline.rs:6-14
    const float m = 1.0f - t;
    w[0] = (1.0f / 6.0f) * m * m * m;
    w[1] = 2.0f / 3.0f - 0.5f * t * t * (2.0f - t);
    w[2] = 2.0f / 3.0f - 0.5f * m * m * (1.0f + t);
    w[3] = (1.0f / 6.0f) * t * t * t;
}

// Sample::sample (math/sample.rs:494-526).  IP 0 Linear, 1 CubicBSpline;
// align 0 Corner, 1 CellCentered (cubic is always cell-centred).
template <int IP>
__device__ __forceinline__ float sample_ip(const GridView &g, float px, float py, float pz, int align, int bc) {
    if constexpr (IP == 0) {
        float x = px, y = py, z = pz;
        if (align == 1) {
            x = x - 0.5f;
            y = y - 0.5f;
            z = z - 0.5f;
        }
        const float ix = floorf(x), iy = floorf(y), iz = floorf(z);
        float c[8];
        gather_map_dev(g, (int)ix, (int)iy, (int)iz, bc, 1, c);
        const float u = x - ix, v = y - iy, w = z - iz;
        const float c00 = lerp_f(c[0], c[1], u), c10 = lerp_f(c[2], c[3], u);
        const float c01 = lerp_f(c[4], c[5], u), c11 = lerp_f(c[6], c[7], u);
        return lerp_f(lerp_f(c00, c10, v), lerp_f(c01, c11, v), w);
    } else {
    const float x = px - 0.5f, y = py - 0.5f, z = pz - 0.5f;
    const float xf = floorf(x), yf = floorf(y), zf = floorf(z);
    float win[64];
    gather_map_dev(g, (int)xf - 1, (int)yf - 1, (int)zf - 1, bc, 3, win);
    float wx[4], wy[4], wz[4];
    cubic_weights_dev(x - xf, wx);
    cubic_weights_dev(y - yf, wy);
    cubic_weights_dev(z - zf, wz);
    float val = 0.0f;
    for (int k = 0; k < 4; ++k)
        for (int j = 0; j < 4; ++j) val = __builtin_fmaf(dot4_seq(win + 16 * k + 4 * j, wx), wy[j] * wz[k], val);
    return val;
    }
}

__device__ float sample_dev(const GridView &g, float px, float py, float pz, int interp, int align, int bc) {
    return interp == 0 ? sample_ip<0>(g, px, py, pz, align, bc) : sample_ip<1>(g, px, py, pz, align, bc);
}

// out[i * stride] = sample at p_i - 1/2 e_axis (axis < 0: no offset).
template <int IP>
__global__ void sample_kernel(GridView g, const float *__restrict__ pos, int64_t n, int align, int bc, int axis,
                              float *__restrict__ out, int stride) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float q[3] = {axis == 0 ? pos[3 * i] - 0.5f : pos[3 * i], axis == 1 ? pos[3 * i + 1] - 0.5f : pos[3 * i + 1],
                            axis == 2 ? pos[3 * i + 2] - 0.5f : pos[3 * i + 2]};
        out[i * stride] = sample_ip<IP>(g, q[0], q[1], q[2], align, bc);
    }
}

void launch_sample(const GridView &g, const float *pos, int64_t n, int interp, int align, int bc, int axis,
                   float *out, int stride) {
    if (interp == 0)
        hipLaunchKernelGGL(sample_kernel<0>, dim3(grid_for(n, 256)), dim3(256), 0, stream(), g, pos, n, align, bc, axis,
                           out, stride);
    else
        hipLaunchKernelGGL(sample_kernel<1>, dim3(grid_for(n, 256)), dim3(256), 0, stream(), g, pos, n, align, bc, axis,
                           out, stride);
}

__global__ void blend_kernel(const float *__restrict__ u_old, const float *__restrict__ u,
                             const float *__restrict__ u_tilde, int64_t n3, float alpha, float *__restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n3; i += (int64_t)gridDim.x * blockDim.x) {
        const float delta = u[i] - u_tilde[i];  // g2p.rs:43-44
        out[i] = (u_old[i] + delta) * alpha + u[i] * (1.0f - alpha);
    }
}

// G2P of a FLIP step, per particle (fluid/g2p.rs:11-45): the staggered
// samples of u and u* (MacSampler::sample: face a at p - 1/2 e_a) and the
// FLIP/PIC blend, with the arithmetic of sample_kernel and blend_kernel.
struct MacViews {
    GridView v[3];
};
__device__ __forceinline__ float flip_blend(float u_old, float su, float st, float alpha) {
    const float delta = su - st;  // g2p.rs:43-44
    return (u_old + delta) * alpha + su * (1.0f - alpha);
}

template <int IP>
__device__ __forceinline__ void g2p_flip_one(const MacViews &u, const MacViews &ut, const float *__restrict__ pos,
                                             const float *__restrict__ u_old, int64_t i, int bc, float alpha,
                                             float *__restrict__ out) {
    const float p[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
#pragma unroll 1
    for (int a = 0; a < 3; ++a) {  // one axis at a time keeps the live registers of one sample pair
        const float q[3] = {a == 0 ? p[0] - 0.5f : p[0], a == 1 ? p[1] - 0.5f : p[1], a == 2 ? p[2] - 0.5f : p[2]};
        const float su = sample_ip<IP>(u.v[a], q[0], q[1], q[2], 1, bc);
        const float st = sample_ip<IP>(ut.v[a], q[0], q[1], q[2], 1, bc);
        out[3 * i + a] = flip_blend(u_old[3 * i + a], su, st, alpha);
    }
}

template <int IP>
__global__ void g2p_flip_kernel(MacViews u, MacViews ut, const float *__restrict__ pos,
                                const float *__restrict__ u_old, int64_t n, int bc, float alpha,
                                float *__restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        g2p_flip_one<IP>(u, ut, pos, u_old, i, bc, alpha, out);
}

// The linear samples of 256 consecutive particles.  A sample waits for its
// position, its blocks' slots and its values in turn, and those waits were the
// kernel's time (87% of its waves', at a quarter of the memory rate).  So the
// slots of the blocks around the work-group's particles go into LDS together,
// and every particle then issues all of its 48 values, x pairs in one load
// where a block holds both: three waits instead of nine.  A FLIP step's
// particles come sorted along a Morton curve, so their blocks are few; a
// work-group whose particles lie in more than `most` (any order is allowed), and
// particles near the domain's bounds, go through sample_ip.  Both give its bits.
// 67 M sorted particles: 5.35 ms through sample_ip, 3.96 so (in step, a
// direction at a time, 4.9; from cells staged in LDS, whose boxes are twice the
// particles' own cells, 5.35).
// Scattered particles share no lines, and then 48 loads at once only crowd the
// caches, so the line lies at a mean number of particles a value block (all
// sorted; sample_ip against this): 61 a block, 0.18 ms against 0.21 (1 M), 244,
// 1.25 against 1.50 (8 M), 488, 1.85 against 1.97 (16 M), 977, 0.41 against
// 0.39 (4 M), 1,950, 1.00 against 0.85 (8 M), 12,000, 1.40 against 0.99 (16 M).
// 1 M unsorted ones in 64 blocks: 0.19 against 0.22, hence 27 blocks at most. A
// few thousand are a chain of latencies, which this shortens when they lie close
// (33 us against 25 in 8 blocks).
constexpr int kFlipThreads = 256, kFlipBlocks = 27, kFlipBlocksFew = 8;
constexpr int64_t kFlipPerBlock = 750, kFlipFew = 4096;
__global__ __launch_bounds__(kFlipThreads) void g2p_flip_linear_kernel(MacViews u, MacViews ut,
                                                                       const float *__restrict__ pos,
                                                                       const float *__restrict__ u_old, int64_t n,
                                                                       int bc, float alpha, int most,
                                                                       float *__restrict__ out) {
    __shared__ int s_box[6], s_slot[6][kFlipBlocks];
    const int t = threadIdx.x;
    const int64_t i = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * kFlipThreads + t;
    const GridView &g = u.v[0];
    if (t < 6) s_box[t] = t < 3 ? INT_MAX : INT_MIN;
    float p[3] = {0.0f, 0.0f, 0.0f};
    bool in = i < n;
    if (in)
#pragma unroll
        for (int d = 0; d < 3; ++d) p[d] = pos[3 * i + d];
    // cells of all three directions: floor(p - 1) .. floor(p - 1/2) + 1, in
    // sample_ip's roundings, all inside the domain (a NaN is not)
    const float top[3] = {(float)(g.sx - 1), (float)(g.sy - 1), (float)(g.sz - 1)};
    int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
#pragma unroll
    for (int d = 0; d < 3; ++d) in = in && floorf((p[d] - 0.5f) - 0.5f) >= 0.0f && floorf(p[d] - 0.5f) + 1.0f <= top[d];
    if (in)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            lo[d] = (int)floorf((p[d] - 0.5f) - 0.5f) >> 4;
            hi[d] = ((int)floorf(p[d] - 0.5f) + 1) >> 4;
        }
#pragma unroll
    for (int d = 0; d < 3; ++d)
        for (int o = 32; o > 0; o >>= 1) {
            lo[d] = min(lo[d], __shfl_xor(lo[d], o));
            hi[d] = max(hi[d], __shfl_xor(hi[d], o));
        }
    __syncthreads();
    if ((t & 63) == 0 && lo[0] <= hi[0])
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            atomicMin(&s_box[d], lo[d]);
            atomicMax(&s_box[3 + d], hi[d]);
        }
    __syncthreads();
    const int bx0 = s_box[0], by0 = s_box[1], bz0 = s_box[2];
    const bool any = s_box[3] >= bx0;
    const int64_t nx = any ? s_box[3] - bx0 + 1 : 0, ny = any ? s_box[4] - by0 + 1 : 0, nz = any ? s_box[5] - bz0 + 1 : 0;
    const bool few = any && nx * ny * nz <= most;  // uniform over the work-group
    const int nxy = (int)(nx * ny);
    if (few)
        for (int e = t; e < 6 * kFlipBlocks; e += kFlipThreads) {
            const int a = e / kFlipBlocks, b = e % kFlipBlocks;
            if (b >= nxy * (int)nz) continue;
            const int64_t bid = (bx0 + b % (int)nx) + (int64_t)(by0 + (b % nxy) / (int)nx) * g.nx +
                                (int64_t)(bz0 + b / nxy) * g.nx * g.ny;
            s_slot[a][b] = a == 0   ? u.v[0].b2s[bid]
                           : a == 1 ? u.v[1].b2s[bid]
                           : a == 2 ? u.v[2].b2s[bid]
                           : a == 3 ? ut.v[0].b2s[bid]
                           : a == 4 ? ut.v[1].b2s[bid]
                                    : ut.v[2].b2s[bid];
        }
    __syncthreads();
    if (i >= n) return;
    if (!few || !in) {
        g2p_flip_one<0>(u, ut, pos, u_old, i, bc, alpha, out);
        return;
    }
    float f[3][3];      // fractions of direction a
    float2 e[3][2][4];  // the x pairs of direction a in u and u*
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        int c[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const float x = (d == a ? p[d] - 0.5f : p[d]) - 0.5f, b = floorf(x);
            f[a][d] = x - b;
            c[d] = (int)b;
        }
        const int vx = c[0] & 15, x0 = min(vx, 14);  // (a pair from 15 on would leave the row)
        const bool X = vx == 15;
        const int bx = (c[0] >> 4) - bx0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int y = c[1] + (k & 1), z = c[2] + (k >> 1);
            const int b = bx + (int)nx * ((y >> 4) - by0) + nxy * ((z >> 4) - bz0), row = (y & 15) << 4 | (z & 15) << 8;
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                const float *slab = (w ? ut : u).v[a].slab;
                float2 v;
                __builtin_memcpy(&v, slab + ((int64_t)s_slot[a + 3 * w][b] << 12) + (row | x0), 8);
                if (X) {
                    v.x = v.y;
                    v.y = slab[((int64_t)s_slot[a + 3 * w][b + 1] << 12) + row];
                }
                e[a][w][k] = v;
            }
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float r[2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const float c00 = lerp_f(e[a][w][0].x, e[a][w][0].y, f[a][0]), c10 = lerp_f(e[a][w][1].x, e[a][w][1].y, f[a][0]);
            const float c01 = lerp_f(e[a][w][2].x, e[a][w][2].y, f[a][0]), c11 = lerp_f(e[a][w][3].x, e[a][w][3].y, f[a][0]);
            r[w] = lerp_f(lerp_f(c00, c10, f[a][1]), lerp_f(c01, c11, f[a][1]), f[a][2]);
        }
        out[3 * i + a] = flip_blend(u_old[3 * i + a], r[0], r[1], alpha);
    }
}

// ---------------------------------------------------------------------------
// Reference MAC P2G (fluid/p2g.rs:221-412).
// ---------------------------------------------------------------------------
__global__ void set_flag_kernel(int32_t *p, int32_t v) { *p = v; }

__global__ void fill_i32_kernel(int32_t *p, int64_t n, int32_t v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Block ids as keys, at most `most` (particles far outside the domain), and
// *ungrouped set to 1 when some particle's block precedes the previous
// particle's in Morton order, or lies past 1,023 on an axis or past the last
// block along x or y (its id is then that of a block of the next row, which has
// a run of its own): otherwise (Morton-sorted input) each block's particles
// already form one run in input order, which is the order the stable bucket sort
// gives within a block.
__global__ void bucket_keys_grouped_kernel(const float *__restrict__ pos, int64_t n, int32_t nx, int32_t ny,
                                           uint32_t most, uint32_t *__restrict__ keys, uint32_t *__restrict__ idx,
                                           int32_t *__restrict__ ungrouped) {
    auto mblock = [](uint32_t x, uint32_t y, uint32_t z) {
        return spread10(x >> 4) | (spread10(y >> 4) << 1) | (spread10(z >> 4) << 2);
    };
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t x = trunc_index(pos[3 * i]), y = trunc_index(pos[3 * i + 1]), z = trunc_index(pos[3 * i + 2]);
        const uint64_t id = (x >> 4) + (uint64_t)nx * ((y >> 4) + (uint64_t)ny * (z >> 4));
        keys[i] = (uint32_t)min(id, (uint64_t)most);
        idx[i] = (uint32_t)i;
        bool down = ((x | y | z) >> 14) != 0 || (x >> 4) >= (uint32_t)nx || (y >> 4) >= (uint32_t)ny;
        if (i > 0) {
            const uint32_t px = trunc_index(pos[3 * i - 3]), py = trunc_index(pos[3 * i - 2]),
                           pz = trunc_index(pos[3 * i - 1]);
            down = down || mblock(x, y, z) < mblock(px, py, pz);
        }
        if (__any(down) && (threadIdx.x & 63) == 0) *ungrouped = 1;  // one store per wave
    }
}

// Gathers (pos, vel, mass) rows into sorted order.
__global__ void gather_payload_kernel(const float *__restrict__ pos, const float *__restrict__ vel,
                                      const float *__restrict__ mass, const uint32_t *__restrict__ perm, int64_t n,
                                      float *__restrict__ spos, float *__restrict__ svel, float *__restrict__ smass) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = perm[i];
        spos[3 * i] = pos[3 * j];
        spos[3 * i + 1] = pos[3 * j + 1];
        spos[3 * i + 2] = pos[3 * j + 2];
        svel[3 * i] = vel[3 * j];
        svel[3 * i + 1] = vel[3 * j + 1];
        svel[3 * i + 2] = vel[3 * j + 2];
        if (smass) smass[i] = mass ? mass[j] : 1.0f;
    }
}

// A work item of the MAC splat: particles p0 .. p1 - 1 (sorted) of block bid.
struct SplatItem {
    int32_t bid, p0, p1;
};
constexpr int kSplatThreads = 1024;  // one group per CU holds the 128 KB window of r_p <= 2: 16 waves
// Particles per item: an item per CU, at most 16,384 and not below 256, where a
// window's clearing and writing outweigh its particles (100,000 particles in 48
// blocks: 20 + 14 us a direction for splat and commit, 25 + 23 with two items
// per CU).
constexpr int kSplatMost = 16384, kSplatLeast = 256, kSplatItems = 256;
constexpr size_t kSplatShared = (size_t)64 << 20;  // bytes of windows in the shared workspace
constexpr int kSplatMaxCells = 8192;  // window cells of the two-channel kernels (m <= 2: 20^3)

// One face direction of the MAC splat (p2g.rs:261-333): work-group i adds up
// the particles of items[i] in its (16 + 2m)^3 window and writes the window's
// (mass, momentum) pairs to win + i (16 + 2m)^3 (mac_commit_kernel adds the
// windows up): first the 16 middle cells of every row, then the rows' m cells
// below, then those above, so that a reader of a margin takes whole lines.
// CH 0 splats the mass m w, CH 1 the momentum m u_a w, CH 2 both.
//
// The window holds float64 sums of the float contributions w m and w (m u_a)
// (16,384 of one sign lose at most 2^-39 of their sum), so it needs no scale,
// and NaN and infinities propagate as in a float sum.  It is bound by its LDS
// adds: 8.4 ns a wave and CU for float64 at random cells.  int64 adds of a
// fixed-point window take 4.4 ns, but small contributions (a slow particle
// beside a fast one, the edge of a support) don't fit one scale, and the
// special path that they need cost six times the adds.
//
// AT is the face direction when it is a template constant (the two-channel
// kernels), or -1 when it comes in `a_rt`.
template <int CH, int AT>
__global__ __launch_bounds__(kSplatThreads) void mac_splat_kernel(int nx, int ny, int a_rt,
                                                                  const SplatItem *__restrict__ items,
                                                                  const float *__restrict__ spos,
                                                                  const float *__restrict__ svel,
                                                                  const float *__restrict__ smass, float r_p,
                                                                  float inv_r2, int m, float2 *__restrict__ win) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    constexpr int NC = CH == 2 ? 2 : 1;  // channels of this pass
    const int a = AT >= 0 ? AT : a_rt;
    const int MSX = 16 + 2 * m, NS = MSX * MSX * MSX;
    double *acc = reinterpret_cast<double *>(smem_raw);  // NC windows
    for (int s = threadIdx.x; s < NC * NS / 2; s += kSplatThreads)
        reinterpret_cast<double2 *>(acc)[s] = make_double2(0.0, 0.0);
    const SplatItem item = items[blockIdx.x];
    const int bx = item.bid % nx, by = (item.bid / nx) % ny, bz = item.bid / (nx * ny);
    const int b0x = bx * 16, b0y = by * 16, b0z = bz * 16;
    const int x0s = b0x - m, y0s = b0y - m, z0s = b0z - m, whi = 16 + m - 1;
    const float ofx = a == 0 ? 1.0f : 0.5f, ofy = a == 1 ? 1.0f : 0.5f, ofz = a == 2 ? 1.0f : 0.5f;
    const int cnt = item.p1 - item.p0;
    __syncthreads();
    // A wave takes 64 particles, `chunks` apart: particles sorted along a curve
    // share cells with their successors, and adds of one wave to one address
    // run one after the other (67 M particles: 2.8 ms a direction and half of
    // them with neighbouring particles in neighbouring lanes, 2.3 so).
    const int chunks = (cnt + 63) >> 6, lane = threadIdx.x & 63;
    for (int t = threadIdx.x >> 6; t < chunks; t += kSplatThreads / 64) {
        const int q = lane * chunks + t;
        if (q >= cnt) continue;
        const int pi = item.p0 + q;
        float sc[NC];
        bool fin = true, live = false;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            // channel k of this pass is the mass when CH is 0, or CH is 2 and k is 0
            sc[k] = (CH == 2 ? k == 0 : CH == 0) ? smass[pi] : smass[pi] * svel[3 * pi + a];
            fin = fin && isfinite(sc[k]);
            live = live || sc[k] != 0.0f;
        }
        if (!live) continue;
        const float px = spos[3 * pi], py = spos[3 * pi + 1], pz = spos[3 * pi + 2];
        const float px0 = px - 0.5f, py0 = py - 0.5f, pz0 = pz - 0.5f;
        const int ix1 = min(max((int)ceilf(px - r_p - ofx), x0s), b0x + whi);
        const int ix2 = min(max((int)floorf(px + r_p - ofx), x0s), b0x + whi);
        const int iy1 = min(max((int)ceilf(py - r_p - ofy), y0s), b0y + whi);
        const int iy2 = min(max((int)floorf(py + r_p - ofy), y0s), b0y + whi);
        const int iz1 = min(max((int)ceilf(pz - r_p - ofz), z0s), b0z + whi);
        const int iz2 = min(max((int)floorf(pz + r_p - ofz), z0s), b0z + whi);
        if (AT >= 0 && fin && ix2 - ix1 <= 3 && iy2 - iy1 <= 3 && iz2 - iz1 <= 3) {
            // r_p <= 2: the footprint is at most 4 cells wide on an axis
            // unless p - of is an integer there (5 wide: the loop below).
            // Offsets past the footprint get an infinite squared distance,
            // hence weight 0.
            float cx[4], cx2[4], cy[4], cy2[4], cz[4], cz2[4];
#pragma unroll
            for (int o = 0; o < 4; ++o) {
                cx[o] = (float)(ix1 + o) - px0;
                cy[o] = (float)(iy1 + o) - py0;
                cz[o] = (float)(iz1 + o) - pz0;
                cx2[o] = ix1 + o <= ix2 ? cx[o] * cx[o] : __builtin_inff();
                cy2[o] = iy1 + o <= iy2 ? cy[o] * cy[o] : __builtin_inff();
                cz2[o] = iz1 + o <= iz2 ? cz[o] * cz[o] : __builtin_inff();
                // computed once per particle: the empty statements keep the
                // compiler from recomputing them at each of the cells
                asm volatile("" : "+v"(cx[o]), "+v"(cx2[o]));
            }
            const int row = MSX, plane = MSX * MSX;
            double *base = acc + ((iz1 - z0s) * MSX + (iy1 - y0s)) * MSX + ix1 - x0s;
            // 1 - df2 / r_p^2 (Eq. 6) of face cell (ox, oy, oz) for the particle at p - 1/2
            auto t_of = [&](int ox, int oy, int oz) {
                const float dist_sq = cx2[ox] + (cz2[oz] + cy2[oy]);
                const float d_a = AT == 0 ? cx[ox] : (AT == 1 ? cy[oy] : cz[oz]);
                const float df2 = dist_sq + d_a + 0.25f;
                return 1.0f - df2 * inv_r2;
            };
            auto add = [&](double *at, float w) {
                if (w > 0.0f) {
                    const float w3 = w * w * w;
#pragma unroll
                    for (int k = 0; k < NC; ++k) unsafeAtomicAdd(at + k * NS, (double)(w3 * sc[k]));
                }
            };
            auto cell = [&](int ox, int oy, int oz) { add(base + oz * plane + oy * row + ox, t_of(ox, oy, oz)); };
            // Two cells of which at most one has a positive weight share an add.
            auto either = [&](int ax, int ay, int az, int bx, int by, int bz) {
                const float ta = t_of(ax, ay, az), tb = t_of(bx, by, bz);
                add(base + (tb > 0.0f ? bz * plane + by * row + bx : az * plane + ay * row + ax), fmaxf(ta, tb));
            };
            // On an axis the cells 0 and 3 lie d and 3 - d from the particle,
            // both at least r_p - 1 (a footprint cut at the domain's lower
            // bound has no cell 3, and its cell 0 is outside the domain).
            // Cells that swap 0 and 3 on two axes have squared distances that
            // sum to at least 4 (3/2)^2 = 9 > 2 r_p^2, so one of them is
            // outside the support.  Two of the 8 corners that differ on one
            // axis only sum to at least 9/2 + 4 (r_p - 1)^2, 1/2 + 2 (r_p - 2)^2
            // above 2 r_p^2: one corner at most is inside.  So 45 adds a
            // channel instead of 64 (4.55 -> 4.16 ms a direction; an add takes
            // 12 to 19 cycles, growing with the lanes that take part).
            float best = t_of(0, 0, 0);
            int at = 0;
#pragma unroll
            for (int c = 1; c < 8; ++c) {
                const int ox = c & 1 ? 3 : 0, oy = c & 2 ? 3 : 0, oz = c & 4 ? 3 : 0;
                const float tc = t_of(ox, oy, oz);
                at = tc > best ? oz * plane + oy * row + ox : at;
                best = fmaxf(best, tc);
            }
            add(base + at, best);
#pragma unroll
            for (int o = 1; o < 3; ++o) {
                either(0, o, 0, 3, o, 3);
                either(3, o, 0, 0, o, 3);
                either(o, 0, 0, o, 3, 3);
                either(o, 3, 0, o, 0, 3);
                either(0, 0, o, 3, 3, o);
                either(3, 0, o, 0, 3, o);
#pragma unroll
                for (int i = 1; i < 3; ++i) {
                    cell(o, i, 0);
                    cell(o, i, 3);
                    cell(o, 0, i);
                    cell(o, 3, i);
                    cell(0, o, i);
                    cell(3, o, i);
                    cell(1, o, i);
                    cell(2, o, i);
                }
            }
        } else {
            for (int iz = iz1; iz <= iz2; ++iz)
                for (int iy = iy1; iy <= iy2; ++iy)
                    for (int ix = ix1; ix <= ix2; ++ix) {
                        const float dz = (float)iz - pz0, dy = (float)iy - py0, dx = (float)ix - px0;
                        const float dist_sq = dx * dx + (dz * dz + dy * dy);
                        const float d_a = a == 0 ? dx : (a == 1 ? dy : dz);
                        const float df2 = dist_sq + d_a + 0.25f;
                        float w = fmaxf(1.0f - df2 * inv_r2, 0.0f);
                        w = w * w * w;
                        // a non-finite scale reaches its whole footprint, weights of 0 included
                        if (w > 0.0f || !fin) {
                            const int cell = ((iz - z0s) * MSX + (iy - y0s)) * MSX + ix - x0s;
#pragma unroll
                            for (int k = 0; k < NC; ++k) unsafeAtomicAdd(&acc[k * NS + cell], (double)(w * sc[k]));
                        }
                    }
        }
    }
    __syncthreads();
    float2 *out = win + (int64_t)blockIdx.x * NS;
    auto put = [&](int at, int s) {
        if (CH == 2)
            out[at] = make_float2((float)acc[s], (float)acc[NS + s]);
        else
            reinterpret_cast<float *>(out + at)[CH] = (float)acc[s];
    };
    const int rows = MSX * MSX;
    for (int s = threadIdx.x; s < rows * 16; s += kSplatThreads) put(s, (s >> 4) * MSX + m + (s & 15));
    for (int r = threadIdx.x; r < rows; r += kSplatThreads)
        for (int x = 0; x < m; ++x) {
            put(rows * 16 + r * m + x, r * MSX + x);
            put(rows * (16 + m) + r * m + x, r * MSX + 16 + m + x);
        }
}

// The commit (p2g.rs:342-411) and MacGrid::normalize_velocity (mac.rs:106-132)
// of one face direction: every cell of the active blocks takes the sum of the
// windows that cover it, in float64 and in a fixed order (own block, then the
// neighbours whose margin it lies in, each block's items in order), rounded
// once, and u = P / M (0 where M <= 0).  `first[b]` is the first item of block
// b and `count[b]` their number.  Source block S commits window region (rx,
// ry, rz), the margin below, its own 16 cells or the margin above on each
// axis, only when that lies inside the domain; a particle on the domain's
// upper z bound makes S a block of the layer above it.  Where the windows come
// in several passes, all but the first add to the grid's cells and only the
// last divides.  Adding the windows into the grid from the splat took 8 colour
// passes a direction, a zero fill before and a division pass after (67 M
// particles: 26 ms, 16 so; 100,000: 2.5 ms, 0.1).  It is bound by the windows'
// bytes on large sets and by its dependent loads on small ones.
//
// A work-group of 256 lanes takes one block, plane after plane; with SPLIT its
// 1,024 lanes take one plane, and the four groups of 256 share the items of
// every region (few blocks of many items).  One plane per work-group
// everywhere took twice as long on large sets (67 M particles: 3.9 ms a
// direction, 1.08 so): its chain of dependent loads (list, slots, ranges,
// windows) weighs as much as the cells of a plane.
template <bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 1024 : 256) void mac_commit_kernel(GridView gm, GridView gv,
                                                                        const int32_t *__restrict__ active,
                                                                        const int32_t *__restrict__ first,
                                                                        const int32_t *__restrict__ count,
                                                                        const float2 *__restrict__ win, int m,
                                                                        bool head, bool last) {
    __shared__ int s_first[27], s_count[27];
    __shared__ double s_part[2][3][SPLIT ? 256 : 1];
    const int bid = active[SPLIT ? blockIdx.x >> 4 : blockIdx.x];
    const int ms = gm.b2s[bid], vs = gv.b2s[bid];
    if (ms < 2 || vs < 2) return;
    const int bx = bid % gm.nx, by = (bid / gm.nx) % gm.ny, bz = bid / (gm.nx * gm.ny);
    if (threadIdx.x < 27) {
        const int t = threadIdx.x;
        const int o[3] = {t % 3 - 1, (t / 3) % 3 - 1, t / 9 - 1};
        const int b[3] = {bx + o[0], by + o[1], bz + o[2]}, nb[3] = {gm.nx, gm.ny, gm.nz + 1}, s[3] = {gm.sx, gm.sy, gm.sz};
        bool in = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            in = in && b[d] >= 0 && b[d] < nb[d];
            // this block is S's upper margin (o < 0), its own cells (0) or its lower margin
            in = in && b[d] * 16 + (o[d] > 0 ? 0 : 16) + (o[d] < 0 ? m : 0) <= s[d];
        }
        const int src = b[0] + gm.nx * (b[1] + gm.ny * b[2]);
        s_count[t] = in ? count[src] : 0;
        s_first[t] = in ? first[src] : 0;
    }
    __syncthreads();
    const int MSX = 16 + 2 * m, NS = MSX * MSX * MSX, rows = MSX * MSX;
    const int cell = threadIdx.x & 255, group = threadIdx.x >> 8;
    const int cx = cell & 15, cy = cell >> 4;
    // the one neighbour on each axis whose margin the cell lies in, or 0
    const int ox = cx < m ? -1 : (cx >= 16 - m ? 1 : 0), oy = cy < m ? -1 : (cy >= 16 - m ? 1 : 0);
    const int step = SPLIT ? 4 : 1;
#pragma unroll 1
    for (int cz = SPLIT ? (int)(blockIdx.x & 15) : 0; cz < 16; cz += SPLIT ? 16 : 1) {
        const int oz = cz < m ? -1 : (cz >= 16 - m ? 1 : 0);
        float *pm = gm.slab + (int64_t)ms * 4096 + cz * 256 + cell;
        float *pv = gv.slab + (int64_t)vs * 4096 + cz * 256 + cell;
        double sm = 0.0, sv = 0.0;
        if (!head && group == 0) {
            sm = (double)*pm;
            sv = (double)*pv;
        }
        // the first window of each region, all loads in flight together, then the rest four at a time
        float2 f[8];
        int n[8], at[8];  // a pass's windows are below 2^31 cells
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            n[k] = 0;
            f[k] = make_float2(0.0f, 0.0f);
            if ((k & 4) && !oz) continue;  // uniform
            const int kx = (k & 1) ? ox : 0, ky = (k & 2) ? oy : 0, kz = (k & 4) ? oz : 0;
            const int t = (kx + 1) + 3 * (ky + 1) + 9 * (kz + 1);
            n[k] = ((k & 1) && !ox) || ((k & 2) && !oy) ? 0 : s_count[t];
            const int row = (cz - 16 * kz + m) * MSX + cy - 16 * ky + m;
            at[k] = (s_first[t] + group) * NS +
                    (kx == 0 ? row * 16 + cx
                             : (kx < 0 ? rows * (16 + m) + row * m + cx : rows * 16 + row * m + cx - 16 + m));
            if (n[k] > group) f[k] = win[at[k]];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            sm += (double)f[k].x;
            sv += (double)f[k].y;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k)
            for (int j = group + step; j < n[k]; j += 4 * step) {
                float2 g[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    g[i] = j + i * step < n[k] ? win[at[k] + (j + i * step - group) * NS] : make_float2(0.0f, 0.0f);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    sm += (double)g[i].x;
                    sv += (double)g[i].y;
                }
            }
        if (SPLIT) {
            if (group > 0) {
                s_part[0][group - 1][cell] = sm;
                s_part[1][group - 1][cell] = sv;
            }
            __syncthreads();
            if (group > 0) return;
            for (int g = 0; g < 3; ++g) {
                sm += s_part[0][g][cell];
                sv += s_part[1][g][cell];
            }
        }
        const float mm = (float)sm, mv = (float)sv;
        *pm = mm;
        *pv = !last ? mv : (mm > 0.0f ? mv / mm : 0.0f);
    }
}

// first / count of each block from its items (first at its first one).
__global__ void splat_ranges_kernel(const SplatItem *__restrict__ items, int n, int32_t *__restrict__ first,
                                    int32_t *__restrict__ count) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int bid = items[i].bid;
    if (i > 0 && items[i - 1].bid == bid) return;
    int e = i + 1;
    while (e < n && items[e].bid == bid) ++e;
    first[bid] = i;
    count[bid] = e - i;
}

// ---------------------------------------------------------------------------
// B-spline transfers.
// ---------------------------------------------------------------------------
template <int ORDER>
__device__ __forceinline__ float bspline_w(float p, int ci) {
    const float x = (p - 0.5f) - (float)ci;
    const float ax = fabsf(x);
    if (ORDER == 1) return ax < 1.0f ? 1.0f - ax : 0.0f;
    if (ax < 0.5f) return 0.75f - x * x;
    if (ax < 1.5f) {
        const float t = 1.5f - ax;
        return 0.5f * t * t;
    }
    return 0.0f;
}

// Sorted particle records for the B-spline P2G, pm = (x, y, z, m) and
// pu = (u, v, w, 0), gathered from the caller-order records rec.
__global__ void gather_records_kernel(const float4 *__restrict__ rec, const uint32_t *__restrict__ perm, int64_t n,
                                      float4 *__restrict__ pm, float4 *__restrict__ pu) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = perm[i];
        pm[i] = rec[2 * j];
        pu[i] = rec[2 * j + 1];
    }
}

// Sort keys of the B-spline P2G, block id and voxel id (x fastest), and the
// particles' records in caller order: x-adjacent voxels of a block are one run
// of the sorted particles, and a voxel's particles keep their input order.  A
// particle outside the domain adds nothing: it becomes one of no mass and no
// velocity in a voxel of its own index's choosing.
__global__ void block_keys_pack_kernel(const float *__restrict__ pos, const float *__restrict__ vel,
                                       const float *__restrict__ mass, int64_t n, int sx, int sy, int sz, int nx,
                                       int ny, uint32_t n_keys, uint32_t *__restrict__ keys,
                                       uint32_t *__restrict__ idx, float4 *__restrict__ rec) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float px = pos[3 * i], py = pos[3 * i + 1], pz = pos[3 * i + 2];
        const uint32_t x = trunc_index(px), y = trunc_index(py), z = trunc_index(pz);
        float4 a = make_float4(px, py, pz, mass ? mass[i] : 1.0f);
        float4 b = make_float4(vel[3 * i], vel[3 * i + 1], vel[3 * i + 2], 0.0f);
        uint32_t key = ((x >> 4) + (uint32_t)nx * ((y >> 4) + (uint32_t)ny * (z >> 4))) << 12 | (x & 15) | (y & 15) << 4 |
                       (z & 15) << 8;
        if (x >= (uint32_t)sx || y >= (uint32_t)sy || z >= (uint32_t)sz) {
            key = (uint32_t)i * 2654435761u % n_keys;
            a = b = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        keys[i] = key;
        idx[i] = (uint32_t)i;
        rec[2 * i] = a;
        rec[2 * i + 1] = b;
    }
}

// The sorted particles [beg, end) of every voxel of the active blocks, indexed
// by slot * 4096 + vid; an empty voxel's range is empty where its particles
// would be, so neighbouring voxels' ranges join.  A work-group per block: its
// run by search, a count per voxel in LDS, their scan.  *widest: the particles of
// the fullest block.
__global__ __launch_bounds__(256) void voxel_ranges_kernel(const uint32_t *__restrict__ keys, uint32_t n,
                                                           const int32_t *__restrict__ active, GridView g,
                                                           uint2 *__restrict__ range, uint32_t *widest) {
    __shared__ uint32_t s_cnt[4096];
    __shared__ uint32_t s_run[2], s_sum[4];
    const uint32_t bid = (uint32_t)active[blockIdx.x];
    const int slot = g.b2s[bid], t = threadIdx.x;
    if (slot < 2) return;
    if (t < 128) {
        // the first particle whose key is not below the block's (wave 0) / the
        // next block's (wave 1): a wave probes 64 places at a time
        const uint32_t key = (bid + (t >> 6)) << 12, lane = t & 63;
        uint32_t lo = 0, hi = n;  // it lies in [lo, hi]
        while (lo < hi) {
            const uint32_t step = (hi - lo + 63) / 64, at = lo + lane * step;
            const uint32_t below = (uint32_t)__popcll(__ballot(at < hi && keys[at] < key));  // probes 0 .. below - 1
            if (below == 0) {
                hi = lo;
            } else {
                hi = min(hi, lo + below * step);
                lo = lo + (below - 1) * step + 1;
            }
        }
        if (lane == 0) s_run[t >> 6] = lo;
    }
    for (int v = t; v < 4096; v += 256) s_cnt[v] = 0;
    __syncthreads();
    const uint32_t b0 = s_run[0], b1 = s_run[1];
    uint4 *out = reinterpret_cast<uint4 *>(range + ((int64_t)slot << 12));
    if (b0 == b1) {  // most active blocks of a sparse set: the footprints' margins
        for (int v = t; v < 2048; v += 256) out[v] = make_uint4(b0, b0, b0, b0);
        return;
    }
    if (widest && t == 0) atomicMax(widest, b1 - b0);
    for (uint32_t i = b0 + t; i < b1; i += 256) atomicAdd(&s_cnt[keys[i] & 4095u], 1u);
    __syncthreads();
    uint32_t c[16], sum = 0;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        c[v] = s_cnt[16 * t + v];
        sum += c[v];
    }
    uint32_t x = sum;  // inclusive scan inside each wave, then wave sums
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if ((t & 63) >= o) x += y;
    }
    if ((t & 63) == 63) s_sum[t >> 6] = x;
    __syncthreads();
    uint32_t at = b0 + x - sum;
    for (int w = 0; w < t >> 6; ++w) at += s_sum[w];
#pragma unroll
    for (int v = 0; v < 16; v += 2) {
        const uint32_t m = at + c[v], e = m + c[v + 1];
        out[8 * t + v / 2] = make_uint4(at, m, m, e);
        at = e;
    }
}

struct Acc4 {
    float m, u0, u1, u2;
};

template <int ORDER>
__device__ __forceinline__ void acc_add(Acc4 &a, float wxy, float pz, int cz, float m, const float4 &u) {
    const float wm = (wxy * bspline_w<ORDER>(pz, cz)) * m;
    a.m = a.m + wm;
    a.u0 = a.u0 + wm * u.x;
    a.u1 = a.u1 + wm * u.y;
    a.u2 = a.u2 + wm * u.z;
}

// Workgroup per active block; lane (lx, ly) owns the cell column (lx, ly, *).
// A cell sums its 27 neighbour voxels, z then y then x from -1 to 1, and each
// voxel's particles in sorted order -- the oracle's order.  The lane walks the
// 18 voxel planes bz*16-1 .. bz*16+16 once: plane v feeds cells v+1 (as their
// dz = -1 plane), v (dz = 0) and v-1 (dz = +1), so each particle is read once
// per column and every cell still receives its planes in increasing z.
//
// A work-group takes the whole column, which has the least to read (18 planes
// for 16 cells), or (split = 4) on few blocks, where a column's chain of dependent
// reads is all the time, a span of 4 (6 planes); there too a quarter of the
// work-groups take whole columns where no block holds more than `even` particles
// (*widest), so that the columns are a full and even load.
// Bound by its arithmetic and by lanes that wait for the fullest of their wave
// (16.8 M particles in 9,000 blocks, quadratic: 1,240 us with 9 voxels a plane
// to step through, most of them empty, 1,025 with joined rows; 1 M in 350
// blocks, linear: 375 and 120).
template <int ORDER>
__global__ __launch_bounds__(256) void p2g_bspline_kernel(GridView mg, GridView v0, GridView v1, GridView v2,
                                                          const int32_t *__restrict__ active,
                                                          const uint32_t *__restrict__ flags,
                                                          const uint2 *__restrict__ range,
                                                          const float4 *__restrict__ pm,
                                                          const float4 *__restrict__ pu, int split,
                                                          const uint32_t *__restrict__ widest, uint32_t even) {
    __shared__ int s_nb[27];
    // voxel ranges of the block's 18 x 18 plane window (the block's columns
    // and a 1-voxel ring), double-buffered: plane v + 1 loads during plane v
    __shared__ uint2 s_pl[2][18 * 18];
    // (the first quarter of the work-groups then: every fourth of them would all
    // fall on two of the 8 XCDs)
    const bool joined = even && *widest <= even;
    if (joined && blockIdx.x >= gridDim.x / split) return;
    const int64_t bid = active[joined ? blockIdx.x : blockIdx.x / split];
    const int part = joined ? 0 : (int)(blockIdx.x % split);
    const int span = joined ? 16 : 16 / split, lz0 = part * span;  // cells of the span, the first of them
    const int bx = (int)(bid % mg.nx), by = (int)((bid / mg.nx) % mg.ny), bz = (int)(bid / ((int64_t)mg.nx * mg.ny));
    if (threadIdx.x < 27) {
        const int t = threadIdx.x;
        const int nx = bx + t % 3 - 1, ny = by + (t / 3) % 3 - 1, nz = bz + t / 9 - 1;
        // only blocks active in this call have ranges; a value block that is not
        // (one of an earlier call, or the caller's own) holds no particle
        int slot = 0;
        if (nx >= 0 && nx < mg.nx && ny >= 0 && ny < mg.ny && nz >= 0 && nz < mg.nz) {
            const int64_t nb = nx + (int64_t)ny * mg.nx + (int64_t)nz * mg.nx * mg.ny;
            const uint32_t on = flags[nb];
            slot = mg.b2s[nb];
            if (!on) slot = 0;
        }
        s_nb[t] = slot;
    }
    __syncthreads();
    const int ms = s_nb[13];
    const int s0 = v0.b2s[bid], s1 = v1.b2s[bid], s2 = v2.b2s[bid];
    if (ms < 2) return;
    const int lx = threadIdx.x & 15, ly = threadIdx.x >> 4;
    const int cx = bx * 16 + lx, cy = by * 16 + ly, cz0 = bz * 16 + lz0;
    Acc4 lo = {0, 0, 0, 0}, mid = {0, 0, 0, 0}, hi = {0, 0, 0, 0};  // cells lv-1, lv, lv+1
    auto store = [&](int lz, const Acc4 &a) {
        const int vid = lx | (ly << 4) | ((lz0 + lz) << 8);
        mg.slab[(int64_t)ms * 4096 + vid] = a.m;
        const bool pos_m = a.m > 0.0f;
        v0.slab[(int64_t)s0 * 4096 + vid] = pos_m ? a.u0 / a.m : 0.0f;
        v1.slab[(int64_t)s1 * 4096 + vid] = pos_m ? a.u1 / a.m : 0.0f;
        v2.slab[(int64_t)s2 * 4096 + vid] = pos_m ? a.u2 / a.m : 0.0f;
    };
    // Ranges of window voxels idx and idx + 256 (idx < 324) of plane vz; an
    // outside or absent voxel is an empty range.
    auto plane_ranges = [&](int vz, uint2 *r) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int idx = threadIdx.x + 256 * h;
            r[h] = make_uint2(0u, 0u);
            if (idx >= 18 * 18 || vz < 0 || vz >= mg.sz) continue;
            const int vy = by * 16 - 1 + idx / 18, vx = bx * 16 - 1 + idx % 18;
            // (not past the domain's last block; a voxel past its last cell has an empty range in its place)
            if (vy < 0 || (vy >> 4) >= mg.ny || vx < 0 || (vx >> 4) >= mg.nx) continue;
            const int slot = s_nb[((vx >> 4) - bx + 1) + 3 * ((vy >> 4) - by + 1) + 9 * ((vz >> 4) - bz + 1)];
            if (slot < 2) continue;
            const int64_t c = (int64_t)slot * 4096 + ((vx & 15) | ((vy & 15) << 4) | ((vz & 15) << 8));
            r[h] = range[c];
        }
    };
    auto put_plane = [&](int buf, const uint2 *r) {
        s_pl[buf][threadIdx.x] = r[0];
        if (threadIdx.x + 256 < 18 * 18) s_pl[buf][threadIdx.x + 256] = r[1];
    };
    uint2 nxt[2];
    plane_ranges(cz0 - 1, nxt);
    put_plane(0, nxt);
    __syncthreads();
    for (int lv = -1; lv <= span; ++lv) {
        const int vz = cz0 + lv, cur = (lv + 1) & 1;
        if (lv < span) plane_ranges(vz + 1, nxt);  // in flight while this plane's particles are added
        if (vz >= 0 && vz < mg.sz) {
            // This lane's 9 voxels are window voxels (ly + dy + 1, lx + dx + 1).
            // The three of a row are one run of the sorted particles, or two
            // where a block ends between them: 6 runs, the second one of a row
            // empty but for the first and the last lane of a row.  One pass
            // over their concatenation: a wave steps as often as its fullest
            // lane has particles.  Per cell, the particles still arrive voxel
            // by voxel in (dy, dx) order, sorted within.
            const uint2 *pl = s_pl[cur] + ly * 18 + lx;
            auto rng = [&](int t) {
                const uint2 *row = pl + (t >> 1) * 18;
                const uint2 a = row[0], m = row[1], b = row[2];
                // lane 0: {-1}, {0, 1}; lane 15: {14, 15}, {16}; the others {-1, 0, 1}
                if (t & 1) return lx == 0 ? make_uint2(m.x, b.y) : (lx == 15 ? b : make_uint2(0u, 0u));
                return make_uint2(a.x, lx == 0 ? a.y : (lx == 15 ? m.y : b.y));
            };
            const int step = lx == 0 || lx == 15 ? 1 : 2;
            int t = 0;
            uint2 rt = rng(0);
            uint32_t j = rt.x, e = rt.y;
            while (j >= e && (t += step) < 6) {
                rt = rng(t);
                j = rt.x;
                e = rt.y;
            }
            float4 pn = make_float4(0.f, 0.f, 0.f, 0.f), un = pn;
            if (t < 6) {
                pn = pm[j];
                un = pu[j];
            }
            while (t < 6) {
                const float4 p = pn, u = un;
                ++j;
                while (j >= e && (t += step) < 6) {
                    rt = rng(t);
                    j = rt.x;
                    e = rt.y;
                }
                if (t < 6) {  // the next particle's records are in flight while this one is added
                    pn = pm[j];
                    un = pu[j];
                }
                const float wxy = bspline_w<ORDER>(p.x, cx) * bspline_w<ORDER>(p.y, cy);
                if (lv >= 1) acc_add<ORDER>(lo, wxy, p.z, cz0 + lv - 1, p.w, u);
                if (lv >= 0 && lv <= span - 1) acc_add<ORDER>(mid, wxy, p.z, cz0 + lv, p.w, u);
                if (lv <= span - 2) acc_add<ORDER>(hi, wxy, p.z, cz0 + lv + 1, p.w, u);
            }
        }
        if (lv < span) put_plane(cur ^ 1, nxt);  // buffer cur ^ 1 was last read before the previous barrier
        __syncthreads();
        if (lv >= 1) store(lv - 1, lo);  // cell lv-1 has its planes lv-2, lv-1, lv
        lo = mid;
        mid = hi;
        hi = Acc4{0, 0, 0, 0};
    }
}

// G2P work-groups: 256 consecutive Morton-sorted particles each.  The grid
// cells their supports reach (the chunk's box of floor(p) -1 .. +1, clipped
// to the domain) are staged in LDS when the box holds at most kG2pWindow
// cells; a chunk with a larger box (it straddles a coarse Morton boundary)
// reads the slabs directly.  Both paths take the same values in the same
// order, so the result does not depend on which one runs.
constexpr int kG2pThreads = 256;
constexpr int kG2pWindow = 3072;
constexpr int kG2pWindowBlocks = 64;  // 16^3 blocks a staged box may touch

// floor(p) as a cell index, held to [-2, s + 1]: beyond that every support
// cell floor(p) - 1 .. floor(p) + 1 lies outside the domain either way, and
// the float -> int conversion stays in range (NaN maps to -2: no cells).
__device__ __forceinline__ int floor_cell(float p, int s) {
    return (int)fminf(fmaxf(floorf(p), -2.0f), (float)(s + 1));
}

// Cell range [lo, hi] of one axis of a particle's support, clipped to the
// domain (empty when lo > hi).
__device__ __forceinline__ void support_range(int f, int s, int &lo, int &hi) {
    lo = max(f - 1, 0);
    hi = min(f + 1, s - 1);
}

// One particle's sum over its 27 support cells (z, then y, then x), the
// oracle's order.  STAGED reads the cells from the LDS window `win` (box
// origin x0, y0, z0, extents ex, ey), else straight from the slabs.
template <int ORDER, bool STAGED>
__device__ __forceinline__ void g2p_sum(const GridView &v0, const GridView &v1, const GridView &v2, float px,
                                        float py, float pz, int fx, int fy, int fz, const float (*win)[kG2pWindow],
                                        int x0, int y0, int z0, int ex, int ey, float &a0, float &a1, float &a2) {
    a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
    for (int dz = -1; dz <= 1; ++dz) {
        const int cz = fz + dz;
        if (cz < 0 || cz >= v0.sz) continue;
        const float wz = bspline_w<ORDER>(pz, cz);
        for (int dy = -1; dy <= 1; ++dy) {
            const int cy = fy + dy;
            if (cy < 0 || cy >= v0.sy) continue;
            const float wy = bspline_w<ORDER>(py, cy);
            for (int dx = -1; dx <= 1; ++dx) {
                const int cx = fx + dx;
                if (cx < 0 || cx >= v0.sx) continue;
                const float w = (bspline_w<ORDER>(px, cx) * wy) * wz;
                float s0, s1, s2;
                if constexpr (STAGED) {  // every in-domain support cell lies in the box
                    const int c = ((cz - z0) * ey + (cy - y0)) * ex + (cx - x0);
                    s0 = win[0][c];
                    s1 = win[1][c];
                    s2 = win[2][c];
                } else {
                    const int64_t bid =
                        (cx >> 4) + (int64_t)(cy >> 4) * v0.nx + (int64_t)(cz >> 4) * v0.nx * v0.ny;
                    const int vid = (cx & 15) | ((cy & 15) << 4) | ((cz & 15) << 8);
                    s0 = v0.slab[(int64_t)v0.b2s[bid] * 4096 + vid];
                    s1 = v1.slab[(int64_t)v1.b2s[bid] * 4096 + vid];
                    s2 = v2.slab[(int64_t)v2.b2s[bid] * 4096 + vid];
                }
                a0 = a0 + w * s0;
                a1 = a1 + w * s1;
                a2 = a2 + w * s2;
            }
        }
    }
}

template <int ORDER>
__global__ __launch_bounds__(kG2pThreads) void g2p_bspline_kernel(GridView v0, GridView v1, GridView v2,
                                                                  const float *__restrict__ pos, int64_t n,
                                                                  const uint32_t *__restrict__ visit,
                                                                  float *__restrict__ out) {
    __shared__ float win[3][kG2pWindow];
    __shared__ int s_box[6];                    // min x, y, z; max x, y, z of the chunk's support cells
    __shared__ int s_slot[3][kG2pWindowBlocks];  // slab slot of each block the box touches, per component
    // Consecutive chunks (neighbouring cells) land on one XCD and share its L2.
    const int64_t k = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * kG2pThreads + threadIdx.x;
    if (threadIdx.x < 3) s_box[threadIdx.x] = INT_MAX;
    else if (threadIdx.x < 6) s_box[threadIdx.x] = INT_MIN;
    int64_t i = -1;
    float px = 0.0f, py = 0.0f, pz = 0.0f;
    int fx = 0, fy = 0, fz = 0;
    // support box of this lane, inverted (no cells) unless it reaches the domain
    int lx = INT_MAX, ly = INT_MAX, lz = INT_MAX, hx = INT_MIN, hy = INT_MIN, hz = INT_MIN;
    if (k < n) {
        i = visit[k];
        px = pos[3 * i], py = pos[3 * i + 1], pz = pos[3 * i + 2];
        fx = floor_cell(px, v0.sx), fy = floor_cell(py, v0.sy), fz = floor_cell(pz, v0.sz);
        int ax, bx, ay, by, az, bz;
        support_range(fx, v0.sx, ax, bx);
        support_range(fy, v0.sy, ay, by);
        support_range(fz, v0.sz, az, bz);
        if (ax <= bx && ay <= by && az <= bz) lx = ax, hx = bx, ly = ay, hy = by, lz = az, hz = bz;
    }
    // wave-level min / max first: one LDS atomic per wave and bound
    for (int o = 32; o > 0; o >>= 1) {
        lx = min(lx, __shfl_xor(lx, o)), ly = min(ly, __shfl_xor(ly, o)), lz = min(lz, __shfl_xor(lz, o));
        hx = max(hx, __shfl_xor(hx, o)), hy = max(hy, __shfl_xor(hy, o)), hz = max(hz, __shfl_xor(hz, o));
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0 && lx <= hx) {
        atomicMin(&s_box[0], lx);
        atomicMin(&s_box[1], ly);
        atomicMin(&s_box[2], lz);
        atomicMax(&s_box[3], hx);
        atomicMax(&s_box[4], hy);
        atomicMax(&s_box[5], hz);
    }
    __syncthreads();
    const int x0 = s_box[0], y0 = s_box[1], z0 = s_box[2];
    // box extents; none of the chunk's lanes reaching the domain leaves the box inverted (ex <= 0)
    const int64_t ex = (int64_t)s_box[3] - x0 + 1, ey = (int64_t)s_box[4] - y0 + 1, ez = (int64_t)s_box[5] - z0 + 1;
    const int bx0 = x0 >> 4, by0 = y0 >> 4, bz0 = z0 >> 4;
    const int64_t nbx = ex > 0 ? ((s_box[3] >> 4) - bx0 + 1) : 0, nby = ex > 0 ? ((s_box[4] >> 4) - by0 + 1) : 0,
                  nbz = ex > 0 ? ((s_box[5] >> 4) - bz0 + 1) : 0;
    float a0, a1, a2;
    // uniform over the work-group
    if (ex > 0 && ex * ey * ez <= kG2pWindow && nbx * nby * nbz <= kG2pWindowBlocks) {
        const int nbxy = (int)(nbx * nby), nb = (int)(nbxy * nbz);
        if (threadIdx.x < nb) {
            const int t = threadIdx.x;
            const int64_t bid = (bx0 + t % (int)nbx) + (int64_t)(by0 + (t % nbxy) / (int)nbx) * v0.nx +
                                (int64_t)(bz0 + t / nbxy) * v0.nx * v0.ny;
            s_slot[0][t] = v0.b2s[bid];
            s_slot[1][t] = v1.b2s[bid];
            s_slot[2][t] = v2.b2s[bid];
        }
        __syncthreads();
        // Each lane's cells are addressed first and loaded back to back.
        constexpr int ITEMS = kG2pWindow / kG2pThreads;
        const int exy = (int)(ex * ey), nw = (int)(exy * ez);
        int64_t off[3][ITEMS];
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) {
            const int c = threadIdx.x + q * kG2pThreads;
            off[0][q] = off[1][q] = off[2][q] = -1;
            if (c < nw) {
                const int cz = z0 + c / exy, cy = y0 + (c % exy) / (int)ex, cx = x0 + c % (int)ex;
                const int b = ((cx >> 4) - bx0) + (int)nbx * ((cy >> 4) - by0) + nbxy * ((cz >> 4) - bz0);
                const int vid = (cx & 15) | ((cy & 15) << 4) | ((cz & 15) << 8);
                off[0][q] = (int64_t)s_slot[0][b] * 4096 + vid;
                off[1][q] = (int64_t)s_slot[1][b] * 4096 + vid;
                off[2][q] = (int64_t)s_slot[2][b] * 4096 + vid;
            }
        }
        float val[3][ITEMS];
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) {
            val[0][q] = off[0][q] >= 0 ? v0.slab[off[0][q]] : 0.0f;
            val[1][q] = off[1][q] >= 0 ? v1.slab[off[1][q]] : 0.0f;
            val[2][q] = off[2][q] >= 0 ? v2.slab[off[2][q]] : 0.0f;
        }
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) {
            const int c = threadIdx.x + q * kG2pThreads;
            if (c < nw) win[0][c] = val[0][q], win[1][c] = val[1][q], win[2][c] = val[2][q];
        }
        __syncthreads();
        if (k >= n) return;
        g2p_sum<ORDER, true>(v0, v1, v2, px, py, pz, fx, fy, fz, win, x0, y0, z0, (int)ex, (int)ey, a0, a1, a2);
    } else {
        if (k >= n) return;
        g2p_sum<ORDER, false>(v0, v1, v2, px, py, pz, fx, fy, fz, win, 0, 0, 0, 0, 0, a0, a1, a2);
    }
    out[3 * i] = a0;
    out[3 * i + 1] = a1;
    out[3 * i + 2] = a2;
}

// Ensures `bids` (host) on every grid and zero-fills them (MacGrid::zero_blocks,
// mac.rs:95-102).
int zero_blocks(msbg_grid *const *grids, int ng, const std::vector<int64_t> &bids) {
    for (int k = 0; k < ng; ++k) {
        int rc = msbg_grid_ensure_blocks(grids[k], bids.data(), (int64_t)bids.size());
        if (rc) return rc;
        rc = msbg_grid_fill_blocks(grids[k], bids.data(), (int64_t)bids.size(), 0.0f);
        if (rc) return rc;
    }
    return MSBG_OK;
}

int check_same_dims(msbg_grid *const *grids, int ng) {
    for (int k = 0; k < ng; ++k) {
        MSBG_CHECK(grids[k], MSBG_EINVAL, "transfer: null grid");
        MSBG_CHECK(grids[k]->L == 4 && grids[k]->sx == grids[0]->sx && grids[k]->sy == grids[0]->sy &&
                       grids[k]->sz == grids[0]->sz,
                   MSBG_EINVAL, "transfer: all channels must be 16^3-block grids over one domain");
    }
    return MSBG_OK;
}

// Active blocks of the particles (device list, and a flag per block), downloaded.
int active_list(const msbg_grid *g, const float *d_pos, int64_t n, float r_scan, std::vector<int64_t> &out,
                int32_t **d_list, const uint32_t **d_flags = nullptr) {
    int rc;
    int32_t *d_act = (int32_t *)workspace(6, sizeof(int32_t) * std::max<int64_t>(g->n_blocks, 1), &rc);
    if (rc) return rc;
    int64_t k = 0;
    const uint32_t *flags = nullptr;
    rc = active_blocks_flagged(g->sx, g->sy, g->sz, d_pos, n, r_scan, d_act, &k, &flags);
    if (rc) return rc;
    if (d_flags) *d_flags = flags;
    std::vector<int32_t> h((size_t)k);
    if (k) MSBG_HIP(hipMemcpy(h.data(), d_act, sizeof(int32_t) * k, hipMemcpyDeviceToHost));
    out.assign(h.begin(), h.end());
    *d_list = d_act;
    return MSBG_OK;
}

// `bytes` of splat windows for `g`: small ones in the shared workspace, large
// ones g's own, kept until it is freed.  (Given back and taken anew by every FLIP
// step of 67 M particles, 53% of the steps waited 10 ms to 2 s for the driver to
// hand out memory that was freed just before; kept, 32%, as in its other buffers.)
int splat_windows(msbg_grid *g, size_t bytes, float2 **win) {
    int rc = MSBG_OK;
    if (bytes <= kSplatShared) {
        *win = (float2 *)workspace(24, bytes, &rc);
        return rc;
    }
    if (bytes > g->window_bytes) {
        constexpr size_t kStep = (size_t)256 << 20;  // (a growing set takes new ones seldom)
        bytes = (bytes + kStep - 1) / kStep * kStep;
        if (g->d_windows) {
            MSBG_HIP(hipStreamSynchronize(stream()));
            (void)hipFree(g->d_windows);
            g->d_windows = nullptr;
            g->window_bytes = 0;
        }
        const hipError_t e = hipMalloc(&g->d_windows, bytes);
        if (e != hipSuccess) {
            g->d_windows = nullptr;
            return e == hipErrorOutOfMemory ? fail(MSBG_ENOMEM, "particles_to_grid: out of device memory")
                                            : hip_fail(e, "particles_to_grid windows");
        }
        g->window_bytes = bytes;
    }
    *win = (float2 *)g->d_windows;
    return MSBG_OK;
}

}  // namespace msbg

using namespace msbg;

extern "C" {

int msbg_sample(const msbg_grid *g, const float *d_pos, int64_t n, int interp, int align, int bc, float *d_out) {
    MSBG_CHECK(g && g->L == 4, MSBG_EINVAL, "sample: 16^3-block grid required");
    MSBG_CHECK(interp == 0 || interp == 1, MSBG_EINVAL, "sample: interp is 0 (Linear) or 1 (CubicBSpline)");
    MSBG_CHECK((align == 0 || align == 1) && bc >= 0 && bc <= 2, MSBG_EINVAL, "sample: bad alignment / boundary");
    MSBG_CHECK(n >= 0 && (n == 0 || (d_pos && d_out)), MSBG_EINVAL, "sample: null argument");
    if (n == 0) return MSBG_OK;
    launch_sample(g->view(), d_pos, n, interp, align, bc, -1, d_out, 1);
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}

int msbg_mac_sample(msbg_grid *const *vel, const float *d_pos, int64_t n, int interp, int bc, float *d_out) {
    MSBG_CHECK(vel, MSBG_EINVAL, "mac sample: null grids");
    int rc = check_same_dims(vel, 3);
    if (rc) return rc;
    MSBG_CHECK(interp == 0 || interp == 1, MSBG_EINVAL, "mac sample: interp is 0 or 1");
    MSBG_CHECK(bc >= 0 && bc <= 2, MSBG_EINVAL, "mac sample: bad boundary");
    MSBG_CHECK(n >= 0 && (n == 0 || (d_pos && d_out)), MSBG_EINVAL, "mac sample: null argument");
    if (n == 0) return MSBG_OK;
    for (int a = 0; a < 3; ++a)
        launch_sample(vel[a]->view(), d_pos, n, interp, 1, bc, a, d_out + a, 3);
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}

int msbg_g2p_blend(const float *d_u_old, const float *d_u, const float *d_u_tilde, int64_t n, float alpha,
                   float *d_out) {
    MSBG_CHECK(n >= 0 && (n == 0 || (d_u_old && d_u && d_u_tilde && d_out)), MSBG_EINVAL, "g2p blend: null argument");
    if (n == 0) return MSBG_OK;
    hipLaunchKernelGGL(blend_kernel, dim3(grid_for(3 * n, 256)), dim3(256), 0, stream(), d_u_old, d_u, d_u_tilde, 3 * n,
                       alpha, d_out);
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}

int msbg_g2p_flip(msbg_grid *const *vel, msbg_grid *const *vel_tilde, const float *d_pos, const float *d_u_old,
                  int64_t n, int interp, int bc, float alpha, float *d_out) {
    MSBG_CHECK(vel && vel_tilde, MSBG_EINVAL, "g2p flip: null grids");
    msbg_grid *all[6] = {vel[0], vel[1], vel[2], vel_tilde[0], vel_tilde[1], vel_tilde[2]};
    int rc = check_same_dims(all, 6);
    if (rc) return rc;
    MSBG_CHECK(interp == 0 || interp == 1, MSBG_EINVAL, "g2p flip: interp is 0 or 1");
    MSBG_CHECK(bc >= 0 && bc <= 2, MSBG_EINVAL, "g2p flip: bad boundary");
    MSBG_CHECK(n >= 0 && (n == 0 || (d_pos && d_u_old && d_out)), MSBG_EINVAL, "g2p flip: null argument");
    if (n == 0) return MSBG_OK;
    MacViews u, ut;
    for (int a = 0; a < 3; ++a) {
        u.v[a] = vel[a]->view();
        ut.v[a] = vel_tilde[a]->view();
    }
    const int64_t groups = (n + kFlipThreads - 1) / kFlipThreads;
    const bool dense = n >= kFlipPerBlock * (vel[0]->n_slots - 2);
    // a lane a particle; past 2^32 lanes stride
    if (interp == 0 && (dense || n <= kFlipFew) && groups <= max_groups(kFlipThreads))
        hipLaunchKernelGGL(g2p_flip_linear_kernel, dim3((unsigned)groups), dim3(kFlipThreads), 0, stream(), u, ut, d_pos,
                           d_u_old, n, bc, alpha, dense ? kFlipBlocks : kFlipBlocksFew, d_out);
    else if (interp == 0)
        hipLaunchKernelGGL(g2p_flip_kernel<0>, dim3(grid_for(n, 256)), dim3(256), 0, stream(), u, ut, d_pos, d_u_old,
                           n, bc, alpha, d_out);
    else
        hipLaunchKernelGGL(g2p_flip_kernel<1>, dim3(grid_for(n, 256)), dim3(256), 0, stream(), u, ut, d_pos, d_u_old,
                           n, bc, alpha, d_out);
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}

int msbg_particles_to_grid_mac(msbg_grid *const *vel, msbg_grid *const *mass, const float *d_pos, const float *d_vel,
                               const float *d_mass, int64_t n, float r_p, int64_t *n_active) {
    MSBG_CHECK(vel && mass && n_active, MSBG_EINVAL, "particles_to_grid: null argument");
    msbg_grid *all[6] = {vel[0], vel[1], vel[2], mass[0], mass[1], mass[2]};
    int rc = check_same_dims(all, 6);
    if (rc) return rc;
    // splat precondition (p2g.rs:32-42, 174-181): 0 < r_p <= margin, staging fits LDS.
    MSBG_CHECK(r_p > 0.0f && r_p <= 3.0f, MSBG_EINVAL, "particles_to_grid: r_p must be in (0, 3]");
    MSBG_CHECK(n >= 0 && n < ((int64_t)1 << 31) && (n == 0 || (d_pos && d_vel && d_mass)), MSBG_EINVAL,
               "particles_to_grid: bad particle arrays");
    const msbg_grid *g = vel[0];
    // active blocks with the (r_p + 1)/bsx footprint (p2g.rs:104-107); the
    // commit writes every cell of them
    std::vector<int64_t> act;
    int32_t *d_act = nullptr;
    rc = active_list(g, d_pos, n, r_p + 1.0f, act, &d_act);
    if (rc) return rc;
    for (msbg_grid *c : all) {
        rc = msbg_grid_ensure_blocks(c, act.data(), (int64_t)act.size());
        if (rc) return rc;
    }
    *n_active = (int64_t)act.size();
    if (n == 0) return MSBG_OK;
    // bucket by block (p2g.rs:149-158).  Particles that arrive grouped by
    // block (Morton-sorted, as a FLIP step passes them) skip the sort and the
    // payload gather: the runs of the input are the buckets.
    uint32_t *keys = (uint32_t *)workspace(4, sizeof(uint32_t) * 2 * n + 2 * sizeof(int32_t), &rc);
    if (rc) return rc;
    uint32_t *perm = keys + n;
    int32_t *d_ungrouped = (int32_t *)(perm + n);
    hipLaunchKernelGGL(set_flag_kernel, dim3(1), dim3(1), 0, stream(), d_ungrouped, 0);
    // block ids, one layer past the upper z bound included, and `most` for all beyond
    const int64_t most = g->n_blocks + (int64_t)g->nx * g->ny;
    hipLaunchKernelGGL(bucket_keys_grouped_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream(), d_pos, n,
                       (int32_t)g->nx, (int32_t)g->ny, (uint32_t)most, keys, perm, d_ungrouped);
    MSBG_HIP(hipGetLastError());
    int32_t ungrouped = 1;
    MSBG_HIP(hipMemcpyAsync(&ungrouped, d_ungrouped, sizeof(int32_t), hipMemcpyDeviceToHost, stream()));
    MSBG_HIP(hipStreamSynchronize(stream()));
    float *pay = (float *)workspace(7, sizeof(float) * 7 * n + sizeof(int32_t) * (2 * n + 2), &rc);
    if (rc) return rc;
    const float *spos = d_pos, *svel = d_vel, *smass = d_mass;
    int32_t *pblocks = (int32_t *)(pay + 7 * n), *starts = pblocks + n;
    if (ungrouped) {
        int key_bits = 1;
        while (key_bits < 32 && ((int64_t)1 << key_bits) <= most) ++key_bits;
        rc = radix_sort_pairs(keys, perm, n, key_bits);
        if (rc) return rc;
        hipLaunchKernelGGL(gather_payload_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream(), d_pos, d_vel, d_mass,
                           perm, n, pay, pay + 3 * n, pay + 6 * n);
        MSBG_HIP(hipGetLastError());
        spos = pay;
        svel = pay + 3 * n;
        smass = pay + 6 * n;
    }
    int64_t nocc = 0;
    rc = run_lengths(keys, n, pblocks, starts, &nocc);
    if (rc) return rc;
    // the blocks' particles, cut into items
    std::vector<int32_t> hb((size_t)nocc), hs((size_t)nocc + 1);
    MSBG_HIP(hipMemcpy(hb.data(), pblocks, sizeof(int32_t) * nocc, hipMemcpyDeviceToHost));
    MSBG_HIP(hipMemcpy(hs.data(), starts, sizeof(int32_t) * (nocc + 1), hipMemcpyDeviceToHost));
    int32_t cut = kSplatLeast;
    while (cut < kSplatMost && (int64_t)cut * kSplatItems < n) cut *= 2;
    std::vector<SplatItem> order;
    order.reserve((size_t)(nocc + n / cut));
    for (int64_t i = 0; i < nocc; ++i) {
        if (hb[i] >= most) continue;
        const int64_t cnt = hs[i + 1] - hs[i], parts = (cnt + cut - 1) / cut;
        for (int64_t p = 0; p < parts; ++p)
            order.push_back(SplatItem{hb[i], (int32_t)(hs[i] + cnt * p / parts), (int32_t)(hs[i] + cnt * (p + 1) / parts)});
    }
    const int n_items = (int)order.size();
    const int m = (int)ceilf(r_p);
    const int msx = 16 + 2 * m, ns = msx * msx * msx;
    // items, and the item range of each block
    SplatItem *d_order = (SplatItem *)workspace(3, sizeof(SplatItem) * n_items + sizeof(int32_t) * 2 * most, &rc);
    if (rc) return rc;
    int32_t *d_first = (int32_t *)(d_order + n_items), *d_count = d_first + most;
    // the windows of at most `chunk` items: up to 2 GiB, less where that does not fit the device
    int chunk = std::max(1, std::min(n_items, (int)(((int64_t)1 << 31) / ((int64_t)sizeof(float2) * ns))));
    float2 *win = nullptr;
    for (;; chunk = (chunk + 1) / 2) {
        rc = splat_windows(mass[0], sizeof(float2) * ns * (size_t)chunk, &win);
        if (!rc) break;
        if (rc != MSBG_ENOMEM || chunk <= 16) return rc;
        (void)hipGetLastError();
    }
    if (n_items)
        MSBG_HIP(hipMemcpyAsync(d_order, order.data(), sizeof(SplatItem) * n_items, hipMemcpyHostToDevice, stream()));
    // both channels in one pass when two float64 windows fit (r_p <= 2), else a pass per channel
    const bool both = ns <= kSplatMaxCells;
    const size_t lds = (both ? 2 : 1) * sizeof(double) * ns;
    {
        int dev = 0, max_lds = 0;
        MSBG_HIP(hipGetDevice(&dev));
        MSBG_HIP(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
        MSBG_CHECK((int64_t)lds <= max_lds, MSBG_EINVAL,
                   "particles_to_grid: the staging window for this r_p exceeds the workgroup LDS limit");
        if (lds > 65536) {
            const void *fns[5] = {(const void *)mac_splat_kernel<0, -1>, (const void *)mac_splat_kernel<1, -1>,
                                  (const void *)mac_splat_kernel<2, 0>, (const void *)mac_splat_kernel<2, 1>,
                                  (const void *)mac_splat_kernel<2, 2>};
            for (const void *f : fns)
                MSBG_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        }
    }
    const float inv_r2 = 1.0f / (r_p * r_p);
    for (int at = 0; at == 0 || at < n_items; at += chunk) {
        const int cnt = std::min(chunk, n_items - at);
        const bool head = at == 0, last = at + chunk >= n_items;
        hipLaunchKernelGGL(fill_i32_kernel, dim3(grid_for(most, 256)), dim3(256), 0, stream(), d_count, most, 0);
        if (cnt > 0)
            hipLaunchKernelGGL(splat_ranges_kernel, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, stream(),
                               d_order + at, cnt, d_first, d_count);
        for (int a = 0; a < 3; ++a) {
            const auto splat = [&](auto kernel) {
                if (cnt > 0)
                    kernel<<<cnt, kSplatThreads, lds, stream()>>>((int)g->nx, (int)g->ny, a, d_order + at, spos, svel,
                                                                  smass, r_p, inv_r2, m, win);
            };
            if (!both) {
                splat(mac_splat_kernel<0, -1>);
                splat(mac_splat_kernel<1, -1>);
            } else if (a == 0) {
                splat(mac_splat_kernel<2, 0>);
            } else if (a == 1) {
                splat(mac_splat_kernel<2, 1>);
            } else {
                splat(mac_splat_kernel<2, 2>);
            }
            // below four blocks a CU a plane per work-group, or the chip idles
            // (48 blocks: 14 us, 106 with a block's items read by one group of lanes)
            const unsigned nact = (unsigned)act.size();
            if (nact > 0 && nact < 1024)
                mac_commit_kernel<true><<<16 * nact, 1024, 0, stream()>>>(mass[a]->view(), vel[a]->view(), d_act, d_first,
                                                                         d_count, win, m, head, last);
            else if (nact > 0)
                mac_commit_kernel<false><<<nact, 256, 0, stream()>>>(mass[a]->view(), vel[a]->view(), d_act, d_first,
                                                                     d_count, win, m, head, last);
            MSBG_HIP(hipGetLastError());
        }
    }
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}

int msbg_p2g_bspline(int order, msbg_grid *mass, msbg_grid *const *vel, const float *d_pos, const float *d_vel,
                     const float *d_mass, int64_t n, int64_t *n_active) {
    MSBG_CHECK(order == 1 || order == 2, MSBG_EINVAL, "p2g_bspline: order is 1 (trilinear) or 2 (quadratic)");
    MSBG_CHECK(mass && vel && n_active, MSBG_EINVAL, "p2g_bspline: null argument");
    msbg_grid *all[4] = {mass, vel[0], vel[1], vel[2]};
    int rc = check_same_dims(all, 4);
    if (rc) return rc;
    MSBG_CHECK(n >= 0 && n < ((int64_t)1 << 31) && (n == 0 || (d_pos && d_vel)), MSBG_EINVAL,
               "p2g_bspline: bad particle arrays");
    MSBG_CHECK(mass->sx <= 1024 && mass->sy <= 1024 && mass->sz <= 1024, MSBG_EINVAL,
               "p2g_bspline: the 30-bit block and voxel key needs a domain of at most 1024^3");
    // support cells floor(p)-1 .. floor(p)+1 lie in the footprint blocks of r_scan 2
    std::vector<int64_t> act;
    int32_t *d_act = nullptr;
    const uint32_t *d_flags = nullptr;
    rc = active_list(mass, d_pos, n, 2.0f, act, &d_act, &d_flags);
    if (rc) return rc;
    rc = zero_blocks(all, 4, act);
    if (rc) return rc;
    *n_active = (int64_t)act.size();
    if (n == 0 || act.empty()) return MSBG_OK;
    // sort by block and voxel (stable) and the sorted payload
    uint32_t *keys = (uint32_t *)workspace(4, sizeof(uint32_t) * 2 * n, &rc);
    if (rc) return rc;
    uint32_t *perm = keys + n;
    float4 *rec = (float4 *)workspace(22, sizeof(float4) * 2 * n, &rc);
    if (rc) return rc;
    const uint32_t n_keys = (uint32_t)mass->n_blocks << 12;  // at most 2^30
    hipLaunchKernelGGL(block_keys_pack_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream(), d_pos, d_vel, d_mass, n,
                       mass->sx, mass->sy, mass->sz, (int)mass->nx, (int)mass->ny, n_keys, keys, perm, rec);
    MSBG_HIP(hipGetLastError());
    rc = radix_sort_pairs(keys, perm, n, bits_for((int64_t)n_keys - 1));
    if (rc) return rc;
    float4 *pay = (float4 *)workspace(7, sizeof(float4) * 2 * n, &rc);
    if (rc) return rc;
    float4 *pm = pay, *pu = pay + n;
    hipLaunchKernelGGL(gather_records_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream(), rec, perm, n, pm, pu);
    // per-voxel ranges of the sorted particles, indexed like the mass slab; those
    // of blocks that are not active are neither written nor looked at
    const size_t n_range = (size_t)mass->n_slots * 4096;
    uint2 *range = (uint2 *)workspace(8, sizeof(uint2) * n_range + sizeof(uint32_t), &rc);
    if (rc) return rc;
    const unsigned na = (unsigned)act.size();
    // Up to 8 columns of a work-group a CU fit at once, and fewer leave it idle
    // (1 M particles, 350 blocks: 375 us whole, 141 in spans of 4, 164 of 2; 16.8 M,
    // 9,000 blocks: 1,265 whole, 1,334 in spans of 4; all before the rows joined).
    // Two columns a CU are load enough where the blocks are alike and full (calls
    // of 4 M / 8 M particles in a box of 512 blocks: 726 / 1,190 us whole, 692 /
    // 1,480 in spans; of 8 M in 768 uneven ones 8,750 and 4,660).
    const unsigned split = na >= 2048 ? 1 : 4;
    const uint32_t even = split > 1 && na >= 512 && n >= 10000 * (int64_t)na ? (uint32_t)(2 * n / na) : 0;
    uint32_t *widest = even ? (uint32_t *)(range + n_range) : nullptr;
    if (widest) hipLaunchKernelGGL(set_flag_kernel, dim3(1), dim3(1), 0, stream(), (int32_t *)widest, 0);
    hipLaunchKernelGGL(voxel_ranges_kernel, dim3(na), dim3(256), 0, stream(), keys, (uint32_t)n, d_act, mass->view(),
                       range, widest);
    MSBG_HIP(hipGetLastError());
    const auto spread = [&](auto kernel) {
        kernel<<<na * split, 256, 0, stream()>>>(mass->view(), vel[0]->view(), vel[1]->view(), vel[2]->view(), d_act,
                                                 d_flags, range, pm, pu, (int)split, widest, even);
    };
    if (order == 1)
        spread(p2g_bspline_kernel<1>);
    else
        spread(p2g_bspline_kernel<2>);
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}

int msbg_g2p_bspline(int order, msbg_grid *const *vel, const float *d_pos, int64_t n, float *d_out) {
    MSBG_CHECK(order == 1 || order == 2, MSBG_EINVAL, "g2p_bspline: order is 1 (trilinear) or 2 (quadratic)");
    MSBG_CHECK(vel, MSBG_EINVAL, "g2p_bspline: null grids");
    int rc = check_same_dims(vel, 3);
    if (rc) return rc;
    MSBG_CHECK(n >= 0 && (n == 0 || (d_pos && d_out)), MSBG_EINVAL, "g2p_bspline: null argument");
    MSBG_CHECK(n < ((int64_t)1 << 31), MSBG_EINVAL, "g2p_bspline: n must be below 2^31");
    if (n == 0) return MSBG_OK;
    uint32_t *keys = (uint32_t *)workspace(9, sizeof(uint32_t) * 2 * n, &rc);
    if (rc) return rc;
    uint32_t *visit = keys + n;
    rc = morton_order_async(d_pos, n, vel[0]->sx, vel[0]->sy, vel[0]->sz, keys, visit);
    if (rc) return rc;
    // one lane per particle (n < 2^31, so the chunk count fits the grid)
    const dim3 chunks((unsigned)((n + kG2pThreads - 1) / kG2pThreads)), lanes(kG2pThreads);
    if (order == 1)
        hipLaunchKernelGGL(g2p_bspline_kernel<1>, chunks, lanes, 0, stream(), vel[0]->view(), vel[1]->view(),
                           vel[2]->view(), d_pos, n, visit, d_out);
    else
        hipLaunchKernelGGL(g2p_bspline_kernel<2>, chunks, lanes, 0, stream(), vel[0]->view(), vel[1]->view(),
                           vel[2]->view(), d_pos, n, visit, d_out);
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}

}  // extern "C"

// ===========================================================================
// MacGrid::divergence -- fluid/mac.rs:137-171 (each cell at its layout index;
// the reference's running index coincides for whole blocks).
// ===========================================================================
namespace msbg {
namespace {

__device__ __forceinline__ float voxel_at(const GridView &g, int x, int y, int z) {
    const int64_t bid = (x >> 4) + (int64_t)(y >> 4) * g.nx + (int64_t)(z >> 4) * g.nx * g.ny;
    return g.slab[((int64_t)g.b2s[bid] << 12) + ((x & 15) | ((y & 15) << 4) | ((z & 15) << 8))];
}

// The divergence and projection kernels run 16 work-groups of 256 cells per
// listed block, so the block's slot lookups (its own and its neighbours')
// are uniform over a work-group and go out once, together; each lane then
// issues its value loads together.  The values are those voxel_at reads.
__global__ __launch_bounds__(256) void divergence_kernel(GridView u, GridView v, GridView w, GridView d,
                                                         const int32_t *__restrict__ bids, int64_t n) {
    const int64_t k = (int64_t)(blockIdx.x >> 4);
    if (k >= n) return;
    const int vid = (int)((blockIdx.x & 15) << 8) | (int)threadIdx.x;
    const int64_t bid = bids[k];
    const int slot = d.b2s[bid];
    if (slot < 2) return;
    const int64_t nxy = (int64_t)d.nx * d.ny;
    const int bx = (int)(bid % d.nx), by = (int)((bid / d.nx) % d.ny), bz = (int)(bid / nxy);
    const int lx = vid & 15, ly = (vid >> 4) & 15, lz = vid >> 8;
    const int x = bx * 16 + lx, y = by * 16 + ly, z = bz * 16 + lz;
    if (x >= d.sx || y >= d.sy || z >= d.sz) return;
    // this block's slots in the face grids and its -x / -y / -z neighbours' (itself where none exists)
    const int64_t su = (int64_t)u.b2s[bid] << 12, sv = (int64_t)v.b2s[bid] << 12, sw = (int64_t)w.b2s[bid] << 12;
    const int64_t sux = (int64_t)u.b2s[bx > 0 ? bid - 1 : bid] << 12;
    const int64_t svy = (int64_t)v.b2s[by > 0 ? bid - d.nx : bid] << 12;
    const int64_t swz = (int64_t)w.b2s[bz > 0 ? bid - nxy : bid] << 12;
    const float ux1 = u.slab[su + vid], vy1 = v.slab[sv + vid], wz1 = w.slab[sw + vid];
    const float um = u.slab[lx > 0 ? su + vid - 1 : sux + vid + 15];
    const float vm = v.slab[ly > 0 ? sv + vid - 16 : svy + vid + 240];
    const float wm = w.slab[lz > 0 ? sw + vid - 256 : swz + vid + 3840];
    const float ux0 = x == 0 ? 0.0f : um, vy0 = y == 0 ? 0.0f : vm, wz0 = z == 0 ? 0.0f : wm;
    d.slab[((int64_t)slot << 12) + vid] = ((ux1 - ux0) + (vy1 - vy0)) + (wz1 - wz0);
}

// Pressure projection of the face velocities: face a of cell c takes
// u_a(c) - scale (p(c + e_a) - p(c)), the neighbour outside the domain being
// the cell itself; one thread per cell, the three faces it owns.  LO: p is
// the compensated pair p + plo (plo over p's slot layout), and the gradient
// is (p(c + e_a) - p(c)) + (plo(c + e_a) - plo(c)).
template <bool LO>
__global__ __launch_bounds__(256) void subtract_gradient_kernel(GridView u, GridView v, GridView w, GridView p,
                                                                const float *__restrict__ plo,
                                                                const int32_t *__restrict__ bids, int64_t n,
                                                                float scale) {
    const int64_t k = (int64_t)(blockIdx.x >> 4);
    if (k >= n) return;
    const int vid = (int)((blockIdx.x & 15) << 8) | (int)threadIdx.x;
    const int64_t bid = bids[k];
    const int64_t nxy = (int64_t)p.nx * p.ny;
    const int bx = (int)(bid % p.nx), by = (int)((bid / p.nx) % p.ny), bz = (int)(bid / nxy);
    const int lx = vid & 15, ly = (vid >> 4) & 15, lz = vid >> 8;
    const int x = bx * 16 + lx, y = by * 16 + ly, z = bz * 16 + lz;
    if (x >= p.sx || y >= p.sy || z >= p.sz) return;
    // p's slots of this block and of its +x / +y / +z neighbours (itself where none exists)
    const int64_t sp = (int64_t)p.b2s[bid] << 12;
    const int64_t spx = (int64_t)p.b2s[bx + 1 < p.nx ? bid + 1 : bid] << 12;
    const int64_t spy = (int64_t)p.b2s[by + 1 < p.ny ? bid + p.nx : bid] << 12;
    const int64_t spz = (int64_t)p.b2s[bz + 1 < p.nz ? bid + nxy : bid] << 12;
    const int64_t cx = lx < 15 ? sp + vid + 1 : spx + vid - 15, cy = ly < 15 ? sp + vid + 16 : spy + vid - 240,
                  cz = lz < 15 ? sp + vid + 256 : spz + vid - 3840;
    const bool hx = x + 1 < p.sx, hy = y + 1 < p.sy, hz = z + 1 < p.sz;  // the neighbour is in the domain
    const float pc = p.slab[sp + vid];
    const float px = p.slab[hx ? cx : sp + vid], py = p.slab[hy ? cy : sp + vid], pz = p.slab[hz ? cz : sp + vid];
    const float pn[3] = {hx ? px : pc, hy ? py : pc, hz ? pz : pc};
    float lc = 0.0f, ln[3] = {0.0f, 0.0f, 0.0f};
    if constexpr (LO) {  // plo has p's slot layout
        lc = plo[sp + vid];
        const float qx = plo[hx ? cx : sp + vid], qy = plo[hy ? cy : sp + vid], qz = plo[hz ? cz : sp + vid];
        ln[0] = hx ? qx : lc;
        ln[1] = hy ? qy : lc;
        ln[2] = hz ? qz : lc;
    }
    const GridView ch[3] = {u, v, w};
    int slots[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) slots[a] = ch[a].b2s[bid];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (slots[a] < 2) continue;
        float *f = ch[a].slab + ((int64_t)slots[a] << 12) + vid;
        float g = pn[a] - pc;
        if constexpr (LO) g = g + (ln[a] - lc);
        const float t = scale * g;
        *f = *f - t;
    }
}

}  // namespace
}  // namespace msbg

namespace msbg {
namespace {

int subtract_gradient(msbg_grid *const *vel, const msbg_grid *p_layout, const float *d_p, const float *d_plo,
                      const int64_t *active, int64_t n, float scale) {
    MSBG_CHECK(vel && vel[0] && vel[1] && vel[2] && p_layout && d_p, MSBG_EINVAL, "subtract gradient: null argument");
    MSBG_CHECK(n >= 0 && (n == 0 || active), MSBG_EINVAL, "subtract gradient: bad active list");
    for (int a = 0; a < 3; ++a)
        MSBG_CHECK(vel[a]->L == 4 && vel[a]->sx == p_layout->sx && vel[a]->sy == p_layout->sy &&
                       vel[a]->sz == p_layout->sz,
                   MSBG_EINVAL, "subtract gradient: grids must share dimensions and 16^3 blocks");
    MSBG_CHECK(p_layout->L == 4, MSBG_EINVAL, "subtract gradient: 16^3-block pressure layout required");
    if (!n) return MSBG_OK;
    for (int64_t k = 0; k < n; ++k)
        MSBG_CHECK(active[k] >= 0 && active[k] < p_layout->n_blocks, MSBG_EINVAL, "subtract gradient: bid out of range");
    int rc;
    int32_t *d_bids = (int32_t *)workspace(19, sizeof(int32_t) * n, &rc);
    if (rc) return rc;
    std::vector<int32_t> h(active, active + n);
    MSBG_HIP(hipMemcpyAsync(d_bids, h.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, stream()));
    GridView pv = p_layout->view();
    pv.slab = const_cast<float *>(d_p);
    const int grid = (int)((n * 4096 + 255) / 256);
    if (d_plo)
        subtract_gradient_kernel<true><<<grid, 256, 0, stream()>>>(vel[0]->view(), vel[1]->view(), vel[2]->view(), pv,
                                                                    d_plo, d_bids, n, scale);
    else
        subtract_gradient_kernel<false><<<grid, 256, 0, stream()>>>(vel[0]->view(), vel[1]->view(), vel[2]->view(),
                                                                     pv, nullptr, d_bids, n, scale);
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}

}  // namespace
}  // namespace msbg

extern "C" int msbg_mac_subtract_gradient(msbg_grid *const *vel, const msbg_grid *p_layout, const float *d_p,
                                          const int64_t *active, int64_t n, float scale) {
    return msbg::subtract_gradient(vel, p_layout, d_p, nullptr, active, n, scale);
}

extern "C" int msbg_mac_subtract_gradient_pair(msbg_grid *const *vel, const msbg_grid *p_layout, const float *d_p,
                                               const float *d_p_lo, const int64_t *active, int64_t n, float scale) {
    MSBG_CHECK(d_p_lo, MSBG_EINVAL, "subtract gradient: null low part");
    return msbg::subtract_gradient(vel, p_layout, d_p, d_p_lo, active, n, scale);
}

extern "C" int msbg_mac_divergence(msbg_grid *const *vel, msbg_grid *dst, const int64_t *active, int64_t n) {
    MSBG_CHECK(vel && vel[0] && vel[1] && vel[2] && dst, MSBG_EINVAL, "divergence: null grid");
    MSBG_CHECK(n >= 0 && (n == 0 || active), MSBG_EINVAL, "divergence: bad active list");
    for (int a = 0; a < 3; ++a)
        MSBG_CHECK(vel[a]->L == 4 && vel[a]->sx == dst->sx && vel[a]->sy == dst->sy && vel[a]->sz == dst->sz,
                   MSBG_EINVAL, "divergence: grids must share dimensions and 16^3 blocks");
    MSBG_CHECK(dst->L == 4, MSBG_EINVAL, "divergence: 16^3-block destination required");
    if (!n) return MSBG_OK;
    int rc = msbg_grid_ensure_blocks(dst, active, n);  // dst.ensure_blocks_parallel(active), mac.rs:142
    if (rc) return rc;
    int32_t *d_bids = (int32_t *)workspace(15, sizeof(int32_t) * n, &rc);
    if (rc) return rc;
    std::vector<int32_t> h(active, active + n);
    MSBG_HIP(hipMemcpyAsync(d_bids, h.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, stream()));
    divergence_kernel<<<(int)((n * 4096 + 255) / 256), 256, 0, stream()>>>(vel[0]->view(), vel[1]->view(),
                                                                             vel[2]->view(), dst->view(), d_bids, n);
    MSBG_HIP(hipGetLastError());
    MSBG_HIP(hipStreamSynchronize(stream()));
    return MSBG_OK;
}
