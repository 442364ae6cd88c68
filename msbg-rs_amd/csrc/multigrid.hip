// Geometric multigrid for the Poisson band (msbg_poisson): one V-cycle on the
// error equation A e = rt of an FP32 iterative-refinement step.
//
// The reference has no solver (docs/roadmap.md:610-702 "HAVEN'T STARTED";
// restriction by the mean of 8 children is its downsample_channel_avg,
// multires/downsample.rs:13-58).  The hierarchy is block-aligned and
// cell-centred:
//   level 0        the band itself (16^3 cells per listed block, storage T)
//   levels 1..3    8^3, 4^3, 2^3 cells per listed block (FP32, structured:
//                  cell (x, y, z) of listed block k at k B^3 + x + B (y + B z))
//   level 4        one cell per listed block (index = position in the list)
//   levels 5..     the block lattice coarsened by 2 per axis, a cell existing
//                  where any child exists
// Levels 4 and coarser are FP32 cell lists whose neighbour, coefficient,
// child and interpolation tables are built on the host once per band; the
// coarsest (<= kCoarseMax cells) is solved in FP64 by conjugate gradients in
// one work-group.
//
// Level l (cell edge h = 2^l fine cells) holds the cells whose first fine
// cell lies inside the domain.  Operators (unscaled):
//   levels 1..3:  (A x)_c = sum over faces of c_f (x_c - x_f), c_f = 1 towards
//                 a cell of the level, 0 towards the domain boundary (Neumann,
//                 as the band mirrors there), w_l = 2 / (1 + 2^-l) towards a
//                 cell of an unlisted block (x_f = 0).  The band's Dirichlet
//                 values sit at the centres of the first outside fine cells,
//                 (h + 1) / 2 from a level-l cell centre; w_l is h over that
//                 distance.
//   levels 4..:   a quarter of the Galerkin product P^T A P of the next finer
//                 level with piecewise-constant P: the coefficient between
//                 two cells is a quarter of the sum of the fine links between
//                 their children, and each cell keeps a quarter of its
//                 children's Dirichlet coefficients, scaled by w_l / w_{l-1}
//                 (for whole cells this is the operator above on level l; for
//                 partly filled cells the band's Dirichlet coupling is
//                 carried down, so no level loses its boundary values).
// Restriction: b_{l+1} = 0.5 * (sum of the child residuals) (4 x their mean:
// h_{l+1}^2 / h_l^2 of the unscaled operators).  Prolongation: trilinear
// (weights 27, 9, 3, 1 / 64), a partner outside the band reading 0 and one
// beyond the domain the clamped cell.  Smoothing: red-black Gauss-Seidel /
// SOR with the caller's omega, colour 0 then 1 before the coarse correction
// and 1 then 0 after it.
#include <algorithm>
#include <cmath>
#include <vector>

#include "coarse_cg.hpp"
#include "poisson.hpp"

namespace msbg {
namespace mg {

struct Level {
    int l = 0;         // cell edge 2^l fine cells
    int B = 0;         // cells per block edge (structured levels 1..3), 0 for cell lists
    int64_t n = 0;     // cells
    float w = 1.0f;    // Dirichlet face coefficient (structured levels)
    float *x = nullptr, *b = nullptr;
    float *y = nullptr;       // structured levels: x and y take turns
    // cell lists (level >= 4)
    int32_t *nb = nullptr;    // [n][6]: -x, +x, -y, +y, -z, +z linked cell, -1 none
    float *cf = nullptr;      // [n][6]: coefficient of the link
    float *diag = nullptr;    // sum of the link and Dirichlet coefficients
    uint8_t *col = nullptr;   // (x + y + z) & 1 of the cell's lattice coordinates
    int32_t *ch = nullptr;    // [n][8]: children in the next finer cell list (level >= 5), -1 none
    int32_t *pn = nullptr;    // [n][8]: interpolation partners in the next coarser level, -1 none
    // coarsest level: connected components, and which have no Dirichlet coupling
    int16_t *comp = nullptr;  // [n]: component of each cell
    uint8_t *sing = nullptr;  // [n_comp]: 1 when the component's operator is singular
    int n_comp = 0, n_sing = 0;
};

struct Hierarchy {
    std::vector<Level> lv;    // lv[k] is level k + 1
    int32_t *nb27 = nullptr;  // [n_active][27]: listed index of block k's neighbour (dx, dy, dz), -1 / -2
    int32_t *slot27 = nullptr;  // its slot, -1 where not listed (then scratch of the set-up)
};

namespace {

constexpr int kT = 256;

__device__ __forceinline__ int nb27_at(int dx, int dy, int dz) { return (dz + 1) * 9 + (dy + 1) * 3 + (dx + 1); }

// Cell (cx, cy, cz) of a listed block with voxel origin o, at cell edge h:
// inside the domain when its first fine cell is.
__device__ __forceinline__ bool live(const PBlock &B, const Dom &d, int h, int cx, int cy, int cz) {
    return B.ox + cx * h < d.sx && B.oy + cy * h < d.sy && B.oz + cz * h < d.sz;
}

// Trilinear value at fine cell (cx, cy, cz) of listed block k from the
// coarse level of C cells per block edge (coarse cell edge hc = 16 / C).
template <int C>
__device__ __forceinline__ float blk_interp(const float *__restrict__ xc, const int32_t *__restrict__ T,
                                            const PBlock &Bk, const Dom &d, i64 k, int cx, int cy, int cz) {
    constexpr int C3 = C * C * C, hc = 16 / C;
    const int c[3] = {cx, cy, cz}, org[3] = {Bk.ox, Bk.oy, Bk.oz}, dom[3] = {d.sx, d.sy, d.sz};
    // Loads in three batches (the -x / -y / -z neighbour ids, the 8 partners'
    // block ids, the 8 values), each load at a valid address whether or not
    // its value is used; the sum runs over the partners in the same order.
    int32_t tm[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) tm[a] = T[nb27_at(a == 0 ? -1 : 0, a == 1 ? -1 : 0, a == 2 ? -1 : 0)];
    int p[3], dd[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        p[a] = c[a] >> 1;
        dd[a] = (c[a] & 1) ? 1 : -1;
        // a partner beyond the domain is the cell itself (clamp)
        if (dd[a] > 0 && org[a] + (p[a] + 1) * hc >= dom[a]) dd[a] = 0;
        if (dd[a] < 0 && p[a] == 0 && tm[a] == -2) dd[a] = 0;
    }
    int qi[8], tix[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
        int q[3], o[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int on = (kk >> a) & 1;
            q[a] = p[a] + (on ? dd[a] : 0);
            o[a] = 0;
            if (q[a] < 0) {
                q[a] += C;
                o[a] = -1;
            } else if (q[a] >= C) {
                q[a] -= C;
                o[a] = 1;
            }
        }
        qi[kk] = q[0] + C * (q[1] + C * q[2]);
        tix[kk] = nb27_at(o[0], o[1], o[2]);  // 13: the block itself
    }
    int32_t tv[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) tv[kk] = T[tix[kk]];
    i64 nbk[8];
    float xv[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
        nbk[kk] = tix[kk] == 13 ? k : (i64)tv[kk];
        xv[kk] = xc[(nbk[kk] >= 0 ? nbk[kk] : k) * C3 + qi[kk]];
    }
    float v = 0.0f;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
        float wt = 1.0f;
#pragma unroll
        for (int a = 0; a < 3; ++a) wt *= ((kk >> a) & 1) ? 0.25f : 0.75f;
        if (nbk[kk] >= 0) v += wt * xv[kk];
    }
    return v;
}

template <int B>
__global__ __launch_bounds__(kT) void prolong_blk_kernel(i64 n_active, const PBlock *__restrict__ blocks, Dom d,
                                                         const int32_t *__restrict__ nb27,
                                                         const float *__restrict__ xc, float *x) {
    constexpr int B3 = B * B * B;
    const i64 i = (i64)blockIdx.x * kT + threadIdx.x;
    if (i >= n_active * B3) return;
    const i64 k = i / B3;
    const int v = (int)(i % B3), cx = v % B, cy = (v / B) % B, cz = v / (B * B);
    const PBlock Bk = blocks[k];
    if (!live(Bk, d, 16 / B, cx, cy, cz)) return;
    x[i] += blk_interp<B / 2>(xc, nb27 + k * 27, Bk, d, k, cx, cy, cz);
}

__device__ __forceinline__ float list_residual(const float *__restrict__ x, const float *__restrict__ b,
                                               const int32_t *__restrict__ nb, const float *__restrict__ cf,
                                               const float *__restrict__ diag, i64 i) {
    // neighbour indices and coefficients, then the neighbour values, each in
    // one batch (an absent neighbour reads the cell itself, unused)
    int32_t q[6];
    float c[6], xv[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        q[f] = nb[i * 6 + f];
        c[f] = cf[i * 6 + f];
    }
#pragma unroll
    for (int f = 0; f < 6; ++f) xv[f] = x[q[f] >= 0 ? (i64)q[f] : i];
    float s = 0.0f;
#pragma unroll
    for (int f = 0; f < 6; ++f)
        if (q[f] >= 0) s += c[f] * xv[f];
    return b[i] + s - diag[i] * x[i];
}

__global__ __launch_bounds__(kT) void relax_list_kernel(i64 n, const int32_t *__restrict__ nb,
                                                        const float *__restrict__ cf, const float *__restrict__ diag,
                                                        const uint8_t *__restrict__ col, float *x,
                                                        const float *__restrict__ b, float omega, int color) {
    const i64 i = (i64)blockIdx.x * kT + threadIdx.x;
    if (i >= n || col[i] != color || !(diag[i] > 0.0f)) return;
    x[i] += omega * list_residual(x, b, nb, cf, diag, i) / diag[i];
}

__global__ __launch_bounds__(kT) void init_list_kernel(i64 n, const float *__restrict__ diag,
                                                       const uint8_t *__restrict__ col, float *x,
                                                       const float *__restrict__ b, float omega) {
    const i64 i = (i64)blockIdx.x * kT + threadIdx.x;
    if (i >= n) return;
    x[i] = (col[i] == 0 && diag[i] > 0.0f) ? omega * b[i] / diag[i] : 0.0f;
}

__global__ __launch_bounds__(kT) void restrict_list_kernel(i64 nc, const int32_t *__restrict__ ch,
                                                           const int32_t *__restrict__ nb,
                                                           const float *__restrict__ cf,
                                                           const float *__restrict__ diag,
                                                           const float *__restrict__ x, const float *__restrict__ b,
                                                           float *bc) {
    const i64 i = (i64)blockIdx.x * kT + threadIdx.x;
    if (i >= nc) return;
    int32_t c[8];
#pragma unroll
    for (int o = 0; o < 8; ++o) c[o] = ch[i * 8 + o];
    // every child's residual is evaluated (an absent child at cell 0, unused),
    // so no branch separates one child's loads from the next one's
    float r[8];
#pragma unroll
    for (int o = 0; o < 8; ++o) r[o] = list_residual(x, b, nb, cf, diag, c[o] >= 0 ? c[o] : 0);
    float sum = 0.0f;
#pragma unroll
    for (int o = 0; o < 8; ++o)
        if (c[o] >= 0) sum += r[o];
    bc[i] = 0.5f * sum;
}

__global__ __launch_bounds__(kT) void prolong_list_kernel(i64 n, const int32_t *__restrict__ pn,
                                                          const float *__restrict__ xc, float *x) {
    const i64 i = (i64)blockIdx.x * kT + threadIdx.x;
    if (i >= n) return;
    int32_t q[8];
    float xv[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) q[kk] = pn[i * 8 + kk];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) xv[kk] = xc[q[kk] >= 0 ? q[kk] : 0];  // an absent partner reads entry 0, unused
    float v = 0.0f;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
        const float wt = ((kk & 1) ? 0.25f : 0.75f) * ((kk & 2) ? 0.25f : 0.75f) * ((kk & 4) ? 0.25f : 0.75f);
        if (q[kk] >= 0) v += wt * xv[kk];
    }
    x[i] += v;
}

// The coarsest level by itself (below the cell lists of more than kCoarseMax blocks).
__global__ __launch_bounds__(kCoarseMax) void coarse_cg_kernel(CoarseArgs A, const float *__restrict__ b, float *x) {
    __shared__ CoarseShared S;
    const int t = threadIdx.x;
    const double v = coarse_cg(A, A.nb, A.cf, t < A.n ? b[t] : 0.0f, S);
    if (t < A.n) x[t] = (float)v;
}

// The listed index of every block (-1 where not listed), and from it the
// listed index and slot of the 27 blocks around each listed block (-1 where not
// listed, -2 and -1 beyond the lattice).
__global__ void unlisted_kernel(int32_t *index, i64 n) {
    const i64 i = (i64)blockIdx.x * kT + threadIdx.x;
    if (i < n) index[i] = -1;
}
__global__ void listed_kernel(const PBlock *__restrict__ blocks, i64 n, int nx, int ny, int32_t *index) {
    const i64 k = (i64)blockIdx.x * kT + threadIdx.x;
    if (k >= n) return;
    const PBlock B = blocks[k];
    index[(B.ox >> 4) + (i64)nx * ((B.oy >> 4) + (i64)ny * (B.oz >> 4))] = (int32_t)k;
}
__global__ void neighbours_kernel(const PBlock *__restrict__ blocks, i64 n, int nx, int ny, int nz,
                                  const int32_t *__restrict__ index, int32_t *__restrict__ nb27,
                                  int32_t *__restrict__ slot27) {
    const i64 i = (i64)blockIdx.x * kT + threadIdx.x;
    if (i >= n * 27) return;
    const int t = (int)(i % 27);
    const PBlock B = blocks[i / 27];
    const int x = (B.ox >> 4) + t % 3 - 1, y = (B.oy >> 4) + (t / 3) % 3 - 1, z = (B.oz >> 4) + t / 9 - 1;
    int32_t v = -2;
    if (x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz) v = index[x + (i64)nx * (y + (i64)ny * z)];
    nb27[i] = v;
    slot27[i] = v >= 0 ? blocks[v].slot : -1;
}

int grid_of(i64 n) { return (int)((n + kT - 1) / kT); }

// nu red-black sweeps of a cell list (colour 0 then 1; rev: 1 then 0);
// from_zero: x = 0 on entry, the first half sweep written without reading x.
void smooth_list(const Level &L, hipStream_t s, float omega, int nu, bool rev, bool from_zero) {
    for (int it = 0; it < nu; ++it)
        for (int h = 0; h < 2; ++h) {
            if (from_zero && it == 0 && h == 0)
                init_list_kernel<<<grid_of(L.n), kT, 0, s>>>(L.n, L.diag, L.col, L.x, L.b, omega);
            else
                relax_list_kernel<<<grid_of(L.n), kT, 0, s>>>(L.n, L.nb, L.cf, L.diag, L.col, L.x, L.b, omega,
                                                              rev ? 1 - h : h);
        }
}

// ---- host construction -----------------------------------------------------

// A level as a cell list on its lattice (cell edge 2^l fine cells), with its
// operator: links (neighbour + coefficient) and Dirichlet coefficients.
struct HostOp {
    int l = 0;
    int64_t dims[3] = {0, 0, 0};
    std::vector<int32_t> pos;    // [n][3] lattice coordinates
    std::vector<uint8_t> alive;  // the cell lies inside the domain
    std::vector<int32_t> nb;     // [n][6] linked cell, -1 none
    std::vector<float> cf;       // [n][6]
    std::vector<float> dir;      // [n] sum of the Dirichlet coefficients
    std::vector<int32_t> dense;  // lattice -> live cell, -1
    int64_t at(int64_t x, int64_t y, int64_t z) const { return x + dims[0] * (y + dims[1] * z); }
    size_t n() const { return alive.size(); }
};

float dirichlet_coef(int l) { return (float)(2.0 / (1.0 + std::ldexp(1.0, -l))); }

// Lattice position q (level l) inside the domain: its first fine cell is.
bool in_domain(const msbg_poisson *p, int l, const int64_t q[3]) {
    const int64_t s[3] = {p->dom.sx, p->dom.sy, p->dom.sz};
    for (int a = 0; a < 3; ++a)
        if (q[a] < 0 || (q[a] << l) >= s[a]) return false;
    return true;
}

// Level 4, one cell per listed block (cell k is block k): the Galerkin product
// of level 3's operator (2^3 cells per block), whose cells all have the same
// links but for the domain's bound and the unlisted blocks, so it is written
// down per block without level 3's list (37,000 blocks: 0.6 ms, 4 ms through
// the list).
void level4_op(const msbg_poisson *p, HostOp &H) {
    const size_t na = (size_t)p->n_active;
    const int64_t dims[3] = {p->nx, p->ny, p->nz}, s[3] = {p->dom.sx, p->dom.sy, p->dom.sz};
    const int64_t stride[3] = {1, dims[0], dims[0] * dims[1]};
    H.l = 4;
    H.dense.assign((size_t)(dims[0] * dims[1] * dims[2]), -1);
    H.pos.resize(na * 3);
    H.alive.assign(na, 1);
    H.nb.assign(na * 6, -1);
    H.cf.assign(na * 6, 0.0f);
    H.dir.assign(na, 0.0f);
    for (int a = 0; a < 3; ++a) H.dims[a] = dims[a];
    for (size_t k = 0; k < na; ++k) H.dense[(size_t)p->bids[k]] = (int32_t)k;
    const float w = dirichlet_coef(3), part = 0.25f * (dirichlet_coef(4) / dirichlet_coef(3));
    for (size_t k = 0; k < na; ++k) {
        const int64_t bid = p->bids[k];
        const int64_t b[3] = {bid % dims[0], (bid / dims[0]) % dims[1], bid / (dims[0] * dims[1])};
        int children[3];  // along each axis, inside the domain
        for (int a = 0; a < 3; ++a) {
            H.pos[k * 3 + a] = (int32_t)b[a];
            children[a] = (2 * b[a] + 1) << 3 < s[a] ? 2 : 1;
        }
        bool open[6], any = false;  // faces towards an unlisted block
        for (int f = 0; f < 6; ++f) {
            const int a = f >> 1;
            open[f] = false;
            const int64_t q = b[a] + ((f & 1) ? 1 : -1);
            if (q < 0 || q >= dims[a]) continue;  // the domain's bound
            const int32_t j = H.dense[(size_t)(bid + ((f & 1) ? stride[a] : -stride[a]))];
            open[f] = j < 0;
            any = any || open[f];
            if (j < 0) continue;
            H.nb[k * 6 + f] = j;
            H.cf[k * 6 + f] = 0.25f * (float)(children[(a + 1) % 3] * children[(a + 2) % 3]);
        }
        if (!any) continue;
        for (int z = 0; z < children[2]; ++z)
            for (int y = 0; y < children[1]; ++y)
                for (int x = 0; x < children[0]; ++x) {
                    const int c[3] = {x, y, z};
                    float d = 0.0f;
                    for (int f = 0; f < 6; ++f)
                        if (open[f] && c[f >> 1] == (f & 1)) d += w;
                    H.dir[k] += part * d;
                }
    }
}

// The next coarser level of F (Galerkin / 4), its child table and F's
// interpolation table.  Coarse cells are numbered in the order of their first
// child.
void aggregate(const msbg_poisson *p, const HostOp &F, HostOp &Cl, std::vector<int32_t> &ch,
               std::vector<int32_t> &pn) {
    Cl.l = F.l + 1;
    for (int a = 0; a < 3; ++a) Cl.dims[a] = (F.dims[a] + 1) >> 1;
    Cl.dense.assign((size_t)(Cl.dims[0] * Cl.dims[1] * Cl.dims[2]), -1);
    Cl.pos.clear();
    std::vector<int32_t> parent(F.n(), -1);
    for (size_t i = 0; i < F.n(); ++i) {
        if (!F.alive[i]) continue;
        const int64_t q[3] = {F.pos[i * 3] >> 1, F.pos[i * 3 + 1] >> 1, F.pos[i * 3 + 2] >> 1};
        int32_t &c = Cl.dense[Cl.at(q[0], q[1], q[2])];
        if (c < 0) {
            c = (int32_t)(Cl.pos.size() / 3);
            for (int a = 0; a < 3; ++a) Cl.pos.push_back((int32_t)q[a]);
        }
        parent[i] = c;
    }
    const size_t nc = Cl.pos.size() / 3;
    Cl.alive.assign(nc, 1);
    Cl.nb.assign(nc * 6, -1);
    Cl.cf.assign(nc * 6, 0.0f);
    Cl.dir.assign(nc, 0.0f);
    const float wr = dirichlet_coef(Cl.l) / dirichlet_coef(F.l);
    for (size_t i = 0; i < F.n(); ++i) {
        if (!F.alive[i]) continue;
        const int32_t c = parent[i];
        Cl.dir[c] += 0.25f * wr * F.dir[i];
        for (int f = 0; f < 6; ++f) {
            const int32_t j = F.nb[i * 6 + f];
            if (j < 0 || parent[j] == c) continue;
            Cl.nb[(size_t)c * 6 + f] = parent[j];
            Cl.cf[(size_t)c * 6 + f] += 0.25f * F.cf[i * 6 + f];
        }
    }
    ch.assign(nc * 8, -1);
    for (size_t c = 0; c < nc; ++c)
        for (int o = 0; o < 8; ++o) {
            const int64_t x = 2 * (int64_t)Cl.pos[c * 3] + (o & 1), y = 2 * (int64_t)Cl.pos[c * 3 + 1] + ((o >> 1) & 1),
                          z = 2 * (int64_t)Cl.pos[c * 3 + 2] + (o >> 2);
            if (x < F.dims[0] && y < F.dims[1] && z < F.dims[2]) ch[c * 8 + o] = F.dense[F.at(x, y, z)];
        }
    pn.assign(F.n() * 8, -1);
    for (size_t i = 0; i < F.n(); ++i) {
        if (!F.alive[i]) continue;
        for (int kk = 0; kk < 8; ++kk) {
            int64_t q[3];
            for (int a = 0; a < 3; ++a) {
                const int64_t c = F.pos[i * 3 + a], pc = c >> 1, d = (c & 1) ? 1 : -1;
                q[a] = ((kk >> a) & 1) ? pc + d : pc;
            }
            for (int a = 0; a < 3; ++a) {  // a partner beyond the domain is the clamped cell
                int64_t axis[3] = {0, 0, 0};
                axis[a] = q[a];
                if (q[a] >= Cl.dims[a] || !in_domain(p, Cl.l, axis)) q[a] = F.pos[i * 3 + a] >> 1;
            }
            pn[i * 8 + kk] = Cl.dense[Cl.at(q[0], q[1], q[2])];
        }
    }
}

template <class T>
hipError_t upload(T **d, const std::vector<T> &h);

// Connected components of a level's link graph, and which of them have no
// Dirichlet coefficient (singular operator), uploaded into L.
hipError_t components(const HostOp &H, Level &L) {
    const size_t n = H.n();
    std::vector<int16_t> comp(n, -1);
    std::vector<uint8_t> sing;
    std::vector<int32_t> stack;
    for (size_t s0 = 0; s0 < n; ++s0) {
        if (comp[s0] >= 0) continue;
        const int16_t id = (int16_t)sing.size();
        double dir = 0.0;
        stack.assign(1, (int32_t)s0);
        comp[s0] = id;
        while (!stack.empty()) {
            const int32_t i = stack.back();
            stack.pop_back();
            dir += H.dir[i];
            for (int f = 0; f < 6; ++f) {
                const int32_t j = H.nb[(size_t)i * 6 + f];
                if (j >= 0 && comp[j] < 0) {
                    comp[j] = id;
                    stack.push_back(j);
                }
            }
        }
        sing.push_back(dir > 0.0 ? 0 : 1);
    }
    L.n_comp = (int)sing.size();
    L.n_sing = 0;
    for (uint8_t v : sing) L.n_sing += v;
    if (!L.n_sing) return hipSuccess;
    hipError_t e = upload(&L.comp, comp);
    if (e == hipSuccess) e = upload(&L.sing, sing);
    return e;
}

template <class T>
hipError_t upload(T **d, const std::vector<T> &h) {
    if (h.empty()) return hipSuccess;
    hipError_t e = hipMalloc(d, sizeof(T) * h.size());
    if (e == hipSuccess) e = hipMemcpy(*d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice);
    return e;
}

hipError_t upload_list(const HostOp &H, Level &L) {
    const size_t n = H.n();
    std::vector<float> diag(n);
    std::vector<uint8_t> col(n);
    for (size_t i = 0; i < n; ++i) {
        float d = H.dir[i];
        for (int f = 0; f < 6; ++f) d += H.cf[i * 6 + f];
        diag[i] = d;
        col[i] = (uint8_t)((H.pos[i * 3] + H.pos[i * 3 + 1] + H.pos[i * 3 + 2]) & 1);
    }
    hipError_t e = hipMalloc(&L.x, sizeof(float) * std::max<size_t>(1, n));
    if (e == hipSuccess) e = hipMalloc(&L.b, sizeof(float) * std::max<size_t>(1, n));
    if (e == hipSuccess) e = upload(&L.nb, H.nb);
    if (e == hipSuccess) e = upload(&L.cf, H.cf);
    if (e == hipSuccess) e = upload(&L.diag, diag);
    if (e == hipSuccess) e = upload(&L.col, col);
    return e;
}

}  // namespace

void release(msbg_poisson *p) {
    if (!p || !p->mg) return;
    Hierarchy *H = p->mg;
    for (Level &L : H->lv) {
        (void)hipFree(L.x);
        (void)hipFree(L.y);
        (void)hipFree(L.b);
        (void)hipFree(L.nb);
        (void)hipFree(L.cf);
        (void)hipFree(L.diag);
        (void)hipFree(L.col);
        (void)hipFree(L.ch);
        (void)hipFree(L.pn);
        (void)hipFree(L.comp);
        (void)hipFree(L.sing);
    }
    (void)hipFree(H->nb27);
    (void)hipFree(H->slot27);
    delete H;
    p->mg = nullptr;
}

int ensure(msbg_poisson *p) {
    if (p->mg) return MSBG_OK;
    const i64 na = p->n_active;
    Hierarchy *H = new Hierarchy();
    p->mg = H;
    // each listed block's 27 neighbours, by way of every block's listed index
    // (behind the slots: hierarchies share no scratch, so several can be built at once)
    const size_t n27 = (size_t)na * 27;
    hipError_t e = hipMalloc(&H->nb27, sizeof(int32_t) * n27);
    if (e == hipSuccess) e = hipMalloc(&H->slot27, sizeof(int32_t) * (n27 + (size_t)p->n_blocks));
    int32_t *index = H->slot27 + n27;
    if (e == hipSuccess) {
        const int nx = (int)p->nx, ny = (int)p->ny, nz = (int)p->nz;
        unlisted_kernel<<<grid_of(p->n_blocks), kT, 0, stream()>>>(index, p->n_blocks);
        listed_kernel<<<grid_of(na), kT, 0, stream()>>>(p->d_blocks, na, nx, ny, index);
        neighbours_kernel<<<grid_of((i64)n27), kT, 0, stream()>>>(p->d_blocks, na, nx, ny, nz, index, H->nb27,
                                                                 H->slot27);
        e = hipGetLastError();
    }
    for (int l = 1; l <= 3 && e == hipSuccess; ++l) {
        Level L;
        L.l = l;
        L.B = 16 >> l;
        L.n = na * L.B * L.B * L.B;
        L.w = dirichlet_coef(l);
        e = hipMalloc(&L.x, sizeof(float) * L.n);
        if (e == hipSuccess) e = hipMalloc(&L.y, sizeof(float) * L.n);
        if (e == hipSuccess) e = hipMalloc(&L.b, sizeof(float) * L.n);
        H->lv.push_back(L);
    }
    // cell lists: level 4 (one cell per block) and coarser, to <= kCoarseMax cells
    HostOp cur;
    level4_op(p, cur);
    std::vector<int32_t> ch, pn;
    bool first = true;
    while (e == hipSuccess) {
        Level L;
        L.l = cur.l;
        L.n = (i64)cur.n();
        e = upload_list(cur, L);
        if (e == hipSuccess && !first) e = upload(&L.ch, ch);
        const bool last = L.n <= kCoarseMax;
        if (last && e == hipSuccess) e = components(cur, L);
        HostOp next;
        if (!last && e == hipSuccess) {
            aggregate(p, cur, next, ch, pn);
            e = upload(&L.pn, pn);
        }
        H->lv.push_back(L);
        if (last) break;
        cur = std::move(next);
        first = false;
    }
    if (e != hipSuccess) {
        release(p);
        return hip_fail(e, "multigrid hierarchy");
    }
    return MSBG_OK;
}

int n_levels(const msbg_poisson *p) { return p->mg ? (int)p->mg->lv.size() + 1 : 0; }

void vcycle(msbg_poisson *p, hipStream_t s, int storage, float omega, int nu, float extra, float *x, float *lo) {
    const Hierarchy &H = *p->mg;
    const int nl = (int)H.lv.size();
    band_before(p, s, storage, H.nb27, H.slot27, omega, nu, extra, H.lv[0].b);
    const Level &Lc = H.lv[nl - 1];
    const CoarseArgs cg{(int)Lc.n, Lc.n_comp, Lc.n_sing, Lc.nb, Lc.cf, Lc.diag, Lc.comp, Lc.sing};
    // Level 4, a cell per block, is the coarsest (up to kCoarseMax blocks): it and the 2^3 level in one launch, 20 us
    // instead of 37 on 144 blocks, 45 instead of 51 on 704.
    const int tail = Lc.l == 4 ? nl - 2 : nl - 1;
    for (int k = 0; k < tail; ++k) {
        const Level &L = H.lv[k], &C = H.lv[k + 1];
        if (L.B) {
            level_before(p, s, H.nb27, L.B, L.w, omega, nu, L.x, L.y, L.b, C.b);
        } else {
            smooth_list(L, s, omega, nu, false, true);
            restrict_list_kernel<<<grid_of(C.n), kT, 0, s>>>(C.n, C.ch, L.nb, L.cf, L.diag, L.x, L.b, C.b);
        }
    }
    if (tail < nl - 1) {
        const Level &L = H.lv[tail];
        level_tail(p, s, H.nb27, L.w, omega, nu, cg, L.b, L.x);
    } else {
        const int cg_threads = (int)std::min<i64>(kCoarseMax, std::max<i64>(64, (Lc.n + 63) / 64 * 64));
        coarse_cg_kernel<<<1, cg_threads, 0, s>>>(cg, Lc.b, Lc.x);
    }
    const float *xc = H.lv[tail].x;  // the next coarser level's result
    for (int k = tail - 1; k >= 0; --k) {
        const Level &L = H.lv[k];
        if (L.B == 2) {
            // its neighbours' cells interpolate from blocks beyond the 27
            float *x = level_field(L.x, L.y, nu);
            prolong_blk_kernel<2><<<grid_of(L.n), kT, 0, s>>>(p->n_active, p->d_blocks, p->dom, H.nb27, xc, x);
            xc = level_after(p, s, H.nb27, L.B, L.w, omega, nu, L.x, L.y, L.b, nullptr);
        } else if (L.B) {
            xc = level_after(p, s, H.nb27, L.B, L.w, omega, nu, L.x, L.y, L.b, xc);
        } else {
            prolong_list_kernel<<<grid_of(L.n), kT, 0, s>>>(L.n, L.pn, xc, L.x);
            smooth_list(L, s, omega, nu, true, false);
            xc = L.x;
        }
    }
    band_after(p, s, storage, H.nb27, H.slot27, omega, nu, extra, xc, x, lo);
}

}  // namespace mg
}  // namespace msbg
