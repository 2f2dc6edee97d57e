// Adaptive PF-FLIP step on an MSBG (pfflip/mr_sim.py:203-310,
// pfflip/mr_kernels.py, pfflip/particles.py).
//
// Faces follow the operator's convention: cell `a` owns its three low faces
// at face[a * 3 + axis].  Per-particle work (refinement map, P2G, G2P,
// resampling, advection) is one thread per particle; per-cell work is one
// thread per cell, fused so that each pass reads the neighbours only after
// the previous pass has finished everywhere:
//   finish        accumulators -> cell phase, liquid tag, face mass, u*
//   face_prepare  face beta, wall faces, the pre-force copy u*, gravity
//   rhs           integrated divergence (+ the optional density correction)
//   project       pressure gradient on owned faces, and du = u - u*
//   max_div       max |div u| after projection
// P2G adds into 64-bit fixed-point accumulators (one power-of-two scale per
// quantity, chosen on the host from the largest single contribution), so
// the sums do not depend on the order of the atomics.
#include <algorithm>

#include "pf_msbg.hpp"

namespace pf {

int fill_u32(void* dst, int64_t n, uint32_t v, hipStream_t s);
int exclusive_scan(const int* in, int64_t n, int* out, int* tmp, hipStream_t s);
int64_t scan_tmp_ints(int64_t n);

constexpr int kAcc = 8;  // cmass, cwsum, fmass x3, fmom x3 (channel-major)

struct MRConst {
    float r0, rho_l, rho_g, rho_min, alpha_phi, rho_0l, rho_tilde_0, k_div;
    float gx, gy, gz, dt, nu_l, nu_g, alpha_cap;
    float lo[3], hi[3];
    int max_level;
    float mass_scale, mom_scale, w_scale;
    double inv_mass, inv_mom, inv_w;
};

static MRConst mrconst(const pf_mr_params& p) {
    MRConst c;
    c.r0 = p.r0;
    c.rho_l = p.rho_l;
    c.rho_g = p.rho_g;
    c.rho_min = p.rho_min;
    c.alpha_phi = p.alpha_phi;
    c.rho_0l = p.rho_0l;
    c.rho_tilde_0 = p.rho_tilde_0;
    c.k_div = p.k_div;
    c.gx = p.gravity[0];
    c.gy = p.gravity[1];
    c.gz = p.gravity[2];
    c.dt = p.dt;
    c.nu_l = p.nu_l;
    c.nu_g = p.nu_g;
    c.alpha_cap = p.alpha_cap;
    for (int a = 0; a < 3; ++a) {
        c.lo[a] = p.lo[a];
        c.hi[a] = p.hi[a];
    }
    c.max_level = p.max_level;
    c.mass_scale = (float)p.mass_scale;
    c.mom_scale = (float)p.mom_scale;
    c.w_scale = (float)p.w_scale;
    c.inv_mass = 1.0 / p.mass_scale;
    c.inv_mom = 1.0 / p.mom_scale;
    c.inv_w = 1.0 / p.w_scale;
    return c;
}

__device__ inline float cell_size(const MGrid& g, int l) { return g.h0 * (float)(1 << l); }

// eq. (7) with the level-0 constants (mr_kernels.py:141-146)
__device__ inline float phase_field(float rho, float rho_min, float alpha_phi, float rho_0l) {
    if (rho < rho_min) return 0.0f;
    return fminf(sqrtf(fmaxf(rho - rho_min, 0.0f) / (alpha_phi * rho_0l)), 1.0f);
}

// ------------------------------------------------------------------ 1. refinement map
// M[block] = min(l_p, M[block]) over the blocks a particle's box of half
// width cfl_eps touches (particles.py:49-85).  Neighbouring particles touch
// the same few blocks, so a wave combines its lanes first: each lane walks
// its blocks in index order; per round the first pending lane's block is
// taken, the lanes at that block reduce min(l), and one lane issues the
// atomic (the map only decreases, so it is skipped where the map already
// holds the value or less).
__global__ __launch_bounds__(256) void k_mr_refine_map(const float* __restrict__ x, const int* __restrict__ lev,
                                                       int64_t n, int* map, int nbx, int nby, int nbz, float bext,
                                                       float eps) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    int i0 = 0, i1 = -1, j0 = 0, j1 = 0, k0 = 0, k1 = 0, l = 0;
    if (p < n) {
        const float px = x[3 * p], py = x[3 * p + 1], pz = x[3 * p + 2];
        l = lev[p];
        i0 = max((int)floorf((px - eps) / bext), 0);
        i1 = min((int)floorf((px + eps) / bext), nbx - 1);
        j0 = max((int)floorf((py - eps) / bext), 0);
        j1 = min((int)floorf((py + eps) / bext), nby - 1);
        k0 = max((int)floorf((pz - eps) / bext), 0);
        k1 = min((int)floorf((pz + eps) / bext), nbz - 1);
        if (j0 > j1 || k0 > k1) i1 = i0 - 1;  // box outside the raster
    }
    int i = i0, j = j0, k = k0;
    for (;;) {
        const bool pending = i <= i1;
        const unsigned long long act = __ballot(pending);
        if (act == 0ull) break;
        const int key = pending ? (i * nby + j) * nbz + k : -1;
        const int first = __ffsll((long long)act) - 1;
        const int lead = __shfl(key, first, 64);
        const bool mine = pending && key == lead;
        int m = mine ? l : 0x7fffffff;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = min(m, __shfl_xor(m, o, 64));
        if (lane == first && map[lead] > m) atomicMin(map + lead, m);
        if (mine) {
            if (++k > k1) {
                k = k0;
                if (++j > j1) {
                    j = j0;
                    ++i;
                }
            }
        }
    }
}

// max |v| over particles (mr_kernels.py:507-510)
__global__ __launch_bounds__(256) void k_mr_max_speed(const float* __restrict__ v, int64_t n, float* __restrict__ out) {
    float m = 0.0f;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
        const float a = v[3 * p], b = v[3 * p + 1], c = v[3 * p + 2];
        m = fmaxf(m, sqrtf(a * a + b * b + c * c));
    }
    __shared__ float sh[4];
    m = block_max(m, sh);
    if (threadIdx.x == 0) atomic_max_nonneg(out, m);
}

// ------------------------------------------------------------------ 4. P2G
// Mass (eq. 3) and momentum (eq. 4) on the low faces, mass and the bare
// weight sum at the centres, over the cells of every block the support
// sphere touches (mr_kernels.py:48-133).  m_p = rho 8^l_p, r_p = r0 2^l_p
// (particles.py:234-248).  `add(cell, values, mask)` receives the
// fixed-point contributions to one cell (bit ch of mask: channel ch set).
// round(v * scale) to the nearest integer (ties to even), for |v * scale| <
// 2^51: adding 1.5 * 2^52 in double leaves the rounded integer in the low
// mantissa bits (3 instructions; the float-to-int64 conversion takes 11).
// The host keeps every single contribution below 2^48.
__device__ inline long long fixed(float v, float scale) {
    const double d = (double)(v * scale) + 6755399441055744.0;
    return __double_as_longlong(d) - 0x4338000000000000LL;
}

// Distance of a cell centre (axis index i of a block with low corner o) from
// a particle, squared distances and eq. (6) weights.  Which products are fused
// is spelled out: left to the compiler it differs from kernel to kernel, and
// the P2G kernels are to agree bit for bit.
__device__ inline float centre_dist(float o, int i, float h, float x) {
#pragma clang fp contract(off)
    return fmaf(h, (float)i + 0.5f, o) - x;
}
__device__ inline float square(float d) {
#pragma clang fp contract(off)
    return d * d;
}
// q = 0: the centre, 1-3: the low face of axis q - 1; x2, y2: squared
// distances, z: the distance
__device__ inline float eq6_weight(int q, float x2, float y2, float z, float inv_r2) {
#pragma clang fp contract(off)
    const float xy = x2 + y2, d2 = q == 0 || q == 3 ? fmaf(z, z, xy) : xy + z * z;
    const float t = fmaxf(fmaf(-d2, inv_r2, 1.0f), 0.0f);
    return t * t * t;
}

// The blocks an axis of a particle's support touches, clamped to the grid.
__device__ inline int2 touched_blocks(float x, float r, float bext, int nb) {
    return make_int2(max((int)floorf((x - r) / bext), 0), min((int)floorf((x + r) / bext), nb - 1));
}

// PARTS threads share a particle: thread `part` takes every PARTS-th row of
// cells its support touches.
template <int PARTS = 1, class Add>
__device__ inline void splat_particle(const MGrid& g, const float* __restrict__ x, const float* __restrict__ v,
                                      const int* __restrict__ type, const int* __restrict__ lev, int64_t p,
                                      const MRConst& c, Add&& add, int part = 0) {
    const float px = x[3 * p], py = x[3 * p + 1], pz = x[3 * p + 2];
    const float vel[3] = {v[3 * p], v[3 * p + 1], v[3 * p + 2]};
    const int lp = lev[p];
    const float mp = (type[p] == 1 ? c.rho_l : c.rho_g) * (float)(1 << (3 * lp));
    const float rp = c.r0 * (float)(1 << lp);
    const float r2 = rp * rp, inv_r2 = 1.0f / r2;
    const float bext = (float)g.n0 * g.h0;
    int row = 0;
    const int2 bi_ = touched_blocks(px, rp, bext, g.nbx), bj_ = touched_blocks(py, rp, bext, g.nby),
               bk_ = touched_blocks(pz, rp, bext, g.nbz);
    for (int bi = bi_.x; bi <= bi_.y; ++bi)
        for (int bj = bj_.x; bj <= bj_.y; ++bj)
            for (int bk = bk_.x; bk <= bk_.y; ++bk) {
                const int s = g.slot[(bi * g.nby + bj) * g.nbz + bk];
                if (s < 0) continue;
                const int l = g.blev[s];
                const int nn = g.n0 >> l;
                const float h = cell_size(g, l), half = 0.5f * h;
                const float ox = (float)bi * bext, oy = (float)bj * bext, oz = (float)bk * bext;
                // cells whose centre ((i + 1/2) h) or low face (i h) lies
                // within r: i in [(x - r)/h - 1/2, (x + r)/h].  A cell this
                // range misses by rounding has w < 2^-49 of a full weight,
                // which is 0 in fixed point (every scale keeps the largest
                // single contribution below 2^48), so the sums equal those
                // of the reference's wider walk (index range +-1).
                const int i0 = max((int)floorf((px - rp - ox) / h - 0.5f), 0);
                const int i1 = min((int)floorf((px + rp - ox) / h), nn - 1);
                const int j0 = max((int)floorf((py - rp - oy) / h - 0.5f), 0);
                const int j1 = min((int)floorf((py + rp - oy) / h), nn - 1);
                const int k0 = max((int)floorf((pz - rp - oz) / h - 0.5f), 0);
                const int k1 = min((int)floorf((pz + rp - oz) / h), nn - 1);
                const int base = g.coff[s];
                for (int i = i0; i <= i1; ++i) {
                    const float dxc = centre_dist(ox, i, h, px), dxf = dxc - half;
                    const float xc2 = square(dxc), xf2 = square(dxf);
                    if (fminf(xc2, xf2) >= r2) continue;
                    for (int j = j0; j <= j1; ++j) {
                        const float dyc = centre_dist(oy, j, h, py), dyf = dyc - half;
                        const float yc2 = square(dyc), yf2 = square(dyf);
                        if (fminf(xc2, xf2) + fminf(yc2, yf2) >= r2) continue;
                        if (PARTS > 1 && row++ % PARTS != part) continue;
                        for (int k = k0; k <= k1; ++k) {
                            const float dzc = centre_dist(oz, k, h, pz), dzf = dzc - half;
                            const int addr = base + (i * nn + j) * nn + k;
                            const float wt[4] = {
                                eq6_weight(0, xc2, yc2, dzc, inv_r2), eq6_weight(1, xf2, yc2, dzc, inv_r2),
                                eq6_weight(2, xc2, yf2, dzc, inv_r2), eq6_weight(3, xc2, yc2, dzf, inv_r2)};
                            long long val[kAcc];
                            unsigned mask = 0u;
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const float w = wt[q];
                                if (!(w > 0.0f)) continue;
                                const float wm = w * mp;
                                if (q == 0) {
                                    val[0] = fixed(wm, c.mass_scale);
                                    val[1] = fixed(w, c.w_scale);
                                    mask |= 3u;
                                } else {
                                    val[1 + q] = fixed(wm, c.mass_scale);
                                    val[4 + q] = fixed(wm * vel[q - 1], c.mom_scale);
                                    mask |= (1u << (1 + q)) | (1u << (4 + q));
                                }
                            }
                            if (mask) add(addr, val, mask);
                        }
                    }
                }
            }
}

// one thread per particle in index order, every contribution a global atomic
__global__ __launch_bounds__(256) void k_mr_p2g(MGrid g, const float* __restrict__ x, const float* __restrict__ v,
                                                const int* __restrict__ type, const int* __restrict__ lev, int64_t n,
                                                MRConst c, unsigned long long* __restrict__ acc) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int64_t nc = g.ncells;
    splat_particle(g, x, v, type, lev, p, c, [&](int addr, const long long* val, unsigned mask) {
#pragma unroll
        for (int ch = 0; ch < kAcc; ++ch)
            if (mask & (1u << ch)) atomicAdd(acc + ch * nc + addr, (unsigned long long)val[ch]);
    });
}

// Visit order for the cached P2G: particles sorted by the address of the
// cell they sit in (key ncells outside the grid); the order inside a cell
// is whatever the counting atomics give, which the fixed-point sums do not
// see.  The particle arrays themselves keep their order.
__global__ __launch_bounds__(256) void k_mr_cell_key(MGrid g, const float* __restrict__ x, int64_t n,
                                                     int* __restrict__ key, int* __restrict__ rank,
                                                     int* __restrict__ count) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const MCell cl = locate_at(g, x[3 * p], x[3 * p + 1], x[3 * p + 2]);
    const int k = cl.addr >= 0 ? cl.addr : g.ncells;
    key[p] = k;
    rank[p] = atomicAdd(count + k, 1);
}

__global__ __launch_bounds__(256) void k_mr_cell_scatter(const int* __restrict__ key, const int* __restrict__ rank,
                                                         const int* __restrict__ start, int64_t n,
                                                         int* __restrict__ perm, int* __restrict__ nlist) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < 2) nlist[p] = 0;  // what k_mr_p2g_tile leaves to the walk: particles, whole tiles
    if (p >= n) return;
    perm[start[key[p]] + rank[p]] = (int)p;
}

// P2G by tiles of 8^3 cells of a block (a coarser block's whole cell range if
// it has fewer).  A workgroup adds its cells' particles into LDS, at plain
// tile coordinates: the tile plus R cells on every side, 8 fixed-point
// channels, then one global atomic per non-zero entry.  This is the uniform
// splat where it applies: R = 1 takes the particles of the block's own level
// (2 candidates per axis and stagger), R = 2 those one level coarser (5 cells
// per axis), which fill a ring of blocks that a neighbouring finer level has
// refined; in both every block the support touches must have this block's
// level.  What remains (about 0.5 % of the particles of a settled dam break,
// along the 2:1 jumps, and those outside the grid) is left to k_mr_p2g_walk: up
// to kP2GLight of a tile by a list, more by naming the tile (they are marked in
// the order, ~p).  The sums are those of the per-particle walk bit for bit: the
// same cells, weights and fixed-point roundings, and integer adds.
// A hash of cells in LDS for every particle (what k_mr_p2g_walk does) was
// bound by its lookups, one per touched cell.
// 128^3 grid, 9.2M particles (6 % one level coarser than their block):
// 4.95 -> 0.95 ms (0.41 own level, 0.32 one coarser, 0.22 the walk).
constexpr int kP2GLight = 512;
template <int R>
struct P2GTile {
    static constexpr int E = 8 + 2 * R, E3 = E * E * E;
    static constexpr int NT = R == 1 ? 512 : 1024;
};

// The block of a tile and the tile in it.
struct TileRef {
    int level, nn, base;   // cells per axis of the block, first cell address
    int b[3], t0[3], tn;   // block coordinates, first local cell, cells per axis
    float h, bext;
};

// position along axis a in cells of the block.  Without contraction: both tile
// kernels and p2g_class place a particle by it, and a particle that they
// placed in different cells would be splatted twice or not at all.
__device__ inline float block_coord(const TileRef& t, int a, float x) {
#pragma clang fp contract(off)
    return (x - (float)t.b[a] * t.bext) / t.h;
}

// How a particle whose centre lies in the tile is splatted: 0, 1: by the
// R = 1, 2 tile kernel, 2: by the walk.  ok: which of the 27 blocks around
// exist at the tile's level.  (The other float operation that decides,
// touched_blocks, has no product to fuse: r is r0 times a power of two.)
__device__ inline int p2g_class(const MGrid& g, const TileRef& t, unsigned ok, const float (&x)[3], float r0,
                                float rp, int lp, int2 (&blk)[3], int (&ic)[3]) {
    const int nb[3] = {g.nbx, g.nby, g.nbz};
    bool in = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        blk[a] = touched_blocks(x[a], rp, t.bext, nb[a]);
        ic[a] = (int)floorf(block_coord(t, a, x[a]));
        in = in && (unsigned)(ic[a] - t.t0[a]) < (unsigned)t.tn && blk[a].x >= t.b[a] - 1 && blk[a].y <= t.b[a] + 1;
    }
    const int d = lp - t.level;
    if (!in || d < 0 || d > 1 || r0 > g.h0) return 2;  // (candidates sized for radii of at most a cell per level)
    for (int i = blk[0].x; i <= blk[0].y; ++i)
        for (int j = blk[1].x; j <= blk[1].y; ++j)
            for (int k = blk[2].x; k <= blk[2].y; ++k)
                if (!(ok >> (((i - t.b[0] + 1) * 3 + j - t.b[1] + 1) * 3 + k - t.b[2] + 1) & 1u)) return 2;
    return d;
}

// distances of cell i's centre and low face along axis a, from the block that
// holds it; a cell of a block the support does not touch gets a distance that
// makes its weight zero
__device__ inline void cell_dist(const TileRef& t, int a, int i, const int2& blk, float x, float& c, float& f) {
    const int side = i < 0 ? -1 : (i >= t.nn ? 1 : 0), b = t.b[a] + side;
    const float d = centre_dist((float)b * t.bext, i - side * t.nn, t.h, x);
    const bool touched = b >= blk.x && b <= blk.y;
    c = touched ? d : 1e15f;
    f = touched ? d - 0.5f * t.h : 1e15f;
}

// Workgroups: one per 512 cells of the grid.  The multiples of 512 among a
// block's cell addresses are as many as its tiles if it has at least 8 cells
// per axis, so the workgroup of such an address takes one of them.  (One
// workgroup for every tile of a block at level 0 left nearly all idle on coarse
// levels of large blocks: 512 blocks of 64^3 finest cells at level 3, 262144
// workgroups for 512 tiles, P2G 1.28 ms instead of 0.17.)  Then up to
// kP2GWhole that look for the blocks of 4 cells per axis, a tile each.  Smaller
// blocks are left to the walk: at 8 particles per cell, P2G of 13824 of 2^3
// cells took 0.38 ms with tiles and takes 0.33, of 32768 of one cell 0.87 and
// 0.16.
constexpr int kP2GWhole = 1024;

template <int R>
__global__ __launch_bounds__(P2GTile<R>::NT) void k_mr_p2g_tile(MGrid g, int chunks, const float* __restrict__ x,
                                                                const float* __restrict__ v,
                                                                const int* __restrict__ type,
                                                                const int* __restrict__ lev,
                                                                int* __restrict__ perm,
                                                                const int* __restrict__ start, MRConst c,
                                                                int* __restrict__ coarse_tile, int* __restrict__ list,
                                                                int2* __restrict__ heavy, int* __restrict__ nlist,
                                                                unsigned long long* __restrict__ acc) {
    using PT = P2GTile<R>;
    constexpr int E = PT::E, E3 = PT::E3, NT = PT::NT;
    __shared__ unsigned long long L[kAcc * E3];
    __shared__ int s_ok, s_n, s_at;
    __shared__ int s_walk[R == 1 ? kP2GLight : 1];
    const bool whole = (int)blockIdx.x >= chunks;
    // (the R = 2 tiles lie together in the order: dealt out over the XCDs)
    const int wg = whole ? 0 : (R == 1 ? xcd_block(blockIdx.x, chunks) : blockIdx.x);
    if (R == 2 && !whole && coarse_tile[wg] == 0) return;
    const int step = whole ? gridDim.x - chunks : g.nslots;
    for (int slot = whole ? blockIdx.x - chunks : g.cslot[512 * wg]; slot < g.nslots; slot += step) {
        TileRef t;
        t.level = g.blev[slot];
        t.nn = g.n0 >> t.level;
        if (whole ? t.nn != 4 : t.nn < 8) continue;
        t.base = g.coff[slot];
        t.tn = min(t.nn, 8);
        const int ns = t.nn / t.tn;  // tiles per axis
        const int sub = whole ? 0 : wg - (t.base + 511) / 512;
        int* flag = coarse_tile + (whole ? chunks + t.base : wg);
        if (R == 2 && *flag == 0) continue;
        const int blk = g.blk[slot];
        t.b[2] = blk % g.nbz;
        t.b[1] = (blk / g.nbz) % g.nby;
        t.b[0] = blk / (g.nbz * g.nby);
        t.t0[0] = sub / (ns * ns) * t.tn;
        t.t0[1] = sub / ns % ns * t.tn;
        t.t0[2] = sub % ns * t.tn;
        t.h = cell_size(g, t.level);
        t.bext = (float)g.n0 * g.h0;
        const int tid = threadIdx.x;
        // entries of the tile and its ring: all E3 of a tile of 8^3 cells
        const int ext = t.tn + 2 * R, ext3 = ext * ext * ext;
        const auto entry = [&](int e, int& i, int& j, int& k) {
            if (ext == E) {  // (divisions by constants)
                k = e % E;
                j = e / E % E;
                i = e / (E * E);
                return e;
            }
            k = e % ext;
            j = e / ext % ext;
            i = e / (ext * ext);
            return (i * E + j) * E + k;
        };
        if (t.tn == 8) {
            for (int e = tid; e < kAcc * E3; e += NT) L[e] = 0ull;
        } else {
            for (int e = tid; e < ext3; e += NT) {
                int i, j, k;
                const int at = entry(e, i, j, k);
#pragma unroll
                for (int ch = 0; ch < kAcc; ++ch) L[ch * E3 + at] = 0ull;
            }
        }
        if (tid == 0) s_n = 0;
        if (tid < 64) {
            bool same = false;
            if (tid < 27) {
                const int i = t.b[0] + tid / 9 - 1, j = t.b[1] + tid / 3 % 3 - 1, k = t.b[2] + tid % 3 - 1;
                if (i >= 0 && j >= 0 && k >= 0 && i < g.nbx && j < g.nby && k < g.nbz) {
                    const int s = g.slot[(i * g.nby + j) * g.nbz + k];
                    same = s >= 0 && g.blev[s] == t.level;
                }
            }
            const unsigned long long m = __ballot(same);
            if (tid == 0) s_ok = (int)(unsigned)m;
        }
        __syncthreads();
        const unsigned ok = (unsigned)s_ok;
        const int tn3 = t.tn * t.tn * t.tn;
        bool coarse = false;
        // lanes of a wave take different cells; the threads beyond one per cell
        // share its particles
        const int parts = tn3 <= NT ? NT / tn3 : 1;
        const int cell0 = tid % tn3, part = min(tid / tn3, parts);
        if (part < parts) {
            const int li = cell0 / (t.tn * t.tn), lj = cell0 / t.tn % t.tn, lk = cell0 % t.tn;
            const int addr = t.base + ((t.t0[0] + li) * t.nn + t.t0[1] + lj) * t.nn + t.t0[2] + lk;
            const unsigned e0 = start[addr + 1];
            for (unsigned q = start[addr] + part; q < e0; q += parts) {
                const int p = perm[q];
                if (R == 2 && p < 0) continue;  // left to the walk
                const float px[3] = {x[3 * (int64_t)p], x[3 * (int64_t)p + 1], x[3 * (int64_t)p + 2]};
                const float vel[3] = {v[3 * (int64_t)p], v[3 * (int64_t)p + 1], v[3 * (int64_t)p + 2]};
                const int lp = lev[p];
                const float mp = (type[p] == 1 ? c.rho_l : c.rho_g) * (float)(1 << (3 * lp));
                const float rp = c.r0 * (float)(1 << lp);
                const float inv_r2 = 1.0f / (rp * rp);
                int2 tb[3];
                int ic[3];
                const int cls = p2g_class(g, t, ok, px, c.r0, rp, lp, tb, ic);
                if (R == 1) {
                    if (cls == 1) coarse = true;
                    if (cls == 2) {
                        const int at = atomicAdd(&s_n, 1);
                        if (at < kP2GLight) s_walk[at] = p;
                        perm[q] = ~p;
                    }
                }
                if (cls != R - 1) continue;
                auto add = [&](int ch, int at, float value, float scale) {
                    atomicAdd(L + ch * E3 + at, (unsigned long long)fixed(value, scale));
                };
                if constexpr (R == 1) {
                    // per axis: the two centres (first index it) and the two low
                    // faces (first index ic) within the radius: squared distances
                    // along x and y, distances along z
                    float dc[3][2], df[3][2];
                    int lc[3], lf[3];
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        const int it = block_coord(t, a, px[a]) - (float)ic[a] < 0.5f ? ic[a] - 1 : ic[a];
                        float unused;
                        cell_dist(t, a, it, tb[a], px[a], dc[a][0], unused);
                        cell_dist(t, a, it + 1, tb[a], px[a], dc[a][1], unused);
                        cell_dist(t, a, ic[a], tb[a], px[a], unused, df[a][0]);
                        cell_dist(t, a, ic[a] + 1, tb[a], px[a], unused, df[a][1]);
#pragma unroll
                        for (int e = 0; e < 2 && a < 2; ++e) {
                            dc[a][e] = square(dc[a][e]);
                            df[a][e] = square(df[a][e]);
                        }
                        lc[a] = it - t.t0[a] + R;
                        lf[a] = ic[a] - t.t0[a] + R;
                    }
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4) {
                        // q4 = 0: centres, 1-3: low faces of axis q4 - 1
                        const int at0 = ((q4 == 1 ? lf[0] : lc[0]) * E + (q4 == 2 ? lf[1] : lc[1])) * E +
                                        (q4 == 3 ? lf[2] : lc[2]);
#pragma unroll
                        for (int m = 0; m < 8; ++m) {
                            const int i = m >> 2, j = (m >> 1) & 1, k = m & 1;
                            const float w = eq6_weight(q4, q4 == 1 ? df[0][i] : dc[0][i], q4 == 2 ? df[1][j] : dc[1][j],
                                                       q4 == 3 ? df[2][k] : dc[2][k], inv_r2);
                            if (!(w > 0.0f)) continue;
                            const int at = at0 + (i * E + j) * E + k;
                            const float wm = w * mp;
                            if (q4 == 0) {
                                add(0, at, wm, c.mass_scale);
                                add(1, at, w, c.w_scale);
                            } else {
                                add(1 + q4, at, wm, c.mass_scale);
                                add(4 + q4, at, wm * vel[q4 - 1], c.mom_scale);
                            }
                        }
                    }
                } else {
                    float zc[5], zf[5];
#pragma unroll
                    for (int k = 0; k < 5; ++k) cell_dist(t, 2, ic[2] - 2 + k, tb[2], px[2], zc[k], zf[k]);
                    const float r2 = rp * rp;
                    for (int i = 0; i < 5; ++i) {
                        float xc, xf;
                        cell_dist(t, 0, ic[0] - 2 + i, tb[0], px[0], xc, xf);
                        xc = square(xc);
                        xf = square(xf);
                        if (fminf(xc, xf) >= r2) continue;
                        for (int j = 0; j < 5; ++j) {
                            float yc, yf;
                            cell_dist(t, 1, ic[1] - 2 + j, tb[1], px[1], yc, yf);
                            yc = square(yc);
                            yf = square(yf);
                            if (fminf(xc, xf) + fminf(yc, yf) >= r2) continue;
                            const int row = ((ic[0] - 2 + i - t.t0[0] + R) * E + ic[1] - 2 + j - t.t0[1] + R) * E +
                                            ic[2] - 2 - t.t0[2] + R;
#pragma unroll
                            for (int k = 0; k < 5; ++k) {
                                const float wt[4] = {
                                    eq6_weight(0, xc, yc, zc[k], inv_r2), eq6_weight(1, xf, yc, zc[k], inv_r2),
                                    eq6_weight(2, xc, yf, zc[k], inv_r2), eq6_weight(3, xc, yc, zf[k], inv_r2)};
#pragma unroll
                                for (int q4 = 0; q4 < 4; ++q4) {
                                    if (!(wt[q4] > 0.0f)) continue;
                                    const float wm = wt[q4] * mp;
                                    if (q4 == 0) {
                                        add(0, row + k, wm, c.mass_scale);
                                        add(1, row + k, wt[0], c.w_scale);
                                    } else {
                                        add(1 + q4, row + k, wm, c.mass_scale);
                                        add(4 + q4, row + k, wm * vel[q4 - 1], c.mom_scale);
                                    }
                                }
                            }
                        }
                    }
                }
            }
        }
        if (R == 1) {
            const bool any = __syncthreads_or(coarse);
            if (tid == 0) *flag = any ? 1 : 0;
            const int walk = s_n;
            if (walk > kP2GLight) {
                if (tid == 0) heavy[atomicAdd(nlist + 1, 1)] = make_int2(slot, sub);
            } else if (walk > 0) {
                if (tid == 0) s_at = atomicAdd(nlist, walk);
                __syncthreads();
                for (int e = tid; e < walk; e += NT) list[s_at + e] = s_walk[e];
            }
        } else {
            __syncthreads();
        }
        // flush: an entry beyond the block belongs to the neighbouring block
        const int64_t nc = g.ncells;
        for (int e0 = tid; e0 < ext3; e0 += NT) {
            int ei, ej, ek;
            const int e = entry(e0, ei, ej, ek);
            bool any = false;
#pragma unroll
            for (int ch = 0; ch < kAcc; ++ch) any = any || L[ch * E3 + e] != 0ull;
            if (!any) continue;
            const int i = t.t0[0] + ei - R, j = t.t0[1] + ej - R, k = t.t0[2] + ek - R;
            const int di = i < 0 ? -1 : (i >= t.nn ? 1 : 0), dj = j < 0 ? -1 : (j >= t.nn ? 1 : 0),
                      dk = k < 0 ? -1 : (k >= t.nn ? 1 : 0);
            int base = t.base;
            if (di | dj | dk)  // (non-zero entries only lie in blocks of this level)
                base = g.coff[g.slot[((t.b[0] + di) * g.nby + t.b[1] + dj) * g.nbz + t.b[2] + dk]];
            const int64_t a = base + ((i - di * t.nn) * t.nn + j - dj * t.nn) * t.nn + k - dk * t.nn;
#pragma unroll
            for (int ch = 0; ch < kAcc; ++ch) {
                const unsigned long long val = L[ch * E3 + e];
                if (val != 0ull) atomicAdd(acc + ch * nc + a, val);
            }
        }
        __syncthreads();
    }
}

// The particles left to the walk: a workgroup keeps a hash of kP2GSlots
// cells in LDS (tag + the 8 fixed-point channels), adds there with LDS
// atomics, and flushes every cached cell with one global atomic per non-zero
// channel.  A contribution whose slot holds another cell goes to global
// memory directly.  Integer sums, so the result equals the uncached kernel's
// bit for bit.
constexpr int kP2GSlots = 512;
constexpr unsigned kP2GWalkBlocks = 1024;
static_assert(kP2GSlots == 1 << 9, "the slot hash keeps 9 bits");

// 256 / PARTS particles, or none (p < 0), one per PARTS threads
template <int PARTS>
__device__ inline void p2g_walk(const MGrid& g, const float* __restrict__ x, const float* __restrict__ v,
                                const int* __restrict__ type, const int* __restrict__ lev, int64_t p, const MRConst& c,
                                int* tag, unsigned long long* lacc, unsigned long long* __restrict__ acc) {
    const int64_t nc = g.ncells;
    for (int s = threadIdx.x; s < kP2GSlots; s += 256) tag[s] = -1;
    for (int s = threadIdx.x; s < kP2GSlots * kAcc; s += 256) lacc[s] = 0ull;
    __syncthreads();
    if (p >= 0)
        splat_particle<PARTS>(g, x, v, type, lev, p, c, [&](int addr, const long long* val, unsigned mask) {
            const int s = (int)(((unsigned)addr * 2654435761u) >> 23);  // 9-bit multiplicative hash
            int t = tag[s];
            if (t != addr && t == -1) {
                t = atomicCAS(tag + s, -1, addr);
                if (t == -1) t = addr;
            }
            if (t == addr) {
#pragma unroll
                for (int ch = 0; ch < kAcc; ++ch)
                    if (mask & (1u << ch)) atomicAdd(lacc + s * kAcc + ch, (unsigned long long)val[ch]);
            } else {
#pragma unroll
                for (int ch = 0; ch < kAcc; ++ch)
                    if (mask & (1u << ch)) atomicAdd(acc + ch * nc + addr, (unsigned long long)val[ch]);
            }
        }, (int)threadIdx.x % PARTS);
    __syncthreads();
    for (int s = threadIdx.x; s < kP2GSlots; s += 256) {
        const int a = tag[s];
        if (a < 0) continue;
#pragma unroll
        for (int ch = 0; ch < kAcc; ++ch) {
            const unsigned long long val = lacc[s * kAcc + ch];
            if (val != 0ull) atomicAdd(acc + ch * nc + a, val);
        }
    }
    __syncthreads();
}

// The listed particles and those outside the grid, kP2GParts threads each:
// one particle's walk is a serial chain over up to a few hundred cells, and 46k
// particles (0.5 % of a 9.2M dam break) at one per thread were 180 workgroups
// waiting for it: 1, 2, 4, 8 threads: 350, 300, 221, 253 us; in a flow that
// lists far more of them 795, 725, 705, 730, and 16 or 32 threads 855 and 1030.
// Then the blocks of fewer than 4 cells per axis, and the tiles that leave many,
// an eighth (8 rows of 8 cells) per workgroup, in the cells' order, in which the
// particles of a workgroup share cells: with jumps between all blocks of 16^3
// cells, alternately of levels 0 and 1, P2G of 16.8M particles took 8.8 ms from
// the list, 4.1 so (3.1 where all are walked: those that a tile has taken leave
// gaps).  nlist NULL: every particle, in that order.
constexpr int kP2GParts = 4;

__global__ __launch_bounds__(256) void k_mr_p2g_walk(MGrid g, const float* __restrict__ x, const float* __restrict__ v,
                                                     const int* __restrict__ type, const int* __restrict__ lev,
                                                     const int* __restrict__ list, const int2* __restrict__ heavy,
                                                     const int* __restrict__ nlist, const int* __restrict__ perm,
                                                     const int* __restrict__ start, int np, MRConst c,
                                                     unsigned long long* __restrict__ acc) {
    __shared__ int tag[kP2GSlots];
    __shared__ unsigned long long lacc[kP2GSlots * kAcc];
    if (!nlist) {
        for (int64_t p0 = blockIdx.x * 256; p0 < np; p0 += gridDim.x * 256) {
            const int64_t q = p0 + threadIdx.x;
            p2g_walk<1>(g, x, v, type, lev, q < np ? perm[q] : -1, c, tag, lacc, acc);
        }
        return;
    }
    const int nl = nlist[0], out0 = start[g.ncells], n = nl + (np - out0);
    constexpr int B = 256 / kP2GParts;
    for (int64_t p0 = blockIdx.x * B; p0 < n; p0 += gridDim.x * B) {
        const int64_t q = p0 + (int)threadIdx.x / kP2GParts;
        const int p = q < n ? (q < nl ? list[q] : perm[out0 + q - nl]) : -1;
        p2g_walk<kP2GParts>(g, x, v, type, lev, p, c, tag, lacc, acc);
    }
    // the blocks of fewer than 4 cells per axis, 32 neighbours in the order at a
    // time and of their particles every fourth 256
    const int groups = (g.nslots + 31) / 32;
    __shared__ int first[32], before[33], some[512], nsome;
    const int lane = threadIdx.x & 63;
    for (int w = blockIdx.x; w < 4 * groups; w += gridDim.x) {
        const int slot = 32 * (w % groups) + (int)threadIdx.x;
        if (threadIdx.x < 64) {
            int f = 0, len = 0;
            if (threadIdx.x < 32 && slot < g.nslots) {
                const int nn = g.n0 >> g.blev[slot], a = g.coff[slot];
                if (nn < 4) {
                    f = start[a];
                    len = start[a + nn * nn * nn] - f;
                }
            }
            int sum = len;
#pragma unroll
            for (int o = 1; o < 32; o <<= 1) {
                const int t = __shfl_up(sum, o, 64);
                sum += lane >= o ? t : 0;
            }
            if (threadIdx.x < 32) {
                first[lane] = f;
                before[lane + 1] = sum;
            }
            if (threadIdx.x == 0) before[0] = 0;
        }
        __syncthreads();
        const int m = before[32];
        for (int q0 = 256 * (w / groups); q0 < m; q0 += 1024) {
            const int q = q0 + (int)threadIdx.x;
            int r = 0;
#pragma unroll
            for (int o = 16; o > 0; o >>= 1) r += q >= before[r + o] ? o : 0;
            p2g_walk<1>(g, x, v, type, lev, q < m ? perm[first[r] + q - before[r]] : -1, c, tag, lacc, acc);
        }
        __syncthreads();
    }
    const int nw = 8 * nlist[1];
    for (int w = blockIdx.x; w < nw; w += gridDim.x) {
        const int2 h = heavy[w >> 3];
        const int nn = g.n0 >> g.blev[h.x], tn = min(nn, 8), ns = nn / tn, li = w & 7;
        if (li >= tn) continue;
        if ((int)threadIdx.x < tn) {
            const int i = h.y / (ns * ns) * tn + li, j = h.y / ns % ns * tn + (int)threadIdx.x, k = h.y % ns * tn;
            const int a = g.coff[h.x] + (i * nn + j) * nn + k;
            first[threadIdx.x] = start[a];
            before[threadIdx.x + 1] = start[a + tn] - start[a];
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            before[0] = 0;
            for (int r = 0; r < tn; ++r) before[r + 1] += before[r];
        }
        __syncthreads();
        const int m = before[tn];
        if (threadIdx.x == 0) nsome = 0;
        __syncthreads();
        for (int q0 = 0; q0 < m; q0 += 256) {
            // the marked ones, walked 256 at a time
            const int q = q0 + (int)threadIdx.x;
            int r = 0;
            while (r + 1 < tn && q >= before[r + 1]) ++r;
            const int e = q < m ? perm[first[r] + q - before[r]] : 0;
            if (e < 0) some[atomicAdd(&nsome, 1)] = ~e;
            __syncthreads();
            const int have = nsome;
            __syncthreads();
            if (have < 256 && q0 + 256 < m) continue;
            p2g_walk<1>(g, x, v, type, lev, (int)threadIdx.x < have ? some[threadIdx.x] : -1, c, tag, lacc, acc);
            const int rest = max(have - 256, 0), later = (int)threadIdx.x < rest ? some[256 + threadIdx.x] : 0;
            if (q0 + 256 >= m && rest > 0)
                p2g_walk<1>(g, x, v, type, lev, (int)threadIdx.x < rest ? later : -1, c, tag, lacc, acc);
            some[threadIdx.x] = later;
            if (threadIdx.x == 0) nsome = rest;
            __syncthreads();
        }
    }
}

// ------------------------------------------------------------------ 5. cell finish
// cwsum; phase field and liquid tag with the per-level normalisation
// (mr_kernels.py:149-165); face mass and u* = P / m (mr_kernels.py:136-146).
// The accumulators are cleared for the next P2G.
__global__ __launch_bounds__(256) void k_mr_finish(MGrid g, MRConst c, int64_t* __restrict__ acc,
                                                   float* __restrict__ cwsum, float* __restrict__ phi,
                                                   int* __restrict__ is_liquid, float* __restrict__ fmass,
                                                   float* __restrict__ fvel) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= g.ncells) return;
    const int64_t nc = g.ncells;
    const int l = g.blev[g.cslot[a]];
    const float norm = (float)(1 << (3 * l));
    const float cm = (float)((double)acc[a] * c.inv_mass);
    cwsum[a] = (float)((double)acc[nc + a] * c.inv_w);
    const float f = phase_field(cm / norm, c.rho_min, c.alpha_phi, c.rho_0l);
    phi[a] = f;
    is_liquid[a] = f >= 0.5f ? 1 : 0;
    const float eps = 1e-12f * c.rho_0l;
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        const double m = (double)acc[(2 + ax) * nc + a] * c.inv_mass;
        const double mom = (double)acc[(5 + ax) * nc + a] * c.inv_mom;
        fmass[a * 3 + ax] = (float)m;
        fvel[a * 3 + ax] = (float)m > eps ? (float)(mom / m) : 0.0f;
    }
#pragma unroll
    for (int q = 0; q < kAcc; ++q) acc[q * nc + a] = 0;
}

// ------------------------------------------------------------------ face coefficients, walls, forces
// beta = 1 / rho(phi_face) on owned faces, phi = 1 / 0 between two liquid /
// two air cells, beta = 0 on domain walls (mr_kernels.py:168-206); zero the
// wall velocities (mr_kernels.py:209-214); u* = u (mr_sim.py:238); gravity on
// open faces (mr_kernels.py:220-227)
__global__ __launch_bounds__(256) void k_mr_face_prepare(MGrid g, MRConst c, const int* __restrict__ is_liquid,
                                                         const float* __restrict__ fmass, float* __restrict__ fbeta,
                                                         float* __restrict__ fvel, float* __restrict__ fvel_star) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= g.ncells) return;
    BlockRef br;
    const int4 o = origin_ref(g, a, br);
    const float norm = (float)(1 << (3 * o.w));
    const int hi = is_liquid[a];
    const float gv[3] = {c.gx, c.gy, c.gz};
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        const MCell nb = locate_near(g, br, o.x - comp(ax, 0), o.y - comp(ax, 1), o.z - comp(ax, 2));
        float beta = 0.0f;
        if (nb.addr >= 0) {
            const int lo = is_liquid[nb.addr];
            float f;
            if (lo == 1 && hi == 1)
                f = 1.0f;
            else if (lo == 0 && hi == 0)
                f = 0.0f;
            else
                f = phase_field(fmass[a * 3 + ax] / norm, c.rho_min, c.alpha_phi, c.rho_0l);
            beta = 1.0f / ((1.0f - f) * c.rho_g + f * c.rho_l);
        }
        fbeta[a * 3 + ax] = beta;
        float u = beta == 0.0f ? 0.0f : fvel[a * 3 + ax];
        fvel_star[a * 3 + ax] = u;
        if (beta != 0.0f) u += gv[ax] * c.dt;
        fvel[a * 3 + ax] = u;
    }
}

// flux-weighted velocity through the high face: a finer neighbour backs the
// face with a 2x2 patch whose mean is taken (mr_kernels.py:230-283)
__device__ inline float face_velocity_high(const MGrid& g, const BlockRef& br, const float* __restrict__ fvel, int4 o,
                                          int ax) {
    const int ext = 1 << o.w;
    const int fx = o.x + comp(ax, 0) * ext, fy = o.y + comp(ax, 1) * ext, fz = o.z + comp(ax, 2) * ext;
    const MCell nb = locate_near(g, br, fx, fy, fz);
    if (nb.addr < 0) return 0.0f;
    if (nb.level >= o.w) return fvel[nb.addr * 3 + ax];
    const int sub = 1 << nb.level;
    const int a1 = (ax + 1) % 3, a2 = (ax + 2) % 3;
    float acc = 0.0f, cnt = 0.0f;
    for (int u = 0; u < 2; ++u)
        for (int v = 0; v < 2; ++v) {
            const int du = u * sub, dv = v * sub;
            const MCell nc = locate_near(g, br, fx + comp(a1, 0) * du + comp(a2, 0) * dv,
                                         fy + comp(a1, 1) * du + comp(a2, 1) * dv, fz + comp(a1, 2) * du + comp(a2, 2) * dv);
            if (nc.addr >= 0) {
                acc += fvel[nc.addr * 3 + ax];
                cnt += 1.0f;
            }
        }
    return cnt > 0.0f ? acc / cnt : 0.0f;
}

// b = -(1/dt) sum_faces u* . A_f, minus the optional density correction
// (mr_kernels.py:286-313)
__global__ __launch_bounds__(256) void k_mr_rhs(MGrid g, MRConst c, const float* __restrict__ fvel,
                                                const float* __restrict__ cwsum, float* __restrict__ rhs) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= g.ncells) return;
    BlockRef br;
    const int4 o = origin_ref(g, a, br);
    const float h = cell_size(g, o.w), area = h * h;
    float flux = 0.0f;
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) flux += (face_velocity_high(g, br, fvel, o, ax) - fvel[a * 3 + ax]) * area;
    float r = -flux / c.dt;
    if (c.k_div > 0.0f) {
        const float excess = (cwsum[a] / (float)(1 << (3 * o.w)) - c.rho_tilde_0) / c.rho_tilde_0;
        r -= c.k_div * fmaxf(excess, 0.0f) * h * h * h / c.dt;
    }
    rhs[a] = r;
}

// u = u* - dt beta (p_a - p_low) / dist on owned faces (mr_kernels.py:316-343),
// then du = u - u* (mr_kernels.py:415-418)
__global__ __launch_bounds__(256) void k_mr_project(MGrid g, MRConst c, const float* __restrict__ pres,
                                                    const float* __restrict__ fbeta, float* __restrict__ fvel,
                                                    const float* __restrict__ fvel_star, float* __restrict__ fdvel) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= g.ncells) return;
    BlockRef br;
    const int4 o = origin_ref(g, a, br);
    const float hA = cell_size(g, o.w);
    const float pa = pres[a];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        float u = fvel[a * 3 + ax];
        const float beta = fbeta[a * 3 + ax];
        if (beta != 0.0f) {
            const MCell nb = locate_near(g, br, o.x - comp(ax, 0), o.y - comp(ax, 1), o.z - comp(ax, 2));
            if (nb.addr >= 0) {
                const float dist = 0.5f * (hA + cell_size(g, nb.level));
                u -= c.dt * beta * (pa - pres[nb.addr]) / dist;
                fvel[a * 3 + ax] = u;
            }
        }
        fdvel[a * 3 + ax] = u - fvel_star[a * 3 + ax];
    }
}

// max |div u| (mr_kernels.py:346-353)
__global__ __launch_bounds__(256) void k_mr_max_div(MGrid g, const float* __restrict__ fvel, float* __restrict__ out) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    float m = 0.0f;
    if (a < g.ncells) {
        BlockRef br;
        const int4 o = origin_ref(g, a, br);
        float d = 0.0f;
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) d += face_velocity_high(g, br, fvel, o, ax) - fvel[a * 3 + ax];
        m = fabsf(d / cell_size(g, o.w));
    }
    __shared__ float sh[4];
    m = block_max(m, sh);
    if (threadIdx.x == 0) atomic_max_nonneg(out, m);
}

// ------------------------------------------------------------------ G2P and advection
// trilinear face sample at the resolution of the cell containing x; taps
// resolve through locate, so a coarser or finer neighbour contributes its own
// face (mr_kernels.py:359-405)
// the cell containing a sample point and its block, resolved once for the
// three staggered components
struct SamplePoint {
    MCell c;
    BlockRef br;
};

__device__ inline SamplePoint sample_point(const MGrid& g, float x, float y, float z) {
    SamplePoint s;
    s.c = locate_at(g, x, y, z);
    if (s.c.addr >= 0) s.br = block_ref(g, s.c.slot);
    return s;
}

// rounded twice, never fused into the sum of the weights, so that both ways to
// sample agree bit for bit
__device__ inline float tap_weight(float wi, float wj, float wk) {
#pragma clang fp contract(off)
    const float w = wi * wj;
    return w * wk;
}

__device__ inline float sample_face(const MGrid& g, const float* __restrict__ f, float x, float y, float z, int ax,
                                    const SamplePoint& sp) {
    const MCell& c = sp.c;
    if (c.addr < 0) return 0.0f;
    const BlockRef& br = sp.br;
    const int ext = 1 << c.level;
    const float h = cell_size(g, c.level);
    const float sx = x / h - (ax == 0 ? 0.0f : 0.5f);
    const float sy = y / h - (ax == 1 ? 0.0f : 0.5f);
    const float sz = z / h - (ax == 2 ? 0.0f : 0.5f);
    const float fi = floorf(sx), fj = floorf(sy), fk = floorf(sz);
    const int i0 = (int)fi, j0 = (int)fj, k0 = (int)fk;
    const float tx = sx - fi, ty = sy - fj, tz = sz - fk;
    float acc = 0.0f, wsum = 0.0f;
    for (int di = 0; di < 2; ++di) {
        const float wi = di == 0 ? 1.0f - tx : tx;
        for (int dj = 0; dj < 2; ++dj) {
            const float wj = dj == 0 ? 1.0f - ty : ty;
            for (int dk = 0; dk < 2; ++dk) {
                const float wk = dk == 0 ? 1.0f - tz : tz;
                const float w = tap_weight(wi, wj, wk);
                if (w <= 0.0f) continue;
                const MCell nc = locate_near(g, br, (i0 + di) * ext, (j0 + dj) * ext, (k0 + dk) * ext);
                if (nc.addr < 0) continue;
                acc = fmaf(w, f[nc.addr * 3 + ax], acc);
                wsum += w;
            }
        }
    }
    return wsum > 0.0f ? acc / wsum : 0.0f;
}

// Without a table (see below), G2P samples two fields at one point through the
// same taps: the taps of the three staggered components (weight and cell
// address; -1: not summed, a zero weight or no cell) are resolved once and the
// 48 values loaded together: 9.2M particles 672 us, 1210 with a walk per
// component and field.  The advection's three samples at three points are
// walked per component: with the taps batched per point it took 1.38 ms instead
// of 1.20 (more registers, the out-of-block lookups still serial), and with
// one body for the three stages 1.65 instead of 1.04.
struct WalkTaps {
    float w[3][8];
    int addr[3][8];
};

__device__ inline void walk_taps(const MGrid& g, float x, float y, float z, const SamplePoint& sp, WalkTaps& t) {
    const MCell& c = sp.c;
    const BlockRef& br = sp.br;
    const int ext = 1 << c.level;
    const float h = cell_size(g, c.level);
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        const float sx = x / h - (ax == 0 ? 0.0f : 0.5f);
        const float sy = y / h - (ax == 1 ? 0.0f : 0.5f);
        const float sz = z / h - (ax == 2 ? 0.0f : 0.5f);
        const float fi = floorf(sx), fj = floorf(sy), fk = floorf(sz);
        const int i0 = (int)fi, j0 = (int)fj, k0 = (int)fk;
        const float tx = sx - fi, ty = sy - fj, tz = sz - fk;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int di = q >> 2, dj = (q >> 1) & 1, dk = q & 1;
            const float w = tap_weight(di ? tx : 1.0f - tx, dj ? ty : 1.0f - ty, dk ? tz : 1.0f - tz);
            t.w[ax][q] = w;
            t.addr[ax][q] =
                w > 0.0f ? locate_near(g, br, (i0 + di) * ext, (j0 + dj) * ext, (k0 + dk) * ext).addr : -1;
        }
    }
}

// The tap values of field f (address -1 reads entry 0, masked in the sum):
// all 24 loads are issued before the first is used.
__device__ inline void walk_values(const float* __restrict__ f, const WalkTaps& t, float (&v)[3][8]) {
#pragma unroll
    for (int ax = 0; ax < 3; ++ax)
#pragma unroll
        for (int q = 0; q < 8; ++q) v[ax][q] = f[max(t.addr[ax][q], 0) * 3 + ax];
}

// sample_face's sums for the three components
__device__ inline void walk_sum(const WalkTaps& t, const float (&v)[3][8], float (&out)[3]) {
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        float acc = 0.0f, wsum = 0.0f;
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (t.addr[ax][q] >= 0) {
                acc = fmaf(t.w[ax][q], v[ax][q], acc);
                wsum += t.w[ax][q];
            }
        out[ax] = wsum > 0.0f ? acc / wsum : 0.0f;
    }
}

// Where a sample's 24 taps are: per axis the two lattice points of a face
// component along its own axis ([0]) and of the others ([1]), each with its
// weight, its part of the address inside a block and which of three blocks
// holds it.  A block's taps reach at most the blocks around it, so with
// nbr[27 slot + ...] (first cell of the neighbours of the block's own level,
// -1 for any other) a tap's address is one load and a few adds instead of a
// walk over slots, levels and offsets, some 60 instructions times 72 taps.
struct SampleTaps {
    float w[3][2][2];
    int at[3][2][2];   // local cell times the axis' stride
    int blk[3][2][2];  // 0, 1, 2 times 9, 3, 1
    int cell[3];       // the sample's cell, in the grid at its level
    bool below[3];     // ... and the one below it (else above) for the others
    int slot, base, level;
    bool cross;        // some tap is in another block
};

// false: no cell here.  A tap outside the grid, or of weight 0 (it may hold no
// number), takes the other one's place with weight 0: it adds nothing to either
// sum.  The sample's own cell has some weight in each component.
__device__ inline bool sample_taps(const MGrid& g, const float (&x)[3], SampleTaps& t) {
    const int nb[3] = {g.nbx, g.nby, g.nbz};
    float u[3];
    int f[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        u[a] = x[a] / g.h0;
        f[a] = (int)floorf(u[a]);
        if (f[a] < 0 || (f[a] >> g.sh0) >= nb[a]) return false;
    }
    t.slot = g.slot[((f[0] >> g.sh0) * nb[1] + (f[1] >> g.sh0)) * nb[2] + (f[2] >> g.sh0)];
    if (t.slot < 0) return false;
    t.level = g.blev[t.slot];
    t.base = g.coff[t.slot];
    const int ln = g.sh0 - t.level, n = 1 << ln;
    const float inv = __int_as_float((127 - t.level) << 23);  // 2^-level: x / h = (x / h0) 2^-level exactly
    t.cross = false;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int shift = (2 - a) * ln, bs = a == 0 ? 9 : (a == 1 ? 3 : 1);
        const float sf = u[a] * inv, sc = sf - 0.5f;
        const int c = f[a] >> t.level, lc = c & (n - 1);  // the cell, in the grid and in the block
        const bool lo = c > 0, hi = c + 1 < nb[a] << ln;  // its neighbours exist
        const int at0 = lc << shift, atm = ((lc - 1) & (n - 1)) << shift, atp = ((lc + 1) & (n - 1)) << shift;
        const int bm = lc == 0 ? 0 : bs, bp = lc == n - 1 ? 2 * bs : bs;
        const float tf = sf - floorf(sf), fc = floorf(sc), tc = sc - fc;
        const bool next = hi && tf != 0.0f;
        t.w[a][0][0] = 1.0f - tf;
        t.w[a][0][1] = next ? tf : 0.0f;
        t.at[a][0][0] = at0;
        t.blk[a][0][0] = bs;
        t.at[a][0][1] = next ? atp : at0;
        t.blk[a][0][1] = next ? bp : bs;
        const bool below = (int)fc < c;  // the cell and the one below it, or above (tc >= 1/2 below)
        const bool other = below ? lo : hi && tc != 0.0f;
        t.cell[a] = c;
        t.below[a] = below;
        const int ao = other ? (below ? atm : atp) : at0, bo = other ? (below ? bm : bp) : bs;
        t.w[a][1][0] = below && !lo ? 0.0f : 1.0f - tc;
        t.w[a][1][1] = !below && !hi ? 0.0f : tc;
        t.at[a][1][0] = below ? ao : at0;
        t.blk[a][1][0] = below ? bo : bs;
        t.at[a][1][1] = below ? at0 : ao;
        t.blk[a][1][1] = below ? bs : bo;
        t.cross = t.cross || t.blk[a][0][1] != bs || bo != bs;
    }
    return true;
}

// The 24 addresses; a tap whose block has another level is looked up by itself.
// (With the whole sample by the walk instead, jumps between levels everywhere
// cost more than no table at all: 2.1M particles over random levels, G2P 132 us
// without it, 292 and now 124 with it; the advection 225, 400 and 284.)  false:
// a tap with weight has no cell.
__device__ inline bool tap_addresses(const MGrid& g, const SampleTaps& t, const int* __restrict__ nbr,
                                     int (&addr)[3][8]) {
#pragma unroll
    for (int ax = 0; ax < 3; ++ax)
#pragma unroll
        for (int q = 0; q < 8; ++q)
            addr[ax][q] = t.at[0][ax != 0][q >> 2] + t.at[1][ax != 1][q >> 1 & 1] + t.at[2][ax != 2][q & 1];
    if (!t.cross) {
#pragma unroll
        for (int ax = 0; ax < 3; ++ax)
#pragma unroll
            for (int q = 0; q < 8; ++q) addr[ax][q] += t.base;
        return true;
    }
    int all = 0;
    const int* nb = nbr + 27 * (int64_t)t.slot;
#pragma unroll
    for (int ax = 0; ax < 3; ++ax)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int b = nb[t.blk[0][ax != 0][q >> 2] + t.blk[1][ax != 1][q >> 1 & 1] + t.blk[2][ax != 2][q & 1]];
            all |= b;
            addr[ax][q] = b < 0 ? -1 : addr[ax][q] + b;
        }
    if (all >= 0) return true;
    bool found = true;
#pragma unroll
    for (int ax = 0; ax < 3; ++ax)
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (addr[ax][q] >= 0) continue;
            const int e[3] = {q >> 2, q >> 1 & 1, q & 1};
            int x[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) x[a] = (t.cell[a] + e[a] - (ax != a && t.below[a] ? 1 : 0)) << t.level;
            const int at = locate(g, x[0], x[1], x[2]).addr;
            found = found && (at >= 0 || !(tap_weight(t.w[0][ax != 0][e[0]], t.w[1][ax != 1][e[1]],
                                                      t.w[2][ax != 2][e[2]]) > 0.0f));
            addr[ax][q] = max(at, 0);
        }
    return found;
}

// the samples of sample_face for all three components: the same values,
// weights and order
__device__ inline void tap_sum(const SampleTaps& t, const int (&addr)[3][8], const float* __restrict__ f,
                               float (&out)[3]) {
    float v[3][8];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax)
#pragma unroll
        for (int q = 0; q < 8; ++q) v[ax][q] = f[(int64_t)addr[ax][q] * 3 + ax];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        float acc = 0.0f, wsum = 0.0f;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float w = tap_weight(t.w[0][ax != 0][q >> 2], t.w[1][ax != 1][q >> 1 & 1], t.w[2][ax != 2][q & 1]);
            acc = fmaf(w, v[ax][q], acc);
            wsum += w;
        }
        out[ax] = wsum > 0.0f ? acc / wsum : 0.0f;
    }
}

__device__ inline void sample_walk(const MGrid& g, const float* __restrict__ f, const float (&x)[3],
                                   float (&out)[3]) {
    const SamplePoint sp = sample_point(g, x[0], x[1], x[2]);
#pragma unroll 1
    for (int ax = 0; ax < 3; ++ax) {
        const float r = sample_face(g, f, x[0], x[1], x[2], ax, sp);
        out[0] = ax == 0 ? r : out[0];
        out[1] = ax == 1 ? r : out[1];
        out[2] = ax == 2 ? r : out[2];
    }
}

// first cells of the 27 blocks around each block that have its level
__global__ __launch_bounds__(256) void k_mr_neighbours(MGrid g, int* __restrict__ nbr) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= 27 * (int64_t)g.nslots) return;
    const int s = (int)(e / 27), d = (int)(e - 27 * (int64_t)s), b = g.blk[s];
    const int i = b / (g.nbz * g.nby) + d / 9 - 1, j = b / g.nbz % g.nby + d / 3 % 3 - 1, k = b % g.nbz + d % 3 - 1;
    int first = -1;
    if (i >= 0 && j >= 0 && k >= 0 && i < g.nbx && j < g.nby && k < g.nbz) {
        const int q = g.slot[(i * g.nby + j) * g.nbz + k];
        if (q >= 0 && g.blev[q] == g.blev[s]) first = g.coff[q];
    }
    nbr[e] = first;
}

// alpha_FLIP from the local grid spacing (particles.py:251-276), then
// u_p = alpha (u_p + I(du)) + (1 - alpha) I(u), eq. (12) (mr_kernels.py:413-430).
// NEAR: with the table of sample_taps, the walk only for a sample with a tap
// that has no cell.  9.2M particles, 6 % of them along 2:1 jumps: 672 us
// without the table, 365 with it.
template <bool NEAR>
__global__ __launch_bounds__(256) void k_mr_g2p(MGrid g, const int* __restrict__ nbr, const float* __restrict__ x,
                                                float* __restrict__ v, const int* __restrict__ type, int64_t n,
                                                MRConst c, const float* __restrict__ fvel,
                                                const float* __restrict__ fdvel) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const float q[3] = {x[3 * p], x[3 * p + 1], x[3 * p + 2]};
    const float vp[3] = {v[3 * p], v[3 * p + 1], v[3 * p + 2]};
    const float nu = type[p] == 1 ? c.nu_l : c.nu_g;
    float delta[3] = {0.0f, 0.0f, 0.0f}, pic[3] = {0.0f, 0.0f, 0.0f};
    int level = 0;
    if constexpr (NEAR) {
        SampleTaps t;
        if (sample_taps(g, q, t)) {
            level = t.level;
            int addr[3][8];
            if (tap_addresses(g, t, nbr, addr)) {
                tap_sum(t, addr, fdvel, delta);
                tap_sum(t, addr, fvel, pic);
            } else {
                sample_walk(g, fdvel, q, delta);
                sample_walk(g, fvel, q, pic);
            }
        }
    } else {
        const SamplePoint sp = sample_point(g, q[0], q[1], q[2]);
        if (sp.c.addr >= 0) {
            level = sp.c.level;
            WalkTaps t;
            walk_taps(g, q[0], q[1], q[2], sp, t);
            float vd[3][8], vu[3][8];
            walk_values(fdvel, t, vd);
            walk_values(fvel, t, vu);
            walk_sum(t, vd, delta);
            walk_sum(t, vu, pic);
        }
    }
    const float dx = cell_size(g, level);
    const float alpha = fminf(fmaxf(1.0f - 6.0f * nu * c.dt / (dx * dx), 0.0f), c.alpha_cap);
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) v[3 * p + ax] = fmaf(1.0f - alpha, pic[ax], alpha * (vp[ax] + delta[ax]));
}

// x + dt (2 k1 + 3 k2 + 4 k3) / 9, with the roundings spelled out
__device__ inline float rk3_end(float x, float dt, float k1, float k2, float k3) {
#pragma clang fp contract(off)
    return fmaf(dt, fmaf(2.0f / 9.0f, k1, (3.0f / 9.0f) * k2) + (4.0f / 9.0f) * k3, x);
}

// Ralston RK3 through the MSBG velocity, clamped to [lo, hi]
// (mr_kernels.py:421-438), then the wall reflection of the velocity
// (mr_kernels.py:441-461).  NEAR as above; one body for the three stages keeps
// it at 128 registers.  9.2M particles: 1036 us without the table, 660 with it.
template <bool NEAR>
__global__ __launch_bounds__(256) void k_mr_advect(MGrid g, const int* __restrict__ nbr, float* __restrict__ x,
                                                   float* __restrict__ v, int64_t n, MRConst c,
                                                   const float* __restrict__ fvel) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const float q[3] = {x[3 * p], x[3 * p + 1], x[3 * p + 2]};
    float k[3] = {0.0f, 0.0f, 0.0f}, k1[3], k2[3];
    if constexpr (NEAR) {
#pragma unroll 1
        for (int s = 0; s < 3; ++s) {
            const float a = s == 0 ? 0.0f : (s == 1 ? 0.5f * c.dt : 0.75f * c.dt);
            float y[3];
#pragma unroll
            for (int ax = 0; ax < 3; ++ax) {
                k1[ax] = s == 1 ? k[ax] : k1[ax];
                k2[ax] = s == 2 ? k[ax] : k2[ax];
                y[ax] = s == 0 ? q[ax] : fmaf(a, k[ax], q[ax]);
                k[ax] = 0.0f;
            }
            SampleTaps t;
            if (sample_taps(g, y, t)) {
                int addr[3][8];
                if (tap_addresses(g, t, nbr, addr))
                    tap_sum(t, addr, fvel, k);
                else
                    sample_walk(g, fvel, y, k);
            }
        }
    } else {
        float y[3];
        SamplePoint sp = sample_point(g, q[0], q[1], q[2]);
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) k1[ax] = sample_face(g, fvel, q[0], q[1], q[2], ax, sp);
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) y[ax] = fmaf(0.5f * c.dt, k1[ax], q[ax]);
        sp = sample_point(g, y[0], y[1], y[2]);
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) k2[ax] = sample_face(g, fvel, y[0], y[1], y[2], ax, sp);
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) y[ax] = fmaf(0.75f * c.dt, k2[ax], q[ax]);
        sp = sample_point(g, y[0], y[1], y[2]);
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) k[ax] = sample_face(g, fvel, y[0], y[1], y[2], ax, sp);
    }
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        float xa = rk3_end(q[ax], c.dt, k1[ax], k2[ax], k[ax]);
        xa = fminf(fmaxf(xa, c.lo[ax]), c.hi[ax]);
        float va = v[3 * p + ax];
        if (xa <= c.lo[ax])
            va = fmaxf(va, 0.0f);
        else if (xa >= c.hi[ax])
            va = fminf(va, 0.0f);
        x[3 * p + ax] = xa;
        v[3 * p + ax] = va;
    }
}

// ------------------------------------------------------------------ 6. resampling
// A block is "interface" when its cells hold both phases (mr_kernels.py:464-477);
// one workgroup per active block reduces its contiguous cell range.
__global__ __launch_bounds__(256) void k_mr_block_phase(MGrid g, const int* __restrict__ is_liquid,
                                                        int* __restrict__ mixed) {
    const int s = blockIdx.x;
    const int c0 = g.coff[s];
    const int nn = g.n0 >> g.blev[s];
    const int cnt = nn * nn * nn;
    int liq = 0, air = 0;
    for (int i = threadIdx.x; i < cnt; i += blockDim.x) {
        const int t = is_liquid[c0 + i];
        liq |= t;
        air |= 1 - t;
    }
    __shared__ int sh[2][4];
    liq = __any(liq) ? 1 : 0;
    air = __any(air) ? 1 : 0;
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = liq;
        sh[1][threadIdx.x >> 6] = air;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int l = 0, a = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
            l |= sh[0][w];
            a |= sh[1][w];
        }
        mixed[g.blk[s]] = (l && a) ? 1 : 0;
    }
}

constexpr int kInfD2 = 1 << 30;

// exact Euclidean distance to the nearest interface block, in block units,
// as separable squared-distance passes along z, y, x (the reference calls
// scipy.ndimage.distance_transform_edt: particles.py:387-419)
__global__ __launch_bounds__(256) void k_mr_edt(int pass, const int* __restrict__ mixed, const int* __restrict__ in,
                                                int* __restrict__ out, float* __restrict__ dist, int nbx, int nby,
                                                int nbz, float max_dist) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nbx * nby * nbz) return;
    const int k = t % nbz, j = (t / nbz) % nby, i = t / (nbz * nby);
    int best = kInfD2;
    if (pass == 0) {
        for (int kk = 0; kk < nbz; ++kk)
            if (mixed[(i * nby + j) * nbz + kk]) best = min(best, (k - kk) * (k - kk));
        out[t] = best;
    } else if (pass == 1) {
        for (int jj = 0; jj < nby; ++jj) {
            const int g = in[(i * nby + jj) * nbz + k];
            if (g < kInfD2) best = min(best, g + (j - jj) * (j - jj));
        }
        out[t] = best;
    } else {
        for (int ii = 0; ii < nbx; ++ii) {
            const int g = in[(ii * nby + j) * nbz + k];
            if (g < kInfD2) best = min(best, g + (i - ii) * (i - ii));
        }
        dist[t] = best >= kInfD2 ? max_dist : fminf((float)sqrt((double)best), max_dist);
    }
}

// l_new = floor(|beta_bw d~|) with d~ interpolated trilinearly from the block
// raster, clamped to [0, max_level] and to one level per step; deferred
// probabilistic coarsening (particles.py:88-168).  nout = 0, 1 or 8.
__global__ __launch_bounds__(256) void k_mr_classify(const float* __restrict__ x, const int* __restrict__ lev,
                                                     int* __restrict__ defer, const float* __restrict__ dist, int nbx,
                                                     int nby, int nbz, float bext, float beta_bw, int max_level,
                                                     int threshold, int seed, int* __restrict__ lnew_out,
                                                     int* __restrict__ nout, int64_t n) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const float gx = x[3 * p] / bext - 0.5f, gy = x[3 * p + 1] / bext - 0.5f, gz = x[3 * p + 2] / bext - 0.5f;
    const float fi = floorf(gx), fj = floorf(gy), fk = floorf(gz);
    const int i0 = (int)fi, j0 = (int)fj, k0 = (int)fk;
    const float tx = gx - fi, ty = gy - fj, tz = gz - fk;
    float d = 0.0f;
    for (int a = 0; a < 2; ++a) {
        const float wa = a == 0 ? 1.0f - tx : tx;
        const int ii = min(max(i0 + a, 0), nbx - 1);
        for (int b = 0; b < 2; ++b) {
            const float wb = b == 0 ? 1.0f - ty : ty;
            const int jj = min(max(j0 + b, 0), nby - 1);
            for (int cc = 0; cc < 2; ++cc) {
                const float wc = cc == 0 ? 1.0f - tz : tz;
                const int kk = min(max(k0 + cc, 0), nbz - 1);
                d += wa * wb * wc * dist[(ii * nby + jj) * nbz + kk];
            }
        }
    }
    const int lp = lev[p];
    int ln = min(max((int)floorf(fabsf(beta_bw * d)), 0), max_level);
    ln = min(max(ln, lp - 1), lp + 1);
    lnew_out[p] = ln;
    if (ln < lp) {
        defer[p] = 0;
        nout[p] = 8;
        return;
    }
    if (ln > lp) {
        const int dp = defer[p] + 1;
        defer[p] = dp;
        if (dp >= threshold) {
            uint32_t st = rng_init(seed, (int32_t)p);
            const float prob_del = 1.0f - ldexpf(1.0f, -3 * (ln - lp));
            if (rng_uniform(st) < prob_del) {
                nout[p] = 0;
                return;
            }
        }
        nout[p] = 1;
        return;
    }
    defer[p] = 0;
    nout[p] = 1;
}

// survivors (promoted when the counter fired) and 8 split children jittered
// inside the octants of the parent's cell (particles.py:171-231)
__global__ __launch_bounds__(256) void k_mr_emit(const float* __restrict__ x, const float* __restrict__ v,
                                                 const int* __restrict__ type, const int* __restrict__ lev,
                                                 const int* __restrict__ defer, const int* __restrict__ lnew,
                                                 const int* __restrict__ nout, const int* __restrict__ off, int64_t n,
                                                 int64_t cap, int threshold, float r0, int seed, float* __restrict__ ox,
                                                 float* __restrict__ ov, int* __restrict__ otype,
                                                 int* __restrict__ olev, int* __restrict__ odefer) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int cnt = nout[p];
    const int64_t o = off[p];
    if (cnt == 0 || o + cnt > cap) return;  // the host sized the output from offsets[n]
    const float px = x[3 * p], py = x[3 * p + 1], pz = x[3 * p + 2];
    const float vx = v[3 * p], vy = v[3 * p + 1], vz = v[3 * p + 2];
    const int t = type[p], lp = lev[p], ln = lnew[p];
    if (cnt == 1) {
        ox[3 * o] = px;
        ox[3 * o + 1] = py;
        ox[3 * o + 2] = pz;
        ov[3 * o] = vx;
        ov[3 * o + 1] = vy;
        ov[3 * o + 2] = vz;
        otype[o] = t;
        const bool promote = ln > lp && defer[p] >= threshold;
        olev[o] = promote ? ln : lp;
        odefer[o] = promote ? 0 : defer[p];
        return;
    }
    const float hp = r0 * (float)(1 << lp);
    const float half = 0.5f * hp;
    uint32_t st = rng_init(seed, (int32_t)p);
    for (int ch = 0; ch < 8; ++ch) {
        const float sx = (float)(ch & 1) - 0.5f, sy = (float)((ch >> 1) & 1) - 0.5f, sz = (float)((ch >> 2) & 1) - 0.5f;
        const float jx = (rng_uniform(st) - 0.5f) * half;
        const float jy = (rng_uniform(st) - 0.5f) * half;
        const float jz = (rng_uniform(st) - 0.5f) * half;
        const int64_t q = o + ch;
        ox[3 * q] = px + sx * half + jx;
        ox[3 * q + 1] = py + sy * half + jy;
        ox[3 * q + 2] = pz + sz * half + jz;
        ov[3 * q] = vx;
        ov[3 * q + 1] = vy;
        ov[3 * q + 2] = vz;
        otype[q] = t;
        olev[q] = lp - 1;
        odefer[q] = 0;
    }
}

}  // namespace pf

using namespace pf;

static int check_mgrid(const pf_msbg_grid* g, const char* who) {
    PF_REQUIRE(g && g->ncells > 0 && g->nslots > 0 && g->n0 == (1 << g->sh0) && g->h0 > 0.f, "%s: bad grid", who);
    PF_REQUIRE(g->level && g->slot && g->blk && g->blev && g->coff && g->cslot, "%s: null grid array", who);
    // face fields are indexed 3 * cell + axis in 32-bit arithmetic
    PF_REQUIRE(g->ncells <= kMsbgMaxCells, "%s: %d cells exceed the limit of %d", who, g->ncells, kMsbgMaxCells);
    return PF_OK;
}

static int check_parts(const pf_mr_particles* ps, const char* who) {
    PF_REQUIRE(ps && ps->n >= 0 && ps->n < ((int64_t)1 << 31), "%s: bad particle set", who);
    PF_REQUIRE(ps->n == 0 || (ps->x && ps->v && ps->type && ps->level && ps->defer), "%s: null particle array",
               who);
    return PF_OK;
}

static unsigned pgrid(int64_t n) { return cdiv(n > 0 ? n : 1, 256); }

PF_API int pf_mr_refine_map(const pf_mr_particles* ps, int32_t* level_map, int32_t nbx, int32_t nby, int32_t nbz,
                            float block_extent, float cfl_eps, int32_t max_level, pf_stream_t stream) {
    int rc = check_parts(ps, "pf_mr_refine_map");
    if (rc) return rc;
    PF_REQUIRE(level_map && nbx > 0 && nby > 0 && nbz > 0 && block_extent > 0.f && max_level >= 0,
               "pf_mr_refine_map: bad block raster");
    rc = fill_u32(level_map, (int64_t)nbx * nby * nbz, (uint32_t)max_level, S(stream));
    if (rc) return rc;
    if (ps->n == 0) return PF_OK;
    k_mr_refine_map<<<pgrid(ps->n), 256, 0, S(stream)>>>(ps->x, ps->level, ps->n, level_map, nbx, nby, nbz,
                                                         block_extent, cfl_eps);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_max_speed(const float* v, int64_t n, float* out, pf_stream_t stream) {
    PF_REQUIRE(out && (n == 0 || v), "pf_mr_max_speed: null pointer");
    int rc = fill_u32(out, 1, 0u, S(stream));
    if (rc || n == 0) return rc;
    const unsigned nb = cdiv(n, 256) < 2048u ? cdiv(n, 256) : 2048u;
    k_mr_max_speed<<<nb, 256, 0, S(stream)>>>(v, n, out);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_p2g(const pf_msbg_grid* g, const pf_mr_particles* ps, const pf_mr_params* prm, pf_mr_fields* f,
                     pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_p2g");
    if (rc) return rc;
    rc = check_parts(ps, "pf_mr_p2g");
    if (rc) return rc;
    PF_REQUIRE(prm && f && f->acc, "pf_mr_p2g: null params / accumulators");
    PF_REQUIRE(prm->mass_scale > 0.0 && prm->mom_scale > 0.0 && prm->w_scale > 0.0, "pf_mr_p2g: bad scales");
    if (ps->n == 0) return PF_OK;
    k_mr_p2g<<<pgrid(ps->n), 256, 0, S(stream)>>>(mgrid(*g), ps->x, ps->v, ps->type, ps->level, ps->n, mrconst(*prm),
                                                  reinterpret_cast<unsigned long long*>(f->acc));
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int64_t pf_mr_p2g_scratch_ints(int64_t n, int32_t ncells) {
    // key, rank, perm (n each); count (ncells + 1, then flags of as many blocks
    // and of ncells / 512 tiles); start (ncells + 2); scan
    return 3 * (n > 0 ? n : 1) + 2 * ((int64_t)ncells + 2) + cdiv(ncells, 512) + scan_tmp_ints((int64_t)ncells + 1);
}

PF_API int pf_mr_p2g_sorted(const pf_msbg_grid* g, const pf_mr_particles* ps, const pf_mr_params* prm,
                            pf_mr_fields* f, int32_t* scratch, pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_p2g_sorted");
    if (rc) return rc;
    rc = check_parts(ps, "pf_mr_p2g_sorted");
    if (rc) return rc;
    PF_REQUIRE(prm && f && f->acc && scratch, "pf_mr_p2g_sorted: null params / accumulators / scratch");
    PF_REQUIRE(prm->mass_scale > 0.0 && prm->mom_scale > 0.0 && prm->w_scale > 0.0, "pf_mr_p2g_sorted: bad scales");
    const int64_t n = ps->n;
    if (n == 0) return PF_OK;
    const int64_t nk = (int64_t)g->ncells + 1;
    int* key = scratch;
    int* rank = key + n;
    int* perm = rank + n;
    int* count = perm + n;
    int* start = count + (nk + 1) + cdiv(g->ncells, 512);
    int* tmp = start + (nk + 1);
    hipStream_t s = S(stream);
    rc = fill_u32(count, nk, 0u, s);
    if (rc) return rc;
    const MGrid m = mgrid(*g);
    k_mr_cell_key<<<pgrid(n), 256, 0, s>>>(m, ps->x, n, key, rank, count);
    PF_CHECK_LAUNCH();
    rc = exclusive_scan(count, nk, start, tmp, s);
    if (rc) return rc;
    // the scan's scratch and the counts are free now: the lengths of the walk's
    // lists, and a flag per workgroup of the tiles (then at the first cell of a
    // block of 4 cells per axis); the lists take the places of the keys and
    // ranks once the scatter has read them
    int* nlist = tmp;
    k_mr_cell_scatter<<<pgrid(n), 256, 0, s>>>(key, rank, start, n, perm, nlist);
    PF_CHECK_LAUNCH();
    const MRConst c = mrconst(*prm);
    unsigned long long* acc = reinterpret_cast<unsigned long long*>(f->acc);
    // (a heavy tile has more than kP2GLight particles: the ranks' place holds
    // their names)
    int2* heavy = reinterpret_cast<int2*>(rank + (reinterpret_cast<uintptr_t>(rank) / 4 & 1));
    // few particles leave most of the chip idle between the tile launches: 33k
    // and 111k in tiles 77 and 80 us, all by the walk 65 and 75; 262k 86 and 109
    const bool tiled = n >= (int64_t)1 << 17;
    if (tiled) {
        const int chunks = (int)cdiv(m.ncells, 512);
        const unsigned tiles = (unsigned)chunks + (unsigned)std::min(m.nslots, kP2GWhole);
        k_mr_p2g_tile<1><<<tiles, P2GTile<1>::NT, 0, s>>>(m, chunks, ps->x, ps->v, ps->type, ps->level, perm, start, c,
                                                          count, key, heavy, nlist, acc);
        PF_CHECK_LAUNCH();
        k_mr_p2g_tile<2><<<tiles, P2GTile<2>::NT, 0, s>>>(m, chunks, ps->x, ps->v, ps->type, ps->level, perm, start, c,
                                                          count, key, heavy, nlist, acc);
        PF_CHECK_LAUNCH();
    }
    k_mr_p2g_walk<<<tiled ? kP2GWalkBlocks : std::min(kP2GWalkBlocks, cdiv(n, 256)), 256, 0, s>>>(m, ps->x, ps->v, ps->type, ps->level, key, heavy,
                                                tiled ? nlist : nullptr, perm, start, (int)n, c, acc);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_finish(const pf_msbg_grid* g, const pf_mr_params* prm, pf_mr_fields* f, pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_finish");
    if (rc) return rc;
    PF_REQUIRE(prm && f && f->acc && f->cwsum && f->phi && f->is_liquid && f->fmass && f->fvel,
               "pf_mr_finish: null field");
    k_mr_finish<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), mrconst(*prm), f->acc, f->cwsum, f->phi,
                                                             f->is_liquid, f->fmass, f->fvel);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_face_prepare(const pf_msbg_grid* g, const pf_mr_params* prm, pf_mr_fields* f, pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_face_prepare");
    if (rc) return rc;
    PF_REQUIRE(prm && f && f->is_liquid && f->fmass && f->fbeta && f->fvel && f->fvel_star,
               "pf_mr_face_prepare: null field");
    k_mr_face_prepare<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), mrconst(*prm), f->is_liquid, f->fmass,
                                                                   f->fbeta, f->fvel, f->fvel_star);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_rhs(const pf_msbg_grid* g, const pf_mr_params* prm, pf_mr_fields* f, pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_rhs");
    if (rc) return rc;
    PF_REQUIRE(prm && f && f->fvel && f->cwsum && f->rhs, "pf_mr_rhs: null field");
    PF_REQUIRE(prm->dt > 0.f, "pf_mr_rhs: dt must be positive");
    k_mr_rhs<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), mrconst(*prm), f->fvel, f->cwsum, f->rhs);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_project(const pf_msbg_grid* g, const pf_mr_params* prm, pf_mr_fields* f, pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_project");
    if (rc) return rc;
    PF_REQUIRE(prm && f && f->pressure && f->fbeta && f->fvel && f->fvel_star && f->fdvel,
               "pf_mr_project: null field");
    k_mr_project<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), mrconst(*prm), f->pressure, f->fbeta,
                                                              f->fvel, f->fvel_star, f->fdvel);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_max_divergence(const pf_msbg_grid* g, const float* fvel, float* out, pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_max_divergence");
    if (rc) return rc;
    PF_REQUIRE(fvel && out, "pf_mr_max_divergence: null pointer");
    rc = fill_u32(out, 1, 0u, S(stream));
    if (rc) return rc;
    k_mr_max_div<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), fvel, out);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_neighbours(const pf_msbg_grid* g, int32_t* nbr, pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_neighbours");
    if (rc) return rc;
    PF_REQUIRE(nbr, "pf_mr_neighbours: null table");
    k_mr_neighbours<<<cdiv(27 * (int64_t)g->nslots, 256), 256, 0, S(stream)>>>(mgrid(*g), nbr);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_g2p(const pf_msbg_grid* g, const pf_mr_particles* ps, const pf_mr_params* prm,
                     const pf_mr_fields* f, pf_stream_t stream) {
    return pf_mr_g2p_near(g, nullptr, ps, prm, f, stream);
}

PF_API int pf_mr_g2p_near(const pf_msbg_grid* g, const int32_t* nbr, const pf_mr_particles* ps,
                          const pf_mr_params* prm, const pf_mr_fields* f, pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_g2p");
    if (rc) return rc;
    rc = check_parts(ps, "pf_mr_g2p");
    if (rc) return rc;
    PF_REQUIRE(prm && f && f->fvel && f->fdvel, "pf_mr_g2p: null field");
    if (ps->n == 0) return PF_OK;
    const auto k = nbr ? k_mr_g2p<true> : k_mr_g2p<false>;
    k<<<pgrid(ps->n), 256, 0, S(stream)>>>(mgrid(*g), nbr, ps->x, ps->v, ps->type, ps->n, mrconst(*prm), f->fvel,
                                           f->fdvel);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_advect(const pf_msbg_grid* g, const pf_mr_particles* ps, const pf_mr_params* prm,
                        const float* fvel, pf_stream_t stream) {
    return pf_mr_advect_near(g, nullptr, ps, prm, fvel, stream);
}

PF_API int pf_mr_advect_near(const pf_msbg_grid* g, const int32_t* nbr, const pf_mr_particles* ps,
                             const pf_mr_params* prm, const float* fvel, pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_advect");
    if (rc) return rc;
    rc = check_parts(ps, "pf_mr_advect");
    if (rc) return rc;
    PF_REQUIRE(prm && fvel, "pf_mr_advect: null pointer");
    if (ps->n == 0) return PF_OK;
    const auto k = nbr ? k_mr_advect<true> : k_mr_advect<false>;
    k<<<pgrid(ps->n), 256, 0, S(stream)>>>(mgrid(*g), nbr, ps->x, ps->v, ps->n, mrconst(*prm), fvel);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mr_block_distance(const pf_msbg_grid* g, const int32_t* is_liquid, int32_t* mixed, int32_t* tmp,
                                float* dist, float max_dist, pf_stream_t stream) {
    int rc = check_mgrid(g, "pf_mr_block_distance");
    if (rc) return rc;
    PF_REQUIRE(is_liquid && mixed && tmp && dist, "pf_mr_block_distance: null pointer");
    const int nblk = g->nbx * g->nby * g->nbz;
    rc = fill_u32(mixed, nblk, 0u, S(stream));
    if (rc) return rc;
    k_mr_block_phase<<<g->nslots, 256, 0, S(stream)>>>(mgrid(*g), is_liquid, mixed);
    PF_CHECK_LAUNCH();
    int* a = tmp;
    int* b = tmp + nblk;
    k_mr_edt<<<cdiv(nblk, 256), 256, 0, S(stream)>>>(0, mixed, nullptr, a, nullptr, g->nbx, g->nby, g->nbz, max_dist);
    PF_CHECK_LAUNCH();
    k_mr_edt<<<cdiv(nblk, 256), 256, 0, S(stream)>>>(1, mixed, a, b, nullptr, g->nbx, g->nby, g->nbz, max_dist);
    PF_CHECK_LAUNCH();
    k_mr_edt<<<cdiv(nblk, 256), 256, 0, S(stream)>>>(2, mixed, b, nullptr, dist, g->nbx, g->nby, g->nbz, max_dist);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int64_t pf_mr_scan_tmp_ints(int64_t n) { return scan_tmp_ints(n > 0 ? n : 1); }

PF_API int pf_mr_classify(const pf_mr_particles* ps, const float* dist, int32_t nbx, int32_t nby, int32_t nbz,
                          float block_extent, float beta_bw, int32_t max_level, int32_t defer_threshold, int32_t seed,
                          int32_t* lnew, int32_t* nout, int32_t* offsets, int32_t* scan_tmp, pf_stream_t stream) {
    int rc = check_parts(ps, "pf_mr_classify");
    if (rc) return rc;
    PF_REQUIRE(dist && lnew && nout && offsets && scan_tmp && nbx > 0 && nby > 0 && nbz > 0 && block_extent > 0.f,
               "pf_mr_classify: bad arguments");
    if (ps->n == 0) return fill_u32(offsets, 1, 0u, S(stream));
    k_mr_classify<<<pgrid(ps->n), 256, 0, S(stream)>>>(ps->x, ps->level, ps->defer, dist, nbx, nby, nbz, block_extent,
                                                       beta_bw, max_level, defer_threshold, seed, lnew, nout, ps->n);
    PF_CHECK_LAUNCH();
    return exclusive_scan(nout, ps->n, offsets, scan_tmp, S(stream));
}

PF_API int pf_mr_emit(const pf_mr_particles* in, const int32_t* lnew, const int32_t* nout, const int32_t* offsets,
                      int32_t defer_threshold, float r0, int32_t seed, pf_mr_particles* out, pf_stream_t stream) {
    int rc = check_parts(in, "pf_mr_emit");
    if (rc) return rc;
    rc = check_parts(out, "pf_mr_emit");
    if (rc) return rc;
    PF_REQUIRE(lnew && nout && offsets, "pf_mr_emit: null pointer");
    if (in->n == 0) return PF_OK;
    k_mr_emit<<<pgrid(in->n), 256, 0, S(stream)>>>(in->x, in->v, in->type, in->level, in->defer, lnew, nout, offsets,
                                                   in->n, out->n, defer_threshold, r0, seed, out->x, out->v, out->type,
                                                   out->level, out->defer);
    PF_CHECK_LAUNCH();
    return PF_OK;
}
