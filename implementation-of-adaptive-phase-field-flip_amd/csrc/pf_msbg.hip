// Multiresolution sparse block grid (MSBG): addressing, the 2:1 variable-
// coefficient Poisson operator and the aggregation multigrid transfers
// (pfflip/msbg.py, pfflip/mr_operator.py, pfflip/mr_multigrid.py).
//
// Blocks have one geometric size; a level-l block holds (n0 >> l)^3 cells.
// Every lookup goes through finest-level integer coordinates: block =
// F >> log2(n0), cell = (F & (n0 - 1)) >> l.  Each cell stores its three
// low-side faces; the face between two cells is read from the cell on its
// high side, so both rows see one coefficient and the operator is symmetric
// across resolution jumps.
//
// The red-black smoother reads one buffer and writes another: every cell of
// the active colour is updated from the values before the half-sweep.  With
// the finest-coordinate colouring two same-colour cells can touch across a
// resolution jump; reading the old values there makes the half-sweep
// deterministic.  Restriction gathers each coarse cell's children in a fixed
// order instead of adding them with atomics.
//
// The cell-parallel operator kernels take their cell range through
// xcd_block: the 16 workgroups of a 16^3 block then run on one XCD and the
// +-z neighbour rows they read from each other stay in that XCD's L2.
#include "pf_msbg.hpp"

namespace pf {

int fill_u32(void* dst, int64_t n, uint32_t v, hipStream_t s);

// Calls f(neighbour address, T) for every coupling of cell `addr`, with
// T = beta * min(hA, hB)^2 / ((hA + hB) / 2), walking the faces in the
// reference's order (mr_operator.py:74-166); across a face to finer cells
// the 2x2 patch behind it.
template <class F>
__device__ inline void for_each_coupling_from(const MGrid& g, const float* __restrict__ bface, int addr,
                                              const int4 o, const BlockRef& br, F&& f) {
    const int la = o.w;
    const int ext = 1 << la;
    const float hA = g.h0 * (float)ext;
    for (int axis = 0; axis < 3; ++axis) {
        const int ex = comp(axis, 0), ey = comp(axis, 1), ez = comp(axis, 2);
        for (int side = 0; side < 2; ++side) {
            int fx, fy, fz;
            if (side == 0) {
                fx = o.x - ex;
                fy = o.y - ey;
                fz = o.z - ez;
            } else {
                fx = o.x + ex * ext;
                fy = o.y + ey * ext;
                fz = o.z + ez * ext;
            }
            const MCell nb = locate_near(g, br, fx, fy, fz);
            if (nb.addr < 0) continue;  // domain wall: no flux
            const float hB = g.h0 * (float)(1 << nb.level);
            if (nb.level >= la) {
                // same size or coarser: one neighbour
                float area = fminf(hA, hB);
                area = area * area;
                const float dist = 0.5f * (hA + hB);
                const float beta = side == 0 ? bface[addr * 3 + axis] : bface[nb.addr * 3 + axis];
                f(nb.addr, beta * area / dist);
            } else {
                // finer: the 2x2 patch across this face
                const int sub = 1 << nb.level;
                const float area = hB * hB;
                const float dist = 0.5f * (hA + hB);
                const int a1 = (axis + 1) % 3, a2 = (axis + 2) % 3;
                for (int u = 0; u < 2; ++u)
                    for (int v = 0; v < 2; ++v) {
                        const int du = u * sub, dv = v * sub;
                        const MCell nc = locate_near(g, br, fx + comp(a1, 0) * du + comp(a2, 0) * dv,
                                                     fy + comp(a1, 1) * du + comp(a2, 1) * dv,
                                                     fz + comp(a1, 2) * du + comp(a2, 2) * dv);
                        if (nc.addr < 0) continue;
                        const float beta = side == 0 ? bface[addr * 3 + axis] : bface[nc.addr * 3 + axis];
                        f(nc.addr, beta * area / dist);
                    }
            }
        }
    }
}

template <class F>
__device__ inline void for_each_coupling(const MGrid& g, const float* __restrict__ bface, int addr, F&& f) {
    BlockRef br;
    const int4 o = origin_ref(g, addr, br);
    for_each_coupling_from(g, bface, addr, o, br, f);
}

// sum_f T_f (p_A - p_B) over the couplings of cell `addr` (origin o, block
// br), or (want_diag) the sum of T_f
__device__ inline float apply_row_from(const MGrid& g, const float* __restrict__ p,
                                       const float* __restrict__ bface, int addr, const int4 o,
                                       const BlockRef& br, bool want_diag) {
    const float pa = want_diag ? 0.0f : p[addr];
    float acc = 0.0f, diag = 0.0f;
    for_each_coupling_from(g, bface, addr, o, br, [&](int nb, float t) {
        diag += t;
        if (!want_diag) acc += t * (pa - p[nb]);
    });
    return want_diag ? diag : acc;
}

__device__ inline float apply_row(const MGrid& g, const float* __restrict__ p, const float* __restrict__ bface,
                                  int addr, bool want_diag) {
    BlockRef br;
    const int4 o = origin_ref(g, addr, br);
    return apply_row_from(g, p, bface, addr, o, br, want_diag);
}

__global__ __launch_bounds__(256) void k_msbg_apply(MGrid g, const float* __restrict__ p,
                                                    const float* __restrict__ bface, float* __restrict__ out,
                                                    int want_diag) {
    const int a = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (a >= g.ncells) return;
    out[a] = apply_row(g, p, bface, a, want_diag != 0);
}

__global__ __launch_bounds__(256) void k_msbg_residual(MGrid g, const float* __restrict__ p,
                                                       const float* __restrict__ b,
                                                       const float* __restrict__ bface, float* __restrict__ r) {
    const int a = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (a >= g.ncells) return;
    r[a] = b[a] - apply_row(g, p, bface, a, false);
}

// Grids from this many cells up take the paired half-sweep: on the 1.4M-cell
// level of a 128^3 dam break it runs 19.6 us against 25.9; on levels of a
// few thousand cells, mostly small blocks, it was up to twice as slow.
constexpr int kMsbgPairMinCells = 1 << 17;

// one cell of the half-sweep: the weighted update if the cell has the
// active colour and diag > 0, else a copy
__device__ inline void rbgs_cell(const MGrid& g, const float* __restrict__ pin, float* __restrict__ pout,
                                 const float* __restrict__ b, const float* __restrict__ bface,
                                 const float* __restrict__ diag, int colour, float omega, int a, const int4 o,
                                 const BlockRef& br) {
    float v = pin[a];
    if ((((o.x >> o.w) + (o.y >> o.w) + (o.z >> o.w)) & 1) == colour) {
        const float d = diag[a];
        if (d > 0.0f) v = v + omega * (b[a] - apply_row_from(g, pin, bface, a, o, br, false)) / d;
    }
    pout[a] = v;
}

// weighted Gauss-Seidel half-sweep of one colour (mr_operator.py:193-212),
// colour from the finest-coordinate checkerboard, pin -> pout; one thread
// per cell
__global__ __launch_bounds__(256) void k_msbg_rbgs(MGrid g, const float* __restrict__ pin, float* __restrict__ pout,
                                                   const float* __restrict__ b, const float* __restrict__ bface,
                                                   const float* __restrict__ diag, int colour, float omega) {
    const int a = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (a >= g.ncells) return;
    BlockRef br;
    const int4 o = origin_ref(g, a, br);
    rbgs_cell(g, pin, pout, b, bface, diag, colour, omega, a, o, br);
}

// The same half-sweep with thread t on cells 2t and 2t + 1.  When 2t sits at
// an even offset of a block with an even edge, the two are k-neighbours in
// one row and exactly one of them has the active colour: the thread updates
// that one and copies the other, so no lane of a wave idles through the
// coupling walk (with one cell per thread the colour alternates from lane to
// lane and half the lanes wait).  Otherwise both cells take the per-cell
// path, one after the other, which costs latency on grids of small blocks.
// Every cell gets the arithmetic of k_msbg_rbgs.
__global__ __launch_bounds__(256) void k_msbg_rbgs_pairs(MGrid g, const float* __restrict__ pin,
                                                         float* __restrict__ pout, const float* __restrict__ b,
                                                         const float* __restrict__ bface,
                                                         const float* __restrict__ diag, int colour, float omega) {
    const int t = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const int a0 = 2 * t;
    if (a0 >= g.ncells) return;
    BlockRef br;
    const int4 o0 = origin_ref(g, a0, br);
    if (br.n >= 2 && ((a0 - br.base) & 1) == 0) {
        // a0 + 1 is the next cell of the same row, of the other colour; the
        // pair is read and written as one 8-byte word (the host checks that
        // pin and pout are 8-byte aligned)
        const bool first = (((o0.x >> o0.w) + (o0.y >> o0.w) + (o0.z >> o0.w)) & 1) == colour;
        const int act = first ? a0 : a0 + 1;
        const int4 oa = first ? o0 : make_int4(o0.x, o0.y, o0.z + (1 << o0.w), o0.w);
        float2 v2 = *reinterpret_cast<const float2*>(pin + a0);
        float v = first ? v2.x : v2.y;
        const float d = diag[act];
        if (d > 0.0f) v = v + omega * (b[act] - apply_row_from(g, pin, bface, act, oa, br, false)) / d;
        if (first)
            v2.x = v;
        else
            v2.y = v;
        *reinterpret_cast<float2*>(pout + a0) = v2;
        return;
    }
    rbgs_cell(g, pin, pout, b, bface, diag, colour, omega, a0, o0, br);
    if (a0 + 1 < g.ncells) {
        BlockRef br1;
        const int4 o1 = origin_ref(g, a0 + 1, br1);
        rbgs_cell(g, pin, pout, b, bface, diag, colour, omega, a0 + 1, o1, br1);
    }
}

// All sweeps of the coarsest level in one workgroup: each row's couplings
// (neighbour, T) are gathered into LDS once, then every half-sweep reads LDS
// only.  Same couplings, same order, same arithmetic as k_msbg_rbgs, so the
// result equals the launched half-sweeps bit for bit.  p is read and
// overwritten; the sweep count is even in half-sweeps, so no copy is left.
constexpr int kRowMax = 24;  // 6 faces x a 2x2 patch
constexpr int kCoarsestThreads = 512;

__host__ __device__ inline size_t coarsest_lds_bytes(int n) {
    return (size_t)n * (kRowMax * (sizeof(float) + sizeof(unsigned short)) + 4 * sizeof(float) + 2);
}

__global__ __launch_bounds__(kCoarsestThreads) void k_msbg_coarsest(MGrid g, float* __restrict__ p,
                                                                    const float* __restrict__ b,
                                                                    const float* __restrict__ bface,
                                                                    const float* __restrict__ diag, int sweeps,
                                                                    float omega) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int n = g.ncells;
    float* coef = reinterpret_cast<float*>(lds);
    float* p0 = coef + (size_t)n * kRowMax;
    float* p1 = p0 + n;
    float* bb = p1 + n;
    float* dd = bb + n;
    unsigned short* nbr = reinterpret_cast<unsigned short*>(dd + n);
    unsigned char* cnt = reinterpret_cast<unsigned char*>(nbr + (size_t)n * kRowMax);
    unsigned char* col = cnt + n;
    // entry k of every row is contiguous (k * n + a): a wave's loads of one
    // entry hit consecutive LDS words, free of bank conflicts
    for (int a = threadIdx.x; a < n; a += blockDim.x) {
        int k = 0;
        for_each_coupling(g, bface, a, [&](int nb, float t) {
            coef[k * n + a] = t;
            nbr[k * n + a] = (unsigned short)nb;
            ++k;
        });
        cnt[a] = (unsigned char)k;
        const int4 o = origin(g, a);
        col[a] = (unsigned char)(((o.x >> o.w) + (o.y >> o.w) + (o.z >> o.w)) & 1);
        p0[a] = p[a];
        bb[a] = b[a];
        dd[a] = diag[a];
    }
    __syncthreads();
    float* pin = p0;
    float* pout = p1;
    for (int s = 0; s < sweeps; ++s)
        for (int c = 0; c < 2; ++c) {
            for (int a = threadIdx.x; a < n; a += blockDim.x) {
                float v = pin[a];
                if (col[a] == c) {
                    const float d = dd[a];
                    if (d > 0.0f) {
                        const float pa = pin[a];
                        float acc = 0.0f;
                        const int m = cnt[a];
                        for (int k = 0; k < m; ++k) acc += coef[k * n + a] * (pa - pin[nbr[k * n + a]]);
                        v = v + omega * (bb[a] - acc) / d;
                    }
                }
                pout[a] = v;
            }
            __syncthreads();
            float* t = pin;
            pin = pout;
            pout = t;
        }
    for (int a = threadIdx.x; a < n; a += blockDim.x) p[a] = pin[a];
}

// The coarsest level's smoothing as a matrix: `sweeps` red-black sweeps
// from zero followed by mean removal are a linear map b -> p, so column j
// is that map applied to the unit vector e_j.  One workgroup per column and
// one thread per cell, in FP64; op[j * n + t] is entry (t, j).  A V-cycle then
// applies it with one matrix-vector product (k_msbg_coarse_apply) instead of
// the sweeps.
// A row's first kOpRow couplings are in registers (a cell without finer
// neighbours has no more; another row walks its rest anew in every sweep) and
// only the iterate is read from LDS.  That leaves 27 KB of LDS per workgroup,
// so all 512 columns run at once instead of in two rounds, and a half-sweep
// is 7 reads: 259 -> 64 us at 512 cells and 80 sweeps, once per solve.
constexpr int kMsbgCoarseOpMax = 512;
constexpr int kOpRow = 6;

__host__ __device__ constexpr size_t coarse_op_lds_bytes(int n) {
    return (size_t)n * (2 * sizeof(double) + kOpRow * (sizeof(float) + sizeof(unsigned short)));
}

__global__ __launch_bounds__(kCoarsestThreads) void k_msbg_coarse_op(MGrid g, const float* __restrict__ bface,
                                                                     const float* __restrict__ diag, int sweeps,
                                                                     double omega, double* __restrict__ op) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    static_assert(kMsbgCoarseOpMax <= kCoarsestThreads, "one cell per thread");
    const int n = g.ncells, j = blockIdx.x, a = threadIdx.x;
    double* p0 = reinterpret_cast<double*>(lds);
    double* p1 = p0 + n;
    float* coef = reinterpret_cast<float*>(p1 + n);
    unsigned short* nbr = reinterpret_cast<unsigned short*>(coef + (size_t)kOpRow * n);
    __shared__ double sh[16];
    __shared__ double shift;
    int cnt = 0, colour = -1;
    double w = 0.0;
    float c[kOpRow];
    int nb[kOpRow];
    if (a < n) {
        for_each_coupling(g, bface, a, [&](int b, float t) {
            if (cnt < kOpRow) {
                coef[cnt * n + a] = t;
                nbr[cnt * n + a] = (unsigned short)b;
            }
            ++cnt;
        });
        const int4 o = origin(g, a);
        if (diag[a] > 0.0f) {
            colour = ((o.x >> o.w) + (o.y >> o.w) + (o.z >> o.w)) & 1;
            w = omega / (double)diag[a];
        }
        p0[a] = 0.0;
    }
#pragma unroll
    for (int k = 0; k < kOpRow; ++k) {  // (written and read by this thread alone)
        const bool has = k < cnt;
        c[k] = has ? coef[k * n + a] : 0.0f;
        nb[k] = has ? nbr[k * n + a] : min(a, n - 1);
    }
    __syncthreads();
    double* pin = p0;
    double* pout = p1;
    for (int sw = 0; sw < sweeps; ++sw)
        for (int col = 0; col < 2; ++col) {
            if (a < n) {
                double v = pin[a];
                if (colour == col) {
                    const double pa = v;
                    double acc = 0.0;
#pragma unroll
                    for (int k = 0; k < kOpRow; ++k) acc += (double)c[k] * (pa - pin[nb[k]]);
                    if (cnt > kOpRow) {
                        int k = 0;
                        for_each_coupling(g, bface, a, [&](int b, float t) {
                            if (k++ >= kOpRow) acc += (double)t * (pa - pin[b]);
                        });
                    }
                    v = pa + ((a == j ? 1.0 : 0.0) - acc) * w;
                }
                pout[a] = v;
            }
            __syncthreads();
            double* t = pin;
            pin = pout;
            pout = t;
        }
    double sm[1] = {a < n ? pin[a] : 0.0};
    block_sum<1>(sm, sh);
    if (a == 0) shift = -(sm[0] / (double)n);
    __syncthreads();
    if (a < n) op[(int64_t)j * n + a] = pin[a] + shift;
}

// p = op b in FP64, rounded to float.  A workgroup takes kApplyRows rows (128
// consecutive bytes of a column) and its 1024 threads 64 columns at a time,
// so 512 cells make 32 workgroups with 8 loads in flight per thread; 64 rows
// per workgroup of 8 waves left 8 CUs to read the 2 MB (22 -> 4.9 us out of
// HBM, 11 -> 5.2 out of L2).  Partials are added in a fixed order.
constexpr int kApplyRows = 16;

__global__ __launch_bounds__(1024) void k_msbg_coarse_apply(const double* __restrict__ op,
                                                            const float* __restrict__ b, float* __restrict__ p,
                                                            int n) {
    __shared__ double part[16][kApplyRows];
    const int r = threadIdx.x % kApplyRows, w = threadIdx.x >> 6;
    const int t = blockIdx.x * kApplyRows + r;
    constexpr int G = 1024 / kApplyRows, M = kMsbgCoarseOpMax / G;
    double acc = 0.0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int j = (int)threadIdx.x / kApplyRows + m * G;
        if (j < n && t < n) acc += op[(int64_t)j * n + t] * (double)b[j];
    }
    acc += __shfl_xor(acc, 16, 64);
    acc += __shfl_xor(acc, 32, 64);
    if ((threadIdx.x & 63) < kApplyRows) part[w][r] = acc;
    __syncthreads();
    if (threadIdx.x < kApplyRows && t < n) {
        double s = part[0][r];
        for (int q = 1; q < 16; ++q) s += part[q][r];
        p[t] = (float)s;
    }
}

// ------------------------------------------------------------------ adaptive relaxation
// Algorithm 2 of the paper as the reference runs it on a GPU
// (adaptive_relax.py:1-241): red-black sweeps restricted to an active block
// set, the per-block effective residual max |delta| diag, a threshold from
// the log-histogram of the first residuals, and re-activation of the blocks
// above it with their face neighbours.  Like k_msbg_rbgs the half-sweep reads
// pin and writes every cell of pout.

// one colour over the active blocks; delta = |update| of the updated cells
// (adaptive_relax.py:84-109)
__global__ __launch_bounds__(256) void k_msbg_rbgs_active(MGrid g, const float* __restrict__ pin,
                                                          float* __restrict__ pout, const float* __restrict__ b,
                                                          const float* __restrict__ bface,
                                                          const float* __restrict__ diag,
                                                          const int* __restrict__ active, int colour, float omega,
                                                          float* __restrict__ delta) {
    const int a = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (a >= g.ncells) return;
    float v = pin[a];
    if (active[g.cslot[a]]) {
        const int4 o = origin(g, a);
        if ((((o.x >> o.w) + (o.y >> o.w) + (o.z >> o.w)) & 1) == colour) {
            const float d = diag[a];
            if (d > 0.0f) {
                const float upd = omega * (b[a] - apply_row(g, pin, bface, a, false)) / d;
                v = v + upd;
                delta[a] = fabsf(upd);
            }
        }
    }
    pout[a] = v;
}

// k_msbg_rbgs_active with thread t on cells 2t and 2t + 1, paired as in
// k_msbg_rbgs_pairs (one cell of each colour in one block row, so both share
// the block's active flag); other cells take the per-cell path.  Same
// arithmetic and the same delta writes per cell.
__device__ inline void rbgs_active_cell(const MGrid& g, const float* __restrict__ pin, float* __restrict__ pout,
                                        const float* __restrict__ b, const float* __restrict__ bface,
                                        const float* __restrict__ diag, const int* __restrict__ active,
                                        int colour, float omega, float* __restrict__ delta, int a) {
    float v = pin[a];
    if (active[g.cslot[a]]) {
        BlockRef br;
        const int4 o = origin_ref(g, a, br);
        if ((((o.x >> o.w) + (o.y >> o.w) + (o.z >> o.w)) & 1) == colour) {
            const float d = diag[a];
            if (d > 0.0f) {
                const float upd = omega * (b[a] - apply_row_from(g, pin, bface, a, o, br, false)) / d;
                v = v + upd;
                delta[a] = fabsf(upd);
            }
        }
    }
    pout[a] = v;
}

__global__ __launch_bounds__(256) void k_msbg_rbgs_active_pairs(MGrid g, const float* __restrict__ pin,
                                                                float* __restrict__ pout,
                                                                const float* __restrict__ b,
                                                                const float* __restrict__ bface,
                                                                const float* __restrict__ diag,
                                                                const int* __restrict__ active, int colour,
                                                                float omega, float* __restrict__ delta) {
    const int t = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const int a0 = 2 * t;
    if (a0 >= g.ncells) return;
    BlockRef br;
    const int4 o0 = origin_ref(g, a0, br);
    if (br.n >= 2 && ((a0 - br.base) & 1) == 0) {
        float2 v2 = *reinterpret_cast<const float2*>(pin + a0);
        if (active[br.slot]) {
            const bool first = (((o0.x >> o0.w) + (o0.y >> o0.w) + (o0.z >> o0.w)) & 1) == colour;
            const int act = first ? a0 : a0 + 1;
            const int4 oa = first ? o0 : make_int4(o0.x, o0.y, o0.z + (1 << o0.w), o0.w);
            const float d = diag[act];
            if (d > 0.0f) {
                const float upd = omega * (b[act] - apply_row_from(g, pin, bface, act, oa, br, false)) / d;
                if (first)
                    v2.x = v2.x + upd;
                else
                    v2.y = v2.y + upd;
                delta[act] = fabsf(upd);
            }
        }
        *reinterpret_cast<float2*>(pout + a0) = v2;
        return;
    }
    rbgs_active_cell(g, pin, pout, b, bface, diag, active, colour, omega, delta, a0);
    if (a0 + 1 < g.ncells) rbgs_active_cell(g, pin, pout, b, bface, diag, active, colour, omega, delta, a0 + 1);
}

// res[slot] = max over the block's cells of delta * diag, 0 when inactive
// (adaptive_relax.py:112-129); one workgroup per block
__global__ __launch_bounds__(256) void k_msbg_block_res(MGrid g, const float* __restrict__ delta,
                                                        const float* __restrict__ diag,
                                                        const int* __restrict__ active, float* __restrict__ res) {
    const int s = blockIdx.x;
    __shared__ float sh[4];
    float m = 0.0f;
    if (active[s]) {
        const int c0 = g.coff[s];
        const int nn = g.n0 >> g.blev[s];
        const int cnt = nn * nn * nn;
        for (int i = threadIdx.x; i < cnt; i += blockDim.x) m = fmaxf(m, delta[c0 + i] * diag[c0 + i]);
    }
    m = block_max(m, sh);
    if (threadIdx.x == 0) res[s] = m;
}

// theta = exp(mean + sigma std) of log(res) over the positive entries
// (population std, two passes, FP64 in a fixed order); +inf when none is
// positive, which stops all further activation (adaptive_relax.py:220-231)
__global__ __launch_bounds__(256) void k_msbg_theta(const float* __restrict__ res, int ns, float sigma,
                                                    float* __restrict__ theta) {
    __shared__ double sh[2 * 16];
    double v[2] = {0.0, 0.0};
    for (int s = threadIdx.x; s < ns; s += blockDim.x)
        if (res[s] > 0.0f) {
            v[0] += log((double)res[s]);
            v[1] += 1.0;
        }
    block_sum<2>(v, sh);
    __shared__ double mean_cnt[2];
    if (threadIdx.x == 0) {
        mean_cnt[0] = v[1] > 0.0 ? v[0] / v[1] : 0.0;
        mean_cnt[1] = v[1];
    }
    __syncthreads();
    const double mean = mean_cnt[0], cnt = mean_cnt[1];
    double w[1] = {0.0};
    for (int s = threadIdx.x; s < ns; s += blockDim.x)
        if (res[s] > 0.0f) {
            const double d = log((double)res[s]) - mean;
            w[0] += d * d;
        }
    block_sum<1>(w, sh);
    if (threadIdx.x == 0)
        *theta = cnt > 0.0 ? (float)exp(mean + (double)sigma * sqrt(w[0] / cnt)) : __int_as_float(0x7f800000);
}

// blocks above theta and their face neighbours form the next active set
// (adaptive_relax.py:132-160); the writers all store 1
__global__ __launch_bounds__(256) void k_msbg_update_active(MGrid g, const float* __restrict__ res,
                                                            const float* __restrict__ theta,
                                                            int* __restrict__ active_next) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.nslots) return;
    if (!(res[s] > *theta)) return;
    active_next[s] = 1;
    const int b = g.blk[s];
    const int bz = b % g.nbz, by = (b / g.nbz) % g.nby, bx = b / (g.nbz * g.nby);
    for (int d = 0; d < 6; ++d) {
        const int ax = d >> 1, sg = (d & 1) ? 1 : -1;
        const int nx = bx + (ax == 0 ? sg : 0), ny = by + (ax == 1 ? sg : 0), nz = bz + (ax == 2 ? sg : 0);
        if (nx < 0 || ny < 0 || nz < 0 || nx >= g.nbx || ny >= g.nby || nz >= g.nbz) continue;
        const int ns = g.slot[(nx * g.nby + ny) * g.nbz + nz];
        if (ns >= 0) active_next[ns] = 1;
    }
}

// coarse face = mean of the 2x2 fine faces it covers (mr_multigrid.py:52-89)
__global__ __launch_bounds__(256) void k_msbg_coarsen_beta(MGrid cg, MGrid fg, const float* __restrict__ bfine,
                                                           float* __restrict__ bcoarse) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= cg.ncells) return;
    const int4 o = origin(cg, a);
    const int half = (1 << o.w) >> 1;
    for (int axis = 0; axis < 3; ++axis) {
        const int a1 = (axis + 1) % 3, a2 = (axis + 2) % 3;
        float acc = 0.0f, cnt = 0.0f;
        for (int u = 0; u < 2; ++u)
            for (int v = 0; v < 2; ++v) {
                const int du = u * half, dv = v * half;
                const MCell nc = locate(fg, o.x + comp(a1, 0) * du + comp(a2, 0) * dv,
                                        o.y + comp(a1, 1) * du + comp(a2, 1) * dv,
                                        o.z + comp(a1, 2) * du + comp(a2, 2) * dv);
                if (nc.addr >= 0) {
                    acc += bfine[nc.addr * 3 + axis];
                    cnt += 1.0f;
                }
            }
        bcoarse[a * 3 + axis] = cnt > 0.0f ? acc / cnt : 0.0f;
    }
}

// R = P^T: each coarse cell sums the fine cells it covers, in x-major order:
// eight, or one where the block has the same resolution on both levels (it
// bottomed out at one cell per block) (mr_multigrid.py:92-99)
__global__ __launch_bounds__(256) void k_msbg_restrict(MGrid fg, MGrid cg, const float* __restrict__ rfine,
                                                       float* __restrict__ bcoarse) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= cg.ncells) return;
    const int4 o = origin(cg, a);
    const MCell f0 = locate(fg, o.x, o.y, o.z);
    float acc = 0.0f;
    if (f0.level == o.w) {
        acc = rfine[f0.addr];
    } else {
        const int hf = 1 << f0.level;
        for (int x = 0; x < 2; ++x)
            for (int y = 0; y < 2; ++y)
                for (int z = 0; z < 2; ++z)
                    acc += rfine[locate(fg, o.x + x * hf, o.y + y * hf, o.z + z * hf).addr];
    }
    bcoarse[a] = acc;
}

// P: piecewise-constant injection added onto the fine level (mr_multigrid.py:102-109)
__global__ __launch_bounds__(256) void k_msbg_prolong_add(MGrid fg, MGrid cg, const float* __restrict__ pcoarse,
                                                          float* __restrict__ pfine) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= fg.ncells) return;
    const int4 o = origin(fg, a);
    pfine[a] += pcoarse[locate(cg, o.x, o.y, o.z).addr];
}

// cell centre, volume and whether all six neighbours exist
// (msbg.py:144-153, mr_operator.py:215-220)
__global__ __launch_bounds__(256) void k_msbg_geometry(MGrid g, float* __restrict__ centre, float* __restrict__ vol,
                                                       int* __restrict__ interior) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= g.ncells) return;
    const int4 o = origin(g, a);
    const int ext = 1 << o.w;
    const float half = (float)ext * 0.5f;
    if (centre) {
        centre[3 * a] = ((float)o.x + half) * g.h0;
        centre[3 * a + 1] = ((float)o.y + half) * g.h0;
        centre[3 * a + 2] = ((float)o.z + half) * g.h0;
    }
    if (vol) {
        const float h = g.h0 * (float)ext;
        vol[a] = h * h * h;
    }
    if (interior) {
        int ok = 1;
        for (int axis = 0; axis < 3; ++axis) {
            const int ex = comp(axis, 0), ey = comp(axis, 1), ez = comp(axis, 2);
            if (locate(g, o.x - ex, o.y - ey, o.z - ez).addr < 0) ok = 0;
            if (locate(g, o.x + ex * ext, o.y + ey * ext, o.z + ez * ext).addr < 0) ok = 0;
        }
        interior[a] = ok;
    }
}

// hits[c] = number of finest coordinates that resolve to cell c
__global__ __launch_bounds__(256) void k_msbg_cover(MGrid g, int* __restrict__ hits) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int fz_n = g.nbz << g.sh0, fy_n = g.nby << g.sh0, fx_n = g.nbx << g.sh0;
    if (t >= (int64_t)fx_n * fy_n * fz_n) return;
    const int fz = (int)(t % fz_n), fy = (int)((t / fz_n) % fy_n), fx = (int)(t / ((int64_t)fz_n * fy_n));
    const MCell c = locate(g, fx, fy, fz);
    if (c.addr >= 0) atomicAdd(hits + c.addr, 1);
}

constexpr int kVecBlocks = 1024;

// FP64 partial sums over blocks, combined in block order by one block
__global__ __launch_bounds__(256) void k_vec_part(int op, const float* __restrict__ x, const float* __restrict__ y,
                                                  int64_t n, double* __restrict__ part) {
    __shared__ double sh[16];
    double v[1] = {0.0};
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        if (op == 0)
            v[0] += (double)x[i];
        else if (op == 1)
            v[0] += (double)x[i] * (double)y[i];
        else
            v[0] = fmax(v[0], fabs((double)x[i]));
    }
    if (op == 2) {
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
        double m = v[0];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
        if (lane == 0) sh[wid] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            double r = sh[0];
            for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = fmax(r, sh[w]);
            part[blockIdx.x] = r;
        }
        return;
    }
    block_sum<1>(v, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = v[0];
}

// one wave combines the partials: lane t takes t, t + 64, ... in order,
// then a fixed butterfly
__global__ __launch_bounds__(64) void k_vec_comb(int op, const double* __restrict__ part, int np,
                                                 double* __restrict__ out) {
    double r = 0.0;
    for (int b = threadIdx.x; b < np; b += 64) r = op == 2 ? fmax(r, part[b]) : r + part[b];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double t = __shfl_xor(r, o, 64);
        r = op == 2 ? fmax(r, t) : r + t;
    }
    if (threadIdx.x == 0) *out = r;
}

// y = a x + b y (x may be NULL: y = b y + a)
__global__ __launch_bounds__(256) void k_vec_axpby(float a, const float* __restrict__ x, float b, float* __restrict__ y,
                                                   int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = x ? a * x[i] + b * y[i] : b * y[i] + a;
}

// y = a x + b y with a = a_sign * st[ia] and b = st[ib] (or 1 when ib < 0)
// rounded to float, the scalars of the flexible PCG kept on the device; a
// no-op once flag[0] is set
__global__ __launch_bounds__(256) void k_vec_axpby_dev(const double* __restrict__ st, int ia, float a_sign,
                                                       const float* __restrict__ x, int ib,
                                                       float* __restrict__ y, int64_t n,
                                                       const int* __restrict__ flag) {
    if (flag && flag[0]) return;
    const float a = ia >= 0 ? (float)((double)a_sign * st[ia]) : a_sign;
    const float b = ib >= 0 ? (float)st[ib] : 1.0f;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = a * x[i] + b * y[i];
}

// y = 1 y + (float)(-sum / n): the mean removal of mr_multigrid.py:181-184
// with the sum left on the device by pf_vec_reduce
__global__ __launch_bounds__(256) void k_vec_sub_mean(float* __restrict__ y, int64_t n,
                                                      const double* __restrict__ sum) {
    const float a = (float)(-*sum / (double)n);
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = 1.0f * y[i] + a;
}

// The scalar steps of the flexible Polak-Ribiere PCG (mr_solver.py:118-165)
// on one thread.  st: 0 rz, 1 alpha, 2 beta, 3 rel, 4 bnorm, 5 tol, 6 qAq,
// 7 a copy of flag[0]; flag[0]: 0 running, 1 stopped at qAq <= 0, 2 converged, 3 stopped at
// rz == 0 or rz_new <= 0.
enum MrcgOp { MRCG_INIT = 0, MRCG_RZ, MRCG_ALPHA, MRCG_REL, MRCG_BETA };

__device__ inline void mrcg_scalar(int op, double* st, int* flag, const double* a, const double* b, double tol) {
    if (op == MRCG_INIT) {  // a = max|b|
        st[4] = *a;
        st[5] = tol;
        st[3] = 1.0;
        flag[0] = 0;
    } else if (op == MRCG_RZ) {
        st[0] = *a;
    } else if (flag[0]) {
        // stopped: the scalars keep their values
    } else if (op == MRCG_ALPHA) {
        st[6] = *a;
        if (*a <= 0.0)
            flag[0] = 1;
        else
            st[1] = st[0] / *a;
    } else if (op == MRCG_REL) {
        st[3] = *a / st[4];
        if (st[3] < st[5]) flag[0] = 2;
    } else if (op == MRCG_BETA) {  // a = <r, z>, b = <r_prev, z>
        const double rz_new = *a;
        if (st[0] == 0.0 || rz_new <= 0.0) {
            flag[0] = 3;
        } else {
            st[2] = fmax((rz_new - *b) / st[0], 0.0);
            st[0] = rz_new;
        }
    }
    st[7] = (double)flag[0];  // the host reads st[0..7] in one copy
}

__global__ void k_mrcg_scalar(int op, double* st, int* flag, const double* a, const double* b, double tol) {
    if (threadIdx.x == 0 && blockIdx.x == 0) mrcg_scalar(op, st, flag, a, b, tol);
}

// One PCG iteration's vector work in five launches (twenty when every vector
// operation, reduction and scalar step had its own; at 32k cells each costs its
// launch, at 1.4M a pass over memory: adaptive 32^3 step 2.26 -> 1.95 ms, 128^3
// 7.83 -> 7.60).  A reduction's partials stay in
// its work buffer (work + 1, kVecBlocks entries, those past the launch's blocks
// zero) and every block of the next kernel combines them anew, in the order of
// k_vec_comb; block 0 leaves the scalars in st.  A block reads no entry of st
// that block 0 of the same launch writes, but the flag: both of its values
// lead a block to the same decision.
__device__ inline double comb_parts(int op, const double* __restrict__ part) {
    __shared__ double total;
    __syncthreads();
    if (threadIdx.x < 64) {
        double x[kVecBlocks / 64], r = 0.0;
#pragma unroll
        for (int q = 0; q < kVecBlocks / 64; ++q) x[q] = part[q * 64 + threadIdx.x];
#pragma unroll
        for (int q = 0; q < kVecBlocks / 64; ++q) r = op == 2 ? fmax(r, x[q]) : r + x[q];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const double t = __shfl_xor(r, o, 64);
            r = op == 2 ? fmax(r, t) : r + t;
        }
        if (threadIdx.x == 0) total = r;
    }
    __syncthreads();
    return total;
}

// alpha = rz / <q, Ap>; x += alpha q, r_prev = r, r -= alpha Ap, and the
// partials of max |r|.  rz: slot of st that holds it.
__global__ __launch_bounds__(256) void k_mrcg_update(double* st, int* flag, int rz, const double* __restrict__ qap,
                                                     const float* __restrict__ q, const float* __restrict__ ap,
                                                     float* __restrict__ x, float* __restrict__ r,
                                                     float* __restrict__ r_prev, int64_t n,
                                                     double* __restrict__ rmax) {
    __shared__ float sh[4];
    const double d = comb_parts(1, qap);
    const bool go = flag[0] == 0 && !(d <= 0.0);
    const double al = go ? st[rz] / d : 0.0;
    const float a = (float)al, am = (float)-al;
    float m = 0.0f;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        float ri = r[i];
        r_prev[i] = ri;
        if (go) {
            x[i] = __fmaf_rn(a, q[i], x[i]);
            ri = __fmaf_rn(am, ap[i], ri);
            r[i] = ri;
        }
        m = fmaxf(m, fabsf(ri));
    }
    m = block_max(m, sh);
    if (threadIdx.x == 0) rmax[blockIdx.x] = (double)m;
    if (blockIdx.x == 0 && threadIdx.x == 0 && flag[0] == 0) {
        st[6] = d;
        if (go)
            st[1] = al;
        else
            flag[0] = 1;
    }
}

// rel = max |r| / |b|, convergence, and the flag where the host reads it
__global__ __launch_bounds__(64) void k_mrcg_rel(double* st, int* flag, const double* __restrict__ rmax) {
    const double m = comb_parts(2, rmax);
    if (threadIdx.x == 0) mrcg_scalar(MRCG_REL, st, flag, &m, nullptr, 0.0);
}

// z = y - mean(y) from the partials of its sum, and the partials of <r, z>
// and <r_prev, z>
__global__ __launch_bounds__(256) void k_mrcg_z(const float* y, float* z, int64_t n,
                                                const double* __restrict__ sum, const float* __restrict__ r,
                                                const float* __restrict__ r_prev, double* __restrict__ rz,
                                                double* __restrict__ rpz) {
    __shared__ double sh[2 * 16];
    const float a = (float)(-comb_parts(0, sum) / (double)n);
    double v[2] = {0.0, 0.0};
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const float zi = 1.0f * y[i] + a;
        z[i] = zi;
        v[0] += (double)r[i] * (double)zi;
        v[1] += (double)r_prev[i] * (double)zi;
    }
    block_sum<2>(v, sh);
    if (threadIdx.x == 0) {
        rz[blockIdx.x] = v[0];
        rpz[blockIdx.x] = v[1];
    }
}

// beta = max((<r, z> - <r_prev, z>) / rz, 0), q = z + beta q; the new rz goes
// to the other slot, since every block reads the old one
__global__ __launch_bounds__(256) void k_mrcg_q(double* st, int* flag, int rz, int rz_next,
                                                const double* __restrict__ rzp, const double* __restrict__ rpzp,
                                                const float* __restrict__ z, float* __restrict__ q, int64_t n) {
    const double rz_new = comb_parts(1, rzp), rpz = comb_parts(1, rpzp), old = st[rz];
    const bool go = flag[0] == 0 && !(old == 0.0 || rz_new <= 0.0);
    const double beta = go ? fmax((rz_new - rpz) / old, 0.0) : 0.0;
    if (go) {
        const float b = (float)beta;
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
#pragma clang fp contract(off)
            const float t = b * q[i];  // rounded, as in k_vec_axpby_dev
            q[i] = z[i] + t;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (go) {
            st[2] = beta;
            st[rz_next] = rz_new;
        } else if (flag[0] == 0) {
            flag[0] = 3;
        }
        st[7] = (double)flag[0];
    }
}

// x -= mean(x) in one workgroup, for a coarsest level
constexpr int kMeanSmallMax = 4096;

__global__ __launch_bounds__(1024) void k_vec_remove_mean_small(float* __restrict__ x, int n,
                                                               double* __restrict__ sum) {
    __shared__ double sh[16];
    __shared__ float shift;
    float v[kMeanSmallMax / 1024];
    double s[1] = {0.0};
#pragma unroll
    for (int q = 0; q < kMeanSmallMax / 1024; ++q) {
        const int i = q * 1024 + (int)threadIdx.x;
        v[q] = i < n ? x[i] : 0.0f;
        s[0] += (double)v[q];
    }
    block_sum<1>(s, sh);
    if (threadIdx.x == 0) {
        *sum = s[0];
        shift = (float)(-s[0] / (double)n);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kMeanSmallMax / 1024; ++q) {
        const int i = q * 1024 + (int)threadIdx.x;
        if (i < n) x[i] = 1.0f * v[q] + shift;
    }
}

// z = r / diag where diag > 0, else 0 (mr_solver.py:64-69)
__global__ __launch_bounds__(256) void k_vec_jacobi(const float* __restrict__ r, const float* __restrict__ diag,
                                                    float* __restrict__ z, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float d = diag[i];
        z[i] = d > 0.0f ? r[i] / d : 0.0f;
    }
}

// ------------------------------------------------------------------ stored rows
// The couplings of every cell as a table, built once per set of face
// coefficients.  Walking the block structure is a chain of five dependent
// loads (cell -> block -> neighbour block -> its offset -> value) and some 300
// instructions per cell, and a solve does it 24 times per level and V-cycle
// with the same result; from the table it is one load and one gather.
// Per half-sweep: 1.4M cells 19.0 -> 12.1 us (bound by reading 48 bytes of rows
// per cell, 5 TB/s in all), 205k 8.4 -> 4.1, 32k 6.6 -> 3.1, 25k 8.1 -> 3.5
// (bound by the launch); A p at 1.4M cells 28 -> 17.6 us; the table takes 48 us
// there and 8 at 32k cells.
//
// Cells 2t and 2t + 1 form pair t.  A pair with one cell of each colour keeps
// its colour-c row at position c H + t (H pairs), so that a half-sweep reads
// its colour's half of the table only, without gaps; any other pair keeps cell
// 2t + s at s H + t.  A row's first kRowIn couplings stand in `in` (entry k of
// all positions is contiguous); rows with more (a cell facing finer ones) are
// marked by bit 31 of the last and keep the rest in `more`, in order of arrival
// (which changes no result).  A coarse cell has 3 couplings more than faces for
// each finer block it faces, however much finer (always a 2x2 patch), and a
// block of (2 m)^3 cells is faced by at most 6 m^2 coarser cells, so 18 m^2 <=
// 9/4 (2 m)^3 bounds `more` for any map of levels, graded 2:1 or not (the
// largest share, on blocks of 2^3 cells between blocks of one).  Same
// couplings, same order and same arithmetic as the kernels without the table.
constexpr int kRowIn = 6;

struct MRows {
    int2* in;    // [kRowIn][2 H] (coefficient bits, neighbour)
    int2* more;  // [cap], cap = 9/4 of the cells
    int2* ext;   // [2 H] (first of `more`, count); set for marked rows
    float* d;    // [2 H] sum of the couplings
    unsigned* used;  // of `more`
    uint8_t* code;  // [H] colours of cells 2t (bit 0) and 2t + 1 (bit 1)
    int H;
    unsigned cap;
};

inline size_t mrows_layout(int ncells, char* base, MRows* r) {
    const size_t H = ((size_t)ncells + 1) / 2, cap = (size_t)ncells * 9 / 4;
    size_t o = 0;
    const auto take = [&](size_t bytes) {
        char* q = base ? base + o : nullptr;
        o += (bytes + 15) & ~(size_t)15;
        return q;
    };
    MRows m;
    m.in = reinterpret_cast<int2*>(take(kRowIn * 2 * H * sizeof(int2)));
    m.more = reinterpret_cast<int2*>(take(cap * sizeof(int2)));
    m.ext = reinterpret_cast<int2*>(take(2 * H * sizeof(int2)));
    m.d = reinterpret_cast<float*>(take(2 * H * sizeof(float)));
    m.used = reinterpret_cast<unsigned*>(take(sizeof(unsigned)));
    m.code = reinterpret_cast<uint8_t*>(take(H));
    m.H = (int)H;
    m.cap = (unsigned)cap;
    if (r) *r = m;
    return o;
}

__device__ inline int cell_colour(const int4 o) { return ((o.x >> o.w) + (o.y >> o.w) + (o.z >> o.w)) & 1; }

// position of cell 2t + s
__device__ inline int row_pos(int code, int s, int t, int H) {
    const int half = (code == 1 || code == 2) ? ((code >> s) & 1) : s;
    return half * H + t;
}

__global__ __launch_bounds__(256) void k_msbg_rows(MGrid g, const float* __restrict__ bface, MRows r,
                                                   float* __restrict__ diag) {
    const int a = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (a >= g.ncells) return;
    BlockRef br;
    const int4 o = origin_ref(g, a, br);
    const int t = a >> 1, s = a & 1, c = cell_colour(o);
    // (the missing partner of an odd last cell counts as the other colour)
    const int cp = (a ^ 1) < g.ncells ? cell_colour(origin(g, a ^ 1)) : 1 - c;
    const int code = s ? (cp | (c << 1)) : (c | (cp << 1));
    const int pos = row_pos(code, s, t, r.H);
    if (s == 0) r.code[t] = (uint8_t)code;
    const size_t W = 2 * (size_t)r.H;
    int k = 0;
    int2 last = make_int2(0, a);
    float sum = 0.0f;
    for_each_coupling_from(g, bface, a, o, br, [&](int nb, float w) {
        sum += w;
        if (k < kRowIn) {
            last = make_int2(__float_as_int(w), nb);
            if (k < kRowIn - 1) r.in[k * W + pos] = last;
        }
        ++k;
    });
    diag[a] = sum;
    r.d[pos] = sum;
    for (int q = k; q < kRowIn - 1; ++q) r.in[q * W + pos] = make_int2(0, a);
    if (k < kRowIn) last = make_int2(0, a);
    if (k > kRowIn) {
        const unsigned cnt = k - kRowIn, at = atomicAdd(r.used, cnt);
        if (at + cnt <= r.cap) {
            r.ext[pos] = make_int2((int)at, (int)cnt);
            last.y |= (int)0x80000000;
            k = 0;
            for_each_coupling_from(g, bface, a, o, br, [&](int nb, float w) {
                if (k >= kRowIn) r.more[at + k - kRowIn] = make_int2(__float_as_int(w), nb);
                ++k;
            });
        }
    }
    r.in[(kRowIn - 1) * W + pos] = last;
}

// the couplings past the first kRowIn added to acc
template <class V>
__device__ inline float row_rest(const MRows& r, int pos, float pa, const V* p, float acc) {
    const int2 e = r.ext[pos];
    for (int q = 0; q < e.y; ++q) {
        const int2 m = r.more[e.x + q];
        acc += __int_as_float(m.x) * (pa - p[m.y]);
    }
    return acc;
}

// sum_f T_f (p_A - p_B) of cell a at position pos
__device__ inline float row_acc(const MRows& r, int pos, float pa, const float* __restrict__ p) {
    const size_t W = 2 * (size_t)r.H;
    int2 e[kRowIn];
#pragma unroll
    for (int k = 0; k < kRowIn; ++k) e[k] = r.in[k * W + pos];
    const bool rest = e[kRowIn - 1].y < 0;
    e[kRowIn - 1].y &= 0x7fffffff;
    float q[kRowIn];
#pragma unroll
    for (int k = 0; k < kRowIn; ++k) q[k] = p[e[k].y];
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < kRowIn; ++k) acc += __int_as_float(e[k].x) * (pa - q[k]);
    if (rest) acc = row_rest(r, pos, pa, p, acc);
    return acc;
}

// One half-sweep, a pair per thread; ZERO: pin is all zeros and not read (the
// first half-sweep of a V-cycle level).
template <bool ZERO>
__global__ __launch_bounds__(256) void k_msbg_rows_sweep(MRows r, int n, const float* __restrict__ pin,
                                                         float* __restrict__ pout, const float* __restrict__ b,
                                                         int colour, float omega) {
    const int t = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (t >= r.H) return;
    const int code = r.code[t];
    const bool two = 2 * t + 1 < n;
    float v[2] = {0.0f, 0.0f};
    if (!ZERO) {
        if (two) {
            const float2 w = reinterpret_cast<const float2*>(pin)[t];
            v[0] = w.x;
            v[1] = w.y;
        } else {
            v[0] = pin[2 * t];
        }
    }
    const auto update = [&](int s, int pos, float x) {
        const int a = 2 * t + s;
        const float d = r.d[pos];
        if (d > 0.0f) x = x + omega * (b[a] - (ZERO ? 0.0f : row_acc(r, pos, x, pin))) / d;
        return x;
    };
    if (code == 1 || code == 2) {  // one of each colour
        const int s = (code & 1) == colour ? 0 : 1;
        if (s == 0 || two) {
            const float x = update(s, colour * r.H + t, s ? v[1] : v[0]);
            v[0] = s ? v[0] : x;
            v[1] = s ? x : v[1];
        }
    } else if ((code & 1) == colour) {
        v[0] = update(0, t, v[0]);
        v[1] = update(1, r.H + t, v[1]);  // (the missing partner makes a pair of two colours)
    }
    if (two)
        reinterpret_cast<float2*>(pout)[t] = make_float2(v[0], v[1]);
    else
        pout[2 * t] = v[0];
}

// All half-sweeps of a smoothing phase in one workgroup, for a level of up to
// 2048 PP cells: rows in registers, the iterate and b in LDS.  New values are
// held until every thread has read the old ones.  Three sweeps: 11.7 us at
// 4096 cells (15.5 with rows past six couplings, whose rest is read from
// memory each time), of which the loads take half; six launches take 19.  Four
// pairs per thread do not fit the registers, hence the limit.
constexpr int kRowsSmallThreads = 1024;
constexpr int kRowsSmallMax = 4096;

template <int PP>
__global__ __launch_bounds__(kRowsSmallThreads) void k_msbg_rows_small(MRows r, int n, float* __restrict__ p,
                                                                       const float* __restrict__ b, int sweeps,
                                                                       int first, int zero, float omega) {
    __shared__ float x[2048 * PP], bb[2048 * PP];
    const size_t W = 2 * (size_t)r.H;
    float w[PP][2][kRowIn], dd[PP][2];
    unsigned nb[PP][2][kRowIn / 2];
    int code[PP];
    unsigned rest = 0;
#pragma unroll
    for (int m = 0; m < PP; ++m) {
        const int t = (int)threadIdx.x + m * kRowsSmallThreads;
        code[m] = 4;  // no pair here
        if (t < r.H) {
            code[m] = r.code[t];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int a = 2 * t + h, pos = h * r.H + t;
                // (an odd last cell's partner has no row)
                const bool has = 2 * t + 1 < n || h == (code[m] & 1);
                dd[m][h] = has ? r.d[pos] : 0.0f;
                int2 e[kRowIn];
#pragma unroll
                for (int k = 0; k < kRowIn; ++k) e[k] = has ? r.in[k * W + pos] : make_int2(0, 0);
                if (e[kRowIn - 1].y < 0) rest |= 1u << (2 * m + h);
#pragma unroll
                for (int k = 0; k < kRowIn; ++k) w[m][h][k] = __int_as_float(e[k].x);
#pragma unroll
                for (int k = 0; k < kRowIn; k += 2)
                    nb[m][h][k / 2] = (unsigned)(e[k].y & 0x7fff) | ((unsigned)(e[k + 1].y & 0x7fff) << 16);
                x[a] = zero || a >= n ? 0.0f : p[a];
                bb[a] = a < n ? b[a] : 0.0f;
            }
        }
    }
    __syncthreads();
    for (int hs = 0; hs < 2 * sweeps; ++hs) {
        const int colour = (hs & 1) ^ first;
        float nv[PP][2];
        int at[PP][2];
#pragma unroll
        for (int m = 0; m < PP; ++m) {
            const int t = (int)threadIdx.x + m * kRowsSmallThreads;
            const bool mixed = code[m] == 1 || code[m] == 2;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                // row h: the cell of colour h, or cell 2t + h
                at[m][h] = -1;
                const bool on = mixed ? h == colour : (code[m] != 4 && (code[m] & 1) == colour);
                if (on && dd[m][h] > 0.0f) {
                    const int s = mixed ? ((code[m] & 1) == h ? 0 : 1) : h;
                    const int a = 2 * t + s;
                    const float pa = x[a];
                    float acc = 0.0f;
#pragma unroll
                    for (int k = 0; k < kRowIn; ++k) {
                        const unsigned q = nb[m][h][k / 2];
                        acc += w[m][h][k] * (pa - x[k & 1 ? q >> 16 : q & 0xffffu]);
                    }
                    if (rest >> (2 * m + h) & 1) acc = row_rest(r, h * r.H + t, pa, x, acc);
                    nv[m][h] = pa + omega * (bb[a] - acc) / dd[m][h];
                    at[m][h] = a;
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < PP; ++m)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (at[m][h] >= 0) x[at[m][h]] = nv[m][h];
        __syncthreads();
    }
    for (int a = threadIdx.x; a < n; a += kRowsSmallThreads) p[a] = x[a];
}

// out = A p, or b - A p, a pair per thread (twelve row loads in flight); DOT:
// part[block] = the block's share of <p, out> too.  At 1.4M cells 18.4 us, 22.6
// with the product (28 + 9 from the blocks and in three launches): 84 MB.
template <bool DOT>
__global__ __launch_bounds__(256) void k_msbg_rows_apply(MRows r, int n, const float* __restrict__ p,
                                                         const float* __restrict__ b, float* __restrict__ out,
                                                         double* __restrict__ part) {
    __shared__ double sh[16];
    double v[1] = {0.0};
    const int nb = (r.H + 255) / 256;
    for (int q = xcd_block(blockIdx.x, gridDim.x); q < nb; q += gridDim.x) {
        const int t = q * 256 + (int)threadIdx.x;
        if (t >= r.H) continue;
        const int code = r.code[t], a = 2 * t;
        const bool two = a + 1 < n, swap = code == 1;  // (the row at t is cell a + 1's)
        const float p0 = p[a], p1 = two ? p[a + 1] : 0.0f;
        const float lo = two || !swap ? row_acc(r, t, swap ? p1 : p0, p) : 0.0f;
        const float hi = two || swap ? row_acc(r, r.H + t, swap ? p0 : p1, p) : 0.0f;
        const float y0 = swap ? hi : lo, y1 = swap ? lo : hi;
        out[a] = b ? b[a] - y0 : y0;
        if (two) out[a + 1] = b ? b[a + 1] - y1 : y1;
        if (DOT) {
            v[0] += (double)p0 * (double)y0;
            if (two) v[0] += (double)p1 * (double)y1;
        }
    }
    if (DOT) {
        block_sum<1>(v, sh);
        if (threadIdx.x == 0) part[blockIdx.x] = v[0];
    }
}

}  // namespace pf

using namespace pf;

static int check_grid(const pf_msbg_grid* g, const char* who) {
    PF_REQUIRE(g, "%s: null grid", who);
    PF_REQUIRE(g->ncells > 0 && g->nslots > 0 && g->n0 == (1 << g->sh0) && g->h0 > 0.f, "%s: bad grid", who);
    PF_REQUIRE(g->level && g->slot && g->blk && g->blev && g->coff && g->cslot, "%s: null grid array", who);
    // face fields are indexed 3 * cell + axis in 32-bit arithmetic
    PF_REQUIRE(g->ncells <= kMsbgMaxCells, "%s: %d cells exceed the limit of %d", who, g->ncells, kMsbgMaxCells);
    return PF_OK;
}

PF_API int pf_msbg_apply(const pf_msbg_grid* g, const float* p, const float* bface, float* out, int32_t want_diag,
                         pf_stream_t stream) {
    int rc = check_grid(g, "pf_msbg_apply");
    if (rc) return rc;
    PF_REQUIRE(bface && out && (want_diag || p), "pf_msbg_apply: null vector");
    k_msbg_apply<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), p, bface, out, want_diag);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_residual(const pf_msbg_grid* g, const float* p, const float* b, const float* bface, float* r,
                            pf_stream_t stream) {
    int rc = check_grid(g, "pf_msbg_residual");
    if (rc) return rc;
    PF_REQUIRE(p && b && bface && r, "pf_msbg_residual: null vector");
    k_msbg_residual<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), p, b, bface, r);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_rbgs(const pf_msbg_grid* g, const float* pin, float* pout, const float* b, const float* bface,
                        const float* diag, int32_t colour, float omega, pf_stream_t stream) {
    int rc = check_grid(g, "pf_msbg_rbgs");
    if (rc) return rc;
    PF_REQUIRE(pin && pout && b && bface && diag, "pf_msbg_rbgs: null vector");
    PF_REQUIRE(pin != pout, "pf_msbg_rbgs: pin and pout must be distinct");
    PF_REQUIRE(colour == 0 || colour == 1, "pf_msbg_rbgs: colour must be 0 or 1");
    if (g->ncells >= kMsbgPairMinCells && ((reinterpret_cast<uintptr_t>(pin) | reinterpret_cast<uintptr_t>(pout)) & 7) == 0)
        k_msbg_rbgs_pairs<<<cdiv(cdiv(g->ncells, 2), 256), 256, 0, S(stream)>>>(mgrid(*g), pin, pout, b, bface, diag,
                                                                               colour, omega);
    else
        k_msbg_rbgs<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), pin, pout, b, bface, diag, colour, omega);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_rbgs_active(const pf_msbg_grid* g, const float* pin, float* pout, const float* b,
                               const float* bface, const float* diag, const int32_t* active, int32_t colour,
                               float omega, float* delta, pf_stream_t stream) {
    int rc = check_grid(g, "pf_msbg_rbgs_active");
    if (rc) return rc;
    PF_REQUIRE(pin && pout && b && bface && diag && active && delta, "pf_msbg_rbgs_active: null vector");
    PF_REQUIRE(pin != pout, "pf_msbg_rbgs_active: pin and pout must be distinct");
    PF_REQUIRE(colour == 0 || colour == 1, "pf_msbg_rbgs_active: colour must be 0 or 1");
    if (g->ncells >= kMsbgPairMinCells && ((reinterpret_cast<uintptr_t>(pin) | reinterpret_cast<uintptr_t>(pout)) & 7) == 0)
        k_msbg_rbgs_active_pairs<<<cdiv(cdiv(g->ncells, 2), 256), 256, 0, S(stream)>>>(
            mgrid(*g), pin, pout, b, bface, diag, active, colour, omega, delta);
    else
        k_msbg_rbgs_active<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), pin, pout, b, bface, diag, active,
                                                                        colour, omega, delta);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_relax_update(const pf_msbg_grid* g, const float* delta, const float* diag, const int32_t* active,
                                float* res, float* theta, int32_t set_theta, float theta_sigma, int32_t* active_next,
                                pf_stream_t stream) {
    int rc = check_grid(g, "pf_msbg_relax_update");
    if (rc) return rc;
    PF_REQUIRE(delta && diag && active && res && theta && active_next, "pf_msbg_relax_update: null pointer");
    PF_REQUIRE(active_next != active, "pf_msbg_relax_update: active_next must be a separate buffer");
    k_msbg_block_res<<<g->nslots, 256, 0, S(stream)>>>(mgrid(*g), delta, diag, active, res);
    PF_CHECK_LAUNCH();
    if (set_theta) {
        k_msbg_theta<<<1, 256, 0, S(stream)>>>(res, g->nslots, theta_sigma, theta);
        PF_CHECK_LAUNCH();
    }
    rc = fill_u32(active_next, g->nslots, 0u, S(stream));
    if (rc) return rc;
    k_msbg_update_active<<<cdiv(g->nslots, 256), 256, 0, S(stream)>>>(mgrid(*g), res, theta, active_next);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int32_t pf_msbg_coarsest_max_cells(void) {
    int dev = 0, lim = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&lim, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) return 0;
    int n = (int)(lim / coarsest_lds_bytes(1));
    return n < 65536 ? n : 65535;  // neighbour indices are 16-bit
}

PF_API int pf_msbg_coarsest_smooth(const pf_msbg_grid* g, float* p, const float* b, const float* bface,
                                   const float* diag, int32_t sweeps, float omega, pf_stream_t stream) {
    int rc = check_grid(g, "pf_msbg_coarsest_smooth");
    if (rc) return rc;
    PF_REQUIRE(p && b && bface && diag && sweeps >= 0, "pf_msbg_coarsest_smooth: bad arguments");
    PF_REQUIRE(g->ncells <= pf_msbg_coarsest_max_cells(),
               "pf_msbg_coarsest_smooth: %d cells exceed the workgroup's LDS", g->ncells);
    const size_t bytes = coarsest_lds_bytes(g->ncells);
    if (bytes > 65536) {
        const hipError_t e = hipFuncSetAttribute((const void*)k_msbg_coarsest,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        PF_REQUIRE(e == hipSuccess, "pf_msbg_coarsest_smooth: cannot raise the LDS limit to %zu bytes", bytes);
    }
    k_msbg_coarsest<<<1, kCoarsestThreads, bytes, S(stream)>>>(mgrid(*g), p, b, bface, diag, sweeps, omega);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int32_t pf_msbg_coarse_op_max_cells(void) {
    int dev = 0, lim = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&lim, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) return 0;
    const int n = (int)(lim / coarse_op_lds_bytes(1));
    return n < kMsbgCoarseOpMax ? n : kMsbgCoarseOpMax;
}

PF_API int pf_msbg_coarse_op(const pf_msbg_grid* g, const float* bface, const float* diag, int32_t sweeps,
                             float omega, double* op, pf_stream_t stream) {
    int rc = check_grid(g, "pf_msbg_coarse_op");
    if (rc) return rc;
    PF_REQUIRE(bface && diag && op && sweeps >= 0, "pf_msbg_coarse_op: bad arguments");
    PF_REQUIRE(g->ncells <= pf_msbg_coarse_op_max_cells(), "pf_msbg_coarse_op: %d cells exceed the limit",
               g->ncells);
    static_assert(coarse_op_lds_bytes(kMsbgCoarseOpMax) <= 60 * 1024, "the default dynamic LDS limit");
    k_msbg_coarse_op<<<g->ncells, kCoarsestThreads, coarse_op_lds_bytes(g->ncells), S(stream)>>>(mgrid(*g), bface, diag, sweeps,
                                                                         (double)omega, op);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_coarse_apply(const double* op, const float* b, float* p, int32_t n, pf_stream_t stream) {
    PF_REQUIRE(op && b && p && n > 0 && n <= kMsbgCoarseOpMax, "pf_msbg_coarse_apply: bad arguments");
    k_msbg_coarse_apply<<<cdiv(n, kApplyRows), 1024, 0, S(stream)>>>(op, b, p, n);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API size_t pf_msbg_rows_bytes(int32_t ncells) {
    return ncells > 0 && ncells <= kMsbgMaxCells ? mrows_layout(ncells, nullptr, nullptr) : 0;
}

static int check_rows(const pf_msbg_grid* g, const void* rows, const char* who, MRows* r) {
    int rc = check_grid(g, who);
    if (rc) return rc;
    PF_REQUIRE(rows && (reinterpret_cast<uintptr_t>(rows) & 15) == 0, "%s: rows must be 16-byte aligned", who);
    mrows_layout(g->ncells, static_cast<char*>(const_cast<void*>(rows)), r);
    return PF_OK;
}

PF_API int pf_msbg_rows_build(const pf_msbg_grid* g, const float* bface, float* diag, void* rows,
                              pf_stream_t stream) {
    MRows r;
    int rc = check_rows(g, rows, "pf_msbg_rows_build", &r);
    if (rc) return rc;
    PF_REQUIRE(bface && diag, "pf_msbg_rows_build: null vector");
    rc = fill_u32(r.used, 1, 0u, S(stream));
    if (rc) return rc;
    k_msbg_rows<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), bface, r, diag);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_rows_smooth(const pf_msbg_grid* g, const void* rows, float* p, float* p2, const float* b,
                               int32_t sweeps, int32_t first_colour, int32_t from_zero, float omega,
                               pf_stream_t stream) {
    MRows r;
    int rc = check_rows(g, rows, "pf_msbg_rows_smooth", &r);
    if (rc) return rc;
    PF_REQUIRE(p && p2 && p != p2 && b, "pf_msbg_rows_smooth: null or equal vectors");
    PF_REQUIRE(((reinterpret_cast<uintptr_t>(p) | reinterpret_cast<uintptr_t>(p2)) & 7) == 0,
               "pf_msbg_rows_smooth: p and p2 must be 8-byte aligned");
    PF_REQUIRE(sweeps >= 0 && (first_colour == 0 || first_colour == 1), "pf_msbg_rows_smooth: bad sweeps or colour");
    if (sweeps == 0) return from_zero ? fill_u32(p, g->ncells, 0u, S(stream)) : PF_OK;
    if (g->ncells <= kRowsSmallMax) {
        const auto k = g->ncells <= 2048 ? k_msbg_rows_small<1> : k_msbg_rows_small<2>;
        k<<<1, kRowsSmallThreads, 0, S(stream)>>>(r, g->ncells, p, b, sweeps, first_colour, from_zero, omega);
        PF_CHECK_LAUNCH();
        return PF_OK;
    }
    const int nb = cdiv(r.H, 256);
    float *in = p, *out = p2;
    for (int h = 0; h < 2 * sweeps; ++h) {  // an even number: the result is in p
        const int c = (h & 1) ^ first_colour;
        if (h == 0 && from_zero)
            k_msbg_rows_sweep<true><<<nb, 256, 0, S(stream)>>>(r, g->ncells, in, out, b, c, omega);
        else
            k_msbg_rows_sweep<false><<<nb, 256, 0, S(stream)>>>(r, g->ncells, in, out, b, c, omega);
        PF_CHECK_LAUNCH();
        float* t = in;
        in = out;
        out = t;
    }
    return PF_OK;
}

PF_API int pf_msbg_rows_apply(const pf_msbg_grid* g, const void* rows, const float* p, const float* b, float* out,
                              pf_stream_t stream) {
    MRows r;
    int rc = check_rows(g, rows, "pf_msbg_rows_apply", &r);
    if (rc) return rc;
    PF_REQUIRE(p && out && out != p, "pf_msbg_rows_apply: null vector, or p == out");
    k_msbg_rows_apply<false><<<cdiv(r.H, 256), 256, 0, S(stream)>>>(r, g->ncells, p, b, out, nullptr);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_rows_apply_dot(const pf_msbg_grid* g, const void* rows, const float* p, float* out, double* work,
                                  pf_stream_t stream) {
    MRows r;
    int rc = check_rows(g, rows, "pf_msbg_rows_apply_dot", &r);
    if (rc) return rc;
    PF_REQUIRE(p && out && out != p && work, "pf_msbg_rows_apply_dot: null vector, or p == out");
    const int nb = cdiv(r.H, 256);
    k_msbg_rows_apply<true><<<nb < kVecBlocks ? nb : kVecBlocks, 256, 0, S(stream)>>>(r, g->ncells, p, nullptr, out,
                                                                                   work + 1);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_coarsen_beta(const pf_msbg_grid* cg, const pf_msbg_grid* fg, const float* bfine, float* bcoarse,
                                pf_stream_t stream) {
    int rc = check_grid(cg, "pf_msbg_coarsen_beta");
    if (rc) return rc;
    rc = check_grid(fg, "pf_msbg_coarsen_beta");
    if (rc) return rc;
    PF_REQUIRE(bfine && bcoarse, "pf_msbg_coarsen_beta: null vector");
    k_msbg_coarsen_beta<<<cdiv(cg->ncells, 256), 256, 0, S(stream)>>>(mgrid(*cg), mgrid(*fg), bfine, bcoarse);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_restrict(const pf_msbg_grid* fg, const pf_msbg_grid* cg, const float* rfine, float* bcoarse,
                            pf_stream_t stream) {
    int rc = check_grid(fg, "pf_msbg_restrict");
    if (rc) return rc;
    rc = check_grid(cg, "pf_msbg_restrict");
    if (rc) return rc;
    PF_REQUIRE(rfine && bcoarse, "pf_msbg_restrict: null vector");
    k_msbg_restrict<<<cdiv(cg->ncells, 256), 256, 0, S(stream)>>>(mgrid(*fg), mgrid(*cg), rfine, bcoarse);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_prolong_add(const pf_msbg_grid* fg, const pf_msbg_grid* cg, const float* pcoarse, float* pfine,
                               pf_stream_t stream) {
    int rc = check_grid(fg, "pf_msbg_prolong_add");
    if (rc) return rc;
    rc = check_grid(cg, "pf_msbg_prolong_add");
    if (rc) return rc;
    PF_REQUIRE(pcoarse && pfine, "pf_msbg_prolong_add: null vector");
    k_msbg_prolong_add<<<cdiv(fg->ncells, 256), 256, 0, S(stream)>>>(mgrid(*fg), mgrid(*cg), pcoarse, pfine);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_geometry(const pf_msbg_grid* g, float* centre, float* volume, int32_t* interior,
                            pf_stream_t stream) {
    int rc = check_grid(g, "pf_msbg_geometry");
    if (rc) return rc;
    k_msbg_geometry<<<cdiv(g->ncells, 256), 256, 0, S(stream)>>>(mgrid(*g), centre, volume, interior);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_msbg_cover(const pf_msbg_grid* g, int32_t* hits, pf_stream_t stream) {
    int rc = check_grid(g, "pf_msbg_cover");
    if (rc) return rc;
    PF_REQUIRE(hits, "pf_msbg_cover: null hits");
    const int64_t nf = ((int64_t)g->nbx << g->sh0) * ((int64_t)g->nby << g->sh0) * ((int64_t)g->nbz << g->sh0);
    PF_REQUIRE(nf < ((int64_t)1 << 31), "pf_msbg_cover: too many finest cells");
    rc = fill_u32(hits, g->ncells, 0u, S(stream));
    if (rc) return rc;
    k_msbg_cover<<<cdiv(nf, 256), 256, 0, S(stream)>>>(mgrid(*g), hits);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API size_t pf_vec_reduce_bytes(void) { return (size_t)(kVecBlocks + 1) * sizeof(double); }

PF_API int pf_vec_reduce(int32_t op, const float* x, const float* y, int64_t n, double* work, pf_stream_t stream) {
    PF_REQUIRE(op >= 0 && op <= 2, "pf_vec_reduce: op must be 0 (sum), 1 (dot) or 2 (max |x|)");
    PF_REQUIRE(x && work && (op != 1 || y), "pf_vec_reduce: null vector");
    PF_REQUIRE(n > 0, "pf_vec_reduce: empty vector");
    const int64_t nb64 = cdiv(n, 256 * 4);
    const int nb = (int)(nb64 < kVecBlocks ? nb64 : kVecBlocks);
    k_vec_part<<<nb, 256, 0, S(stream)>>>(op, x, y, n, work + 1);
    PF_CHECK_LAUNCH();
    k_vec_comb<<<1, 64, 0, S(stream)>>>(op, work + 1, nb, work);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_vec_axpby(float a, const float* x, float b, float* y, int64_t n, pf_stream_t stream) {
    PF_REQUIRE(y && n > 0, "pf_vec_axpby: null or empty y");
    const int64_t nb64 = cdiv(n, 256 * 4);
    const int nb = (int)(nb64 < kVecBlocks ? nb64 : kVecBlocks);
    k_vec_axpby<<<nb, 256, 0, S(stream)>>>(a, x, b, y, n);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_vec_axpby_dev(const double* st, int32_t ia, float a_sign, const float* x, int32_t ib, float* y,
                            int64_t n, const int32_t* flag, pf_stream_t stream) {
    PF_REQUIRE(st && x && y && n > 0, "pf_vec_axpby_dev: null or empty vector");
    PF_REQUIRE(ia < 8 && ib < 8, "pf_vec_axpby_dev: scalar slot out of range");
    const int64_t nb64 = cdiv(n, 256 * 4);
    const int nb = (int)(nb64 < kVecBlocks ? nb64 : kVecBlocks);
    k_vec_axpby_dev<<<nb, 256, 0, S(stream)>>>(st, ia, a_sign, x, ib, y, n, flag);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_vec_remove_mean(float* x, int64_t n, double* work, pf_stream_t stream) {
    PF_REQUIRE(x && work && n > 0, "pf_vec_remove_mean: null or empty vector");
    if (n <= kMeanSmallMax) {
        k_vec_remove_mean_small<<<1, 1024, 0, S(stream)>>>(x, (int)n, work);
        PF_CHECK_LAUNCH();
        return PF_OK;
    }
    int rc = pf_vec_reduce(0, x, nullptr, n, work, stream);
    if (rc) return rc;
    const int64_t nb64 = cdiv(n, 256 * 4);
    const int nb = (int)(nb64 < kVecBlocks ? nb64 : kVecBlocks);
    k_vec_sub_mean<<<nb, 256, 0, S(stream)>>>(x, n, work);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mrcg_scalar(int32_t op, double* st, int32_t* flag, const double* a, const double* b, double tol,
                          pf_stream_t stream) {
    PF_REQUIRE(st && flag && (op < MRCG_ALPHA || a), "pf_mrcg_scalar: null pointer");
    PF_REQUIRE(op >= MRCG_INIT && op <= MRCG_BETA && (op != MRCG_BETA || b) && (op > MRCG_RZ || a),
               "pf_mrcg_scalar: bad op");
    k_mrcg_scalar<<<1, 64, 0, S(stream)>>>(op, st, flag, a, b, tol);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_vec_jacobi(const float* r, const float* diag, float* z, int64_t n, pf_stream_t stream) {
    PF_REQUIRE(r && diag && z && n > 0, "pf_vec_jacobi: null or empty vector");
    const int64_t nb64 = cdiv(n, 256 * 4);
    const int nb = (int)(nb64 < kVecBlocks ? nb64 : kVecBlocks);
    k_vec_jacobi<<<nb, 256, 0, S(stream)>>>(r, diag, z, n);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

static int vec_blocks(int64_t n) {
    const int64_t nb = cdiv(n, 256 * 4);
    return (int)(nb < kVecBlocks ? nb : kVecBlocks);
}

PF_API int pf_mrcg_update(double* st, int32_t* flag, int32_t rz, const double* qap, const float* q, const float* ap,
                          float* x, float* r, float* r_prev, int64_t n, double* rmax, pf_stream_t stream) {
    PF_REQUIRE(st && flag && qap && q && ap && x && r && r_prev && rmax && n > 0, "pf_mrcg_update: null or empty");
    PF_REQUIRE(rz == 0 || rz == 8, "pf_mrcg_update: rz is st[0] or st[8]");
    k_mrcg_update<<<vec_blocks(n), 256, 0, S(stream)>>>(st, flag, rz, qap + 1, q, ap, x, r, r_prev, n, rmax + 1);
    PF_CHECK_LAUNCH();
    k_mrcg_rel<<<1, 64, 0, S(stream)>>>(st, flag, rmax + 1);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

PF_API int pf_mrcg_direction(double* st, int32_t* flag, int32_t rz, const float* y, float* z, const float* r,
                             const float* r_prev, float* q, int64_t n, double* sum, double* rzw, double* rpzw,
                             pf_stream_t stream) {
    PF_REQUIRE(st && flag && y && z && r && r_prev && q && sum && rzw && rpzw && n > 0,
               "pf_mrcg_direction: null or empty");
    PF_REQUIRE(rz == 0 || rz == 8, "pf_mrcg_direction: rz is st[0] or st[8]");
    const int nb = vec_blocks(n);
    k_vec_part<<<nb, 256, 0, S(stream)>>>(0, y, nullptr, n, sum + 1);
    PF_CHECK_LAUNCH();
    k_mrcg_z<<<nb, 256, 0, S(stream)>>>(y, z, n, sum + 1, r, r_prev, rzw + 1, rpzw + 1);
    PF_CHECK_LAUNCH();
    k_mrcg_q<<<nb, 256, 0, S(stream)>>>(st, flag, rz, 8 - rz, rzw + 1, rpzw + 1, z, q, n);
    PF_CHECK_LAUNCH();
    return PF_OK;
}
