// Multigrid-preconditioned flexible CG for A p = b with
// (A p)_i = sum_f beta_f (p_i - p_nbr) on the MAC grid.
//
// Hierarchy: unsmoothed-aggregation Galerkin (coarse face = sum of 4 fine
// faces), red-black weighted Gauss-Seidel (omega = 6/7), V-cycle with
// pre (0,1) / post (1,0) colour orders.  Large levels run one kernel per
// red-black sweep out of HBM (one per half-sweep on request), levels of up
// to about 64^3 cells one kernel per smoothing phase; every level
// from `small_from` down is solved inside one workgroup with all its data
// in LDS.  The FPCG scalars live on the
// device; dot products are deterministic FP64 block reductions, and the
// host polls a "done" flag while the GPU still has queued work.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <new>
#include <type_traits>
#include <vector>

#include "pf_common.hpp"

namespace pf {

int fill_u32(void* dst, int64_t n, uint32_t v, hipStream_t s);

constexpr int MAXB = 1024;  // blocks of a reduction launch
constexpr int PS = 8192;    // entries per quantity of the partial-sum arrays (the sweeps write one per tile)
constexpr int RT = 256;     // threads of element-wise / reduction kernels
// k_cg_apply and k_cg_beta: few, wide blocks, so the kernel that combines
// their partials itself reads few of them
constexpr int WT = 1024;
constexpr int WB = 256;

// Largest coarsest level whose smoother is applied as a precomputed matrix.
constexpr int kCoarseOpMax = 512;

struct CGState {
    double alpha, beta, mu, b_norm, rel, qAq, mu_x, tol;
    // <r, z - mu> of the iteration whose search direction parity is the
    // index: the k_cg_apply of iteration `slot` forms its value from the
    // previous one's, so the two never share a word
    double rz[2];
    int it, done, seq;  // seq: residual tests run in this solve
    int beta_parts;     // 1: the FPCG beta partials in part[0..5) are this iteration's to combine
    // 16-bit V-cycles: the level-0 right-hand side is read times vscale (a
    // power of two putting max|r| in [1/2, 1)) and z is read back times
    // vscale_inv, so the FP16 iterates stay in range as r shrinks
    float vscale, vscale_inv;
    unsigned ticket[8];
    double part[6 * PS];  // [0, 5 PS): dot-product partials; [5 PS, 6 PS): <q, Aq> partials
    float fpart[MAXB];
    // the coarsest level's `coarsest` red-black sweeps from zero followed by
    // mean removal, a linear map of its right-hand side: column j (the image
    // of the unit vector e_j) at [j * n, (j + 1) * n), built by pf_mg_build.
    // FP64: at 1000:1 contrast its entries are large and of both signs, and
    // an FP32 map loses the result to cancellation
    double coarse_op[kCoarseOpMax * kCoarseOpMax];
};

// vscale = 2^-e with m = f 2^e, f in [1/2, 1): m * vscale in [1/2, 1)
__device__ inline int vscale_exponent(float m) {
    int e = 0;
    if (m > 0.0f && m < 3.0e38f) {
        (void)frexpf(m, &e);
        e = max(min(e, 120), -120);
    }
    return e;
}

__device__ inline void set_vscale(CGState* st, float m) {
    const int e = vscale_exponent(m);
    st->vscale = ldexpf(1.0f, -e);
    st->vscale_inv = ldexpf(1.0f, e);
}

// The residual test (poisson.py:394-398) on m = max|r|, recorded by one
// thread: rel, done, the 16-bit input scale, then (number of tests so far) *
// 2 + (done != 0) to host_flag (pinned host memory, may be NULL) with a
// system-scope store the polling host sees without any event.  A solve that
// is already done only publishes.
__device__ inline void residual_test_record(CGState* st, float m, int* host_flag) {
    if (!st->done) {
        const double rel = (double)m / st->b_norm;
        st->rel = rel;
        if (rel < st->tol) st->done = 1;
        set_vscale(st, m);
    }
    st->seq += 1;
    if (host_flag)
        __hip_atomic_store(host_flag, st->seq * 2 + (st->done != 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Pinned host words of a solver: the residual tests' flag, then the
// solve's result (its number, the iteration count, the residual as the bits
// of a double).
// HW_WANT: the number the next result is to carry, written by the host
// before the launch (a captured graph cannot take it as an argument).
enum HostWord { HW_FLAG = 0, HW_RESULT_NO = 1, HW_IT = 2, HW_WANT = 3, HW_REL = 4, HW_WORDS = 8 };

// The solve's result for the host: the iteration count and the residual,
// then the solve's number, into pinned host memory with system-scope stores
// (the number last, with release order), so the host spins on one word
// instead of copying the scalars back and synchronising the stream.  The
// kernels before it on the stream have completed when it runs.
__global__ void k_publish_result(const CGState* st, int* words) {
    if (threadIdx.x != 0) return;
    const int number = __hip_atomic_load(words + HW_WANT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    const int it = st->it;
    const unsigned long long rel = (unsigned long long)__double_as_longlong(st->rel);
    __hip_atomic_store(words + HW_IT, it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(words + HW_REL), rel, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(words + HW_RESULT_NO, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The residual test folded into the V-cycle's first kernel (the zero-start
// level-0 sweep): every block takes the max of k_cg_update's partials itself
// (max is exact, so all blocks agree) and so knows whether to store and the
// 16-bit input scale; block 0 records the test.  st == NULL: no fold.
struct UpdateFold {
    CGState* st;
    int nparts;
    int* host_flag;
};

// The flexible CG's inner products after the preconditioner (k_cg_beta's
// work), folded into the V-cycle's last level-0 sweep, which has the final
// z and the residual r (its right-hand side) of its tile in registers: per
// workgroup the FP64 partials of sum z, sum r, sum Ap, <r, z>, <Ap, z> of
// its tile's cells, with z as stored (times zscale for 16-bit iterates).
struct DotFold {
    const float* Ap;
    const float* zscale;
    CGState* st;
};

static unsigned red_blocks(int64_t n) {
    const int64_t nb = cdiv(n, (int64_t)RT * 4);
    return (unsigned)(nb < 1 ? 1 : (nb > MAXB ? MAXB : nb));
}

// Combine per-block partials in the last block: every thread sums a fixed
// strided subset, then a fixed-order block reduction (deterministic).
template <int NV>
__device__ inline void combine_sums(const double* part, int nparts, double (&v)[NV], double* sh) {
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = 0.0;
#pragma unroll 4
    for (int b = threadIdx.x; b < nparts; b += blockDim.x)
#pragma unroll
        for (int q = 0; q < NV; ++q) v[q] += part[q * PS + b];
    block_sum<NV>(v, sh);
}

__device__ inline float combine_max(const float* part, int nparts, float* sh) {
    float m = 0.0f;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x) m = fmaxf(m, part[b]);
    return block_max(m, sh);
}

// ================================================================ stencil
template <typename FT, typename PT>
__device__ inline void stencil_s(const Dims& d, const FT* __restrict__ bx, const FT* __restrict__ by,
                                 const FT* __restrict__ bz, const PT* p, int i, int j, int k,
                                 float& diag, float& s, float& pc) {
    const float bxl = to_f32(bx[face_index<0>(d, i, j, k)]);
    const float bxh = to_f32(bx[face_index<0>(d, i + 1, j, k)]);
    const float byl = to_f32(by[face_index<1>(d, i, j, k)]);
    const float byh = to_f32(by[face_index<1>(d, i, j + 1, k)]);
    const float bzl = to_f32(bz[face_index<2>(d, i, j, k)]);
    const float bzh = to_f32(bz[face_index<2>(d, i, j, k + 1)]);
    // compute_diag order (poisson.py:49-51)
    diag = bxl + bxh + byl + byh + bzl + bzh;
    pc = to_f32(p[cell_index(d, i, j, k)]);
    // _apply_row order, neighbours clamped at the walls (poisson.py:69-75)
    s = bxl * to_f32(p[cell_index(d, max(i - 1, 0), j, k)]);
    s += bxh * to_f32(p[cell_index(d, min(i + 1, d.nx - 1), j, k)]);
    s += byl * to_f32(p[cell_index(d, i, max(j - 1, 0), k)]);
    s += byh * to_f32(p[cell_index(d, i, min(j + 1, d.ny - 1), k)]);
    s += bzl * to_f32(p[cell_index(d, i, j, max(k - 1, 0))]);
    s += bzh * to_f32(p[cell_index(d, i, j, min(k + 1, d.nz - 1))]);
}

// A p in the difference form sum_f beta_f (p_i - p_f).  It equals
// diag*p_i - sum_f beta_f p_f (the reference's form, poisson.py:75), but in
// FP32 the subtractions of nearby values are exact, so the product carries
// no cancellation error: the reference's form limits the recursively
// updated CG residual to ~3e-6 (FP32) / ~4e-5 (16-bit preconditioner) at a
// 1000:1 coefficient jump, this form to ~1e-9 / ~5e-8.
// f = (x-low, x-high, y-low, y-high, z-low, z-high) faces, pn the matching
// neighbour values.  Every smoother and residual kernel goes through these
// helpers, so all of them round identically: the fused multiply-adds are
// written out and contraction is off, since the compiler could otherwise
// fuse either product of the first sum and choose differently per kernel.
__device__ inline void stencil_vals(float pc, const float (&f)[6], const float (&pn)[6], float& diag,
                                    float& Ap) {
#pragma clang fp contract(off)
    diag = f[0] + f[1] + f[2] + f[3] + f[4] + f[5];
    float s = f[0] * (pc - pn[0]);
    s = fmaf(f[1], pc - pn[1], s);
    s = fmaf(f[2], pc - pn[2], s);
    s = fmaf(f[3], pc - pn[3], s);
    s = fmaf(f[4], pc - pn[4], s);
    s = fmaf(f[5], pc - pn[5], s);
    Ap = s;
}

// weighted Gauss-Seidel update of one cell (poisson.py:120-126)
__device__ inline float rb_relax(float pc, float b, float Ap, float dg, float omega) {
    return pc + omega * (b - Ap) / dg;
}
// the same update from p = 0 (every neighbour and the cell itself zero)
__device__ inline float rb_first(float b, float dg, float omega) { return omega * b / dg; }

template <typename ST>
__device__ inline float round_st(float v) { return to_f32(from_f32<ST>(v)); }

template <typename FT, typename PT>
__device__ inline void stencil(const Dims& d, const FT* __restrict__ bx, const FT* __restrict__ by,
                               const FT* __restrict__ bz, const PT* p, int i, int j, int k,
                               float& diag, float& Ap, float& pc) {
    const float f[6] = {to_f32(bx[face_index<0>(d, i, j, k)]), to_f32(bx[face_index<0>(d, i + 1, j, k)]),
                        to_f32(by[face_index<1>(d, i, j, k)]), to_f32(by[face_index<1>(d, i, j + 1, k)]),
                        to_f32(bz[face_index<2>(d, i, j, k)]), to_f32(bz[face_index<2>(d, i, j, k + 1)])};
    pc = to_f32(p[cell_index(d, i, j, k)]);
    const float pn[6] = {to_f32(p[cell_index(d, max(i - 1, 0), j, k)]),
                         to_f32(p[cell_index(d, min(i + 1, d.nx - 1), j, k)]),
                         to_f32(p[cell_index(d, i, max(j - 1, 0), k)]),
                         to_f32(p[cell_index(d, i, min(j + 1, d.ny - 1), k)]),
                         to_f32(p[cell_index(d, i, j, max(k - 1, 0))]),
                         to_f32(p[cell_index(d, i, j, min(k + 1, d.nz - 1))])};
    stencil_vals(pc, f, pn, diag, Ap);
}

// ================================================================ hierarchy build
// Coarse face = sum of the 4 fine faces it covers (poisson.py:130-163).
__global__ __launch_bounds__(RT) void k_galerkin(Dims df, Dims dc, const float* __restrict__ fx,
                                                 const float* __restrict__ fy,
                                                 const float* __restrict__ fz, float* __restrict__ cx,
                                                 float* __restrict__ cy, float* __restrict__ cz) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int ez = dc.nz + 1, ey = dc.ny + 1;
    if (t >= (int64_t)(dc.nx + 1) * ey * ez) return;
    const int K = (int)(t % ez), J = (int)((t / ez) % ey), I = (int)(t / ((int64_t)ez * ey));
    const int i0 = 2 * I, j0 = 2 * J, k0 = 2 * K;
    if (J < dc.ny && K < dc.nz) {
        float acc = 0.f;
        for (int a = 0; a < 2; ++a)
            for (int b = 0; b < 2; ++b) {
                const int jj = j0 + a, kk = k0 + b;
                if (i0 <= df.nx && jj < df.ny && kk < df.nz) acc += fx[face_index<0>(df, i0, jj, kk)];
            }
        cx[face_index<0>(dc, I, J, K)] = acc;
    }
    if (I < dc.nx && K < dc.nz) {
        float acc = 0.f;
        for (int a = 0; a < 2; ++a)
            for (int b = 0; b < 2; ++b) {
                const int ii = i0 + a, kk = k0 + b;
                if (ii < df.nx && j0 <= df.ny && kk < df.nz) acc += fy[face_index<1>(df, ii, j0, kk)];
            }
        cy[face_index<1>(dc, I, J, K)] = acc;
    }
    if (I < dc.nx && J < dc.ny) {
        float acc = 0.f;
        for (int a = 0; a < 2; ++a)
            for (int b = 0; b < 2; ++b) {
                const int ii = i0 + a, jj = j0 + b;
                if (ii < df.nx && jj < df.ny && k0 <= df.nz) acc += fz[face_index<2>(df, ii, jj, k0)];
            }
        cz[face_index<2>(dc, I, J, K)] = acc;
    }
}

// diag (poisson.py:40-51) and, for levels run out of HBM in reduced
// precision, the 16-bit copies of the face coefficients.
template <typename ST>
__global__ __launch_bounds__(RT) void k_diag_copy(Dims d, const float* __restrict__ bx,
                                                  const float* __restrict__ by,
                                                  const float* __restrict__ bz, float* diag, ST* hx,
                                                  ST* hy, ST* hz) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int ez = d.nz + 1, ey = d.ny + 1;
    if (t >= (int64_t)(d.nx + 1) * ey * ez) return;
    const int k = (int)(t % ez), j = (int)((t / ez) % ey), i = (int)(t / ((int64_t)ez * ey));
    const bool ci = i < d.nx, cj = j < d.ny, ck = k < d.nz;
    if (hx) {
        if (cj && ck) hx[face_index<0>(d, i, j, k)] = from_f32<ST>(bx[face_index<0>(d, i, j, k)]);
        if (ci && ck) hy[face_index<1>(d, i, j, k)] = from_f32<ST>(by[face_index<1>(d, i, j, k)]);
        if (ci && cj) hz[face_index<2>(d, i, j, k)] = from_f32<ST>(bz[face_index<2>(d, i, j, k)]);
    }
    if (diag && ci && cj && ck)
        diag[cell_index(d, i, j, k)] = bx[face_index<0>(d, i, j, k)] + bx[face_index<0>(d, i + 1, j, k)] +
                                       by[face_index<1>(d, i, j, k)] + by[face_index<1>(d, i, j + 1, k)] +
                                       bz[face_index<2>(d, i, j, k)] + bz[face_index<2>(d, i, j, k + 1)];
}

// ================================================================ HBM smoother / transfers
// Red-black half-sweep (poisson.py:105-126).  One thread per cell of the
// active colour.  ZINIT: p is known to be zero (a freshly cleared level),
// so res = b and every cell of the other colour is written as 0.
template <typename ST, bool ZINIT>
__global__ __launch_bounds__(RT) void k_rbgs(Dims d, const ST* __restrict__ bx,
                                             const ST* __restrict__ by, const ST* __restrict__ bz,
                                             ST* p, const float* __restrict__ b, int colour,
                                             float omega, const int* __restrict__ done,
                                             const float* __restrict__ bscale) {
    // the flag is only consulted at the stores, so its load does not delay
    // the stencil loads (a converged solve's extra iteration stores nothing)
    const bool skip = done && *done;
    const float bs = bscale ? *bscale : 1.0f;
    const int nkp = (d.nz + 1) >> 1;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)d.nx * d.ny * nkp) return;
    const int kp = (int)(t % nkp);
    const int row = (int)(t / nkp);
    const int j = row % d.ny, i = row / d.ny;
    if (ZINIT) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int k = 2 * kp + q;
            if (k >= d.nz) break;
            float v = 0.0f;
            if (((i + j + k) & 1) == colour) {
                const float dg = to_f32(bx[face_index<0>(d, i, j, k)]) + to_f32(bx[face_index<0>(d, i + 1, j, k)]) +
                                 to_f32(by[face_index<1>(d, i, j, k)]) + to_f32(by[face_index<1>(d, i, j + 1, k)]) +
                                 to_f32(bz[face_index<2>(d, i, j, k)]) + to_f32(bz[face_index<2>(d, i, j, k + 1)]);
                if (dg > 0.0f) v = rb_first(b[cell_index(d, i, j, k)] * bs, dg, omega);
            }
            if (!skip) p[cell_index(d, i, j, k)] = from_f32<ST>(v);
        }
    } else {
        const int k = 2 * kp + ((i + j + colour) & 1);
        if (k >= d.nz) return;
        float dg, Ap, pc;
        stencil(d, bx, by, bz, p, i, j, k, dg, Ap, pc);
        if (dg <= 0.0f) return;
        const int c = cell_index(d, i, j, k);
        if (!skip) p[c] = from_f32<ST>(rb_relax(pc, b[c] * bs, Ap, dg, omega));
    }
}

// Pair loads/stores: cells (i,j,k) and (i,j,k+1) with k even, adjacent in
// memory and 2-element aligned whenever the row length is even.
template <typename ST>
__device__ inline void ld_pair(const ST* p, int idx, float& a, float& b);
template <>
__device__ inline void ld_pair<float>(const float* p, int idx, float& a, float& b) {
    const float2 v = *reinterpret_cast<const float2*>(p + idx);
    a = v.x;
    b = v.y;
}
template <typename ST>
__device__ inline void ld_pair(const ST* p, int idx, float& a, float& b) {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(p + idx);
    a = to_f32(ST{(uint16_t)(w & 0xFFFFu)});
    b = to_f32(ST{(uint16_t)(w >> 16)});
}
template <typename ST>
__device__ inline void st_pair(ST* p, int idx, float a, float b);
template <>
__device__ inline void st_pair<float>(float* p, int idx, float a, float b) {
    *reinterpret_cast<float2*>(p + idx) = make_float2(a, b);
}
template <typename ST>
__device__ inline void st_pair(ST* p, int idx, float a, float b) {
    const uint32_t w = (uint32_t)from_f32<ST>(a).u | ((uint32_t)from_f32<ST>(b).u << 16);
    *reinterpret_cast<uint32_t*>(p + idx) = w;
}

// One full red-black sweep (colour c1, then the other colour) in one launch,
// bitwise equal to two in-place half-sweeps.  A workgroup owns a TI x TJ x TK
// tile.  It stages the iterate of the tile plus a 2-cell halo in LDS
// (coordinates clamped into the grid, which reproduces the reference's
// clamped neighbour indices: a clamped neighbour is the cell itself), updates
// the first colour on the tile and on its 1-cell halo shell (the shell
// updates duplicate work of the neighbouring tiles), then the second colour
// on the tile, and writes the whole tile to `pout`.  Reading `pin` and
// writing `pout` (ping-pong) keeps neighbouring tiles' halo reads race-free.
// Each thread owns pairs of cells (k, k+1) of the tile and keeps the pair's
// faces in registers between the two colours, so faces, b and p are read
// from memory once per sweep.  Every global load (staging, the tile's faces
// and b, the shell cells' faces and b) is issued before the first wait, so
// a workgroup is exposed to memory latency once.  Needs nz even.
// ZINIT: the input is zero (no staging loads).
template <int TI, int TJ, int TK, int NTH>
struct RbTile {
    static constexpr int NT = NTH;
    static constexpr int PI = TI + 4, PJ = TJ + 4, PK = TK + 4;
    static constexpr int NP = PI * PJ * PK;
    static constexpr int NPR = PK / 2;                    // staged pairs per row
    static constexpr int NSP = PI * PJ * NPR;             // staged pairs
    static constexpr int SPT = (NSP + NT - 1) / NT;       // staged pairs per thread
    static constexpr int PAIRS = TI * TJ * TK / 2;
    static constexpr int PPT = PAIRS / NT;
    // first-colour shell cells: i-planes and j-planes hold rows along k of
    // TK+2 cells (half of each row has colour c1); k-planes rows along j
    static constexpr int RK = (TK + 2) / 2;
    static constexpr int S1 = 2 * (TJ + 2) * RK, S2 = 2 * TI * RK, S3 = 2 * TI * (TJ / 2);
    static constexpr int NS = S1 + S2 + S3;
    static constexpr int SHT = (NS + NT - 1) / NT;
    static_assert(PAIRS % NT == 0 && TK % 2 == 0 && TJ % 2 == 0 && PPT >= 1, "tile shape");
};

// (4 waves per SIMD: a 128^3 level's 512 workgroups of 8x8x64 tiles are all
// resident at once, so the sweep costs one memory round trip, not two)
// PROL: the sweep's input is pin plus the piecewise-constant prolongation of
// the coarse iterate pc (poisson.py:178-182), formed in LDS while staging
// (rounded to ST as the separate prolongation stores it): the first
// post-sweep of a level without a separate prolongation pass.
// DOTS: the CG's inner products of the sweep's output (DotFold), with Ap
// staged into LDS alongside the iterate and the sums formed after the
// stores, when the face registers are free.
template <typename ST, bool ZINIT, int TI, int TJ, int TK, int NTH = 256, bool PROL = false, typename CT = float,
          bool DOTS = false>
__global__ __launch_bounds__(NTH, 4) void k_rbgs_full(Dims d, const ST* __restrict__ bx,
                                                   const ST* __restrict__ by, const ST* __restrict__ bz,
                                                   const ST* __restrict__ pin, ST* __restrict__ pout,
                                                   const float* __restrict__ b, int c1, float omega,
                                                   const int* __restrict__ done,
                                                   const float* __restrict__ bscale,
                                                   const CT* __restrict__ pcoarse, Dims dc, UpdateFold uf,
                                                   DotFold df) {
    using T = RbTile<TI, TJ, TK, NTH>;
    __shared__ __attribute__((aligned(16))) float P[T::NP];
    __shared__ float s_fm[NTH / 64];
    const int tid = threadIdx.x;
    // the residual test's inputs, loaded with everything else
    const bool fold = uf.st != nullptr;
    int was_done = 0;
    float fm = 0.0f;
    if (fold) {
        was_done = uf.st->done;
        for (int e = tid; e < uf.nparts; e += T::NT) fm = fmaxf(fm, uf.st->fpart[e]);
    }
    const int ntk = (d.nz + TK - 1) / TK, ntj = (d.ny + TJ - 1) / TJ;
    const int tile = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = (tile / (ntk * ntj)) * TI, j0 = ((tile / ntk) % ntj) * TJ, k0 = (tile % ntk) * TK;
    constexpr int SI = T::PJ * T::PK, SJ = T::PK;
    auto lidx = [&](int i, int j, int k) { return ((i - i0 + 2) * T::PJ + (j - j0 + 2)) * T::PK + (k - k0 + 2); };

    // (1) staging: the iterate of the tile + 2-cell halo goes straight from
    // memory into LDS (global_load_lds: lane l of a wave writes its dword to
    // the wave's LDS base + 4 l, no registers).  FP32: one element per lane
    // from clamped coordinates.  16-bit: raw pairs (k, k+1) from the nearest
    // in-grid pair into R, converted into P after the barrier.
    constexpr bool F32 = sizeof(ST) == 4;
    __shared__ uint32_t R[F32 ? 1 : T::NSP];
    if (!ZINIT) {
        if constexpr (F32) {
            for (int e0 = 0; e0 < T::NP; e0 += T::NT) {
                const int e = e0 + tid;
                if (e < T::NP) {
                    const int kk = e % T::PK, jj = (e / T::PK) % T::PJ, ii = e / SI;
                    const int gi = min(max(i0 - 2 + ii, 0), d.nx - 1);
                    const int gj = min(max(j0 - 2 + jj, 0), d.ny - 1);
                    const int gk = min(max(k0 - 2 + kk, 0), d.nz - 1);
                    __builtin_amdgcn_global_load_lds(
                        (const void*)(pin + cell_index(d, gi, gj, gk)),
                        (__attribute__((address_space(3))) void*)(P + e0 + (tid & ~63)), 4, 0, 0);
                }
            }
        } else {
            for (int e0 = 0; e0 < T::NSP; e0 += T::NT) {
                const int e = e0 + tid;
                if (e < T::NSP) {
                    const int q = e % T::NPR, row = e / T::NPR;
                    const int gi = min(max(i0 - 2 + row / T::PJ, 0), d.nx - 1);
                    const int gj = min(max(j0 - 2 + row % T::PJ, 0), d.ny - 1);
                    const int kc = min(max(k0 - 2 + 2 * q, 0), d.nz - 2);
                    __builtin_amdgcn_global_load_lds(
                        (const void*)(pin + cell_index(d, gi, gj, kc)),
                        (__attribute__((address_space(3))) void*)(R + e0 + (tid & ~63)), 4, 0, 0);
                }
            }
        }
    }

    // (1b) PROL: the coarse iterate under the staged region, parents
    // [i0/2 - 1, i0/2 + TI/2 + 1) per axis (coordinates clamped)
    constexpr int CI = TI / 2 + 2, CJ = TJ / 2 + 2, CK = TK / 2 + 2, CN = CI * CJ * CK;
    constexpr int CPT = PROL ? (CN + T::NT - 1) / T::NT : 1;
    float cv[CPT];
    if constexpr (PROL) {
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            const int e = tid + q * T::NT;
            cv[q] = 0.0f;
            if (e < CN) {
                const int ck = e % CK, cj = (e / CK) % CJ, ci = e / (CK * CJ);
                const int gi = min(max(i0 / 2 - 1 + ci, 0), dc.nx - 1);
                const int gj = min(max(j0 / 2 - 1 + cj, 0), dc.ny - 1);
                const int gk = min(max(k0 / 2 - 1 + ck, 0), dc.nz - 1);
                cv[q] = to_f32(pcoarse[cell_index(dc, gi, gj, gk)]);
            }
        }
    }

    // (2) the tile's pairs: faces and b into registers
    float f[T::PPT][11], bb[T::PPT][2];
    int li[T::PPT];
    bool ok[T::PPT];
#pragma unroll
    for (int q = 0; q < T::PPT; ++q) {
        const int pq = tid + q * T::NT;
        const int kp = pq % (TK / 2), jl = (pq / (TK / 2)) % TJ, il = pq / ((TK / 2) * TJ);
        const int i = i0 + il, j = j0 + jl, k = k0 + 2 * kp;
        ok[q] = i < d.nx && j < d.ny && k < d.nz;
        li[q] = ((il + 2) * T::PJ + (jl + 2)) * T::PK + (2 * kp + 2);
        if (ok[q]) {
            ld_pair(bx, face_index<0>(d, i, j, k), f[q][0], f[q][1]);      // x-low of k, k+1
            ld_pair(bx, face_index<0>(d, i + 1, j, k), f[q][2], f[q][3]);  // x-high
            ld_pair(by, face_index<1>(d, i, j, k), f[q][4], f[q][5]);      // y-low
            ld_pair(by, face_index<1>(d, i, j + 1, k), f[q][6], f[q][7]);  // y-high
            const int z = face_index<2>(d, i, j, k);
            f[q][8] = to_f32(bz[z]);
            f[q][9] = to_f32(bz[z + 1]);
            f[q][10] = to_f32(bz[z + 2]);
            ld_pair(b, cell_index(d, i, j, k), bb[q][0], bb[q][1]);
        }
    }
    // (1c) DOTS: Ap of the tile into LDS, cell (il, jl, kl) at its tile-linear
    // index (every lane loads: coordinates clamped into the grid)
    constexpr int TC = TI * TJ * TK;
    __shared__ float A[DOTS ? TC : 1];
    if constexpr (DOTS) {
        static_assert(TC % T::NT == 0, "whole passes");
        for (int e0 = 0; e0 < TC; e0 += T::NT) {
            const int e = e0 + tid;
            const int kl = e % TK, jl = (e / TK) % TJ, il = e / (TK * TJ);
            const int gi = min(i0 + il, d.nx - 1), gj = min(j0 + jl, d.ny - 1), gk = min(k0 + kl, d.nz - 1);
            __builtin_amdgcn_global_load_lds((const void*)(df.Ap + cell_index(d, gi, gj, gk)),
                                             (__attribute__((address_space(3))) void*)(A + e0 + (tid & ~63)), 4,
                                             0, 0);
        }
    }

    // (3) first-colour cells of the 1-cell halo shell that lie in the grid
    float sf[T::SHT][6], sb[T::SHT];
    int sc[T::SHT];
    bool sok[T::SHT];
#pragma unroll
    for (int r = 0; r < T::SHT; ++r) {
        int e = tid + r * T::NT, i, j, k;
        if (e < T::S1) {  // i = i0-1 and i0+TI, all j of the shell, rows along k
            i = e < T::S1 / 2 ? i0 - 1 : i0 + TI;
            e %= T::S1 / 2;
            j = j0 - 1 + e / T::RK;
            const int m = e % T::RK, base = k0 - 1;
            k = base + 2 * m + ((c1 - (i + j + base)) & 1);
        } else if ((e -= T::S1) < T::S2) {  // j = j0-1 and j0+TJ, i in the tile
            j = e < T::S2 / 2 ? j0 - 1 : j0 + TJ;
            e %= T::S2 / 2;
            i = i0 + e / T::RK;
            const int m = e % T::RK, base = k0 - 1;
            k = base + 2 * m + ((c1 - (i + j + base)) & 1);
        } else {  // k = k0-1 and k0+TK, i and j in the tile, rows along j
            e -= T::S2;
            k = e < T::S3 / 2 ? k0 - 1 : k0 + TK;
            e %= T::S3 / 2;
            i = i0 + e / (TJ / 2);
            const int m = e % (TJ / 2);
            j = j0 + 2 * m + ((c1 - (i + j0 + k)) & 1);
        }
        sok[r] = (tid + r * T::NT) < T::NS && i >= 0 && j >= 0 && k >= 0 && i < d.nx && j < d.ny && k < d.nz;
        sc[r] = lidx(i, j, k);
        if (sok[r]) {
            sf[r][0] = to_f32(bx[face_index<0>(d, i, j, k)]);
            sf[r][1] = to_f32(bx[face_index<0>(d, i + 1, j, k)]);
            sf[r][2] = to_f32(by[face_index<1>(d, i, j, k)]);
            sf[r][3] = to_f32(by[face_index<1>(d, i, j + 1, k)]);
            sf[r][4] = to_f32(bz[face_index<2>(d, i, j, k)]);
            sf[r][5] = to_f32(bz[face_index<2>(d, i, j, k + 1)]);
            sb[r] = b[cell_index(d, i, j, k)];
        }
    }
    bool skip = !fold && done && *done;
    if (fold) {
        fm = wave_max(fm);
        if ((tid & 63) == 0) s_fm[tid >> 6] = fm;
    }

    if (ZINIT) {
        for (int e = tid; e < T::NP; e += T::NT) P[e] = 0.0f;
    } else {
        __builtin_amdgcn_s_waitcnt(0);  // the LDS-destined loads have landed
    }
    __syncthreads();
    float bs = 1.0f;
    if (fold) {
        float mm = s_fm[0];
#pragma unroll
        for (int w = 1; w < NTH / 64; ++w) mm = fmaxf(mm, s_fm[w]);
        const bool conv = (double)mm / uf.st->b_norm < uf.st->tol;
        skip = was_done || conv;
        bs = ldexpf(1.0f, -vscale_exponent(mm));
        if (blockIdx.x == 0 && tid == 0) residual_test_record(uf.st, mm, uf.host_flag);
    } else if (bscale) {
        bs = *bscale;
    }
    // a finished solve's queued iterations stop here: after the loads (the
    // flag is not waited for before issuing them) but before any arithmetic
    // (every load has landed; skip is the same in the whole workgroup)
    if (skip) return;
    if (bscale) {
#pragma unroll
        for (int q = 0; q < T::PPT; ++q) {
            bb[q][0] *= bs;
            bb[q][1] *= bs;
        }
#pragma unroll
        for (int r = 0; r < T::SHT; ++r) sb[r] *= bs;
    }
    if constexpr (!F32) {
        if (!ZINIT) {
            // raw pairs -> floats (LDS index 2 * pair index); past either end
            // of a row both entries clamp to the end cell
            for (int e = tid; e < T::NSP; e += T::NT) {
                const uint32_t w = R[e];
                float x = to_f32(ST{(uint16_t)(w & 0xFFFFu)}), y = to_f32(ST{(uint16_t)(w >> 16)});
                const int kk = k0 - 2 + 2 * (e % T::NPR);
                if (kk < 0) y = x;
                if (kk > d.nz - 2) x = y;
                P[2 * e] = x;
                P[2 * e + 1] = y;
            }
            __syncthreads();
        }
    }
    if constexpr (PROL) {
        __shared__ float C[PROL ? CN : 1];
#pragma unroll
        for (int q = 0; q < CPT; ++q)
            if (tid + q * T::NT < CN) C[tid + q * T::NT] = cv[q];
        __syncthreads();
        // staged pairs (k, k+1) with k even share their parent, clamping
        // included (k0 is even, so a clamped pair clamps to one cell)
        for (int e2 = tid; e2 < T::NP / 2; e2 += T::NT) {
            const int m = e2 % (T::PK / 2), row = e2 / (T::PK / 2);
            const int jj = row % T::PJ, ii = row / T::PJ;
            const int gi = min(max(i0 - 2 + ii, 0), d.nx - 1);
            const int gj = min(max(j0 - 2 + jj, 0), d.ny - 1);
            const int gk = min(max(k0 - 2 + 2 * m, 0), d.nz - 1);
            const int ci = (gi >> 1) - (i0 / 2 - 1), cj = (gj >> 1) - (j0 / 2 - 1), ck = (gk >> 1) - (k0 / 2 - 1);
            const float c = C[(ci * CJ + cj) * CK + ck];
            float2 v = *reinterpret_cast<float2*>(P + 2 * e2);
            v.x = round_st<ST>(v.x + c);
            v.y = round_st<ST>(v.y + c);
            *reinterpret_cast<float2*>(P + 2 * e2) = v;
        }
        __syncthreads();
    }

    // first colour on the tile
#pragma unroll
    for (int q = 0; q < T::PPT; ++q) {
        if (!ok[q]) continue;
        const int pq = tid + q * T::NT;
        const int jl = (pq / (TK / 2)) % TJ, il = pq / ((TK / 2) * TJ);
        const int h = ((i0 + il + j0 + jl) & 1) == c1 ? 0 : 1;  // which cell of the pair has colour c1
        const int c = li[q] + h;
        const float fc[6] = {f[q][h], f[q][2 + h], f[q][4 + h], f[q][6 + h], f[q][8 + h], f[q][9 + h]};
        float v;
        if (ZINIT) {
            const float dg = fc[0] + fc[1] + fc[2] + fc[3] + fc[4] + fc[5];
            v = dg > 0.0f ? rb_first(bb[q][h], dg, omega) : 0.0f;
        } else {
            const float pc = P[c];
            const float pn[6] = {P[c - SI], P[c + SI], P[c - SJ], P[c + SJ], P[c - 1], P[c + 1]};
            float dg, Ap;
            stencil_vals(pc, fc, pn, dg, Ap);
            v = dg > 0.0f ? rb_relax(pc, bb[q][h], Ap, dg, omega) : pc;
        }
        P[c] = round_st<ST>(v);
    }
    // first colour on the halo shell
#pragma unroll
    for (int r = 0; r < T::SHT; ++r) {
        if (!sok[r]) continue;
        const int c = sc[r];
        const float fc[6] = {sf[r][0], sf[r][1], sf[r][2], sf[r][3], sf[r][4], sf[r][5]};
        float v;
        if (ZINIT) {
            const float dg = fc[0] + fc[1] + fc[2] + fc[3] + fc[4] + fc[5];
            v = dg > 0.0f ? rb_first(sb[r], dg, omega) : 0.0f;
        } else {
            const float pc = P[c];
            const float pn[6] = {P[c - SI], P[c + SI], P[c - SJ], P[c + SJ], P[c - 1], P[c + 1]};
            float dg, Ap;
            stencil_vals(pc, fc, pn, dg, Ap);
            v = dg > 0.0f ? rb_relax(pc, sb[r], Ap, dg, omega) : pc;
        }
        P[c] = round_st<ST>(v);
    }
    __syncthreads();

    // second colour on the tile, then the pair goes out
#pragma unroll
    for (int q = 0; q < T::PPT; ++q) {
        if (!ok[q]) continue;
        const int pq = tid + q * T::NT;
        const int kp = pq % (TK / 2), jl = (pq / (TK / 2)) % TJ, il = pq / ((TK / 2) * TJ);
        const int h = ((i0 + il + j0 + jl) & 1) == c1 ? 1 : 0;  // the cell of the other colour
        const int c = li[q] + h;
        const float fc[6] = {f[q][h], f[q][2 + h], f[q][4 + h], f[q][6 + h], f[q][8 + h], f[q][9 + h]};
        const float pc = P[c];
        const float pn[6] = {P[c - SI], P[c + SI], P[c - SJ], P[c + SJ], P[c - 1], P[c + 1]};
        float dg, Ap;
        stencil_vals(pc, fc, pn, dg, Ap);
        const float v = dg > 0.0f ? rb_relax(pc, bb[q][h], Ap, dg, omega) : pc;
        const float other = P[li[q] + (1 - h)];
        if (!skip)
            st_pair(pout, cell_index(d, i0 + il, j0 + jl, k0 + 2 * kp), h ? other : v, h ? v : other);
        // DOTS: the cell's value as stored (no other thread reads a
        // second-colour cell in this half-sweep)
        if (DOTS) P[c] = round_st<ST>(v);
    }
    if constexpr (DOTS) {
        // k_cg_beta's sums over the tile: z as stored times zscale (its
        // zval), r = b unscaled (b * bs * zscale, powers of two), Ap
        const float zsc = df.zscale ? *df.zscale : 1.0f;
        // (A landed before the first barrier; a pair's two cells were
        // written by this thread)
        double dsum[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < T::PPT; ++q) {
            if (!ok[q]) continue;
            const int pq = tid + q * T::NT;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const double zz = (double)(P[li[q] + e] * zsc), rr = (double)(bb[q][e] * zsc);
                const double ap = (double)A[2 * pq + e];
                dsum[0] += zz;
                dsum[1] += rr;
                dsum[2] += ap;
                dsum[3] += rr * zz;
                dsum[4] += ap * zz;
            }
        }
        __shared__ double s_dot[5 * 16];
        block_sum<5>(dsum, s_dot);
        if (tid == 0 && !skip) {
#pragma unroll
            for (int q = 0; q < 5; ++q) df.st->part[q * PS + blockIdx.x] = dsum[q];
            if (blockIdx.x == 0) df.st->beta_parts = 1;  // read by the next k_cg_apply
        }
    }
}

// residual (poisson.py:91-102) fused with R = P^T (poisson.py:166-175)
template <typename ST>
__global__ __launch_bounds__(RT) void k_resid_restrict(Dims d, Dims dc, const ST* __restrict__ bx,
                                                       const ST* __restrict__ by,
                                                       const ST* __restrict__ bz,
                                                       const ST* __restrict__ p,
                                                       const float* __restrict__ b,
                                                       float* __restrict__ bc,
                                                       const int* __restrict__ done,
                                                       const float* __restrict__ bscale) {
    const bool skip = done && *done;
    const float bs = bscale ? *bscale : 1.0f;
    // 32-bit index arithmetic (levels hold fewer than 2^31 cells)
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= dc.nx * dc.ny * dc.nz) return;
    const int K = t % dc.nz, J = (t / dc.nz) % dc.ny, I = t / (dc.nz * dc.ny);
    // The 2x2x2 children share their inputs: each row (i, j) of the block
    // and its four side rows are read as (k0, k0+1) pairs (k0 even and the
    // fine rows even, so a pair is aligned; the z-faces' rows are odd and
    // read singly), 48 loads instead of 8 separate stencils' 112.  The
    // neighbours are clamped at the walls as in stencil().
    const int i0 = 2 * I, j0 = 2 * J, k0 = 2 * K;
    const int im = max(i0 - 1, 0), ip = min(i0 + 2, d.nx - 1);
    const int jm = max(j0 - 1, 0), jp = min(j0 + 2, d.ny - 1);
    const int km = max(k0 - 1, 0), kp = min(k0 + 2, d.nz - 1);
    // pc[a][bb][c]: the block; px[0|1][bb][c]: rows im / ip; py[a][0|1][c]:
    // rows jm / jp; pz[a][bb][0|1]: k0-1 / k0+2 of the block's rows
    float pc[2][2][2], px[2][2][2], py[2][2][2], pz[2][2][2];
    float fx[3][2][2], fy[2][3][2], fz[2][2][3], bv[2][2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int bb = 0; bb < 2; ++bb) {
            const int i = i0 + a, j = j0 + bb;
            ld_pair(p, cell_index(d, i, j, k0), pc[a][bb][0], pc[a][bb][1]);
            ld_pair(p, cell_index(d, a ? ip : im, j, k0), px[a][bb][0], px[a][bb][1]);
            ld_pair(p, cell_index(d, i, bb ? jp : jm, k0), py[a][bb][0], py[a][bb][1]);
            pz[a][bb][0] = to_f32(p[cell_index(d, i, j, km)]);
            pz[a][bb][1] = to_f32(p[cell_index(d, i, j, kp)]);
            ld_pair(b, cell_index(d, i, j, k0), bv[a][bb][0], bv[a][bb][1]);
            const int z = face_index<2>(d, i, j, k0);
            fz[a][bb][0] = to_f32(bz[z]);
            fz[a][bb][1] = to_f32(bz[z + 1]);
            fz[a][bb][2] = to_f32(bz[z + 2]);
        }
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int bb = 0; bb < 2; ++bb) {
            ld_pair(bx, face_index<0>(d, i0 + a, j0 + bb, k0), fx[a][bb][0], fx[a][bb][1]);
            ld_pair(by, face_index<1>(d, i0 + bb, j0 + a, k0), fy[bb][a][0], fy[bb][a][1]);
        }
    float acc = 0.0f;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int bb = 0; bb < 2; ++bb)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float f[6] = {fx[a][bb][c], fx[a + 1][bb][c], fy[a][bb][c],
                                    fy[a][bb + 1][c], fz[a][bb][c], fz[a][bb][c + 1]};
                // -x, +x, -y, +y, -z, +z (the sibling inside the block, or
                // the side row)
                const float pn[6] = {a ? pc[0][bb][c] : px[0][bb][c], a ? px[1][bb][c] : pc[1][bb][c],
                                     bb ? pc[a][0][c] : py[a][0][c], bb ? py[a][1][c] : pc[a][1][c],
                                     c ? pc[a][bb][0] : pz[a][bb][0], c ? pz[a][bb][1] : pc[a][bb][1]};
                float dg, Ap;
                stencil_vals(pc[a][bb][c], f, pn, dg, Ap);
                acc += bv[a][bb][c] * bs - Ap;
            }
    if (!skip) bc[t] = acc;
}

// P: piecewise-constant injection added onto the fine level (poisson.py:178-182)
// (pin and pout may be the same array)
template <typename ST, typename CT>
__global__ __launch_bounds__(RT) void k_prolong(Dims d, Dims dc, const ST* pin, ST* pout,
                                                const CT* __restrict__ pc, const int* __restrict__ done) {
    const bool skip = done && *done;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)d.nx * d.ny * d.nz) return;
    const int k = (int)(t % d.nz), j = (int)((t / d.nz) % d.ny), i = (int)(t / ((int64_t)d.nz * d.ny));
    const float v = to_f32(pin[t]) + to_f32(pc[cell_index(dc, i / 2, j / 2, k / 2)]);
    if (!skip) pout[t] = from_f32<ST>(v);
}

// ================================================================ one launch per smoothing phase
// A level's whole pre-smoothing phase (sweeps from zero, colour order (0,1),
// then the residual restricted to the coarse level) or whole post-smoothing
// phase (input pin plus the prolongation of the coarse iterate, colour order
// (1,0)) in one launch: a level of up to about 64^3 cells is bound by its
// launches' latency (about 5 us per sweep for 64^3 and for 32^3 alike), not
// by its bytes.  A workgroup owns a T x T x TK tile.  It holds the faces, b
// and diagonals of the tile plus an H-cell halo (two cells per sweep) in
// registers and their iterate in LDS, so no workgroup waits for another: each
// half-sweep runs on the region the tile's result still depends on (margin M
// of the box, one cell more per half-sweep) and repeats the neighbouring
// tiles' work there.
//  - The box's columns (x, y) are numbered from the tile outwards in rings,
//    so the columns at margin >= M are a prefix, and a thread's slots (pairs
//    of cells along k, one of each colour) drop out from the last one on.
//    Along k the whole column is updated; its ends beyond the margin are not
//    read again.
//  - The cells of even and odd k are in two arrays indexed by pair: one
//    colour's cells then cover all LDS banks, and every neighbour is at a
//    compile-time offset from one of two addresses.
//  - A face on a wall has weight 0 in the sum (its neighbour is the cell
//    itself, so its flux is 0) but counts in the diagonal; cells outside the
//    grid have diagonal 0 and keep their value.
// Every update has the operations of the per-sweep kernels in their order,
// so the results are bitwise those of the per-sweep path.
// VALU issue bounds it (the repeated updates are 4.7 times the tile's own at
// 64^3, 16.5 at 32^3), so the columns' indices and walls are worked out once
// per column, in LDS, and b is in LDS, which leaves the rest in registers.
// One phase of 3 sweeps with its restriction / prolongation, in the solve's
// graph: 64^3 15 / 15 us (one launch per sweep: 20 / 17), 32^3 8.6 / 7.8 us
// (faces and b in LDS instead of registers: 10 / 10).  FPCG iteration at
// 128^3 216 -> 207 us (BF16 212 -> 199), at 64^3 106 -> 99, at 32^3 78 -> 67.
template <int T, int TK, int NSW>
struct PhBox {
    static constexpr int NT = 1024;
    static constexpr int H = 2 * NSW;
    static constexpr int B = T + 2 * H, BM = (TK + 2 * H) / 2;  // box: B x B columns of BM pairs
    static constexpr int SY = BM, SX = B * BM, N = B * SX;      // LDS strides, pairs
    static constexpr int OFF = (N + 63) & ~63;                  // odd-k array behind the even one
    static constexpr int pairs(int M) { return (T + 2 * (H - M)) * (T + 2 * (H - M)) * BM; }  // at margin >= M
    static constexpr int slots(int M) { return (pairs(M) + NT - 1) / NT; }
    static_assert(T % 2 == 0 && TK % 2 == 0, "tiles restrict to whole coarse cells");
    static_assert((T & (T - 1)) == 0, "column numbering");
};

// column c of the ring numbering -> (x, y) in the box
template <typename BX, int T>
__device__ inline void ph_column(int c, int& x, int& y) {
    int s = 0;
#pragma unroll
    for (int r = 0; r < BX::H; ++r) s += c >= (T + 2 * r) * (T + 2 * r);
    const int in = T + 2 * (s - 1), e = T + 2 * s - 1;  // inner square's side, this ring's side - 1
    int r = c - in * in;
    const int lo = BX::H - s, hi = BX::H + T - 1 + s;
    const int w = (r >= e) + (r >= 2 * e) + (r >= 3 * e);
    r -= w * e;
    x = w == 0 ? lo : (w == 1 ? lo + r : (w == 2 ? hi : hi - r));
    y = w == 0 ? lo + r : (w == 1 ? hi : (w == 2 ? hi - r : lo));
    if (s == 0) {
        x = BX::H + c / T;
        y = BX::H + c % T;
    }
}

// two adjacent values as stored
template <typename ST>
struct RawPair {
    ST v[2];
    __device__ float get(bool second) const { return to_f32(second ? v[1] : v[0]); }
};

// a T at byte offset o of a uniform base (4-byte aligned; 2-byte for one
// 16-bit value)
template <typename T, typename B>
__device__ inline T at_byte(const B* base, unsigned o) {
    T v;
    __builtin_memcpy(&v, reinterpret_cast<const char*>(base) + o, sizeof(T));
    return v;
}

// One pair's data in registers, by colour: faces x-low, x-high, y-low,
// y-high of each cell; the z face between the cells and each cell's other
// one; b; the diagonal; the pair's LDS index * 2 + (x + y) & 1 (the k parity
// of its colour-0 cell).
struct PhSlot {
    float f[2][4], zm, zo[2], dg[2];
    int pk;
};

template <typename BX>
__device__ inline void ph_addr(int pk, int col, int& own, int& hi, bool& odd) {
    const int h = (pk ^ col) & 1, base = pk >> 1;
    odd = h != 0;
    own = base + h * BX::OFF;
    hi = base + BX::OFF + h * (1 - BX::OFF);  // the cell above along k; below: one entry before
}

template <typename BX>
__device__ inline void ph_stencil(const float* P, const PhSlot& S, int col, int own, int hi, bool odd, float pc,
                                  float& Ap) {
    const float f[6] = {S.f[col][0], S.f[col][1], S.f[col][2],
                        S.f[col][3], odd ? S.zm : S.zo[col], odd ? S.zo[col] : S.zm};
    const float pn[6] = {P[own - BX::SX], P[own + BX::SX], P[own - BX::SY],
                         P[own + BX::SY], P[hi - 1],       P[hi]};
    float dg;
    stencil_vals(pc, f, pn, dg, Ap);
}

// half-sweeps h .. 2*NSW-1 at margins M0 + h, colours c1, 1 - c1, ...; ZI: the
// first one starts from zero everywhere
template <typename ST, typename BX, int M0, int h, bool ZI, int NS>
__device__ inline void ph_sweeps(float* P, const float* B, PhSlot (&S)[NS], float omega) {
    if constexpr (h < BX::H) {
        constexpr int M = M0 + h;
#pragma unroll
        for (int q = 0; q < BX::slots(M); ++q) {
            // (the addresses are formed anew in every half-sweep: held, they spill)
            asm volatile("" : "+v"(S[q].pk));
            if ((q + 1) * BX::NT > BX::pairs(M) && (int)threadIdx.x + q * BX::NT >= BX::pairs(M)) continue;
            const int col = h & 1;  // slots are ordered by colour: first colour at [0]
            int own, hi;
            bool odd;
            ph_addr<BX>(S[q].pk, col, own, hi, odd);
            const float dg = S[q].dg[col];
            if constexpr (ZI && h == 0) {
                const float v = dg > 0.0f ? rb_first(B[own], dg, omega) : 0.0f;
                P[own] = round_st<ST>(v);
                P[odd ? hi - 1 : hi] = 0.0f;  // the pair's other cell
            } else {
                const float pc = P[own], bc = B[own];
                float Ap;
                ph_stencil<BX>(P, S[q], col, own, hi, odd, pc, Ap);
                // (formed unconditionally: every read is issued at once)
                const float v = rb_relax(pc, bc, Ap, dg, omega);
                P[own] = round_st<ST>(dg > 0.0f ? v : pc);
            }
        }
        __syncthreads();
        ph_sweeps<ST, BX, M0, h + 1, ZI, NS>(P, B, S, omega);
    }
}

// PRE: pin is unused (the level starts from zero), pout gets the smoothed
// iterate and bc the restricted residual (k_resid_restrict's order); uf: the
// residual test rides along (level 0).  !PRE: pout gets the post-smoothed
// iterate of pin + P pcoarse; df: with the CG's inner products (level 0).
template <typename ST, bool PRE, int T, int TK, int NSW, typename CT = float>
__global__ __launch_bounds__(1024) void k_phase(Dims d, Dims dc, const ST* __restrict__ bx,
                                                const ST* __restrict__ by, const ST* __restrict__ bz,
                                                const float* __restrict__ b, const ST* __restrict__ pin,
                                                const CT* __restrict__ pcoarse, ST* __restrict__ pout,
                                                float* __restrict__ bc, float omega,
                                                const int* __restrict__ done, const float* __restrict__ bscale,
                                                UpdateFold uf, DotFold df) {
    using BX = PhBox<T, TK, NSW>;
    constexpr int M0 = PRE ? 0 : 1, NS = BX::slots(M0), H = BX::H, NT = BX::NT;
    constexpr int c1 = PRE ? 0 : 1;
    __shared__ float P[2 * BX::OFF], B[2 * BX::OFF];
    const int tid = threadIdx.x;
    const bool fold = PRE && uf.st != nullptr;
    int was_done = 0;
    float fm = 0.0f;
    if (fold) {
        was_done = uf.st->done;
        for (int e = tid; e < uf.nparts; e += NT) fm = fmaxf(fm, uf.st->fpart[e]);
    }
    const int ntk = (d.nz + TK - 1) / TK, ntj = (d.ny + T - 1) / T;
    const int tile = xcd_block(blockIdx.x, gridDim.x);
    const int i0 = (tile / (ntk * ntj)) * T, j0 = ((tile / ntk) % ntj) * T, k0 = (tile % ntk) * TK;
    const int ox = i0 - H, oy = j0 - H, oz = k0 - H;  // even

    // staging of the iterate (every pair of the box, from clamped coordinates)
    constexpr int NST = PRE ? 1 : (BX::N + NT - 1) / NT;
    RawPair<ST> lp[NST];
    CT lc[NST];
    if constexpr (!PRE) {
#pragma unroll
        for (int q = 0; q < NST; ++q) {
            const int e = min(tid + q * NT, BX::N - 1);
            const int m = e % BX::BM, y = (e / BX::BM) % BX::B, x = e / BX::SX;
            const int gi = min(max(ox + x, 0), d.nx - 1), gj = min(max(oy + y, 0), d.ny - 1),
                      gk = min(max(oz + 2 * m, 0), d.nz - 2);
            lp[q] = at_byte<RawPair<ST>>(pin, (unsigned)cell_index(d, gi, gj, gk) * sizeof(ST));
            lc[q] = at_byte<CT>(pcoarse, (unsigned)cell_index(dc, gi >> 1, gj >> 1, gk >> 1) * sizeof(CT));
        }
    }
    // the box's columns: their first cell's index, what leads from a cell to
    // its y and z faces, and the column's LDS index * 2 + the k parity of the
    // first colour's cells, with the walls in bits 20-23 (low x, high x, low
    // y, high y) and bit 26: outside the grid
    constexpr int NC = BX::pairs(M0) / BX::BM;
    __shared__ uint4 col[NC];
    static_assert(2 * BX::N < 1 << 20 && NC <= NT, "column word");
    if (tid < NC) {
        int x, y;
        ph_column<BX, T>(tid, x, y);
        const int i = min(max(ox + x, 0), d.nx - 1), j = min(max(oy + y, 0), d.ny - 1);
        const unsigned walls = (i == 0) | (i == d.nx - 1) << 1 | (j == 0) << 2 | (j == d.ny - 1) << 3 |
                               (unsigned)(i != ox + x || j != oy + y) << 6;
        col[tid] = make_uint4((i * d.ny + j) * d.nz, i * d.nz, i * d.ny + j,
                              (2 * (x * BX::SX + y * BX::SY) + ((x + y + c1) & 1)) | walls << 20);
    }
    __syncthreads();
    // the slots: every load from clamped coordinates (byte offsets of 32 bits
    // from uniform bases), all issued before the first use
    PhSlot S[NS];
    RawPair<ST> rx[NS][2], ry[NS][2];
    ST rz[NS][3];
    float2 rb[NS];
    unsigned wall[NS];
    float2 ap = make_float2(0.0f, 0.0f);
#pragma unroll
    for (int q = 0; q < NS; ++q) {
        const int t = min(tid + q * NT, BX::pairs(M0) - 1);
        const int c = t / BX::BM, m = t - c * BX::BM;
        const uint4 cl = col[c];
        const int kb = oz + 2 * m, k = min(max(kb, 0), d.nz - 2);
        const unsigned cell = cl.x + k, fy = cell + cl.y, fz = cell + cl.z;
        rx[q][0] = at_byte<RawPair<ST>>(bx, cell * sizeof(ST));
        rx[q][1] = at_byte<RawPair<ST>>(bx, (cell + d.ny * d.nz) * sizeof(ST));
        ry[q][0] = at_byte<RawPair<ST>>(by, fy * sizeof(ST));
        ry[q][1] = at_byte<RawPair<ST>>(by, (fy + d.nz) * sizeof(ST));
#pragma unroll
        for (int e = 0; e < 3; ++e) rz[q][e] = at_byte<ST>(bz, (fz + e) * sizeof(ST));
        rb[q] = at_byte<float2>(b, cell * 4u);
        if (!PRE && q == 0 && df.Ap) ap = at_byte<float2>(df.Ap, cell * 4u);
        S[q].pk = (int)(cl.w & 0xFFFFFu) + 2 * m;
        wall[q] = (cl.w >> 20) | (k == 0) << 4 | (k == d.nz - 2) << 5 | (k != kb) << 6;
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!PRE) {
#pragma unroll
        for (int q = 0; q < NST; ++q) {
            const int e = tid + q * NT;
            if (e < BX::N) {
                P[e] = round_st<ST>(lp[q].get(false) + to_f32(lc[q]));
                P[e + BX::OFF] = round_st<ST>(lp[q].get(true) + to_f32(lc[q]));
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < NS; ++q) {
        const int par = S[q].pk & 1;
        const unsigned wl = wall[q];
        const float z[3] = {to_f32(rz[q][0]), to_f32(rz[q][1]), to_f32(rz[q][2])};
#pragma unroll
        for (int col = 0; col < 2; ++col) {
            const bool odd = (par ^ col) != 0;
            const float fc[6] = {rx[q][0].get(odd), rx[q][1].get(odd), ry[q][0].get(odd),
                                 ry[q][1].get(odd), odd ? z[1] : z[0], odd ? z[2] : z[1]};
            const float dg = fc[0] + fc[1] + fc[2] + fc[3] + fc[4] + fc[5];
            S[q].dg[col] = dg;
#pragma unroll
            for (int e = 0; e < 4; ++e) S[q].f[col][e] = fc[e];
            S[q].zo[col] = odd ? z[2] : z[0];
        }
        // bits 0-5: the pair has a wall on the low / high side of an axis;
        // 6: it lies outside the grid
        if (__any(wl)) {
#pragma unroll
            for (int col = 0; col < 2; ++col) {
                const bool odd = (par ^ col) != 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) S[q].f[col][e] = (wl >> e & 1u) ? 0.0f : S[q].f[col][e];
                S[q].zo[col] = (wl & (odd ? 32u : 16u)) ? 0.0f : S[q].zo[col];
                S[q].dg[col] = (wl & 64u) ? 0.0f : S[q].dg[col];
            }
        }
        S[q].zm = z[1];
        // (b: written and read by this thread alone, unscaled until bs is known)
        if (tid + q * NT < BX::pairs(M0)) {
            B[S[q].pk >> 1] = rb[q].x;
            B[(S[q].pk >> 1) + BX::OFF] = rb[q].y;
        }
#pragma unroll
        for (int col = 0; col < 2; ++col)  // formed here and now, not at every use
            asm volatile("" : "+v"(S[q].f[col][0]), "+v"(S[q].f[col][1]), "+v"(S[q].f[col][2]), "+v"(S[q].f[col][3]),
                              "+v"(S[q].zo[col]), "+v"(S[q].dg[col]));
    }
    bool skip = !fold && done && *done;
    __shared__ float s_fm[NT / 64];
    if (fold) {
        fm = wave_max(fm);
        if ((tid & 63) == 0) s_fm[tid >> 6] = fm;
        __syncthreads();
    }
    float bs = 1.0f;
    if (fold) {
        float mm = s_fm[0];
#pragma unroll
        for (int w = 1; w < NT / 64; ++w) mm = fmaxf(mm, s_fm[w]);
        const bool conv = (double)mm / uf.st->b_norm < uf.st->tol;
        skip = was_done || conv;
        bs = ldexpf(1.0f, -vscale_exponent(mm));
        if (blockIdx.x == 0 && tid == 0) residual_test_record(uf.st, mm, uf.host_flag);
    } else if (bscale) {
        bs = *bscale;
    }
    if (skip) return;  // a finished solve's queued iteration (uniform)
    if (bscale) {
#pragma unroll
        for (int q = 0; q < NS; ++q) {
            if (tid + q * NT < BX::pairs(M0)) {
                B[S[q].pk >> 1] *= bs;
                B[(S[q].pk >> 1) + BX::OFF] *= bs;
            }
        }
    }
    if (!PRE) __syncthreads();
    // PRE: the first half-sweep from zero runs on the whole box (it reads no
    // neighbour), the last at margin H - 1; !PRE: margins 1 .. H
    ph_sweeps<ST, BX, M0, 0, PRE, NS>(P, B, S, omega);

    // the tile goes out: its pairs are all in slot 0
    static_assert(T * T * BX::BM <= NT, "the tile's columns fit slot 0");
    const int col0 = tid / BX::BM, m = tid - col0 * BX::BM;
    const int il = col0 / T, jl = col0 % T, kl = 2 * m - H;
    const bool mine = tid < T * T * BX::BM && kl >= 0 && kl < TK && i0 + il < d.nx && j0 + jl < d.ny && k0 + kl < d.nz;
    __shared__ float Rs[PRE ? T * T * TK : 1];
    double dsum[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (mine) {
        const int base = S[0].pk >> 1;
        const float p0 = P[base], p1 = P[base + BX::OFF];
        st_pair(pout, cell_index(d, i0 + il, j0 + jl, k0 + kl), p0, p1);
        if constexpr (PRE) {
#pragma unroll
            for (int col = 0; col < 2; ++col) {
                int own, hi;
                bool odd;
                ph_addr<BX>(S[0].pk, col, own, hi, odd);
                float Ap;
                ph_stencil<BX>(P, S[0], col, own, hi, odd, odd ? p1 : p0, Ap);
                Rs[(il * T + jl) * TK + kl + (odd ? 1 : 0)] = B[own] - Ap;
            }
        } else if (df.Ap) {
            // k_cg_beta's sums: z as stored times zscale, r = b unscaled, Ap
            const float zsc = df.zscale ? *df.zscale : 1.0f;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const double zz = (double)((e ? p1 : p0) * zsc);
                const double rr = (double)(B[base + e * BX::OFF] * zsc);
                const double aa = (double)(e ? ap.y : ap.x);
                dsum[0] += zz;
                dsum[1] += rr;
                dsum[2] += aa;
                dsum[3] += rr * zz;
                dsum[4] += aa * zz;
            }
        }
    }
    if constexpr (PRE) {
        __syncthreads();
        constexpr int CJ = T / 2, CK = TK / 2;
        for (int e = tid; e < T * T * TK / 8; e += NT) {
            const int K = e % CK, J = (e / CK) % CJ, I = e / (CK * CJ);
            const int gI = i0 / 2 + I, gJ = j0 / 2 + J, gK = k0 / 2 + K;
            if (gI >= dc.nx || gJ >= dc.ny || gK >= dc.nz) continue;
            float acc = 0.0f;
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int bb = 0; bb < 2; ++bb)
#pragma unroll
                    for (int c = 0; c < 2; ++c) acc += Rs[((2 * I + a) * T + 2 * J + bb) * TK + 2 * K + c];
            bc[cell_index(dc, gI, gJ, gK)] = acc;
        }
    } else if (df.Ap) {
        __shared__ double s_dot[5 * 16];
        block_sum<5>(dsum, s_dot);
        if (tid == 0) {
#pragma unroll
            for (int q = 0; q < 5; ++q) df.st->part[q * PS + blockIdx.x] = dsum[q];
            if (blockIdx.x == 0) df.st->beta_parts = 1;  // read by the next k_cg_apply
        }
    }
}

// ================================================================ reductions
// Reductions are fence-free: a kernel writes one partial per block, and a
// one-block combine kernel (k_comb) forms the scalar.  The kernel boundary
// orders the two, so no device-scope fence (an L2 write-back per block on
// this multi-XCD part) is needed, and the fixed combine order keeps every
// result bitwise reproducible.
template <typename T>
__global__ __launch_bounds__(RT) void k_part_sum(const T* __restrict__ x, int64_t n, double* part) {
    __shared__ double sh[16];
    double v[1] = {0.0};
    for (int64_t c = (int64_t)blockIdx.x * RT + threadIdx.x; c < n; c += (int64_t)gridDim.x * RT)
        v[0] += (double)to_f32(x[c]);
    block_sum<1>(v, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = v[0];
}

// y = x + shift (FP32 shift of the FP64 mean, as _remove_mean's shift_kernel)
template <typename TI, typename TO>
__global__ __launch_bounds__(RT) void k_shift(const TI* x, TO* y, int64_t n, const double* mean) {
    const float c = (float)(-*mean);
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < n; i += (int64_t)gridDim.x * RT)
        y[i] = from_f32<TO>(to_f32(x[i]) + c);
}

template <typename T>
__global__ __launch_bounds__(RT) void k_zero(T* x, int64_t n, const int* __restrict__ done) {
    if (done && *done) return;
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < n; i += (int64_t)gridDim.x * RT)
        x[i] = from_f32<T>(0.0f);
}

// ================================================================ levels of one workgroup
constexpr int kSmallThreads = 1024;

// A level (or all of a coarsest one) held by one workgroup: thread t has the
// pairs of cells along k t, t + 1024, ... (row * nkp + kp), one cell of each
// colour per pair, with their faces, b and omega / diag in registers.  Only
// the iterate is in LDS, the cells of even and of odd k in two arrays indexed
// by pair: one colour's cells of a row then lie next to each other, and a
// wave's reads fall on all LDS banks (in cell order one colour uses every
// other bank: 108 us instead of 69 for 60 sweeps of 26 x 19 x 13 cells).
// Faces on a wall are given weight 0 in the sum (their neighbour is the cell
// itself, so their flux is 0; they stay in the diagonal), so the neighbour
// addresses need no clamps: zeros on either side of the arrays keep them
// inside.  ZL: the low z faces are in LDS too (a cell's high z face is the
// next cell's low one), which holds 8 pairs per thread without spilling in
// the sweeps.
struct PairGeom {
    Dims d;
    int nkp, npair, SP, OFF;  // pairs per row / in all; pairs per i; the odd array behind the even one
};

// floats from the even-k array to the odd-k one: the pairs, with room on both
// sides, in whole rounds of the LDS banks
__host__ __device__ inline int pair_stride(const Dims& d) {
    const int nkp = (d.nz + 1) >> 1;
    return (d.nx * d.ny * nkp + 2 * d.ny * nkp + 63) & ~63;
}

__device__ inline PairGeom pair_geom(const Dims& d) {
    PairGeom g;
    g.d = d;
    g.nkp = (d.nz + 1) >> 1;
    g.npair = d.nx * d.ny * g.nkp;
    g.SP = d.ny * g.nkp;
    g.OFF = pair_stride(d);
    return g;
}

template <int KP, bool ZL>
struct RegPairs {
    static constexpr int NF = ZL ? 4 : 6;
    int own0[KP];  // index of the pair's colour-0 cell; -1: no pair
    float f[2][KP][NF], rb[2][KP];
    float w[2][KP];  // omega / diag; 0: a cell that is never updated (none there, or no faces)

    // cell of colour col of a pair with colour-0 index own0: its index in
    // the pair arrays, and that of the cell above along k (below: one before)
    __device__ inline void cell(const PairGeom& g, int q, int col, int& c, int& hi) const {
        const int t = (int)threadIdx.x + q * kSmallThreads;
        c = col == 0 ? own0[q] : 2 * t + g.OFF - own0[q];
        hi = c == t ? t + g.OFF : t + 1;
    }

    __device__ inline void load(const PairGeom& g, const float* __restrict__ bx, const float* __restrict__ by,
                                const float* __restrict__ bz, float omega, float* Z) {
        const Dims& d = g.d;
        const int SJ = d.nz, SI = d.ny * d.nz;
#pragma unroll
        for (int q = 0; q < KP; ++q) {
            const int t = (int)threadIdx.x + q * kSmallThreads, tc = min(t, g.npair - 1);
            const int row = tc / g.nkp, kp = tc - row * g.nkp;
            const int i = row / d.ny, j = row - i * d.ny;
            const int par = (i + j) & 1;  // k = 2 kp + par has colour 0
            own0[q] = t < g.npair ? t + (par ? g.OFF : 0) : -1;
#pragma unroll
            for (int col = 0; col < 2; ++col) {
                const int kk = 2 * kp + (par ^ col), k = min(kk, d.nz - 1);
                const int c = row * d.nz + k;
                const int fy = c + i * d.nz, fz = c + row;
                float v[6] = {bx[c], bx[c + SI], by[fy], by[fy + SJ], bz[fz], bz[fz + 1]};
                const float dg = v[0] + v[1] + v[2] + v[3] + v[4] + v[5];
                const bool own = t < g.npair && kk < d.nz;
                if (i == 0) v[0] = 0.0f;
                if (i == d.nx - 1) v[1] = 0.0f;
                if (j == 0) v[2] = 0.0f;
                if (j == d.ny - 1) v[3] = 0.0f;
                if (k == 0) v[4] = 0.0f;
                if (k == d.nz - 1) v[5] = 0.0f;
#pragma unroll
                for (int m = 0; m < NF; ++m) f[col][q][m] = v[m];
                if (ZL && t < g.npair) Z[t + ((par ^ col) ? g.OFF : 0)] = own ? v[4] : 0.0f;
                w[col][q] = own && dg > 0.0f ? omega / dg : 0.0f;
            }
        }
    }

    // cell index (i ny + j) nz + k of a pair's cell of either colour; nz odd:
    // the last pair of a row has no odd cell (exists = false)
    __device__ inline int grid_cell(const PairGeom& g, int q, int col, bool& exists) const {
        const int t = (int)threadIdx.x + q * kSmallThreads;
        const int row = t / g.nkp, kp = t - row * g.nkp;
        const bool odd = (own0[q] != t) != (col != 0);
        const int k = 2 * kp + (odd ? 1 : 0);
        exists = own0[q] >= 0 && k < g.d.nz;
        return row * g.d.nz + k;
    }

    // the right-hand side, in cell order
    __device__ inline void load_b(const PairGeom& g, const float* b) {
#pragma unroll
        for (int q = 0; q < KP; ++q)
#pragma unroll
            for (int col = 0; col < 2; ++col) {
                bool ex;
                const int c = grid_cell(g, q, col, ex);
                rb[col][q] = ex ? b[c] : 0.0f;
            }
    }

    // A p at a cell (stencil_vals' operations)
    __device__ inline float Ap(const PairGeom& g, const float* P, const float* Z, int q, int col, int c, int hi,
                               float pc) const {
#pragma clang fp contract(off)
        const float* p = P + c;
        float s = f[col][q][0] * (pc - p[-g.SP]);
        s = fmaf(f[col][q][1], pc - p[g.SP], s);
        s = fmaf(f[col][q][2], pc - p[-g.nkp], s);
        s = fmaf(f[col][q][3], pc - p[g.nkp], s);
        s = fmaf(ZL ? Z[c] : f[col][q][NF - 2], pc - P[hi - 1], s);
        s = fmaf(ZL ? Z[hi] : f[col][q][NF - 1], pc - P[hi], s);
        return s;
    }

    // AHEAD: every pair's reads before the first write (cells of one colour
    // never neighbour each other).  Two pairs in a row of 60 sweeps: 6x22x16
    // 59 -> 47 us; in the V-cycle's 3 + 3 it costs 1 us of 29.
    template <bool AHEAD = false>
    __device__ inline void half(const PairGeom& g, float* P, const float* Z, int col) {
        if constexpr (AHEAD) {
            int c[KP], hi;
            float v[KP];
#pragma unroll
            for (int q = 0; q < KP; ++q) {
                c[q] = -1;
                if (own0[q] < 0 || w[col][q] == 0.0f) continue;
                cell(g, q, col, c[q], hi);
                const float pc = P[c[q]];
                v[q] = fmaf(rb[col][q] - Ap(g, P, Z, q, col, c[q], hi, pc), w[col][q], pc);
            }
#pragma unroll
            for (int q = 0; q < KP; ++q)
                if (c[q] >= 0) P[c[q]] = v[q];
            return;
        }
#pragma unroll
        for (int q = 0; q < KP; ++q) {
            // many pairs: form the addresses anew each time (kept across the
            // loop they spill)
            if constexpr (KP >= 5) asm volatile("" : "+v"(own0[q]));
            if (own0[q] < 0 || w[col][q] == 0.0f) continue;
            int c, hi;
            cell(g, q, col, c, hi);
            const float pc = P[c];
            P[c] = fmaf(rb[col][q] - Ap(g, P, Z, q, col, c, hi, pc), w[col][q], pc);
        }
    }
};

// ================================================================ small levels in LDS
struct SmallArgs {
    int s, L, pre, post;
    int nreg;  // levels s .. s + nreg - 1 are held in registers (RegPairs), the rest in LDS
    float omega;
    Dims d[PF_MAX_LEVELS];
    int off[PF_MAX_LEVELS][5];  // LDS float offsets of bx, by, bz, p, b (register levels: p and b, not s)
    int poff[2];                // and of the register levels' pair arrays
    int scratch;                // LDS float offset of the residual scratch
    const float* rf[2][3];      // the register levels' faces
    const float* b_top;
    // global -> LDS copies at entry: segment q copies seg_len[q] floats from
    // seg_src[q] to LDS offset seg_dst[q] (the LDS levels' faces, b of a
    // hierarchy without register levels, the coarsest level's matrix)
    int nseg;
    const float* seg_src[3 * PF_MAX_LEVELS + 2];
    int seg_dst[3 * PF_MAX_LEVELS + 2];
    int seg_len[3 * PF_MAX_LEVELS + 2];
    void* p_top;
    const int* done;
    const double* cop;  // the coarsest level's smoother as a matrix
    int cop_lds;        // >= 0: LDS float offset of a staged copy of that matrix
};

constexpr int kTopPairs = 2;  // pairs of cells per thread on the largest level

// Pairs along k of a level.  The largest level of the single-workgroup V-cycle
// has at most kSmallThreads * kTopPairs of them (4096 cells), so the third
// one, the first in LDS, at most 64 cells: 32 pairs, smoothed by one wave.
__host__ __device__ inline int colour_space(const Dims& d) { return d.nx * d.ny * ((d.nz + 1) >> 1); }

// floor(t / d) for 0 <= t < 2^22 and 1 <= d, with inv = 1.0f / d: t + 1/2
// stays at least 1/(2d) away from a multiple of d, far more than the float
// rounding of the product.
__device__ inline int fdiv(int t, float inv) { return (int)(((float)t + 0.5f) * inv); }

struct LdsLevel {
    Dims d;
    float* bx;
    float* by;
    float* bz;
    float* p;
    float* b;
};

__device__ inline LdsLevel lds_level(const SmallArgs& a, float* lds, int l) {
    LdsLevel v;
    v.d = a.d[l];
    v.bx = lds + a.off[l][0];
    v.by = lds + a.off[l][1];
    v.bz = lds + a.off[l][2];
    v.p = lds + a.off[l][3];
    v.b = lds + a.off[l][4];
    return v;
}

// One cell that a thread updates on one level, decoded once per level visit:
// its index, the indices of its six neighbours with the reference's clamp at
// the walls (a missing neighbour is the cell itself), its y / z low faces
// (the x low face shares the cell index), its parent on the next coarser
// level, its right-hand side and omega / diag (0 where diag <= 0: no update).
struct Slot {
    int c, n[6], par;
    float f[6];  // x-low, x-high, y-low, y-high, z-low, z-high faces
    float b, w;
};

__device__ inline void make_slot(const LdsLevel& v, int colour, int t, float omega, const Dims* dc, Slot& S) {
    const Dims& d = v.d;
    const int nkp = (d.nz + 1) >> 1;
    S.c = -1;
    if (t >= d.nx * d.ny * nkp) return;
    const int row = fdiv(t, 1.0f / (float)nkp), kp = t - row * nkp;
    const int i = fdiv(row, 1.0f / (float)d.ny), j = row - i * d.ny;
    const int k = 2 * kp + ((i + j + colour) & 1);
    if (k >= d.nz) return;
    const int SI = d.ny * d.nz, SJ = d.nz;
    const int c = (i * d.ny + j) * d.nz + k;
    S.c = c;
    S.n[0] = i > 0 ? c - SI : c;
    S.n[1] = i < d.nx - 1 ? c + SI : c;
    S.n[2] = j > 0 ? c - SJ : c;
    S.n[3] = j < d.ny - 1 ? c + SJ : c;
    S.n[4] = k > 0 ? c - 1 : c;
    S.n[5] = k < d.nz - 1 ? c + 1 : c;
    const int fy = c + i * d.nz;        // face_index<1>(d, i, j, k)
    const int fz = c + (i * d.ny + j);  // face_index<2>(d, i, j, k)
    S.par = dc ? cell_index(*dc, i >> 1, j >> 1, k >> 1) : 0;
    S.f[0] = v.bx[c];
    S.f[1] = v.bx[c + SI];
    S.f[2] = v.by[fy];
    S.f[3] = v.by[fy + SJ];
    S.f[4] = v.bz[fz];
    S.f[5] = v.bz[fz + 1];
    const float dg = S.f[0] + S.f[1] + S.f[2] + S.f[3] + S.f[4] + S.f[5];
    S.b = v.b[c];
    S.w = dg > 0.0f ? omega / dg : 0.0f;
}

// A p at a slot's cell in the difference form (stencil_vals' operations)
__device__ inline float slot_Ap(const LdsLevel& v, const Slot& S, float pc) {
#pragma clang fp contract(off)
    float s = S.f[0] * (pc - v.p[S.n[0]]);
    s = fmaf(S.f[1], pc - v.p[S.n[1]], s);
    s = fmaf(S.f[2], pc - v.p[S.n[2]], s);
    s = fmaf(S.f[3], pc - v.p[S.n[3]], s);
    s = fmaf(S.f[4], pc - v.p[S.n[4]], s);
    s = fmaf(S.f[5], pc - v.p[S.n[5]], s);
    return s;
}

// One half-sweep of a wave's slots (cells of one colour never neighbour each
// other, and a wave's reads are all issued before its writes).
__device__ inline void slot_sweep(const LdsLevel& v, const Slot& S) {
    if (S.c < 0) return;
    const float pc = v.p[S.c];
    v.p[S.c] = pc + (S.b - slot_Ap(v, S, pc)) * S.w;
}

__device__ inline void wave_sync() {
    // LDS operations of one wave execute in issue order; this only keeps the
    // compiler from moving LDS accesses across the colour boundary
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Workgroup barrier over LDS only: unlike __syncthreads it does not wait
// for loads in flight, so the coarser levels' staging overlaps the top
// level's descent.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The slots of both colours of one LDS level for this thread (colour c0
// first); the threads beyond the first wave have none.
struct LevelSlots {
    Slot s0, s1;
};

__device__ inline void make_level_slots(const LdsLevel& v, int c0, float omega, const Dims* dc, LevelSlots& L) {
    L.s0.c = L.s1.c = -1;
    if (threadIdx.x < 64) {
        make_slot(v, c0, threadIdx.x, omega, dc, L.s0);
        make_slot(v, 1 - c0, threadIdx.x, omega, dc, L.s1);
    }
}

// `sweeps` red-black sweeps (colour c0 first); ends with a workgroup barrier
__device__ inline void small_smooth(const LdsLevel& v, const LevelSlots& L, int sweeps) {
    if (threadIdx.x < 64)
        for (int sw = 0; sw < sweeps; ++sw) {
            slot_sweep(v, L.s0);
            wave_sync();
            slot_sweep(v, L.s1);
            wave_sync();
        }
    lds_barrier();
}

// One register level's way down: smooth from zero (pair arrays cleared, b
// loaded), then the residual restricted into the next level's b (cell order).
template <int KP>
__device__ inline void reg_descend(RegPairs<KP, false>& R, const PairGeom& g, float* P, int sweeps, float* scr,
                                   const Dims& dc, float* bc) {
    for (int sw = 0; sw < sweeps; ++sw) {
        R.half(g, P, nullptr, 0);
        lds_barrier();
        R.half(g, P, nullptr, 1);
        lds_barrier();
    }
#pragma unroll
    for (int q = 0; q < KP; ++q)
#pragma unroll
        for (int col = 0; col < 2; ++col) {
            bool ex;
            const int gc = R.grid_cell(g, q, col, ex);
            if (!ex) continue;
            int c, hi;
            R.cell(g, q, col, c, hi);
            scr[gc] = R.rb[col][q] - R.Ap(g, P, nullptr, q, col, c, hi, P[c]);
        }
    lds_barrier();
    const int nc = dc.nx * dc.ny * dc.nz;
    const float inz = 1.0f / (float)dc.nz, iny = 1.0f / (float)dc.ny;
    for (int t = threadIdx.x; t < nc; t += kSmallThreads) {
        const int row = fdiv(t, inz), K = t - row * dc.nz;
        const int I = fdiv(row, iny), J = row - I * dc.ny;
        float acc = 0.0f;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int z = 0; z < 2; ++z) acc += scr[cell_index(g.d, 2 * I + x, 2 * J + y, 2 * K + z)];
        bc[t] = acc;
    }
    lds_barrier();
}

// and its way up: add the parents (cell order; a pair's two cells share one),
// smooth with colours (1,0)
template <int KP>
__device__ inline void reg_ascend(RegPairs<KP, false>& R, const PairGeom& g, float* P, int sweeps, const Dims& dc,
                                  const float* pc) {
#pragma unroll
    for (int q = 0; q < KP; ++q) {
        if (R.own0[q] < 0) continue;
        const int t = (int)threadIdx.x + q * kSmallThreads;
        const int row = t / g.nkp, kp = t - row * g.nkp;
        const int i = row / g.d.ny, j = row - i * g.d.ny;
        const float v = pc[cell_index(dc, i >> 1, j >> 1, kp)];
        P[t] += v;
        P[t + g.OFF] += v;
    }
    lds_barrier();
    for (int sw = 0; sw < sweeps; ++sw) {
        R.half(g, P, nullptr, 1);
        lds_barrier();
        R.half(g, P, nullptr, 0);
        lds_barrier();
    }
}

// p of a register level to an array in cell order
template <int KP, typename OT>
__device__ inline void reg_store(const RegPairs<KP, false>& R, const PairGeom& g, const float* P, OT* out) {
#pragma unroll
    for (int q = 0; q < KP; ++q)
#pragma unroll
        for (int col = 0; col < 2; ++col) {
            bool ex;
            const int gc = R.grid_cell(g, q, col, ex);
            if (!ex) continue;
            int c, hi;
            R.cell(g, q, col, c, hi);
            out[gc] = from_f32<OT>(P[c]);
        }
}

// The whole V-cycle from level s down in one workgroup.  The two largest
// levels (16^3 and 8^3 of a 128^3 grid) keep their cells' faces, b and
// omega / diag in registers, loaded straight from memory once and used on the
// way down and up; smaller ones are in LDS, decoded per visit.  The coarsest
// level is a matrix product (any hierarchy that gets here has at most
// kCoarseOpMax coarsest cells).
// Latency of one CU bounds it.  From 16^3 down, in the solve's graphs of a
// 128^3 / 32^3 grid: 21.8 / 19.8 us; with every level's faces staged in LDS
// and its cells decoded on each visit 27.2 / 25.2.
template <typename OT>
__global__ __launch_bounds__(kSmallThreads) void k_small_vcycle(SmallArgs a) {
    extern __shared__ float lds[];
    const int tid = threadIdx.x, nt = kSmallThreads;
    const int dn = a.done ? *a.done : 0;
    // segments straight from memory into LDS (lane l of a wave writes its
    // dword to the wave's LDS base + 4 l)
    for (int q = 0; q < a.nseg; ++q) {
        const float* src = a.seg_src[q];
        const int len = a.seg_len[q];
        float* dst = lds + a.seg_dst[q];
        for (int e0 = 0; e0 < len; e0 += nt)
            if (e0 + tid < len)
                __builtin_amdgcn_global_load_lds(
                    (const void*)(src + e0 + tid), (__attribute__((address_space(3))) void*)(dst + e0 + (tid & ~63)),
                    4, 0, 0);
    }
    if (dn) {
        __builtin_amdgcn_s_waitcnt(0);  // nothing may land in LDS after the workgroup has gone
        return;                         // uniform: no workgroup barrier has been reached yet
    }
    float* scr = lds + a.scratch;
    const PairGeom g0 = pair_geom(a.d[a.s]), g1 = pair_geom(a.d[a.nreg > 1 ? a.s + 1 : a.s]);
    float* P0 = lds + a.poff[0] + g0.SP;
    float* P1 = lds + a.poff[1] + g1.SP;
    RegPairs<kTopPairs, false> R0;
    RegPairs<1, false> R1;
    if (a.nreg > 0) {
        R0.load(g0, a.rf[0][0], a.rf[0][1], a.rf[0][2], a.omega, nullptr);
        R0.load_b(g0, a.b_top);
        for (int e = tid; e < 2 * g0.OFF; e += nt) lds[a.poff[0] + e] = 0.0f;
    }
    if (a.nreg > 1) {
        R1.load(g1, a.rf[1][0], a.rf[1][1], a.rf[1][2], a.omega, nullptr);
        for (int e = tid; e < 2 * g1.OFF; e += nt) lds[a.poff[1] + e] = 0.0f;
    }
    __builtin_amdgcn_s_waitcnt(0);
    lds_barrier();
    LevelSlots S;
    // descend: smooth from zero, restrict the residual (poisson.py:323-336)
    if (a.nreg > 0) reg_descend(R0, g0, P0, a.pre, scr, a.d[a.s + 1], lds + a.off[a.s + 1][4]);
    if (a.nreg > 1) {
        R1.load_b(g1, lds + a.off[a.s + 1][4]);
        reg_descend(R1, g1, P1, a.pre, scr, a.d[a.s + 2], lds + a.off[a.s + 2][4]);
    }
    for (int l = a.s + a.nreg; l < a.L - 1; ++l) {
        const LdsLevel v = lds_level(a, lds, l);
        const LdsLevel c = lds_level(a, lds, l + 1);
        const int n = v.d.nx * v.d.ny * v.d.nz;
        for (int e = tid; e < n; e += nt) v.p[e] = 0.0f;
        make_level_slots(v, 0, a.omega, &c.d, S);
        lds_barrier();
        small_smooth(v, S, a.pre);
        // residual of every fine cell into the scratch, then R = P^T
        if (S.s0.c >= 0) scr[S.s0.c] = S.s0.b - slot_Ap(v, S.s0, v.p[S.s0.c]);
        if (S.s1.c >= 0) scr[S.s1.c] = S.s1.b - slot_Ap(v, S.s1, v.p[S.s1.c]);
        lds_barrier();
        const int nc = c.d.nx * c.d.ny * c.d.nz;
        for (int t = tid; t < nc; t += nt) {
            const int K = t % c.d.nz, J = (t / c.d.nz) % c.d.ny, I = t / (c.d.nz * c.d.ny);
            float acc = 0.0f;
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y)
#pragma unroll
                    for (int z = 0; z < 2; ++z) acc += scr[cell_index(v.d, 2 * I + x, 2 * J + y, 2 * K + z)];
            c.b[t] = acc;
        }
        lds_barrier();
    }
    // coarsest: sweeps, then the mean removed (poisson.py:325-328), as the
    // precomputed matrix: p = M b (column j of M contiguous).  Each output's
    // sum is split over G groups of n threads (a contiguous range of j each;
    // a wave reads 64 consecutive entries of one column), and the G partials
    // are added in group order (the FP64 partials go through the scratch,
    // 8-byte aligned).
    {
        const LdsLevel v = lds_level(a, lds, a.L - 1);
        const int n = v.d.nx * v.d.ny * v.d.nz;
        const int G = min(nt / n, 16), J = (n + G - 1) / G;
        double* part = reinterpret_cast<double*>(scr);
        // (one instance per memory kind, so the loads are LDS or global
        // loads, not generic ones)
        auto partial = [&](const auto* M) {
            if (tid < n * G) {
                const int t = tid % n, g = tid / n;
                const int j1 = min(n, (g + 1) * J);
                double acc = 0.0;
#pragma unroll 4
                for (int j = g * J; j < j1; ++j) acc += M[(int64_t)j * n + t] * (double)v.b[j];
                part[g * n + t] = acc;
            }
        };
        // the matrix staged in LDS with the faces, else read from memory
        if (a.cop_lds >= 0)
            partial(reinterpret_cast<const double*>(lds + a.cop_lds));
        else
            partial(a.cop);
        lds_barrier();
        for (int t = tid; t < n; t += nt) {
            double acc = part[t];
            for (int g = 1; g < G; ++g) acc += part[g * n + t];
            v.p[t] = (float)acc;
        }
        lds_barrier();
    }
    // ascend: prolong (poisson.py:178-182), smooth (colours (1,0))
    for (int l = a.L - 2; l >= a.s + a.nreg; --l) {
        const LdsLevel v = lds_level(a, lds, l);
        const LdsLevel c = lds_level(a, lds, l + 1);
        make_level_slots(v, 1, a.omega, &c.d, S);
        if (S.s0.c >= 0) v.p[S.s0.c] += c.p[S.s0.par];
        if (S.s1.c >= 0) v.p[S.s1.c] += c.p[S.s1.par];
        lds_barrier();
        small_smooth(v, S, a.post);
    }
    OT* out = static_cast<OT*>(a.p_top);
    if (a.nreg > 1) {
        reg_ascend(R1, g1, P1, a.post, a.d[a.s + 2], lds + a.off[a.s + 2][3]);
        reg_store(R1, g1, P1, lds + a.off[a.s + 1][3]);
        lds_barrier();
    }
    if (a.nreg > 0) {
        reg_ascend(R0, g0, P0, a.post, a.d[a.s + 1], lds + a.off[a.s + 1][3]);
        reg_store(R0, g0, P0, out);
    } else {
        const LdsLevel v = lds_level(a, lds, a.s);
        const int n = v.d.nx * v.d.ny * v.d.nz;
        for (int e = tid; e < n; e += nt) out[e] = from_f32<OT>(v.p[e]);
    }
}

// ================================================================ a coarsest level by its sweeps
// The coarsest level's `sweeps` red-black sweeps from zero and its mean
// removal in one workgroup (RegPairs), for a level that is too large for the
// precomputed matrix (a grid whose extents stop halving early: 96 x 72 x 120
// ends at 12 x 9 x 15, 104 x 76 x 52 at 26 x 19 x 13, 200^3 at 25^3).  One
// launch per half-sweep costs about 3 us of launch and memory latency, 120
// times per V-cycle; here a half-sweep is LDS reads and a barrier.
// FP32 faces and iterate in every precision, like k_small_vcycle; p is
// rounded to ST once, when stored.
// What is left is VALU issue and LDS bandwidth of one CU, 0.6 us per
// half-sweep of 26 x 19 x 13, and latency on the smallest: 12 x 9 x 15 takes
// 24 us (40 from LDS with the cells decoded on each visit).  A V-cycle on the grid of twice the extents,
// launched half-sweeps -> this: 26 x 19 x 13 365 -> 113 us, 33 x 25 x 11 371
// -> 157, 27 x 27 x 15 472 -> 188, 25^3 384 -> 297 (beyond 8 pairs per thread
// one CU would be slower than the launches).
constexpr int kCoarsestPairs = 8;        // largest KP
constexpr int kCoarsestPairsRegs = 5;    // largest KP with the z faces in registers
constexpr int kCoarsestBytes = 156 * 1024;

template <typename ST, int KP, bool ZL>
__global__ __launch_bounds__(kSmallThreads) void k_coarsest(Dims d, const float* __restrict__ bx,
                                                            const float* __restrict__ by,
                                                            const float* __restrict__ bz,
                                                            const float* __restrict__ b, ST* __restrict__ pout,
                                                            int sweeps, float omega, const int* __restrict__ done) {
    extern __shared__ float lds[];
    __shared__ double sh[16];
    __shared__ float shift;
    const int tid = threadIdx.x;
    const PairGeom g = pair_geom(d);
    const int n = d.nx * d.ny * d.nz;
    float* P = lds + g.SP;         // pair t: even k at P[t], odd k at P[OFF + t]
    float* Z = lds + 2 * g.OFF;    // low z faces, the same layout
    if (done && *done) return;  // uniform: no barrier has been reached yet
    for (int e = tid; e < 2 * g.OFF; e += kSmallThreads) lds[e] = 0.0f;
    if (ZL && tid == 0) Z[g.npair] = Z[g.OFF + g.npair] = 0.0f;
    RegPairs<KP, ZL> R;
    R.load(g, bx, by, bz, omega, Z);
    R.load_b(g, b);
    __syncthreads();
    for (int sw = 0; sw < sweeps; ++sw) {
        R.template half<KP == 2>(g, P, Z, 0);
        __syncthreads();
        R.template half<KP == 2>(g, P, Z, 1);
        __syncthreads();
    }
    // everything outside the cells is still 0
    double sm[1] = {0.0};
    for (int e = tid; e < 2 * g.OFF; e += kSmallThreads) sm[0] += (double)lds[e];
    block_sum<1>(sm, sh);
    if (tid == 0) shift = (float)(-(sm[0] / (double)n));
    __syncthreads();
    for (int e = tid; e < n; e += kSmallThreads) {
        const int row = e / d.nz, k = e - row * d.nz;
        pout[e] = from_f32<ST>(P[row * g.nkp + (k >> 1) + ((k & 1) ? g.OFF : 0)] + shift);
    }
}

static int64_t coarsest_lds_bytes(const Dims& d, int kp) {
    const int64_t npair = (int64_t)d.nx * d.ny * ((d.nz + 1) / 2), off = pair_stride(d);
    return (2 * off + (kp > kCoarsestPairsRegs ? off + npair + 1 : 0)) * (int64_t)sizeof(float);
}

// pairs per thread of k_coarsest on a level, 0 if it does not take it
static int coarsest_pairs(const Dims& d) {
    const int64_t npair = (int64_t)d.nx * d.ny * ((d.nz + 1) / 2);
    const int64_t kp = cdiv(npair, kSmallThreads);
    if (kp > kCoarsestPairs) return 0;
    return coarsest_lds_bytes(d, (int)kp) <= kCoarsestBytes ? (int)kp : 0;
}

template <typename ST, int KP>
static int launch_coarsest_kp(const Dims& d, const pf_mg_level& lv, const float* b, ST* p, int sweeps, float omega,
                              const int* done, hipStream_t s) {
    constexpr bool ZL = KP > kCoarsestPairsRegs;
    static std::atomic<uint64_t> done_mask{0};  // devices whose LDS limit has been raised
    int dev = 0;
    PF_CHECK_HIP(hipGetDevice(&dev));
    const uint64_t bit = 1ull << (dev & 63);
    if (!(done_mask.load() & bit)) {
        PF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_coarsest<ST, KP, ZL>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, kCoarsestBytes));
        done_mask.fetch_or(bit);
    }
    k_coarsest<ST, KP, ZL><<<1, kSmallThreads, (size_t)coarsest_lds_bytes(d, KP), s>>>(d, lv.bx, lv.by, lv.bz, b, p, sweeps, omega, done);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

template <typename ST>
static int launch_coarsest(int kp, const Dims& d, const pf_mg_level& lv, const float* b, ST* p, int sweeps, float omega,
                           const int* done, hipStream_t s) {
    switch (kp) {
    case 1: return launch_coarsest_kp<ST, 1>(d, lv, b, p, sweeps, omega, done, s);
    case 2: return launch_coarsest_kp<ST, 2>(d, lv, b, p, sweeps, omega, done, s);
    case 3: return launch_coarsest_kp<ST, 3>(d, lv, b, p, sweeps, omega, done, s);
    case 4: return launch_coarsest_kp<ST, 4>(d, lv, b, p, sweeps, omega, done, s);
    case 5: return launch_coarsest_kp<ST, 5>(d, lv, b, p, sweeps, omega, done, s);
    case 6: return launch_coarsest_kp<ST, 6>(d, lv, b, p, sweeps, omega, done, s);
    case 7: return launch_coarsest_kp<ST, 7>(d, lv, b, p, sweeps, omega, done, s);
    case 8: return launch_coarsest_kp<ST, 8>(d, lv, b, p, sweeps, omega, done, s);
    }
    PF_REQUIRE(false, "launch_coarsest: at most 8 pairs per thread");
    return PF_OK;
}

// Column j of the coarsest level's smoother map: `sweeps` red-black sweeps
// (colours (0,1)) from p = 0 with b = e_j, then mean removal, as the
// single-workgroup V-cycle runs them, in FP64.  One workgroup per column,
// one thread per cell (n <= kCoarseOpMax).
__global__ __launch_bounds__(kCoarseOpMax) void k_coarse_op(Dims d, const float* __restrict__ bx,
                                                            const float* __restrict__ by,
                                                            const float* __restrict__ bz, int sweeps, float omega,
                                                            double* __restrict__ op) {
    __shared__ double P[kCoarseOpMax];
    __shared__ double sh[16];
    __shared__ double shift;
    const int n = d.nx * d.ny * d.nz, j = blockIdx.x, t = threadIdx.x;
    const bool own = t < n;
    double f[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int nb[6] = {0, 0, 0, 0, 0, 0};
    int colour = 0;
    double dg = 0.0;
    if (own) {
        const int k = t % d.nz, jj = (t / d.nz) % d.ny, i = t / (d.nz * d.ny);
        f[0] = bx[face_index<0>(d, i, jj, k)];
        f[1] = bx[face_index<0>(d, i + 1, jj, k)];
        f[2] = by[face_index<1>(d, i, jj, k)];
        f[3] = by[face_index<1>(d, i, jj + 1, k)];
        f[4] = bz[face_index<2>(d, i, jj, k)];
        f[5] = bz[face_index<2>(d, i, jj, k + 1)];
        nb[0] = cell_index(d, max(i - 1, 0), jj, k);
        nb[1] = cell_index(d, min(i + 1, d.nx - 1), jj, k);
        nb[2] = cell_index(d, i, max(jj - 1, 0), k);
        nb[3] = cell_index(d, i, min(jj + 1, d.ny - 1), k);
        nb[4] = cell_index(d, i, jj, max(k - 1, 0));
        nb[5] = cell_index(d, i, jj, min(k + 1, d.nz - 1));
        colour = (i + jj + k) & 1;
        dg = f[0] + f[1] + f[2] + f[3] + f[4] + f[5];
        P[t] = 0.0;
    }
    const double b = t == j ? 1.0 : 0.0, w = (double)omega;
    __syncthreads();
    for (int sw = 0; sw < sweeps; ++sw) {
        for (int c = 0; c < 2; ++c) {
            const bool upd = own && colour == c && dg > 0.0;
            double v = 0.0;
            if (upd) {
                const double pc = P[t];
                double ap = 0.0;
#pragma unroll
                for (int q = 0; q < 6; ++q) ap += f[q] * (pc - P[nb[q]]);
                v = pc + w * (b - ap) / dg;
            }
            __syncthreads();
            if (upd) P[t] = v;
            __syncthreads();
        }
    }
    double sm[1] = {own ? P[t] : 0.0};
    block_sum<1>(sm, sh);
    if (t == 0) shift = -(sm[0] / (double)n);
    __syncthreads();
    if (own) op[(int64_t)j * n + t] = P[t] + shift;
}

static bool use_coarse_op(const pf_mg& mg) {
    const pf_mg_level& c = mg.lev[mg.nlev - 1];
    return mg.small_from < mg.nlev && (int64_t)c.nx * c.ny * c.nz <= kCoarseOpMax;
}

// ================================================================ FPCG kernels
template <typename ZT>
struct CGK {
    Dims d;
    int64_t n;
    const float* bx;
    const float* by;
    const float* bz;
    const float* b;
    float* rhs;
    float* x;
    float* r;
    float* q;            // search direction written by this iteration
    const float* q_old;  // the previous one (the two alternate between iterations)
    float* Ap;
    const ZT* z;
    const float* zscale;  // NULL: z as stored; else z times *zscale
    CGState* st;
    double tol;
    int slot;      // parity of the iteration (selects q / q_old and rz)
    int np_apply;  // blocks of k_cg_apply (its <q, Aq> partials)
    int np_beta;   // blocks of k_cg_beta (its dot-product partials)
};

template <typename ZT>
__device__ inline float zval(const CGK<ZT>& a, float zs, int64_t i) {
    return to_f32(a.z[i]) * zs;
}

// r = b - mean(b); x = 0; q = 0; partial max|r| (poisson.py:363-372)
template <typename ZT>
__global__ __launch_bounds__(RT) void k_cg_init(CGK<ZT> a) {
    __shared__ float sh[4];
    const float c = (float)(-a.st->mu);
    float m = 0.0f;
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * RT) {
        const float v = a.b[i] + c;
        a.r[i] = v;
        a.x[i] = 0.0f;
        a.q[i] = 0.0f;  // the first iteration's previous direction (beta = 0)
        m = fmaxf(m, fabsf(v));
    }
    m = block_max(m, sh);
    if (threadIdx.x == 0) a.st->fpart[blockIdx.x] = m;
}

// partials of sum(z), sum(r), <r, z> after the first V-cycle
template <typename ZT>
__global__ __launch_bounds__(RT) void k_cg_first(CGK<ZT> a) {
    __shared__ double sh[3 * 16];
    if (a.st->done) return;
    const float zs = a.zscale ? *a.zscale : 1.0f;
    double v[3] = {0.0, 0.0, 0.0};
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * RT) {
        const double zz = (double)zval(a, zs, i), rr = (double)a.r[i];
        v[0] += zz;
        v[1] += rr;
        v[2] += rr * zz;
    }
    block_sum<3>(v, sh);
    if (threadIdx.x == 0)
        for (int q = 0; q < 3; ++q) a.st->part[q * PS + blockIdx.x] = v[q];
}

// q = (z - mu) + beta q_old (the search direction, poisson.py:406; beta = 0
// on the first iteration), evaluated at the cell and its six neighbours;
// then Ap = A q and the partial <q, Ap> (poisson.py:385-386).  Writes q and Ap
// of the cell; q_old is a different buffer, so neighbours read old values.
// From the second iteration on it first combines k_cg_beta's partials into
// the mean of z and the Polak-Ribiere beta (poisson.py:400-406) itself:
// every block sums them in the same fixed order, so all blocks hold the same
// scalars, and block 0 records them (no separate combine launch).
template <typename ZT>
__global__ __launch_bounds__(WT) void k_cg_apply(CGK<ZT> a) {
    __shared__ double sh[5 * 16];
    __shared__ float s_cm, s_be;
    CGState* st = a.st;
    const Dims d = a.d;
    // 32-bit indices (the level's face arrays hold fewer than 2^31
    // entries): the thread's first cell and the grid stride are decoded into
    // (i, j, k) once, and the loop adds the stride with carries; the faces
    // and the clamped neighbours are offsets from the cell index
    // (face_index and cell_index written out).  64-bit division per cell
    // made this loop several times longer.
    const int n = (int)a.n, sjk = d.ny * d.nz;
    const int c0 = blockIdx.x * WT + threadIdx.x, S = gridDim.x * WT;
    int k = c0 % d.nz, j = (c0 / d.nz) % d.ny, i = c0 / sjk;
    const int sk = S % d.nz, sj = (S / d.nz) % d.ny, si = S / sjk;
    // a cell's inputs: faces, then z (as FP32, unscaled) and q_old at the
    // cell and its six clamped neighbours (-x, +x, -y, +y, -z, +z)
    float f[6], zr[7], qo[7];
    auto load_cell = [&](int c) {
        const int fy = c + i * d.nz, fz = c + i * d.ny + j;
        f[0] = a.bx[c];
        f[1] = a.bx[c + sjk];
        f[2] = a.by[fy];
        f[3] = a.by[fy + d.nz];
        f[4] = a.bz[fz];
        f[5] = a.bz[fz + 1];
        const int nb[7] = {c, i > 0 ? c - sjk : c, i < d.nx - 1 ? c + sjk : c, j > 0 ? c - d.nz : c,
                           j < d.ny - 1 ? c + d.nz : c, k > 0 ? c - 1 : c, k < d.nz - 1 ? c + 1 : c};
#pragma unroll
        for (int t = 0; t < 7; ++t) {
            zr[t] = to_f32(a.z[nb[t]]);
            qo[t] = a.q_old[nb[t]];
        }
    };
    // the first cell's loads are issued before the flag test and the
    // combine below, so their round trip overlaps that work (a finished
    // solve's queued launch returns with them in flight)
    if (c0 < n) load_cell(c0);
    const float zs = a.zscale ? *a.zscale : 1.0f;
    if (st->done) return;
    if (st->beta_parts) {
        // z' = z - mean(z); rz_new = <r, z'>; num = rz_new - <r_prev, z'> =
        // -alpha <Ap, z'> because r_prev = r + alpha Ap
        double t[5];
        combine_sums<5>(st->part, a.np_beta, t, sh);
        if (threadIdx.x == 0) {
            const double mu = t[0] / (double)a.n;
            const double rz_new = t[3] - mu * t[1];
            const double apz = t[4] - mu * t[2];
            const double num = -st->alpha * apz;
            const double rz = st->rz[a.slot ^ 1];
            const double beta = (rz != 0.0) ? fmax(num / rz, 0.0) : 0.0;
            s_cm = (float)(-mu);
            s_be = (float)beta;
            if (blockIdx.x == 0) {
                st->mu = mu;
                st->beta = beta;
                st->rz[a.slot] = rz_new;
            }
        }
    } else if (threadIdx.x == 0) {  // the first iteration: k_comb(C_FIRST) set them
        s_cm = (float)(-st->mu);
        s_be = (float)st->beta;
    }
    __syncthreads();
    const float cm = s_cm;
    const float be = s_be;
    double v[1] = {0.0};
    // q at input point t: (z - mu) + beta q_old
    auto qv = [&](int t) {
        const float zz = zr[t] * zs + cm;
        return zz + be * qo[t];
    };
    for (int c = c0; c < n; c += S) {
        if (c != c0) load_cell(c);
        const float pc = qv(0);
        const float pn[6] = {qv(1), qv(2), qv(3), qv(4), qv(5), qv(6)};
        float dg, Ap;
        stencil_vals(pc, f, pn, dg, Ap);
        a.q[c] = pc;
        a.Ap[c] = Ap;
        v[0] += (double)pc * (double)Ap;
        k += sk;
        if (k >= d.nz) {
            k -= d.nz;
            ++j;
        }
        j += sj;
        if (j >= d.ny) {
            j -= d.ny;
            ++i;
        }
        i += si;
    }
    block_sum<1>(v, sh);
    if (threadIdx.x == 0) st->part[5 * PS + blockIdx.x] = v[0];
}

// x += alpha q; r -= alpha Ap; partial max|r| (poisson.py:390-394), after
// combining k_cg_apply's partials into <q, Aq> and alpha = rz / <q, Aq> in
// every block (fixed order, so all blocks agree); <q, Aq> <= 0 ends the
// solve before any update (poisson.py:386-389).  Block 0 records the
// scalars and the iteration count.
template <typename ZT>
__global__ __launch_bounds__(RT) void k_cg_update(CGK<ZT> a) {
    __shared__ float sh[4];
    __shared__ double shd[16];
    __shared__ float s_al;
    __shared__ int s_ok;
    CGState* st = a.st;
    // the first element's inputs are loaded before the flag test and the
    // combine, so their round trip overlaps that work
    const int64_t i0 = (int64_t)blockIdx.x * RT + threadIdx.x, stride = (int64_t)gridDim.x * RT;
    float x0 = 0.f, q0 = 0.f, r0 = 0.f, ap0 = 0.f;
    if (i0 < a.n) {
        x0 = a.x[i0];
        q0 = a.q[i0];
        r0 = a.r[i0];
        ap0 = a.Ap[i0];
    }
    if (st->done) return;
    double t[1];
    combine_sums<1>(st->part + 5 * PS, a.np_apply, t, shd);
    if (threadIdx.x == 0) {
        const double qAq = t[0];
        const bool ok = qAq > 0.0;
        const double alpha = ok ? st->rz[a.slot] / qAq : 0.0;
        s_ok = ok ? 1 : 0;
        s_al = (float)alpha;
        if (blockIdx.x == 0) {
            st->qAq = qAq;
            st->it += 1;
            if (ok)
                st->alpha = alpha;
            else
                st->done = 1;
        }
    }
    __syncthreads();
    if (!s_ok) return;
    const float al = s_al, nal = -s_al;
    float m = 0.0f;
    for (int64_t i = i0; i < a.n; i += stride) {
        if (i != i0) {
            x0 = a.x[i];
            q0 = a.q[i];
            r0 = a.r[i];
            ap0 = a.Ap[i];
        }
        a.x[i] = x0 + al * q0;
        const float rn = r0 + nal * ap0;
        a.r[i] = rn;
        m = fmaxf(m, fabsf(rn));
    }
    m = block_max(m, sh);
    if (threadIdx.x == 0) a.st->fpart[blockIdx.x] = m;
}

// partials of sum(z), sum(r), sum(Ap), <r,z>, <Ap,z> after a V-cycle
template <typename ZT>
__global__ __launch_bounds__(WT) void k_cg_beta(CGK<ZT> a) {
    __shared__ double sh[5 * 16];
    if (a.st->done) return;
    const float zs = a.zscale ? *a.zscale : 1.0f;
    double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int64_t i = (int64_t)blockIdx.x * WT + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * WT) {
        const double zz = (double)zval(a, zs, i), rr = (double)a.r[i], ap = (double)a.Ap[i];
        v[0] += zz;
        v[1] += rr;
        v[2] += ap;
        v[3] += rr * zz;
        v[4] += ap * zz;
    }
    block_sum<5>(v, sh);
    if (threadIdx.x == 0) {
        for (int q = 0; q < 5; ++q) a.st->part[q * PS + blockIdx.x] = v[q];
        if (blockIdx.x == 0) a.st->beta_parts = 1;  // read by the next k_cg_apply
    }
}

// One-block combine of the previous kernel's partials, then the scalar step.
enum CombOp { C_MEAN = 0, C_MEAN_RESET, C_INIT, C_FIRST, C_UPDATE };


__global__ __launch_bounds__(RT) void k_comb(CGState* st, int op, int nparts, int64_t n,
                                             double* out, double tol, int* host_flag = nullptr) {
    __shared__ double sh[5 * 16];
    __shared__ float shf[4];
    if (op == C_MEAN || op == C_MEAN_RESET) {
        double t[1];
        combine_sums<1>(st->part, nparts, t, sh);
        if (threadIdx.x == 0) {
            *out = t[0] / (double)n;
            if (op == C_MEAN_RESET) {
                st->done = 0;
                st->it = 0;
                st->seq = 0;
                st->beta_parts = 0;
                st->rel = 1.0;
            }
        }
        return;
    }
    if (op == C_INIT) {
        // b_norm = max|rhs|; b == 0 returns x = 0 (poisson.py:365-368)
        const float mm = combine_max(st->fpart, nparts, shf);
        if (threadIdx.x == 0) {
            st->b_norm = (double)mm;
            st->tol = tol;
            set_vscale(st, mm);
            if (mm == 0.0f) {
                st->done = 2;
                st->rel = 0.0;
            }
        }
        return;
    }
    if (op == C_UPDATE) {
        // rel = max|r| / max|b| (poisson.py:394-398)
        const float mm = st->done ? 0.0f : combine_max(st->fpart, nparts, shf);
        if (threadIdx.x == 0) residual_test_record(st, mm, host_flag);
        return;
    }
    if (st->done) return;
    if (op == C_FIRST) {
        // mu = mean(z); rz = <r, z - mu>
        double t[3];
        combine_sums<3>(st->part, nparts, t, sh);
        if (threadIdx.x == 0) {
            // iteration 1 has parity 1: its k_cg_update reads rz[1]
            const double mu = t[0] / (double)n;
            st->mu = mu;
            st->rz[1] = t[2] - mu * t[1];
            st->beta = 0.0;
            st->beta_parts = 0;
        }
    }
}

__global__ __launch_bounds__(RT) void k_apply_A(Dims d, const float* __restrict__ p,
                                                const float* __restrict__ bx,
                                                const float* __restrict__ by,
                                                const float* __restrict__ bz,
                                                const float* __restrict__ diag, float* out) {
    const int64_t c = (int64_t)blockIdx.x * RT + threadIdx.x;
    if (c >= (int64_t)d.nx * d.ny * d.nz) return;
    const int k = (int)(c % d.nz), j = (int)((c / d.nz) % d.ny), i = (int)(c / ((int64_t)d.nz * d.ny));
    float dg, sn, pc;
    stencil_s(d, bx, by, bz, p, i, j, k, dg, sn, pc);
    out[c] = (diag ? diag[c] : dg) * pc - sn;
}

// ================================================================ host side
static Dims ldims(const pf_mg_level& l) { return Dims{l.nx, l.ny, l.nz}; }
static int64_t ncell(const pf_mg_level& l) { return (int64_t)l.nx * l.ny * l.nz; }

// LDS layout of the single-workgroup V-cycle from level s down: the register
// levels' pair arrays; the face arrays of the LDS levels back to back (of the
// coarsest one none: it is a matrix product); p and b of every level but a
// register level s; the scratch.
static int small_reg_levels(const pf_mg& mg, int s) { return std::min(2, mg.nlev - 1 - s); }

static int64_t small_lds_floats(const pf_mg& mg, int s, int (*off)[5], int* poff, int* scratch) {
    const int nreg = small_reg_levels(mg, s);
    int64_t o = 0;
    for (int r = 0; r < 2; ++r) {
        if (poff) poff[r] = (int)o;
        if (r < nreg) o += 2 * (int64_t)pair_stride(ldims(mg.lev[s + r]));
    }
    for (int l = s + nreg; l < mg.nlev - 1; ++l) {
        const Dims d = ldims(mg.lev[l]);
        for (int q = 0; q < 3; ++q) {
            if (off) off[l][q] = (int)o;
            o += face_count(d, q);
        }
    }
    for (int l = s + (nreg > 0 ? 1 : 0); l < mg.nlev; ++l) {
        const int64_t nc = ncell(mg.lev[l]);
        if (off) off[l][3] = (int)o;
        o += nc;
        if (off) off[l][4] = (int)o;
        o += nc;
    }
    // the scratch: a level's residual, and the FP64 partials of the coarsest
    // level's matrix product (8-byte aligned, at most kSmallThreads)
    o = (o + 1) & ~(int64_t)1;
    if (scratch) *scratch = (int)o;
    return o + std::max<int64_t>(ncell(mg.lev[s]), 2 * kSmallThreads);
}

constexpr int64_t kSmallMaxCells = 8192;
constexpr int64_t kSmallMaxBytes = 150 * 1024;

template <typename ST>
struct Lv {
    static const ST* fx(const pf_mg_level& l) { return reinterpret_cast<const ST*>(l.bx_h); }
    static const ST* fy(const pf_mg_level& l) { return reinterpret_cast<const ST*>(l.by_h); }
    static const ST* fz(const pf_mg_level& l) { return reinterpret_cast<const ST*>(l.bz_h); }
    static ST* p(const pf_mg_level& l) { return reinterpret_cast<ST*>(l.p_h); }
};
template <>
struct Lv<float> {
    static const float* fx(const pf_mg_level& l) { return l.bx; }
    static const float* fy(const pf_mg_level& l) { return l.by; }
    static const float* fz(const pf_mg_level& l) { return l.bz; }
    static float* p(const pf_mg_level& l) { return l.p; }
};

// The single-workgroup kernel needs more than the default 64 KB of dynamic
// LDS; raise the limit once per device (gfx950 has 160 KB per workgroup).
static int ensure_small_lds() {
    static std::atomic<uint64_t> done_mask{0};
    int dev = 0;
    PF_CHECK_HIP(hipGetDevice(&dev));
    const uint64_t bit = 1ull << (dev & 63);
    if (done_mask.load() & bit) return PF_OK;
    const int bytes = (int)kSmallMaxBytes;
    PF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_small_vcycle<float>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    PF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_small_vcycle<bf16s>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    PF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_small_vcycle<fp16s>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    done_mask.fetch_or(bit);
    return PF_OK;
}

// Fused full sweep on one level: tile shape by level size.  Long tiles cut
// the redundant halo work, small ones keep enough workgroups in flight.
// us per sweep, FP32 / BF16 (HIP events, 60 sweeps), by tile and threads:
//                  8x8x64/512    8x8x32/512    8x8x16/256
//   80^3            8.4 /  8.6    7.6 /  7.8    6.7 /  6.9
//   128x96x64       8.0 /  8.4    7.4 /  7.5    7.7 /  7.8
//   96x72x120       8.6 /  8.6    8.1 /  7.8    9.3 /  9.2
//   128^3          13.2 / 11.9   13.5 / 12.7   16.5 / 14.8
//   192x128x96     17.3 / 18.2   14.8 / 14.1   17.5 / 15.3
//   160^3          26.6 / 28.1   24.0 / 21.6   29.4 / 25.3
//   256^3           112 / 82.4    123 / 73.0    164 / 89.8
//   320x320x8        --           17.6 / 16.6   11.4 / 10.8
//   512x512x16      66.2 / 73.1   34.0 / 35.4   21.3 / 21.0
//   300x300x18      27.2 / 26.5   15.0 / 15.0   16.8 / 16.5
//   160x160x40       --           11.2 / 11.2    9.4 /  9.1
//   192x192x40      16.0 / 16.4   13.3 / 13.1   12.6 / 11.4
//   256x256x48      20.5 / 21.0   19.7 / 20.1   20.8 / 17.9
//   200x200x80      25.6 / 27.7   20.5 / 20.7   23.5 / 20.6
// So 8x8x64 where its tiles are whole along k, in 16 bits only while they are
// all resident at once (two per CU); otherwise 8x8x32 from 5 x 2^17 cells,
// unless it is padded by another 8x8x16 tile of one or of three: that is its
// whole gain and more up to 16 cells along k, and from 33 to 48 in 16 bits or
// below 2^21 cells.
enum SweepShape { SWEEP_64, SWEEP_32, SWEEP_16, SWEEP_SMALL };

static int64_t sweep_tiles(const Dims& d, SweepShape s) {
    const int tk = s == SWEEP_64 ? 64 : (s == SWEEP_32 ? 32 : 16);
    return (int64_t)cdiv(d.nx, s == SWEEP_SMALL ? 4 : 8) * cdiv(d.ny, 8) * cdiv(d.nz, tk);
}

static SweepShape sweep_shape(const Dims& d, bool half) {
    const int64_t n = (int64_t)d.nx * d.ny * d.nz;
    if (n >= (int64_t)1 << 20 && d.nz % 64 == 0 && (!half || sweep_tiles(d, SWEEP_64) <= 512)) return SWEEP_64;
    const bool padded = d.nz <= 16 || (d.nz > 32 && d.nz <= 48 && (half || n < (int64_t)1 << 21));
    if (n >= (int64_t)5 << 17 && !padded) return SWEEP_32;
    return n >= (int64_t)1 << 17 ? SWEEP_16 : SWEEP_SMALL;
}

// PROL (CT = the coarse iterate's type): the input is pin plus the
// prolongation of pcoarse (dims dc); the fine dims must be twice dc.
template <typename ST, bool ZINIT, bool PROL = false, typename CT = float>
static int launch_full_sweep(const Dims& d, const ST* fx, const ST* fy, const ST* fz, const ST* pin,
                             ST* pout, const float* b, int c1, float omega, const int* done,
                             const float* bscale, hipStream_t s, const CT* pcoarse = nullptr,
                             Dims dc = Dims{1, 1, 1}, UpdateFold uf = UpdateFold{nullptr, 0, nullptr},
                             DotFold df = DotFold{nullptr, nullptr, nullptr}) {
    const SweepShape shape = sweep_shape(d, sizeof(ST) == 2);
    const unsigned tiles = (unsigned)sweep_tiles(d, shape);
    if constexpr (!ZINIT && !PROL) {
        if (df.Ap) {  // the plain sweep with the CG's inner products
            switch (shape) {
            case SWEEP_64:
                k_rbgs_full<ST, false, 8, 8, 64, 512, false, float, true><<<tiles, 512, 0, s>>>(
                    d, fx, fy, fz, pin, pout, b, c1, omega, done, bscale, nullptr, dc, uf, df);
                break;
            case SWEEP_32:
                k_rbgs_full<ST, false, 8, 8, 32, 512, false, float, true><<<tiles, 512, 0, s>>>(
                    d, fx, fy, fz, pin, pout, b, c1, omega, done, bscale, nullptr, dc, uf, df);
                break;
            case SWEEP_16:
                k_rbgs_full<ST, false, 8, 8, 16, 256, false, float, true><<<tiles, 256, 0, s>>>(
                    d, fx, fy, fz, pin, pout, b, c1, omega, done, bscale, nullptr, dc, uf, df);
                break;
            case SWEEP_SMALL:
                k_rbgs_full<ST, false, 4, 8, 16, 256, false, float, true><<<tiles, 256, 0, s>>>(
                    d, fx, fy, fz, pin, pout, b, c1, omega, done, bscale, nullptr, dc, uf, df);
                break;
            }
            PF_CHECK_LAUNCH();
            return PF_OK;
        }
    }
    PF_REQUIRE(!df.Ap, "launch_full_sweep: inner products only on a plain sweep");
    switch (shape) {
    case SWEEP_64:
        k_rbgs_full<ST, ZINIT, 8, 8, 64, 512, PROL, CT><<<tiles, 512, 0, s>>>(
            d, fx, fy, fz, pin, pout, b, c1, omega, done, bscale, pcoarse, dc, uf, df);
        break;
    case SWEEP_32:
        k_rbgs_full<ST, ZINIT, 8, 8, 32, 512, PROL, CT><<<tiles, 512, 0, s>>>(
            d, fx, fy, fz, pin, pout, b, c1, omega, done, bscale, pcoarse, dc, uf, df);
        break;
    case SWEEP_16:
        k_rbgs_full<ST, ZINIT, 8, 8, 16, 256, PROL, CT><<<tiles, 256, 0, s>>>(
            d, fx, fy, fz, pin, pout, b, c1, omega, done, bscale, pcoarse, dc, uf, df);
        break;
    case SWEEP_SMALL:
        k_rbgs_full<ST, ZINIT, 4, 8, 16, 256, PROL, CT><<<tiles, 256, 0, s>>>(
            d, fx, fy, fz, pin, pout, b, c1, omega, done, bscale, pcoarse, dc, uf, df);
        break;
    }
    PF_CHECK_LAUNCH();
    return PF_OK;
}

// Levels whose pre and post phases run as one k_phase launch each: those of
// at most one workgroup per CU, with 4 x 4 x 8 tiles (up to 32^3), else with
// 8 x 8 x 16 ones (up to 64^3).  A second round of workgroups costs more than
// the per-sweep launches: a V-cycle of 80^3 (500 tiles) took 121 us with its
// level 0 in phases, 111 without; 64^3 (256 tiles) 82 and 90.
constexpr unsigned kPhaseTiles = 256;

static unsigned phase_tiles(const Dims& d, int t) {
    return (unsigned)(cdiv(d.nx, t) * cdiv(d.ny, t) * cdiv(d.nz, 2 * t));
}
// tile edge of a level's k_phase launches, 0: too large for them
static int phase_tile(const Dims& d) {
    for (int t = 4; t <= 8; t *= 2)
        if (phase_tiles(d, t) <= kPhaseTiles) return t;
    return 0;
}

template <typename ST, bool PRE, int T, typename CT>
static int launch_phase_tile(const Dims& d, const Dims& dc, int nsw, const ST* fx, const ST* fy, const ST* fz,
                             const float* b, const ST* pin, const CT* pcoarse, ST* pout, float* bc, float omega,
                             const int* done, const float* bscale, UpdateFold uf, DotFold df, hipStream_t s) {
    const unsigned grid = phase_tiles(d, T);
    switch (nsw) {
    case 1:
        k_phase<ST, PRE, T, 2 * T, 1, CT><<<grid, 1024, 0, s>>>(d, dc, fx, fy, fz, b, pin, pcoarse, pout, bc, omega,
                                                               done, bscale, uf, df);
        break;
    case 2:
        k_phase<ST, PRE, T, 2 * T, 2, CT><<<grid, 1024, 0, s>>>(d, dc, fx, fy, fz, b, pin, pcoarse, pout, bc, omega,
                                                               done, bscale, uf, df);
        break;
    case 3:
        k_phase<ST, PRE, T, 2 * T, 3, CT><<<grid, 1024, 0, s>>>(d, dc, fx, fy, fz, b, pin, pcoarse, pout, bc, omega,
                                                               done, bscale, uf, df);
        break;
    default:
        PF_REQUIRE(false, "launch_phase: 1 to 3 sweeps");
    }
    PF_CHECK_LAUNCH();
    return PF_OK;
}

// One k_phase launch: PRE (the pre-smoothing phase from zero and the
// restricted residual into bc) or the post phase (pin plus the prolongation
// of pcoarse, dims dc, into pout); nsw sweeps, 1..3.
template <typename ST, bool PRE, typename CT = float>
static int launch_phase(const Dims& d, const Dims& dc, int nsw, const ST* fx, const ST* fy, const ST* fz,
                        const float* b, const ST* pin, const CT* pcoarse, ST* pout, float* bc, float omega,
                        const int* done, const float* bscale, UpdateFold uf, DotFold df, hipStream_t s) {
    PF_REQUIRE(d.nx == 2 * dc.nx && d.ny == 2 * dc.ny && d.nz == 2 * dc.nz, "launch_phase: fine dims must be 2x coarse");
    return phase_tile(d) == 4
               ? launch_phase_tile<ST, PRE, 4, CT>(d, dc, nsw, fx, fy, fz, b, pin, pcoarse, pout, bc, omega, done,
                                                   bscale, uf, df, s)
               : launch_phase_tile<ST, PRE, 8, CT>(d, dc, nsw, fx, fy, fz, b, pin, pcoarse, pout, bc, omega, done,
                                                   bscale, uf, df, s);
}

// The two iterate buffers of an HBM level: the level's own (level 0: the
// output z0) and the fused smoother's second buffer.
template <typename ST>
static ST* second_buffer(const pf_mg& mg, int l) {
    if (sizeof(ST) == 4 && l == 0) return reinterpret_cast<ST*>(mg.lev[0].p);
    return reinterpret_cast<ST*>(mg.lev[l].r);
}

static bool fused_smoother(const pf_mg& mg, int l) {
    return !(mg.options & PF_MG_UNFUSED_SMOOTHER) && (mg.lev[l].nz % 2) == 0;
}

// level l (restricted to l + 1) runs each smoothing phase as one k_phase
// launch
static bool level_fused(const pf_mg& mg, int l) {
    const int G = mg.small_from < mg.nlev ? mg.small_from : mg.nlev - 1;
    return l < G && !(mg.options & PF_MG_SPLIT_LEVELS) && fused_smoother(mg, l) && phase_tile(ldims(mg.lev[l])) &&
           mg.pre >= 1 && mg.pre <= 3 && mg.post >= 1 && mg.post <= 3;
}

// One V-cycle: z0 = M^{-1} r0 (no mean removal at level 0).
template <typename ST>
// dfold: the CG's inner products ride on the last level-0 post-sweep
// (*dot_done tells whether one took them).
static int vcycle(const pf_mg& mg, const float* r0, ST* z0, const int* done, const float* bscale,
                  hipStream_t s, const UpdateFold* uf = nullptr, const DotFold* dfold = nullptr,
                  bool* dot_done = nullptr) {
    const int L = mg.nlev;
    const int sm = mg.small_from;             // first LDS level (L if none)
    const int G = sm < L ? sm : L - 1;        // levels 0..G-1 run out of HBM with restriction
    auto P = [&](int l) -> ST* { return l == 0 ? z0 : Lv<ST>::p(mg.lev[l]); };
    auto B = [&](int l) -> const float* { return l == 0 ? r0 : mg.lev[l].b; };
    ST* cur[PF_MAX_LEVELS];  // buffer holding each HBM level's current iterate
    auto other = [&](int l, const ST* x) -> ST* { return x == P(l) ? second_buffer<ST>(mg, l) : P(l); };

    // `sweeps` red-black sweeps of level l (colour order (0,1), or (1,0) if
    // reverse), starting from zero if from_zero, else from cur[l]
    auto smooth = [&](int l, int sweeps, bool reverse, bool from_zero) -> int {
        const pf_mg_level& lv = mg.lev[l];
        const Dims d = ldims(lv);
        const ST *fx = Lv<ST>::fx(lv), *fy = Lv<ST>::fy(lv), *fz = Lv<ST>::fz(lv);
        const float* b = B(l);
        const float* bsc = l == 0 ? bscale : nullptr;
        if (from_zero) cur[l] = P(l);
        if (from_zero && sweeps == 0) {
            k_zero<ST><<<red_blocks(ncell(lv)), RT, 0, s>>>(cur[l], ncell(lv), done);
            PF_CHECK_LAUNCH();
        }
        if (fused_smoother(mg, l)) {
            for (int sw = 0; sw < sweeps; ++sw) {
                ST* out = other(l, cur[l]);
                const int c1 = reverse ? 1 : 0;
                // the V-cycle's first kernel takes the residual test with it
                const UpdateFold f = (uf && l == 0 && sw == 0) ? *uf : UpdateFold{nullptr, 0, nullptr};
                const bool dots = dfold && l == 0 && !from_zero && sw == sweeps - 1;
                const int rc = (from_zero && sw == 0)
                                   ? launch_full_sweep<ST, true>(d, fx, fy, fz, cur[l], out, b, c1, mg.omega, done,
                                                                 bsc, s, static_cast<const float*>(nullptr),
                                                                 Dims{1, 1, 1}, f)
                                   : launch_full_sweep<ST, false>(d, fx, fy, fz, cur[l], out, b, c1, mg.omega, done,
                                                                  bsc, s, static_cast<const float*>(nullptr),
                                                                  Dims{1, 1, 1}, UpdateFold{nullptr, 0, nullptr},
                                                                  dots ? *dfold : DotFold{nullptr, nullptr, nullptr});
                if (dots && dot_done) *dot_done = true;
                if (rc) return rc;
                cur[l] = out;
            }
            return PF_OK;
        }
        const int64_t nthr = (int64_t)d.nx * d.ny * ((d.nz + 1) / 2);
        const unsigned grid = cdiv(nthr, RT);
        for (int sw = 0; sw < sweeps; ++sw) {
            for (int h = 0; h < 2; ++h) {
                const int colour = reverse ? 1 - h : h;
                if (from_zero && sw == 0 && h == 0)
                    k_rbgs<ST, true><<<grid, RT, 0, s>>>(d, fx, fy, fz, cur[l], b, colour, mg.omega, done, bsc);
                else
                    k_rbgs<ST, false><<<grid, RT, 0, s>>>(d, fx, fy, fz, cur[l], b, colour, mg.omega, done, bsc);
                PF_CHECK_LAUNCH();
            }
        }
        return PF_OK;
    };

    for (int l = 0; l < G; ++l) {
        const pf_mg_level& lv = mg.lev[l];
        const pf_mg_level& cv = mg.lev[l + 1];
        if (level_fused(mg, l)) {
            // (level 0: the post phase then lands in z0)
            cur[l] = l == 0 ? second_buffer<ST>(mg, 0) : P(l);
            const int rc = launch_phase<ST, true>(ldims(lv), ldims(cv), mg.pre, Lv<ST>::fx(lv), Lv<ST>::fy(lv),
                                                  Lv<ST>::fz(lv), B(l), static_cast<const ST*>(nullptr),
                                                  static_cast<const float*>(nullptr), cur[l], mg.lev[l + 1].b,
                                                  mg.omega, done, l == 0 ? bscale : nullptr,
                                                  uf && l == 0 ? *uf : UpdateFold{nullptr, 0, nullptr},
                                                  DotFold{nullptr, nullptr, nullptr}, s);
            if (rc) return rc;
            continue;
        }
        int rc = smooth(l, mg.pre, false, true);
        if (rc) return rc;
        k_resid_restrict<ST><<<cdiv(ncell(cv), RT), RT, 0, s>>>(ldims(lv), ldims(cv), Lv<ST>::fx(lv),
                                                              Lv<ST>::fy(lv), Lv<ST>::fz(lv), cur[l], B(l),
                                                              mg.lev[l + 1].b, done, l == 0 ? bscale : nullptr);
        PF_CHECK_LAUNCH();
    }
    const bool swept = sm >= L - 1 && !use_coarse_op(mg);  // the coarsest level by its sweeps
    if (sm < L && !swept) {
        int rc0 = ensure_small_lds();
        if (rc0) return rc0;
        SmallArgs a;
        a.s = sm;
        a.L = L;
        a.pre = mg.pre;
        a.post = mg.post;
        a.nreg = small_reg_levels(mg, sm);
        a.omega = mg.omega;
        for (int l = sm; l < L; ++l) a.d[l] = ldims(mg.lev[l]);
        const int64_t nf = small_lds_floats(mg, sm, a.off, a.poff, &a.scratch);
        for (int r = 0; r < 2; ++r) {
            const pf_mg_level& v = mg.lev[std::min(sm + r, L - 1)];
            a.rf[r][0] = v.bx;
            a.rf[r][1] = v.by;
            a.rf[r][2] = v.bz;
        }
        a.b_top = B(sm);
        a.nseg = 0;
        auto seg = [&](const float* src, int dst, int64_t n) {
            a.seg_src[a.nseg] = src;
            a.seg_dst[a.nseg] = dst;
            a.seg_len[a.nseg++] = (int)n;
        };
        for (int l = sm + a.nreg; l < L - 1; ++l) {
            seg(mg.lev[l].bx, a.off[l][0], face_count(a.d[l], 0));
            seg(mg.lev[l].by, a.off[l][1], face_count(a.d[l], 1));
            seg(mg.lev[l].bz, a.off[l][2], face_count(a.d[l], 2));
        }
        if (a.nreg == 0) seg(B(sm), a.off[sm][4], ncell(mg.lev[sm]));
        a.done = done;
        a.cop = static_cast<CGState*>(mg.scalars)->coarse_op;
        // stage the coarsest level's matrix too when it fits the LDS budget:
        // its loads then overlap the others instead of costing round trips of
        // their own in the middle of the V-cycle
        a.cop_lds = -1;
        int64_t nlds = nf;
        const int64_t ncop = ncell(mg.lev[L - 1]);
        const int64_t cop_off = (nf + 3) & ~(int64_t)3;  // 16-byte aligned
        if ((cop_off + 2 * ncop * ncop) * (int64_t)sizeof(float) <= kSmallMaxBytes) {
            a.cop_lds = (int)cop_off;
            seg(reinterpret_cast<const float*>(a.cop), (int)cop_off, 2 * ncop * ncop);
            nlds = cop_off + 2 * ncop * ncop;
        }
        const size_t lds = (size_t)nlds * sizeof(float);
        if (sm == 0) {
            a.p_top = z0;
            k_small_vcycle<ST><<<1, kSmallThreads, lds, s>>>(a);
        } else {
            a.p_top = mg.lev[sm].p;
            k_small_vcycle<float><<<1, kSmallThreads, lds, s>>>(a);
        }
        PF_CHECK_LAUNCH();
    } else {
        // the coarsest level's sweeps, then mean removal, in one workgroup
        // where it fits (a one-level hierarchy that is too large for the
        // single-workgroup V-cycle has its own right-hand side scale and
        // residual test and stays launched)
        const int l = L - 1;
        const int kp = L > 1 || sm == 0 ? coarsest_pairs(ldims(mg.lev[l])) : 0;
        if (kp) {
            const Dims d = ldims(mg.lev[l]);
            int rc;
            if (l == sm && l > 0) {  // an FP32 level in every precision, as k_small_vcycle's
                rc = launch_coarsest<float>(kp, d, mg.lev[l], B(l), mg.lev[l].p, mg.coarsest, mg.omega, done, s);
            } else {
                cur[l] = P(l);
                rc = launch_coarsest<ST>(kp, d, mg.lev[l], B(l), cur[l], mg.coarsest, mg.omega, done, s);
            }
            if (rc) return rc;
        } else {
            int rc = smooth(l, mg.coarsest, false, true);
            if (rc) return rc;
            CGState* st = static_cast<CGState*>(mg.scalars);
            const int64_t n = ncell(mg.lev[l]);
            // p is ST; the mean is taken in FP64 and the shifted value stored back
            k_part_sum<ST><<<red_blocks(n), RT, 0, s>>>(cur[l], n, st->part);
            PF_CHECK_LAUNCH();
            k_comb<<<1, RT, 0, s>>>(st, C_MEAN, (int)red_blocks(n), n, &st->mu_x, 0.0);
            PF_CHECK_LAUNCH();
            // (an odd number of sweeps ends in the second buffer)
            k_shift<ST, ST><<<red_blocks(n), RT, 0, s>>>(cur[l], P(l), n, &st->mu_x);
            PF_CHECK_LAUNCH();
            cur[l] = P(l);
        }
    }
    for (int l = G - 1; l >= 0; --l) {
        const pf_mg_level& lv = mg.lev[l];
        const pf_mg_level& cv = mg.lev[l + 1];
        if (level_fused(mg, l)) {
            ST* out = other(l, cur[l]);
            const float* bsc = l == 0 ? bscale : nullptr;
            const UpdateFold nf{nullptr, 0, nullptr};
            const bool dots = dfold && l == 0;
            const DotFold df = dots ? *dfold : DotFold{nullptr, nullptr, nullptr};
            const int rc =
                (l + 1 == sm)
                    ? launch_phase<ST, false, float>(ldims(lv), ldims(cv), mg.post, Lv<ST>::fx(lv), Lv<ST>::fy(lv),
                                                     Lv<ST>::fz(lv), B(l), cur[l], cv.p, out, nullptr, mg.omega,
                                                     done, bsc, nf, df, s)
                    : launch_phase<ST, false, ST>(ldims(lv), ldims(cv), mg.post, Lv<ST>::fx(lv), Lv<ST>::fy(lv),
                                                  Lv<ST>::fz(lv), B(l), cur[l], cur[l + 1], out, nullptr,
                                                  mg.omega, done, bsc, nf, df, s);
            if (dots && dot_done) *dot_done = true;
            if (rc) return rc;
            cur[l] = out;
            continue;
        }
        // the first post-sweep forms the prolongation itself when the last
        // post-sweep then lands where it must (level 0: in z0)
        if (fused_smoother(mg, l) && mg.post > 0 &&
            (l > 0 || ((mg.post % 2) ? other(0, cur[0]) : cur[0]) == z0)) {
            const Dims d = ldims(lv);
            ST* out = other(l, cur[l]);
            const float* bsc = l == 0 ? bscale : nullptr;
            int rc = (l + 1 == sm)
                         ? launch_full_sweep<ST, false, true, float>(d, Lv<ST>::fx(lv), Lv<ST>::fy(lv),
                                                                           Lv<ST>::fz(lv), cur[l], out, B(l), 1,
                                                                           mg.omega, done, bsc, s, cv.p, ldims(cv))
                               : launch_full_sweep<ST, false, true, ST>(d, Lv<ST>::fx(lv), Lv<ST>::fy(lv),
                                                                        Lv<ST>::fz(lv), cur[l], out, B(l), 1,
                                                                        mg.omega, done, bsc, s, cur[l + 1],
                                                                        ldims(cv));
            if (rc) return rc;
            cur[l] = out;
            rc = smooth(l, mg.post - 1, true, false);
            if (rc) return rc;
            continue;
        }
        // prolongation target: in place, except on level 0 where the last
        // post-sweep must land in z0
        ST* dst = cur[l];
        if (l == 0) dst = (fused_smoother(mg, 0) && (mg.post % 2)) ? second_buffer<ST>(mg, 0) : z0;
        const unsigned grid = cdiv(ncell(lv), RT);
        if (l + 1 == sm)
            k_prolong<ST, float><<<grid, RT, 0, s>>>(ldims(lv), ldims(cv), cur[l], dst, cv.p, done);
        else
            k_prolong<ST, ST><<<grid, RT, 0, s>>>(ldims(lv), ldims(cv), cur[l], dst, cur[l + 1], done);
        PF_CHECK_LAUNCH();
        cur[l] = dst;
        int rc = smooth(l, mg.post, true, false);
        if (rc) return rc;
    }
    return PF_OK;
}

// Host-side state of one solver (caller-owned through pf_mgpcg_state_*):
// the pinned int the residual tests publish to (the host polls it, no
// events), and the HIP graphs captured for this solver's buffers.  Bound to the device current at
// creation.
struct SolveGraphs;
struct SolverState {
    int device = -1;
    int* flag = nullptr;    // HW_WORDS pinned ints (host address)
    int* flag_d = nullptr;  // the same memory as the device addresses it
    int solves = 0;         // results published so far
    std::vector<SolveGraphs>* graphs = nullptr;
};

static void release_state(SolverState& st);

static int init_state(SolverState& st) {
    PF_CHECK_HIP(hipGetDevice(&st.device));
    // coherent: the device's stores reach host memory without cache flushes
    PF_CHECK_HIP(hipHostMalloc(reinterpret_cast<void**>(&st.flag), HW_WORDS * sizeof(int),
                               hipHostMallocMapped | hipHostMallocCoherent));
    for (int w = 0; w < HW_WORDS; ++w) st.flag[w] = 0;
    PF_CHECK_HIP(hipHostGetDevicePointer(reinterpret_cast<void**>(&st.flag_d), st.flag, 0));
    return PF_OK;
}

// The V-cycle's right-hand-side scale of a solve that reads z scaled.
template <typename ST>
static const float* vcycle_scale(const CGK<ST>& a) {
    return a.zscale ? &a.st->vscale : nullptr;
}

// Kernels of one FPCG iteration; `flag` (the device address of pinned host
// memory) receives the done flag from the residual test's combine kernel.
// Every kernel returns at once when the flag is set, so an iteration
// enqueued past convergence does nothing.
// The residual test rides in the V-cycle's first kernel when that is the
// fused zero-start sweep or pre phase of an HBM level 0.
static bool fold_residual_test(const pf_mg& mg) {
    return mg.small_from > 0 && mg.pre > 0 && fused_smoother(mg, 0);
}

// The inner products after the V-cycle ride on its last level-0 kernel when
// that is the post phase or a plain fused sweep (at least two post-sweeps on
// an HBM level 0) whose workgroups fit the partials array.  A grid that cannot
// be halved has no post-smoothing: its only level ends with the mean removal.
static int64_t dot_blocks(const pf_mg& mg) {
    const Dims d = ldims(mg.lev[0]);
    return level_fused(mg, 0) ? (int64_t)phase_tiles(d, phase_tile(d)) : sweep_tiles(d, sweep_shape(d, mg.precision != 0));
}
static bool fold_dots(const pf_mg& mg) {
    return !(mg.options & PF_MG_SEPARATE_DOTS) && mg.nlev > 1 && mg.small_from > 0 &&
           (mg.post >= 2 || level_fused(mg, 0)) && fused_smoother(mg, 0) && dot_blocks(mg) <= PS;
}

template <typename ST>
static int enqueue_iteration(const pf_mg& mg, const CGK<ST>& a, ST* z, const int* done, int* flag,
                             unsigned nb, hipStream_t s) {
    CGState* st = a.st;
    k_cg_apply<ST><<<a.np_apply, WT, 0, s>>>(a);
    PF_CHECK_LAUNCH();
    k_cg_update<ST><<<nb, RT, 0, s>>>(a);
    PF_CHECK_LAUNCH();
    const UpdateFold uf{st, (int)nb, flag};
    const bool fold = fold_residual_test(mg);
    if (!fold) {
        k_comb<<<1, RT, 0, s>>>(st, C_UPDATE, (int)nb, a.n, nullptr, 0.0, flag);
        PF_CHECK_LAUNCH();
    }
    const DotFold df{a.Ap, a.zscale, st};
    const bool dots = fold_dots(mg);
    bool dot_done = false;
    int rc = vcycle<ST>(mg, a.r, z, done, vcycle_scale(a), s, fold ? &uf : nullptr, dots ? &df : nullptr,
                        &dot_done);
    if (rc) return rc;
    PF_REQUIRE(dot_done == dots, "pf_mgpcg_solve: the V-cycle's last level-0 kernel is not a plain fused sweep");
    if (!dots) {
        k_cg_beta<ST><<<a.np_beta, WT, 0, s>>>(a);
        PF_CHECK_LAUNCH();
    }
    return PF_OK;
}

// First preconditioner application (poisson.py:378-380); the first search
// direction is formed inside the first iteration's k_cg_apply (beta = 0).
template <typename ST>
static int enqueue_prologue(const pf_mg& mg, const CGK<ST>& a, ST* z, const int* done, unsigned nb,
                            hipStream_t s) {
    int rc = vcycle<ST>(mg, a.r, z, done, vcycle_scale(a), s);
    if (rc) return rc;
    k_cg_first<ST><<<nb, RT, 0, s>>>(a);
    PF_CHECK_LAUNCH();
    k_comb<<<1, RT, 0, s>>>(a.st, C_FIRST, (int)nb, a.n, nullptr, 0.0);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

// _remove_mean(x) (poisson.py:408), then the result for the host
static int enqueue_epilogue(CGState* st, float* x, int64_t n, unsigned nb, int* words, hipStream_t s) {
    k_part_sum<float><<<nb, RT, 0, s>>>(x, n, st->part);
    PF_CHECK_LAUNCH();
    k_comb<<<1, RT, 0, s>>>(st, C_MEAN, (int)nb, n, &st->mu_x, 0.0);
    PF_CHECK_LAUNCH();
    k_shift<float, float><<<nb, RT, 0, s>>>(x, x, n, &st->mu_x);
    PF_CHECK_LAUNCH();
    k_publish_result<<<1, 64, 0, s>>>(st, words);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

// HIP graphs of the prologue, of one iteration (two instances that differ
// only in which search-direction buffer they write) and of an odd and an
// even iteration together, cached per solver layout.  A solve issues one
// graph launch per two iterations instead of ~20 kernel launches each.
// pair: an odd iteration and the even one after it in one graph; the GPU
// spends ~8 us between two graphs, none between two kernels of one graph
struct SolveGraphs {
    std::vector<uint64_t> key;
    hipGraphExec_t pro = nullptr;
    hipGraphExec_t it[2] = {nullptr, nullptr};
    hipGraphExec_t pair = nullptr;
    hipGraphExec_t epi = nullptr;  // mean removal and the result for the host
};

static void destroy_graphs(SolveGraphs& g) {
    if (g.pro) (void)hipGraphExecDestroy(g.pro);
    for (auto& e : g.it)
        if (e) (void)hipGraphExecDestroy(e);
    if (g.pair) (void)hipGraphExecDestroy(g.pair);
    if (g.epi) (void)hipGraphExecDestroy(g.epi);
    g.pro = g.it[0] = g.it[1] = g.pair = g.epi = nullptr;
}

template <typename F>
static int capture(hipStream_t cs, F&& enqueue, hipGraphExec_t* out) {
    PF_CHECK_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeRelaxed));
    const int rc = enqueue(cs);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(cs, &g);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return set_error((int)e, "hipStreamEndCapture: %s", hipGetErrorString(e));
    const hipError_t ei = hipGraphInstantiate(out, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ei != hipSuccess) return set_error((int)ei, "hipGraphInstantiate: %s", hipGetErrorString(ei));
    return PF_OK;
}

// Iteration `slot` (= iteration number & 1) writes its search direction to
// mg.q (slot 0) or mg.rhs (slot 1) and reads the other one.
template <typename ST>
static CGK<ST> slot_args(const CGK<ST>& a, const pf_mg& mg, int slot) {
    CGK<ST> b = a;
    b.q = slot ? mg.rhs : mg.q;
    b.q_old = slot ? mg.q : mg.rhs;
    b.slot = slot;
    return b;
}

// Everything a captured graph bakes in: the hierarchy's sizes, scalars and
// buffer addresses, the solve's vectors, the flag slot and the launch shape.
template <typename ST>
static std::vector<uint64_t> graph_key(const pf_mg& mg, const CGK<ST>& a, const ST* z, const int* flag,
                                       unsigned nb) {
    std::vector<uint64_t> k;
    auto ptr = [&](const void* p) { k.push_back((uint64_t)(uintptr_t)p); };
    uint32_t om;
    std::memcpy(&om, &mg.omega, sizeof(om));
    k.insert(k.end(), {(uint64_t)mg.nlev, (uint64_t)mg.pre, (uint64_t)mg.post, (uint64_t)mg.coarsest, om,
                       (uint64_t)mg.precision, (uint64_t)mg.small_from, (uint64_t)mg.options,
                       (uint64_t)sizeof(ST), (uint64_t)nb});
    for (int l = 0; l < mg.nlev; ++l) {
        const pf_mg_level& v = mg.lev[l];
        k.insert(k.end(), {(uint64_t)v.nx, (uint64_t)v.ny, (uint64_t)v.nz});
        for (const void* p : {(const void*)v.bx, (const void*)v.by, (const void*)v.bz, (const void*)v.diag,
                              (const void*)v.p, (const void*)v.b, (const void*)v.r, (const void*)v.bx_h,
                              (const void*)v.by_h, (const void*)v.bz_h, (const void*)v.p_h})
            ptr(p);
    }
    for (const void* p : {(const void*)mg.rhs, (const void*)mg.res, (const void*)mg.z, (const void*)mg.q,
                          (const void*)mg.Ap, (const void*)mg.scalars, (const void*)a.b, (const void*)a.x,
                          (const void*)z, (const void*)flag})
        ptr(p);
    return k;
}

template <typename ST>
static int get_graphs(SolverState& st, const pf_mg& mg, const CGK<ST>& a, ST* z, const int* done,
                      unsigned nb, SolveGraphs*& out) {
    std::vector<SolveGraphs>& cache = *st.graphs;
    std::vector<uint64_t> key = graph_key<ST>(mg, a, z, st.flag, nb);
    for (auto& c : cache)
        if (c.key == key) {
            out = &c;
            return PF_OK;
        }
    int rc = ensure_small_lds();
    if (rc) return rc;
    SolveGraphs g;
    g.key = std::move(key);
    hipStream_t cs = nullptr;
    PF_CHECK_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
    rc = capture(cs, [&](hipStream_t t) { return enqueue_prologue<ST>(mg, a, z, done, nb, t); }, &g.pro);
    for (int q = 0; q < 2 && !rc; ++q) {
        const CGK<ST> aq = slot_args(a, mg, q);
        rc = capture(cs, [&](hipStream_t t) { return enqueue_iteration<ST>(mg, aq, z, done, st.flag_d, nb, t); },
                     &g.it[q]);
    }
    if (!rc) {
        const CGK<ST> a1 = slot_args(a, mg, 1), a0 = slot_args(a, mg, 0);
        rc = capture(
            cs,
            [&](hipStream_t t) {
                const int r1 = enqueue_iteration<ST>(mg, a1, z, done, st.flag_d, nb, t);
                return r1 ? r1 : enqueue_iteration<ST>(mg, a0, z, done, st.flag_d, nb, t);
            },
            &g.pair);
    }
    if (!rc)
        rc = capture(
            cs, [&](hipStream_t t) { return enqueue_epilogue(a.st, a.x, a.n, nb, st.flag_d, t); }, &g.epi);
    (void)hipStreamDestroy(cs);
    if (rc) {
        destroy_graphs(g);
        return rc;
    }
    // a solver is normally solved with one set of vectors; keep a few
    if (cache.size() >= 4) {
        destroy_graphs(cache.front());
        cache.erase(cache.begin());
    }
    cache.push_back(std::move(g));
    out = &cache.back();
    return PF_OK;
}

static void release_state(SolverState& st) {
    if (st.graphs) {
        for (auto& g : *st.graphs) destroy_graphs(g);
        delete st.graphs;
        st.graphs = nullptr;
    }
    if (st.flag) (void)hipHostFree(st.flag);
    st.flag = st.flag_d = nullptr;
}

static bool use_graphs() {
    static const bool on = [] {
        const char* e = std::getenv("PFFLIP_SOLVER_GRAPHS");
        return !(e && e[0] == '0');
    }();
    return on;
}

// Spin until the published counter (see publish_done) reaches `seq`; *stop
// = the solve is done.  The stream running dry without that publication is
// an error, so the loop cannot spin forever.
static int wait_published(const int* flag, int seq, hipStream_t s, bool* stop) {
    const volatile int* f = flag;
    for (unsigned spin = 0;; ++spin) {
        const int v = *f;
        if ((v >> 1) >= seq) {
            *stop = (v & 1) != 0;
            return PF_OK;
        }
        if ((spin & 255) == 255) {
            const hipError_t q = hipStreamQuery(s);
            if (q == hipSuccess) {
                const int w = *f;
                if ((w >> 1) >= seq) {
                    *stop = (w & 1) != 0;
                    return PF_OK;
                }
                return set_error(PF_ERR_INVALID, "pf_mgpcg_solve: residual test %d was never published", seq);
            }
            if (q != hipErrorNotReady)
                return set_error((int)q, "pf_mgpcg_solve: %s", hipGetErrorString(q));
        }
        __builtin_ia32_pause();
    }
}

// Spin until k_publish_result stored `number` (the stream running dry
// without it is an error, so the loop cannot spin forever); the result
// words are read after it (x86 keeps loads in order).
static int wait_result(const int* words, int number, hipStream_t s) {
    const volatile int* f = words + HW_RESULT_NO;
    for (unsigned spin = 0;; ++spin) {
        if (*f == number) break;
        if ((spin & 255) == 255) {
            const hipError_t q = hipStreamQuery(s);
            if (q == hipSuccess) {
                if (*f == number) break;
                return set_error(PF_ERR_INVALID, "pf_mgpcg_solve: the result was never published");
            }
            if (q != hipErrorNotReady) return set_error((int)q, "pf_mgpcg_solve: %s", hipGetErrorString(q));
        }
        __builtin_ia32_pause();
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return PF_OK;
}

template <typename ST>
static int solve_impl(const pf_mg& mg, const float* b, float* x, double tol, int max_iter,
                      int* it_out, double* rel_out, hipStream_t s) {
    CGState* st = static_cast<CGState*>(mg.scalars);
    const pf_mg_level& l0 = mg.lev[0];
    const Dims d = ldims(l0);
    const int64_t n = ncell(l0);
    ST* z = (sizeof(ST) == 4) ? reinterpret_cast<ST*>(mg.z) : Lv<ST>::p(l0);
    CGK<ST> a;
    a.d = d;
    a.n = n;
    a.bx = l0.bx;
    a.by = l0.by;
    a.bz = l0.bz;
    a.b = b;
    a.rhs = mg.rhs;
    a.x = x;
    a.r = mg.res;
    a.q = mg.q;  // zeroed by k_cg_init: iteration 1 (slot 1) reads it as q_old
    a.q_old = mg.rhs;
    a.Ap = mg.Ap;
    a.z = z;
    // 16-bit iterates: scale the V-cycle's input (not for a whole hierarchy
    // in LDS, which computes in FP32 and rounds only its output)
    a.zscale = (sizeof(ST) == 2 && mg.small_from > 0) ? &st->vscale_inv : nullptr;
    a.st = st;
    a.tol = tol;
    const unsigned nb = red_blocks(n);
    a.slot = 1;
    a.np_apply = a.np_beta = (int)std::min<int64_t>(WB, (n + WT - 1) / WT);
    if (fold_dots(mg)) a.np_beta = (int)dot_blocks(mg);  // one partial per level-0 tile
    const int* done = &st->done;

    k_part_sum<float><<<nb, RT, 0, s>>>(b, n, st->part);
    PF_CHECK_LAUNCH();
    k_comb<<<1, RT, 0, s>>>(st, C_MEAN_RESET, (int)nb, n, &st->mu, 0.0);
    PF_CHECK_LAUNCH();
    k_cg_init<ST><<<nb, RT, 0, s>>>(a);
    PF_CHECK_LAUNCH();
    // b == 0 after mean removal (poisson.py:366-368): C_INIT sets done = 2
    // and rel = 0, x stays k_cg_init's zeros, every later kernel exits on the
    // flag and the first residual test stops the host loop, so the result
    // is (0, 0) without a synchronisation here
    k_comb<<<1, RT, 0, s>>>(st, C_INIT, (int)nb, n, nullptr, tol);
    PF_CHECK_LAUNCH();
    // the caller's solver state (graphs, flags), or a temporary one for this
    // call (no graphs)
    SolverState local;
    struct LocalGuard {
        SolverState& s;
        ~LocalGuard() { release_state(s); }
    } guard{local};
    SolverState* hp = static_cast<SolverState*>(mg.host_state);
    int rc = PF_OK;
    if (hp) {
        int dev = 0;
        PF_CHECK_HIP(hipGetDevice(&dev));
        PF_REQUIRE(dev == hp->device, "pf_mgpcg_solve: solver state was created on device %d, current is %d",
                   hp->device, dev);
    } else {
        rc = init_state(local);
        if (rc) return rc;
        hp = &local;
    }
    // the previous solve's last publication must not be read as this one's
    // (its kernels have all completed: it ended with a stream synchronize)
    static_cast<volatile int*>(hp->flag)[0] = 0;
    SolveGraphs* gr = nullptr;
    if (use_graphs() && max_iter > 0 && hp->graphs) {
        rc = get_graphs<ST>(*hp, mg, a, z, done, nb, gr);
        if (rc) return rc;
    }
    if (gr) {
        PF_CHECK_HIP(hipGraphLaunch(gr->pro, s));
    } else {
        rc = enqueue_prologue<ST>(mg, a, z, done, nb, s);
        if (rc) return rc;
    }
    for (int it = 1; it <= max_iter;) {
        const int slot = it & 1;
        // graphs: iterations in (odd, even) pairs, one graph each (single
        // iterations without graphs and for an odd max_iter's last).  Then
        // wait for the last launched iteration's residual test: it opens
        // that iteration's first kernel, so the rest of the iteration (about
        // 200 us at 128^3) is still queued while the host launches the next
        // one, and after convergence at most the iteration that found it and
        // one more run (as early exits).
        int step = 1;
        if (gr) {
            if (slot == 1 && it < max_iter) {
                PF_CHECK_HIP(hipGraphLaunch(gr->pair, s));
                step = 2;
            } else {
                PF_CHECK_HIP(hipGraphLaunch(gr->it[slot], s));
            }
        } else {
            rc = enqueue_iteration<ST>(mg, slot_args(a, mg, slot), z, done, hp->flag_d, nb, s);
            if (rc) return rc;
        }
        bool stop = false;
        rc = wait_published(hp->flag, it + step - 1, s, &stop);
        if (rc) return rc;
        if (stop) break;
        it += step;
    }
    // _remove_mean(x) (poisson.py:408) and the result, published under the
    // solve's number
    const int number = ++hp->solves;
    static_cast<volatile int*>(hp->flag)[HW_WANT] = number;
    if (gr) {
        PF_CHECK_HIP(hipGraphLaunch(gr->epi, s));
    } else {
        rc = enqueue_epilogue(st, x, n, nb, hp->flag_d, s);
        if (rc) return rc;
    }
    rc = wait_result(hp->flag, number, s);
    if (rc) return rc;
    const volatile int* w = hp->flag;
    *it_out = w[HW_IT];
    *rel_out = __builtin_bit_cast(double, *reinterpret_cast<const volatile unsigned long long*>(w + HW_REL));
    return PF_OK;
}

template <typename ST>
static int precondition_impl(const pf_mg& mg, const float* r, float* z, hipStream_t s) {
    CGState* st = static_cast<CGState*>(mg.scalars);
    const int64_t n = ncell(mg.lev[0]);
    ST* zt = (sizeof(ST) == 4) ? reinterpret_cast<ST*>(z) : Lv<ST>::p(mg.lev[0]);
    int rc = vcycle<ST>(mg, r, zt, nullptr, nullptr, s);
    if (rc) return rc;
    k_part_sum<ST><<<red_blocks(n), RT, 0, s>>>(zt, n, st->part);
    PF_CHECK_LAUNCH();
    k_comb<<<1, RT, 0, s>>>(st, C_MEAN, (int)red_blocks(n), n, &st->mu_x, 0.0);
    PF_CHECK_LAUNCH();
    k_shift<ST, float><<<red_blocks(n), RT, 0, s>>>(zt, z, n, &st->mu_x);
    PF_CHECK_LAUNCH();
    return PF_OK;
}

static int check_mg(const pf_mg* mg) {
    PF_REQUIRE(mg, "null pf_mg");
    PF_REQUIRE(mg->nlev >= 1 && mg->nlev <= PF_MAX_LEVELS, "pf_mg: bad level count %d", mg->nlev);
    PF_REQUIRE(mg->precision >= 0 && mg->precision <= 2, "pf_mg: bad precision %d", mg->precision);
    PF_REQUIRE(mg->pre >= 0 && mg->post >= 0 && mg->coarsest >= 0, "pf_mg: negative sweep count");
    PF_REQUIRE(mg->scalars, "pf_mg: null scalar workspace");
    PF_REQUIRE(mg->small_from >= 0 && mg->small_from <= mg->nlev, "pf_mg: call pf_mg_setup first");
    for (int l = 0; l < mg->nlev; ++l) {
        const pf_mg_level& v = mg->lev[l];
        PF_REQUIRE(v.nx > 0 && v.ny > 0 && v.nz > 0, "pf_mg: level %d has bad dims", l);
        // the kernels index cells and faces with 32-bit ints
        PF_REQUIRE((int64_t)(v.nx + 1) * (v.ny + 1) * (v.nz + 1) < ((int64_t)1 << 31), "pf_mg: level %d too large", l);
        PF_REQUIRE(v.bx && v.by && v.bz && v.b, "pf_mg: level %d missing arrays", l);
        if (l > 0) {
            const pf_mg_level& f = mg->lev[l - 1];
            PF_REQUIRE(f.nx == 2 * v.nx && f.ny == 2 * v.ny && f.nz == 2 * v.nz,
                       "pf_mg: level %d is not the 2x coarsening of level %d", l, l - 1);
        }
        if (mg->precision != 0 && l < mg->small_from)
            PF_REQUIRE(v.bx_h && v.by_h && v.bz_h && v.p_h, "pf_mg: level %d missing 16-bit arrays", l);
        // level 0's 16-bit iterate holds the preconditioned vector z
        if (mg->precision != 0 && l == 0) PF_REQUIRE(v.p_h, "pf_mg: level 0 missing its 16-bit iterate");
        if (l > 0 && (mg->precision == 0 || l >= mg->small_from)) PF_REQUIRE(v.p, "pf_mg: level %d missing p", l);
        // the fused smoother's second iterate buffer on the HBM levels
        if (l < mg->small_from) {
            PF_REQUIRE(v.r, "pf_mg: level %d missing r (second smoother buffer)", l);
            if (l == 0 && mg->precision == 0) PF_REQUIRE(v.p, "pf_mg: level 0 missing p (second smoother buffer)");
        }
    }
    return PF_OK;
}

}  // namespace pf

using namespace pf;

PF_API size_t pf_mg_scalar_bytes(void) { return sizeof(CGState); }

PF_API int pf_mg_setup(pf_mg* mg) {
    PF_REQUIRE(mg, "pf_mg_setup: null pf_mg");
    PF_REQUIRE(mg->nlev >= 1 && mg->nlev <= PF_MAX_LEVELS, "pf_mg_setup: bad level count");
    int sm = mg->nlev;
    for (int l = mg->nlev - 1; l >= 0; --l) {
        const int64_t nc = (int64_t)mg->lev[l].nx * mg->lev[l].ny * mg->lev[l].nz;
        const int64_t bytes = small_lds_floats(*mg, l, nullptr, nullptr, nullptr) * (int64_t)sizeof(float);
        const Dims d{mg->lev[l].nx, mg->lev[l].ny, mg->lev[l].nz};
        if (nc <= kSmallMaxCells && bytes <= kSmallMaxBytes && colour_space(d) <= kSmallThreads * kTopPairs)
            sm = l;
        else
            break;
    }
    mg->small_from = sm;
    return PF_OK;
}

PF_API int pf_mg_build(const pf_mg* mg, const float* bx, const float* by, const float* bz,
                       pf_stream_t stream) {
    int rc = check_mg(mg);
    if (rc) return rc;
    PF_REQUIRE(bx && by && bz, "pf_mg_build: null coefficients");
    hipStream_t s = S(stream);
    const pf_mg_level& l0 = mg->lev[0];
    const Dims d0 = ldims(l0);
    const float* src[3] = {bx, by, bz};
    float* dst[3] = {l0.bx, l0.by, l0.bz};
    for (int q = 0; q < 3; ++q)
        if (src[q] != dst[q])
            PF_CHECK_HIP(hipMemcpyAsync(dst[q], src[q], face_count(d0, q) * sizeof(float),
                                        hipMemcpyDeviceToDevice, s));
    for (int l = 0; l < mg->nlev; ++l) {
        const pf_mg_level& v = mg->lev[l];
        const Dims d = ldims(v);
        if (l > 0) {
            const pf_mg_level& f = mg->lev[l - 1];
            const int64_t n = (int64_t)(d.nx + 1) * (d.ny + 1) * (d.nz + 1);
            k_galerkin<<<cdiv(n, RT), RT, 0, s>>>(ldims(f), d, f.bx, f.by, f.bz, v.bx, v.by, v.bz);
            PF_CHECK_LAUNCH();
        }
        const int64_t n = (int64_t)(d.nx + 1) * (d.ny + 1) * (d.nz + 1);
        const bool copy = mg->precision != 0 && l < mg->small_from;
        if (mg->precision == 2)
            k_diag_copy<fp16s><<<cdiv(n, RT), RT, 0, s>>>(
                d, v.bx, v.by, v.bz, v.diag, copy ? reinterpret_cast<fp16s*>(v.bx_h) : nullptr,
                reinterpret_cast<fp16s*>(v.by_h), reinterpret_cast<fp16s*>(v.bz_h));
        else
            k_diag_copy<bf16s><<<cdiv(n, RT), RT, 0, s>>>(
                d, v.bx, v.by, v.bz, v.diag, copy ? reinterpret_cast<bf16s*>(v.bx_h) : nullptr,
                reinterpret_cast<bf16s*>(v.by_h), reinterpret_cast<bf16s*>(v.bz_h));
        PF_CHECK_LAUNCH();
    }
    if (use_coarse_op(*mg)) {
        const pf_mg_level& c = mg->lev[mg->nlev - 1];
        const int n = c.nx * c.ny * c.nz;
        const int threads = ((n + 63) / 64) * 64;
        k_coarse_op<<<n, threads, 0, s>>>(ldims(c), c.bx, c.by, c.bz, mg->coarsest, mg->omega,
                                          static_cast<CGState*>(mg->scalars)->coarse_op);
        PF_CHECK_LAUNCH();
    }
    return PF_OK;
}

PF_API int pf_mg_precondition(const pf_mg* mg, const float* r, float* z, pf_stream_t stream) {
    int rc = check_mg(mg);
    if (rc) return rc;
    PF_REQUIRE(r && z, "pf_mg_precondition: null vector");
    switch (mg->precision) {
        case 0: return precondition_impl<float>(*mg, r, z, S(stream));
        case 1: return precondition_impl<bf16s>(*mg, r, z, S(stream));
        default: return precondition_impl<fp16s>(*mg, r, z, S(stream));
    }
}

// One V-cycle from a zero guess, without the final mean removal of
// pf_mg_precondition.  FP32 hierarchies only: the 16-bit V-cycles keep their
// level-0 iterate in 16-bit storage with a scale that pf_mg_precondition
// and pf_mgpcg_solve undo.
PF_API int pf_mg_vcycle(const pf_mg* mg, const float* r, float* z, pf_stream_t stream) {
    int rc = check_mg(mg);
    if (rc) return rc;
    PF_REQUIRE(r && z, "pf_mg_vcycle: null vector");
    PF_REQUIRE(mg->precision == 0, "pf_mg_vcycle: FP32 hierarchies only (precision %d)", mg->precision);
    // level 0 ping-pongs between z and the hierarchy's own p
    PF_REQUIRE((const void*)z != (const void*)r && (const void*)z != (const void*)mg->lev[0].p &&
                   (const void*)r != (const void*)mg->lev[0].p,
               "pf_mg_vcycle: r, z and the level-0 p buffer must be distinct");
    return vcycle<float>(*mg, r, z, nullptr, nullptr, S(stream));
}

PF_API int pf_mgpcg_state_create(void** out) {
    PF_REQUIRE(out, "pf_mgpcg_state_create: null argument");
    *out = nullptr;
    SolverState* st = new (std::nothrow) SolverState();
    PF_REQUIRE(st, "pf_mgpcg_state_create: out of host memory");
    int rc = init_state(*st);
    if (!rc) {
        st->graphs = new (std::nothrow) std::vector<SolveGraphs>();
        if (!st->graphs) rc = set_error(PF_ERR_INVALID, "pf_mgpcg_state_create: out of host memory");
    }
    if (rc) {
        release_state(*st);
        delete st;
        return rc;
    }
    *out = st;
    return PF_OK;
}

PF_API int pf_mgpcg_state_destroy(void* state) {
    if (!state) return PF_OK;
    SolverState* st = static_cast<SolverState*>(state);
    int cur = 0;
    const bool switched = hipGetDevice(&cur) == hipSuccess && cur != st->device;
    if (switched) (void)hipSetDevice(st->device);
    release_state(*st);
    if (switched) (void)hipSetDevice(cur);
    delete st;
    return PF_OK;
}

PF_API int pf_mgpcg_solve(const pf_mg* mg, const float* b, float* x, double tol, int32_t max_iter,
                          int32_t* it_out, double* rel_out, pf_stream_t stream) {
    int rc = check_mg(mg);
    if (rc) return rc;
    PF_REQUIRE(b && x && it_out && rel_out, "pf_mgpcg_solve: null argument");
    PF_REQUIRE(mg->rhs && mg->res && mg->q && mg->Ap, "pf_mgpcg_solve: missing CG vectors");
    PF_REQUIRE(mg->precision != 0 || mg->z, "pf_mgpcg_solve: missing z");
    PF_REQUIRE(max_iter >= 0, "pf_mgpcg_solve: negative max_iter");
    switch (mg->precision) {
        case 0: return solve_impl<float>(*mg, b, x, tol, max_iter, it_out, rel_out, S(stream));
        case 1: return solve_impl<bf16s>(*mg, b, x, tol, max_iter, it_out, rel_out, S(stream));
        default: return solve_impl<fp16s>(*mg, b, x, tol, max_iter, it_out, rel_out, S(stream));
    }
}

template <typename ST>
static int time_smoother_impl(const pf_mg& mg, int level, int reps, float* ms_out, hipStream_t s) {
    const pf_mg_level& lv = mg.lev[level];
    const Dims d = ldims(lv);
    ST* pa = level == 0 ? (sizeof(ST) == 4 ? reinterpret_cast<ST*>(mg.z) : Lv<ST>::p(lv)) : Lv<ST>::p(lv);
    ST* pb = second_buffer<ST>(mg, level);
    const float* b = level == 0 ? mg.res : lv.b;
    const bool fused = fused_smoother(mg, level);
    const int64_t nthr = (int64_t)d.nx * d.ny * ((d.nz + 1) / 2);
    const unsigned grid = cdiv(nthr, RT);
    hipEvent_t e0, e1;
    PF_CHECK_HIP(hipEventCreate(&e0));
    PF_CHECK_HIP(hipEventCreate(&e1));
    auto run = [&]() -> int {
        for (int r = 0; r < reps; ++r) {
            if (fused) {
                const int rc = launch_full_sweep<ST, false>(d, Lv<ST>::fx(lv), Lv<ST>::fy(lv), Lv<ST>::fz(lv),
                                                            r % 2 ? pb : pa, r % 2 ? pa : pb, b, 0, mg.omega,
                                                            nullptr, nullptr, s);
                if (rc) return rc;
            } else {
                for (int c = 0; c < 2; ++c) {
                    k_rbgs<ST, false><<<grid, RT, 0, s>>>(d, Lv<ST>::fx(lv), Lv<ST>::fy(lv), Lv<ST>::fz(lv), pa,
                                                          b, c, mg.omega, nullptr, nullptr);
                    PF_CHECK_LAUNCH();
                }
            }
        }
        return PF_OK;
    };
    int rc = run();  // warm-up
    if (!rc) {
        PF_CHECK_HIP(hipEventRecord(e0, s));
        rc = run();
    }
    if (!rc) {
        PF_CHECK_HIP(hipEventRecord(e1, s));
        PF_CHECK_HIP(hipEventSynchronize(e1));
        float ms = 0.f;
        PF_CHECK_HIP(hipEventElapsedTime(&ms, e0, e1));
        *ms_out = ms / (fused ? (float)reps : 2.0f * reps);
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return rc;
}

PF_API int pf_mg_time_smoother(const pf_mg* mg, int32_t level, int32_t reps, float* ms_out,
                               pf_stream_t stream) {
    int rc = check_mg(mg);
    if (rc) return rc;
    PF_REQUIRE(ms_out && reps > 0, "pf_mg_time_smoother: bad arguments");
    PF_REQUIRE(level >= 0 && level < mg->nlev && level < mg->small_from,
               "pf_mg_time_smoother: level %d is not smoothed out of HBM", level);
    PF_REQUIRE(level > 0 || mg->precision != 0 || mg->z, "pf_mg_time_smoother: missing z");
    switch (mg->precision) {
        case 0: return time_smoother_impl<float>(*mg, level, reps, ms_out, S(stream));
        case 1: return time_smoother_impl<bf16s>(*mg, level, reps, ms_out, S(stream));
        default: return time_smoother_impl<fp16s>(*mg, level, reps, ms_out, S(stream));
    }
}

PF_API int pf_apply_A(int nx, int ny, int nz, const float* p, const float* bx, const float* by,
                      const float* bz, const float* diag, float* out, pf_stream_t stream) {
    PF_REQUIRE(nx > 0 && ny > 0 && nz > 0, "pf_apply_A: bad grid");
    PF_REQUIRE(p && bx && by && bz && out, "pf_apply_A: null argument");
    const int64_t n = (int64_t)nx * ny * nz;
    k_apply_A<<<cdiv(n, RT), RT, 0, S(stream)>>>(Dims{nx, ny, nz}, p, bx, by, bz, diag, out);
    PF_CHECK_LAUNCH();
    return PF_OK;
}
