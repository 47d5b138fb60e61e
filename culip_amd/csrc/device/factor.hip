// Numeric BILDLt factor for gfx950, one level at a time.
//
// Reference: libs/la/preconditioner/block_ildlt.impl.cuh:1519-1671 (schedule)
// and block_ildlt_kernels.impl.cuh:1146-2074 (kernels). Per level:
//   k_pivots_pairs
//               one or four waves per pivot block: A_ii -= sum_k U_ki' D_k U_ki over
//               the block column, 1x1/2x2 LDL' of the tile (static or
//               numeric pivots), row sums; in the same launch, one lane per
//               small off-diagonal block: its Schur updates
//   k_offdiag_tiny_scale
//               those blocks through U_ii' and D, row partial sums, compact
//               entries
//   k_offdiag   one wave per off-diagonal block: A_ij -= sum_k U_ki' D_k U_kj
//               over the block's symbolic Schur pairs, U_ij = D_i \ (U_ii' \
//               A_ij), per-row partial sums of squares; the result leaves as
//               a dense tile or as a compact (index, value) list of the
//               entries with |v| > 1e-10
//   k_drop      one workgroup per row group: row sums of squares in a fixed
//               order, entries surviving the threshold, leftover-space pool in
//               level-list order, granted extra space, the factored metadata
//               and the final storage of blocks with few entries
//   k_store     one wave per remaining block: compacted final storage
//
// The dependency blocks of a tile are walked with their metadata fetched
// lane-parallel up front. A block (or pair of blocks) of few entries has its
// whole update formed by its own lane, and the updates are applied in block
// order; other blocks are staged as tiles. The update U' D U is applied over the nonzero rows
// of the right factor only, with D applied on the fly: every term the
// reference adds is added, in the same order with the same fused
// multiply-adds as the CPU oracle's restatement; the skipped terms are exact
// zeros. FP64 factors therefore agree with the oracle bit for bit.
#include "factor.hpp"
#include "wave.hpp"

#include <hip/hip_runtime.h>

namespace culip {

namespace {

constexpr double NZ_EPS = 1e-10;

template<typename T>
__device__ __forceinline__ bool finite_value(T v) { return fabs(v) < (T) INFINITY; }

// first Schur pair of an off-diagonal task: low and high 32 bits in the
// third int4's x and w
__device__ __forceinline__ int64_t pair_first(int4 t2)
{
    return (int64_t) (((uint64_t) (uint32_t) t2.w << 32) | (uint32_t) t2.x);
}

__device__ __forceinline__ double lane_value(double v, int src)
{
    const unsigned long long b = (unsigned long long) __double_as_longlong(v);
    const unsigned lo = (unsigned) __builtin_amdgcn_readlane((int) (unsigned) b, src);
    const unsigned hi = (unsigned) __builtin_amdgcn_readlane((int) (unsigned) (b >> 32), src);
    return __longlong_as_double((long long) (((unsigned long long) hi << 32) | lo));
}

__device__ __forceinline__ float lane_value(float v, int src)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}

// ix / w for an entry index ix < 1024 and a width 1 <= w <= 32 as
// (ix * m) >> 20, m = ceil(2^20 / w): the excess ix (m w - 2^20) / (2^20 w) is
// below 1023 * 31 / 2^20 / w < 1 / w
struct RowOf {
    uint32_t m;
    int w;
    __device__ __forceinline__ explicit RowOf(int w_) : m(((1u << 20) + w_ - 1) / w_), w(w_) {}
    __device__ __forceinline__ int row(int ix) const { return (int) (((uint32_t) ix * m) >> 20); }
    // 32 row + column
    __device__ __forceinline__ int at(int ix) const
    {
        const int r = row(ix);
        return 32 * r + (ix - r * w);
    }
};

template<typename VT>
__device__ __forceinline__ void tile_zero(VT* T)
{
    const int lane = lane_id();
#pragma unroll
    for(int t = 0; t < 16; ++t) T[64 * t + lane] = (VT) 0;
}

template<typename VT>
__device__ __forceinline__ void tile_copy(VT* dst, const VT* src)
{
    const int lane = lane_id();
#pragma unroll
    for(int t = 0; t < 16; ++t) dst[64 * t + lane] = src[64 * t + lane];
}

// d_load_block (kernels :22-81) for an input block of h x w, m its {format,
// nnz, col_ptr, val_ptr}: zero, then fill
template<typename VT>
__device__ void tile_load(VT* T, int4 m, int h, int w, const int32_t* ixs, const VT* vals)
{
    const int lane = lane_id();
    const RowOf width(w);
    tile_zero(T);
    wave_sync();
    if(m.x == FMT_DENSE) {
#pragma unroll
        for(int t = 0; t < 16; ++t) {
            const int idx = 64 * t + lane, r = idx >> 5, c = idx & 31;
            if(r < h && c < w) T[idx] = vals[(int64_t) m.w + r * w + c];
        }
    } else {
        for(int e = lane; e < m.y; e += 64) {
            T[width.at(ixs[(int64_t) m.z + e])] = vals[(int64_t) m.w + e];
        }
    }
    wave_sync();
}

// metadata of a factored dependency block, one per lane
struct Dep {
    int fmt, nnz, cp, vp, rb, rk;
};

__device__ __forceinline__ Dep load_dep(const BlockMeta* bout, const int32_t* bs, int blk)
{
    const BlockMeta m = bout[blk];
    Dep d;
    d.fmt = m.format;
    d.nnz = m.nnz;
    d.cp = m.col_ptr;
    d.vp = m.val_ptr;
    d.rb = bs[m.block_row];
    d.rk = bs[m.block_row + 1] - d.rb;
    return d;
}

// src is uniform across the wave: the result lives in scalar registers
__device__ __forceinline__ Dep bcast(const Dep& d, int src)
{
    Dep o;
    o.fmt = __builtin_amdgcn_readlane(d.fmt, src);
    o.nnz = __builtin_amdgcn_readlane(d.nnz, src);
    o.cp = __builtin_amdgcn_readlane(d.cp, src);
    o.vp = __builtin_amdgcn_readlane(d.vp, src);
    o.rb = __builtin_amdgcn_readlane(d.rb, src);
    o.rk = __builtin_amdgcn_readlane(d.rk, src);
    return o;
}

// registers holding one dependency block: its (up to 64) sparse entries and
// the tridiagonal D of its rows
template<typename VT>
struct Pre {
    int ix;
    VT v;
    VT sup, dia, sub;
};

template<typename VT>
__device__ __forceinline__ bool small_sparse(const Dep& d)
{
    return d.fmt == FMT_SPARSE && d.nnz <= 64;
}

template<typename VT>
__device__ __forceinline__ Pre<VT> prefetch(const Dep& d, const int32_t* ixs, const VT* vals,
    const double* tri, bool want_d)
{
    const int lane = lane_id();
    Pre<VT> p;
    p.ix = 0;
    p.v = 0;
    p.sup = p.dia = p.sub = 0;
    if(small_sparse<VT>(d) && lane < d.nnz) {
        p.ix = ixs[(int64_t) d.cp + lane];
        p.v = vals[(int64_t) d.vp + lane];
    }
    const int l = lane & 31;
    if(want_d && l < d.rk) {
        const double* t = tri + 3 * (int64_t) (d.rb + l);
        p.sup = (VT) t[0];
        p.dia = (VT) t[1];
        p.sub = (VT) t[2];
    }
    return p;
}

// Writes a dependency block (width w) into tile X and, when mask is set,
// the nonzero rows of each column into mask[c] (LDS, integer atomics).
template<typename VT>
__device__ void stage(VT* X, uint32_t* mask, const Dep& d, const Pre<VT>& p, const RowOf& wd,
    const int32_t* ixs, const VT* vals)
{
    const int lane = lane_id(), w = wd.w;
    if(small_sparse<VT>(d)) {
        if(lane < d.nnz) {
            const int k = wd.at(p.ix);
            X[k] = p.v;
            if(mask && p.v != (VT) 0) atomicOr(&mask[k & 31], 1u << (k >> 5));
        }
    } else if(d.fmt == FMT_DENSE) {
#pragma unroll
        for(int t = 0; t < 16; ++t) {
            const int idx = 64 * t + lane, r = idx >> 5, c = idx & 31;
            if(r < d.rk && c < w) {
                const VT v = vals[(int64_t) d.vp + r * w + c];
                X[idx] = v;
                if(mask && v != (VT) 0) atomicOr(&mask[c], 1u << r);
            }
        }
    } else {
        for(int e = lane; e < d.nnz; e += 64) {
            const int ix = ixs[(int64_t) d.cp + e];
            const VT v = vals[(int64_t) d.vp + e];
            const int k = wd.at(ix);
            X[k] = v;
            if(mask && v != (VT) 0) atomicOr(&mask[k & 31], 1u << (k >> 5));
        }
    }
}

template<typename VT>
__device__ void unstage(VT* X, uint32_t* mask, const Dep& d, const Pre<VT>& p, const RowOf& wd)
{
    const int lane = lane_id();
    if(small_sparse<VT>(d)) {
        if(lane < d.nnz) X[wd.at(p.ix)] = (VT) 0;
    } else {
        tile_zero(X);
    }
    if(mask && lane < 32) mask[lane] = 0;
}

template<typename VT>
__device__ __forceinline__ void stage_d(VT* cs, VT* cd, VT* cb, const Pre<VT>& p)
{
    const int lane = lane_id();
    if(lane < 32) {
        cs[lane] = p.sup;
        cd[lane] = p.dia;
        cb[lane] = p.sub;
    }
}

// T[c][j] -= sum_l R[l][j] * Lt[c][l] over the nonzero rows l of R's column
// j, ascending, with Lt[c][l] = (A' D)[c][l] formed from A[l-1..l+1][c] as
// d_multiply_block_by_block_diagonal does (kernels :372-456)
template<typename VT>
__device__ void product(VT* T, const VT* A, const VT* R, const uint32_t* mask, const VT* cs,
    const VT* cd, const VT* cb, int lh, int rh)
{
    const int lane = lane_id();
    const int j = lane & 31;
    const int c0 = lane >> 5;
    uint32_t mk = (j < rh) ? mask[j] : 0u;
    if(mk) {
        VT acc[16];
#pragma unroll
        for(int t = 0; t < 16; ++t) acc[t] = 0;
        while(mk) {
            const int l = __ffs(mk) - 1;
            mk &= mk - 1;
            const VT r = R[32 * l + j];
            const VT sup = cs[l], dia = cd[l], sub = cb[l];
#pragma unroll
            for(int t = 0; t < 16; ++t) {
                const int c = c0 + 2 * t;
                const VT left = (l == 0) ? (VT) 0 : A[32 * (l - 1) + c];
                const VT mid = A[32 * l + c];
                const VT right = (l == 31) ? (VT) 0 : A[32 * (l + 1) + c];
                const VT lt = fma(sub, right, fma(dia, mid, sup * left));
                acc[t] = fma(r, lt, acc[t]);
            }
        }
#pragma unroll
        for(int t = 0; t < 16; ++t) {
            const int c = c0 + 2 * t;
            if(c < lh) T[32 * c + j] -= acc[t];
        }
    }
}

// The Givens-form solve of d_left_solve_with_D_Ut (kernels :1533-1566) for
// row l of a block of hgt rows, D pointing at row l's tridiagonal triple:
// x1 for row l, x2 for row l + 1 when a 2x2 pivot starts at l (p2). The
// arithmetic runs in AT: the factor's type as the reference computes it,
// or FP64 for an FP32 factor whose 2x2 pivots are inverted in FP64. A 1x1
// pivot (d12 = 0) gives x1 = rl / d11 exactly either way.
template<typename VT, typename AT>
__device__ __forceinline__ void givens_d_solve(const double* D, int l, int hgt, VT rl_, VT right_,
    bool p2, VT& x1_, VT& x2_)
{
    const AT rl = (AT) rl_, right = (AT) right_;
    const AT d11 = (AT) D[1];
    const AT d12 = (AT) D[2];
    AT d22 = (l + 1 < hgt) ? (AT) D[4] : (AT) 0;
    if(l == 31) d22 = d11;
    const AT r = sqrt(fma(d11, d11, d12 * d12));
    const AT c = d11 / r, sn = d12 / r;
    AT x1 = fma(c, rl, sn * right);
    AT x2 = fma(-sn, rl, c * right);
    const AT t11 = fma(c, d11, sn * d12);
    const AT t12 = fma(c, d12, sn * d22);
    const AT t22 = fma(-sn, d12, c * d22);
    x2 = p2 ? (x2 / t22) : (AT) 0;
    x1 = fma(-t12, x2, x1) / t11;
    x1_ = (VT) x1;
    x2_ = (VT) x2;
}

template<typename VT>
__device__ __forceinline__ void givens_d_solve(bool f64, const double* D, int l, int hgt, VT rl,
    VT right, bool p2, VT& x1, VT& x2)
{
    if(f64) givens_d_solve<VT, double>(D, l, hgt, rl, right, p2, x1, x2);
    else givens_d_solve<VT, VT>(D, l, hgt, rl, right, p2, x1, x2);
}

// What a pivot step came upon: a D that is not finite; a multiplier that is
// not, after which rows and columns beyond the pivot row's nonzero ones have
// changed (0 inf and 0 NaN are NaN).
constexpr uint32_t STEP_BAD_D = 1, STEP_BAD_ROW = 2;

// d_ldlt_1x1_step (kernels :538-585)
template<typename VT>
__device__ uint32_t step_1x1(VT* T, double* tri, int p, int len)
{
    const int lane = lane_id();
    const int j = lane & 31, half = lane >> 5;
    VT d = T[32 * p + p];
    bool mod = false;
    if(fabs((double) d) < 1e-8) { d = (VT) 1e-6; mod = true; }
    const VT a = (j < p) ? (VT) 0 : T[32 * p + j];
    const VT u = a / d;
    const VT ru = u * d;
    wave_sync();
    if(half == 0) T[32 * p + j] = u;
    // trailing rows i > p, two per pass: only rows with a nonzero multiplier
    // ru_i change, and only if the pivot row has a nonzero u_j right of the
    // diagonal; the other updates would add exact zeros
    const uint64_t ucols = wave_ballot(half == 0 && j > p && j < len && u != (VT) 0);
    uint64_t rows = ucols ? wave_ballot(half == 0 && j > p && j < len && ru != (VT) 0) : 0ull;
    while(rows) {
        const int ia = __ffsll((long long) rows) - 1;
        rows &= rows - 1;
        const int ib = rows ? __ffsll((long long) rows) - 1 : -1;
        if(rows) rows &= rows - 1;
        const VT ra = wave_bcast(ru, ia);
        const VT rb = wave_bcast(ru, ib < 0 ? ia : ib);
        const int i = half ? ib : ia;
        const VT rui = half ? rb : ra;
        if(i >= 0 && j < len) T[32 * i + j] = fma(-rui, u, T[32 * i + j]);
    }
    wave_sync();
    if(mod && lane == 0) T[32 * p + p] = 1;
    if(lane < 3) tri[3 * p + lane] = (lane == 1) ? (double) d : 0.0;
    wave_sync();
    return (finite_value(d) ? 0u : STEP_BAD_D) |
        (wave_ballot(!finite_value(u) || !finite_value(ru)) ? STEP_BAD_ROW : 0u);
}

// d_ldlt_2x2_step (kernels :589-675): Givens rotation of the 2x2 pivot.
// The arithmetic runs in AT (see givens_d_solve); the multipliers are
// stored in the factor's type and the trailing update subtracts their
// products with the FP64-exact row factors r1, r2. A replaced near-singular
// pivot is (VT) 1e-6 on the diagonal in both forms.
template<typename VT, typename AT>
__device__ uint32_t step_2x2(VT* T, double* tri, int p, int len)
{
    const int lane = lane_id();
    const int j = lane & 31, half = lane >> 5;
    bool mod = false;
    AT d11 = (AT) T[32 * p + p];
    const AT d12 = (AT) T[32 * p + p + 1];
    AT d22 = (AT) T[32 * (p + 1) + p + 1];
    const AT det = fma(d11, d22, -(d12 * d12));
    if(fabs((double) det) < 1e-8) { d11 = (AT) (VT) 1e-6; d22 = (AT) (VT) 1e-6; mod = true; }
    const AT r = sqrt(fma(d11, d11, d12 * d12));
    const AT c = d11 / r, s = d12 / r;
    const AT t11 = fma(c, d11, s * d12);
    const AT t12 = fma(c, d12, s * d22);
    const AT t22 = fma(-s, d12, c * d22);
    const AT a1 = (j < p) ? (AT) 0 : (AT) T[32 * p + j];
    const AT a2 = (j < p) ? (AT) 0 : ((j == p) ? d12 : (AT) T[32 * (p + 1) + j]);
    AT x1 = fma(c, a1, s * a2);
    AT x2 = fma(-s, a1, c * a2);
    x2 = x2 / t22;
    x1 = fma(-t12, x2, x1) / t11;
    const VT u1 = (VT) x1, u2 = (VT) x2;
    const AT r1 = fma(x1, d11, x2 * d12);
    const AT r2 = fma(x1, d12, x2 * d22);
    wave_sync();
    if(half == 0) {
        T[32 * p + j] = (j < p) ? (VT) 0 : u1;
        T[32 * (p + 1) + j] = (j < p) ? (VT) 0 : u2;
    }
    // trailing rows i > p + 1 as in step_1x1: rows with a nonzero (r1_i,
    // r2_i), when the pivot rows have a nonzero (u1_j, u2_j) beyond them
    const uint64_t ucols = wave_ballot(half == 0 && j > p + 1 && j < len &&
        (u1 != (VT) 0 || u2 != (VT) 0));
    uint64_t rows = ucols ? wave_ballot(half == 0 && j > p + 1 && j < len &&
        (r1 != (AT) 0 || r2 != (AT) 0)) : 0ull;
    while(rows) {
        const int ia = __ffsll((long long) rows) - 1;
        rows &= rows - 1;
        const int ib = rows ? __ffsll((long long) rows) - 1 : -1;
        if(rows) rows &= rows - 1;
        const AT r1a = wave_bcast(r1, ia), r2a = wave_bcast(r2, ia);
        const AT r1b = wave_bcast(r1, ib < 0 ? ia : ib), r2b = wave_bcast(r2, ib < 0 ? ia : ib);
        const int i = half ? ib : ia;
        const AT r1i = half ? r1b : r1a, r2i = half ? r2b : r2a;
        if(i >= 0 && j < len)
            T[32 * i + j] = (VT) ((AT) T[32 * i + j] - fma(r1i, (AT) u1, r2i * (AT) u2));
    }
    wave_sync();
    if(mod && lane == 0) {
        T[32 * p + p] = 1;
        T[32 * p + p + 1] = 0;
        T[32 * (p + 1) + p + 1] = 1;
    }
    if(lane < 3) {
        tri[3 * p + lane] = (lane == 0) ? 0.0 : ((lane == 1) ? (double) d11 : (double) d12);
        tri[3 * (p + 1) + lane] = (lane == 0) ? (double) d12 : ((lane == 1) ? (double) d22 : 0.0);
    }
    wave_sync();
    // two products of finite factors may also overflow and meet as NaN, first
    // of all on the diagonal
    const VT dj = T[33 * j];
    const bool bad = !finite_value(u1) || !finite_value(u2) || !finite_value(r1) ||
        !finite_value(r2) || dj != dj;
    return (finite_value(fabs(d11) + fabs(d12) + fabs(d22)) ? 0u : STEP_BAD_D) |
        (wave_ballot(bad) ? STEP_BAD_ROW : 0u);
}

// entries of a block taken by the one-lane forms, and updates beside the
// diagonal one such block may make in a pivot tile
constexpr int LIGHT_E = 8;
constexpr int LIGHT_OFF = 4;

template<typename VT>
struct alignas(16) OffLds {
    VT T[1024];
    VT A[1024];
    VT R[1024];
    VT cs[32], cd[32], cb[32];
    uint32_t mask[32];
    uint32_t umask[32];
};

// ---------------------------------------------------------------------------

// ---------------------------------------------------------------------------
// Numeric pivoting inside a pivot tile T (stride 32, the matrix in its upper
// triangle), one wave. Lane l < 32 stands for row / column l, as a warp lane
// of the reference does.

// largest value over the wave and the lowest lane holding it among the
// lanes with `in` set (the reference's shuffle reduction keeps the lower
// lane on ties); NaN is never the largest
template<typename VT>
__device__ __forceinline__ int wave_argmax_first(VT v, bool in, VT& best)
{
    best = wave_max(in ? v : (VT) 0);
    const uint64_t at = wave_ballot(in && v == best);
    return at ? __ffsll((long long) at) - 1 : -1;
}

template<typename VT>
__device__ __forceinline__ VT sym_abs(const VT* T, int a, int b)
{
    return (a < b) ? fabs(T[32 * a + b]) : fabs(T[32 * b + a]);
}

// d_select_pivot_bunch_kaufman (kernels :743-834); alpha = (1 + sqrtf(17))
// / 8 evaluated in float as the reference writes it
template<typename VT>
__device__ void select_bk(const VT* T, int len, int p, int& order, int& p0, int& p1)
{
    const int l = lane_id();
    const VT alpha = (VT) ((1.0f + sqrtf(17.0f)) / 8.0f);
    order = 1;
    p0 = p;
    p1 = p + 1;
    VT w1;
    const VT v = (l > p && l < len) ? fabs(T[32 * p + min(l, 31)]) : (VT) 0;
    const int r = wave_argmax_first(v, l > p && l < len, w1);
    if(!(w1 > (VT) 0)) return;
    const VT app = fabs(T[32 * p + p]);
    if(app >= alpha * w1) return;
    const bool in = l >= p && l < len && l != r;
    const VT wr = wave_max(in ? sym_abs(T, min(l, 31), r) : (VT) 0);
    if(app * wr >= alpha * w1 * w1) return;
    if(fabs(T[32 * r + r]) >= alpha * wr) { p0 = r; return; }
    order = 2;
    p1 = r;
}

// d_select_pivot_rook (kernels :838-948). The search ends: wi is the
// magnitude of an entry of row r, so the largest of row r is at least wi, and
// the loop goes on only while it grows.
template<typename VT>
__device__ void select_rook(const VT* T, int len, int p, int& order, int& p0, int& p1)
{
    const int l = lane_id();
    const VT alpha = (VT) ((1.0f + sqrtf(17.0f)) / 8.0f);
    order = 1;
    p0 = p;
    p1 = p + 1;
    VT wi;
    const VT v = (l > p && l < len) ? fabs(T[32 * p + min(l, 31)]) : (VT) 0;
    int r = wave_argmax_first(v, l > p && l < len, wi);
    if(!(wi > (VT) 0)) return;
    int i = p;
    if(fabs(T[32 * p + p]) >= alpha * wi) return;
    for(;;) {
        VT wr;
        const bool in = l >= p && l < len && l != r;
        int q = wave_argmax_first(in ? sym_abs(T, min(l, 31), r) : (VT) 0, in, wr);
        // no nonzero candidate: the reference's reduction leaves lane 0's
        // start index, max(0, p)
        if(!(wr > (VT) 0)) q = p;
        if(fabs(T[32 * r + r]) >= alpha * wr) { p0 = r; return; }
        if(wi == wr) { order = 2; p0 = i; p1 = r; return; }
        i = r;
        r = q;
        wi = wr;
    }
}

// d_dense_pivot_op (kernels :679-739): symmetric interchange of rows and
// columns a and b of the tile (earlier, factored rows included, their
// entries in the two columns move too) and of perm[a], perm[b]
template<typename VT>
__device__ void dense_pivot_op(VT* T, int32_t* perm, int len, int pa, int pb)
{
    const int l = lane_id();
    wave_sync();
    if(l < len) {
        int x, y;
        if(l < pa) { x = 32 * l + pa; y = 32 * l + pb; }
        else if(l == pa) { x = 32 * pa + pa; y = 32 * pb + pb; }
        else if(l < pb) { x = 32 * pa + l; y = 32 * l + pb; }
        else if(l == pb) { x = y = 32 * pa + pb; }
        else { x = 32 * pa + l; y = 32 * pb + l; }
        const VT tx = T[x], ty = T[y];
        T[x] = ty;
        T[y] = tx;
    }
    if(l == 0) {
        const int32_t t = perm[pa];
        perm[pa] = perm[pb];
        perm[pb] = t;
    }
    wave_sync();
}

// ---------------------------------------------------------------------------
// Which Schur pairs do anything. The product of a pair (k, i), (k, j) is
// sum_l R[l][j] (A' D)[c][l] over the rows l of block row k: a pair whose
// blocks share no row adds exact zeros. At level-0 fill nearly every pair is
// such a pair (blocks of 1-3 entries in 32 rows: 97 % at kkt-400k, about
// 70 % at n = 2,000), and walking one costs a chain of four dependent
// loads, so each stored block leaves a 32-bit mask of its rows and a pair's
// masks are compared first. A 2x2 pivot couples neighbouring rows (the mask
// is widened by one row each way), and a non-finite entry or D makes the
// products of unmatched rows NaN (the mask ALL_ROWS matches every block).
constexpr uint32_t ALL_ROWS = 0xffffffffu;

// the mask of a stored block with entries in the rows m (dense blocks:
// ALL_ROWS), any_bad: one of them is not finite; flag: its row's row_flag
__device__ __forceinline__ uint32_t store_row_mask(uint32_t m, bool any_bad, int32_t flag)
{
    if(any_bad || (flag & ROW_NONFINITE)) return ALL_ROWS;
    if(flag & ROW_2X2) m |= (m << 1) | (m >> 1);
    return m;
}

// Most Schur pairs share no row. Leaving those out by two 4-byte masks instead
// of the blocks' metadata and entries: refactor 10.3 -> 7.7 ms at n = 2,000,
// 11.9 -> 10.6 ms at n = 400,000.
__device__ __forceinline__ bool pair_matches(uint32_t mi, uint32_t mj)
{
    return (mi & mj) != 0u || mi == ALL_ROWS || mj == ALL_ROWS;
}

// LDS of a pivot block: the tile, and either the one-lane updates of a round
// of blocks or one staged block
template<typename VT, int NW>
struct alignas(16) PivLds {
    VT T[1024];
    union {
        struct {
            VT val[NW][64 * LIGHT_E];                          // in block order
            uint32_t cols[NW][32][64 * LIGHT_E / 32 + 1];      // per column: which are its own
        } d;
        struct {
            VT X[1024];
            VT cs[32], cd[32], cb[32];
            uint32_t mask[32];
        } h;
    } u;
    VT dia[32];
    uint64_t heavy[NW];
    Dep dep;
    int32_t runs[NW];
    uint32_t plain, tiny;  // rows scaled together last, of them with a replaced pivot
    int32_t rflag;
    int32_t perm[32];      // old place of each row (numeric pivoting)
};

// What a dependency block U_ki with at most LIGHT_E entries subtracts from the
// pivot tile, formed by one lane with product()'s operations in its order: per
// column c of the block the update of T[c][c], and for two entries in one row
// the update of T[c1][c2], c1 < c2 (the lower triangle is never read). False
// for a block outside the form: more entries, a 2x2 pivot or a non-finite D
// among its rows, or more than LIGHT_OFF updates beside the diagonal.
template<typename VT>
struct LightUpd {
    uint32_t cols;             // columns with entries
    VT acc[LIGHT_E];           // update of the diagonal for the columns head[e]
    int head[LIGHT_E];         // column of entry e when it is its first, else -1
    int noff;
    int oe[LIGHT_OFF];         // 32 c1 + c2
    VT ov[LIGHT_OFF];
};

template<typename VT, int E>
__device__ __forceinline__ bool light_update(const Dep& d, const RowOf& w, const int32_t* ixs,
    const VT* vals, const double* tri, LightUpd<VT>& o)
{
    o.cols = 0;
    o.noff = 0;
#pragma unroll
    for(int e = 0; e < LIGHT_E; ++e) { o.acc[e] = (VT) 0; o.head[e] = -1; }
#pragma unroll
    for(int k = 0; k < LIGHT_OFF; ++k) { o.oe[k] = 0; o.ov[k] = (VT) 0; }
    if(d.fmt != FMT_SPARSE || d.nnz > E) return false;
    if(d.nnz == 0) return true;
    constexpr int NONE = 1 << 20;
    int key[E];          // 32 row + column, ascending
    VT v[E];
    bool sorted = true;
#pragma unroll
    for(int e = 0; e < E; ++e) {
        const int at = min(e, d.nnz - 1);
        const int ix = ixs[(int64_t) d.cp + at];
        v[e] = vals[(int64_t) d.vp + at];
        key[e] = (e < d.nnz && v[e] != (VT) 0) ? w.at(ix) : NONE;
    }
#pragma unroll
    for(int e = 1; e < E; ++e) sorted = sorted && key[e - 1] <= key[e];
    if(!sorted) {
        // odd-even transposition (entries over capacity are stored by size)
#pragma unroll
        for(int p = 0; p < E; ++p)
#pragma unroll
            for(int e = p & 1; e + 1 < E; e += 2)
                if(key[e + 1] < key[e]) {
                    const int tk = key[e]; key[e] = key[e + 1]; key[e + 1] = tk;
                    const VT tv = v[e]; v[e] = v[e + 1]; v[e + 1] = tv;
                }
    }
    VT lt[E];
    bool ok = true;
#pragma unroll
    for(int e = 0; e < E; ++e) {
        const double* t = tri + 3 * (int64_t) (d.rb + ((key[e] != NONE) ? key[e] >> 5 : 0));
        const double sup = t[0], dia = t[1], sub = t[2];
        ok = ok && (key[e] == NONE ||
            (sup == 0.0 && sub == 0.0 && fabs(dia) < (double) INFINITY && finite_value(v[e])));
        lt[e] = (VT) dia * v[e];
    }
    if(!ok) return false;
#pragma unroll
    for(int e = 0; e < E; ++e) {
        if(key[e] == NONE) continue;
        const int c = key[e] & 31;
        bool first = true;
#pragma unroll
        for(int f = 0; f < e; ++f) first = first && (key[f] & 31) != c;
        if(first) {
            VT acc = fma(v[e], lt[e], (VT) 0);
#pragma unroll
            for(int f = e + 1; f < E; ++f)
                if(key[f] != NONE && (key[f] & 31) == c) acc = fma(v[f], lt[f], acc);
            o.acc[e] = acc;
            o.head[e] = c;
            o.cols |= 1u << c;
        }
#pragma unroll
        for(int f = e + 1; f < E; ++f)
            if(key[f] != NONE && (key[f] >> 5) == (key[e] >> 5)) {
                const int el = 32 * c + (key[f] & 31);
                const VT acc = fma(v[f], lt[e], (VT) 0);
#pragma unroll
                for(int k = 0; k < LIGHT_OFF; ++k) {
                    ok = ok && !(k < o.noff && o.oe[k] == el);
                    if(k == o.noff) { o.oe[k] = el; o.ov[k] = acc; }
                }
                ++o.noff;
            }
    }
    return ok && o.noff <= LIGHT_OFF;
}

// The same for a block with a 2x2 pivot among its rows and at most COL_E entries,
// all in one column c: it updates T[c][c] alone, the rows above and below coupled
// by D. Among static 2x2 pivots two blocks in five are such; staged as tiles
// instead, a refactor at n = 5,000 in blocks of up to 8 rows took 11.6 ms
// instead of 7.0 (f64).
constexpr int COL_E = 4;

template<typename VT>
__device__ __forceinline__ bool column_update(const Dep& d, const RowOf& w, const int32_t* ixs,
    const VT* vals, const double* tri, LightUpd<VT>& o)
{
    if(d.fmt != FMT_SPARSE || d.nnz > COL_E || d.nnz == 0) return false;
    constexpr int NONE = 1 << 20;
    int key[COL_E];          // 32 row + column, ascending
    VT v[COL_E];
#pragma unroll
    for(int e = 0; e < COL_E; ++e) {
        const int at = min(e, d.nnz - 1);
        const int ix = ixs[(int64_t) d.cp + at];
        v[e] = vals[(int64_t) d.vp + at];
        key[e] = (e < d.nnz && v[e] != (VT) 0) ? w.at(ix) : NONE;
    }
    auto order = [&](int x, int y) {
        if(key[y] < key[x]) {
            const int tk = key[x]; key[x] = key[y]; key[y] = tk;
            const VT tv = v[x]; v[x] = v[y]; v[y] = tv;
        }
    };
    static_assert(COL_E == 4, "sorting network on four");
    order(0, 1); order(2, 3); order(0, 2); order(1, 3); order(1, 2);
    bool ok = true;
    VT acc = (VT) 0;
#pragma unroll
    for(int e = 0; e < COL_E; ++e) {
        if(key[e] == NONE) continue;
        const double* t = tri + 3 * (int64_t) (d.rb + (key[e] >> 5));
        const VT sup = (VT) t[0], dia = (VT) t[1], sub = (VT) t[2];
        ok = ok && (key[e] & 31) == (key[0] & 31) && finite_value(sup) && finite_value(dia) &&
            finite_value(sub) && finite_value(v[e]);
        const VT left = (e > 0 && key[max(e - 1, 0)] == key[e] - 32) ? v[max(e - 1, 0)] : (VT) 0;
        const VT right = (e + 1 < COL_E && key[min(e + 1, COL_E - 1)] == key[e] + 32)
            ? v[min(e + 1, COL_E - 1)] : (VT) 0;
        acc = fma(v[e], fma(sub, right, fma(dia, v[e], sup * left)), acc);
    }
    if(!ok) return false;
    o.cols = (key[0] != NONE) ? 1u << (key[0] & 31) : 0u;
    o.noff = 0;
#pragma unroll
    for(int e = 0; e < LIGHT_E; ++e) o.head[e] = -1;
    if(o.cols) {
        o.head[0] = key[0] & 31;
        o.acc[0] = acc;
    }
    return true;
}

// T -= A' D A for the block staged in h.X by all NW waves: the arithmetic and
// order of product() with R = A
template<typename VT, int NW>
__device__ __forceinline__ void product_staged(PivLds<VT, NW>& s, int len)
{
    const int j = (int) threadIdx.x & 31;
    const int c0 = (int) threadIdx.x >> 5;
    constexpr int NR = 16 / NW, ST = 2 * NW;
    const VT* A = s.u.h.X;
    const uint32_t mk = (j < len) ? s.u.h.mask[j] : 0u;
    if(mk) {
        VT acc[NR];
#pragma unroll
        for(int t = 0; t < NR; ++t) acc[t] = 0;
        for(uint32_t bits = mk; bits; bits &= bits - 1) {
            const int l = __ffs(bits) - 1;
            const VT r = A[32 * l + j];
            const VT sup = s.u.h.cs[l], dia = s.u.h.cd[l], sub = s.u.h.cb[l];
#pragma unroll
            for(int t = 0; t < NR; ++t) {
                const int c = c0 + ST * t;
                const VT left = (l == 0) ? (VT) 0 : A[32 * (l - 1) + c];
                const VT mid = A[32 * l + c];
                const VT right = (l == 31) ? (VT) 0 : A[32 * (l + 1) + c];
                const VT lt = fma(sub, right, fma(dia, mid, sup * left));
                acc[t] = fma(r, lt, acc[t]);
            }
        }
#pragma unroll
        for(int t = 0; t < NR; ++t) {
            const int c = c0 + ST * t;
            if(c < len) s.T[32 * c + j] -= acc[t];
        }
    }
}

// one dependency block of any form, by all NW waves
template<typename VT, int NW>
__device__ __forceinline__ void heavy_update(const FactorArgs<VT>& a, PivLds<VT, NW>& s, const Dep& d, int len)
{
    constexpr int TPB = 64 * NW;
    const int t = (int) threadIdx.x;
    for(int e = t; e < 1024; e += TPB) s.u.h.X[e] = (VT) 0;
    if(t < 32) {
        s.u.h.mask[t] = 0;
        VT sup = 0, dia = 0, sub = 0;
        if(t < d.rk) {
            const double* td = a.tri + 3 * (int64_t) (d.rb + t);
            sup = (VT) td[0];
            dia = (VT) td[1];
            sub = (VT) td[2];
        }
        s.u.h.cs[t] = sup;
        s.u.h.cd[t] = dia;
        s.u.h.cb[t] = sub;
    }
    __syncthreads();
    auto put = [&](int r, int c, VT v) {
        s.u.h.X[32 * r + c] = v;
        if(v != (VT) 0) atomicOr(&s.u.h.mask[c], 1u << r);
    };
    if(d.fmt == FMT_DENSE) {
        for(int e = t; e < d.rk * len; e += TPB) {
            const int r = e / len;
            put(r, e - r * len, a.val_out[(int64_t) d.vp + e]);
        }
    } else {
        for(int e = t; e < d.nnz; e += TPB) {
            const int ix = a.ix_out[(int64_t) d.cp + e];
            const int r = ix / len;
            put(r, ix - r * len, a.val_out[(int64_t) d.vp + e]);
        }
    }
    __syncthreads();
    product_staged<VT, NW>(s, len);
    __syncthreads();
}

// the one-lane updates of the lanes with `mine` set, in block order
template<typename VT, int NW>
__device__ __forceinline__ void apply_light(PivLds<VT, NW>& s, const LightUpd<VT>& o, bool mine)
{
    const int t = (int) threadIdx.x, lane = lane_id(), wv = t / WAVE;
    const int n = mine ? __popc(o.cols) : 0;
    int off = n;
#pragma unroll
    for(int k = 1; k < WAVE; k <<= 1) {
        const int u = __shfl_up(off, k, WAVE);
        if(lane >= k) off += u;
    }
    const int total = __shfl(off, WAVE - 1, WAVE);
    off -= n;
    const int words = (total + 31) / 32;
    for(int k = lane; k < 32 * words; k += WAVE) s.u.d.cols[wv][k & 31][k >> 5] = 0u;
    if(lane == 0) s.runs[wv] = words;
    wave_sync();
    if(n) {
#pragma unroll
        for(int e = 0; e < LIGHT_E; ++e)
            if(o.head[e] >= 0) {
                const int c = o.head[e];
                const int at = off + __popc(o.cols & ((1u << c) - 1));
                s.u.d.val[wv][at] = o.acc[e];
                atomicOr(&s.u.d.cols[wv][c][at >> 5], 1u << (at & 31));
            }
    }
    __syncthreads();
    if(t < 32) {
        VT d = s.T[33 * t];
        for(int u = 0; u < NW; ++u)
            for(int wd = 0; wd < s.runs[u]; ++wd)
                for(uint32_t bits = s.u.d.cols[u][t][wd]; bits; bits &= bits - 1)
                    d -= s.u.d.val[u][32 * wd + __ffs(bits) - 1];
        s.T[33 * t] = d;
    }
    // updates beside the diagonal (few), one block after the other
    const bool off_any = mine && o.noff > 0;
    if(__syncthreads_or(off_any))
        for(int u = 0; u < NW; ++u) {
            if(u == wv)
                for(uint64_t b = wave_ballot(off_any); b; b &= b - 1) {
                    if(lane == __ffsll((long long) b) - 1) {
#pragma unroll
                        for(int k = 0; k < LIGHT_OFF; ++k)
                            if(k < o.noff) s.T[o.oe[k]] -= o.ov[k];
                    }
                    wave_sync();
                }
            __syncthreads();
        }
}

// piv_flag: an entry right of the diagonal, a 2x2 pivot, a non-finite D, rows
// out of their order
constexpr uint32_t PIV_ANY = 1, PIV_2X2 = 2, PIV_NONFINITE = 4, PIV_PERM = 8;

// k_factor_pivot_blocks (kernels :1146-1283) for the pivot block at level
// position q, NW waves.
// Bound by latency: the level's pivot blocks are far fewer than the chip has
// CUs, and each waits for its tile, the ids of the blocks above it, their
// metadata, their entries and D, five dependent round trips. All blocks above
// it take these trips together, one per lane, and the updates are then added
// per element in block order from LDS; blocks outside the one-lane form are
// staged one by one in their place in that order. Of the pivot steps only
// rows with an entry right of the diagonal (or a 2x2 pivot, or a NaN on the
// diagonal, which reaches all rows below) are steps; the others scale a row and
// change nothing else, so they are done together last.
// FP64 refactor, blocks above taken by rounds of one wave -> at once: 7.1 ->
// 5.2 ms at n = 2,000, 8.3 -> 6.4 ms at n = 400,000.
// TWO: there may be 2x2 pivots, static ones or numerically chosen. Without them
// their code stays out: a level's kernels follow each other through the
// instruction cache (n = 400,000: 4.16 ms, with it 4.21).
template<typename VT, int NW, bool TWO>
__device__ __forceinline__ void pivots_one(const FactorArgs<VT>& a, const LevelRange& lr, const int q,
    PivLds<VT, NW>& s)
{
    constexpr int TPB = 64 * NW;
    const int t = (int) threadIdx.x, lane = lane_id(), wv = t / WAVE;
    const int4 t0 = ((const int4*) a.off_task)[3 * ((int64_t) lr.lo + q)];
    const int4 t1 = ((const int4*) a.off_task)[3 * ((int64_t) lr.lo + q) + 1];
    const int4 t2 = ((const int4*) a.off_task)[3 * ((int64_t) lr.lo + q) + 2];
    // the pool before the level: its pivot blocks come first in it
    const int32_t pool = a.carry[4 * (lr.level & 1)];
    const int i = t0.w;
    const int fr = t0.y;
    const int len = t0.z;
    const int cb0 = t2.x;
    const int nd = t2.y;
    // the tile: dense input values (the factor's blocks on the diagonal are)
    int blk = (t < nd) ? a.csc_idx[cb0 + t] : -1;
    int piv = 1;
    if(t < 32 && t < len) piv = a.is_piv[fr + t];
    const RowOf width(len);
    if(t1.x == FMT_DENSE) {
        // all of a thread's loads in flight at once, at places within the block
        // (one by one under their own conditions: 5 us of a one-wave block's 25)
        VT v[1024 / TPB];
#pragma unroll
        for(int k = 0; k < 1024 / TPB; ++k) {
            const int e = t + TPB * k, r = min(e >> 5, len - 1), c = min(e & 31, len - 1);
            v[k] = a.val_in[(int64_t) t1.w + r * len + c];
        }
#pragma unroll
        for(int k = 0; k < 1024 / TPB; ++k) {
            const int e = t + TPB * k;
            s.T[e] = ((e >> 5) < len && (e & 31) < len) ? v[k] : (VT) 0;
        }
    } else {
        for(int e = t; e < 1024; e += TPB) s.T[e] = (VT) 0;
        __syncthreads();
        for(int e = t; e < t1.y; e += TPB)
            s.T[width.at(a.ix_in[(int64_t) t1.z + e])] = a.val_in[(int64_t) t1.w + e];
    }
    __syncthreads();
    // updates from the blocks (k, i) above the diagonal, in CSC order
    for(int c0 = 0; c0 < nd; c0 += TPB) {
        if(c0) blk = (c0 + t < nd) ? a.csc_idx[cb0 + c0 + t] : -1;
        Dep d{};
        LightUpd<VT> up;
        up.cols = 0;
        up.noff = 0;
        bool light = false;
        if(blk >= 0) {
            d = load_dep(a.bout, a.bs, blk);
        }
        // blocks of one or two entries (nearly all on large sparse patterns)
        // without the eight-entry form's work
        if(wave_ballot(blk >= 0 && !(d.fmt == FMT_SPARSE && d.nnz <= 2)) == 0ull)
            light = blk >= 0 && light_update<VT, 2>(d, width, a.ix_out, a.val_out, a.tri, up);
        else
            light = blk >= 0 && light_update<VT, LIGHT_E>(d, width, a.ix_out, a.val_out, a.tri, up);
        if(TWO && wave_ballot(blk >= 0 && !light && d.fmt == FMT_SPARSE && d.nnz <= COL_E))
            light = light || (blk >= 0 &&
                column_update<VT>(d, width, a.ix_out, a.val_out, a.tri, up));
        const uint64_t hm = wave_ballot(blk >= 0 && !light);
        if(lane == 0) s.heavy[wv] = hm;
        __syncthreads();
        for(int start = 0, w = 0;;) {
            // the next block outside the form
            int h = -1;
            for(; w < NW; ++w) {
                uint64_t m = s.heavy[w];
                if(start > 64 * w) m &= (start - 64 * w >= 64) ? 0ull : ~0ull << (start - 64 * w);
                if(m) { h = 64 * w + __ffsll((long long) m) - 1; break; }
            }
            apply_light<VT, NW>(s, up, light && t >= start && (h < 0 || t < h));
            __syncthreads();
            if(h < 0) break;
            if(t == h) s.dep = d;
            __syncthreads();
            const Dep hd = s.dep;
            heavy_update<VT, NW>(a, s, hd, len);
            start = h + 1;
        }
    }
    // d_factor_pivot_factorize (kernels :956-1083): static pivots, or a
    // numeric choice per step with symmetric interchanges (the pivot starts
    // and the block's rows in perm are rewritten as pivots are chosen)
    double* tri = a.tri + 3 * (int64_t) fr;
    VT* T0 = s.T;
    const uint32_t live = len == 32 ? ~0u : (1u << len) - 1;
    uint32_t M = 0;   // wave 0: columns right of the diagonal of row `lane`
    if(wv == 0) {
        int32_t rflag = 0;
        uint32_t plain = 0, tiny = 0;
        if(TWO && a.pivoting) {
            int32_t* fpiv = a.is_piv + fr;
            int32_t* bperm = s.perm;
            if(lane < 32) bperm[lane] = lane;
            wave_sync();
            int p = 0;
            while(p < len) {
                int order = 1, p0 = p, p1 = p + 1;
                if(p < len - 1) {
                    if(a.pivoting == 1) select_bk(T0, len, p, order, p0, p1);
                    else select_rook(T0, len, p, order, p0, p1);
                }
                if(order == 1) {
                    if(p0 != p) dense_pivot_op(T0, bperm, len, p, p0);
                    if(step_1x1(T0, tri, p, len) & STEP_BAD_D) rflag |= ROW_NONFINITE;
                    if(lane == 0) fpiv[p] = 1;
                } else {
                    if(p0 != p) dense_pivot_op(T0, bperm, len, p, p0);
                    dense_pivot_op(T0, bperm, len, p + 1, p1);
                    const uint32_t bad = a.piv64 ? step_2x2<VT, double>(T0, tri, p, len)
                                                 : step_2x2<VT, VT>(T0, tri, p, len);
                    rflag |= (bad & STEP_BAD_D) ? (ROW_2X2 | ROW_NONFINITE) : ROW_2X2;
                    if(lane == 0) {
                        fpiv[p] = 1;
                        fpiv[p + 1] = 0;
                    }
                }
                wave_sync();
                p += order;
            }
            if(lane < 32) M = (lane < 31) ? ~0u << (lane + 1) : 0u;
        } else {
            // columns right of the diagonal per row: a superset while steps fill
            // rows in (all of them after a multiplier that is not finite)
#pragma unroll
            for(int k = 0; k < 16; ++k) {
                const int r = 2 * k + (lane >> 5), c = lane & 31;
                const uint64_t b = wave_ballot(c > r && c < len && T0[64 * k + lane] != (VT) 0);
                if(lane == 2 * k) M = (uint32_t) b;
                if(lane == 2 * k + 1) M = (uint32_t) (b >> 32);
            }
            const uint32_t right = lane < len ? live & (~1u << lane) : 0u;
            const VT d0 = T0[33 * (lane & 31)];
            if(d0 != d0) M = right;
            const uint32_t starts = (uint32_t) wave_ballot(lane < 32 && lane < len && piv != 0);
            const uint32_t two = TWO ? (~starts & live) >> 1 : 0u;   // rows where a 2x2 pivot starts
            uint32_t done = 0;
            for(int p = 0; p < len;) {
                const uint32_t cand = ((uint32_t) wave_ballot(lane < len && M != 0u) | two) &
                    (~0u << p);
                if(!cand) break;
                p = __ffs(cand) - 1;
                uint32_t bad;
                if(TWO && ((two >> p) & 1u)) {
                    bad = a.piv64 ? step_2x2<VT, double>(T0, tri, p, len)
                                  : step_2x2<VT, VT>(T0, tri, p, len);
                    rflag |= ROW_2X2;
                    const uint32_t mm = (uint32_t) (__builtin_amdgcn_readlane((int) M, p) |
                        __builtin_amdgcn_readlane((int) M, p + 1));
                    if(lane > p + 1 && lane < 32 && ((mm >> lane) & 1u)) M |= mm & (~1u << lane);
                    if(lane == p || lane == p + 1) M |= mm & (~1u << lane);
                    done |= 3u << p;
                    p += 2;
                } else {
                    bad = step_1x1(T0, tri, p, len);
                    const uint32_t mm = (uint32_t) __builtin_amdgcn_readlane((int) M, p);
                    if(lane > p && lane < 32 && ((mm >> lane) & 1u)) M |= mm & (~1u << lane);
                    done |= 1u << p;
                    p += 1;
                }
                if(bad & STEP_BAD_D) rflag |= ROW_NONFINITE;
                if(bad & STEP_BAD_ROW) M = right;
                wave_sync();
            }
            plain = live & ~done;
            const bool own = lane < 32 && ((plain >> lane) & 1u);
            VT d = T0[33 * (lane & 31)];
            const bool rep = fabs((double) d) < 1e-8;
            if(rep) d = (VT) 1e-6;
            if(lane < 32) s.dia[lane] = d;
            tiny = plain & (uint32_t) wave_ballot(own && rep);
            if(own) {
                tri[3 * lane] = 0.0;
                tri[3 * lane + 1] = (double) d;
                tri[3 * lane + 2] = 0.0;
            }
            if(wave_ballot(own && !finite_value(d))) rflag |= ROW_NONFINITE;
        }
        if(lane == 0) {
            s.plain = plain;
            s.tiny = tiny;
            s.rflag = rflag;
        }
    }
    __syncthreads();
    // the remaining rows' steps: step_1x1 without its trailing update
    if(s.plain) {
        const uint32_t rows = s.plain, ones = s.tiny;
#pragma unroll 4
        for(int e = t; e < 1024; e += TPB) {
            const int r = e >> 5, c = e & 31;
            const VT u = ((c < r) ? (VT) 0 : T0[e]) / s.dia[r];
            if((rows >> r) & 1u) T0[e] = (c == r && ((ones >> r) & 1u)) ? (VT) 1 : u;
        }
        __syncthreads();
    }
    if(wv == 0) {
        // row sums of squares, and the nonzero columns right of the diagonal
        // for the U_ii' solves (every other entry of a row is zero)
        uint32_t um = 0;
        bool bounded = true;
        if(lane < len) {
            VT v = T0[33 * lane];
            VT ssq = fma(v, v, (VT) 0);
            bounded = fabs(v) > (VT) 0.5 && fabs(v) < (VT) 0x1p30;
            for(uint32_t bits = M & live; bits; bits &= bits - 1) {
                v = T0[32 * lane + __ffs(bits) - 1];
                ssq = fma(v, v, ssq);
                if(v != (VT) 0) um |= bits & (0u - bits);
                bounded = bounded && fabs(v) < (VT) 0x1p30;
            }
            a.rn[fr + lane] = ssq;
        }
        if(lane < 32) a.piv_umask[(int64_t) q * 32 + lane] = um;   // all 32 words defined
        // what the off-diagonal blocks of the row ask first
        uint32_t flags = wave_ballot(um != 0u) ? PIV_ANY : 0u;
        if(s.rflag & ROW_2X2) flags |= PIV_2X2;
        if(s.rflag & ROW_NONFINITE) flags |= PIV_NONFINITE;
        const bool unbounded = wave_ballot(!bounded) != 0ull;
        if(TWO && a.pivoting) {
            const int p = (lane < len) ? s.perm[lane] : lane;
            if(wave_ballot(lane < len && p != lane)) flags |= PIV_PERM;
            if(lane < len) {
                a.perm[fr + lane] = fr + p;
                a.piv_iperm[(int64_t) q * 32 + p] = (uint8_t) lane;
            }
        }
        if(lane == 0) {
            a.piv_flag[q] = flags;
            a.row_flag[i] = s.rflag | ((flags & PIV_ANY) ? ROW_COUPLED : 0) |
                (unbounded ? ROW_UNBOUNDED : 0);
            a.piv_loc[i] = q;
        }
    }
    // the tile for the level's off-diagonal blocks, and its final storage:
    // dense blocks keep their size, so the offset follows from the pool alone
    // (k_drop)
    VT* out = a.if_val + (int64_t) q * 1024;
    VT* fin = a.val_out + ((int64_t) t1.w - pool);
#pragma unroll 4
    for(int e = t; e < len * len; e += TPB) {
        const VT v = T0[width.at(e)];
        out[e] = v;
        fin[e] = v;
    }
}

// the entry list of position q: its first LIST_C entries in the compact
// store, the others in the large one
template<typename VT>
struct EntryList {
    VT* cv;
    uint16_t* ci;
    VT* v;
    uint16_t* ix;
    __device__ __forceinline__ VT val(int e) const { return e < LIST_C ? cv[e] : v[e]; }
    __device__ __forceinline__ int idx(int e) const { return e < LIST_C ? ci[e] : ix[e]; }
    __device__ __forceinline__ void set(int e, int i, VT x) const
    {
        (e < LIST_C ? ci : ix)[e] = (uint16_t) i;
        (e < LIST_C ? cv : v)[e] = x;
    }
};

template<typename VT>
__device__ __forceinline__ EntryList<VT> entry_list(const FactorArgs<VT>& a, int q)
{
    return {a.c_val + (int64_t) q * LIST_C, a.c_idx + (int64_t) q * LIST_C,
        a.if_val + (int64_t) q * 1024, a.if_idx + (int64_t) q * 1024};
}

// An off-diagonal tile X (one wave, stride 32, zero outside hgt x wid) as
// position q leaves it: divided by D where that is left to do (by_d; d_row
// holds row l's 1x1 pivot in lane l; a finite D leaves a row of zeros as it
// is), then the row sums of squares and the dense tile or the entries above
// NZ_EPS. The tile is mostly zeros: the loop takes the pairs of rows that have
// an entry.
template<typename VT>
__device__ __forceinline__ void offdiag_output(const FactorArgs<VT>& a, int q, VT* X, bool by_d,
    bool nonfinite, double d_row, int hgt, int wid, int format)
{
    const int lane = lane_id();
    const EntryList<VT> o = entry_list(a, q);
    uint32_t act = 0;
#pragma unroll
    for(int t = 0; t < 16; ++t)
        if(wave_ballot(X[64 * t + lane] != (VT) 0)) act |= 1u << t;
    if(by_d && nonfinite) act = (uint32_t) ((1ull << ((hgt + 1) / 2)) - 1ull);
    // nonzero entries per row; a row's sum skips exact zeros
    uint32_t nz = 0;
    int base = 0;
#pragma unroll 1
    for(; act; act &= act - 1) {
        const int t = __ffs(act) - 1;
        VT x = X[64 * t + lane];
        if(by_d) {
            const uint64_t b = wave_ballot(x != (VT) 0);
            const double lo = lane_value(d_row, 2 * t), hi = lane_value(d_row, 2 * t + 1);
            const bool some = (lane < 32 ? (uint32_t) b : (uint32_t) (b >> 32)) != 0u;
            const bool in = (lane & 31) < wid && 2 * t + (lane >> 5) < hgt;
            const VT y = (VT) ((double) x / (lane < 32 ? lo : hi));
            if(in && (some || nonfinite)) {
                x = y;
                X[64 * t + lane] = y;
            }
        }
        const uint64_t b = wave_ballot(x != (VT) 0);
        if(lane == 2 * t) nz = (uint32_t) b;
        if(lane == 2 * t + 1) nz = (uint32_t) (b >> 32);
        if(format != FMT_DENSE) {
            const bool live = fabs((double) x) > NZ_EPS;
            const uint64_t msk = wave_ballot(live);
            if(live) o.set(base + lanes_below(msk), 64 * t + lane, x);
            base += __popcll(msk);
        }
    }
    wave_sync();
    VT ssq = (VT) 0;
#pragma unroll 1
    for(uint32_t bits = nz; bits; bits &= bits - 1) {
        const VT v = X[32 * lane + __ffs(bits) - 1];
        ssq = fma(v, v, ssq);
    }
    const uint64_t rows = wave_ballot(!(ssq == (VT) 0));
    if((rows >> lane) & 1ull) {
        const int j = lanes_below(rows);
        if(j == 0) a.rn_first[q] = ssq;
        else a.rn_part[(int64_t) q * 32 + j] = ssq;
    }
    if(format == FMT_DENSE) {
        VT* oval = a.if_val + (int64_t) q * 1024;
#pragma unroll 4
        for(int t = 0; t < 16; ++t) {
            const int r = 2 * t + (lane >> 5), c = lane & 31;
            if(r < hgt && c < wid) oval[r * wid + c] = X[64 * t + lane];
        }
        base = hgt * wid;
    }
    if(lane == 0) {
        a.part_mask[q] = (uint32_t) rows;
        a.if_cnt[q] = base;
    }
}

// k_update_scale_offdiagonal_blocks (kernels :1628-1803) with
// d_left_solve_with_D_Ut (:1489-1570): general form, all dependency blocks
// staged as tiles; takes the positions k_offdiag leaves to it.
template<typename VT>
__device__ void offdiag_general_one(const FactorArgs<VT>& a, const LevelRange& lr, int q,
    OffLds<VT>& s);

template<typename VT>
__device__ __forceinline__ void offdiag_general_body(const FactorArgs<VT>& a, const LevelRange& lr,
    int bid_, int nblk_)
{
    __shared__ OffLds<VT> s;
    const int ndef = a.defer_cnt[lr.level];
    for(int t = bid_; t < ndef; t += nblk_) {
        offdiag_general_one(a, lr, a.defer_list[t], s);
        __syncthreads();
    }
}

template<typename VT>
__device__ void offdiag_general_one(const FactorArgs<VT>& a, const LevelRange& lr, int q,
    OffLds<VT>& s)
{
    const int lane = lane_id();
    const int b = a.lvlb_idx[lr.lo + q];
    const BlockMeta m = a.bin[b];
    const int i = m.block_row, jb = m.block_col;
    const int fr = a.bs[i];
    const int hgt = a.bs[i + 1] - fr;
    const int wid = a.bs[jb + 1] - a.bs[jb];
    const int64_t p0 = a.upd_off[b];
    const int np = (int) (a.upd_off[b + 1] - p0);
    const int pq = a.piv_loc[i];
    const bool all1x1 = (wave_ballot(lane < hgt && !a.is_piv[fr + (lane & 31)]) == 0);
    const RowOf height(hgt), width(wid);
    tile_zero(s.A);
    if(lane < 32) { s.mask[lane] = 0; s.umask[lane] = 0; }
    if(np > 0) tile_zero(s.R);
    tile_load(s.T, make_int4(m.format, m.nnz, m.col_ptr, m.val_ptr), hgt, wid, a.ix_in, a.val_in);
    for(int c0 = 0; c0 < np; c0 += 64) {
        Dep mi{}, mj{};
        bool hit = false;
        if(c0 + lane < np) {
            const int ki = a.upd_ki[p0 + c0 + lane], kj = a.upd_kj[p0 + c0 + lane];
            hit = pair_matches(a.row_mask[ki], a.row_mask[kj]);
            if(hit) {
                mi = load_dep(a.bout, a.bs, ki);
                mj = load_dep(a.bout, a.bs, kj);
            }
        }
        uint64_t hits = wave_ballot(hit);
        if(!hits) continue;
        int d = __ffsll((long long) hits) - 1;
        Dep ci = bcast(mi, d), cj = bcast(mj, d);
        Pre<VT> pi = prefetch(ci, a.ix_out, a.val_out, a.tri, true);
        Pre<VT> pj = prefetch(cj, a.ix_out, a.val_out, a.tri, false);
        while(hits) {
            hits &= hits - 1;
            Dep ni = ci, nj = cj;
            Pre<VT> qi = pi, qj = pj;
            if(hits) {
                d = __ffsll((long long) hits) - 1;
                ni = bcast(mi, d);
                nj = bcast(mj, d);
                qi = prefetch(ni, a.ix_out, a.val_out, a.tri, true);
                qj = prefetch(nj, a.ix_out, a.val_out, a.tri, false);
            }
            stage(s.A, (uint32_t*) nullptr, ci, pi, height, a.ix_out, a.val_out);
            stage(s.R, s.mask, cj, pj, width, a.ix_out, a.val_out);
            stage_d(s.cs, s.cd, s.cb, pi);
            wave_sync();
            product(s.T, s.A, s.R, s.mask, s.cs, s.cd, s.cb, hgt, wid);
            wave_sync();
            unstage(s.A, (uint32_t*) nullptr, ci, pi, height);
            unstage(s.R, s.mask, cj, pj, width);
            wave_sync();
            ci = ni; cj = nj; pi = qi; pj = qj;
        }
    }

    // rows in the block row's pivoting order (kernels :1733-1751)
    if(a.pivoting) {
        tile_copy(s.A, s.T);
        wave_sync();
        for(int e = lane; e < hgt * 32; e += 64) {
            const int r = e >> 5, c = e & 31;
            s.T[e] = s.A[32 * (a.perm[fr + r] - fr) + c];
        }
        wave_sync();
        tile_zero(s.A);
        wave_sync();
    }
    // pivot tile U_ii (row-major) into A; umask[r] = nonzero columns > r
    const VT* piv = a.if_val + (int64_t) pq * 1024;
    for(int e = lane; e < hgt * hgt; e += 64) {
        const int r = e / hgt, c = e - r * hgt;
        const VT v = piv[e];
        s.A[32 * r + c] = v;
        if(c > r && v != (VT) 0) atomicOr(&s.umask[r], 1u << c);
    }
    wave_sync();

    // column j per lane (lanes >= 32 idle): forward substitution with U_ii'
    // (terms with a zero multiplier are exact no-ops and are skipped)
    const int j = lane;
    const VT* U = s.A;
    VT rhs[32];
#pragma unroll
    for(int l = 0; l < 32; ++l) rhs[l] = (l < hgt && j < wid) ? s.T[32 * l + j] : (VT) 0;
#pragma unroll
    for(int ii = 0; ii < 32; ++ii) {
        if(ii < hgt) {
            const uint32_t um = s.umask[ii];
            if(rhs[ii] != (VT) 0 && um) {
                const VT pv = rhs[ii] / U[32 * ii + ii];
#pragma unroll
                for(int l = ii + 1; l < 32; ++l)
                    if((um >> l) & 1u) rhs[l] = fma(-U[32 * ii + l], pv, rhs[l]);
            }
        }
    }
    const double* D = a.tri + 3 * (int64_t) fr;
    const int32_t* ip = a.is_piv + fr;
    wave_sync();
    if(all1x1) {
        // 1x1 pivots: the Givens-form solve reduces exactly to rhs / d
#pragma unroll
        for(int l = 0; l < 32; ++l)
            if(l < hgt && j < wid) s.T[32 * l + j] = (VT) ((double) rhs[l] / D[3 * l + 1]);
    } else {
#pragma unroll
        for(int l = 0; l < 32; ++l) {
            if(l < hgt) {
                const bool p1 = ip[l] != 0;
                const bool p2 = (l + 1 < hgt) && !ip[l + 1];
                const VT rl = rhs[l];
                const VT right = (l < 31) ? rhs[l + 1] : rhs[31];
                VT x1, x2;
                givens_d_solve(a.piv64 != 0, D + 3 * l, l, hgt, rl, right, p2, x1, x2);
                if(j < wid) {
                    if(p1) s.T[32 * l + j] = x1;
                    if(p2) s.T[32 * (l + 1) + j] = x2;
                }
            }
        }
    }
    wave_sync();
    offdiag_output(a, q, s.T, false, false, 0.0, hgt, wid, m.format);
}

// ---------------------------------------------------------------------------
// Off-diagonal blocks outside the one-lane form, one wave each, the output
// tile in LDS. The matching pairs of a chunk of 64 are taken one per lane
// where both blocks have at most LIGHT_E entries: each lane forms its pair's
// few updates (entries that share a row), all lanes together going through
// the chain of dependent loads once, and the updates are applied in pair
// order. Other pairs are staged one at a time in their place in that order:
// U_ki as a tile, U_kj (at most 64 entries, else the block is handed to
// k_offdiag_general) as a list ordered by (column, row). Arithmetic and order
// are those of the general form. Bound by latency, at small sizes by the few
// blocks with staged pairs: FP64, a level at n = 2,000 took 36.9 us with every
// step of substitution, scaling and output written out, 24.8 with loops over
// what is there (refactor 3.73 -> 3.27 ms; 4.23 -> 3.65 at n = 33,333 with
// Bunch-Kaufman pivots).

template<typename VT>
struct alignas(16) OffLdsSmall {
    VT X[1024];   // the output tile
    VT A[1024];   // a staged U_ki, the rows' old order, U_ii
    VT cs[32], cd[32], cb[32];
    VT rv[64];
    int32_t cst[33];
    uint8_t rl[64];
};

__device__ __forceinline__ Dep dep_meta(const BlockMeta* bout, int blk, int rb, int rk)
{
    const BlockMeta m = bout[blk];
    return Dep{m.format, m.nnz, m.col_ptr, m.val_ptr, rb, rk};
}

// nonzero entries of a small sparse block (width w, one per lane) sorted by
// (column, row) into rl / rv; cst[c] = entries in columns < c, c = 0..32
template<typename VT>
__device__ void list_build(VT* rv, uint8_t* rl, int32_t* cst, const Dep& d, const Pre<VT>& p,
    int w)
{
    const int lane = lane_id();
    constexpr int NONE = 0x7fffffff;
    int key = NONE, r = 0;
    if(lane < d.nnz && p.v != (VT) 0) {
        r = p.ix / w;
        key = (p.ix - r * w) * 32 + r;
    }
    int rank = 0, below = 0;
    for(int f = 0; f < d.nnz; ++f) {
        const int kf = wave_bcast(key, f);
        rank += (kf < key);
        below += (kf != NONE) && ((kf >> 5) < lane);
    }
    if(key != NONE) {
        rl[rank] = (uint8_t) r;
        rv[rank] = p.v;
    }
    if(lane <= 32) cst[lane] = below;
}

// T[c][j] -= sum_l R[l][j] * Lt[c][l] over the listed rows l of column j,
// ascending, Lt as in product()
template<typename VT>
__device__ void product_list(VT* T, const VT* A, const VT* rv, const uint8_t* rl,
    const int32_t* cst, const VT* cs, const VT* cd, const VT* cb, int lh, int rh)
{
    const int lane = lane_id();
    const int j = lane & 31;
    const int c0 = lane >> 5;
    const int k0 = (j < rh) ? cst[j] : 0;
    const int k1 = (j < rh) ? cst[j + 1] : 0;
    if(k0 < k1) {
        // four output rows of a lane together: their LDS reads are in flight at
        // once (one row at a time waits for them 16 times: 5.8 us a pair)
#pragma unroll 1
        for(int c4 = c0; c4 < lh; c4 += 8) {
            VT acc[4];
#pragma unroll
            for(int t = 0; t < 4; ++t) acc[t] = 0;
#pragma unroll 1
            for(int k = k0; k < k1; ++k) {
                const int l = rl[k];
                const VT r = rv[k];
                const VT sup = cs[l], dia = cd[l], sub = cb[l];
                const VT* Al = A + 32 * l + c4;
                const VT* Ap = l == 0 ? Al : Al - 32;
                const VT* An = l == 31 ? Al : Al + 32;
#pragma unroll
                for(int t = 0; t < 4; ++t) {
                    const VT left = (l == 0) ? (VT) 0 : Ap[2 * t];
                    const VT right = (l == 31) ? (VT) 0 : An[2 * t];
                    const VT lt = fma(sub, right, fma(dia, Al[2 * t], sup * left));
                    acc[t] = fma(r, lt, acc[t]);
                }
            }
#pragma unroll
            for(int t = 0; t < 4; ++t)
                if(c4 + 2 * t < lh) T[32 * (c4 + 2 * t) + j] -= acc[t];
        }
    }
}

// What a Schur pair of blocks with at most LIGHT_E entries each subtracts,
// formed by one lane with product()'s operations: one update per pair of
// entries in a common row. False outside the form: more entries, a 2x2 pivot
// or a non-finite value among the rows, more than LIGHT_OFF updates or two of
// one element.
template<typename VT>
struct PairUpd {
    int n;
    int el[LIGHT_OFF];   // 32 row + column of the tile
    VT v[LIGHT_OFF];
};

template<typename VT, int E>
__device__ __forceinline__ bool light_pair(const Dep& di, const Dep& dj, const RowOf& hgt,
    const RowOf& wid,
    const int32_t* ixs, const VT* vals, const double* tri, PairUpd<VT>& o)
{
    o.n = 0;
#pragma unroll
    for(int k = 0; k < LIGHT_OFF; ++k) { o.el[k] = -1; o.v[k] = (VT) 0; }
    if(di.fmt != FMT_SPARSE || di.nnz > E || di.nnz == 0 || dj.fmt != FMT_SPARSE ||
        dj.nnz > E || dj.nnz == 0)
        return false;
    int ki[E], kj[E];   // 32 row + column, -1 for no entry
    VT vi[E], vj[E], dd[E];
#pragma unroll
    for(int e = 0; e < E; ++e) {
        const int ai = min(e, di.nnz - 1), aj = min(e, dj.nnz - 1);
        ki[e] = ixs[(int64_t) di.cp + ai];
        vi[e] = vals[(int64_t) di.vp + ai];
        kj[e] = ixs[(int64_t) dj.cp + aj];
        vj[e] = vals[(int64_t) dj.vp + aj];
    }
    bool ok = true;
#pragma unroll
    for(int e = 0; e < E; ++e) {
        ki[e] = hgt.at(ki[e]);
        kj[e] = wid.at(kj[e]);
        const double* t = tri + 3 * (int64_t) (dj.rb + (kj[e] >> 5));
        const double sup = t[0], dia = t[1], sub = t[2];
        ok = ok && sup == 0.0 && sub == 0.0 && fabs(dia) < (double) INFINITY &&
            finite_value(vi[e]) && finite_value(vj[e]);
        dd[e] = (VT) dia;
        if(e >= di.nnz) ki[e] = -1;
        if(e >= dj.nnz || vj[e] == (VT) 0) kj[e] = -1;
    }
#pragma unroll
    for(int f = 0; f < E; ++f)
#pragma unroll
        for(int e = 0; e < E; ++e)
            if(kj[f] >= 0 && (ki[e] >> 5) == (kj[f] >> 5)) {
                const int el = 32 * (ki[e] & 31) + (kj[f] & 31);
                const VT lt = dd[f] * vi[e];
                const VT acc = fma(vj[f], lt, (VT) 0);
#pragma unroll
                for(int k = 0; k < LIGHT_OFF; ++k) {
                    ok = ok && !(k < o.n && o.el[k] == el);
                    if(k == o.n) { o.el[k] = el; o.v[k] = acc; }
                }
                ++o.n;
            }
    return ok && o.n <= LIGHT_OFF;
}

template<typename VT>
__device__ __forceinline__ void offdiag_small_one(const FactorArgs<VT>& a, const LevelRange& lr, int q,
    OffLdsSmall<VT>& s)
{
    const int lane = lane_id();
    const int64_t p = (int64_t) lr.lo + q;
    const int4 t0 = ((const int4*) a.off_task)[3 * p];
    const int4 t1 = ((const int4*) a.off_task)[3 * p + 1];
    const int4 t2 = ((const int4*) a.off_task)[3 * p + 2];
    const int fr = t0.y;
    const int hgt = t0.z & 255, wid = (t0.z >> 8) & 255;
    const int pq = t0.w;
    const int np = t2.y;
    const int4* pairs = (const int4*) a.upd4 + pair_first(t2);
    // what the end needs, in flight meanwhile
    const uint32_t flags = a.piv_flag[pq];
    const uint32_t um_row = (lane < hgt) ? a.piv_umask[(int64_t) pq * 32 + lane] : 0u;
    const double d_row = a.tri[3 * (int64_t) (fr + min(lane, hgt - 1)) + 1];
    tile_load(s.X, t1, hgt, wid, a.ix_in, a.val_in);
    // U_ii for the end, rows 2 t and 2 t + 1 in register t (what lies beyond
    // its hgt x hgt elements is not used)
    VT u[16];
#pragma unroll
    for(int t = 0; t < 16; ++t) u[t] = (VT) 0;
    if(flags & PIV_ANY) {
        const VT* piv = a.if_val + (int64_t) pq * 1024;
        const int u0 = (lane >> 5) * hgt + (lane & 31);
#pragma unroll
        for(int t = 0; t < 16; ++t) u[t] = piv[min(u0 + 2 * t * hgt, 1023)];
    }
    bool staging = false;   // s.A is zero
    const RowOf height(hgt), width(wid);

    // A_ij -= U_ki' D_k U_kj over the Schur pairs, in order
    for(int e0 = 0; e0 < np; e0 += 64) {
        Dep mi{}, mj{};
        PairUpd<VT> up;
        up.n = 0;
        bool hit = false, light = false;
        if(e0 + lane < np) {
            const int4 pr = pairs[e0 + lane];
            hit = pair_matches(a.row_mask[pr.x], a.row_mask[pr.y]);
            if(hit) {
                mi = dep_meta(a.bout, pr.x, pr.z, pr.w);
                mj = dep_meta(a.bout, pr.y, pr.z, pr.w);
            }
        }
        if(!wave_ballot(hit)) continue;
        // the form costs the square of its entries: the short one where no
        // pair in it would need more
        const bool in_form = hit && mi.fmt == FMT_SPARSE && mi.nnz <= LIGHT_E &&
            mj.fmt == FMT_SPARSE && mj.nnz <= LIGHT_E;
        const bool longer = wave_ballot(in_form && max(mi.nnz, mj.nnz) > LIGHT_E / 2) != 0ull;
        if(in_form)
            light = longer ?
                light_pair<VT, LIGHT_E>(mi, mj, height, width, a.ix_out, a.val_out, a.tri, up) :
                light_pair<VT, LIGHT_E / 2>(mi, mj, height, width, a.ix_out, a.val_out, a.tri, up);
        if(wave_ballot(hit && !light && !small_sparse<VT>(mj))) {
            if(lane == 0) a.defer_list[atomicAdd(a.defer_cnt + lr.level, 1)] = q;
            return;
        }
        const uint64_t heavy = wave_ballot(hit && !light);
        for(uint64_t m = wave_ballot(hit && (!light || up.n > 0)); m; m &= m - 1) {
            const int d = __ffsll((long long) m) - 1;
            if(!((heavy >> d) & 1ull)) {
                if(lane == d) {
#pragma unroll
                    for(int k = 0; k < LIGHT_OFF; ++k)
                        if(k < up.n) s.X[up.el[k]] -= up.v[k];
                }
                wave_sync();
                continue;
            }
            if(!staging) {
                tile_zero(s.A);
                wave_sync();
                staging = true;
            }
            const Dep ci = bcast(mi, d), cj = bcast(mj, d);
            const Pre<VT> pi = prefetch(ci, a.ix_out, a.val_out, a.tri, true);
            const Pre<VT> pj = prefetch(cj, a.ix_out, a.val_out, a.tri, false);
            stage(s.A, (uint32_t*) nullptr, ci, pi, height, a.ix_out, a.val_out);
            list_build(s.rv, s.rl, s.cst, cj, pj, wid);
            stage_d(s.cs, s.cd, s.cb, pi);
            wave_sync();
            product_list(s.X, s.A, s.rv, s.rl, s.cst, s.cs, s.cd, s.cb, hgt, wid);
            wave_sync();
            unstage(s.A, (uint32_t*) nullptr, ci, pi, height);
            wave_sync();
        }
    }
    // rows in the block row's pivoting order (kernels :1733-1751)
    if(flags & PIV_PERM) {
        tile_copy(s.A, s.X);
        wave_sync();
        for(int e = lane; e < hgt * 32; e += 64) {
            const int r = e >> 5, c = e & 31;
            s.X[e] = s.A[32 * (a.perm[fr + r] - fr) + c];
        }
        wave_sync();
    }
    // U_ii' forward substitution over the pivot rows with an element beyond the
    // diagonal and a nonzero in the tile (exact no-ops are skipped): the lanes
    // of both halves hold the row, lane l updates elements 64 t + l of the
    // tile. Short loops: with all 32 x 32 steps written out the code did not
    // fit beside the rest in the instruction cache, and a CU's first block of a
    // launch took 11-24 us here, where later ones took 0.7
    if(flags & PIV_ANY) {
#pragma unroll
        for(int t = 0; t < 16; ++t) s.A[64 * t + lane] = u[t];
        wave_sync();
#pragma unroll 1
        for(uint64_t m = wave_ballot(um_row != 0u); m; m &= m - 1) {
            const int ii = __ffsll((long long) m) - 1;
            const uint32_t um = (uint32_t) __builtin_amdgcn_readlane((int) um_row, ii);
            const VT x = s.X[32 * ii + (lane & 31)];
            const bool on = x != (VT) 0;
            if(wave_ballot(on) == 0ull) continue;
            const VT pv = x / s.A[33 * ii];
#pragma unroll 1
            for(int g = 0; g < 4; ++g) {
                const uint32_t bits = (um >> (8 * g)) & 255u;
                if(bits == 0u) continue;
                VT* X = s.X + 256 * g + lane;
                const VT* U = s.A + 32 * ii + 8 * g + (lane >> 5);
                VT y[4];
#pragma unroll
                for(int t = 0; t < 4; ++t) y[t] = fma(-U[2 * t], pv, X[64 * t]);
#pragma unroll
                for(int t = 0; t < 4; ++t)
                    if(on && ((bits >> (2 * t + (lane >> 5))) & 1u)) X[64 * t] = y[t];
            }
            wave_sync();
        }
    }
    const int jc = lane;
    VT* col = s.X + jc;
    // D solve in place (d_left_solve_with_D_Ut, kernels :1533-1566); a row
    // is written only after both rows it reads have been read
    if((flags & PIV_2X2) && jc < wid) {
        const double* D = a.tri + 3 * (int64_t) fr;
        const int32_t* ip = a.is_piv + fr;
        for(int l = 0; l < hgt; ++l) {
            const bool p1 = ip[l] != 0;
            const bool p2 = (l + 1 < hgt) && !ip[l + 1];
            const VT rl = col[32 * l];
            const VT right = (l < 31) ? col[32 * (l + 1)] : rl;
            VT x1, x2;
            givens_d_solve(a.piv64 != 0, D + 3 * l, l, hgt, rl, right, p2, x1, x2);
            if(p1) col[32 * l] = x1;
            if(p2) col[32 * (l + 1)] = x2;
        }
    }
    wave_sync();
    offdiag_output(a, q, s.X, !(flags & PIV_2X2), flags & PIV_NONFINITE, d_row, hgt, wid, t1.x);
}

// the positions the one-lane form leaves to the wave form, grid-stride
template<typename VT>
__device__ __forceinline__ void offdiag_body(const FactorArgs<VT>& a, const LevelRange& lr,
    int bid_, int nblk_)
{
    __shared__ OffLdsSmall<VT> s;
    const int nw = a.wave_cnt[lr.level];
    for(int t = bid_; t < nw; t += nblk_) {
        offdiag_small_one(a, lr, a.wave_list[t], s);
        wave_sync();
    }
}

// ---------------------------------------------------------------------------
// One lane per off-diagonal block for small blocks (at level-0 fill of the
// KKT workloads: 1-2 entries each; a wave then works on 64 blocks instead of
// one). Static eligibility (task bit, set by the host): sparse input with at
// most LIGHT_E entries, at most 8 Schur pairs (16 at a level with 8192 or
// more off-diagonal blocks), 1x1 pivots in the block row.
// At run time every matching pair must be within light_pair's form and the
// tile must stay within TINY_P nonzeros (TINY_T while it is scaled);
// otherwise the position goes to the wave form before anything is written.
// The tile is a list of (row * 32 + col, value) in LDS, one column of the
// list arrays per lane; every value is formed by the same operations in the
// same order as in the wave form (terms that are exact zeros there are
// skipped).
constexpr int TINY_T = 16;
constexpr int TINY_P = 12;  // the same while its Schur updates are added up
constexpr int TINY_F = 6;   // pairs whose row masks are fetched together

template<typename VT, int CAP, int TPB>
struct TinyLds {
    VT v[CAP][TPB];
    int16_t ix[CAP][TPB];
};

template<typename VT>
__device__ __forceinline__ void to_wave_form(const FactorArgs<VT>& a, const LevelRange& lr, int q)
{
    a.wave_list[atomicAdd(a.wave_cnt + lr.level, 1)] = q;
}

// One-lane form, first phase: the Schur updates of the off-diagonal block at
// level position q (thread tid of its workgroup), which read only blocks of
// earlier levels and so run beside the level's pivot blocks. The tile list
// is parked as the position's entry list (EntryList: the first LIST_C in c_idx /
// c_val, the others in if_idx / if_val, count in if_cnt); if_cnt[q] = -1 marks a position left to the other kernels.
template<typename VT, int TPB>
__device__ __forceinline__ void tiny_pairs_one(const FactorArgs<VT>& a, const LevelRange& lr, const int q,
    const int tid, TinyLds<VT, TINY_P, TPB>& s)
{
    if(q >= lr.size) return;
    a.if_cnt[q] = -1;
    const int64_t p = (int64_t) lr.lo + q;
    const int4 t0 = ((const int4*) a.off_task)[3 * p];
    const int4 t1 = ((const int4*) a.off_task)[3 * p + 1];
    const int4 t2 = ((const int4*) a.off_task)[3 * p + 2];
    if(!(t2.z & 1)) { to_wave_form(a, lr, q); return; }
    const int hgt = t0.z & 255, wid = (t0.z >> 8) & 255;
    const int np = t2.y;
    const int4* pairs = (const int4*) a.upd4 + pair_first(t2);
    VT* tv = &s.v[0][tid];
    int16_t* ti = &s.ix[0][tid];
    auto V = [&](int k) -> VT& { return tv[k * TPB]; };
    auto I = [&](int k) -> int16_t& { return ti[k * TPB]; };
    int n = 0;
    auto find = [&](int idx) {
        for(int k = 0; k < n; ++k)
            if(I(k) == idx) return k;
        return -1;
    };
    const RowOf height(hgt), width(wid);
    // the first pairs' records beside the input entries
    int4 rec[TINY_F];
    auto records = [&](int p0) {
#pragma unroll
        for(int u = 0; u < TINY_F; ++u) rec[u] = pairs[min(p0 + u, np - 1)];
    };
    if(np > 0) records(0);
    n = t1.y;
    for(int e0 = 0; e0 < n; e0 += 4) {
        int ix[4];
        VT v[4];
#pragma unroll
        for(int u = 0; u < 4; ++u) {
            const int e = min(e0 + u, n - 1);
            ix[u] = a.ix_in[(int64_t) t1.z + e];
            v[u] = a.val_in[(int64_t) t1.w + e];
        }
#pragma unroll
        for(int u = 0; u < 4; ++u)
            if(e0 + u < n) {
                I(e0 + u) = (int16_t) width.at(ix[u]);
                V(e0 + u) = v[u];
            }
    }
    // A_ij -= U_ki' D_k U_kj over the Schur pairs, in order: the row masks
    // of TINY_F pairs are fetched together, and of the pairs that match (few)
    // the metadata, entries and D are read one pair after the other. A pair
    // outside light_pair's form leaves the block to the one-wave form.
    for(int p0 = 0; p0 < np; p0 += TINY_F) {
        if(p0) records(p0);
        uint32_t hits = 0;
        {
            uint32_t mi[TINY_F], mj[TINY_F];
#pragma unroll
            for(int u = 0; u < TINY_F; ++u) {
                mi[u] = a.row_mask[rec[u].x];
                mj[u] = a.row_mask[rec[u].y];
            }
#pragma unroll
            for(int u = 0; u < TINY_F; ++u)
                if(p0 + u < np && pair_matches(mi[u], mj[u])) hits |= 1u << u;
        }
        for(; hits; hits &= hits - 1) {
            const int at = __ffs(hits) - 1;
            int4 pc = rec[0];
#pragma unroll
            for(int u = 1; u < TINY_F; ++u)
                if(u == at) pc = rec[u];
            const Dep mi = dep_meta(a.bout, pc.x, pc.z, pc.w);
            const Dep mj = dep_meta(a.bout, pc.y, pc.z, pc.w);
            PairUpd<VT> up;
            const bool ok = wave_ballot(mi.nnz > 2 || mj.nnz > 2) == 0ull
                ? light_pair<VT, 2>(mi, mj, height, width, a.ix_out, a.val_out, a.tri, up)
                : light_pair<VT, LIGHT_E>(mi, mj, height, width, a.ix_out, a.val_out, a.tri, up);
            if(!ok) {
                to_wave_form(a, lr, q);
                return;
            }
#pragma unroll
            for(int u = 0; u < LIGHT_OFF; ++u) {
                if(u >= up.n) continue;
                int k = find(up.el[u]);
                if(k < 0) {
                    if(up.v[u] == (VT) 0) continue;
                    if(n == TINY_P) {
                        to_wave_form(a, lr, q);
                        return;
                    }
                    k = n++;
                    I(k) = (int16_t) up.el[u];
                    V(k) = 0;
                }
                V(k) -= up.v[u];
            }
        }
    }
    // the tile list for the second phase
    const EntryList<VT> o = entry_list(a, q);
    for(int k = 0; k < n; ++k) o.set(k, I(k), V(k));
    a.if_cnt[q] = n;
}

// One-lane form, second phase (after the level's pivot blocks): the tile
// list of the first phase in the block row's pivoting order, through U_ii'
// and D, then the row sums of squares and the compact entries. Lists of at
// most LIST_C entries whose rows have nothing right of the diagonal of U_ii
// (nearly all at level-0 fill) stay in registers; the others go through LDS.
template<typename VT>
__device__ __forceinline__ void offdiag_tiny_scale_body(const FactorArgs<VT>& a, const LevelRange& lr,
    int bid_)
{
    __shared__ TinyLds<VT, TINY_T, TINY_TPB> s;
    const int tid = threadIdx.x;
    const int q = lr.npiv + bid_ * TINY_TPB + tid;
    if(q >= lr.size) return;
    // the parked count, the first entries and the task record together
    // (none waits for the others)
    const int64_t p = (int64_t) lr.lo + q;
    const int4 t0 = ((const int4*) a.off_task)[3 * p];
    int n = a.if_cnt[q];
    VT v[LIST_C];
    int ix[LIST_C];
#pragma unroll
    for(int e = 0; e < LIST_C; ++e) {
        v[e] = a.c_val[(int64_t) q * LIST_C + e];
        ix[e] = a.c_idx[(int64_t) q * LIST_C + e];
    }
    if(n < 0) return;
    const int fr = t0.y;
    const int hgt = t0.z & 255;
    const int pq = t0.w;
    const uint32_t flags = a.piv_flag[pq];
    if(flags & PIV_2X2) {
        // numeric pivoting chose a 2x2 pivot
        to_wave_form(a, lr, q);
        return;
    }
    const uint8_t* iperm = a.piv_iperm + (int64_t) pq * 32;
    const uint32_t* umask = a.piv_umask + (int64_t) pq * 32;
    const double* D = a.tri + 3 * (int64_t) fr;
    const EntryList<VT> o = entry_list(a, q);
    bool plain = n <= LIST_C;
    if(plain) {
        if(flags & PIV_PERM) {
#pragma unroll
            for(int e = 0; e < LIST_C; ++e)
                if(e < n) ix[e] = 32 * iperm[ix[e] >> 5] + (ix[e] & 31);
        }
        if(flags & PIV_ANY) {
#pragma unroll
            for(int e = 0; e < LIST_C; ++e)
                if(e < n) plain = plain && (umask[ix[e] >> 5] == 0u || v[e] == (VT) 0);
        }
    }
    if(plain) {
        constexpr int NONE = 1 << 20;
        double dv[LIST_C];
#pragma unroll
        for(int e = 0; e < LIST_C; ++e) dv[e] = (e < n) ? D[3 * (ix[e] >> 5) + 1] : 1.0;
#pragma unroll
        for(int e = 0; e < LIST_C; ++e) {
            if(e < n) v[e] = (VT) ((double) v[e] / dv[e]);
            else ix[e] = NONE;
        }
        // tile order (row-major)
        auto order = [&](int x, int y) {
            if(ix[y] < ix[x]) {
                const int ti = ix[x]; ix[x] = ix[y]; ix[y] = ti;
                const VT tv = v[x]; v[x] = v[y]; v[y] = tv;
            }
        };
        static_assert(LIST_C == 4, "sorting network on four");
        order(0, 1); order(2, 3); order(0, 2); order(1, 3); order(1, 2);
        uint32_t rows = 0;
        int nr = 0, cnt = 0;
        VT ssq = 0;
#pragma unroll
        for(int e = 0; e < LIST_C; ++e) {
            if(ix[e] == NONE) continue;
            ssq = fma(v[e], v[e], ssq);
            // the row ends here
            if(e == LIST_C - 1 || (ix[min(e + 1, LIST_C - 1)] >> 5) != (ix[e] >> 5)) {
                if(!(ssq == (VT) 0)) {
                    if(nr == 0) a.rn_first[q] = ssq;
                    else a.rn_part[(int64_t) q * 32 + nr] = ssq;
                    rows |= 1u << (ix[e] >> 5);
                    ++nr;
                }
                ssq = 0;
            }
            if(fabs((double) v[e]) > NZ_EPS) {
                o.cv[cnt] = v[e];
                o.ci[cnt] = (uint16_t) ix[e];
                ++cnt;
            }
        }
        a.part_mask[q] = rows;
        a.if_cnt[q] = cnt;
        return;
    }
    VT* tv = &s.v[0][tid];
    int16_t* ti = &s.ix[0][tid];
    auto V = [&](int k) -> VT& { return tv[k * TINY_TPB]; };
    auto I = [&](int k) -> int16_t& { return ti[k * TINY_TPB]; };
    auto find = [&](int idx) {
        for(int k = 0; k < n; ++k)
            if(I(k) == idx) return k;
        return -1;
    };
    for(int k = 0; k < n; ++k) {
        int at = o.idx(k);
        if(flags & PIV_PERM) at = 32 * iperm[at >> 5] + (at & 31);
        I(k) = (int16_t) at;
        V(k) = o.val(k);
    }
    // U_ii' forward substitution over the rows in ascending order: the next
    // row with an entry and something right of its diagonal
    const VT* piv = a.if_val + (int64_t) pq * 1024;
    for(int ii = -1; flags & PIV_ANY;) {
        int nxt = 32;
        for(int k = 0; k < n; ++k) {
            const int r = I(k) >> 5;
            if(r > ii && r < nxt && V(k) != (VT) 0) nxt = r;
        }
        if(nxt >= hgt) break;
        ii = nxt;
        const uint32_t um = umask[ii];
        if(!um) continue;
        const VT d = piv[ii * hgt + ii];
        const int n0 = n;
        for(int k = 0; k < n0; ++k) {
            if((I(k) >> 5) != ii || V(k) == (VT) 0) continue;
            const int jc = I(k) & 31;
            const VT pv = V(k) / d;
            for(uint32_t bits = um; bits; bits &= bits - 1) {
                const int l = __ffs(bits) - 1;
                const int idx = 32 * l + jc;
                int m = find(idx);
                if(m < 0) {
                    if(n == TINY_T) { to_wave_form(a, lr, q); return; }
                    m = n++;
                    I(m) = (int16_t) idx;
                    V(m) = 0;
                }
                V(m) = fma(-piv[ii * hgt + l], pv, V(m));
            }
        }
    }
    // D solve (1x1 pivots): the Givens-form solve reduces to a division;
    // the divisors of eight entries are loaded together
    for(int k0 = 0; k0 < n; k0 += 8) {
        double dv[8];
#pragma unroll
        for(int u = 0; u < 8; ++u) dv[u] = D[3 * (I(min(k0 + u, n - 1)) >> 5) + 1];
#pragma unroll
        for(int u = 0; u < 8; ++u)
            if(k0 + u < n) V(k0 + u) = (VT) ((double) V(k0 + u) / dv[u]);
    }
    // tile order (row-major)
    for(int k = 1; k < n; ++k) {
        const int16_t ik = I(k);
        const VT vk = V(k);
        int m = k - 1;
        while(m >= 0 && I(m) > ik) {
            I(m + 1) = I(m);
            V(m + 1) = V(m);
            --m;
        }
        I(m + 1) = ik;
        V(m + 1) = vk;
    }
    // row sums of squares (columns ascending) and the compact list
    uint32_t rows = 0;
    int nr = 0;
    for(int k = 0; k < n;) {
        const int r = I(k) >> 5;
        VT ssq = 0;
        while(k < n && (I(k) >> 5) == r) {
            ssq = fma(V(k), V(k), ssq);
            ++k;
        }
        if(!(ssq == (VT) 0)) {
            if(nr == 0) a.rn_first[q] = ssq;
            else a.rn_part[(int64_t) q * 32 + nr] = ssq;
            rows |= 1u << r;
            ++nr;
        }
    }
    a.part_mask[q] = rows;
    int pos = 0;
    for(int m = 0; m < n; ++m)
        if(fabs((double) V(m)) > NZ_EPS) o.set(pos++, I(m), V(m));
    a.if_cnt[q] = pos;
}
// The level's pivot blocks (workgroups 0 .. npiv - 1) and the first phase
// of the one-lane off-diagonal form (the rest, 64 NW positions each) in one
// launch: the two read disjoint data and never wait for each other.
template<typename VT, int NW>
union PivPairsLds {
    PivLds<VT, NW> piv;
    TinyLds<VT, TINY_P, 64 * NW> tiny;
};

template<typename VT, int NW, bool TWO>
__device__ __forceinline__ void pivots_pairs_body(const FactorArgs<VT>& a, const LevelRange& lr,
    int bid_)
{
    __shared__ PivPairsLds<VT, NW> u;
    const int w = bid_;
    if(w < lr.npiv) {
        pivots_one<VT, NW, TWO>(a, lr, w, u.piv);
        return;
    }
    const int q0 = lr.npiv + (w - lr.npiv) * 64 * NW;
    tiny_pairs_one<VT, 64 * NW>(a, lr, q0 + (int) threadIdx.x, (int) threadIdx.x, u.tiny);
}


template<typename VT>
__device__ __forceinline__ VT drop_norm(VT rn) { return (VT) sqrtf((float) rn); }

// Leftover pool and granted extra space of a level's blocks in level-list
// order (kernels :1948-2008 with the atomics serialised in that order). The
// pool after a sparse block is max(pool + max_nnz - kept candidates, 0); such
// maps p -> max(p + a, b) compose associatively, so the pool sequence is a
// scan. A block stores cap + (pool before) - (pool after) entries whatever
// it was granted, so the sizes stored before a position add up to the
// capacities before it (a static prefix sum) minus the pool at it: output
// offsets need no scan of their own.
struct PoolMap {
    int64_t a, b;
    __device__ static PoolMap shfl_up(const PoolMap& m, int o)
    {
        return {__shfl_up(m.a, o, WAVE), __shfl_up(m.b, o, WAVE)};
    }
};
struct MapOp {
    // first x, then y
    __device__ PoolMap operator()(const PoolMap& x, const PoolMap& y) const
    {
        const int64_t nb = x.b + y.a;
        return {x.a + y.a, nb > y.b ? nb : y.b};
    }
};
__device__ __forceinline__ int64_t map_apply(const PoolMap& m, int64_t p)
{
    const int64_t v = p + m.a;
    return v > m.b ? v : m.b;
}
constexpr int DR_TPB = GROUP_BLOCKS;
constexpr int DR_NW = DR_TPB / WAVE;
constexpr int DR_RUNS = 512;        // row sums a wave lays out at once
constexpr int32_t CAP_NONE = -0x7fffffff;
constexpr int LIST_GROUP = 16;      // entries of a block taken by sixteen lanes
constexpr int GROUP_SPIN_LIMIT = 1 << 22;

template<typename VT>
struct DropLds {
    VT val[DR_NW][DR_RUNS];                            // row sums, in block order
    uint32_t rows[DR_NW][GROUP_ROWS][DR_RUNS / 32 + 1];   // per fine row: which are its own
    int32_t runs[DR_NW];
    VT nrm[GROUP_ROWS];
    int32_t frow[GROUP_ROWS], rflag[GROUP_ROWS];
    PoolMap sh[DR_NW];
    int64_t pool;
    int32_t ticket;
};

// Words of a row group's state: each carries its own validity in the low two
// bits, so that readers need no ordering between them (relaxed 8-byte
// agent-coherent stores and loads, no fences).
__device__ __forceinline__ void publish(int64_t* p, int64_t v)
{
    __hip_atomic_store(p, (int64_t) ((uint64_t) v << 2) | 1, __ATOMIC_RELAXED,
        __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int64_t published_word(const int64_t* p)
{
    return __hip_atomic_load(const_cast<int64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The pool before row group g of a level (one wave): the groups before it are
// looked at 64 at a time, nearest first, until one whose pool is known or the
// level's start (pool0); the maps in between are composed in order. A wait
// that gives up records 2 in *err and goes on.
__device__ int64_t pool_before(const int64_t* st, int g, int64_t pool0, int32_t* err)
{
    const int lane = lane_id();
    PoolMap acc{0, 0};
    int spins = 0;
    for(int base = g - 1;; base -= WAVE) {
        const int idx = base - lane;
        int64_t wa = 0, wb = 0, wp = 0;
        bool known = idx < 0, have = known;
        int near;
        for(;;) {
            if(!have) {
                wp = published_word(st + 3 * (int64_t) idx + 2);
                wa = published_word(st + 3 * (int64_t) idx);
                wb = published_word(st + 3 * (int64_t) idx + 1);
                known = wp != 0;
                have = known || (wa != 0 && wb != 0);
            }
            const uint64_t km = wave_ballot(known);
            near = km ? __ffsll((long long) km) - 1 : WAVE;
            const uint64_t need = near < WAVE ? (1ull << near) - 1 : ~0ull;
            if((wave_ballot(!have) & need) == 0ull) break;
            __builtin_amdgcn_s_sleep(1);
            if(++spins > GROUP_SPIN_LIMIT) {
                if(lane == 0 && err)
                    __hip_atomic_store(err, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                break;
            }
        }
        // lane 0 holds the latest group of the window
        PoolMap m{0, 0};
        if(lane < near) m = PoolMap{wa >> 2, wb >> 2};
#pragma unroll
        for(int o = 1; o < WAVE; o <<= 1) {
            const PoolMap u{__shfl_down(m.a, o, WAVE), __shfl_down(m.b, o, WAVE)};
            if(lane + o < WAVE) m = MapOp()(u, m);
        }
        acc = MapOp()(PoolMap{__shfl(m.a, 0, WAVE), __shfl(m.b, 0, WAVE)}, acc);
        if(near < WAVE) {
            const int64_t p = __shfl(idx < 0 ? pool0 : wp >> 2, near, WAVE);
            return map_apply(acc, p);
        }
    }
}

// the position a thread of k_drop works on, with its first LIST_C entries
template<typename VT>
struct DropPos {
    int cap, row0, w, col, val, blk, cnt;
    VT v[LIST_C];
    int ix[LIST_C];
};

template<typename VT>
__device__ __forceinline__ void drop_load(const FactorArgs<VT>& a, const LevelRange& lr, int q,
    bool in, DropPos<VT>& p)
{
    const int qc = in ? q : 0;
    const int4 l = a.lq[lr.lo + qc];
    p.cap = in ? l.x : CAP_NONE;
    p.row0 = l.y;
    p.w = l.z;
    p.col = l.w;
    p.val = a.lq_val[lr.lo + qc];
    p.blk = a.lvlb_idx[lr.lo + qc];
    p.cnt = in ? a.if_cnt[qc] : 0;
#pragma unroll
    for(int e = 0; e < LIST_C; ++e) {
        p.v[e] = a.c_val[(int64_t) qc * LIST_C + e];
        p.ix[e] = a.c_idx[(int64_t) qc * LIST_C + e];
    }
}

// Lists of LIST_C + 1 to LIST_GROUP entries (and any of at most LIST_GROUP
// that overflow) are taken by sixteen lanes each, four at a time. visit(src,
// e, on): this lane is entry e of lane src's list (src < 0: no list); on:
// which four lists, as lanes of the wave.
template<typename Visit>
__device__ __forceinline__ void by_sixteen(uint64_t lanes, Visit visit)
{
    const int g = lane_id() >> 4;
    while(lanes) {
        int on[4];
        int src = -1;
#pragma unroll
        for(int k = 0; k < 4; ++k) {
            on[k] = lanes ? __ffsll((long long) lanes) - 1 : -1;
            lanes &= lanes - 1;
            if(g == k) src = on[k];
        }
        visit(src, lane_id() & 15, on);
    }
}

// entries of a sparse position that survive |v| >= tau * sqrtf(norm)
// (kernels :1919-1946); lists over LIST_GROUP entries by the whole wave
template<typename VT>
__device__ __forceinline__ int drop_count(const FactorArgs<VT>& a, int q, const DropPos<VT>& p,
    const VT* nrm)
{
    auto keeps = [&](VT v, VT n) { return !(fabs(v) < a.threshold * n); };
    int keep = 0;
    if(p.cap >= 0 && p.cnt <= LIST_C) {
#pragma unroll
        for(int e = 0; e < LIST_C; ++e)
            if(e < p.cnt) keep += keeps(p.v[e], nrm[p.row0 + (p.ix[e] >> 5)]);
    }
    by_sixteen(wave_ballot(p.cap >= 0 && p.cnt > LIST_C && p.cnt <= LIST_GROUP),
        [&](int src, int e, const int (&on)[4]) {
            const int from = max(src, 0);
            const int bq = __shfl(q, from), bc = __shfl(p.cnt, from), br = __shfl(p.row0, from);
            const EntryList<VT> l = entry_list(a, bq);
            const bool in = src >= 0 && e < bc;
            const bool k = in && keeps(l.val(in ? e : 0), nrm[br + ((in ? l.idx(e) : 0) >> 5)]);
            const uint64_t kb = wave_ballot(k);
#pragma unroll
            for(int u = 0; u < 4; ++u)
                if(lane_id() == on[u]) keep = __popc((uint32_t) (kb >> (16 * u)) & 0xffffu);
        });
    for(uint64_t bm = wave_ballot(p.cap >= 0 && p.cnt > LIST_GROUP); bm; bm &= bm - 1) {
        const int src = __ffsll((long long) bm) - 1;
        const int bq = __shfl(q, src), bc = __shfl(p.cnt, src), br = __shfl(p.row0, src);
        const EntryList<VT> l = entry_list(a, bq);
        int k = 0;
        for(int e0 = 0; e0 < bc; e0 += WAVE) {
            const int e = min(e0 + lane_id(), bc - 1);
            const bool on = e0 + lane_id() < bc && keeps(l.val(e), nrm[br + (l.idx(e) >> 5)]);
            k += __popcll(wave_ballot(on));
        }
        if(lane_id() == src) keep = k;
    }
    return keep;
}

// Final storage of the wave's sparse blocks with at most LIST_GROUP entries
// (`mine`: this lane has one; the selection and order of store_one), and
// their row masks. NaN entries are counted but never written.
template<typename VT>
__device__ __forceinline__ void drop_store(const FactorArgs<VT>& a, int q, const DropPos<VT>& p,
    const VT* nrm, const int32_t* rflags, int px, int pv, bool mine, bool overflow, int max_nnz)
{
    auto keeps = [&](VT v, VT n) { return !(fabs(v) < a.threshold * n); };
    const bool shared = mine && (overflow || p.cnt > LIST_C);
    if(mine && !shared) {
        uint32_t rows = 0;
        bool bad = false;
        int pos = 0;
#pragma unroll
        for(int e = 0; e < LIST_C; ++e) {
            const int r = p.ix[e] >> 5;
            if(e < p.cnt && keeps(p.v[e], nrm[p.row0 + r])) {
                bad = bad || !finite_value(p.v[e]);
                if(fabs(p.v[e]) >= (VT) 0) {
                    a.ix_out[(int64_t) px + pos] = r * p.w + (p.ix[e] & 31);
                    a.val_out[(int64_t) pv + pos] = p.v[e];
                    rows |= 1u << r;
                    ++pos;
                }
            }
        }
        a.row_mask[p.blk] = store_row_mask(rows, bad, rflags[p.row0]);
    }
    by_sixteen(wave_ballot(shared), [&](int src, int e, const int (&)[4]) {
        const int from = max(src, 0), base = lane_id() & 48;
        const int bq = __shfl(q, from), bc = __shfl(p.cnt, from), br = __shfl(p.row0, from);
        const int bw = __shfl(p.w, from), bx = __shfl(px, from), bv = __shfl(pv, from);
        const int bm = __shfl(max_nnz, from), bb = __shfl(p.blk, from);
        const bool bo = __shfl((int) overflow, from) != 0;
        const EntryList<VT> l = entry_list(a, bq);
        const bool in = src >= 0 && e < bc;
        const VT v = in ? l.val(e) : (VT) 0;
        const int ix = in ? l.idx(e) : 0;
        const bool k = in && keeps(v, nrm[br + (ix >> 5)]);
        const bool bad = k && !finite_value(v);
        // -1: no entry or a dropped one
        const VT key = k ? (VT) fabs(v) : (VT) -1;
        const bool w = key >= (VT) 0;
        const uint32_t wg = (uint32_t) (wave_ballot(w) >> base) & 0xffffu;
        int at = __popc(wg & ((1u << e) - 1));
        if(wave_ballot(src >= 0 && bo)) {
            // over capacity: the max_nnz largest, ties to the lower index
            int rank = 0;
#pragma unroll
            for(int f = 0; f < LIST_GROUP; ++f) {
                const VT kf = __shfl(key, base + f);
                const int xf = __shfl(ix, base + f);
                rank += kf > key || (kf == key && xf < ix);
            }
            if(bo) at = rank;
        }
        uint32_t row = 0;
        if(w && !(bo && at >= bm)) {
            a.ix_out[(int64_t) bx + at] = (ix >> 5) * bw + (ix & 31);
            a.val_out[(int64_t) bv + at] = v;
            row = 1u << (ix >> 5);
        }
#pragma unroll
        for(int o = 1; o < 16; o <<= 1) row |= (uint32_t) __shfl_xor((int) row, o);
        const bool any_bad = ((wave_ballot(bad) >> base) & 0xffffull) != 0;
        if(src >= 0 && e == 0) a.row_mask[bb] = store_row_mask(row, any_bad, rflags[br]);
    });
}

// One launch per level, one workgroup per row group (its ticket's, so every
// group it waits for belongs to a workgroup that is already running). The
// row sums of its blocks, published by the off-diagonal kernels as (row mask,
// sums), are laid out in block order in LDS and added up per fine row in that
// order; each thread then counts what survives of its block, the group's pool
// map goes out, the pool before the group comes from the groups before it,
// and each thread writes its block's metadata and entries.
// Bound by latency: about eight dependent memory round trips. It replaced a
// row-norm launch, a chunked scan with two waits and a store launch (11.6 +
// 36 + 8 us per level at n = 400,000, 5 + 44 + 18 us at n = 2,000); itself 21
// and 29 us.
template<typename VT>
__device__ __forceinline__ void drop_body(const FactorArgs<VT>& a, const LevelRange& lr)
{
    __shared__ DropLds<VT> s;
    const int t = (int) threadIdx.x;
    const int lane = lane_id(), wv = t / WAVE;
    const int64_t pool0 = a.carry[4 * (lr.level & 1)];
    if(t == 0) s.ticket = atomicAdd(a.grp_ticket + lr.level, 1);
    __syncthreads();
    const int g = s.ticket;
    const int4 grp = a.groups[lr.grp_lo + g];
    const int pp0 = grp.x, np = grp.y, q0 = grp.z, nblk = grp.w;
    int64_t* state = a.grp_state + 3 * (int64_t) lr.grp_lo;
    DropPos<VT> pos;
    drop_load(a, lr, q0 + t, t < nblk, pos);
    // the group's block rows: fine rows, flags, pivot block metadata
    if(t < GROUP_ROWS) s.frow[t] = -1;
    __syncthreads();
    if(t < np) {
        const int64_t p = (int64_t) lr.lo + pp0 + t;
        const int4 r = ((const int4*) a.off_task)[3 * p];   // {block, first row, rows, block row}
        const int4 l = a.lq[p];
        const int32_t fl = a.row_flag[r.w];
        for(int k = 0; k < r.z; ++k) {
            s.frow[l.y + k] = r.y + k;
            s.rflag[l.y + k] = fl;
        }
        BlockMeta& o = a.bout[r.x];
        o.nnz = 0;
        o.col_ptr = (int32_t) (l.w - pool0);
        o.val_ptr = (int32_t) (a.lq_val[p] - pool0);
    }
    __syncthreads();
    const int frow = (t < GROUP_ROWS) ? s.frow[t] : -1;
    VT acc = (frow >= 0) ? a.rn[frow] : (VT) 0;
    // row sums of squares: pivot block, then the off-diagonal blocks by id
    for(int c0 = 0; c0 < nblk; c0 += DR_TPB) {
        const int q = q0 + c0 + t;
        const bool in = c0 + t < nblk;
        const uint32_t m = in ? a.part_mask[q] : 0u;
        const VT first = in ? a.rn_first[q] : (VT) 0;
        const int row0 = in ? a.lq[lr.lo + q].y : 0;
        const int n = __popc(m);
        int off = n;
#pragma unroll
        for(int o = 1; o < WAVE; o <<= 1) {
            const int u = __shfl_up(off, o, WAVE);
            if(lane >= o) off += u;
        }
        const int total = __shfl(off, WAVE - 1, WAVE);
        off -= n;
        // all lanes at once, or sixteen (at most DR_RUNS sums) at a time, one
        // wave after the other
        const bool split = __syncthreads_or(total > DR_RUNS) != 0;
        for(int step = 0; step < (split ? 4 * DR_NW : 1); ++step) {
            const int l0 = split ? 16 * (step & 3) : 0;
            const bool mine = !split || step / 4 == wv;
            const int base = __shfl(off, l0, WAVE);
            const int end = (split && l0 < 48) ? __shfl(off, min(l0 + 16, WAVE - 1), WAVE) : total;
            for(int k = lane; k < GROUP_ROWS * (DR_RUNS / 32); k += WAVE)
                s.rows[wv][k / (DR_RUNS / 32)][k % (DR_RUNS / 32)] = 0u;
            if(lane == 0) s.runs[wv] = mine ? end - base : 0;
            wave_sync();
            if(mine && (!split || lane / 16 == l0 / 16)) {
                int j = 0;
                for(uint32_t bits = m; bits; bits &= bits - 1, ++j) {
                    const int at = off - base + j;
                    s.val[wv][at] = (j == 0) ? first : a.rn_part[(int64_t) q * 32 + j];
                    atomicOr(&s.rows[wv][row0 + __ffs(bits) - 1][at >> 5], 1u << (at & 31));
                }
            }
            __syncthreads();
            if(t < GROUP_ROWS)
                for(int u = 0; u < DR_NW; ++u)
                    for(int wd = 0; 32 * wd < s.runs[u]; ++wd)
                        for(uint32_t bits = s.rows[u][t][wd]; bits; bits &= bits - 1)
                            acc += s.val[u][32 * wd + __ffs(bits) - 1];
            __syncthreads();
        }
    }
    if(t < GROUP_ROWS) {
        if(frow >= 0) a.rn[frow] = acc;
        s.nrm[t] = drop_norm(acc);
    }
    __syncthreads();
    // survivors and the group's pool map
    PoolMap tot{0, 0}, ex{0, 0};
    int dcnt = 0;
    for(int c0 = 0; c0 < nblk; c0 += DR_TPB) {
        const int q = q0 + c0 + t;
        const bool in = c0 + t < nblk;
        if(c0) drop_load(a, lr, q, in, pos);
        dcnt = drop_count(a, q, pos, s.nrm);
        if(nblk > DR_TPB && in) a.drop_cnt[q] = dcnt;
        const PoolMap m = pos.cap >= 0 ? PoolMap{(int64_t) pos.cap - dcnt, 0} : PoolMap{0, 0};
        PoolMap ctot;
        ex = block_exclusive_scan<PoolMap, MapOp, DR_NW>(m, MapOp(), PoolMap{0, 0}, s.sh, &ctot);
        tot = MapOp()(tot, ctot);
    }
    if(t == 0) {
        publish(state + 3 * (int64_t) g, tot.a);
        publish(state + 3 * (int64_t) g + 1, tot.b);
    }
    if(wv == 0) {
        const int64_t before = pool_before(state, g, pool0, a.err);
        if(t == 0) {
            const int64_t after = map_apply(tot, before);
            publish(state + 3 * (int64_t) g + 2, after);
            s.pool = before;
            if(g == lr.ngrp - 1) {
                int32_t* cout = a.carry + 4 * ((lr.level + 1) & 1);
                cout[0] = (int32_t) after;
                cout[1] = (int32_t) (lr.end_ix - after);
                cout[2] = (int32_t) (lr.end_val - after);
            }
        }
    }
    __syncthreads();
    // pools, grants, metadata and storage
    int64_t pool = s.pool;
    for(int c0 = 0; c0 < nblk; c0 += DR_TPB) {
        const int q = q0 + c0 + t;
        const bool in = c0 + t < nblk;
        if(nblk > DR_TPB) {
            drop_load(a, lr, q, in, pos);
            dcnt = in ? a.drop_cnt[q] : 0;
            const PoolMap m = pos.cap >= 0 ? PoolMap{(int64_t) pos.cap - dcnt, 0} : PoolMap{0, 0};
            PoolMap ctot;
            ex = block_exclusive_scan<PoolMap, MapOp, DR_NW>(m, MapOp(), PoolMap{0, 0}, s.sh,
                &ctot);
            tot = ctot;
        }
        const int64_t pl = map_apply(ex, pool);
        const int32_t px = (int32_t) (pos.col - pl), pv = (int32_t) (pos.val - pl);
        bool overflow = false, mine = false;
        int32_t room = 0;
        if(in) {
            BlockMeta& o = a.bout[pos.blk];
            o.col_ptr = px;
            o.val_ptr = pv;
            o.nnz = 0;
            if(pos.cap >= 0) {
                const int64_t e = (int64_t) dcnt - pos.cap;
                const int32_t gr = (int32_t) (e > 0 ? (e < pl ? e : pl) : 0);
                room = pos.cap + gr;
                overflow = dcnt > room;
                o.nnz = overflow ? room : dcnt;
                o.max_nnz = room;
                o.got_extra = gr;
                mine = pos.cnt <= LIST_GROUP;
            }
            if(!mine) {
                a.overflow[q] = overflow ? 1 : 0;
                a.store_list[atomicAdd(a.store_cnt + lr.level, 1)] = q;
            }
        }
        drop_store(a, q, pos, s.nrm, s.rflag, px, pv, mine, overflow, room);
        pool = map_apply(tot, pool);
    }
}

// final compacted storage (kernels :2011-2073, d_save_block :85-173), one
// wave per block
template<typename VT>
__device__ void store_one(const FactorArgs<VT>& a, const LevelRange& lr, int q, VT* nrm, VT* key,
    uint16_t* kix)
{
    const int lane = lane_id();
    const int b = a.lvlb_idx[lr.lo + q];
    const BlockMeta mo = a.bout[b];
    const int fr = a.bs[mo.block_row];
    const int h = a.bs[mo.block_row + 1] - fr;
    const int w = a.bs[mo.block_col + 1] - a.bs[mo.block_col];
    const VT* vals = a.if_val + (int64_t) q * 1024;
    VT* out_v = a.val_out + mo.val_ptr;
    if(mo.format == FMT_DENSE) {
        for(int e = lane; e < h * w; e += 64) out_v[e] = vals[e];
        if(lane == 0) a.row_mask[b] = ALL_ROWS;
        return;
    }
    const int32_t rflag = a.row_flag[mo.block_row];
    uint32_t rows = 0;
    bool bad = false;
    auto keep_mask = [&]() {
#pragma unroll
        for(int o = WAVE / 2; o > 0; o >>= 1) rows |= (uint32_t) __shfl_xor((int) rows, o, WAVE);
        const bool any_bad = wave_ballot(bad) != 0ull;
        if(lane == 0) a.row_mask[b] = store_row_mask(rows, any_bad, rflag);
    };
    const EntryList<VT> l = entry_list(a, q);
    int32_t* out_i = a.ix_out + mo.col_ptr;
    if(lane < h) nrm[lane] = drop_norm(a.rn[fr + lane]);
    wave_sync();
    const int cnt = a.if_cnt[q];
    if(!a.overflow[q]) {
        int base = 0;
        for(int e0 = 0; e0 < cnt; e0 += 64) {
            const int e = e0 + lane;
            bool k = false;
            VT v = 0;
            int ix = 0;
            if(e < cnt) {
                v = l.val(e);
                ix = l.idx(e);
                k = !(fabs(v) < a.threshold * nrm[ix >> 5]);
            }
            const uint64_t mask = wave_ballot(k);
            if(k) {
                const int pos = base + lanes_below(mask);
                out_i[pos] = (ix >> 5) * w + (ix & 31);
                out_v[pos] = v;
                rows |= 1u << (ix >> 5);
                bad = bad || !finite_value(v);
            }
            base += __popcll(mask);
        }
        keep_mask();
        return;
    }
    // over capacity: keep the max_nnz largest |v|, ties to the lower tile
    // index, written in that order (CUB BlockRadixSort descending, stable)
    for(int e = lane; e < cnt; e += 64) {
        const VT v = l.val(e);
        const int ix = l.idx(e);
        const bool k = !(fabs(v) < a.threshold * nrm[ix >> 5]);
        key[e] = k ? (VT) fabs(v) : (VT) -1;
        kix[e] = (uint16_t) ix;
    }
    wave_sync();
    for(int e = lane; e < cnt; e += 64) {
        const VT ke = key[e];
        if(ke < (VT) 0) continue;
        const int ie = kix[e];
        int rank = 0;
        for(int f = 0; f < cnt; ++f) {
            const VT kf = key[f];
            rank += (kf > ke) || (kf == ke && (int) kix[f] < ie);
        }
        if(rank < mo.max_nnz) {
            out_i[rank] = (ie >> 5) * w + (ie & 31);
            out_v[rank] = l.val(e);
            rows |= 1u << (ie >> 5);
            bad = bad || !finite_value(l.val(e));
        }
    }
    keep_mask();
}

// the positions k_drop leaves to the wave form, grid-stride
template<typename VT>
__device__ __forceinline__ void store_body(const FactorArgs<VT>& a, const LevelRange& lr,
    int bid_, int nblk_)
{
    __shared__ VT nrm[32];
    __shared__ VT key[1024];
    __shared__ uint16_t kix[1024];
    const int ns = a.store_cnt[lr.level];
    for(int t = bid_; t < ns; t += nblk_) {
        store_one(a, lr, a.store_list[t], nrm, key, kix);
        wave_sync();
    }
}

// Waves per SIMD the pivot, pair and one-wave off-diagonal kernels are compiled
// for at least: as many as their registers allow with few spills. With three, FP32
// spills too (k_offdiag 45 registers, bk_offdiag 18): refactor at n = 2,000 2.98
// ms, with two 2.86; a burst of 24 requests 44.0 and 41.5 ms.
constexpr int PP_WAVES = 2;

// the single-system kernels: the bodies at their own grid position
template<typename VT>
__global__ __launch_bounds__(64) void k_offdiag_general(FactorArgs<VT> a, LevelRange lr)
{
    offdiag_general_body<VT>(a, lr, blockIdx.x, gridDim.x);
}

template<typename VT>
__global__ __launch_bounds__(64, PP_WAVES) void k_offdiag(FactorArgs<VT> a, LevelRange lr)
{
    offdiag_body<VT>(a, lr, blockIdx.x, gridDim.x);
}

template<typename VT>
__global__ __launch_bounds__(TINY_TPB) void k_offdiag_tiny_scale(FactorArgs<VT> a, LevelRange lr)
{
    offdiag_tiny_scale_body<VT>(a, lr, blockIdx.x);
}

template<typename VT, int NW, bool TWO>
__global__ __launch_bounds__(64 * NW, PP_WAVES) void k_pivots_pairs(FactorArgs<VT> a, LevelRange lr)
{
    pivots_pairs_body<VT, NW, TWO>(a, lr, blockIdx.x);
}

template<typename VT>
__global__ __launch_bounds__(DR_TPB) void k_drop(FactorArgs<VT> a, LevelRange lr)
{
    drop_body<VT>(a, lr);
}

template<typename VT>
__global__ __launch_bounds__(64) void k_store(FactorArgs<VT> a, LevelRange lr)
{
    store_body<VT>(a, lr, blockIdx.x, gridDim.x);
}

// k_pivot_col_blocks (kernels :1352-1418) with d_col_pivot_block
// (:1290-1348): one wave per block row of the level; the stored blocks above
// its pivot block (earlier levels, final storage) take its pivoting order in
// their columns: sparse entries get new column indices in place, dense rows
// are gathered column by column.
template<typename VT>
__global__ __launch_bounds__(64) void k_pivot_cols(FactorArgs<VT> a, LevelRange lr)
{
    __shared__ int inv[32];
    const int lane = lane_id();
    const int i = a.lvl_rows[lr.row_lo + blockIdx.x];
    const int fr = a.bs[i];
    const int w = a.bs[i + 1] - fr;
    const int lp = (lane < w) ? a.perm[fr + lane] - fr : lane;
    if(lane < w) inv[lp] = lane;
    if(wave_ballot(lane < w && lp != lane) == 0) return;
    wave_sync();
    for(int ci = a.csc_off[i]; ci < a.csc_off[i + 1] - 1; ++ci) {
        const BlockMeta m = a.bout[a.csc_idx[ci]];
        if(m.format == FMT_SPARSE) {
            int32_t* ix = a.ix_out + m.col_ptr;
            for(int e = lane; e < m.nnz; e += 64) {
                const int v = ix[e];
                ix[e] = (v / w) * w + inv[v % w];
            }
        } else {
            const int h = a.bs[m.block_row + 1] - a.bs[m.block_row];
            VT* v = a.val_out + m.val_ptr;
            for(int r = 0; r < h; ++r) {
                const VT x = (lane < w) ? v[(int64_t) r * w + lp] : (VT) 0;
                wave_sync();
                if(lane < w) v[(int64_t) r * w + lane] = x;
                wave_sync();
            }
        }
    }
}

template<typename VT>
__global__ void k_zero_carry(int32_t* carry)
{
    if(threadIdx.x < 8) carry[threadIdx.x] = 0;
}

template<typename VT>
__global__ void k_gather(const double* vals, const int64_t* slot, int64_t nnz, VT* val_in)
{
    const int64_t q = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if(q < nnz && slot[q] >= 0) val_in[slot[q]] = (VT) vals[q];
}

template<typename VT>
__global__ void k_zero(VT* a, int64_t n)
{
    const int64_t q = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if(q < n) a[q] = (VT) 0;
}

// ---------------------------------------------------------------------------
// Batched refactor: one launch per step covers every listed system; item
// {s, q} is workgroup q of the single-system launch on system s (the same
// grid position and grid size, so the same results).

// factor_reset_pivots, the zeroing of gather_values and factor_begin
template<typename VT>
__global__ void bk_factor_begin(const FactorSys<VT>* fs, const int2* items)
{
    const int2 it = items[blockIdx.x];
    const FactorSys<VT>& F = fs[it.x];
    const FactorArgs<VT>& a = F.a;
    const int64_t g = (int64_t) it.y * 256 + threadIdx.x;
    if(g < a.n) {
        a.is_piv[g] = F.static_is_piv[g];
        a.perm[g] = (int32_t) g;
    }
    if(g < F.val_space) F.val_in[g] = (VT) 0;
    if(g < a.state_words) ((int32_t*) a.grp_state)[g] = 0;
    if(g < a.num_levels) {
        a.defer_cnt[g] = 0;
        a.wave_cnt[g] = 0;
        a.store_cnt[g] = 0;
    }
    if(it.y == 0 && threadIdx.x < 8) a.carry[threadIdx.x] = 0;
}

// the gather of gather_values
template<typename VT>
__global__ void bk_gather(const FactorSys<VT>* fs, const int2* items)
{
    const int2 it = items[blockIdx.x];
    const FactorSys<VT>& F = fs[it.x];
    const int64_t q = (int64_t) it.y * 256 + threadIdx.x;
    if(q < F.nnz && F.value_slot[q] >= 0) F.val_in[F.value_slot[q]] = (VT) F.vals[q];
}

template<typename VT, bool TWO>
__global__ __launch_bounds__(64, PP_WAVES) void bk_pivots_pairs(const FactorSys<VT>* fs, const int2* items,
    int32_t level)
{
    const int2 it = items[blockIdx.x];
    const FactorSys<VT>& F = fs[it.x];
    const LevelRange lr = F.lr[level];
    pivots_pairs_body<VT, 1, TWO>(F.a, lr, it.y);
}

template<typename VT>
__global__ __launch_bounds__(TINY_TPB) void bk_offdiag_tiny_scale(const FactorSys<VT>* fs,
    const int2* items, int32_t level)
{
    const int2 it = items[blockIdx.x];
    const FactorSys<VT>& F = fs[it.x];
    const LevelRange lr = F.lr[level];
    offdiag_tiny_scale_body<VT>(F.a, lr, it.y);
}

template<typename VT>
__global__ __launch_bounds__(64, PP_WAVES) void bk_offdiag(const FactorSys<VT>* fs, const int2* items,
    int32_t level)
{
    const int2 it = items[blockIdx.x];
    const FactorSys<VT>& F = fs[it.x];
    const LevelRange lr = F.lr[level];
    offdiag_body<VT>(F.a, lr, it.y, fl_grid_tasks(lr.size - lr.npiv, BATCH_TASK_GRID));
}

template<typename VT>
__global__ __launch_bounds__(64) void bk_offdiag_general(const FactorSys<VT>* fs,
    const int2* items, int32_t level)
{
    const int2 it = items[blockIdx.x];
    const FactorSys<VT>& F = fs[it.x];
    const LevelRange lr = F.lr[level];
    offdiag_general_body<VT>(F.a, lr, it.y, fl_grid_tasks(lr.size - lr.npiv, BATCH_TASK_GRID));
}

template<typename VT>
__global__ __launch_bounds__(DR_TPB) void bk_drop(const FactorSys<VT>* fs, const int2* items,
    int32_t level)
{
    const FactorSys<VT>& F = fs[items[blockIdx.x].x];
    const LevelRange lr = F.lr[level];
    drop_body<VT>(F.a, lr);
}

template<typename VT>
__global__ __launch_bounds__(64) void bk_store(const FactorSys<VT>* fs, const int2* items,
    int32_t level)
{
    const int2 it = items[blockIdx.x];
    const FactorSys<VT>& F = fs[it.x];
    const LevelRange lr = F.lr[level];
    store_body<VT>(F.a, lr, it.y, fl_grid_tasks(lr.size - lr.npiv, BATCH_TASK_GRID));
}

}  // namespace

__global__ void k_reset_pivots(int32_t n, const int32_t* sp, int32_t* is_piv, int32_t* perm)
{
    const int32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if(g < n) {
        is_piv[g] = sp[g];
        perm[g] = g;
    }
}

void factor_reset_pivots(int32_t n, const int32_t* static_is_piv, int32_t* is_piv, int32_t* perm,
    void* stream)
{
    if(n > 0)
        k_reset_pivots<<<(n + 255) / 256, 256, 0, (hipStream_t) stream>>>(n, static_is_piv, is_piv,
            perm);
}

template<typename VT>
void gather_values(const double* vals, const int64_t* slot, int64_t nnz, VT* val_in,
    int64_t val_space, void* stream)
{
    hipStream_t st = (hipStream_t) stream;
    if(val_space > 0) k_zero<VT><<<(unsigned) ((val_space + 255) / 256), 256, 0, st>>>(val_in, val_space);
    if(nnz > 0) k_gather<VT><<<(unsigned) ((nnz + 255) / 256), 256, 0, st>>>(vals, slot, nnz, val_in);
}

template<typename VT>
void factor_begin(const FactorArgs<VT>& a, void* stream)
{
    hipStream_t st = (hipStream_t) stream;
    k_zero_carry<VT><<<1, 64, 0, st>>>(a.carry);
    if(a.state_words > 0)
        k_zero<int32_t><<<(unsigned) ((a.state_words + 255) / 256), 256, 0, st>>>(
            (int32_t*) a.grp_state, a.state_words);
    if(a.num_levels > 0) {
        const unsigned g = (unsigned) ((a.num_levels + 255) / 256);
        k_zero<int32_t><<<g, 256, 0, st>>>(a.defer_cnt, a.num_levels);
        k_zero<int32_t><<<g, 256, 0, st>>>(a.wave_cnt, a.num_levels);
        k_zero<int32_t><<<g, 256, 0, st>>>(a.store_cnt, a.num_levels);
    }
}

template<typename VT>
void factor_level(const FactorArgs<VT>& a, const LevelRange& r, void* stream)
{
    hipStream_t st = (hipStream_t) stream;
    const int noff = r.size - r.npiv;
    const int tiny_blocks = fl_tiny_blocks(r);
    if(r.size > 0) {
        const bool four = r.piv_waves == 4;
        auto k = four ? (a.two ? k_pivots_pairs<VT, 4, true> : k_pivots_pairs<VT, 4, false>)
                      : (a.two ? k_pivots_pairs<VT, 1, true> : k_pivots_pairs<VT, 1, false>);
        k<<<fl_grid_pivots_pairs(r, r.piv_waves), 64 * r.piv_waves, 0, st>>>(a, r);
    }
    if(noff > 0) {
        const int grid = fl_grid_tasks(noff, 2048);
        k_offdiag_tiny_scale<VT><<<tiny_blocks, TINY_TPB, 0, st>>>(a, r);
        k_offdiag<VT><<<grid, 64, 0, st>>>(a, r);
        k_offdiag_general<VT><<<grid, 64, 0, st>>>(a, r);
    }
    if(a.pivoting && r.npiv > 0) k_pivot_cols<VT><<<r.npiv, 64, 0, st>>>(a, r);
    if(r.ngrp > 0) k_drop<VT><<<r.ngrp, DR_TPB, 0, st>>>(a, r);
    if(noff > 0) k_store<VT><<<fl_grid_tasks(noff, 2048), 64, 0, st>>>(a, r);
}

template void gather_values<double>(const double*, const int64_t*, int64_t, double*, int64_t, void*);
template void gather_values<float>(const double*, const int64_t*, int64_t, float*, int64_t, void*);
template void factor_begin<double>(const FactorArgs<double>&, void*);
template void factor_begin<float>(const FactorArgs<float>&, void*);
template void factor_level<double>(const FactorArgs<double>&, const LevelRange&, void*);
template void factor_level<float>(const FactorArgs<float>&, const LevelRange&, void*);


int64_t factor_batch_chunks(int32_t n, int64_t nnz, int64_t val_space, int32_t num_levels,
    int32_t state_words)
{
    int64_t m = std::max<int64_t>(std::max<int64_t>(n, nnz), std::max<int64_t>(val_space, 1));
    m = std::max<int64_t>(m, state_words);
    m = std::max<int64_t>(m, num_levels);
    return (m + 255) / 256;
}

template<typename VT>
void factor_batch_begin(const FactorSys<VT>* fs, FactorItems chunks, hipStream_t st)
{
    if(chunks.count <= 0) return;
    bk_factor_begin<VT><<<(unsigned) chunks.count, 256, 0, st>>>(fs, chunks.items);
    bk_gather<VT><<<(unsigned) chunks.count, 256, 0, st>>>(fs, chunks.items);
}

// the launches of factor_level, in its order, each over the level's items
// of every system that has the level
template<typename VT>
void factor_batch_level(const FactorSys<VT>* fs, const FactorBatchLevel& L, int32_t level,
    hipStream_t st)
{
    auto grid = [](const FactorItems& f) { return (unsigned) f.count; };
    if(L.pp.count) {
        auto k = L.two ? bk_pivots_pairs<VT, true> : bk_pivots_pairs<VT, false>;
        k<<<grid(L.pp), 64, 0, st>>>(fs, L.pp.items, level);
    }
    if(L.ts.count) bk_offdiag_tiny_scale<VT><<<grid(L.ts), TINY_TPB, 0, st>>>(fs, L.ts.items, level);
    if(L.off.count) {
        bk_offdiag<VT><<<grid(L.off), 64, 0, st>>>(fs, L.off.items, level);
        bk_offdiag_general<VT><<<grid(L.off), 64, 0, st>>>(fs, L.off.items, level);
    }
    if(L.dr.count) bk_drop<VT><<<grid(L.dr), DR_TPB, 0, st>>>(fs, L.dr.items, level);
    if(L.st.count) bk_store<VT><<<grid(L.st), 64, 0, st>>>(fs, L.st.items, level);
}

template void factor_batch_begin<double>(const FactorSys<double>*, FactorItems, hipStream_t);
template void factor_batch_begin<float>(const FactorSys<float>*, FactorItems, hipStream_t);
template void factor_batch_level<double>(const FactorSys<double>*, const FactorBatchLevel&, int32_t, hipStream_t);
template void factor_batch_level<float>(const FactorSys<float>*, const FactorBatchLevel&, int32_t, hipStream_t);

}  // namespace culip
