// Solve layout construction and level-scheduled block triangular solves.
//
// Reference: solve_U_block / solve_Ut_block (block_ildlt.impl.cuh:2378-2426,
// 2557-2606) with k_solve_blocks_offdiagonal_atomic / _diagonal_atomic
// (block_ildlt_kernels.impl.cuh:2354-2606): per level, x[rows] -= U_blk x
// for the level's off-diagonal blocks, then a 32-step substitution with the
// pivot block. Here the factor is first re-laid out per fine row (entries of
// a block row contiguous), the pivot blocks are inverted once, and each level
// is one launch: one wave per block row gathers its rows with coalesced loads
// and a segmented wave reduction (fixed order, no atomics), then applies
// U_ii^-1. k_solve_D follows helper_kernels.impl.cuh:720-772.
// Factor entries are read in their storage precision (FP32 for an FP32
// factor) and every product and sum runs in FP64: the preconditioner stays
// one fixed linear operator to FP64 rounding, which SQMR's short
// recurrences need (FP32 sums make it vary by ~1e-7 from apply to apply and
// cost the recurrence most of its progress below that level).
#include "solve.hpp"
#include "batch.hpp"
#include "wave.hpp"
#include <atomic>

#include <hip/hip_runtime.h>

namespace culip {

namespace {

// diag_inverse with every term added, also those with a zero of U (0 inf and
// 0 NaN are NaN); a tile without an entry beside its diagonal has none in X.
// For the tiles whose inverse may not be finite (ROW_UNBOUNDED).
template<typename VT>
__device__ __forceinline__ void diag_inverse_all_terms(const VT* U, int h, double* X, int hm)
{
    const int c = lane_id();
    bool beside = false;
    if(c < h)
#pragma unroll 1
        for(int k = c + 1; k < h; ++k) beside = beside || (U[c * h + k] != (VT) 0);
    const bool coupled = wave_ballot(beside) != 0ull;
#pragma unroll 1
    for(int r = hm - 1; r >= 0; --r) {
        double v = 0.0;
        if(r <= c && c < h) {
            const double d = (double) U[r * h + r];
            double s = 0.0;
#pragma unroll 1
            for(int k = r + 1; k <= c; ++k) s = fma((double) U[r * h + k], X[hm * k + c], s);
            v = (r == c) ? 1.0 / d : (coupled ? -s / d : 0.0);
        }
        if(c < hm) X[hm * r + c] = v;
    }
    wave_sync();
}

// columns of U_ii^-1 by back substitution, in double; X[r][c] at X[hm r + c]
// (hm x hm LDS, hm >= h: the largest block height of the launch). Lane c forms
// column c. U's rows come in with one round of loads, and only their nonzero
// entries are visited, ascending (the others would add exact zeros to a finite
// X).
template<typename VT>
__device__ void diag_inverse(const VT* U, int h, double* X, int hm)
{
    const int c = lane_id();
    VT u[32];   // U's column c
#pragma unroll
    for(int r = 0; r < 32; ++r) u[r] = (r < h && c < h) ? U[r * h + c] : (VT) 0;
#pragma unroll
    for(int r = 31; r >= 0; --r) {
        if(r < hm) {
            const double d = (double) wave_bcast(u[r], r);
            double s = 0.0;
            for(uint64_t m = wave_ballot(c > r && u[r] != (VT) 0); m; m &= m - 1) {
                const int k = __ffsll((long long) m) - 1;
                const double uk = (double) wave_bcast(u[r], k);
                if(k <= c && c < hm) s = fma(uk, X[hm * k + c], s);
            }
            if(c < hm) {
                double v = 0.0;
                if(c < h && r < h && r <= c) v = (r == c) ? 1.0 / d : -s / d;
                X[hm * r + c] = v;
            }
            wave_sync();
        }
    }
}

// up to 64 factored blocks staged one per lane: metadata, and the entries
// of sparse blocks with at most PLAN_E of them
constexpr int PLAN_E = 8;

template<typename VT>
struct PlanStage {
    int32_t fmt[64], nnz[64], cp[64], vp[64], off[64], ext[64];
    uint8_t small[64];
    uint8_t rr[64 * PLAN_E], cc[64 * PLAN_E];   // local row and column of each entry
    VT v[64 * PLAN_E];
};

// off / ext: first fine index and size of the block's other dimension; w:
// the block's width (the stride of its entry indices)
template<typename VT>
__device__ void plan_stage(PlanStage<VT>& sg, int k, const BlockMeta& m, int off, int ext, int w,
    const int32_t* ix_out, const VT* val_out)
{
    sg.fmt[k] = m.format;
    sg.nnz[k] = m.nnz;
    sg.cp[k] = m.col_ptr;
    sg.vp[k] = m.val_ptr;
    sg.off[k] = off;
    sg.ext[k] = ext;
    const bool sm = m.format == FMT_SPARSE && m.nnz <= PLAN_E;
    sg.small[k] = sm ? 1 : 0;
    if(sm)
        for(int e = 0; e < m.nnz; ++e) {
            const int q = ix_out[(int64_t) m.col_ptr + e];
            const int r = q / w;
            sg.rr[PLAN_E * k + e] = (uint8_t) r;
            sg.cc[PLAN_E * k + e] = (uint8_t) (q - r * w);
            sg.v[PLAN_E * k + e] = val_out[(int64_t) m.val_ptr + e];
        }
}

// true when every staged block of the round is small with at most one
// entry (nearly every off-diagonal block at level-0 fill): the round is then
// placed in parallel instead of walked block by block
template<typename VT>
__device__ __forceinline__ bool plan_one_entry_round(const PlanStage<VT>& sg, int nblk)
{
    const int lane = lane_id();
    const bool simple = lane >= nblk || (sg.small[lane] && sg.nnz[lane] <= 1);
    return wave_ballot(!simple) == 0;
}

// For a one-entry round: key = the local row (by_row) or column of lane k's
// entry (64: none), rank = entries of the same key on lower lanes (earlier
// blocks), and on lane r < ext the round's number of entries with key r.
template<typename VT>
__device__ __forceinline__ void plan_rank(const PlanStage<VT>& sg, int nblk, int ext, bool by_row,
    int& key, int& rank, int& add)
{
    const int lane = lane_id();
    const bool has = lane < nblk && sg.nnz[lane] == 1;
    key = has ? (by_row ? sg.rr[PLAN_E * lane] : sg.cc[PLAN_E * lane]) : 64;
    rank = 0;
    add = 0;
    for(int r = 0; r < ext; ++r) {
        const uint64_t m = wave_ballot(key == r);
        if(key == r) rank = lanes_below(m);
        if(lane == r) add = __popcll(m);
    }
}

// LDS of a plan_rows workgroup: the pivot block's inverse (hm x hm doubles, hm
// >= every block height of the launch), then the staged blocks in its place
template<typename VT>
inline size_t plan_rows_lds(int hm)
{
    const size_t x = sizeof(double) * (size_t) hm * (size_t) hm;
    return x > sizeof(PlanStage<VT>) ? x : sizeof(PlanStage<VT>);
}

template<typename VT, bool FILL>
__device__ __forceinline__ void plan_rows_body(const SolveTopo& t, const VT* val_out,
    const SolvePlan<VT>& p, int bid_, void* lds, int hm)
{
    const int lane = lane_id();
    const int i = bid_;
    const int fr = t.bs[i];
    const int h = t.bs[i + 1] - fr;
    // pivot block inverse rows (ui) and columns (ti)
    const int32_t flag = t.row_flag[i];
    if(flag == 0) {
        // U_ii is the identity (most pivot blocks of a sparse pattern): its
        // tile is not read
        if(lane < h) {
            if(FILL) {
                const int32_t wr = p.ui_ptr[fr + lane], wc = p.ti_ptr[fr + lane];
                p.ui_col[wr] = fr + lane; p.ui_val[wr] = (VT) 1; p.ui_lr[wr] = (uint8_t) lane;
                p.ti_col[wc] = fr + lane; p.ti_val[wc] = (VT) 1; p.ti_lr[wc] = (uint8_t) lane;
            } else {
                p.ui_ptr[fr + lane + 1] = 1;
                p.ti_ptr[fr + lane + 1] = 1;
            }
        }
    } else {
        double* X = (double*) lds;
        const BlockMeta dm = t.bout[t.csr_off[i]];
        if(flag & ROW_UNBOUNDED) diag_inverse_all_terms(val_out + dm.val_ptr, h, X, hm);
        else diag_inverse(val_out + dm.val_ptr, h, X, hm);
        if(lane < h) {
            int cr = 0, cc = 0;
            int32_t wr = 0, wc = 0;
            if(FILL) { wr = p.ui_ptr[fr + lane]; wc = p.ti_ptr[fr + lane]; }
            for(int c = 0; c < h; ++c) {
                const double v = X[hm * lane + c];  // row lane of U^-1
                if(v != 0.0) {
                    if(FILL) { p.ui_col[wr + cr] = fr + c; p.ui_val[wr + cr] = (VT) v; p.ui_lr[wr + cr] = (uint8_t) lane; }
                    ++cr;
                }
                const double u = X[hm * c + lane];  // column lane of U^-1
                if(u != 0.0) {
                    if(FILL) { p.ti_col[wc + cc] = fr + c; p.ti_val[wc + cc] = (VT) u; p.ti_lr[wc + cc] = (uint8_t) lane; }
                    ++cc;
                }
            }
            if(!FILL) { p.ui_ptr[fr + lane + 1] = cr; p.ti_ptr[fr + lane + 1] = cc; }
        }
    }
    // off-diagonal blocks of block row i (uo), by block id; 64 blocks at a
    // time are staged (metadata and small entry lists) one per lane, then
    // walked in order by the lanes of the fine rows
    PlanStage<VT>& sg = *(PlanStage<VT>*) lds;
    int cnt = 0;
    const int32_t base = (FILL && lane < h) ? p.uo_ptr[fr + lane] : 0;
    const int b0 = t.csr_off[i] + 1, b1 = t.csr_off[i + 1];
    for(int c0 = b0; c0 < b1; c0 += 64) {
        const int nblk = min(64, b1 - c0);
        wave_sync();
        if(lane < nblk) {
            const BlockMeta m = t.bout[c0 + lane];
            const int wb = t.bs[m.block_col + 1] - t.bs[m.block_col];
            plan_stage(sg, lane, m, t.bs[m.block_col], wb, wb, t.ix_out, val_out);
        }
        wave_sync();
        if(plan_one_entry_round(sg, nblk)) {
            // every staged block holds at most one entry: lane k places block
            // k's entry after the entries of its row from earlier blocks
            int key, rank, add;
            plan_rank(sg, nblk, h, true, key, rank, add);
            const int prev = __shfl(cnt, key & 63, 64);
            const int32_t rbase = __shfl(base, key & 63, 64);
            if(FILL && key < 64) {
                const int32_t pos = rbase + prev + rank;
                p.uo_col[pos] = sg.off[lane] + sg.cc[PLAN_E * lane];
                p.uo_val[pos] = sg.v[PLAN_E * lane];
                p.uo_lr[pos] = (uint8_t) key;
            }
            cnt += add;
            continue;
        }
        for(int k = 0; k < nblk; ++k) {
            const int fc = sg.off[k], w = sg.ext[k];
            if(sg.small[k]) {
                for(int e = 0; e < sg.nnz[k]; ++e) {
                    if(sg.rr[PLAN_E * k + e] == lane) {
                        if(FILL) { p.uo_col[base + cnt] = fc + sg.cc[PLAN_E * k + e]; p.uo_val[base + cnt] = sg.v[PLAN_E * k + e]; p.uo_lr[base + cnt] = (uint8_t) lane; }
                        ++cnt;
                    }
                }
            } else if(lane < h) {
                const VT* v = val_out + sg.vp[k];
                if(sg.fmt[k] == FMT_DENSE) {
                    for(int c = 0; c < w; ++c) {
                        const VT x = v[lane * w + c];
                        if(x != (VT) 0) {
                            if(FILL) { p.uo_col[base + cnt] = fc + c; p.uo_val[base + cnt] = x; p.uo_lr[base + cnt] = (uint8_t) lane; }
                            ++cnt;
                        }
                    }
                } else {
                    const int32_t* ix = t.ix_out + sg.cp[k];
                    for(int e = 0; e < sg.nnz[k]; ++e) {
                        const int q = ix[e];
                        const int r = q / w;
                        if(r == lane) {
                            if(FILL) { p.uo_col[base + cnt] = fc + (q - r * w); p.uo_val[base + cnt] = v[e]; p.uo_lr[base + cnt] = (uint8_t) lane; }
                            ++cnt;
                        }
                    }
                }
            }
        }
    }
    if(!FILL && lane < h) p.uo_ptr[fr + lane + 1] = cnt;
}

template<typename VT, bool FILL>
__global__ __launch_bounds__(64) void k_plan_rows(SolveTopo t, const VT* val_out, SolvePlan<VT> p)
{
    extern __shared__ double plan_x[];
    plan_rows_body<VT, FILL>(t, val_out, p, blockIdx.x, plan_x, 32);
}

template<typename VT, bool FILL>
__device__ __forceinline__ void plan_cols_body(const SolveTopo& t, const VT* val_out,
    const SolvePlan<VT>& p, int bid_)
{
    __shared__ PlanStage<VT> sg;
    const int lane = lane_id();
    const int j = bid_;
    const int fc = t.bs[j];
    const int w = t.bs[j + 1] - fc;
    int cnt = 0;
    const int32_t base = (FILL && lane < w) ? p.to_ptr[fc + lane] : 0;
    // blocks of column j above the diagonal, ascending block row, staged 64
    // at a time as in k_plan_rows
    const int q0 = t.csc_off[j], q1 = t.csc_off[j + 1] - 1;
    for(int c0 = q0; c0 < q1; c0 += 64) {
        const int nblk = min(64, q1 - c0);
        wave_sync();
        if(lane < nblk) {
            const BlockMeta m = t.bout[t.csc_idx[c0 + lane]];
            plan_stage(sg, lane, m, t.bs[m.block_row], t.bs[m.block_row + 1] - t.bs[m.block_row], w,
                t.ix_out, val_out);
        }
        wave_sync();
        if(plan_one_entry_round(sg, nblk)) {
            // as in k_plan_rows, by column
            int key, rank, add;
            plan_rank(sg, nblk, w, false, key, rank, add);
            const int prev = __shfl(cnt, key & 63, 64);
            const int32_t cbase = __shfl(base, key & 63, 64);
            if(FILL && key < 64) {
                const int32_t pos = cbase + prev + rank;
                p.to_col[pos] = sg.off[lane] + sg.rr[PLAN_E * lane];
                p.to_val[pos] = sg.v[PLAN_E * lane];
                p.to_lr[pos] = (uint8_t) key;
            }
            cnt += add;
            continue;
        }
        for(int k = 0; k < nblk; ++k) {
            const int fr = sg.off[k], h = sg.ext[k];
            if(sg.small[k]) {
                for(int e = 0; e < sg.nnz[k]; ++e) {
                    if(sg.cc[PLAN_E * k + e] == lane) {
                        if(FILL) { p.to_col[base + cnt] = fr + sg.rr[PLAN_E * k + e]; p.to_val[base + cnt] = sg.v[PLAN_E * k + e]; p.to_lr[base + cnt] = (uint8_t) lane; }
                        ++cnt;
                    }
                }
            } else if(lane < w) {
                const VT* v = val_out + sg.vp[k];
                if(sg.fmt[k] == FMT_DENSE) {
                    for(int r = 0; r < h; ++r) {
                        const VT x = v[r * w + lane];
                        if(x != (VT) 0) {
                            if(FILL) { p.to_col[base + cnt] = fr + r; p.to_val[base + cnt] = x; p.to_lr[base + cnt] = (uint8_t) lane; }
                            ++cnt;
                        }
                    }
                } else {
                    const int32_t* ix = t.ix_out + sg.cp[k];
                    for(int e = 0; e < sg.nnz[k]; ++e) {
                        const int qq = ix[e];
                        const int r = qq / w;
                        if(qq - r * w == lane) {
                            if(FILL) { p.to_col[base + cnt] = fr + r; p.to_val[base + cnt] = v[e]; p.to_lr[base + cnt] = (uint8_t) lane; }
                            ++cnt;
                        }
                    }
                }
            }
        }
    }
    if(!FILL && lane < w) p.to_ptr[fc + lane + 1] = cnt;
}

template<typename VT, bool FILL>
__global__ __launch_bounds__(64) void k_plan_cols(SolveTopo t, const VT* val_out, SolvePlan<VT> p)
{
    plan_cols_body<VT, FILL>(t, val_out, p, blockIdx.x);
}

// inclusive scan of a[1..n] in place (a[0] = 0), one workgroup, in chunks
// prefix sums of a[1..n] in place, in chunks of PS_TPB * PS_IPT entries:
// chunk totals first, then each chunk adds the totals before it
constexpr int PS_TPB = 256;
constexpr int PS_IPT = 8;
constexpr int PS_CHUNK = PS_TPB * PS_IPT;

struct ISum {
    int32_t s;
    __device__ static ISum shfl_up(const ISum& v, int o) { return {__shfl_up(v.s, o, WAVE)}; }
};
struct ISumOp {
    __device__ ISum operator()(const ISum& p, const ISum& q) const { return {p.s + q.s}; }
};

__device__ __forceinline__ void chunk_sums_body(const int32_t* a, int32_t n, int32_t* tmp, int bid_)
{
    __shared__ ISum sh[PS_TPB / WAVE];
    int32_t v = 0;
#pragma unroll
    for(int k = 0; k < PS_IPT; ++k) {
        const int64_t i = 1 + (int64_t) bid_ * PS_CHUNK + (int64_t) threadIdx.x * PS_IPT + k;
        if(i <= n) v += a[i];
    }
    ISum tot;
    (void) block_exclusive_scan<ISum, ISumOp, PS_TPB / WAVE>(ISum{v}, ISumOp(), ISum{0}, sh, &tot);
    if(threadIdx.x == 0) tmp[bid_] = tot.s;
}

__global__ __launch_bounds__(PS_TPB) void k_chunk_sums(const int32_t* a, int32_t n, int32_t* tmp)
{
    chunk_sums_body(a, n, tmp, blockIdx.x);
}

__device__ __forceinline__ void chunk_scan_body(int32_t* a, int32_t n, const int32_t* tmp,
    int32_t* total, int bid_, int nblk_)
{
    __shared__ ISum sh[PS_TPB / WAVE];
    const int c = bid_;
    // totals of the chunks before this one
    int32_t pre = 0;
    for(int q = threadIdx.x; q < c; q += PS_TPB) pre += tmp[q];
    ISum ptot;
    (void) block_exclusive_scan<ISum, ISumOp, PS_TPB / WAVE>(ISum{pre}, ISumOp(), ISum{0}, sh, &ptot);
    int32_t v[PS_IPT];
    int32_t s = 0;
    const int64_t i0 = 1 + (int64_t) c * PS_CHUNK + (int64_t) threadIdx.x * PS_IPT;
#pragma unroll
    for(int k = 0; k < PS_IPT; ++k) {
        v[k] = (i0 + k <= n) ? a[i0 + k] : 0;
        s += v[k];
    }
    ISum tot;
    const ISum ex = block_exclusive_scan<ISum, ISumOp, PS_TPB / WAVE>(ISum{s}, ISumOp(), ISum{0}, sh, &tot);
    int32_t run = ptot.s + ex.s;
#pragma unroll
    for(int k = 0; k < PS_IPT; ++k) {
        run += v[k];
        if(i0 + k <= n) a[i0 + k] = run;
    }
    if(threadIdx.x == 0) {
        if(c == 0) a[0] = 0;
        if(c == nblk_ - 1 && total) *total = ptot.s + tot.s;
    }
}

__global__ __launch_bounds__(PS_TPB) void k_chunk_scan(int32_t* a, int32_t n, const int32_t* tmp,
    int32_t* total)
{
    chunk_scan_body(a, n, tmp, total, blockIdx.x, gridDim.x);
}

// task descriptors of the block rows in level order, two int4 each:
// {fr, h, off-diagonal begin, end}, {inverse begin, end, 0, 0}
__device__ __forceinline__ void plan_tasks_body(int32_t nb, const int32_t* lvl_rows,
    const int32_t* bs, const int32_t* o_ptr, const int32_t* i_ptr, int4* task, int bid_)
{
    const int t = bid_ * blockDim.x + threadIdx.x;
    if(t >= nb) return;
    const int i = lvl_rows[t];
    const int fr = bs[i], h = bs[i + 1] - fr;
    task[2 * t] = make_int4(fr, h, o_ptr[fr], o_ptr[fr + h]);
    task[2 * t + 1] = make_int4(i_ptr[fr], i_ptr[fr + h], 0, 0);
}

__global__ void k_plan_tasks(int32_t nb, const int32_t* lvl_rows, const int32_t* bs,
    const int32_t* o_ptr, const int32_t* i_ptr, int4* task)
{
    plan_tasks_body(nb, lvl_rows, bs, o_ptr, i_ptr, task, blockIdx.x);
}

// res = U_ii^-1 y for one block row (y, res: LDS, res zeroed; all lanes
// active), from the
// row-ordered entries ib..ie of U_ii^-1; ic0 / iv0 / il0: this lane's entry
// of the first 64. Returns res[lane] (lanes < h). A diagonal U_ii^-1 (one
// entry per row, on the diagonal) is applied lane by lane; the
// general form sums each row's products by segmented scans. Both give
// 0 + (products in row order), the same bits.
template<typename VT>
__device__ __forceinline__ double apply_inverse(int fr, int h, int ib, int ie, int ic0, VT iv0,
    int il0, const int32_t* i_col, const VT* i_val, const uint8_t* i_lr, const double* y,
    double* res)
{
    const int lane = lane_id();
    if(ie - ib == h && wave_ballot(lane < h && (il0 != lane || ic0 != fr + lane)) == 0)
        return (lane < h) ? fma((double) iv0, y[lane], 0.0) : 0.0;
    const bool in0 = ib + lane < ie;
    int icol = in0 ? ic0 : fr;
    VT ival = in0 ? iv0 : (VT) 0;
    int isg = in0 ? il0 : 64;
    for(int e0 = ib; e0 < ie; e0 += 64) {
        if(e0 != ib) {
            const int e = e0 + lane;
            isg = 64;
            if(e < ie) { icol = i_col[e]; ival = i_val[e]; isg = i_lr[e]; }
        }
        double p = seg_scan_runs_fma((isg < 64) ? (double) ival : 0.0, y[icol - fr], isg);
        const int nsg = next_lane(isg, -1);
        if(isg < 64 && (lane == 63 || nsg != isg)) res[isg] += p;
        wave_sync();
    }
    return (lane < h) ? res[lane] : 0.0;
}

constexpr int TRSV_PF = 4;   // 64-entry chunks whose loads are issued together

// one level: one wave per block row; y = x_i - sum(off-diag) ; x_i = Uinv y.
// All entry loads of up to TRSV_PF chunks are issued before the x gathers;
// the chunks' segmented sums are then applied to y in chunk order.
// One block row of U x = b: x_i = U_ii^-1 (b_i - sum_j U_ij x_j) with FP64
// sums, the off-diagonal products summed in entry order by segmented scans
// over 64-entry chunks, then the rows of U_ii^-1. Every load that does not
// depend on another block row's result is issued before the first wait (b_i,
// the first 64 entries of U_ii^-1, the first off-diagonal chunk and, once its
// columns are in, its gathers of x), so a level costs two dependent memory
// round trips.
template<typename VT>
__device__ __forceinline__ void block_row_solve(int4 t0, int4 t1, bool offdiag,
    const int32_t* o_col, const VT* o_val, const uint8_t* o_lr, const int32_t* i_col,
    const VT* i_val, const uint8_t* i_lr, const double* b, const double* xsrc, double* xout,
    double* y, double* res)
{
    const int lane = lane_id();
    const int fr = t0.x, h = t0.y, ob = t0.z, oe = offdiag ? t0.w : t0.z, ib = t1.x, ie = t1.y;
    // loads run from clamped (in-range) indices without branches, and the
    // lanes past the end are masked afterwards, so the compiler issues them
    // all before the first wait
    const double bo_raw = b[fr + min(lane, h - 1)];
    const double bo = (lane < h) ? bo_raw : 0.0;
    // the first 64 entries of U_ii^-1 (every block row has at least its
    // diagonal there), selected only where they are used
    const int ei = ib + min(lane, max(ie - ib - 1, 0));
    const int ic0 = i_col[ei];
    const VT iv0 = i_val[ei];
    const int il0 = i_lr[ei];
    int c[TRSV_PF], sg[TRSV_PF];
    VT v[TRSV_PF];
    double xv[TRSV_PF];
    auto load = [&](int e0) {
        int cr[TRSV_PF], sr[TRSV_PF];
        VT vr[TRSV_PF];
#pragma unroll
        for(int k = 0; k < TRSV_PF; ++k) {
            const int e = min(e0 + 64 * k + lane, oe - 1);
            cr[k] = o_col[e];
            vr[k] = o_val[e];
            sr[k] = o_lr[e];
        }
        double xr[TRSV_PF];
#pragma unroll
        for(int k = 0; k < TRSV_PF; ++k) xr[k] = xsrc[cr[k]];
#pragma unroll
        for(int k = 0; k < TRSV_PF; ++k) {
            const bool in = e0 + 64 * k + lane < oe;
            c[k] = in ? cr[k] : 0;
            v[k] = in ? vr[k] : (VT) 0;
            sg[k] = in ? sr[k] : 64;
            xv[k] = in ? xr[k] : 0.0;
        }
    };
    if(ob < oe) load(ob);
    if(lane < h) { y[lane] = bo; res[lane] = 0; }
    for(int e0 = ob; e0 < oe; e0 += 64 * TRSV_PF) {
        if(e0 != ob) load(e0);
        wave_sync();
#pragma unroll
        for(int k = 0; k < TRSV_PF; ++k) {
            if(e0 + 64 * k >= oe) break;
            double p = seg_scan_runs_fma((double) v[k], xv[k], sg[k]);
            const int nsg = next_lane(sg[k], -1);
            if(sg[k] < 64 && (lane == 63 || nsg != sg[k])) y[sg[k]] -= p;
            wave_sync();
        }
    }
    wave_sync();
    // every lane takes part (the general form scans across the wave)
    const double r = apply_inverse<VT>(fr, h, ib, ie, ic0, iv0, il0, i_col, i_val, i_lr, y, res);
    if(lane < h) xout[fr + lane] = r;
}

template<typename VT>
__global__ __launch_bounds__(64) void k_trsv_level(const int4* task, const int32_t* o_col,
    const VT* o_val, const uint8_t* o_lr, const int32_t* i_col, const VT* i_val,
    const uint8_t* i_lr, double* x)
{
    __shared__ double y[33];     // FP64 accumulation for both factor precisions
    __shared__ double res[33];
    block_row_solve<VT>(task[2 * blockIdx.x], task[2 * blockIdx.x + 1], true, o_col, o_val,
        o_lr, i_col, i_val, i_lr, x, x, x, y, res);
}

// One block-Jacobi sweep over all block rows (solve_U_jacobi /
// solve_Ut_jacobi, block_ildlt.impl.cuh:2454-2493, 2637-2676, with
// k_solve_block_stripe_level): x_out_i = U_ii^-1 (b_i - sum_j U_ij x_in_j).
// x_in == nullptr is the first sweep from x_0 = 0. The per-row sums run in
// the same order as in k_trsv_level, so once x_in is the exact solution the
// sweep reproduces the level-scheduled solve bit for bit.
template<typename VT>
__global__ __launch_bounds__(64) void k_jacobi_sweep(const int4* task, const int32_t* o_col,
    const VT* o_val, const uint8_t* o_lr, const int32_t* i_col, const VT* i_val,
    const uint8_t* i_lr, const double* b, const double* xin, double* xout)
{
    __shared__ double y[33];
    __shared__ double res[33];
    block_row_solve<VT>(task[2 * blockIdx.x], task[2 * blockIdx.x + 1], xin != nullptr, o_col,
        o_val, o_lr, i_col, i_val, i_lr, b, xin, xout, y, res);
}

// Whole triangular solve in one launch of G resident waves:
// wave g takes the block rows at processing indices g, g + G, g + 2G, ... of
// the level order (reverse level order for the U solve), so every block row
// it depends on has a smaller index. The lowest unfinished index always has
// its inputs published and every wave is resident, so the solve drains.
// Results are published value by value: before the solve every entry of pub
// holds CHAIN_EMPTY, a signalling NaN that no arithmetic produces, and a
// block row writes its x values there with 8-byte agent-coherent stores (the
// L2 of each XCD is separate). A reader loads the values it needs with
// agent-coherent loads and takes each one once it differs from CHAIN_EMPTY,
// reloading the missing ones until all are there; no flag and no
// store-completion wait sits between a producer and its readers. While a
// block row waits and computes, the wave already loads the task and first
// entries of its next one. Each wave also presets its rows of next_pub, the
// buffer of the next single-launch solve. Every wait is bounded: past
// spin_limit polls the wave records an error in *err, and the block row and
// all that depend on it become NaN.
constexpr unsigned long long CHAIN_EMPTY = 0x7ff4c0de5eed1234ull;

__device__ __forceinline__ double pub_load(const double* p)
{
    return __hip_atomic_load(const_cast<double*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ bool published(double v)
{
    return (unsigned long long) __double_as_longlong(v) != CHAIN_EMPTY;
}

// waits until every lane's value xv[k] (column c[k]) is published; rdy[k]
// on entry: xv[k] already usable. What is missing when it gives up stays
// CHAIN_EMPTY, a NaN.
__device__ void wait_published(const double* pub, const int (&c)[TRSV_PF], double (&xv)[TRSV_PF],
    bool (&rdy)[TRSV_PF], int32_t* err, int32_t spin_limit, int& spins)
{
    bool all = true;
#pragma unroll
    for(int k = 0; k < TRSV_PF; ++k) all = all && rdy[k];
    while(wave_ballot(!all)) {
        __builtin_amdgcn_s_sleep(1);
        if(++spins > spin_limit) {
            // err is pinned host memory: the host reads it without a copy
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return;
        }
        all = true;
#pragma unroll
        for(int k = 0; k < TRSV_PF; ++k) {
            if(!rdy[k]) {
                xv[k] = pub_load(pub + c[k]);
                rdy[k] = published(xv[k]);
            }
            all = all && rdy[k];
        }
    }
}

// One group of up to TRSV_PF 64-entry chunks of a block row's off-diagonal
// entries: columns, values and local rows (64: no entry).
template<typename VT>
struct ChainGroup {
    int c[TRSV_PF], sg[TRSV_PF];
    VT v[TRSV_PF];
};

// what a block row loads before it can wait: its first group (clamped in
// range), its own right-hand side and the first 64 entries of U_ii^-1
template<typename VT>
struct ChainHead {
    ChainGroup<VT> g;
    double bo;
    int ic, il;
    VT iv;
};

// The segmented sums over a chunk as far as they follow from its local rows
// alone, formed while the x values are on their way, in one register: how many
// lanes of this lane's 16-lane row before it belong to its segment, whether the
// segment reaches into the rows before (scan steps over lanes 15 and 31), and
// on lane r < 32 the lane that ends row r's segment (-1: no entry of the row).
struct ScanPlan {
    int bits;
    __device__ __forceinline__ int dist() const { return bits & 15; }
    __device__ __forceinline__ bool cross15() const { return (bits & 16) != 0; }
    __device__ __forceinline__ bool cross31() const { return (bits & 32) != 0; }
    __device__ __forceinline__ int end() const { return bits >> 8; }
};

__device__ __forceinline__ ScanPlan scan_plan(int sg, int8_t* ends)
{
    int lane = lane_id();
    // what follows from the lane alone is formed here, not held over the loop
    asm volatile("" : "+v"(lane));
    const int before = dpp_move<0x138, 0xf>(-1, sg);   // every lane active
    const uint64_t heads = wave_ballot(before != sg) | 1ull;
    // the first lane of this lane's segment
    const int start = 63 - __clzll((long long) (heads & (~0ull >> (63 - lane))));
    int bits = min(lane - start, lane & 15);
    if((lane & 16) != 0 && start < (lane & ~15)) bits |= 16;
    if(lane >= 32 && start < 32) bits |= 32;
    const int nsg = next_lane(sg, -1);
    wave_sync();
    if(lane < 32) ends[lane] = -1;
    wave_sync();
    if(sg < 64 && (lane == 63 || nsg != sg)) ends[sg] = (int8_t) lane;
    wave_sync();
    return ScanPlan{bits | (int) ends[lane & 31] * 256};
}

// a lane move whose result is used only where the lane has a source
template<int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_take(double v)
{
    const int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(__builtin_amdgcn_mov_dpp(hi, CTRL, ROW_MASK, 0xf, false),
        __builtin_amdgcn_mov_dpp(lo, CTRL, ROW_MASK, 0xf, false));
}

// seg_scan_runs_fma(a, x, .) with the plan of its local rows: the same tree
// and roundings
__device__ __forceinline__ double planned_scan(double a, double x, const ScanPlan& p)
{
    double v = a * x;
    const double f = fma(a, x, dpp_take<0x111, 0xf>(v));
    const int dist = p.dist();
    v = dist >= 1 ? f : v;
    double s = v + dpp_take<0x112, 0xf>(v);
    v = dist >= 2 ? s : v;
    s = v + dpp_take<0x114, 0xf>(v);
    v = dist >= 4 ? s : v;
    s = v + dpp_take<0x118, 0xf>(v);
    v = dist >= 8 ? s : v;
    s = v + dpp_take<0x142, 0xa>(v);
    v = p.cross15() ? s : v;
    s = v + dpp_take<0x143, 0xc>(v);
    return p.cross31() ? s : v;
}

// Reloads the x values (byte offsets off[k]) of the lanes set in m[k], all in
// one round trip. One block with its own wait: written as loads under
// conditions, the compiler waits for each before it issues the next.
__device__ __forceinline__ void reload_missing(const double* pub, const uint32_t (&off)[TRSV_PF],
    const uint64_t (&m)[TRSV_PF], double (&xv)[TRSV_PF])
{
    static_assert(TRSV_PF == 4, "four chunks");
    uint64_t saved;
    asm volatile("s_mov_b64 %[sv], exec\n\t"
                 "s_mov_b64 exec, %[m0]\n\t"
                 "global_load_dwordx2 %[x0], %[o0], %[pub] sc1\n\t"
                 "s_mov_b64 exec, %[m1]\n\t"
                 "global_load_dwordx2 %[x1], %[o1], %[pub] sc1\n\t"
                 "s_mov_b64 exec, %[m2]\n\t"
                 "global_load_dwordx2 %[x2], %[o2], %[pub] sc1\n\t"
                 "s_mov_b64 exec, %[m3]\n\t"
                 "global_load_dwordx2 %[x3], %[o3], %[pub] sc1\n\t"
                 "s_mov_b64 exec, %[sv]\n\t"
                 "s_waitcnt vmcnt(0)"
                 : [x0] "+&v"(xv[0]), [x1] "+&v"(xv[1]), [x2] "+&v"(xv[2]), [x3] "+&v"(xv[3]),
                 [sv] "=&s"(saved)
                 : [m0] "s"(m[0]), [m1] "s"(m[1]), [m2] "s"(m[2]), [m3] "s"(m[3]), [o0] "v"(off[0]),
                 [o1] "v"(off[1]), [o2] "v"(off[2]), [o3] "v"(off[3]), [pub] "s"(pub)
                 : "memory");
}

// waits until all x values of a group are there; what is missing when it gives
// up stays CHAIN_EMPTY, a NaN
__device__ __forceinline__ void wait_group(const double* pub, const uint32_t (&off)[TRSV_PF],
    const int (&sg)[TRSV_PF], double (&xv)[TRSV_PF], int32_t* err, int32_t spin_limit, int& spins)
{
    for(;;) {
        uint64_t m[TRSV_PF], any = 0;
#pragma unroll
        for(int k = 0; k < TRSV_PF; ++k) {
            m[k] = wave_ballot(sg[k] < 64 && !published(xv[k]));
            any |= m[k];
        }
        if(any == 0) return;
        if(++spins > spin_limit) {
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return;
        }
        __builtin_amdgcn_s_sleep(1);
        reload_missing(pub, off, m, xv);
    }
}

// y (lane r: row r) minus the row sums of a group, chunk after chunk. A
// chunk is scanned as soon as its values are there, while the others are
// still on their way: the latest values of a block row all belong to the
// levels next to its own, so they sit in one chunk (the last for U', the first
// for U) and only that chunk's scan follows the last arrival. off: the byte
// offsets of the values in pub; chunks: how many of the group have entries;
// their values past the row's end are cleared. xv[k] becomes chunk k's sum.
// NaN when the wait gives up, so that no partial sum is taken for a solution.
template<typename VT>
__device__ __forceinline__ double chain_sums(const double* pub, const uint32_t (&off)[TRSV_PF],
    const VT (&a)[TRSV_PF], const int (&sg)[TRSV_PF], double (&xv)[TRSV_PF],
    const ScanPlan (&p)[TRSV_PF], int chunks, double y, int32_t* err, int32_t spin_limit,
    int& spins)
{
    uint32_t open = chunks >= TRSV_PF ? (1u << TRSV_PF) - 1 : (1u << chunks) - 1;
    for(;;) {
        uint64_t m[TRSV_PF];
#pragma unroll
        for(int k = 0; k < TRSV_PF; ++k) {
            m[k] = 0;
            if((open >> k) & 1u) {
                m[k] = wave_ballot(sg[k] < 64 && !published(xv[k]));
                if(m[k] == 0) {
                    const double v = planned_scan((double) a[k], sg[k] < 64 ? xv[k] : 0.0, p[k]);
                    xv[k] = __shfl(v, max(p[k].end(), 0), WAVE);
                    open &= ~(1u << k);
                }
            }
        }
        if(open == 0) break;
        if(++spins > spin_limit) {
            // err is pinned host memory: the host reads it without a copy
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            // a quiet NaN, which readers of the row take as published
            return __longlong_as_double(0x7ff8000000000000ll);
        }
        __builtin_amdgcn_s_sleep(1);
        reload_missing(pub, off, m, xv);
    }
#pragma unroll
    for(int k = 0; k < TRSV_PF; ++k)
        if(k < chunks) y = p[k].end() >= 0 ? y - xv[k] : y;
    return y;
}

// The right-hand side of one block row as K src (rows fr .. fr + h - 1 of a
// CSR matrix), formed exactly as k_csr_spmv forms those rows: eight lanes
// per row, lane sub summing entries s + sub, s + sub + 8, ... by fma in that
// order, then the xor tree over the eight lanes. Four rounds of eight rows
// issue their loads together. Returns row fr + lane's value (lanes < h).
struct CsrRhs {
    const int32_t* rp;
    const int32_t* ci;
    const double* cv;
    const double* src;
};

// RHS_U: entries per lane and row whose loads go together (the same sums for any)
template<int RHS_U>
__device__ double block_rhs(const CsrRhs& k, int fr, int h)
{
    int lane = lane_id();
    asm volatile("" : "+v"(lane));
    const int sub = lane & 7, g = lane >> 3;
    int s[4], e[4];
#pragma unroll
    for(int r = 0; r < 4; ++r) {
        const int row = fr + min(8 * r + g, h - 1);
        s[r] = k.rp[row];
        e[r] = k.rp[row + 1];
    }
    double acc[4];
#pragma unroll
    for(int r = 0; r < 4; ++r) acc[r] = 0.0;
    for(int q0 = sub;; q0 += 8 * RHS_U) {
        int c[4][RHS_U];
        double v[4][RHS_U], xv[4][RHS_U];
#pragma unroll
        for(int r = 0; r < 4; ++r)
#pragma unroll
            for(int u = 0; u < RHS_U; ++u) {
                const int q = max(min(s[r] + q0 + 8 * u, e[r] - 1), 0);
                const int cq = k.ci[q];
                c[r][u] = (s[r] + q0 + 8 * u < e[r]) ? cq : 0;
                v[r][u] = k.cv[q];
            }
#pragma unroll
        for(int r = 0; r < 4; ++r)
#pragma unroll
            for(int u = 0; u < RHS_U; ++u) xv[r][u] = k.src[c[r][u]];
        bool more = false;
#pragma unroll
        for(int r = 0; r < 4; ++r) {
#pragma unroll
            for(int u = 0; u < RHS_U; ++u)
                if(s[r] + q0 + 8 * u < e[r]) acc[r] = fma(v[r][u], xv[r][u], acc[r]);
            more = more || s[r] + q0 + 8 * RHS_U < e[r];
        }
        if(wave_ballot(more) == 0) break;
    }
    double mine = 0.0;
#pragma unroll
    for(int r = 0; r < 4; ++r) {
        double a = acc[r];
#pragma unroll
        for(int o = 4; o > 0; o >>= 1) a += __shfl_xor(a, o, 8);
        const double row_val = 1.0 * a;          // y = alpha (A x), alpha = 1
        const double got = __shfl(row_val, 8 * (lane & 7), 64);
        if((lane >> 3) == r) mine = got;
    }
    return mine;
}

template<typename VT>
__device__ __forceinline__ void chain_group(int e0, int oe, const int32_t* o_col, const VT* o_val,
    const uint8_t* o_lr, ChainGroup<VT>& g)
{
#pragma unroll
    for(int k = 0; k < TRSV_PF; ++k) {
        const int e = max(min(e0 + 64 * k + lane_id(), oe - 1), 0);
        g.c[k] = o_col[e];
        g.v[k] = o_val[e];
        g.sg[k] = o_lr[e];
    }
}

template<typename VT>
__device__ __forceinline__ void chain_fetch(int4 t0, int4 t1, const int32_t* o_col, const VT* o_val,
    const uint8_t* o_lr, const int32_t* i_col, const VT* i_val, const uint8_t* i_lr,
    const double* x, bool rhs_fused, ChainHead<VT>& f)
{
    const int lane = lane_id();
    const int fr = t0.x, h = t0.y, ib = t1.x, ie = t1.y;
    chain_group<VT>(t0.z, t0.w, o_col, o_val, o_lr, f.g);
    // this block row's own right-hand side: no other wave writes x (with a
    // fused product it is formed after the current block row instead)
    f.bo = rhs_fused ? 0.0 : x[fr + min(lane, h - 1)];
    const int ei = ib + min(lane, max(ie - ib - 1, 0));
    f.ic = i_col[ei];
    f.iv = i_val[ei];
    f.il = i_lr[ei];
}

// Two forms with the same values (chain_form). Walked: a row's groups one after
// the other, each awaited as a whole, the chunks summed into LDS. Planned:
// between the arrival of a block row's last x value and the store of its results
// lies the part of every level that no other wave hides, so of a row of one
// group all that does not depend on x is done before (ScanPlan), the chunks that
// are complete are summed while the last one is awaited, and rows are summed by
// lane reads instead of LDS updates; rows of more groups are summed as in the
// walked form (their values are mostly there, and plans only cost: 13.4 ms
// instead of 11.1 for a factor with fill of n = 10,000); U_ii^-1 of up to 64
// entries stays in registers. Measured (publish to arrival / arrival to publish,
// per level, n = 400,000): 0.9-1.1 us / 0.5-0.6 us; a lone pair of waves on two
// XCDs exchanges a value in 0.4-0.5 us.
template<typename VT, bool FUSED, bool PLANNED>
__global__ __launch_bounds__(64, 4) void k_trsv_chain(const int4* task, int32_t nb, int32_t reverse,
    const int32_t* o_col, const VT* o_val, const uint8_t* o_lr, const int32_t* i_col,
    const VT* i_val, const uint8_t* i_lr, double* pub, double* next_pub, int32_t* err,
    int32_t spin_limit, double* x, CsrRhs rhs)
{
    __shared__ double y_lds[33];     // FP64 accumulation for both factor precisions
    __shared__ double res[33];
    __shared__ int8_t ends[32];
    const int lane = lane_id();
    const int G = gridDim.x;
    constexpr bool fused = FUSED;
    const double empty = __longlong_as_double((long long) CHAIN_EMPTY);
    auto task_at = [&](int w, int4& a, int4& b) {
        const int q = min(w, nb - 1);
        const int pos = reverse ? (nb - 1 - q) : q;
        a = task[2 * pos];
        b = task[2 * pos + 1];
    };
    int spins = 0;
    int w = blockIdx.x;
    int4 t0, t1;
    task_at(w, t0, t1);
    ChainHead<VT> cur;
    chain_fetch<VT>(t0, t1, o_col, o_val, o_lr, i_col, i_val, i_lr, x, fused, cur);
    if(fused) cur.bo = block_rhs<3>(rhs, t0.x, t0.y);
    constexpr int RHS_U = PLANNED ? 2 : 3;   // beside the loop's registers
    for(;;) {
        int4 n0, n1;
        task_at(w + G, n0, n1);
        ChainHead<VT> nxt;
        const int fr = t0.x, h = t0.y, ob = t0.z, oe = t0.w, ib = t1.x, ie = t1.y;
        if(lane < h) next_pub[fr + lane] = empty;
        double r;
        if(PLANNED) {
            // U_ii^-1: diagonal (one entry per row, on the diagonal), or up to
            // 64 entries taken by one planned scan, or in chunks of 64
            const bool diagonal = ie - ib == h &&
                wave_ballot(lane < h && (cur.il != lane || cur.ic != fr + lane)) == 0;
            const bool one_chunk = ie - ib <= 64;
            double y = cur.bo;
            ScanPlan ip;
            if(!diagonal && one_chunk) ip = scan_plan(ib + lane < ie ? cur.il : 64, ends);
            double xv[TRSV_PF];
            uint32_t off[TRSV_PF];
            if(ob < oe)
#pragma unroll
                for(int k = 0; k < TRSV_PF; ++k) {
                    off[k] = 8u * (uint32_t) cur.g.c[k];
                    xv[k] = pub_load((const double*) ((const char*) pub + off[k]));
                }
#pragma unroll
            for(int k = 0; k < TRSV_PF; ++k) {
                const bool in = ob + 64 * k + lane < oe;
                cur.g.v[k] = in ? cur.g.v[k] : (VT) 0;
                cur.g.sg[k] = in ? cur.g.sg[k] : 64;
            }
            // the next loads go out here: they are younger than the reads
            // above, so a row whose values are all there does not wait for them
            if(w + G < nb)
                chain_fetch<VT>(n0, n1, o_col, o_val, o_lr, i_col, i_val, i_lr, x, fused, nxt);
            if(oe - ob > 64 * TRSV_PF) {
                // several groups: awaited as a whole and summed into LDS
                wave_sync();
                if(lane < h) y_lds[lane] = y;
                wave_sync();
#pragma unroll 1
                for(int e0 = ob;;) {
                    wait_group(pub, off, cur.g.sg, xv, err, spin_limit, spins);
#pragma unroll
                    for(int k = 0; k < TRSV_PF; ++k) {
                        if(e0 + 64 * k >= oe) break;
                        const int sg = cur.g.sg[k];
                        const double q = seg_scan_runs_fma((double) cur.g.v[k],
                            sg < 64 ? xv[k] : 0.0, sg);
                        const int nsg = next_lane(sg, -1);
                        if(sg < 64 && (lane == 63 || nsg != sg)) y_lds[sg] -= q;
                        wave_sync();
                    }
                    e0 += 64 * TRSV_PF;
                    if(e0 >= oe) break;
                    chain_group<VT>(e0, oe, o_col, o_val, o_lr, cur.g);
#pragma unroll
                    for(int k = 0; k < TRSV_PF; ++k) {
                        off[k] = 8u * (uint32_t) cur.g.c[k];
                        xv[k] = pub_load((const double*) ((const char*) pub + off[k]));
                    }
#pragma unroll
                    for(int k = 0; k < TRSV_PF; ++k) {
                        const bool in = e0 + 64 * k + lane < oe;
                        cur.g.v[k] = in ? cur.g.v[k] : (VT) 0;
                        cur.g.sg[k] = in ? cur.g.sg[k] : 64;
                    }
                }
                y = y_lds[min(lane, 32)];
            } else if(ob < oe) {
                ScanPlan plan[TRSV_PF];
                const int chunks = (oe - ob + 63) / 64;
                plan[0] = scan_plan(cur.g.sg[0], ends);
                if(chunks > 1) plan[1] = scan_plan(cur.g.sg[1], ends);
                if(chunks > 2) plan[2] = scan_plan(cur.g.sg[2], ends);
                if(chunks > 3) plan[3] = scan_plan(cur.g.sg[3], ends);
                y = chain_sums<VT>(pub, off, cur.g.v, cur.g.sg, xv, plan, chunks, y, err, spin_limit,
                    spins);
            }
            if(diagonal) {
                r = fma((double) cur.iv, y, 0.0);
            } else if(one_chunk) {
                const bool in = ib + lane < ie;
                const double yy = __shfl(y, in ? cur.ic - fr : 0, WAVE);
                const double v = planned_scan(in ? (double) cur.iv : 0.0, yy, ip);
                r = 0.0 + __shfl(v, max(ip.end(), 0), WAVE);
                r = ip.end() >= 0 ? r : 0.0;
            } else {
                wave_sync();
                if(lane < h) { y_lds[lane] = y; res[lane] = 0; }
                wave_sync();
                r = apply_inverse<VT>(fr, h, ib, ie, cur.ic, cur.iv, cur.il, i_col, i_val, i_lr,
                    y_lds, res);
            }
        } else {
            wave_sync();
            if(lane < h) { y_lds[lane] = cur.bo; res[lane] = 0; }
            ChainGroup<VT> g = cur.g;
            bool fetched = false;
            for(int e0 = ob; e0 < oe; e0 += 64 * TRSV_PF) {
                if(e0 != ob) chain_group<VT>(e0, oe, o_col, o_val, o_lr, g);
                double xv[TRSV_PF];
                bool rdy[TRSV_PF];
#pragma unroll
                for(int k = 0; k < TRSV_PF; ++k) xv[k] = pub_load(pub + g.c[k]);
#pragma unroll
                for(int k = 0; k < TRSV_PF; ++k) {
                    const bool in = e0 + 64 * k + lane < oe;
                    g.v[k] = in ? g.v[k] : (VT) 0;
                    g.sg[k] = in ? g.sg[k] : 64;
                    rdy[k] = !in || published(xv[k]);
                }
                wait_published(pub, g.c, xv, rdy, err, spin_limit, spins);
                if(!fetched) {
                    chain_fetch<VT>(n0, n1, o_col, o_val, o_lr, i_col, i_val, i_lr, x, fused, nxt);
                    fetched = true;
                }
                wave_sync();
#pragma unroll
                for(int k = 0; k < TRSV_PF; ++k) {
                    if(e0 + 64 * k >= oe) break;
                    const double p = seg_scan_runs_fma((double) g.v[k], g.sg[k] < 64 ? xv[k] : 0.0,
                        g.sg[k]);
                    const int nsg = next_lane(g.sg[k], -1);
                    if(g.sg[k] < 64 && (lane == 63 || nsg != g.sg[k])) y_lds[g.sg[k]] -= p;
                    wave_sync();
                }
            }
            if(!fetched)
                chain_fetch<VT>(n0, n1, o_col, o_val, o_lr, i_col, i_val, i_lr, x, fused, nxt);
            wave_sync();
            r = apply_inverse<VT>(fr, h, ib, ie, cur.ic, cur.iv, cur.il, i_col, i_val, i_lr, y_lds,
                res);
        }
        if(lane < h) {
            __hip_atomic_store(pub + fr + lane, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            x[fr + lane] = r;
        }
        w += G;
        if(w >= nb) break;
        // the next block row's K src: its loads overlap the wait for its
        // inputs, which rarely have all arrived by now
        if(fused) nxt.bo = block_rhs<RHS_U>(rhs, n0.x, n0.y);
        t0 = n0;
        t1 = n1;
        cur = nxt;
    }
}

// The first block-Jacobi sweep with b = K src: each block row forms its rows
// of K src as block_rhs does (the values k_csr_spmv gives), keeps them in b
// for the later sweeps and solves from x_0 = 0 as k_jacobi_sweep does.
template<typename VT>
__global__ __launch_bounds__(64) void k_jacobi_first_product(const int4* task,
    const int32_t* o_col, const VT* o_val, const uint8_t* o_lr, const int32_t* i_col,
    const VT* i_val, const uint8_t* i_lr, CsrRhs rhs, double* b, double* xout)
{
    __shared__ double y[33];
    __shared__ double res[33];
    const int4 t0 = task[2 * blockIdx.x];
    const double bo = block_rhs<3>(rhs, t0.x, t0.y);
    // each lane reads back only the row it wrote (lanes >= h are masked)
    if(lane_id() < t0.y) b[t0.x + lane_id()] = bo;
    block_row_solve<VT>(t0, task[2 * blockIdx.x + 1], false, o_col, o_val, o_lr, i_col, i_val,
        i_lr, b, nullptr, xout, y, res);
}

// Batched block-Jacobi sweeps. Item {s, c} is block rows JACOBI_ROWS c ..
// JACOBI_ROWS c + JACOBI_ROWS - 1 of system s, one after the other in one
// wave; each block row is computed exactly as block_row_solve computes it
// (the workgroup of k_jacobi_sweep for that block row): the same masked
// 64-entry chunks, segmented sums in chunk order and U_ii^-1 rows. What a
// block row reads before its first wait (its first chunk, the x values of
// that chunk, its b and its first 64 entries of U_ii^-1) is loaded while the
// block row before it computes; the task records of all the item's block
// rows come in with one load. tr selects the layout (0 the U solve, 1 the
// U' solve). b may be the output vector itself: a block row reads its own
// rows of b before it writes its own rows of the output, and no other block
// row reads them.
constexpr int JACOBI_ROWS = JACOBI_BATCH_ROWS;

template<typename VT>
struct JacobiHead {
    int c, sg;
    VT v;
    double xv;
    double bo;
    int ic, il;
    VT iv;
};

// The item's block rows two at a time, lanes 0-31 one and lanes 32-63 the
// next, for block rows of at most 64 entries (one chunk). A chunk's first 32
// entries are scanned by the half's lanes, where the steps within 16 lanes and
// over lane 15 are the same as in a chunk of its own; where some block row of
// the item has more (wide), the other 32 are scanned the same way, and the
// step over lane 31 is the sum of the first half's last lane, added where the
// segment goes on: the chunk's tree. A sweep over small blocks is bound by
// instructions, not by bytes (about 300 per block row; 28 of a chunk's 64 lanes
// are in use at a block height of 8). All loads of the item (two passes) go
// out together. 256 systems of 1,000-40,000 primal rows: 91.2 us per sweep one block
// row at a time, 67.5 us so. offdiag: the item has an off-diagonal entry, so
// o_col may be read at the clamped places. y64, res64: 64 doubles of LDS each.
template<typename VT>
__device__ __forceinline__ void jacobi_pairs(int4 tk, int cnt, bool offdiag, bool wide,
    const int32_t* o_col,
    const VT* o_val, const uint8_t* o_lr, const int32_t* i_col, const VT* i_val,
    const uint8_t* i_lr, const double* b, const double* xsrc, double* xout, double* y64,
    double* res64)
{
    constexpr int PASSES = JACOBI_BATCH_ROWS / 2;
    const int lane = lane_id(), l = lane & 31, half = lane & 32;
    int fr[PASSES], h[PASSES], sg[PASSES], ic[PASSES], il[PASSES], ni[PASSES], c[PASSES];
    int sg2[PASSES], c2[PASSES];
    VT v[PASSES], v2[PASSES], iv[PASSES];
    double bo[PASSES], xv[PASSES], xv2[PASSES];
#pragma unroll
    for(int q = 0; q < PASSES; ++q) {
        const int j = 2 * q + (lane >> 5);
        const int jc = min(j, cnt - 1);
        fr[q] = __shfl(tk.x, 2 * jc);
        h[q] = j < cnt ? __shfl(tk.y, 2 * jc) : 0;
        const int hc = max(__shfl(tk.y, 2 * jc), 1);
        const int ob = __shfl(tk.z, 2 * jc), ow = __shfl(tk.w, 2 * jc);
        const int oe = offdiag && j < cnt ? ow : ob;
        const int ib = __shfl(tk.x, 2 * jc + 1), ie = __shfl(tk.y, 2 * jc + 1);
        ni[q] = j < cnt ? ie - ib : 0;
        bo[q] = b[fr[q] + min(l, hc - 1)];
        const int ei = ib + min(l, max(ie - ib - 1, 0));
        ic[q] = i_col[ei];
        iv[q] = i_val[ei];
        il[q] = i_lr[ei];
        c[q] = 0;
        v[q] = (VT) 0;
        sg[q] = 64;
        if(offdiag) {
            const int e = max(min(ob + l, oe - 1), 0);
            c[q] = o_col[e];
            const VT vr = o_val[e];
            const int sr = o_lr[e];
            if(ob + l < oe) {
                v[q] = vr;
                sg[q] = sr;
            }
        }
        c2[q] = 0;
        v2[q] = (VT) 0;
        sg2[q] = 64;
        if(wide) {
            const int e = max(min(ob + 32 + l, oe - 1), 0);
            c2[q] = o_col[e];
            const VT vr = o_val[e];
            const int sr = o_lr[e];
            if(ob + 32 + l < oe) {
                v2[q] = vr;
                sg2[q] = sr;
            }
        }
    }
#pragma unroll
    for(int q = 0; q < PASSES; ++q) {
        xv[q] = offdiag && sg[q] < 64 ? xsrc[c[q]] : 0.0;
        xv2[q] = wide && sg2[q] < 64 ? xsrc[c2[q]] : 0.0;
    }
#pragma unroll
    for(int q = 0; q < PASSES; ++q) {
        if(2 * q >= cnt) break;
        double y = l < h[q] ? bo[q] : 0.0;
        y64[lane] = y;
        wave_sync();
        if(offdiag) {
            // distinct segments in the two halves
            const int seg = sg[q] < 64 ? sg[q] + half : 64;
            const double p = seg_scan_runs_fma((double) v[q], xv[q], half ? seg + 64 : seg);
            int nsg = next_lane(seg, -1);
            if(wide) {
                const int seg2 = sg2[q] < 64 ? sg2[q] + half : 64;
                double p2 = seg_scan_runs_fma((double) v2[q], xv2[q], half ? seg2 + 64 : seg2);
                const double last = __shfl(p, half + 31);
                const int seg31 = __shfl(seg, half + 31);
                if(seg2 < 64 && seg31 == seg2) p2 = p2 + last;
                const int first2 = __shfl(seg2, half);
                if(l == 31) nsg = first2;
                if(seg < 64 && nsg != seg) y64[seg] -= p;
                const int nsg2 = next_lane(seg2, -1);
                wave_sync();
                if(seg2 < 64 && (l == 31 || nsg2 != seg2)) y64[seg2] -= p2;
            } else if(seg < 64 && (l == 31 || nsg != seg)) {
                y64[seg] -= p;
            }
            wave_sync();
            y = y64[lane];
        }
        // U_ii^-1: one entry per row on the diagonal in both block rows, or
        // one scan over the entries of both
        double r;
        if(wave_ballot(l < h[q] && (ni[q] != h[q] || il[q] != l || ic[q] != fr[q] + l)) == 0ull) {
            r = fma((double) iv[q], y, 0.0);
        } else {
            const bool in = l < ni[q];
            const int seg = in ? il[q] + half : 64;
            res64[lane] = 0.0;
            const double yv = y64[in ? half + ic[q] - fr[q] : lane];
            const double p = seg_scan_runs_fma(in ? (double) iv[q] : 0.0, yv, half ? seg + 64 : seg);
            const int nsg = next_lane(seg, -1);
            wave_sync();
            if(seg < 64 && (l == 31 || nsg != seg)) res64[seg] += p;
            wave_sync();
            r = res64[lane];
        }
        if(l < h[q]) xout[fr[q] + l] = r;
        wave_sync();
    }
}

template<typename VT>
__global__ __launch_bounds__(64) void bk_jacobi_sweep(const int2* items, const BatchSys* sys,
    int32_t tr, int32_t b_id, int32_t in, int32_t out)
{
    __shared__ double y64[64], res64[64];
    double* y = y64;
    double* res = res64;
    const int lane = lane_id();
    const int2 it = items[blockIdx.x];
    if(it.x < 0) return;   // a hole of an XCD-aware list
    const BatchSys& S = sys[it.x];
    const int4* task = S.task[tr];
    const int32_t* o_col = S.o_col[tr];
    const VT* o_val = (const VT*) S.o_val[tr];
    const uint8_t* o_lr = S.o_lr[tr];
    const int32_t* i_col = S.i_col[tr];
    const VT* i_val = (const VT*) S.i_val[tr];
    const uint8_t* i_lr = S.i_lr[tr];
    const double* xsrc = in == BV_NONE ? nullptr : batch_vec(S, in);
    const double* b = batch_vec(S, b_id);
    double* xout = batch_vec(S, out);
    const bool offdiag = xsrc != nullptr;
    const int r0 = it.y * JACOBI_ROWS;
    const int cnt = min(JACOBI_ROWS, S.nb - r0);
    // lane 2 j holds block row r0 + j's first task record, lane 2 j + 1 its
    // second
    const int4 tk = task[2 * r0 + min(lane, 2 * cnt - 1)];
    auto rec = [&](int j, int4& t0, int4& t1) {
        t0.x = __shfl(tk.x, 2 * j);
        t0.y = __shfl(tk.y, 2 * j);
        t0.z = __shfl(tk.z, 2 * j);
        t0.w = __shfl(tk.w, 2 * j);
        t1.x = __shfl(tk.x, 2 * j + 1);
        t1.y = __shfl(tk.y, 2 * j + 1);
    };
    // the loads of block row j that do not depend on other rows' results
    auto head = [&](int j, JacobiHead<VT>& H) {
        int4 t0, t1;
        rec(j, t0, t1);
        const int fr = t0.x, h = t0.y, ob = t0.z, oe = offdiag ? t0.w : t0.z;
        const int ib = t1.x, ie = t1.y;
        H.bo = b[fr + min(lane, h - 1)];
        const int ei = ib + min(lane, max(ie - ib - 1, 0));
        H.ic = i_col[ei];
        H.iv = i_val[ei];
        H.il = i_lr[ei];
        H.c = 0;
        H.v = (VT) 0;
        H.sg = 64;
        if(ob < oe) {
            const int e = min(ob + lane, oe - 1);
            H.c = o_col[e];
            H.v = o_val[e];
            H.sg = o_lr[e];
        }
    };
    auto gather = [&](int j, JacobiHead<VT>& H) {
        int4 t0, t1;
        rec(j, t0, t1);
        const int ob = t0.z, oe = offdiag ? t0.w : t0.z;
        H.xv = 0.0;
        if(ob < oe) {
            const double xr = xsrc[H.c];
            const bool in0 = ob + lane < oe;
            H.c = in0 ? H.c : 0;
            H.v = in0 ? H.v : (VT) 0;
            H.sg = in0 ? H.sg : 64;
            H.xv = in0 ? xr : 0.0;
        }
    };
    auto apply_chunk = [&](int c, VT v, int sg, double xv) {
        (void) c;
        const double p = seg_scan_runs_fma((double) v, xv, sg);
        const int nsg = next_lane(sg, -1);
        if(sg < 64 && (lane == 63 || nsg != sg)) y[sg] -= p;
        wave_sync();
    };
    auto compute = [&](int j, const JacobiHead<VT>& H) {
        int4 t0, t1;
        rec(j, t0, t1);
        const int fr = t0.x, h = t0.y, ob = t0.z, oe = offdiag ? t0.w : t0.z;
        const int ib = t1.x, ie = t1.y;
        const double bo = (lane < h) ? H.bo : 0.0;
        if(lane < h) { y[lane] = bo; res[lane] = 0; }
        wave_sync();
        if(ob < oe) {
            apply_chunk(H.c, H.v, H.sg, H.xv);
            for(int e0 = ob + 64; e0 < oe; e0 += 64) {
                const int e = min(e0 + lane, oe - 1);
                const int cr = o_col[e];
                const VT vr = o_val[e];
                const int sr = o_lr[e];
                const double xr = xsrc[cr];
                const bool in0 = e0 + lane < oe;
                apply_chunk(in0 ? cr : 0, in0 ? vr : (VT) 0, in0 ? sr : 64, in0 ? xr : 0.0);
            }
        }
        wave_sync();
        const double r = apply_inverse<VT>(fr, h, ib, ie, H.ic, H.iv, H.il, i_col, i_val, i_lr,
            y, res);
        if(lane < h) xout[fr + lane] = r;
        wave_sync();
    };
    // two block rows per pass where every block row of the item has at most
    // 64 entries off the diagonal and 32 in U_ii^-1
    const int off_cnt = offdiag ? tk.w - tk.z : 0, inv_cnt = __shfl(tk.y - tk.x, lane | 1);
    const bool mine = lane < 2 * cnt && (lane & 1) == 0;
    if(wave_ballot(mine && (off_cnt > 64 || inv_cnt > 32)) == 0ull) {
        const bool some = wave_ballot(mine && off_cnt > 0) != 0ull;
        const bool wide = wave_ballot(mine && off_cnt > 32) != 0ull;
        jacobi_pairs<VT>(tk, cnt, some, wide, o_col, o_val, o_lr, i_col, i_val, i_lr, b, xsrc,
            xout, y64, res64);
        return;
    }
    JacobiHead<VT> A, B;
    head(0, A);
    gather(0, A);
    for(int j = 0; j < cnt; j += 2) {
        if(j + 1 < cnt) head(j + 1, B);
        compute(j, A);
        if(j + 1 >= cnt) break;
        gather(j + 1, B);
        if(j + 2 < cnt) head(j + 2, A);
        compute(j + 1, B);
        if(j + 2 < cnt) gather(j + 2, A);
    }
}

// Batched layout build: item {s, q} is workgroup q of the single-system
// launch on system s.
template<typename VT, bool FILL>
__global__ __launch_bounds__(64) void bk_plan_rows(const PlanSys<VT>* ps, const int2* items,
    int32_t hm)
{
    extern __shared__ double plan_x[];
    const int2 it = items[blockIdx.x];
    const PlanSys<VT>& P = ps[it.x];
    plan_rows_body<VT, FILL>(P.t, P.val_out, P.p, it.y, plan_x, hm);
}

template<typename VT, bool FILL>
__global__ __launch_bounds__(64) void bk_plan_cols(const PlanSys<VT>* ps, const int2* items)
{
    const int2 it = items[blockIdx.x];
    const PlanSys<VT>& P = ps[it.x];
    plan_cols_body<VT, FILL>(P.t, P.val_out, P.p, it.y);
}

template<typename VT>
__device__ __forceinline__ int32_t* plan_ptr(const SolvePlan<VT>& p, int q)
{
    return q == 0 ? p.uo_ptr : q == 1 ? p.ui_ptr : q == 2 ? p.to_ptr : p.ti_ptr;
}

template<typename VT>
__global__ __launch_bounds__(PS_TPB) void bk_chunk_sums(const PlanSys<VT>* ps, const int2* items,
    int32_t q)
{
    const int2 it = items[blockIdx.x];
    const PlanSys<VT>& P = ps[it.x];
    chunk_sums_body(plan_ptr(P.p, q), P.t.n, P.scan_tmp, it.y);
}

template<typename VT>
__global__ __launch_bounds__(PS_TPB) void bk_chunk_scan(const PlanSys<VT>* ps, const int2* items,
    int32_t q)
{
    const int2 it = items[blockIdx.x];
    const PlanSys<VT>& P = ps[it.x];
    chunk_scan_body(plan_ptr(P.p, q), P.t.n, P.scan_tmp, P.totals + q, it.y,
        (P.t.n + PS_CHUNK - 1) / PS_CHUNK);
}

template<typename VT>
__global__ void bk_plan_tasks(const PlanSys<VT>* ps, const int2* items, int32_t transpose)
{
    const int2 it = items[blockIdx.x];
    const PlanSys<VT>& P = ps[it.x];
    if(transpose)
        plan_tasks_body(P.t.nb, P.t.lvl_rows, P.t.bs, P.p.to_ptr, P.p.ti_ptr, P.p.task_t, it.y);
    else
        plan_tasks_body(P.t.nb, P.t.lvl_rows, P.t.bs, P.p.uo_ptr, P.p.ui_ptr, P.p.task_u, it.y);
}

__global__ void k_fill_bits(double* p, int64_t n, unsigned long long bits)
{
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if(i < n) p[i] = __longlong_as_double((long long) bits);
}

__global__ void k_solve_D(int32_t n, const double* tri, const int32_t* is_piv, const double* b,
    double* x)
{
    const int32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if(g >= n) return;
    const int this_piv = is_piv[g];
    const int next_piv = (g < n - 1) ? is_piv[g + 1] : 1;
    const double p11 = tri[3 * (int64_t) g + 1];
    const double p12 = tri[3 * (int64_t) g + 2];
    const double p22 = !next_piv ? tri[3 * (int64_t) (g + 1) + 1] : 1.0;
    const double r1 = b[g];
    const double r2 = (g < n - 1) ? b[g + 1] : 0.0;
    const double gr = sqrt(fma(p11, p11, p12 * p12));
    const double c = p11 / gr, s = p12 / gr;
    double g1 = fma(c, r1, s * r2);
    double g2 = fma(-s, r1, c * r2);
    const double t12 = fma(c, p12, s * p22);
    const double t22 = fma(-s, p12, c * p22);
    g2 = g2 / t22;
    g1 = fma(-t12, g2, g1) / gr;
    if(this_piv) x[g] = g1;
    if(!next_piv) x[g + 1] = g2;
}

}  // namespace

template<typename VT>
void solve_plan_count(const SolveTopo& t, const VT* val_out, VT*, SolvePlan<VT>& p, void* stream)
{
    hipStream_t st = (hipStream_t) stream;
    k_plan_rows<VT, false><<<t.nb, 64, plan_rows_lds<VT>(32), st>>>(t, val_out, p);
    k_plan_cols<VT, false><<<t.nb, 64, 0, st>>>(t, val_out, p);
}

template<typename VT>
void solve_plan_fill(const SolveTopo& t, const VT* val_out, const VT*, SolvePlan<VT>& p,
    void* stream)
{
    hipStream_t st = (hipStream_t) stream;
    k_plan_rows<VT, true><<<t.nb, 64, plan_rows_lds<VT>(32), st>>>(t, val_out, p);
    k_plan_cols<VT, true><<<t.nb, 64, 0, st>>>(t, val_out, p);
    const unsigned g = (unsigned) ((t.nb + 255) / 256);
    k_plan_tasks<<<g, 256, 0, st>>>(t.nb, t.lvl_rows, t.bs, p.uo_ptr, p.ui_ptr, p.task_u);
    k_plan_tasks<<<g, 256, 0, st>>>(t.nb, t.lvl_rows, t.bs, p.to_ptr, p.ti_ptr, p.task_t);
}

size_t scan_tmp_ints(int32_t n) { return (size_t) ((n + PS_CHUNK - 1) / PS_CHUNK) + 1; }

void scan_counts(int32_t* ptr, int32_t n, int32_t* total_dev, int32_t* tmp, void* stream)
{
    hipStream_t st = (hipStream_t) stream;
    const unsigned nch = (unsigned) ((n + PS_CHUNK - 1) / PS_CHUNK);
    if(nch == 0) {
        k_chunk_scan<<<1, PS_TPB, 0, st>>>(ptr, n, tmp, total_dev);
        return;
    }
    k_chunk_sums<<<nch, PS_TPB, 0, st>>>(ptr, n, tmp);
    k_chunk_scan<<<nch, PS_TPB, 0, st>>>(ptr, n, tmp, total_dev);
}

template<typename VT>
void trsv_upper(const SolveTopo& t, const SolvePlan<VT>& p, double* x, void* stream)
{
    hipStream_t st = (hipStream_t) stream;
    for(int l = t.num_levels - 1; l >= 0; --l) {
        const int lo = t.lvl_off_h[l], cnt = t.lvl_off_h[l + 1] - lo;
        if(cnt > 0)
            k_trsv_level<VT><<<cnt, 64, 0, st>>>(p.task_u + 2 * lo, p.uo_col, p.uo_val, p.uo_lr,
                p.ui_col, p.ui_val, p.ui_lr, x);
    }
}

template<typename VT>
void trsv_upper_t(const SolveTopo& t, const SolvePlan<VT>& p, double* x, void* stream)
{
    hipStream_t st = (hipStream_t) stream;
    for(int l = 0; l < t.num_levels; ++l) {
        const int lo = t.lvl_off_h[l], cnt = t.lvl_off_h[l + 1] - lo;
        if(cnt > 0)
            k_trsv_level<VT><<<cnt, 64, 0, st>>>(p.task_t + 2 * lo, p.to_col, p.to_val, p.to_lr,
                p.ti_col, p.ti_val, p.ti_lr, x);
    }
}

__global__ void k_perm_pull(int32_t n, const int32_t* perm, const double* in, double* out)
{
    const int32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if(g < n) out[g] = in[perm[g]];
}

__global__ void k_perm_push(int32_t n, const int32_t* perm, const double* in, double* out)
{
    const int32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if(g < n) out[perm[g]] = in[g];
}

void permute_pull(int32_t n, const int32_t* perm, const double* in, double* out, void* stream)
{
    if(n > 0) k_perm_pull<<<(n + 255) / 256, 256, 0, (hipStream_t) stream>>>(n, perm, in, out);
}

void permute_push(int32_t n, const int32_t* perm, const double* in, double* out, void* stream)
{
    if(n > 0) k_perm_push<<<(n + 255) / 256, 256, 0, (hipStream_t) stream>>>(n, perm, in, out);
}

void solve_D(int32_t n, const double* tri, const int32_t* is_piv, const double* b, double* x,
    void* stream)
{
    k_solve_D<<<(n + 255) / 256, 256, 0, (hipStream_t) stream>>>(n, tri, is_piv, b, x);
}

template void solve_plan_count<double>(const SolveTopo&, const double*, double*, SolvePlan<double>&, void*);
template void solve_plan_count<float>(const SolveTopo&, const float*, float*, SolvePlan<float>&, void*);
template void solve_plan_fill<double>(const SolveTopo&, const double*, const double*, SolvePlan<double>&, void*);
template void solve_plan_fill<float>(const SolveTopo&, const float*, const float*, SolvePlan<float>&, void*);
// Waves of k_trsv_chain per CU at most. A solve needs all of its waves resident.
// TRSV_SINGLE_MAX_CONCURRENT = 4 such solves, of any instances, have to fit on
// the GPU at the same time (other kernels end on their own): all are compiled
// for 16 waves per CU (at most 128 registers), a quarter of them each.
constexpr int CHAIN_WAVES_PER_CU = 4;

template<typename VT>
using ChainKernel = void (*)(const int4*, int32_t, int32_t, const int32_t*, const VT*,
    const uint8_t*, const int32_t*, const VT*, const uint8_t*, double*, double*, int32_t*, int32_t,
    double*, CsrRhs);

template<typename VT>
ChainKernel<VT> chain_kernel(bool fused, bool planned)
{
    if(fused) return planned ? k_trsv_chain<VT, true, true> : k_trsv_chain<VT, true, false>;
    return planned ? k_trsv_chain<VT, false, true> : k_trsv_chain<VT, false, false>;
}

// CUs of the current device and waves per CU a solve may have: as many as let
// TRSV_SINGLE_MAX_CONCURRENT solves of any instance fit (queried once per device)
struct ChainRoom {
    int cus, per_cu;
};

template<typename VT>
ChainRoom chain_room()
{
    // both numbers in one word, since threads may get here at the same time
    static std::atomic<int> room[64] = {};
    int dev = 0;
    if(hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return {};
    int r = room[dev].load(std::memory_order_relaxed);
    if(r == 0) {
        hipDeviceProp_t pr;
        if(hipGetDeviceProperties(&pr, dev) != hipSuccess) return {};
        int per = CHAIN_WAVES_PER_CU;
        for(int k = 0; k < 4; ++k) {
            int o = 0;
            if(hipOccupancyMaxActiveBlocksPerMultiprocessor(&o,
                    chain_kernel<VT>((k & 1) != 0, (k & 2) != 0), 64, 0) != hipSuccess)
                return {};
            per = min(per, o / TRSV_SINGLE_MAX_CONCURRENT);
        }
        r = 8 * pr.multiProcessorCount + max(1, per);
        room[dev].store(r, std::memory_order_relaxed);
    }
    return {r / 8, r % 8};
}

// The form of a solve by its block rows per level. Few (up to 3 in 2 CUs): the
// levels' latency counts, the planned form, with three waves per CU up to one
// row in 2 CUs, since more waves only poll. Many: the waves are busy with rows
// whose values are there, and the walked form takes less time for each. us, U'
// / U / U' with K src on 256 CUs, rows per level: planned 3, planned 4, walked
//   36 (n = 40,000, blocks of 32)      82 /  96 /  80    86 /  98 /  84    91 / 111 /  91
//   262 (n = 300,000, blocks of 32)    95 / 106 / 119    93 / 107 / 111   104 / 122 / 121
//   365 (n = 100,000, blocks of 16)    45 /  44 /  54    44 /  43 /  48    44 /  45 /  48
//   437 (n = 40,000, blocks of 8)      34 /  33 /  38    32 /  32 /  35    32 /  32 /  33
//   3,090 (n = 300,000, blocks of 8)  131 / 122 / 249   106 /  99 / 196    89 /  82 / 187
struct ChainForm {
    bool planned;
    int per_cu;
};

inline ChainForm chain_form(const SolveTopo& t, int cus)
{
    const int64_t rows2 = 2 * (int64_t) t.nb, levels = t.num_levels;
    // the planned form reaches values by 32-bit byte offsets
    if(rows2 > 3 * levels * cus || t.n >= (1 << 29)) return {false, CHAIN_WAVES_PER_CU};
    return {true, rows2 <= levels * cus ? 3 : CHAIN_WAVES_PER_CU};
}

template<typename VT>
hipError_t trsv_chain(const int4* task, int32_t reverse, const int32_t* o_col, const VT* o_val,
    const uint8_t* o_lr, const int32_t* i_col, const VT* i_val, const uint8_t* i_lr, double* pub,
    double* next_pub, const SolveTopo& t, double* x, CsrRhs rhs, hipStream_t st)
{
    const ChainRoom room = chain_room<VT>();
    if(room.cus <= 0) return hipErrorInvalidConfiguration;
    const ChainForm form = chain_form(t, room.cus);
    const int g = min(room.cus * min(form.per_cu, room.per_cu), (int) t.nb);
    chain_kernel<VT>(rhs.rp != nullptr, form.planned)<<<g, 64, 0, st>>>(task, t.nb, reverse, o_col,
        o_val, o_lr, i_col, i_val, i_lr, pub, next_pub, t.err, t.spin_limit, x, rhs);
    return hipGetLastError();
}

template<typename VT>
int trsv_upper_single(const SolveTopo& t, const SolvePlan<VT>& p, double* x, int32_t parity,
    void* stream)
{
    if(t.nb <= 0) return 0;
    double* pub = t.chain_pub + (parity ? t.n : 0);
    double* next = t.chain_pub + (parity ? 0 : t.n);
    return (int) trsv_chain<VT>(p.task_u, 1, p.uo_col, p.uo_val, p.uo_lr, p.ui_col, p.ui_val,
        p.ui_lr, pub, next, t, x, CsrRhs{nullptr, nullptr, nullptr, nullptr},
        (hipStream_t) stream);
}

template<typename VT>
int trsv_upper_t_single(const SolveTopo& t, const SolvePlan<VT>& p, double* x, int32_t parity,
    void* stream)
{
    return trsv_upper_t_single_product<VT>(t, p, nullptr, nullptr, x, parity, stream);
}

template<typename VT>
int trsv_upper_t_single_product(const SolveTopo& t, const SolvePlan<VT>& p, const DevCsr* K,
    const double* src, double* x, int32_t parity, void* stream)
{
    if(t.nb <= 0) return 0;
    double* pub = t.chain_pub + (parity ? t.n : 0);
    double* next = t.chain_pub + (parity ? 0 : t.n);
    const CsrRhs rhs = K ? CsrRhs{K->row_ptr, K->col, K->val, src}
                         : CsrRhs{nullptr, nullptr, nullptr, nullptr};
    return (int) trsv_chain<VT>(p.task_t, 0, p.to_col, p.to_val, p.to_lr, p.ti_col, p.ti_val,
        p.ti_lr, pub, next, t, x, rhs, (hipStream_t) stream);
}

void chain_reset(double* pub, int64_t count, void* stream)
{
    if(count <= 0) return;
    k_fill_bits<<<(unsigned) ((count + 255) / 256), 256, 0, (hipStream_t) stream>>>(pub, count,
        CHAIN_EMPTY);
}

template<typename VT>
void jacobi_sweeps(const SolveTopo& t, const SolvePlan<VT>& p, bool transpose, double* x,
    int32_t sweeps, double* b_tmp, double* x_a, double* x_b, void* stream)
{
    jacobi_sweeps_product<VT>(t, p, transpose, nullptr, nullptr, x, sweeps, b_tmp, x_a, x_b, stream);
}

template<typename VT>
void jacobi_sweeps_product(const SolveTopo& t, const SolvePlan<VT>& p, bool transpose,
    const DevCsr* K, const double* src, double* x, int32_t sweeps, double* b_tmp, double* x_a,
    double* x_b, void* stream)
{
    if(t.nb <= 0 || sweeps <= 0) return;
    hipStream_t st = (hipStream_t) stream;
    const int4* task = transpose ? p.task_t : p.task_u;
    const int32_t* oc = transpose ? p.to_col : p.uo_col;
    const VT* ov = transpose ? p.to_val : p.uo_val;
    const uint8_t* ol = transpose ? p.to_lr : p.uo_lr;
    const int32_t* ic = transpose ? p.ti_col : p.ui_col;
    const VT* iv = transpose ? p.ti_val : p.ui_val;
    const uint8_t* il = transpose ? p.ti_lr : p.ui_lr;
    const double* in = nullptr;
    for(int32_t s = 0; s < sweeps; ++s) {
        double* out = (s == sweeps - 1) ? x : ((s & 1) ? x_b : x_a);
        if(s == 0 && K)
            k_jacobi_first_product<VT><<<t.nb, 64, 0, st>>>(task, oc, ov, ol, ic, iv, il,
                CsrRhs{K->row_ptr, K->col, K->val, src}, b_tmp, out);
        else
            k_jacobi_sweep<VT><<<t.nb, 64, 0, st>>>(task, oc, ov, ol, ic, iv, il, b_tmp, in, out);
        in = out;
    }
}

template void jacobi_sweeps<double>(const SolveTopo&, const SolvePlan<double>&, bool, double*, int32_t, double*, double*, double*, void*);
template void jacobi_sweeps<float>(const SolveTopo&, const SolvePlan<float>&, bool, double*, int32_t, double*, double*, double*, void*);
template void jacobi_sweeps_product<double>(const SolveTopo&, const SolvePlan<double>&, bool, const DevCsr*, const double*, double*, int32_t, double*, double*, double*, void*);
template void jacobi_sweeps_product<float>(const SolveTopo&, const SolvePlan<float>&, bool, const DevCsr*, const double*, double*, int32_t, double*, double*, double*, void*);
template int trsv_upper_single<double>(const SolveTopo&, const SolvePlan<double>&, double*, int32_t, void*);
template int trsv_upper_single<float>(const SolveTopo&, const SolvePlan<float>&, double*, int32_t, void*);
template int trsv_upper_t_single<double>(const SolveTopo&, const SolvePlan<double>&, double*, int32_t, void*);
template int trsv_upper_t_single<float>(const SolveTopo&, const SolvePlan<float>&, double*, int32_t, void*);
template int trsv_upper_t_single_product<double>(const SolveTopo&, const SolvePlan<double>&, const DevCsr*, const double*, double*, int32_t, void*);
template int trsv_upper_t_single_product<float>(const SolveTopo&, const SolvePlan<float>&, const DevCsr*, const double*, double*, int32_t, void*);
template void trsv_upper<double>(const SolveTopo&, const SolvePlan<double>&, double*, void*);
template void trsv_upper<float>(const SolveTopo&, const SolvePlan<float>&, double*, void*);
template void trsv_upper_t<double>(const SolveTopo&, const SolvePlan<double>&, double*, void*);
template void trsv_upper_t<float>(const SolveTopo&, const SolvePlan<float>&, double*, void*);


// the batched form of Bildlt::jacobi (copy, then jacobi_sweeps) and of
// left_product (K src, then the sweeps): the same sweeps and values. The
// product is the batched CSR product, whose rows equal those the fused
// first sweep forms; the sweeps read b from the target itself instead of a
// copy.
template<typename VT>
void batch_jacobi(const BatchLists& L, const BatchSys* sys, bool transpose, int32_t sweeps,
    int32_t target, int32_t product_src, hipStream_t st)
{
    if(L.blk.count <= 0 || sweeps <= 0) return;
    if(product_src != BV_NONE) batch_csr_spmv(L, sys, product_src, target, st);
    const int32_t tr = transpose ? 1 : 0;
    int32_t in = BV_NONE;
    for(int32_t s = 0; s < sweeps; ++s) {
        const int32_t out = (s == sweeps - 1) ? target : ((s & 1) ? BV_JB2 : BV_JB1);
        bk_jacobi_sweep<VT><<<(unsigned) L.blk.count, 64, 0, st>>>(L.blk.items, sys, tr, target,
            in, out);
        in = out;
    }
}

template void batch_jacobi<double>(const BatchLists&, const BatchSys*, bool, int32_t, int32_t, int32_t, hipStream_t);
template void batch_jacobi<float>(const BatchLists&, const BatchSys*, bool, int32_t, int32_t, int32_t, hipStream_t);


int32_t scan_chunks(int32_t n) { return (n + PS_CHUNK - 1) / PS_CHUNK; }

template<typename VT>
void plan_batch(const PlanSys<VT>* ps, FactorItems blk, FactorItems scan, FactorItems task,
    int32_t hm, hipStream_t st)
{
    if(blk.count <= 0) return;
    const unsigned nb = (unsigned) blk.count;
    const size_t lds = plan_rows_lds<VT>(hm);
    bk_plan_rows<VT, false><<<nb, 64, lds, st>>>(ps, blk.items, hm);
    bk_plan_cols<VT, false><<<nb, 64, 0, st>>>(ps, blk.items);
    for(int32_t q = 0; q < 4; ++q) {
        bk_chunk_sums<VT><<<(unsigned) scan.count, PS_TPB, 0, st>>>(ps, scan.items, q);
        bk_chunk_scan<VT><<<(unsigned) scan.count, PS_TPB, 0, st>>>(ps, scan.items, q);
    }
    bk_plan_rows<VT, true><<<nb, 64, lds, st>>>(ps, blk.items, hm);
    bk_plan_cols<VT, true><<<nb, 64, 0, st>>>(ps, blk.items);
    bk_plan_tasks<VT><<<(unsigned) task.count, 256, 0, st>>>(ps, task.items, 0);
    bk_plan_tasks<VT><<<(unsigned) task.count, 256, 0, st>>>(ps, task.items, 1);
}

template void plan_batch<double>(const PlanSys<double>*, FactorItems, FactorItems, FactorItems, int32_t, hipStream_t);
template void plan_batch<float>(const PlanSys<float>*, FactorItems, FactorItems, FactorItems, int32_t, hipStream_t);

}  // namespace culip
