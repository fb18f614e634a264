// gefenx_work.h -- the per-tensor work descriptor of the step kernels, the
// launch segment table, and the launchers the host code calls.
#pragma once

#include "gefenx_device.h"

#include <algorithm>
#include <type_traits>

namespace gx {

constexpr int kThreads = 256;
constexpr int kChunk = 8;
constexpr int64_t kWaves = kThreads / 64;
constexpr int64_t kApplyChunksPerThread = 8;   // apply: 4 iterations of 2 chunks
constexpr int64_t kFinBlocksPerWg = 1024;
constexpr int64_t kDefaultCohortElems = 0;  // one cohort per step (see cohort_limit)
constexpr int kTv = 64;                        // transposed views: square tiles of this side
constexpr int kTvLdsBlocks = 512;              // ... stats: LDS block accumulators per workgroup
constexpr int kTvTilesPerWave = 2;             // apply: consecutive tiles per wave
constexpr int64_t kRowSegCols = 64 * kChunk;   // apply_tasks: most columns of a task
constexpr int kRowsPerTask = 8;                // apply_tasks: row steps of a task
constexpr int64_t kSmallApplyElems = 1 << 22;  // ... in launches of at least so many elements, else 2
constexpr int kDetIters = 8;                   // block stats: items per thread
// Stats records per block from which the block finalize takes a workgroup per block.
constexpr int64_t kFinWideRecords = 32;

struct StepScalars {
    float lr, inv_bc2, inv_bc1, wdf;
};

// Everything one phase needs about one parameter.  Built on the host
// (build_work) from the C-ABI arguments; lives in kernel arguments (single
// parameter) or in device memory (multi-tensor).
struct TensorWork {
    void* p;
    const void* grad;
    uint8_t* idx;
    float* mag;          // m_magnitude
    float* v0;           // factored: v_row; block: vmean
    float* v1;           // factored: v_col
    double* row_part;    // factored workspace
    double* col_part;
    double* vsum;
    double* blk_sq;      // block workspace
    float* step;
    uint32_t* magbits;
    float* mag_old;
    float* minv;
    float* vcs;          // factored: sqrt(v_col), written by finalize
    uint32_t* fin;       // factored: {finalize counter, bits of mean(v_row)}
    struct DetRec* det_rec;  // block: per-workgroup first / last block partials
    const QTable* qt;
    const float* step_scalars;
    const int64_t* seed_dev;
    int64_t R, C, N, P, nb;
    double invC, invP;
    int64_t ps0, ps1, gs0, gs1;
    // factored stats: column tiles of the launch, rows and columns of a
    // workgroup, rows (views: columns) of a granule
    int64_t ct, tile_rows, tile_cols, gran, shards;
    // finalize: row and column tiles; column (row) partials per tile and in all
    int64_t f_rt, f_ct, pc_per, pc_n, pr_per, pr_n;
    // where a granule is a workgroup: the granules' column partials (views: row
    // partials), in a plan's host image their byte offset in its buffer; else null
    double* part;
    int64_t stats_wgs, nr, nc, nbw, fin_wgs, apply_wgs;
    int64_t det_elems;   // block stats: elements per workgroup
    int64_t fB, fP;          // flat apply: block advance for a stride of 256*8 elements
    int64_t a_segs, a_cols;  // apply_tasks: segments per row, columns of a segment
    int32_t a_lg, a_steps;   // ... log2 lanes per segment, row steps of a task
    uint64_t seed;
    int32_t dtype, mode;
    int32_t fast_stats, fast_apply;  // kernel variant: 0 general, 1 contiguous (apply: HOT), 2 transposed view, 3 apply of any alignment
    int32_t write_p, sr, bf16_mean, det_epl;  // det_epl: block stats elements per item (8 or 1)
    int32_t det_vec;     // block stats items: vector loads (grad 16-byte, indices 8-byte aligned)
    int32_t partial;     // block path with the caller's per-block stepsize (no vmean)
    int32_t fin_wide;    // block finalize: one workgroup per block (blocks span many stats records)
    int32_t lg_lanes;    // factored contiguous stats on lane tiles: log2 lanes per row (stats_lanes), else -1
    int32_t csplit;      // factored finalize: threads per column (1, 2, 4 or 8), each over a run of row tiles
    float eps, beta2, alpha2;
    float bc2_div;       // reference-order divisor (factored bc2, block sqrt(bc2)) or 0
    StepScalars sc;
    MomentumCoef mc;
};

__device__ __forceinline__ StepScalars read_scalars(const TensorWork& w) {
    StepScalars s = w.sc;
    if (w.step_scalars != nullptr) {
        s.lr = w.step_scalars[0];
        s.inv_bc2 = w.step_scalars[1];
        s.inv_bc1 = w.step_scalars[2];
        s.wdf = w.step_scalars[3];
    }
    return s;
}

// The factored stepsize of one element in the rounding order of the
// reference's decomposed step (gefen.py:2996-3006): vh = (v_row*v_col)/mean,
// h = sqrt(vh/bc2) + eps, (1/h) * (1/bc1), one fp32 rounding per operation.
// The divisions by the tensor-wide mean and bc2 take div_by_const; sqrt and
// 1/h are the correctly rounded operations.  Used for fp32 parameters when
// the host gave bc2 (w.bc2_div); otherwise the kernels take the cheaper
// sqrt(v_row*s) * sqrt(v_col) form, within 1e-6 of this.
struct RefStep {
    float mean, rmean, bc2, rbc2, eps, inv_bc1;
    bool on;
};

__device__ __forceinline__ RefStep make_ref_step(const TensorWork& w, const StepScalars& sc, float mean) {
    RefStep r;
    r.on = w.bc2_div > 0.0f;
    r.mean = mean;
    r.rmean = block_recip(mean);
    r.bc2 = w.bc2_div;
    r.rbc2 = block_recip(w.bc2_div);
    r.eps = w.eps;
    r.inv_bc1 = sc.inv_bc1;
    return r;
}

__device__ __forceinline__ float ref_step(const RefStep& r, float v_row, float v_col) {
    const float vh = div_by_const(v_row * v_col, r.mean, r.rmean);
    const float h = sqrtf(div_by_const(vh, r.bc2, r.rbc2)) + r.eps;
    return (1.0f / h) * r.inv_bc1;
}

// mean(v_row) as finalize stored it (already clamped at FLT_MIN).
__device__ __forceinline__ float stored_mean(const TensorWork& w) {
    return __uint_as_float(*gbl(w.fin + 1));
}

// Where the stats leave their column and row partials.
__device__ __forceinline__ double* col_partials(const TensorWork& w) {
    return w.part != nullptr && w.fast_stats != 2 ? w.part : w.col_part;
}
__device__ __forceinline__ double* row_partials(const TensorWork& w) {
    return w.part != nullptr && w.fast_stats == 2 ? w.part : w.row_part;
}

struct Seg {
    int32_t t;         // descriptor index
    int32_t pad_;
    int64_t wg_begin;  // first launch workgroup of this descriptor
};

// Launch workgroup -> segment.  coarse[j] is the segment holding workgroup
// j << gshift (the host picks gshift so the table stays small), so a lookup
// is one load plus a binary search inside one granule (usually empty).
struct SegTable {
    const Seg* segs;
    const int32_t* coarse;
    int nseg;
    int gshift;
};

__device__ __forceinline__ Seg find_seg(const SegTable& tb, int64_t wg) {
    const int64_t j = wg >> tb.gshift;
    int lo = gbl(tb.coarse)[j];
    int hi = gbl(tb.coarse)[j + 1] + 1;  // last seg with wg_begin <= wg lies in [lo, hi)
    hi = hi > tb.nseg ? tb.nseg : hi;
    const Seg* sg = tb.segs;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (*gbl(&sg[mid].wg_begin) <= wg) lo = mid; else hi = mid;
    }
    Seg r;
    r.t = *gbl(&sg[lo].t);
    r.pad_ = 0;
    r.wg_begin = *gbl(&sg[lo].wg_begin);
    return r;
}

// Launchers of the kernels that depend on the dtype (gefenx_step_kernels.h,
// instantiated by one source file per dtype).  key_mode: 0 a launch of
// factored tensors and of the block-path tensors that ride along, 1 one of
// block-path transposed views; fast: the kernel variant (TensorWork::fast_*).
template <int DT>
struct StepKernels {
    static void stats(const TensorWork& w, hipStream_t s);
    static void apply(const TensorWork& w, hipStream_t s);
    static void mt_stats(int key_mode, int fast, dim3 grid, hipStream_t s, const TensorWork* ws, SegTable sg);
    static void mt_apply(int key_mode, int fast, int sr, dim3 grid, hipStream_t s, const TensorWork* ws,
                         SegTable sg);
};

}  // namespace gx
