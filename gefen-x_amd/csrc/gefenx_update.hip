// gefenx_update.hip -- fused Gefen update kernels for MI355X (gfx950, wave64).
//
// Per parameter the step has three phases:
//   stats    one pass over grad + stored indices: per-block max |u| (u = the
//            updated momentum) and the second-moment sums (per-tile row/column
//            partial sums of g^2 for the factored path, per-block sums for the
//            block path);
//   finalize tiny: EMA of the second moment, new magnitudes and their
//            reciprocals, per-block stepsizes (block path), partial sums of
//            v_row; re-zeroes the workspace accumulators;
//   apply    one pass: recompute u, normalise by the new magnitude,
//            requantise through the exact threshold table, write the indices
//            and the parameter (decoupled weight decay folded in).
// Every phase is a device function of (TensorWork, workgroup index): the
// single-parameter entry points launch it for one descriptor passed by value,
// the multi-tensor launcher (gefenx_multi_tensor_step) launches it for a
// cohort of parameters whose workgroups are laid end to end.
// The math follows the reference's decomposed step (gefen.py:2959-3018,
// 3329-3486, 3776-3818); gefenx_device.h holds the bit-exact momentum,
// division and quantisation primitives.
#include "gefenx_work.h"
#include "gefenx_internal.h"
#include "gefenx_profile.h"
#include "gefenx.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>
#include <vector>

namespace gx {

// New magnitude (max over the shards), its reciprocal and the old magnitude.
__device__ __forceinline__ void finalize_magnitude(const TensorWork& w, int64_t b) {
    const float old = w.mag[b];
    w.mag_old[b] = old;
    uint32_t bits = 0u;
    drain_shards(w.magbits, w.shards, w.nb, b, [&](uint32_t v) { bits = v > bits ? v : bits; });
    const float m = __uint_as_float(bits);
    w.mag[b] = m;
    w.minv[b] = block_recip(m);
}

// Sum of the tiles [t0, t1), in order, of n partials p[0], p[stride], ..., of
// which `per` in order make a tile; the loads issued eight at a time.
__device__ __forceinline__ double tile_sum(const double* __restrict__ p, int64_t t0, int64_t t1, int64_t per, int64_t n,
                                           int64_t stride) {
    const int64_t end = t1 * per < n ? t1 * per : n;
    double s = 0.0, t = 0.0;
    int left = (int)per;
    const auto add = [&](double a) {  // 0 + a is a: with one partial to a tile, s += a
        t += a;
        if (--left == 0) {
            s += t;
            t = 0.0;
            left = (int)per;
        }
    };
    int64_t i = t0 * per;
    const auto run = [&](auto n_loads) {
        constexpr int kLoads = decltype(n_loads)::value;
        for (; i + kLoads <= end; i += kLoads) {
            double a[kLoads];
#pragma unroll
            for (int k = 0; k < kLoads; ++k) a[k] = *gbl(p + (i + k) * stride);
#pragma unroll
            for (int k = 0; k < kLoads; ++k) add(a[k]);
        }
    };
    run(std::integral_constant<int, 8>{});
    run(std::integral_constant<int, 2>{});
    for (; i < end; ++i) add(*gbl(p + i * stride));
    return left != (int)per ? s + t : s;
}

// ====================================================================
// Factored finalize.  Workgroups [0, nr): v_row EMA from the row partials of
// the f_ct column tiles plus one float64 partial of sum(v_row); [nr, nr+nc):
// v_col EMA from the column partials of the f_rt row tiles in order, csplit
// threads per column: thread p sums the p-th run of ceil(f_rt / csplit) tiles
// in order, then the runs are added in order; the rest: magnitudes.
// v <- fma(sum/n, 1-beta2, v*beta2)  (gefen.py:2994-2996)
// ====================================================================
__device__ __forceinline__ void finalize_factored(const TensorWork& w, int64_t wg) {
    const int tid = threadIdx.x;
    if (wg < w.nr) {
        __shared__ double s_part[kWaves];
        const int64_t i = wg * kFinRowsPerWg + tid;
        double v64 = 0.0;
        if (i < w.R) {
            const double s = tile_sum(row_partials(w) + i, 0, w.f_ct, w.pr_per, w.pr_n, w.R);
            const float ms = (float)s / (float)w.C;
            const float v = __builtin_fmaf(ms, w.alpha2, w.v0[i] * w.beta2);
            w.v0[i] = v;
            v64 = (double)v;
        }
        v64 = wave_sum_d(v64);
        if ((tid & 63) == 0) s_part[tid >> 6] = v64;
        __syncthreads();
        if (tid == 0) {
            double s = 0.0;
            for (int ww = 0; ww < kWaves; ++ww) s += s_part[ww];
            w.vsum[wg] = s;
        }
        return;
    }
    if (wg < w.nr + w.nc) {
        __shared__ double s_run[kThreads];
        const int sp = w.csplit;
        const int cpw = kThreads / sp;  // columns per workgroup
        const int part = tid / cpw;
        const int64_t j = (wg - w.nr) * cpw + tid % cpw;
        const int64_t per = (w.f_rt + sp - 1) / sp;
        const int64_t t0 = std::min<int64_t>((int64_t)part * per, w.f_rt);
        const int64_t t1 = std::min<int64_t>(t0 + per, w.f_rt);
        double tot = j < w.C ? tile_sum(col_partials(w) + j, t0, t1, w.pc_per, w.pc_n, w.C) : 0.0;
        if (sp > 1) {
            s_run[tid] = tot;
            __syncthreads();
            if (part == 0)
                for (int q = 1; q < sp; ++q) tot += s_run[q * cpw + tid];
        }
        if (part == 0 && j < w.C) {
            const float ms = (float)tot / (float)w.R;
            const float v = __builtin_fmaf(ms, w.alpha2, w.v1[j] * w.beta2);
            w.v1[j] = v;
            w.vcs[j] = sqrtf(v);
        }
        return;
    }
    const int64_t gtid = (wg - w.nr - w.nc) * kThreads + tid;
    const int64_t gstride = w.nbw * kThreads;
    for (int64_t b = gtid; b < w.nb; b += gstride) finalize_magnitude(w, b);
}

// vmean EMA + per-block stepsize of block b from its sum of squares
// (gefen.py:180-190, 3794-3805), then its magnitude.
__device__ __forceinline__ void finalize_block_one(const TensorWork& w, const StepScalars& sc, int64_t b, double sq) {
    float mean = (float)sq / (float)w.P;
    if (w.bf16_mean) mean = round_dt<BF16>(mean);
    const float v = __builtin_fmaf(mean, w.alpha2, w.v0[b] * w.beta2);
    w.v0[b] = v;
    // the reference divides by sqrt(bc2) (gefen.py:3794-3805); without that
    // divisor from the host, multiply by the scalar row's 1/sqrt(bc2)
    const float h = (w.bc2_div > 0.0f ? sqrtf(v) / w.bc2_div : sqrtf(v) * sc.inv_bc2) + w.eps;
    w.step[b] = (1.0f / h) * sc.inv_bc1;
    finalize_magnitude(w, b);
}

// Wide form: workgroup b sums block b's stored sum and the records of the
// workgroups it spans (thread t takes records t, t+256, ... in order, then a
// fixed-order reduction), so a block of tens of millions of elements is not
// one thread's serial walk.
__device__ __forceinline__ void finalize_block_wide(const TensorWork& w, int64_t b) {
    __shared__ double s_part[kWaves];
    const int tid = threadIdx.x;
    double part = 0.0;
    if (!w.partial) {
        const int64_t wlo = (b * w.P) / w.det_elems;
        const int64_t whi = ((b + 1) * w.P - 1) / w.det_elems;
        for (int64_t r = wlo + tid; r <= whi; r += kThreads) {
            const DetRec d = w.det_rec[r];
            if (d.kf == b) part += d.sf;
            if (d.kl == b) part += d.sl;
        }
    }
    part = wave_sum_d(part);
    if ((tid & 63) == 0) s_part[tid >> 6] = part;
    __syncthreads();
    if (tid != 0) return;
    double sq = 0.0;
    drain_shards(w.blk_sq, w.shards, w.nb, b, [&](double v) { sq += v; });
    if (w.partial) {  // the stepsize comes from the caller: magnitudes only
        finalize_magnitude(w, b);
        return;
    }
    for (int ww = 0; ww < kWaves; ++ww) sq += s_part[ww];
    finalize_block_one(w, read_scalars(w), b, sq);
}

// vmean EMA + per-block stepsize (gefen.py:180-190, 3794-3805) + magnitudes.
__device__ __forceinline__ void finalize_block(const TensorWork& w, int64_t wg) {
    if (w.fin_wide) {
        if (wg < w.nb) finalize_block_wide(w, wg);
        return;
    }
    const StepScalars sc = read_scalars(w);
    for (int64_t b = wg * kThreads + threadIdx.x; b < w.nb; b += w.nbw * kThreads) {
        // the fixed-order stats store a block's sum (in shard 0) when the
        // block is complete inside one workgroup, or leave it in the records
        // of the workgroups it spans; the transposed-view stats accumulate
        // into the shards
        double sq = 0.0;
        drain_shards(w.blk_sq, w.shards, w.nb, b, [&](double v) { sq += v; });
        if (w.partial) {  // the stepsize comes from the caller: magnitudes only
            finalize_magnitude(w, b);
            continue;
        }
        if (w.det_rec != nullptr) {
            const int64_t wlo = (b * w.P) / w.det_elems;
            const int64_t whi = ((b + 1) * w.P - 1) / w.det_elems;
            for (int64_t r = wlo; r <= whi; ++r) {
                const DetRec d = w.det_rec[r];
                if (d.kf == b) sq += d.sf;
                if (d.kl == b) sq += d.sl;
            }
        }
        finalize_block_one(w, sc, b, sq);
    }
}

// mean(v_row) of one factored parameter from the finalize partials, in a
// fixed order, clamped at FLT_MIN (gefen.py:2998-3000); one workgroup.
__device__ __forceinline__ void mean_phase(const TensorWork& w) {
    __shared__ double s_part[kWaves];
    const int tid = threadIdx.x;
    double acc = 0.0;
    for (int64_t k = tid; k < w.nr; k += kThreads) acc += *gbl(w.vsum + k);
    acc = wave_sum_d(acc);
    if ((tid & 63) == 0) s_part[tid >> 6] = acc;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int ww = 0; ww < kWaves; ++ww) t += s_part[ww];
        float mean = (float)t / (float)w.R;
        if (!(mean >= 1.17549435e-38f) && mean == mean) mean = 1.17549435e-38f;
        w.fin[1] = __float_as_uint(mean);
    }
}

__global__ void __launch_bounds__(kThreads) k_finalize(TensorWork w) {
    if (w.mode == 0) finalize_factored(w, blockIdx.x);
    else finalize_block(w, blockIdx.x);
}

__global__ void __launch_bounds__(kThreads) k_mean(TensorWork w) { mean_phase(w); }

__global__ void __launch_bounds__(kThreads) k_mt_finalize(const TensorWork* __restrict__ ws,
                                                          SegTable tb) {
    const Seg sg = find_seg(tb, blockIdx.x);
    const TensorWork& w = ws[sg.t];
    const int64_t local = (int64_t)blockIdx.x - sg.wg_begin;
    if (w.mode == 0) finalize_factored(w, local);
    else finalize_block(w, local);
}

__global__ void __launch_bounds__(kThreads) k_mt_mean(const TensorWork* __restrict__ ws, SegTable tb) {
    const Seg sg = find_seg(tb, blockIdx.x);
    mean_phase(ws[sg.t]);
}

// ====================================================================
// Host side
// ====================================================================

static MomentumCoef make_coef_w(float w1) {
    MomentumCoef mc;
    mc.w = w1;
    mc.wm1 = mc.w - 1.0f;
    mc.small = std::fabs(mc.w) < 0.5f ? 1 : 0;
    return mc;
}

static inline bool aligned(const void* ptr, size_t a) {
    return (reinterpret_cast<uintptr_t>(ptr) % a) == 0;
}

static int launch_check(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(GEFENX_ELAUNCH, "%s: %s", what, hipGetErrorString(e));
    return GEFENX_OK;
}

static inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

static size_t elem_size(int dtype) { return dtype == F32 ? 4 : 2; }

// Fill the derived fields of a descriptor.  Everything that depends only on
// shapes, strides, pointers and the workspace layout is computed here.
struct WorkInput {
    void* p;
    const void* grad;
    int dtype;
    int mode;  // 0 factored, 1 block
    int64_t R, C, ps0, ps1, gs0, gs1, period;
    uint8_t* idx;
    float* mag;
    float* v0;
    float* v1;
    const void* qt;
    float lerp_w, beta2, alpha2, eps;
    float bc2_div;  // reference-order divisor or 0 (gefenx_tensor_desc.bc2_div)
    StepScalars sc;
    int sr;
    uint64_t seed;
    const float* step_scalars;
    const int64_t* seed_dev;
    void* workspace;
    size_t ws_bytes;
};

// The divisor of the reference's decomposed step (bc2, or sqrt(bc2) on the
// block path) from the reciprocal the C ABI passes, in double then rounded
// once: (float)(1/(1/x)) equals (float)x unless x lies within ~2^-52 of an
// fp32 rounding midpoint (none for beta2 in {0.5, 0.9, 0.95, ..., 0.9999}
// over 200,000 steps).  Python descriptors carry the same value.
static float reference_divisor(double inv) {
    if (!(inv > 0.0) || !std::isfinite(inv)) return 0.0f;
    return (float)(1.0 / inv);
}

// Workgroup = tile q of the contiguous (lane or 1024-column) or view stats.
static void set_tiles(TensorWork& w, const Tiling& q) {
    w.ct = w.f_ct = w.pr_n = q.ct;
    w.f_rt = w.pc_n = q.rt;
    w.pc_per = w.pr_per = 1;
    w.tile_rows = q.rows;
    w.tile_cols = q.cols;
    w.gran = q.gran;
    w.stats_wgs = q.ct * q.rt;
}

// Granules of the launch's workgroups where a granule is one (0 columns or rows
// of partials each: the block path's views leave none).
struct Granules {
    int64_t wgs, doubles;
};

static Granules granules(const TensorWork& w) {
    if (w.fast_stats == 2) {
        const int64_t ng = ceil_div(w.C, w.gran);
        return Granules{ng * w.f_rt, w.mode == 0 ? ng * w.R : 0};
    }
    const int64_t ng = ceil_div(w.R, w.gran);
    return Granules{w.f_ct * ng, ng * w.C};
}

// Workgroup = granule; the caller says where the partials are (part, or
// col_part / row_part of a single tensor).
static void take_granules(TensorWork& w) {
    w.stats_wgs = granules(w).wgs;
    if (w.fast_stats == 2) {
        w.pr_per = w.tile_cols / w.gran;
        w.ct = w.pr_n = ceil_div(w.C, w.gran);
        w.tile_cols = w.gran;
    } else {
        w.pc_per = ceil_div(w.tile_rows, w.gran);
        w.pc_n = ceil_div(w.R, w.gran);
        w.tile_rows = w.gran;
    }
}

// A granule is a workgroup where the tile holds more than this share of its
// launch's elements: the 256 CUs take four workgroups each (the LDS of one
// allows four), and fewer than two leave them waiting for loads.  Measured (stats
// kernel, us; tiles of N/32 alone -> about 1/512, 1/1024, 1/2048 of the launch):
// one decoder layer (218M bf16) 282 -> 154, 129, 136; 4096x4096 fp32 140 -> 28,
// 30, 35; 43M fp16 elements in odd sizes 470 -> 57, 46, 47; 7.5M bf16 in 8 matrices
// 258 -> 76, 75, 75; but 20 of 4096x4096 bf16, 640 tiles, 727 us a step in tiles
// and 757 in 1024 parts.
constexpr int64_t kFactLaunchWgs = 512;
constexpr int64_t kTvLaunchWgs = 2048;  // kTvStatsMaxRows has the figures
// Views whose bands hold more blocks than a workgroup's LDS send an atomic per
// chunk, more of them to one block at a time the narrower the workgroups are
// (4096 x 11008 in 256-element blocks, 176 tiles: 350 us a step in tiles, 385 and
// 408 in 256 and 128 columns; 4096 x 4096, 64 tiles: 175 in tiles, 145 in 128).
constexpr int64_t kTvManyBlockTiles = 128;

static bool wants_granules(const TensorWork& w, int64_t launch_elems) {
    if ((w.mode != 0 && w.fast_stats != 2) || granules(w).wgs <= w.stats_wgs) return false;
    if (w.fast_stats == 2 && w.tile_rows * w.C / w.P > kTvLdsBlocks && w.stats_wgs >= kTvManyBlockTiles) return false;
    const int64_t tile = std::min<int64_t>(w.tile_rows, w.R) * std::min<int64_t>(w.tile_cols, w.C);
    return tile > launch_elems / (w.fast_stats == 2 ? kTvLaunchWgs : kFactLaunchWgs);
}

// Row steps of an apply task (apply_tasks), by the elements of its launch.
static void set_apply_steps(TensorWork& w, int64_t launch_elems) {
    if (w.mode != 0 || !(w.fast_apply & 1)) return;
    w.a_steps = launch_elems < kSmallApplyElems ? 2 : kRowsPerTask;
    const int64_t task_rows = (int64_t)w.a_steps * (64 >> w.a_lg);
    w.apply_wgs = ceil_div(w.a_segs * ceil_div(w.R, task_rows), (int64_t)kWaves);
}

// Transposed views the view kernels take: strides (1, ld), storage rows 16-byte
// aligned, chunks that cross no row, column or block border.
static bool view_shape(int64_t R, int64_t C, int64_t P, const void* idx) {
    return R > 1 && R % kChunk == 0 && C % kChunk == 0 && P % kChunk == 0 && aligned(idx, 8);
}
static bool view_strides(int64_t R, int64_t s0, int64_t s1, int dtype, const void* data) {
    return s0 == 1 && s1 >= R && (s1 * (int64_t)elem_size(dtype)) % 16 == 0 && aligned(data, 16);
}

// The factored stats' variant and tiles.
static void set_factored_stats(TensorWork& w, const FactTiles& t) {
    const bool dense = w.gs1 == 1 && w.gs0 == w.C;
    w.fast_stats = dense && w.C >= kChunk ? 1
                 : view_shape(w.R, w.C, w.P, w.idx) && view_strides(w.R, w.gs0, w.gs1, w.dtype, w.grad) ? 2 : 0;
    w.lg_lanes = w.fast_stats == 1 ? (int32_t)t.lg_lanes : -1;
    set_tiles(w, w.fast_stats == 2 ? t.tv : w.lg_lanes >= 0 ? t.lane : t.wide);
}

static int build_work(const WorkInput& in, TensorWork& w) {
    std::memset(&w, 0, sizeof(w));
    const int64_t N = in.R * in.C;
    const int64_t nb = N / in.period;
    w.p = in.p; w.grad = in.grad; w.idx = in.idx; w.mag = in.mag; w.v0 = in.v0; w.v1 = in.v1;
    w.qt = static_cast<const QTable*>(in.qt);
    w.step_scalars = in.step_scalars; w.seed_dev = in.seed_dev;
    w.R = in.R; w.C = in.C; w.N = N; w.P = in.period; w.nb = nb;
    w.invC = 1.0 / (double)in.C; w.invP = 1.0 / (double)in.period;
    w.ps0 = in.ps0; w.ps1 = in.ps1; w.gs0 = in.gs0; w.gs1 = in.gs1;
    w.shards = mag_shards(nb);
    w.seed = in.seed;
    w.dtype = in.dtype; w.mode = in.mode; w.sr = in.sr;
    w.bf16_mean = in.dtype == BF16 ? 1 : 0;
    w.eps = in.eps; w.beta2 = in.beta2; w.alpha2 = in.alpha2;
    // the divisor describes the host scalars; a device scalar row carries 1/bc2 only
    w.bc2_div = in.step_scalars == nullptr && in.bc2_div > 0.0f ? in.bc2_div : 0.0f;
    w.sc = in.sc;
    w.mc = make_coef_w(in.lerp_w);
    w.write_p = (in.step_scalars != nullptr) || !(in.sc.lr == 0.0f && in.sc.wdf == 1.0f);
    char* ws = static_cast<char*>(in.workspace);
    const int64_t nchunks = ceil_div(N, kChunk);
    const bool tv_shape = view_shape(in.R, in.C, in.period, in.idx);
    const bool tv_g = view_strides(in.R, in.gs0, in.gs1, in.dtype, in.grad);
    const bool tv_p = view_strides(in.R, in.ps0, in.ps1, in.dtype, in.p);
    if (in.mode == 0) {
        const FactoredWs L = FactoredWs::make(in.R, in.C, nb);
        if (in.ws_bytes < L.total)
            return set_error(GEFENX_EINVAL, "factored update: workspace %zu bytes < required %zu", in.ws_bytes, L.total);
        w.row_part = reinterpret_cast<double*>(ws + L.off_rowp);
        w.col_part = reinterpret_cast<double*>(ws + L.off_colp);
        w.magbits = reinterpret_cast<uint32_t*>(ws + L.off_magbits);
        w.mag_old = reinterpret_cast<float*>(ws + L.off_magold);
        w.minv = reinterpret_cast<float*>(ws + L.off_minv);
        w.vsum = reinterpret_cast<double*>(ws + L.off_vsum);
        w.vcs = reinterpret_cast<float*>(ws + L.off_vcs);
        w.fin = reinterpret_cast<uint32_t*>(ws + L.off_fin);
        w.nr = ceil_div(in.R, kFinRowsPerWg);
        w.nbw = std::max<int64_t>(1, std::min<int64_t>(1024, ceil_div(nb, kFinBlocksPerWg)));
        const bool contig_g = (in.gs1 == 1 && in.gs0 == in.C);
        const bool contig_p = (in.ps1 == 1 && in.ps0 == in.C);
        set_factored_stats(w, L.tiles);
        w.fast_apply = 0;
        if (contig_g && contig_p && in.C >= kChunk && in.period >= kChunk) {
            const bool hot = !in.sr && in.C >= kRowSegCols && in.C % kChunk == 0 && in.period % kChunk == 0 &&
                             in.period >= kShortPeriod && aligned(in.grad, 16) && aligned(in.p, 16) &&
                             aligned(in.idx, 8);
            w.fast_apply = hot ? 1 : 3;
        }
        // column sums over many granules split into up to 8 runs (of <= 32
        // values up to 256 of them), so no thread waits on a long load chain
        const int64_t col_values = w.fast_stats == 2 ? w.f_rt : ceil_div(in.R, w.gran);
        w.csplit = 1;
        while (w.csplit < 8 && ceil_div(col_values, (int64_t)w.csplit) > 32) w.csplit *= 2;
        w.nc = ceil_div(in.C, kThreads / w.csplit);
        w.fin_wgs = w.nr + w.nc + w.nbw;
        // the view apply reads v_row and sqrt(v_col) (v_col on the fp32
        // reference path) 8 floats at a time
        if (!w.fast_apply && tv_shape && tv_g && tv_p && !in.sr && w.write_p && aligned(in.v0, 16) &&
            aligned(in.v1, 16))
            w.fast_apply = 2;
    } else {
        const BlockWs L = BlockWs::make(nb, N);
        if (in.ws_bytes < L.total)
            return set_error(GEFENX_EINVAL, "block update: workspace %zu bytes < required %zu", in.ws_bytes, L.total);
        w.blk_sq = reinterpret_cast<double*>(ws + L.off_sq);
        w.magbits = reinterpret_cast<uint32_t*>(ws + L.off_magbits);
        w.mag_old = reinterpret_cast<float*>(ws + L.off_magold);
        w.step = reinterpret_cast<float*>(ws + L.off_step);
        w.minv = reinterpret_cast<float*>(ws + L.off_minv);
        w.det_rec = reinterpret_cast<DetRec*>(ws + L.off_rec);
        // fixed-order stats: 8 elements per item when chunks never cross a
        // block (P and N multiples of 8), else 1.  The summation order then
        // depends on the shape alone, not on where the grad starts in memory
        // (a view into a flat bucket sums like a fresh tensor); a misaligned
        // grad or index array loads its items element by element.
        w.det_epl = (in.period % kChunk == 0 && N % kChunk == 0) ? (int32_t)kChunk : 1;
        w.det_vec = aligned(in.grad, 16) && aligned(in.idx, 8) ? 1 : 0;
        w.det_elems = (int64_t)kDetIters * kThreads * w.det_epl;
        w.stats_wgs = std::max<int64_t>(1, ceil_div(N, w.det_elems));
        w.nbw = std::max<int64_t>(1, std::min<int64_t>(4096, ceil_div(nb, kThreads)));
        w.fin_wgs = w.nbw;
        w.fast_stats = aligned(in.grad, 16) && aligned(in.idx, 8);
        w.fast_apply = 0;
        if (in.period >= kChunk) {
            const bool hot = !in.sr && in.period % kChunk == 0 && aligned(in.grad, 16) && aligned(in.p, 16) &&
                             aligned(in.idx, 8);
            w.fast_apply = hot ? 1 : 3;
        }
        if (in.R > 1) {
            // a 2D descriptor that is not contiguous (the callers flatten the
            // contiguous ones): the grad must be contiguous (flat stats) or a
            // transposed view; p any strides (general apply) or a view too
            const bool g_contig = in.gs1 == 1 && in.gs0 == in.C;
            const bool p_contig = in.ps1 == 1 && in.ps0 == in.C;
            if (tv_shape && tv_g) {
                set_tiles(w, FactTiles::make(in.R, in.C, in.period, false).tv);
                w.fast_stats = 2;
                w.det_rec = nullptr;  // the view tiles accumulate into the shards
            } else if (!g_contig) {
                return set_error(GEFENX_EINVAL,
                                 "block update: grad strides (%lld, %lld) of [%lld, %lld] are neither contiguous nor "
                                 "a transposed view with rows, cols and period multiples of 8",
                                 (long long)in.gs0, (long long)in.gs1, (long long)in.R, (long long)in.C);
            }
            w.fast_apply = (tv_shape && tv_g && tv_p && !in.sr && w.write_p) ? 2
                         : (g_contig && p_contig) ? w.fast_apply : 0;
        }
        // blocks that span many stats workgroups sum their records with a
        // whole workgroup each (a thread would walk thousands of them)
        if (w.det_rec != nullptr && w.P / w.det_elems + 2 >= kFinWideRecords) {
            w.fin_wide = 1;
            w.nbw = nb;
            w.fin_wgs = nb;
        }
    }
    w.apply_wgs = std::max<int64_t>(1, ceil_div(nchunks, kThreads * kApplyChunksPerThread));
    if (in.mode == 0 && (w.fast_apply & 1)) {  // 1 or 3
        // even segments of at most 512 columns, a whole number of chunks each
        // but the last; short rows share a wave.  kRowsPerTask row steps a
        // task, fewer where the launch would leave CUs idle.
        w.a_segs = ceil_div(in.C, kRowSegCols);
        w.a_cols = ceil_div(ceil_div(in.C, w.a_segs), (int64_t)kChunk) * kChunk;
        w.a_segs = ceil_div(in.C, w.a_cols);
        // no last segment of fewer than 8 columns: its lanes would step back
        // into the segment before it, which another wave updates
        while (w.a_segs > 1 && in.C - (w.a_segs - 1) * w.a_cols < kChunk) {
            w.a_cols -= kChunk;
            w.a_segs = ceil_div(in.C, w.a_cols);
        }
        w.a_lg = 0;
        while ((kChunk << w.a_lg) < w.a_cols) ++w.a_lg;
        set_apply_steps(w, N);
    }
    if (w.fast_apply == 2)
        w.apply_wgs = ceil_div(ceil_div(in.R, kTv) * ceil_div(in.C, kTv), (int64_t)kWaves * kTvTilesPerWave);
    const int64_t F = kThreads * kChunk;
    w.fB = F / w.P;
    w.fP = F - w.fB * w.P;
    return GEFENX_OK;
}

// 8% of the apply of so many 16-bit elements (8 B each at ~5.5 TB/s) are about
// the 5 us of a launch.
constexpr int64_t kMergeApplyElems = (int64_t)1 << 25;

// Algorithmic bytes of one parameter's step: p r/w, g r, idx r/w per element
// plus the fp32 state vectors read and written.
static double algo_bytes(const TensorWork& w) {
    const double es = (double)elem_size(w.dtype);
    const double vec = w.mode == 0 ? 8.0 * (double)(w.R + w.C + w.nb) : 16.0 * (double)w.nb;
    return (double)w.N * (3.0 * es + 2.0) + vec;
}

// f(StepKernels<DT>{}) for the dtype code dt.
template <class F>
static void with_dtype(int dt, F&& f) {
    switch (dt) {
        case F32: f(StepKernels<F32>{}); break;
        case F16: f(StepKernels<F16>{}); break;
        default: f(StepKernels<BF16>{}); break;
    }
}

// Run the three phases of one parameter (single-parameter entry points).
static int run_single(const TensorWork& w, hipStream_t s) {
    const double es = (double)elem_size(w.dtype);
    int ph = prof_begin(w.mode == 0 ? GEFENX_K_STATS : GEFENX_K_BLOCK_STATS, (double)w.N * (es + 1.0), 0.0, s);
    const dim3 block(kThreads);
    with_dtype(w.dtype, [&](auto k) { k.stats(w, s); });
    prof_end(ph, s);
    int rc = launch_check("stats");
    if (rc) return rc;
    ph = prof_begin(GEFENX_K_FINALIZE, 16.0 * (double)(w.R + w.C + w.nb), 0.0, s);
    hipLaunchKernelGGL(k_finalize, dim3((unsigned)w.fin_wgs), block, 0, s, w);
    if (w.mode == 0) hipLaunchKernelGGL(k_mean, dim3(1), block, 0, s, w);
    prof_end(ph, s);
    rc = launch_check("finalize");
    if (rc) return rc;
    ph = prof_begin(w.mode == 0 ? GEFENX_K_APPLY : GEFENX_K_BLOCK_APPLY, algo_bytes(w), 0.0, s);
    with_dtype(w.dtype, [&](auto k) { k.apply(w, s); });
    prof_end(ph, s);
    return launch_check("apply");
}

// ------------------------------------------------------------ multi-tensor

// Launch-group key: tensors of one cohort that share a kernel variant.
struct GroupKey {
    int mode, dtype, fast, sr;
    bool operator<(const GroupKey& o) const {
        return std::tie(mode, dtype, fast, sr) < std::tie(o.mode, o.dtype, o.fast, o.sr);
    }
};

struct Launch {
    int phase;       // 0 stats, 1 finalize, 2 apply, 3 mean(v_row)
    int cohort;      // index of the cohort the launch belongs to
    GroupKey key;
    size_t seg_off;  // index of the first Seg in the segment array
    int nseg;
    size_t coarse_off;  // index of the first coarse entry
    int gshift;
    int64_t wgs;
    double bytes;
};

// Pinned, double-buffered staging for the per-step descriptor upload.
struct Staging {
    void* host[2] = {nullptr, nullptr};
    size_t cap[2] = {0, 0};
    hipEvent_t done[2] = {nullptr, nullptr};
    int next = 0;
};
static std::mutex g_stage_mu;
static std::map<int, Staging> g_stage;  // per device; never freed (process lifetime)

// Cohorts: consecutive parameters whose summed element count stays within
// the limit.  Each cohort runs stats -> finalize -> mean -> apply; with more
// than one cohort, the stats of cohort k+1 run on a side stream while cohort
// k applies.  Default: one cohort per step (on the Llama-3-8B set, 256M-element
// cohorts overlapped this way measured no faster: both passes already share
// the same HBM ceiling).  GEFENX_COHORT_ELEMS sets the limit (<= 0: one
// cohort); GEFENX_PIPELINE=0 keeps every launch on the caller's stream.
// Both are read at every plan build (a getenv per step), so a process can
// change them between steps.
static int64_t cohort_limit() {
    const char* e = std::getenv("GEFENX_COHORT_ELEMS");
    int64_t v = e ? std::atoll(e) : kDefaultCohortElems;
    return v > 0 ? v : (int64_t)1 << 62;
}

static bool pipeline_enabled() {
    const char* e = std::getenv("GEFENX_PIPELINE");
    return !(e && std::atoi(e) == 0);
}

struct MtLayout {
    std::vector<TensorWork> works;
    std::vector<Seg> segs;
    std::vector<int32_t> coarse;
    std::vector<Launch> launches;
    size_t part_bytes = 0;  // granule partials
};

// Granule partials of one call: at most so many bytes (a decoder layer of the
// Llama-3-8B set takes 30 MB; launches of half a billion elements and more run
// on tiles and take none).  Tensors past it keep their tiles as workgroups, with
// the same sums.
constexpr size_t kGranuleBytes = (size_t)64 << 20;

// Stats launch of a tensor.  Block-path tensors other than transposed views
// join the factored launches of their dtype (the kernels branch per tensor):
// two launches fewer per step when both paths occur.
static GroupKey stats_key(const TensorWork& w) {
    if (w.mode == 1 && w.fast_stats != 2) return GroupKey{0, w.dtype, 1, 0};
    return GroupKey{w.mode, w.dtype, w.fast_stats, 0};
}

static int64_t group_elems(const std::vector<TensorWork>& works, const std::vector<int>& group) {
    int64_t n = 0;
    for (int t : group) n += works[(size_t)t].N;
    return n;
}

// Granules as workgroups for those tensors of a stats launch that want it,
// partials from address at + used on, within cap bytes.
static void cut_stats(std::vector<TensorWork>& works, const std::vector<int>& group, uintptr_t at, size_t cap,
                      size_t& used) {
    const int64_t elems = group_elems(works, group);
    for (int t : group) {
        TensorWork& w = works[(size_t)t];
        if (!wants_granules(w, elems)) continue;
        const size_t bytes = align256(sizeof(double) * (size_t)granules(w).doubles);
        if (used + bytes > cap) continue;
        if (bytes > 0) w.part = reinterpret_cast<double*>(at + used);
        used += bytes;
        take_granules(w);
    }
}

// Cohort of consecutive tensors that starts at c0: its end.
static int cohort_end(const std::vector<TensorWork>& works, int c0) {
    const int64_t limit = cohort_limit();
    const int n = (int)works.size();
    int c1 = c0;
    int64_t acc = 0;
    while (c1 < n && (c1 == c0 || acc + works[(size_t)c1].N <= limit)) acc += works[(size_t)c1++].N;
    return c1;
}

// part: part_cap bytes for granule partials (a device address, or for a plan the
// offset in its buffer).
static void plan_multi(const std::vector<TensorWork>& works_in, uintptr_t part, size_t part_cap, MtLayout& L) {
    L.works = works_in;
    L.segs.clear();
    L.coarse.clear();
    L.launches.clear();
    L.part_bytes = 0;
    std::vector<TensorWork>& works = L.works;
    const int n = (int)works.size();
    int c0 = 0, cohort = 0;
    while (c0 < n) {
        const int c1 = cohort_end(works, c0);
        // phases in launch order: 0 stats, 1 finalize, 3 mean(v_row), 2 apply
        for (int phase : {0, 1, 3, 2}) {
            std::map<GroupKey, std::vector<int>> groups;
            for (int t = c0; t < c1; ++t) {
                const TensorWork& w = works[(size_t)t];
                GroupKey k{0, 0, 0, 0};
                if (phase == 0) k = stats_key(w);
                if (phase == 2) {
                    k = GroupKey{w.mode, w.dtype, w.fast_apply, w.sr};
                    if (w.fast_apply != 2) k.mode = 0;  // as in stats_key
                }
                if (phase == 3 && w.mode != 0) continue;
                groups[k].push_back(t);
            }
            // transposed-view stats before the contiguous ones: their index
            // loads go through L2, so the contiguous stats' partials, which
            // the finalize reads next, stay cached (measured on the Qwen3-4B
            // set: stats 2.04 -> 1.98 ms, finalize 65 -> 58 us)
            std::vector<std::pair<GroupKey, std::vector<int>>> ordered(groups.begin(), groups.end());
            if (phase == 2) {
                for (const auto& kv : ordered) {
                    const int64_t elems = group_elems(works, kv.second);
                    for (int t : kv.second) set_apply_steps(works[(size_t)t], elems);
                }
            }
            if (phase == 0) {
                for (const auto& kv : ordered) cut_stats(works, kv.second, part, part_cap, L.part_bytes);
                std::stable_sort(ordered.begin(), ordered.end(), [](const auto& a, const auto& b) {
                    return (a.first.fast == 2) > (b.first.fast == 2);
                });
                // inside a launch, tensors with the largest stats tiles first
                // and the smallest last, so the launch's last round of
                // workgroups, which leaves CUs idle, is one of short tiles
                for (auto& kv : ordered)
                    std::stable_sort(kv.second.begin(), kv.second.end(), [&](int a, int b) {
                        const TensorWork& wa = works[(size_t)a];
                        const TensorWork& wb = works[(size_t)b];
                        return (double)wa.N * (double)wb.stats_wgs > (double)wb.N * (double)wa.stats_wgs;
                    });
            }
            for (auto& kv : ordered) {
                Launch l;
                l.phase = phase;
                l.cohort = cohort;
                l.key = kv.first;
                l.seg_off = L.segs.size();
                l.nseg = (int)kv.second.size();
                l.wgs = 0;
                l.bytes = 0.0;
                for (int t : kv.second) {
                    const TensorWork& w = works[(size_t)t];
                    L.segs.push_back(Seg{t, 0, l.wgs});
                    const int64_t wgs = phase == 0 ? w.stats_wgs : phase == 1 ? w.fin_wgs
                                      : phase == 3 ? 1 : w.apply_wgs;
                    l.wgs += wgs;
                    const double es = (double)elem_size(w.dtype);
                    l.bytes += phase == 0 ? (double)w.N * (es + 1.0)
                             : phase == 1 ? 16.0 * (double)(w.R + w.C + w.nb)
                             : phase == 3 ? 8.0 * (double)w.nr : algo_bytes(w);
                }
                // coarse table: at most 4 entries per segment (+2)
                int gs = 0;
                while ((l.wgs >> gs) > 4 * (int64_t)l.nseg) ++gs;
                l.gshift = gs;
                l.coarse_off = L.coarse.size();
                const int64_t ncoarse = (l.wgs >> gs) + 2;
                int cur = 0;
                for (int64_t j = 0; j < ncoarse; ++j) {
                    const int64_t wgj = j << gs;
                    while (cur + 1 < l.nseg && L.segs[l.seg_off + (size_t)cur + 1].wg_begin <= wgj) ++cur;
                    L.coarse.push_back(cur);
                }
                L.launches.push_back(l);
            }
        }
        c0 = c1;
        ++cohort;
    }
}

// Byte offsets of the descriptor image [works | segments | coarse index] that
// the multi-tensor launches read from device memory.
struct MtImage {
    size_t works, segs, coarse, end;
};

static MtImage image_layout(const MtLayout& L, size_t base) {
    MtImage im;
    im.works = base;
    im.segs = im.works + align256(sizeof(TensorWork) * L.works.size());
    im.coarse = im.segs + align256(sizeof(Seg) * L.segs.size());
    im.end = im.coarse + align256(sizeof(int32_t) * L.coarse.size());
    return im;
}

static void write_image(const MtLayout& L, const MtImage& im, char* h) {
    std::memcpy(h + im.works, L.works.data(), sizeof(TensorWork) * L.works.size());
    std::memcpy(h + im.segs, L.segs.data(), sizeof(Seg) * L.segs.size());
    std::memcpy(h + im.coarse, L.coarse.data(), sizeof(int32_t) * L.coarse.size());
}

static int launch_layout(const MtLayout& L, char* dev, const MtImage& im, hipStream_t s, bool prof);

static int run_multi(const MtLayout& L, void* scratch, size_t scratch_bytes, hipStream_t s) {
    const MtImage im = image_layout(L, 0);
    const size_t need = im.end;
    if (scratch_bytes < need)
        return set_error(GEFENX_EINVAL, "gefenx_multi_tensor_step: scratch %zu bytes < required %zu", scratch_bytes, need);
    int dev = 0;
    hipGetDevice(&dev);
    {
        std::lock_guard<std::mutex> lk(g_stage_mu);
        Staging& st = g_stage[dev];
        const int b = st.next;
        st.next ^= 1;
        if (st.done[b] == nullptr && hipEventCreateWithFlags(&st.done[b], hipEventDisableTiming) != hipSuccess)
            return set_error(GEFENX_ELAUNCH, "gefenx_multi_tensor_step: event creation failed");
        if (st.host[b] != nullptr) hipEventSynchronize(st.done[b]);  // previous upload from this buffer finished
        if (st.cap[b] < need) {
            if (st.host[b]) hipHostFree(st.host[b]);
            st.host[b] = nullptr;
            st.cap[b] = 0;
            if (hipHostMalloc(&st.host[b], need, hipHostMallocDefault) != hipSuccess)
                return set_error(GEFENX_ENOMEM, "gefenx_multi_tensor_step: pinned staging of %zu bytes failed", need);
            st.cap[b] = need;
        }
        char* h = static_cast<char*>(st.host[b]);
        write_image(L, im, h);
        if (hipMemcpyAsync(scratch, h, need, hipMemcpyHostToDevice, s) != hipSuccess)
            return set_error(GEFENX_ELAUNCH, "gefenx_multi_tensor_step: descriptor upload failed");
        hipEventRecord(st.done[b], s);
    }
    return launch_layout(L, static_cast<char*>(scratch), im, s, true);
}

// Enqueue one phase launch of a layout whose descriptor image is at dev.
static int enqueue_launch(const Launch& l, char* dev, const MtImage& im, hipStream_t s, bool prof) {
    const TensorWork* dws = reinterpret_cast<const TensorWork*>(dev + im.works);
    const Seg* dsegs = reinterpret_cast<const Seg*>(dev + im.segs);
    const int32_t* dcoarse = reinterpret_cast<const int32_t*>(dev + im.coarse);
    {
        if (l.wgs <= 0) return GEFENX_OK;
        if (l.wgs > 2147483647LL) return set_error(GEFENX_EINVAL, "gefenx_multi_tensor_step: launch too large");
        const dim3 grid((unsigned)l.wgs), block(kThreads);
        const SegTable sg{dsegs + l.seg_off, dcoarse + l.coarse_off, l.nseg, l.gshift};
        const int kinds[4] = {GEFENX_K_STATS, GEFENX_K_FINALIZE, GEFENX_K_APPLY, GEFENX_K_FINALIZE};
        int kind = kinds[l.phase];
        if (l.key.mode == 1 && l.phase == 0) kind = GEFENX_K_BLOCK_STATS;
        if (l.key.mode == 1 && l.phase == 2) kind = GEFENX_K_BLOCK_APPLY;
        int ph = prof ? prof_begin(kind, l.bytes, 0.0, s) : -1;
        if (l.phase == 0) {
            with_dtype(l.key.dtype, [&](auto k) { k.mt_stats(l.key.mode, l.key.fast, grid, s, dws, sg); });
        } else if (l.phase == 3) {
            hipLaunchKernelGGL(k_mt_mean, grid, block, 0, s, dws, sg);
        } else if (l.phase == 1) {
            hipLaunchKernelGGL(k_mt_finalize, grid, block, 0, s, dws, sg);
        } else {
            with_dtype(l.key.dtype, [&](auto k) { k.mt_apply(l.key.mode, l.key.fast, l.key.sr, grid, s, dws, sg); });
        }
        prof_end(ph, s);
        int rc = launch_check("multi-tensor launch");
        if (rc) return rc;
    }
    return GEFENX_OK;
}

// Side stream and event pool of one device for the cohort pipeline (default
// priority; created on first use, kept for the process lifetime).
struct Pipe {
    hipStream_t side = nullptr;
    std::vector<hipEvent_t> ev;
};
static std::mutex g_pipe_mu;
static std::map<int, Pipe> g_pipe;

static int pipe_get(size_t n_events, Pipe*& out) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> lk(g_pipe_mu);
    Pipe& p = g_pipe[dev];
    if (p.side == nullptr && hipStreamCreateWithFlags(&p.side, hipStreamNonBlocking) != hipSuccess) {
        p.side = nullptr;
        return set_error(GEFENX_ELAUNCH, "gefenx_multi_tensor_step: side stream creation failed");
    }
    while (p.ev.size() < n_events) {
        hipEvent_t e = nullptr;
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess)
            return set_error(GEFENX_ELAUNCH, "gefenx_multi_tensor_step: event creation failed");
        p.ev.push_back(e);
    }
    out = &p;
    return GEFENX_OK;
}

// Enqueue the phase launches of L reading the descriptor image at dev.
// One cohort: everything on s in plan order.  Several: the stats, finalize
// and mean launches of every cohort go to the device's side stream, which
// first waits for all work enqueued on s so far; cohort k's applies wait on
// the event recorded after its mean launch, so the side stream runs the
// stats of later cohorts while s applies earlier ones.  s ends after the
// last apply, which follows every side-stream launch, so work enqueued on s
// afterwards sees the whole step.  Calls that overlap on one device must
// come from one host thread at a time (the side stream is shared).
static int launch_layout(const MtLayout& L, char* dev, const MtImage& im, hipStream_t s, bool prof) {
    const int n_cohorts = L.launches.empty() ? 0 : L.launches.back().cohort + 1;
    if (n_cohorts <= 1 || !pipeline_enabled()) {
        for (const Launch& l : L.launches) {
            int rc = enqueue_launch(l, dev, im, s, prof);
            if (rc) return rc;
        }
        return GEFENX_OK;
    }
    Pipe* pp = nullptr;
    int rc = pipe_get((size_t)n_cohorts + 1, pp);
    if (rc) return rc;
    hipStream_t side = pp->side;
    if (hipEventRecord(pp->ev[0], s) != hipSuccess || hipStreamWaitEvent(side, pp->ev[0], 0) != hipSuccess)
        return set_error(GEFENX_ELAUNCH, "gefenx_multi_tensor_step: stream fork failed");
    size_t i = 0;
    const size_t nl = L.launches.size();
    for (int c = 0; c < n_cohorts; ++c) {
        size_t j = i;
        for (; j < nl && L.launches[j].cohort == c; ++j)
            if (L.launches[j].phase != 2) {
                rc = enqueue_launch(L.launches[j], dev, im, side, prof);
                if (rc) return rc;
            }
        hipEvent_t ready = pp->ev[(size_t)c + 1];
        if (hipEventRecord(ready, side) != hipSuccess || hipStreamWaitEvent(s, ready, 0) != hipSuccess)
            return set_error(GEFENX_ELAUNCH, "gefenx_multi_tensor_step: cohort hand-off failed");
        for (size_t k = i; k < j; ++k)
            if (L.launches[k].phase == 2) {
                rc = enqueue_launch(L.launches[k], dev, im, s, prof);
                if (rc) return rc;
            }
        i = j;
    }
    return GEFENX_OK;
}

static size_t multi_scratch_bytes(int n_works, size_t n_segs) {
    // coarse tables: <= 4 entries per segment + 2 per launch, and every launch
    // holds at least one segment
    return align256(sizeof(TensorWork) * (size_t)n_works) + align256(sizeof(Seg) * n_segs) +
           align256(sizeof(int32_t) * 6 * n_segs);
}

// ------------------------------------------------------------ capturable plan

// Descriptor image upload as a kernel node: src is the plan's pinned host
// image (device-visible), dst the plan's device buffer; n 8-byte words.  The
// first n_works descriptors' partials become addresses in that buffer.
__global__ __launch_bounds__(kThreads) void k_image_copy(const uint64_t* __restrict__ src, uint64_t* __restrict__ dst,
                                                         int64_t n, int64_t n_works) {
    constexpr int64_t kWords = sizeof(TensorWork) / 8, kPart = offsetof(TensorWork, part) / 8;
    static_assert(sizeof(TensorWork) % 8 == 0 && offsetof(TensorWork, part) % 8 == 0, "whole words");
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
        uint64_t v = src[i];
        if (v != 0 && i < n_works * kWords && i % kWords == kPart) v += reinterpret_cast<uint64_t>(dst);
        dst[i] = v;
    }
}

__device__ __forceinline__ double capt_lr(const gefenx_capt_desc& c) {
    if (c.lr_dev == nullptr) return c.lr;
    switch (c.lr_dtype) {
        case F64: return *static_cast<const double*>(c.lr_dev);
        case F16: return (double)f16_to_f32(*static_cast<const uint16_t*>(c.lr_dev));
        case BF16: return (double)bf16_to_f32(*static_cast<const uint16_t*>(c.lr_dev));
        default: return (double)*static_cast<const float*>(c.lr_dev);
    }
}

// One thread per parameter: step counters += 1 (fp32, as torch's add_ on a
// 0-dim fp32 tensor), then the scalar row in float64 cast to fp32 --
// bc = 1 - beta^step, sqrt for the block path, reciprocal (the op chain of
// gefen.py:1984-1995).  lr: the device value when given (the weight-decay
// factor from its float64 value, gefen.py:1996-2001), else the host value
// (gefen.py:2003-2004).  Thread 0 also advances {global step, next seed,
// seed of this step}.
__global__ __launch_bounds__(kThreads) void k_capt_prologue(const gefenx_capt_desc* __restrict__ d, int n,
                                                            int64_t* __restrict__ counter) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i == 0 && counter != nullptr) {
        const int64_t seed = counter[1];
        counter[2] = seed;
        counter[1] = seed + 1;
        counter[0] = counter[0] + 1;
    }
    if (i >= n) return;
    const gefenx_capt_desc c = d[i];
    const float st = *c.step + 1.0f;
    *c.step = st;
    float st2 = st;
    if (c.bc2_step != nullptr) {
        st2 = *c.bc2_step + 1.0f;
        *c.bc2_step = st2;
    }
    double bc2 = 1.0 - pow(c.beta2, (double)st2);
    if (c.sqrt_bc2) bc2 = sqrt(bc2);
    const double bc1 = 1.0 - pow(c.beta1, (double)st);
    const double lr = capt_lr(c);
    c.scalars[0] = (float)lr;
    c.scalars[1] = (float)(1.0 / bc2);
    c.scalars[2] = (float)(1.0 / bc1);
    c.scalars[3] = c.weight_decay != 0.0 ? (float)(1.0 - lr * c.weight_decay) : 1.0f;
}

}  // namespace gx

// A fixed tensor set's descriptor image and launch list (include/gefenx.h).
struct gefenx_mt_plan {
    gx::MtLayout L;
    gx::MtImage im;
    size_t capt_off = 0;
    int n_capt = 0;
    int64_t* counter = nullptr;
    size_t image_bytes = 0;    // image and capturable descriptors
    size_t bytes = 0;          // of the device buffer
    int device = 0;
    void* host = nullptr;      // pinned image
    void* host_dev = nullptr;  // its device-visible address
    bool uploaded = false;     // an eager launch copied the image into uploaded_to on uploaded_on
    void* uploaded_to = nullptr;
    hipStream_t uploaded_on = nullptr;
};

using namespace gx;

static int check_dtype(int dtype, const char* fn) {
    if (dtype == F64)
        return set_error(GEFENX_EDTYPE, "%s: not implemented for 'Double' (fp32/fp16/bf16 only)", fn);
    if (dtype != F32 && dtype != F16 && dtype != BF16)
        return set_error(GEFENX_EINVAL, "%s: unknown dtype code %d", fn, dtype);
    return GEFENX_OK;
}

// ------------------------------------------------------------ static scratch
// Device scratch of gefenx_factored_update_noalloc: a file-scope array, one
// copy per GPU the library runs on, held until the process ends.  In host
// code the array's name is not a device address: scratch_on_device() resolves
// it once per device (hipGetSymbolAddress with that device current) and every
// host use -- kernel arguments, the clearing launch -- goes through the
// resolved pointer.
static __device__ __align__(256) unsigned char scratch[GEFENX_NOALLOC_SCRATCH_BYTES];
static_assert(kNoallocScratch == GEFENX_NOALLOC_SCRATCH_BYTES, "FactoredWs::make keeps tensors within it");

constexpr int kScratchDevices = 64;
static void* g_scratch_addr[kScratchDevices];  // per device; nullptr until resolved
static std::mutex g_scratch_mu;

static int scratch_on_device(void** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kScratchDevices)
        return set_error(GEFENX_ELAUNCH, "gefenx_factored_update_noalloc: no usable current device");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_addr[dev] == nullptr) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || ptr == nullptr)
            return set_error(GEFENX_ELAUNCH, "gefenx_factored_update_noalloc: hipGetSymbolAddress of the scratch "
                             "array failed on device %d: %s", dev, hipGetErrorString(e));
        g_scratch_addr[dev] = ptr;
    }
    *out = g_scratch_addr[dev];
    return GEFENX_OK;
}

// Zero n 32-bit words (a kernel, not a memset node, so a captured graph
// replays it like any other launch).
__global__ __launch_bounds__(kThreads) void k_zero_words(uint32_t* __restrict__ p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
        p[i] = 0u;
}

extern "C" {

// Validation and work description shared by the factored entry points.
static int factored_input(const char* fn, void* p, const void* grad, int dtype, int64_t rows, int64_t cols,
                          int64_t ps0, int64_t ps1, int64_t gs0, int64_t gs1, uint8_t* m_codebook,
                          float* m_magnitude, float* v_row, float* v_col, int64_t period, const void* qtable_dev,
                          double beta1, double beta2, double lr, double eps, double inv_bias_correction_2,
                          double inv_bias_correction_1, double weight_decay_factor, int stochastic_round,
                          int64_t rng_seed, const float* step_scalars, const int64_t* seed_dev, WorkInput& in,
                          bool& empty) {
    empty = false;
    int rc = check_dtype(dtype, fn);
    if (rc) return rc;
    if (rows < 0 || cols < 0) return set_error(GEFENX_EINVAL, "%s: negative shape", fn);
    const int64_t N = rows * cols;
    if (N == 0) {  // empty tensors are a no-op
        empty = true;
        return GEFENX_OK;
    }
    if (period <= 0 || N % period != 0)
        return set_error(GEFENX_EINVAL, "%s: period %lld does not divide numel %lld", fn, (long long)period,
                         (long long)N);
    if (!p || !grad || !m_codebook || !m_magnitude || !v_row || !v_col || !qtable_dev)
        return set_error(GEFENX_EINVAL, "%s: null pointer argument", fn);
    in = WorkInput{};
    in.p = p; in.grad = grad; in.dtype = dtype; in.mode = 0;
    in.R = rows; in.C = cols; in.ps0 = ps0; in.ps1 = ps1; in.gs0 = gs0; in.gs1 = gs1; in.period = period;
    in.idx = m_codebook; in.mag = m_magnitude; in.v0 = v_row; in.v1 = v_col; in.qt = qtable_dev;
    in.lerp_w = (float)(1.0 - beta1); in.beta2 = (float)beta2; in.alpha2 = (float)(1.0 - beta2);
    in.eps = (float)eps;
    in.sc = StepScalars{(float)lr, (float)inv_bias_correction_2, (float)inv_bias_correction_1,
                        (float)weight_decay_factor};
    in.bc2_div = reference_divisor(inv_bias_correction_2);
    in.sr = stochastic_round ? 1 : 0; in.seed = (uint64_t)rng_seed;
    in.step_scalars = step_scalars; in.seed_dev = seed_dev;
    return GEFENX_OK;
}

// Granules as workgroups of a single tensor's launch where they fit at mem.
static void cut_single(TensorWork& w, void* mem, size_t cap) {
    if (!wants_granules(w, w.N) || align256(sizeof(double) * (size_t)granules(w).doubles) > cap) return;
    (w.fast_stats == 2 ? w.row_part : w.col_part) = static_cast<double*>(mem);
    take_granules(w);
}

int gefenx_factored_update(
    void* p, const void* grad, int dtype, int64_t rows, int64_t cols,
    int64_t ps0, int64_t ps1, int64_t gs0, int64_t gs1,
    uint8_t* m_codebook, float* m_magnitude, float* v_row, float* v_col,
    int64_t period, const void* qtable_dev,
    double beta1, double beta2, double lr, double eps,
    double inv_bias_correction_2, double inv_bias_correction_1,
    double weight_decay_factor, int stochastic_round, int64_t rng_seed,
    const float* step_scalars, const int64_t* seed_dev,
    void* workspace, size_t workspace_bytes, void* stream) {
    WorkInput in;
    bool empty = false;
    int rc = factored_input("gefenx_factored_update", p, grad, dtype, rows, cols, ps0, ps1, gs0, gs1, m_codebook,
                            m_magnitude, v_row, v_col, period, qtable_dev, beta1, beta2, lr, eps,
                            inv_bias_correction_2, inv_bias_correction_1, weight_decay_factor, stochastic_round,
                            rng_seed, step_scalars, seed_dev, in, empty);
    if (rc || empty) return rc;
    if (!workspace) return set_error(GEFENX_EINVAL, "gefenx_factored_update: null workspace");
    in.workspace = workspace; in.ws_bytes = workspace_bytes;
    TensorWork w;
    rc = build_work(in, w);
    if (rc) return rc;
    const size_t need = gefenx_workspace_bytes(GEFENX_WS_FACTORED, rows, cols, w.nb);
    cut_single(w, static_cast<char*>(workspace) + need, workspace_bytes - need);
    return run_single(w, static_cast<hipStream_t>(stream));
}

int gefenx_factored_update_noalloc(
    void* p, const void* grad, int dtype, int64_t rows, int64_t cols,
    int64_t ps0, int64_t ps1, int64_t gs0, int64_t gs1,
    uint8_t* m_codebook, float* m_magnitude, float* v_row, float* v_col,
    int64_t period, const void* qtable_dev,
    double beta1, double beta2, double lr, double eps,
    double inv_bias_correction_2, double inv_bias_correction_1,
    double weight_decay_factor, int stochastic_round, int64_t rng_seed,
    const float* step_scalars, const int64_t* seed_dev, void* stream) {
    const char* fn = "gefenx_factored_update_noalloc";
    WorkInput in;
    bool empty = false;
    int rc = factored_input(fn, p, grad, dtype, rows, cols, ps0, ps1, gs0, gs1, m_codebook, m_magnitude, v_row,
                            v_col, period, qtable_dev, beta1, beta2, lr, eps, inv_bias_correction_2,
                            inv_bias_correction_1, weight_decay_factor, stochastic_round, rng_seed, step_scalars,
                            seed_dev, in, empty);
    if (rc || empty) return rc;
    const FactoredWs L = FactoredWs::make(rows, cols, rows * cols / period);
    if (L.total > (size_t)GEFENX_NOALLOC_SCRATCH_BYTES)
        return set_error(GEFENX_EINVAL, "%s: a [%lld, %lld] parameter with period %lld needs %zu bytes of scratch; "
                         "the static scratch holds %zu (use gefenx_factored_update with a workspace)", fn,
                         (long long)rows, (long long)cols, (long long)period, L.total,
                         (size_t)GEFENX_NOALLOC_SCRATCH_BYTES);
    void* ptr = nullptr;
    rc = scratch_on_device(&ptr);
    if (rc) return rc;
    in.workspace = ptr;
    in.ws_bytes = GEFENX_NOALLOC_SCRATCH_BYTES;
    TensorWork w;
    rc = build_work(in, w);
    if (rc) return rc;
    cut_single(w, static_cast<char*>(ptr) + L.total, (size_t)GEFENX_NOALLOC_SCRATCH_BYTES - L.total);
    // the accumulators that must start at zero: block maxima and the
    // finalize counter (the previous call on this GPU left them zero unless
    // it failed part-way)
    hipStream_t s = static_cast<hipStream_t>(stream);
    char* base = static_cast<char*>(ptr);
    const int64_t nmag = (int64_t)((L.off_magold - L.off_magbits) / sizeof(uint32_t));
    hipLaunchKernelGGL(k_zero_words, dim3((unsigned)std::min<int64_t>(1024, ceil_div(nmag, kThreads))),
                       dim3(kThreads), 0, s, reinterpret_cast<uint32_t*>(base + L.off_magbits), nmag);
    hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(kThreads), 0, s, reinterpret_cast<uint32_t*>(base + L.off_fin),
                       (int64_t)(256 / sizeof(uint32_t)));
    rc = launch_check(fn);
    if (rc) return rc;
    return run_single(w, s);
}

int gefenx_block_update(
    void* p, const void* grad, int dtype, int64_t numel, int64_t period,
    uint8_t* m_codebook, float* m_magnitude, float* vmean, const void* qtable_dev,
    double beta1, double beta2, double lr, double eps,
    double inv_sqrt_bias_correction_2, double inv_bias_correction_1,
    double weight_decay_factor, int stochastic_round, int64_t rng_seed,
    const float* step_scalars, const int64_t* seed_dev,
    void* workspace, size_t workspace_bytes, void* stream) {
    int rc = check_dtype(dtype, "gefenx_block_update");
    if (rc) return rc;
    if (numel < 0) return set_error(GEFENX_EINVAL, "gefenx_block_update: negative numel");
    if (numel == 0) return GEFENX_OK;
    if (period <= 0 || numel % period != 0)
        return set_error(GEFENX_EINVAL, "gefenx_block_update: period %lld does not divide numel %lld",
                         (long long)period, (long long)numel);
    if (!p || !grad || !m_codebook || !m_magnitude || !vmean || !qtable_dev || !workspace)
        return set_error(GEFENX_EINVAL, "gefenx_block_update: null pointer argument");
    WorkInput in{};
    in.p = p; in.grad = grad; in.dtype = dtype; in.mode = 1;
    in.R = 1; in.C = numel; in.ps0 = numel; in.ps1 = 1; in.gs0 = numel; in.gs1 = 1; in.period = period;
    in.idx = m_codebook; in.mag = m_magnitude; in.v0 = vmean; in.v1 = nullptr; in.qt = qtable_dev;
    in.lerp_w = (float)(1.0 - beta1); in.beta2 = (float)beta2; in.alpha2 = (float)(1.0 - beta2);
    in.eps = (float)eps;
    in.sc = StepScalars{(float)lr, (float)inv_sqrt_bias_correction_2, (float)inv_bias_correction_1,
                        (float)weight_decay_factor};
    in.bc2_div = reference_divisor(inv_sqrt_bias_correction_2);
    in.sr = stochastic_round ? 1 : 0; in.seed = (uint64_t)rng_seed;
    in.step_scalars = step_scalars; in.seed_dev = seed_dev;
    in.workspace = workspace; in.ws_bytes = workspace_bytes;
    TensorWork w;
    rc = build_work(in, w);
    if (rc) return rc;
    return run_single(w, static_cast<hipStream_t>(stream));
}

int gefenx_momentum_apply(
    void* p, const void* grad, int dtype, int64_t numel, int64_t period,
    uint8_t* m_codebook, float* m_magnitude, const float* stepsize, const void* qtable_dev,
    double beta1, double lr, void* workspace, size_t workspace_bytes, void* stream) {
    int rc = check_dtype(dtype, "gefenx_momentum_apply");
    if (rc) return rc;
    if (numel < 0) return set_error(GEFENX_EINVAL, "gefenx_momentum_apply: negative numel");
    if (numel == 0) return GEFENX_OK;
    if (period <= 0 || numel % period != 0)
        return set_error(GEFENX_EINVAL, "gefenx_momentum_apply: period %lld does not divide numel %lld",
                         (long long)period, (long long)numel);
    if (!p || !grad || !m_codebook || !m_magnitude || !stepsize || !qtable_dev || !workspace)
        return set_error(GEFENX_EINVAL, "gefenx_momentum_apply: null pointer argument");
    WorkInput in{};
    in.p = p; in.grad = grad; in.dtype = dtype; in.mode = 1;
    in.R = 1; in.C = numel; in.ps0 = numel; in.ps1 = 1; in.gs0 = numel; in.gs1 = 1; in.period = period;
    in.idx = m_codebook; in.mag = m_magnitude; in.v0 = nullptr; in.v1 = nullptr; in.qt = qtable_dev;
    in.lerp_w = (float)(1.0 - beta1); in.beta2 = 0.0f; in.alpha2 = 0.0f; in.eps = 0.0f;
    in.sc = StepScalars{(float)lr, 1.0f, 1.0f, 1.0f};
    in.workspace = workspace; in.ws_bytes = workspace_bytes;
    TensorWork w;
    rc = build_work(in, w);
    if (rc) return rc;
    w.partial = 1;
    w.step = const_cast<float*>(stepsize);  // read by the apply, never written in this mode
    return run_single(w, static_cast<hipStream_t>(stream));
}

static int desc_to_work(const gefenx_tensor_desc& d, int i, const void* const* qtables, int sr,
                        int64_t seed, const float* step_scalars, const int64_t* seed_dev, TensorWork& w) {
    int rc = check_dtype(d.dtype, "gefenx_multi_tensor_step");
    if (rc) return rc;
    const int64_t N = d.rows * d.cols;
    if (d.rows < 0 || d.cols < 0 || d.period <= 0 || N % d.period != 0)
        return set_error(GEFENX_EINVAL, "gefenx_multi_tensor_step: descriptor %d has period %lld not dividing [%lld, %lld]",
                         i, (long long)d.period, (long long)d.rows, (long long)d.cols);
    if (!d.p || !d.grad || !d.m_codebook || !d.m_magnitude || !d.v0 || (d.factored && !d.v1) || !d.workspace)
        return set_error(GEFENX_EINVAL, "gefenx_multi_tensor_step: descriptor %d has a null pointer", i);
    const void* qt = qtables[d.dtype];
    if (!qt) return set_error(GEFENX_EINVAL, "gefenx_multi_tensor_step: no quantisation table for dtype %d", d.dtype);
    WorkInput in{};
    in.p = d.p; in.grad = d.grad; in.dtype = d.dtype; in.mode = d.factored ? 0 : 1;
    if (d.factored) {
        in.R = d.rows; in.C = d.cols; in.ps0 = d.ps0; in.ps1 = d.ps1; in.gs0 = d.gs0; in.gs1 = d.gs1;
    } else if (d.rows <= 1 || (d.ps1 == 1 && d.gs1 == 1 && d.ps0 == d.cols && d.gs0 == d.cols)) {
        in.R = 1; in.C = N; in.ps0 = N; in.ps1 = 1; in.gs0 = N; in.gs1 = 1;  // contiguous: flat
    } else {
        in.R = d.rows; in.C = d.cols; in.ps0 = d.ps0; in.ps1 = d.ps1; in.gs0 = d.gs0; in.gs1 = d.gs1;
    }
    in.period = d.period;
    in.idx = d.m_codebook; in.mag = d.m_magnitude; in.v0 = d.v0; in.v1 = d.v1; in.qt = qt;
    in.lerp_w = d.lerp_w; in.beta2 = d.beta2; in.alpha2 = d.alpha2; in.eps = d.eps;
    in.bc2_div = d.bc2_div;
    in.sc = StepScalars{d.lr, d.inv_bc2, d.inv_bc1, d.wd_factor};
    in.sr = sr ? 1 : 0; in.seed = (uint64_t)seed;
    in.step_scalars = step_scalars; in.seed_dev = seed_dev;
    in.workspace = d.workspace;
    in.ws_bytes = d.factored ? gefenx_workspace_bytes(GEFENX_WS_FACTORED, d.rows, d.cols, N / d.period)
                             : gefenx_workspace_bytes(GEFENX_WS_BLOCK, d.rows, d.cols, N / d.period);
    return build_work(in, w);
}

// Tensors of the HOT apply join the launch of the others (which takes every
// tensor, some 8% slower) where they are few: a launch of their own costs ~5 us.
static void merge_small_applies(std::vector<TensorWork>& works) {
    for (int dt : {F32, F16, BF16}) {
        int64_t hot = 0, any = 0;
        for (const TensorWork& w : works)
            if (w.dtype == dt) (w.fast_apply == 1 ? hot : any) += (w.fast_apply & 1) ? w.N : 0;
        if (any == 0 || hot > kMergeApplyElems) continue;
        for (TensorWork& w : works)
            if (w.dtype == dt && w.fast_apply == 1) w.fast_apply = 3;
    }
}

static int build_works(const gefenx_tensor_desc* descs, int n, const void* const* qtables, int sr, int64_t seed,
                       const float* const* step_scalars, const int64_t* seed_dev, std::vector<TensorWork>& works) {
    if (n < 0 || (n > 0 && (!descs || !qtables)))
        return set_error(GEFENX_EINVAL, "gefenx_multi_tensor_step: bad descriptor array");
    works.reserve((size_t)n);
    for (int i = 0; i < n; ++i) {
        if (descs[i].rows * descs[i].cols == 0) continue;  // empty tensors are a no-op
        TensorWork w;
        int rc = desc_to_work(descs[i], i, qtables, sr, seed, step_scalars ? step_scalars[i] : nullptr, seed_dev, w);
        if (rc) return rc;
        works.push_back(w);
    }
    merge_small_applies(works);
    return GEFENX_OK;
}

size_t gefenx_multi_tensor_scratch_bytes(int n) {
    if (n <= 0) return 256;
    // each tensor is one segment of one launch per phase (4 phases)
    return multi_scratch_bytes(n, (size_t)n * 4);
}

size_t gefenx_multi_tensor_scratch_bytes_for(const gefenx_tensor_desc* descs, int n) {
    const size_t base = gefenx_multi_tensor_scratch_bytes(n);
    if (n <= 0 || !descs) return base;
    // the stats launches of these tensors, from what decides their cut (views of
    // the block path leave no partials)
    std::vector<TensorWork> works;
    std::map<GroupKey, std::vector<int>> groups;
    size_t used = 0;
    int64_t largest = 0;
    for (int i = 0; i < n; ++i) largest = std::max<int64_t>(largest, descs[i].rows * descs[i].cols);
    if (largest <= kFactGranuleElems) return base;  // a granule each
    works.reserve((size_t)n);
    for (int i = 0; i < n; ++i) {
        const gefenx_tensor_desc& d = descs[i];
        if (d.rows <= 0 || d.cols <= 0 || d.period <= 0 || (d.rows * d.cols) % d.period != 0) continue;
        TensorWork w;
        std::memset(&w, 0, sizeof(w));
        w.R = d.rows; w.C = d.cols; w.P = d.period; w.N = d.rows * d.cols;
        w.gs0 = d.gs0; w.gs1 = d.gs1; w.grad = d.grad; w.idx = d.m_codebook;
        w.dtype = d.dtype; w.mode = d.factored ? 0 : 1;
        if (d.factored) {
            set_factored_stats(w, FactoredWs::make(d.rows, d.cols, w.N / d.period).tiles);
        } else if (d.rows > 1 && view_strides(d.rows, d.gs0, d.gs1, d.dtype, d.grad)) {
            w.fast_stats = 2;
            set_tiles(w, FactTiles::make(d.rows, d.cols, d.period, false).tv);
        }
        works.push_back(w);
    }
    for (int c0 = 0; c0 < (int)works.size();) {
        const int c1 = cohort_end(works, c0);
        groups.clear();
        for (int t = c0; t < c1; ++t) groups[stats_key(works[(size_t)t])].push_back(t);
        for (const auto& kv : groups) cut_stats(works, kv.second, 256, kGranuleBytes, used);
        c0 = c1;
    }
    return base + used;
}

int gefenx_multi_tensor_step(const gefenx_tensor_desc* descs, int n, const void* const* qtables_dev,
                             int stochastic_round, int64_t rng_seed, void* desc_scratch_dev,
                             size_t desc_scratch_bytes, void* stream) {
    std::vector<TensorWork> works;
    int rc = build_works(descs, n, qtables_dev, stochastic_round, rng_seed, nullptr, nullptr, works);
    if (rc) return rc;
    if (works.empty()) return GEFENX_OK;
    if (!desc_scratch_dev) return set_error(GEFENX_EINVAL, "gefenx_multi_tensor_step: null scratch");
    const size_t base = gefenx_multi_tensor_scratch_bytes(n);
    MtLayout L;
    plan_multi(works, reinterpret_cast<uintptr_t>(desc_scratch_dev) + base,
               desc_scratch_bytes > base ? std::min(desc_scratch_bytes - base, kGranuleBytes) : 0, L);
    return run_multi(L, desc_scratch_dev, desc_scratch_bytes, static_cast<hipStream_t>(stream));
}

int gefenx_mt_plan_create(const gefenx_tensor_desc* descs, int n, const float* const* step_scalars,
                          const void* const* qtables_dev, int stochastic_round, int64_t rng_seed,
                          const gefenx_capt_desc* capt, int n_capt, int64_t* counter_dev,
                          gefenx_mt_plan** plan_out) {
    if (!plan_out) return set_error(GEFENX_EINVAL, "gefenx_mt_plan_create: null plan_out");
    *plan_out = nullptr;
    if (n_capt < 0 || (n_capt > 0 && !capt))
        return set_error(GEFENX_EINVAL, "gefenx_mt_plan_create: bad capturable descriptor array");
    for (int i = 0; i < n_capt; ++i) {
        const gefenx_capt_desc& c = capt[i];
        if (!c.step || !c.scalars)
            return set_error(GEFENX_EINVAL, "gefenx_mt_plan_create: capturable descriptor %d has a null pointer", i);
        if (c.lr_dev && (c.lr_dtype < GEFENX_F32 || c.lr_dtype > GEFENX_F64))
            return set_error(GEFENX_EINVAL, "gefenx_mt_plan_create: capturable descriptor %d: lr dtype code %d", i,
                             c.lr_dtype);
    }
    const int64_t* seed_dev = counter_dev ? counter_dev + 2 : nullptr;
    auto plan = std::make_unique<gefenx_mt_plan>();
    std::vector<TensorWork> works;
    int rc = build_works(descs, n, qtables_dev, stochastic_round, rng_seed, step_scalars, seed_dev, works);
    if (rc) return rc;
    // [image | capturable descriptors | granule partials]
    const size_t capt_bytes = align256(sizeof(gefenx_capt_desc) * (size_t)n_capt);
    const size_t part_off = gefenx_multi_tensor_scratch_bytes(n) + capt_bytes;
    plan_multi(works, part_off, kGranuleBytes, plan->L);
    plan->im = image_layout(plan->L, 0);
    plan->capt_off = plan->im.end;
    plan->n_capt = n_capt;
    plan->counter = counter_dev;
    (void)hipGetDevice(&plan->device);
    plan->image_bytes = std::max<size_t>(plan->capt_off + capt_bytes, 256);
    plan->bytes = plan->L.part_bytes > 0 ? part_off + plan->L.part_bytes : plan->image_bytes;
    // Pinned allocation is host work; let it through while this thread's
    // stream is being captured.
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    const hipError_t e = hipHostMalloc(&plan->host, plan->image_bytes, hipHostMallocDefault);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) {
        plan->host = nullptr;
        return set_error(GEFENX_ENOMEM, "gefenx_mt_plan_create: pinned image of %zu bytes failed", plan->image_bytes);
    }
    if (hipHostGetDevicePointer(&plan->host_dev, plan->host, 0) != hipSuccess) {
        (void)hipHostFree(plan->host);
        plan->host = nullptr;
        return set_error(GEFENX_ELAUNCH, "gefenx_mt_plan_create: pinned image has no device address");
    }
    char* h = static_cast<char*>(plan->host);
    std::memset(h, 0, plan->image_bytes);
    write_image(plan->L, plan->im, h);
    if (n_capt > 0) std::memcpy(h + plan->capt_off, capt, sizeof(gefenx_capt_desc) * (size_t)n_capt);
    *plan_out = plan.release();
    return GEFENX_OK;
}

size_t gefenx_mt_plan_device_bytes(const gefenx_mt_plan* plan) { return plan ? plan->bytes : 0; }

int gefenx_mt_plan_launch(gefenx_mt_plan* plan, void* dev_buf, size_t dev_bytes, void* stream) {
    if (!plan || !dev_buf) return set_error(GEFENX_EINVAL, "gefenx_mt_plan_launch: null plan or buffer");
    if (dev_bytes < plan->bytes)
        return set_error(GEFENX_EINVAL, "gefenx_mt_plan_launch: buffer %zu bytes < required %zu", dev_bytes,
                         plan->bytes);
    if (reinterpret_cast<uintptr_t>(dev_buf) % 256 != 0)
        return set_error(GEFENX_EINVAL, "gefenx_mt_plan_launch: buffer not 256-byte aligned");
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cs) != hipSuccess)
        return set_error(GEFENX_ELAUNCH, "gefenx_mt_plan_launch: stream capture query failed");
    const bool capturing = cs != hipStreamCaptureStatusNone;
    const dim3 block(kThreads);
    if (capturing || !plan->uploaded || plan->uploaded_to != dev_buf || plan->uploaded_on != s) {
        const int64_t n8 = (int64_t)(plan->image_bytes / 8);
        const unsigned grid = (unsigned)std::min<int64_t>((n8 + kThreads - 1) / kThreads, 1024);
        hipLaunchKernelGGL(k_image_copy, dim3(grid), block, 0, s, static_cast<const uint64_t*>(plan->host_dev),
                           static_cast<uint64_t*>(dev_buf), n8, (int64_t)plan->L.works.size());
        int rc = launch_check("plan image copy");
        if (rc) return rc;
        if (!capturing) {
            plan->uploaded = true;
            plan->uploaded_to = dev_buf;
            plan->uploaded_on = s;
        }
    }
    char* dev = static_cast<char*>(dev_buf);
    if (plan->n_capt > 0 || plan->counter != nullptr) {
        const unsigned grid = (unsigned)std::max(1, (plan->n_capt + kThreads - 1) / kThreads);
        hipLaunchKernelGGL(k_capt_prologue, dim3(grid), block, 0, s,
                           reinterpret_cast<const gefenx_capt_desc*>(dev + plan->capt_off), plan->n_capt,
                           plan->counter);
        int rc = launch_check("capturable prologue");
        if (rc) return rc;
    }
    if (plan->L.works.empty()) return GEFENX_OK;
    return launch_layout(plan->L, dev, plan->im, s, !capturing);
}

void gefenx_mt_plan_destroy(gefenx_mt_plan* plan) {
    if (!plan) return;
    if (plan->host) {
        // the last launch's image copy may still be reading the pinned image
        int cur = 0;
        (void)hipGetDevice(&cur);
        (void)hipSetDevice(plan->device);
        (void)hipDeviceSynchronize();
        (void)hipHostFree(plan->host);
        (void)hipSetDevice(cur);
    }
    delete plan;
}

}  // extern "C"
