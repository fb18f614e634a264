// gefenx_common.h -- shared host/device definitions of the MI355X Gefen step.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace gx {

enum DType : int { F32 = 0, F16 = 1, BF16 = 2, F64 = 3 };

constexpr int kCodebookMax = 256;
constexpr int kBuckets = 4096;        // bucket index over [-1, 1] (2^12)
constexpr int kLutEntries = kBuckets + 1;
constexpr int kFqEntries = kBuckets + 8;  // fast-quantiser entries incl. padding (x = 1 lands in 4096)

// Byte image of the quantisation table (gefenx_qtable_build).  Plain data,
// copied verbatim to device memory; kernels stage the parts they need in LDS.
struct QTable {
    int32_t k;                       // codebook size (1..256)
    int32_t dtype;                   // grad dtype the dequant table rounds through
    int32_t n_thr;                   // k - 1 decision thresholds
    int32_t max_cnt;                 // most thresholds falling in one bucket
    float cb[kCodebookMax];          // raw fp32 codebook (padded with its last entry)
    float cbr[kCodebookMax];         // codebook rounded through the grad dtype
    float thr[kCodebookMax];         // thr[i] = largest x in [-1,1] with nearest(x) <= i
    uint32_t bucket[kBuckets];       // base | (count << 16) of thresholds per bucket
    int16_t lut[kLutEntries + 7];    // reference search LUT (stochastic rounding)
    // Fast quantiser, one 8-byte entry per bucket: {bits of thr[base], base}.
    // When no bucket holds more than one threshold (max_cnt <= 1) the nearest
    // index of x in bucket b is base + (thr[base] < x).
    uint32_t fq[2 * kFqEntries];
};

static_assert(sizeof(QTable) % 16 == 0, "QTable must stay 16-byte aligned in size");

// Workspace layouts (all sub-arrays 256-byte aligned).  Accumulators are
// zero on entry and left zero on exit by the finalize kernels.
inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// Factored stats tiling: a workgroup covers kFactTileCols columns (64 lanes x
// two 8-column chunks) of `tile_rows` consecutive rows.  A tile's size has two
// bounds.  Per tensor: about N/32 elements, between 64K and 1M (in a launch of
// billions of elements larger tiles spend less of the pass on set-up and
// flushes: on the Llama-3-8B set caps of 256K / 512K / 1M / 2M measured
// 4.30 / 4.08 / 3.97 / 3.96 ms).  Per launch: launch_elems / kFactLaunchWgs,
// so that a launch of any size fills the 256 CUs' four workgroups each (the
// LDS of a workgroup allows four); with N/32 alone a single tensor is 32
// workgroups and a decoder layer 298, one wave per SIMD and most of the chip
// idle.  Not below kFactTileSmallElems, where a tile's set-up and its column
// partials cost more than the waves it adds.  Measured (stats kernel, us;
// N/32 alone -> launch_elems / 512, / 1024, / 2048 with 16K): one decoder
// layer (218M bf16) 282 -> 154, 129, 136; 4096x4096 fp32 140 -> 28, 30, 35;
// 43M fp16 elements in odd sizes 470 -> 57, 46, 47; 7.5M bf16 in 8 matrices
// 258 -> 76, 75, 75.
// Tiles start at multiples of 32 rows, so the rows whose squares meet in one
// fp32 column partial are the same in every launch; the launch decides the
// order of the float64 additions of those partials only.
constexpr int64_t kFactTileCols = 1024;
constexpr int64_t kFactTileMinElems = 1 << 16;
constexpr int64_t kFactTileMaxElems = 1 << 20;
constexpr int64_t kFactTileSmallElems = 1 << 14;
constexpr int64_t kFactLaunchWgs = 1024;

// Contiguous matrices (C >= 8) of at most kNarrowMaxCols columns, or with
// blocks shorter than kShortPeriod, take tiles of up to kLaneTileCols columns
// (stats_lanes): with few columns a 1024-column tile leaves lanes idle, and
// with short blocks nearly every 1024-column row segment holds block borders.
constexpr int64_t kNarrowMaxCols = 256;
constexpr int64_t kShortPeriod = 1024;
constexpr int64_t kLaneTileCols = 512;
inline bool lane_tiles(int64_t cols, int64_t period) {
    return cols >= 8 && (cols <= kNarrowMaxCols || (period < kShortPeriod && period < cols));
}

// As launch_elems: the largest tiles whatever the launch, for the scratch of
// fixed size.  Short blocks of wide matrices then stay on 1024-column tiles: the
// twice as many row partials of the lane tiles would take shapes out of it
// (21920 x 21920 in 512-element blocks 30.3 -> 34.0 MB of 33.6).
constexpr int64_t kCoarseTiles = (int64_t)1 << 62;

// Transposed-view stats (strides (1, ld)): tiles of up to four 64-row bands,
// one for each wave of the workgroup, and a multiple of 64 columns, half as
// many elements as the contiguous tiles (a wave walks its columns one 64 x 64
// tile at a time, with nothing else in flight: on 51M elements of a decoder
// layer 1024-column tiles 59 us, the share of 1/1024 of the launch 42 us, of
// 1/2048 37 us).
constexpr int64_t kTvStatsMaxRows = 256;

struct FactTiles {
    int64_t ct, rt, tile_rows;                            // 1024-column tiles
    int64_t ct_l, rt_l, l_rows, l_cols, lg_lanes;         // lane tiles (lg_lanes: log2 lanes per row; -1: not taken)
    int64_t ct_tv, rt_tv, tv_rows, tv_cols;               // transposed-view tiles
    // launch_elems: elements of all tensors of the launch (>= rows * cols)
    static FactTiles make(int64_t rows, int64_t cols, int64_t period, int64_t launch_elems) {
        FactTiles t;
        const auto ceil_div = [](int64_t x, int64_t d) { return x > 0 ? (x + d - 1) / d : 1; };
        int64_t elems = rows * cols / 32;
        elems = elems < kFactTileMinElems ? kFactTileMinElems : (elems > kFactTileMaxElems ? kFactTileMaxElems : elems);
        int64_t share = launch_elems / kFactLaunchWgs;
        if (share < kFactTileSmallElems) share = kFactTileSmallElems;
        if (elems > share) elems = share;
        // rows of a tile of `width` columns: whole 8-row fp32 column groups of
        // each wave (lane tiles: of each lane), `gran` rows together
        const auto tile_rows = [&](int64_t width, int64_t gran) {
            const int64_t w = cols < width ? (cols < 1 ? 1 : cols) : width;
            int64_t r = ceil_div(ceil_div(elems, w), gran) * gran;
            if (r > rows) r = rows;
            return r < 1 ? 1 : r;
        };
        t.ct = ceil_div(cols, kFactTileCols);
        t.tile_rows = tile_rows(kFactTileCols, 32);
        t.rt = ceil_div(rows, t.tile_rows);
        t.lg_lanes = -1;
        t.ct_l = t.rt_l = 0;
        t.l_rows = t.l_cols = 0;
        if (lane_tiles(cols, period) && (cols <= kNarrowMaxCols || launch_elems < kCoarseTiles)) {
            t.l_cols = (ceil_div(cols, ceil_div(cols, kLaneTileCols)) + 7) & ~int64_t(7);  // even column tiles
            t.lg_lanes = 0;
            while ((8 << t.lg_lanes) < t.l_cols) ++t.lg_lanes;
            t.ct_l = ceil_div(cols, t.l_cols);
            t.l_rows = tile_rows(t.l_cols, 32 * (64 >> t.lg_lanes));
            t.rt_l = ceil_div(rows, t.l_rows);
        }
        t.tv_rows = rows < 1 ? 1 : (rows < kTvStatsMaxRows ? rows : kTvStatsMaxRows);
        t.rt_tv = ceil_div(rows, t.tv_rows);
        const int64_t vc = (share / (2 * kTvStatsMaxRows) + 63) & ~int64_t(63);
        t.tv_cols = vc < 64 ? 64 : vc > kFactTileCols ? kFactTileCols : vc;
        t.ct_tv = ceil_div(cols, t.tv_cols);
        return t;
    }
};

// Block-max (and block-path sum-of-squares) accumulators are sharded when
// there are few blocks: workgroup w folds into shard (w % shards), so one huge
// block is not a single atomic hot spot; the finalize kernels reduce the
// shards in a fixed order.
constexpr int64_t kMagShardMaxBlocks = 4096;
constexpr int64_t kMagShards = 32;
inline int64_t mag_shards(int64_t nb) { return nb <= kMagShardMaxBlocks ? kMagShards : 1; }

// Rows of v_row handled per finalize workgroup (one float64 partial of
// sum(v_row) each; the apply kernel adds the partials in a fixed order).
constexpr int64_t kFinRowsPerWg = 256;

struct FactoredWs {
    // double row_part[max of the tilings' ct][rows], double col_part[max rt][cols] (per-tile
    // partial sums, fully rewritten every step; launch_elems = rows * cols sizes them for the
    // smallest tiles, so one workspace serves the tensor in every launch), uint32 magbits[shards][nb] (zero
    // between steps), float mag_old[nb], float minv[nb],
    // double vrow_sum[ceil(rows/256)] (partials of sum(v_row)), float vcs[cols] (sqrt(v_col)),
    // {uint32 finalize counter (zero between steps), float mean(v_row)}
    size_t off_rowp, off_colp, off_magbits, off_magold, off_minv, off_vsum, off_vcs, off_fin, total;
    static FactoredWs make(int64_t rows, int64_t cols, int64_t nb, int64_t launch_elems) {
        FactoredWs w;
        const FactTiles t = FactTiles::make(rows, cols, nb > 0 ? rows * cols / nb : 1, launch_elems);
        size_t o = 0;
        // any of the three tilings fits
        const auto max3 = [](int64_t x, int64_t y, int64_t z) { return x > y ? (x > z ? x : z) : (y > z ? y : z); };
        const int64_t ct = max3(t.ct, t.ct_l, t.ct_tv), rt = max3(t.rt, t.rt_l, t.rt_tv);
        w.off_rowp = o;    o += align256(sizeof(double) * (size_t)(ct * rows));
        w.off_colp = o;    o += align256(sizeof(double) * (size_t)(rt * cols));
        w.off_magbits = o; o += align256(sizeof(uint32_t) * (size_t)(nb * mag_shards(nb)));
        w.off_magold = o;  o += align256(sizeof(float) * (size_t)nb);
        w.off_minv = o;    o += align256(sizeof(float) * (size_t)nb);
        w.off_vsum = o;    o += align256(sizeof(double) * (size_t)((rows + kFinRowsPerWg - 1) / kFinRowsPerWg));
        w.off_vcs = o;     o += align256(sizeof(float) * (size_t)cols);
        w.off_fin = o;     o += 256;
        w.total = o;
        return w;
    }
};

// Block stats record of one workgroup: the sums of squares of its first and
// last block (key -1: none), which may continue in neighbouring workgroups.
struct DetRec {
    int64_t kf;
    double sf;
    int64_t kl;
    double sl;
};

// Elements per workgroup of the block stats with one element per item (the
// smallest geometry, so it bounds the record count).
constexpr int64_t kBlockStatsMinElems = 8 * 256;

struct BlockWs {
    // double blk_sq[shards][nb] (zero between steps), uint32
    // magbits[shards][nb] (zero between steps), float mag_old[nb], float
    // step[nb], float minv[nb], DetRec rec[ceil(numel / kBlockStatsMinElems)]
    size_t off_sq, off_magbits, off_magold, off_step, off_minv, off_rec, total;
    static BlockWs make(int64_t nb, int64_t numel) {
        BlockWs w;
        size_t o = 0;
        w.off_sq = o;      o += align256(sizeof(double) * (size_t)(nb * mag_shards(nb)));
        w.off_magbits = o; o += align256(sizeof(uint32_t) * (size_t)(nb * mag_shards(nb)));
        w.off_magold = o;  o += align256(sizeof(float) * (size_t)nb);
        w.off_step = o;    o += align256(sizeof(float) * (size_t)nb);
        w.off_minv = o;    o += align256(sizeof(float) * (size_t)nb);
        w.off_rec = o;     o += align256(sizeof(DetRec) * (size_t)((numel + kBlockStatsMinElems - 1) /
                                                                   kBlockStatsMinElems));
        w.total = o;
        return w;
    }
};

struct MomentumWs {
    size_t off_magbits, off_magold, off_minv, total;
    static MomentumWs make(int64_t nb) {
        MomentumWs w;
        size_t o = 0;
        w.off_magbits = o; o += align256(sizeof(uint32_t) * (size_t)(nb * mag_shards(nb)));
        w.off_magold = o;  o += align256(sizeof(float) * (size_t)nb);
        w.off_minv = o;    o += align256(sizeof(float) * (size_t)nb);
        w.total = o;
        return w;
    }
};

}  // namespace gx
