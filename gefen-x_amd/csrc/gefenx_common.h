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

// Factored stats tiling.  A tensor's sums of squares are added up in an order
// that its shape and block length alone decide, whatever else the call holds:
// fp32 over 8 rows (float64 for fp32 grads), four such values to a granule,
// granules in order to a tile, tiles in order to the total.  Granules and tiles
// are rows of a column tile (transposed views: columns of a row band).
// How the launch is cut is another matter: a workgroup takes a tile, or, where
// that would leave CUs idle, a granule, whose sum then goes to scratch of the
// call and which finalize adds up in the same order.
//   tiles: about N/32 elements, between 64K and 1M.  In a launch of billions of
// elements large ones spend less of the pass on set-up and flushes (on the
// Llama-3-8B set caps of 256K / 512K / 1M / 2M measured 4.30 / 4.08 / 3.97 /
// 3.96 ms), and their sums are what stays resident per tensor.
//   granules: multiples of 32 rows (each of the 4 waves 8), at least 8K elements,
// as many as leave a tensor at most kFactGranules of them, the workgroups that the
// CUs hold: a second round of a few costs as much as the first (11008 x 4096 in
// 256-element blocks, stats kernel: 920 workgroups 59.9 us, 1376 of them 69.7; in
// rows as blocks 688 of them 36.9, 460 45.4).  A workgroup on a tile meets after
// each (about 2 us: twenty of 4096 x 4096 in 32 rows 239 us against 201 without),
// so 1024-column tiles take 128 rows where that leaves kFactGranulesOf128 of them
// (the Llama-3-8B set's step 15.89 ms against 16.08 in 64 rows).
// Tiles hold equal numbers of them (14336 x 4096 in 1024 rows against 1056 and a
// short last tile: 3% of the stats of twelve).
constexpr int64_t kFactTileCols = 1024;
constexpr int64_t kFactTileMinElems = 1 << 16;
constexpr int64_t kFactTileMaxElems = 1 << 20;
constexpr int64_t kFactGranules = 1024;
constexpr int64_t kFactGranulesOf128 = 448;
constexpr int64_t kFactGranuleElems = 1 << 13;

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

// Transposed-view stats (strides (1, ld)): bands of up to 256 rows, 64 for each
// wave of the workgroup, tiles of 1024 columns, granules of 64 to 512.  A wave
// walks its columns one 64 x 64 tile at a time, with nothing else in flight, so
// half as large a share of the launch as for the contiguous tiles is the faster
// one (on 51M elements of a decoder layer 1024-column tiles 59 us, 1/1024 of the
// launch 42 us, 1/2048 37 us).  Not below 16K elements: with few rows, one
// finalize workgroup adds up all partials of a row (16 x 100000 in 64 columns
// 154 us a step against 88 in 1024).  The block path leaves no such partials and
// takes 64 columns there (49 against 92).
constexpr int64_t kTvStatsMaxRows = 256;
constexpr int64_t kTvGranules = 512;

struct Tiling {
    int64_t ct, rt;      // tiles: columns, rows
    int64_t rows, cols;  // of a tile
    int64_t gran, ng;    // granule: rows (views: columns) and count
};

struct FactTiles {
    Tiling wide, lane, tv;  // 1024-column tiles, lane tiles, transposed views
    int64_t lg_lanes;       // lane tiles: log2 lanes per row; -1: not taken
    static FactTiles make(int64_t rows, int64_t cols, int64_t period, bool factored = true) {
        FactTiles t;
        const auto ceil_div = [](int64_t x, int64_t d) { return x > 0 ? (x + d - 1) / d : 1; };
        const int64_t N = rows * cols;
        int64_t elems = N / 32;
        elems = elems < kFactTileMinElems ? kFactTileMinElems : (elems > kFactTileMaxElems ? kFactTileMaxElems : elems);
        // tiles of `width` columns; `unit` rows hold 8 rows of every wave (lane tiles: of every lane)
        const auto tiling = [&](int64_t width, int64_t unit) {
            Tiling q;
            const int64_t w = cols < width ? (cols < 1 ? 1 : cols) : width;
            q.gran = unit;
            while (q.gran * w < kFactGranuleElems) q.gran *= 2;
            q.gran *= ceil_div(N, kFactGranules * q.gran * w);
            if (width == kFactTileCols && q.gran < 128 && N >= kFactGranulesOf128 * 128 * w) q.gran = 128;
            q.cols = width;
            q.ct = ceil_div(cols, width);
            q.ng = ceil_div(rows, q.gran);
            q.rt = ceil_div(q.ng, ceil_div(elems, q.gran * w));
            q.rows = ceil_div(q.ng, q.rt) * q.gran;
            q.rt = ceil_div(rows, q.rows);
            if (q.rows > rows) q.rows = rows < 1 ? 1 : rows;
            return q;
        };
        t.wide = tiling(kFactTileCols, 32);
        t.lg_lanes = -1;
        t.lane = Tiling{};
        if (lane_tiles(cols, period)) {
            const int64_t width = (ceil_div(cols, ceil_div(cols, kLaneTileCols)) + 7) & ~int64_t(7);  // even column tiles
            t.lg_lanes = 0;
            while ((8 << t.lg_lanes) < width) ++t.lg_lanes;
            t.lane = tiling(width, 32 * (64 >> t.lg_lanes));
        }
        t.tv.rows = rows < 1 ? 1 : (rows < kTvStatsMaxRows ? rows : kTvStatsMaxRows);
        t.tv.rt = ceil_div(rows, t.tv.rows);
        t.tv.cols = kFactTileCols;
        t.tv.ct = ceil_div(cols, kFactTileCols);
        t.tv.gran = 64;
        while (t.tv.gran < kFactTileCols &&
               ((factored && t.tv.rows * t.tv.gran < kFactGranuleElems) || 2 * t.tv.rows * t.tv.gran <= N / kTvGranules))
            t.tv.gran *= 2;
        t.tv.ng = ceil_div(cols, t.tv.gran);
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

// Static scratch of gefenx_factored_update_noalloc.
constexpr size_t kNoallocScratch = (size_t)32 << 20;

struct FactoredWs {
    // double row_part[most ct of the tilings][rows], double col_part[most rt][cols] (per-tile
    // partial sums, fully rewritten every step), uint32 magbits[shards][nb] (zero
    // between steps), float mag_old[nb], float minv[nb],
    // double vrow_sum[ceil(rows/256)] (partials of sum(v_row)), float vcs[cols] (sqrt(v_col)),
    // {uint32 finalize counter (zero between steps), float mean(v_row)}
    FactTiles tiles;
    size_t off_rowp, off_colp, off_magbits, off_magold, off_minv, off_vsum, off_vcs, off_fin, total;
    // The lane tiles of short blocks have twice the row partials of 1024-column
    // tiles.  Where these alone would take a tensor out of the static scratch
    // (21920 x 21920 in 512-element blocks 30.3 -> 34.0 MB of 33.6), it keeps
    // the 1024-column tiles, in every entry point.
    static FactoredWs make(int64_t rows, int64_t cols, int64_t nb) {
        FactoredWs w;
        w.tiles = FactTiles::make(rows, cols, nb > 0 ? rows * cols / nb : 1);
        w.lay_out(rows, cols, nb);
        if (w.tiles.lg_lanes >= 0 && cols > kNarrowMaxCols && w.total > kNoallocScratch) {
            FactoredWs v = w;
            v.tiles.lg_lanes = -1;
            v.tiles.lane = Tiling{};
            v.lay_out(rows, cols, nb);
            if (v.total <= kNoallocScratch) return v;
        }
        return w;
    }

private:
    void lay_out(int64_t rows, int64_t cols, int64_t nb) {
        size_t o = 0;
        // any of the three tilings fits
        const auto most = [](int64_t x, int64_t y) { return x > y ? x : y; };
        const int64_t ct = most(tiles.wide.ct, tiles.lane.ct);
        const int64_t rt = most(most(tiles.wide.rt, tiles.lane.rt), tiles.tv.rt);
        off_rowp = o;    o += align256(sizeof(double) * (size_t)(ct * rows));
        off_colp = o;    o += align256(sizeof(double) * (size_t)(rt * cols));
        off_magbits = o; o += align256(sizeof(uint32_t) * (size_t)(nb * mag_shards(nb)));
        off_magold = o;  o += align256(sizeof(float) * (size_t)nb);
        off_minv = o;    o += align256(sizeof(float) * (size_t)nb);
        off_vsum = o;    o += align256(sizeof(double) * (size_t)((rows + kFinRowsPerWg - 1) / kFinRowsPerWg));
        off_vcs = o;     o += align256(sizeof(float) * (size_t)cols);
        off_fin = o;     o += 256;
        total = o;
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
