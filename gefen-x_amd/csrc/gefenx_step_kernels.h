// gefenx_step_kernels.h -- stats and apply kernels of the Gefen step, templates
// over the dtype.  Included by one source file per dtype (gefenx_step_*.hip),
// so the three instantiations compile in parallel.
#pragma once

#include "gefenx_work.h"

namespace gx {

// Wave-uniform running block max of |u| as ordered uint bits (NaN > inf >
// finite, so the integer max propagates NaN like torch's amax).
struct WaveMax {
    int64_t blk;
    uint32_t bits;
};

__device__ __forceinline__ void wavemax_flush(uint32_t* __restrict__ mb, WaveMax& wm) {
    if (wm.blk >= 0) {
        const uint32_t m = wave_max_u(wm.bits);
        if ((threadIdx.x & 63) == 0 && m != 0u) gatomic_max(mb + wm.blk, m);
    }
    wm.bits = 0u;
}

// Flush a wave-uniform running block max: one atomic per wave.
__device__ __forceinline__ void wavemax_flush63(uint32_t* __restrict__ mb, WaveMax& wm) {
    if (wm.blk >= 0) {
        const uint32_t m = wave_max_u63(wm.bits);
        if ((threadIdx.x & 63) == 63 && m != 0u) gatomic_max(mb + wm.blk, m);
    }
    wm.bits = 0u;
}

// ====================================================================
// Factored stats: workgroup = 4 waves over a tile of tile_rows rows x 1024
// columns; lane l owns the chunks at columns c0 + 8l and c0 + 512 + 8l, wave
// w takes rows r0 + w, r0 + w + 4, ... two at a time.  Per row: squares and
// the momentum max over the lane's 16 elements, then a float64 DPP reduction
// of the row sum (one value per row per column tile).  Column sums: fp32 in
// registers over 8 rows, then float64 in LDS, where the 4 waves meet after each
// granule and join the tile's partial (FactTiles has the order).
// Both go out as float64 partials (no float atomics, deterministic).
// FAST: contiguous grad and C >= 8, any alignment, any C and P (the vector
// loads take any address; a row's last chunk, when C % 8 != 0, loads the row's
// last 8 elements and shifts its own down).  Blocks that end inside a wave's
// row segment combine over the lanes first (wave_block_max): one atomic per
// block and wave where each lane used to send its own.  Measured, us: 43M fp16
// elements of which two matrices are odd-sized 46 + 48 (the odd ones through
// element loads in a launch of their own) -> 49; 7.5M bf16 elements with
// 256-element blocks 75 -> 40.
// ====================================================================
// A granule's column sum joins the tile's partial, which one thread owns: a
// plain store of the first, then atomics that return nothing, performed in
// order (a sum in registers would cost 8 of the stats kernel's 128).
__device__ __forceinline__ void put_granule(double* p, double v, bool first) {
    if (first) *gbl(p) = v;
    else gatomic_add(p, v);
}

// v, as far as the compiler knows another value each time: what follows from it
// is computed where it is used instead of held in registers across a loop.
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

struct FactStatsLds {
    float cbr[kCodebookMax];
    // float64 column sums of a granule: [wave][k][64 h + lane]; the padding puts
    // the 64 columns that a wave reads in order into different banks
    double col[kWaves][kChunk][2 * 64 + 8];
    int64_t wblk[kWaves];
    uint32_t wbits[kWaves];
};

template <int DT, bool FAST, int LF>
__device__ __forceinline__ void stats_factored(const TensorWork& wr, int64_t wg, FactStatsLds& lds) {
    using T = typename Elem<DT>::T;
    // fp32 grads: every square into a float64 accumulator, as the reference
    // sums them; 16-bit grads: exact squares in 8-row / 16-column fp32 partials
    using Acc = std::conditional_t<DT == F32, double, float>;
    constexpr int H = 2;  // chunks per lane per row
    float* s_cbr = lds.cbr;
    auto& s_col = lds.col;
    int64_t* s_wblk = lds.wblk;
    uint32_t* s_wbits = lds.wbits;
    const QTable* qt = wr.qt;
    if (threadIdx.x < kCodebookMax) s_cbr[threadIdx.x] = *gbl(qt->cbr + threadIdx.x);

    const T* g = static_cast<const T*>(wr.grad);
    const uint8_t* idxp = wr.idx;
    const float* mag_old = wr.mag;
    double* row_part = wr.row_part;
    double* col_part = col_partials(wr);
    const int64_t R = wr.R, C = wr.C, P = wr.P, gs0 = wr.gs0, gs1 = wr.gs1;
    const int64_t ct = wr.ct, tile_rows = wr.tile_rows, nb = wr.nb;
    const double invP = wr.invP;
    const MomentumCoef mc = wr.mc;
    uint32_t* mb = wr.magbits + (wg % wr.shards) * nb;
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: row state in SGPRs
    const int64_t ctile = wg % ct;
    const int64_t rtile = wg / ct;
    const int64_t tc0 = ctile * kFactTileCols;
    const int64_t span = std::min<int64_t>(kFactTileCols, C - tc0);
    int64_t cc[H], ccl[H];
    int nv[H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
        cc[h] = tc0 + h * (kFactTileCols / 2) + (int64_t)lane * kChunk;
        nv[h] = (int)std::max<int64_t>(0, std::min<int64_t>(kChunk, C - cc[h]));
        // FAST loads every chunk unconditionally: a chunk past C (nv == 0,
        // skipped by the math) or cut by it reads the row's last 8 elements
        ccl[h] = nv[h] == kChunk ? cc[h] : C - kChunk;
    }
    const int64_t r_begin = rtile * tile_rows;
    const int64_t r_end = std::min<int64_t>(r_begin + tile_rows, R);

    // block position of the first element of the wave's row segment, and its
    // advance for 4 rows: (blk, pin) += divmod(4C, P)
    int64_t blk = 0, pin = 0;
    {
        const int64_t e = (r_begin + wave) * C + tc0;
        blk = div_floor(e, P, invP);
        pin = e - blk * P;
    }
    const int64_t d4 = 4 * C;
    const int64_t dB4 = div_floor(d4, P, invP);
    const int64_t dP4 = d4 - dB4 * P;

    // column sums: in registers over 8 rows, then added into the wave's
    // float64 slots in LDS (each lane owns its 16 columns' slots); the first of
    // a granule is stored
    Acc colf[H][kChunk];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
        for (int k = 0; k < kChunk; ++k) { colf[h][k] = 0; s_col[wave][k][64 * h + lane] = 0.0; }
    auto flush_cols = [&]() {
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                s_col[wave][k][64 * h + lane] += (double)colf[h][k];
                colf[h][k] = 0;
            }
    };
    // A granule's end: waves summed in order 0..3 (and cleared, where the tile
    // goes on); thread t takes columns t, t + 256, ...  The bare barriers leave
    // the next rows' loads in flight.
    double* const col_out = col_part + rtile * C + tc0;
    auto fold = [&](bool first, auto goes_on) {
        lds_barrier();
        const unsigned t = (unsigned)opaque((int)threadIdx.x);
        double* src = &s_col[0][t % kChunk][t / kChunk];
        constexpr int kWaveStride = kChunk * (2 * 64 + 8), kStride = kThreads / kChunk;
#pragma unroll 2
        for (int j = 0; j < kFactTileCols / kThreads; ++j) {
            double sum = src[j * kStride];
#pragma unroll
            for (int ww = 1; ww < kWaves; ++ww) sum += src[ww * kWaveStride + j * kStride];
            if constexpr (decltype(goes_on)::value) {
#pragma unroll
                for (int ww = 0; ww < kWaves; ++ww) src[ww * kWaveStride + j * kStride] = 0.0;
            }
            const int c = (int)t + j * kThreads;
            if (c < span) put_granule(col_out + c, sum, first);
        }
        if constexpr (decltype(goes_on)::value) lds_barrier();
    };
    const int gran = (int)wr.gran;
    int64_t fold_at = r_begin + gran;  // first row of the next granule
    int nrows_f = 0;
    WaveMax wm{-1, 0u};
    float mag_cur = 0.0f;
    bool mag_ok = false;
    // chunk h of every lane inside C (hall) / of some lane (hany): wave-uniform
    bool hall[H], hany[H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
        hall[h] = tc0 + (h + 1) * (kFactTileCols / 2) <= C;
        hany[h] = tc0 + h * (kFactTileCols / 2) < C;
    }
    const bool cut = (C & 7) != 0;  // a chunk cut by C may sit in a half that is not full

    // One batch = the wave's next two rows (r0, r0 + 4): raw grads and
    // indices, plus (FAST) the old magnitude of each row segment's first
    // block.  FAST keeps the next batch in flight while the current one is
    // reduced, so a wave never waits for a load it issued in the same step.
    struct Batch {
        Raw8<DT> graw[2][H];
        RawIdx8 iraw[2][H];
        float gsc[2][H][kChunk];
        uint32_t isc[2][H][kChunk];
        float mo[2];
    };
    int64_t pblk = blk, ppin = pin;  // block position of the next batch to load
    auto load_batch = [&](int64_t rr0, Batch& b) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int64_t r = rr0 + (int64_t)u * kWaves;
            if constexpr (FAST) {
                // rows past the tile re-read the tile's last row; the math
                // stops before them
                const int64_t rl = r < r_end ? r : r_end - 1;
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const int64_t el = rl * C + ccl[h];
                    load_raw8_any<DT>(g + el, b.graw[u][h]);
                    b.iraw[u][h] = load_raw_idx8_any(idxp + el);
                }
                b.mo[u] = sload(mag_old + (pblk < nb ? pblk : nb - 1));  // uniform: scalar load
                ppin += dP4;
                pblk += dB4;
                if (ppin >= P) { ppin -= P; ++pblk; }
            } else {
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const int64_t e0 = r * C + cc[h];
#pragma unroll
                    for (int k = 0; k < kChunk; ++k) {
                        const bool ok = r < r_end && k < nv[h];
                        b.gsc[u][h][k] = ok ? to_f32<DT>(*gbl(g + r * gs0 + (cc[h] + k) * gs1)) : 0.0f;
                        b.isc[u][h][k] = ok ? (uint32_t)*gbl(idxp + e0 + k) : 0u;
                    }
                }
            }
        }
    };
    auto reduce_batch = [&](int64_t rr0, Batch& b) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int64_t r = rr0 + (int64_t)u * kWaves;
            if (r >= r_end) break;
            if constexpr (FAST) {
                if (cut) {
#pragma unroll
                    for (int h = 0; h < H; ++h)
                        if (hany[h] && !hall[h]) shift_down<DT>(b.graw[u][h], b.iraw[u][h], (kChunk - nv[h]) & 7);
                }
            }
            Acc rs[H];
            const bool uniform = (pin + span - 1) < P;
            if (uniform) {
                if (blk != wm.blk) {
                    wavemax_flush63(mb, wm);
                    wm.blk = blk;
                    if constexpr (FAST) {
                        mag_cur = b.mo[u];
                        mag_ok = (__float_as_uint(mag_cur) & 0x7fffffffu) < 0x7e967699u;  // |m| < 1e38, not NaN
                    } else {
                        mag_cur = *gbl(mag_old + blk);
                    }
                }
                if constexpr (FAST) {
                    // |u| max as floats (v_max3 with |.| modifiers).  Exact when
                    // every u is finite, which holds when the old magnitude is
                    // below 1e38 and every g^2 is finite (then |g - cm| cannot
                    // overflow); otherwise the row is redone with the ordered
                    // integer max, which ranks NaN above inf like torch's amax.
                    float mf = 0.0f;
                    auto chunk = [&](int h, auto masked) {
                        rs[h] = 0;
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) {
                            float gv = raw_elem<DT>(b.graw[u][h], k);
                            if constexpr (decltype(masked)::value) gv = nv[h] > k ? gv : 0.0f;
                            const float uu = momentum_value<LF>(s_cbr[raw_idx(b.iraw[u][h], k)], mag_cur, gv, mc);
                            if constexpr (decltype(masked)::value) mf = nv[h] > k ? __builtin_fmaxf(mf, fabsf(uu)) : mf;
                            else mf = __builtin_fmaxf(mf, fabsf(uu));
                            sq_add(rs[h], gv);
                            sq_add(colf[h][k], gv);
                        }
                    };
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        if (hall[h]) chunk(h, std::false_type{});
                        else if (hany[h]) chunk(h, std::true_type{});
                        else rs[h] = 0;
                    }
                    // integer test: NaN and inf both fail it, whatever the
                    // compiler assumes about float compares (a square that
                    // overflows fp32 is inf in either accumulator)
                    const bool fin = (__float_as_uint((float)(rs[0] + rs[1])) & 0x7fffffffu) < 0x7f800000u;
                    if (__builtin_expect(mag_ok && __all(fin), 1)) {
                        const uint32_t mb_ = __float_as_uint(mf);
                        wm.bits = mb_ > wm.bits ? mb_ : wm.bits;
                    } else {
                        uint32_t m = wm.bits;
#pragma unroll
                        for (int h = 0; h < H; ++h) {
                            if (nv[h] == 0) continue;
#pragma unroll
                            for (int k = 0; k < kChunk; ++k) {
                                if (k >= nv[h]) continue;
                                const float uu = momentum_value<LF>(s_cbr[raw_idx(b.iraw[u][h], k)], mag_cur,
                                                                    raw_elem<DT>(b.graw[u][h], k), mc);
                                const uint32_t ub = __float_as_uint(uu) & 0x7fffffffu;
                                m = ub > m ? ub : m;
                            }
                        }
                        wm.bits = m;
                    }
                } else {
                    uint32_t m = wm.bits;
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        rs[h] = 0;
                        if (nv[h] == 0) continue;  // columns past C (last tile)
#pragma unroll
                        for (int k = 0; k < kChunk; ++k) {
                            if (k >= nv[h]) continue;
                            const float gv = b.gsc[u][h][k];
                            const float uu = momentum_value<LF>(s_cbr[b.isc[u][h][k]], mag_cur, gv, mc);
                            const uint32_t ub = __float_as_uint(uu) & 0x7fffffffu;
                            m = ub > m ? ub : m;
                            sq_add(rs[h], gv);
                            sq_add(colf[h][k], gv);
                        }
                    }
                    wm.bits = m;
                }
            } else {
                // blocks end inside this row segment: per-lane blocks; a
                // block that ends inside a chunk (P % 8 != 0) sends its part
                // at once, each chunk's last block meets its neighbours'
                wavemax_flush63(mb, wm);
                wm.blk = -1;
                int64_t bb[H], pp[H];
                float mo[H];
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const int64_t off = pin + (cc[h] - tc0);
                    const int64_t db = div_floor(off, P, invP);
                    bb[h] = nv[h] > 0 ? blk + db : -1;
                    pp[h] = off - db * P;
                    mo[h] = nv[h] > 0 ? *gbl(mag_old + bb[h]) : 0.0f;
                }
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    rs[h] = 0;
                    if (!hany[h]) continue;
                    uint32_t m = 0u;
#pragma unroll
                    for (int k = 0; k < kChunk; ++k) {
                        if (k < nv[h]) {
                            float gv;
                            uint32_t ix;
                            if constexpr (FAST) { gv = raw_elem<DT>(b.graw[u][h], k); ix = raw_idx(b.iraw[u][h], k); }
                            else { gv = b.gsc[u][h][k]; ix = b.isc[u][h][k]; }
                            const float uu = momentum_value<LF>(s_cbr[ix], mo[h], gv, mc);
                            const uint32_t ub = __float_as_uint(uu) & 0x7fffffffu;
                            m = ub > m ? ub : m;
                            sq_add(rs[h], gv);
                            sq_add(colf[h][k], gv);
                            if (++pp[h] == P && k + 1 < nv[h]) {
                                if (m) gatomic_max(mb + bb[h], m);
                                m = 0u;
                                pp[h] = 0;
                                ++bb[h];
                                mo[h] = *gbl(mag_old + bb[h]);
                            }
                        }
                    }
                    wave_block_max(mb, bb[h], m);
                }
            }
            double rsum = 0.0;
#pragma unroll
            for (int h = 0; h < H; ++h) rsum += (double)rs[h];
            rsum = wave_sum_d63(rsum);
            if (lane == 63) *gbl(row_part + ctile * R + r) = rsum;
            if (++nrows_f == 8) {
                flush_cols();
                nrows_f = 0;
            }
            pin += dP4;
            blk += dB4;
            if (pin >= P) { pin -= P; ++blk; }
        }
    };

    constexpr int64_t kStep = 2 * kWaves;
    // A granule ends inside the tile before row r - wave.  Every wave comes here
    // with that row: one that left the loop before has r >= r_end, so r_end lies
    // within the 3 rows after an r - wave below it.  A granule is a multiple of
    // 32 rows, 8 of each wave, so the fp32 sums are flushed.
    auto granule_ends = [&](int64_t r) { return r - wave == fold_at && fold_at < r_end; };
    auto end_granule = [&]() {
        fold(fold_at - gran == r_begin, std::true_type{});
        fold_at += gran;
    };
    int64_t r0 = r_begin + wave;
    if (r0 < r_end) {
        Batch ba, bb;
        load_batch(r0, ba);
        if constexpr (FAST) {
            // The prefetch is unconditional (past the tile it re-reads the
            // tile's last row, which is still in cache), so every step has
            // the same loads in flight and the compiler can wait for the
            // current batch alone instead of draining the queue.
            for (;;) {
                load_batch(r0 + kStep, bb);
                reduce_batch(r0, ba);
                r0 += kStep;
                if (r0 >= r_end) break;
                load_batch(r0 + kStep, ba);
                reduce_batch(r0, bb);
                r0 += kStep;
                if (granule_ends(r0)) end_granule();
                if (r0 >= r_end) break;
            }
        } else {
            for (;;) {
                reduce_batch(r0, ba);
                r0 += kStep;
                if (granule_ends(r0)) end_granule();
                if (r0 >= r_end) break;
                load_batch(r0, ba);
            }
        }
    }
    flush_cols();

    // final block-max flush: one atomic per workgroup when the waves agree
    const uint32_t wbits = wm.blk >= 0 ? wave_max_u63(wm.bits) : 0u;
    if (lane == 63) {
        s_wblk[wave] = wm.blk;
        s_wbits[wave] = wbits;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        bool same = true;
        uint32_t m = 0u;
        for (int ww = 0; ww < kWaves; ++ww) {
            same = same && (s_wblk[ww] == s_wblk[0]);
            m = s_wbits[ww] > m ? s_wbits[ww] : m;
        }
        if (same) {
            if (s_wblk[0] >= 0 && m) gatomic_max(mb + s_wblk[0], m);
        } else {
            for (int ww = 0; ww < kWaves; ++ww)
                if (s_wblk[ww] >= 0 && s_wbits[ww]) gatomic_max(mb + s_wblk[ww], s_wbits[ww]);
        }
    }
    fold(fold_at - gran == r_begin, std::false_type{});  // the last granule
}

// ====================================================================
// Factored stats with per-lane blocks, for contiguous matrices (C >= 8, any
// alignment and P) of at most kNarrowMaxCols columns or of short blocks.  The
// workgroup covers tile_rows rows of tile_cols <= 512 columns; L lanes (a
// power of two, 8 columns each) take a row of the tile, a wave 64 / L rows at a
// time, four such steps in flight, each lane's old magnitude loaded with its
// chunk.  A row's lanes add up its sum of squares, a lane keeps its columns'
// sums (fp32 over 8 rows, then float64), the lanes of one column meet in LDS
// after each granule in a fixed order.  stats_factored would leave all but C / 16 of a
// wave's lanes idle on few columns and walk the rows one by one (a set of
// 16-column and 16-row fp32 adapters 246 -> 16 us), and would wait for the
// magnitudes of every row whose blocks end inside it (7.5M bf16 elements with
// 256-element blocks 40 -> 21 us).
// ====================================================================
template <int DT, int LF>
__device__ __forceinline__ void stats_lanes(const TensorWork& wr, int64_t wg, FactStatsLds& lds) {
    using T = typename Elem<DT>::T;
    using Acc = std::conditional_t<DT == F32, double, float>;
    constexpr int Q = 4;  // steps in flight
    float* s_cbr = lds.cbr;
    if (threadIdx.x < kCodebookMax) s_cbr[threadIdx.x] = *gbl(wr.qt->cbr + threadIdx.x);
    const T* g = static_cast<const T*>(wr.grad);
    const uint8_t* idxp = wr.idx;
    const float* mag_old = wr.mag;
    const int64_t R = wr.R, C = wr.C, P = wr.P;
    const double invP = wr.invP;
    const MomentumCoef mc = wr.mc;
    uint32_t* mb = wr.magbits + (wg % wr.shards) * wr.nb;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lgL = wr.lg_lanes, L = 1 << lgL, rpw = 64 >> lgL;
    const int64_t ct = wr.ct, ctile = wg % ct, rtile = wg / ct;
    const int64_t tc0 = ctile * wr.tile_cols;
    const int span = (int)std::min<int64_t>(wr.tile_cols, C - tc0);
    const int sub = lane >> lgL;
    const int64_t c = tc0 + (lane & (L - 1)) * kChunk;
    const int nv = (int)std::max<int64_t>(0, std::min<int64_t>(kChunk, tc0 + span - c));
    const int64_t cl = nv == kChunk ? c : tc0 + span - kChunk;  // a lane past the tile or cut by it: its last 8
    const int sh = (kChunk - nv) & 7;
    const bool cut = (span & 7) != 0;
    const int64_t r_begin = rtile * wr.tile_rows;
    const int64_t r_end = std::min<int64_t>(r_begin + wr.tile_rows, R);
    __syncthreads();
    Acc colf[kChunk];
#pragma unroll
    for (int k = 0; k < kChunk; ++k) colf[k] = 0;
    bool fresh = true;
    auto flush_cols = [&]() {  // as in stats_factored
        const auto flush = [&](auto add) {
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                double& slot = lds.col[wave][k][lane];
                slot = fresh ? (double)colf[k] : slot + (double)colf[k];
                colf[k] = 0;
            }
        };
        flush(std::true_type{});
        fresh = false;
    };
    // A granule's end: per column the waves in order, and the rows of a wave
    double* const col_part = col_partials(wr) + rtile * C + tc0;
    auto fold = [&](bool first) {
        lds_barrier();
        for (int col = opaque(threadIdx.x); col < span; col += kThreads) {
            const int j = col / kChunk, k = col % kChunk;
            double sum = 0.0;
            for (int ww = 0; ww < kWaves; ++ww)
                for (int s = 0; s < rpw; ++s) sum += lds.col[ww][k][s * L + j];
            put_granule(col_part + col, sum, first);
        }
    };
    constexpr int64_t kStep = Q * kWaves;
    int64_t fold_at = r_begin + wr.gran;  // first row of the next granule
    int nf = 0;
    for (int64_t r0 = r_begin + wave * rpw; r0 < r_end; r0 += kStep * rpw) {
        Raw8<DT> gr[Q];
        RawIdx8 ir[Q];
        int64_t bb[Q], pp[Q];
        float mo[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int64_t r = r0 + (int64_t)q * kWaves * rpw + sub;
            const int64_t rl = r < r_end ? r : r_end - 1;
            load_raw8_any<DT>(g + rl * C + cl, gr[q]);
            ir[q] = load_raw_idx8_any(idxp + rl * C + cl);
            const int64_t e = rl * C + (nv > 0 ? c : cl);
            bb[q] = div_floor(e, P, invP);
            pp[q] = e - bb[q] * P;
            mo[q] = *gbl(mag_old + bb[q]);
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int64_t r = r0 + (int64_t)q * kWaves * rpw + sub;
            if (r - sub >= r_end) break;
            if (cut) shift_down<DT>(gr[q], ir[q], sh);
            const int n = r < r_end ? nv : 0;
            Acc rs = 0;
            uint32_t m = 0u;
            int64_t key = n > 0 ? bb[q] : -1;
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                if (k < n) {
                    const float gv = raw_elem<DT>(gr[q], k);
                    const float uu = momentum_value<LF>(s_cbr[raw_idx(ir[q], k)], mo[q], gv, mc);
                    const uint32_t ub = __float_as_uint(uu) & 0x7fffffffu;
                    m = ub > m ? ub : m;
                    sq_add(rs, gv);
                    sq_add(colf[k], gv);
                    if (++pp[q] == P && k + 1 < n) {
                        if (m) gatomic_max(mb + key, m);
                        m = 0u;
                        pp[q] = 0;
                        ++key;
                        mo[q] = *gbl(mag_old + key);
                    }
                }
            }
            wave_block_max(mb, key, m);
            double rsum = (double)rs;
            if (lgL > 0) rsum += dpp64<0xB1, 0xf>(rsum);   // lane ^ 1
            if (lgL > 1) rsum += dpp64<0x4E, 0xf>(rsum);   // lane ^ 2
            if (lgL > 2) rsum += dpp64<0x141, 0xf>(rsum);  // the other half of 8
            if (lgL > 3) rsum += dpp64<0x140, 0xf>(rsum);  // the other half of 16
            if (lgL > 4) rsum += __shfl_xor(rsum, 16, 64);
            if (lgL > 5) rsum += __shfl_xor(rsum, 32, 64);
            if ((lane & (L - 1)) == 0 && r < r_end) *gbl(wr.row_part + ctile * R + r) = rsum;
            if (++nf == 8) {
                nf = 0;
                flush_cols();
            }
        }
        // every wave comes here for each granule that ends inside the tile
        // (one that left the loop has its r0, so every later granule, past r_end)
        const int64_t next = r0 - wave * rpw + kStep * rpw;
        if (next == fold_at && fold_at < r_end) {
            fold(fold_at - wr.gran == r_begin);
            lds_barrier();
            fresh = true;
            fold_at += wr.gran;
        }
    }
    flush_cols();
    fold(fold_at - wr.gran == r_begin);  // the last granule
}

// ====================================================================
// Transposed views: g (and p) with strides (1, ld), ld >= R -- the layout of
// x.t() for a contiguous [C, R] tensor x.  Logical row-major order still
// fixes the blocks, the indices and v_row / v_col, but g and p run along
// logical columns.  The view kernels walk 64 x 64 logical tiles, one per
// wave at a time; lane l = 8b + a owns the 8 x 8 sub-block at tile rows
// 8a .. 8a+7 and tile columns 8b .. 8b+7.  It loads g (and p) as 8 vectors
// along storage rows (tile column 8b+k, rows 8a .. 8a+7: the 8 lanes of one
// b read one 128-byte run for 16-bit types) and the indices as 8 logical
// chunks (row 8a+j, columns 8b .. 8b+7: the 8 lanes of one a read one
// 64-byte run).  Element (j, k) of the sub-block is element j of g vector k
// and element k of index chunk j, so no data passes through LDS.  Chunk j
// (8 elements of one logical row) lies in one block since P % 8 == 0.
// Requires R, C, P multiples of 8 and 16-byte aligned storage rows.
// ====================================================================
constexpr int kTvFew = 4;           // blocks a tile may touch on the scalar-load path

// A value every lane of the wave holds, moved to scalar registers.
__device__ __forceinline__ int64_t uniform64(int64_t v) {
    const uint64_t u = (uint64_t)v;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Blocks of a lane's 8 chunks (rows r .. r+7 at column c) relative to b_lo;
// (dB, dP) = divmod(C, P) advances one row.
__device__ __forceinline__ void tv_chunk_blocks(int64_t r, int64_t c, int64_t C, int64_t P, double invP,
                                                int64_t dB, int64_t dP, int64_t b_lo, int q[kChunk]) {
    const int64_t e = r * C + c;
    int64_t b = div_floor(e, P, invP);
    int64_t pin = e - b * P;
#pragma unroll
    for (int j = 0; j < kChunk; ++j) {
        q[j] = (int)(b - b_lo);
        pin += dP;
        b += dB;
        if (pin >= P) { pin -= P; ++b; }
    }
}

__device__ __forceinline__ float tv_pick(int q, const float v[kTvFew]) {
    return q == 0 ? v[0] : (q == 1 ? v[1] : (q == 2 ? v[2] : v[3]));
}

// The first kTvFew values of a per-block array from block b_lo on (indices
// clamped to the array), as scalar loads.
__device__ __forceinline__ void tv_sload_few(const float* arr, int64_t b_lo, int64_t nb, float v[kTvFew]) {
#pragma unroll
    for (int i = 0; i < kTvFew; ++i) v[i] = sload(arr + (b_lo + i < nb ? b_lo + i : nb - 1));
}

// Reduce-scatter of 8 float64 values over the 8 lanes of a group (lane bits
// 0-2): lane i ends with the group's sum of v[i].  Partners at the three
// steps: i ^ 7 (row_half_mirror), i ^ 2, i ^ 1 (quad_perm); a fixed order of
// float64 adds.
__device__ __forceinline__ double tv_scatter_lo(const double v[kChunk], int i) {
    const bool hi = (i & 4) != 0, mid = (i & 2) != 0, lo = (i & 1) != 0;
    double w[4], x[2];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const double send = hi ? v[t] : v[t + 4];
        w[t] = (hi ? v[t + 4] : v[t]) + dpp64<0x141, 0xf>(send);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const double send = mid ? w[t] : w[t + 2];
        x[t] = (mid ? w[t + 2] : w[t]) + dpp64<0x4E, 0xf>(send);
    }
    const double send = lo ? x[0] : x[1];
    return (lo ? x[1] : x[0]) + dpp64<0xB1, 0xf>(send);
}

// The same over lane bits 3-5 (partners lane ^ 32, lane ^ 16, lane ^ 8):
// lane 8i + a ends with the sum of v[i] over its 8 lanes a + 8i'.
__device__ __forceinline__ double tv_scatter_hi(const double v[kChunk], int i) {
    const bool hi = (i & 4) != 0, mid = (i & 2) != 0, lo = (i & 1) != 0;
    double w[4], x[2];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const double send = hi ? v[t] : v[t + 4];
        w[t] = (hi ? v[t + 4] : v[t]) + __shfl_xor(send, 32, 64);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const double send = mid ? w[t] : w[t + 2];
        x[t] = (mid ? w[t + 2] : w[t]) + __shfl_xor(send, 16, 64);
    }
    const double send = lo ? x[0] : x[1];
    return (lo ? x[1] : x[0]) + dpp64<0x128, 0xf>(send);  // row_ror:8 = lane ^ 8 within 16
}

template <int MODE>
struct TvStatsLds {
    float cbr[kCodebookMax];
    double colp[MODE == 0 ? kWaves : 1][MODE == 0 ? kFactTileCols : 1];
    uint32_t bmax[kTvLdsBlocks];
    double bsum[MODE == 1 ? kTvLdsBlocks : 1];
};

// Stats of a transposed view.  Workgroup (ctile, rtile) covers tile_cols
// (<= kFactTileCols) columns and tile_rows (<= 256) rows; wave w takes the 64-row band w and
// walks the workgroup's columns in 64 x 64 tiles, so the 4 waves read 512-byte
// runs of the same storage rows at about the same time (measured 6% faster
// than 4 waves on 4 column ranges) and a wave reads the two halves of each
// 128-byte index line in consecutive tiles.  MODE 0 (factored): squares in
// fp32 over a chunk's 8 columns and over a vector's 8 rows (float64 for fp32
// grads), then float64: a row's sum over a granule's columns collects in its
// lanes and joins the row partial (reduce-scatter over the 8 column groups),
// a column's over the band in one lane (reduce-scatter over the 8 row
// groups of each tile), and the 4 bands' column sums meet in LDS in band
// order.  Block max |u| (and, MODE 1, the block's sum of squares, each square
// rounded to bf16 for bf16 grads, in float64): when a tile touches at most
// kTvFew blocks (the common case) its old magnitudes are scalar loads, the
// lanes keep one value per block and the wave reduces each; otherwise per
// chunk.  Either way the values go to the workgroup's LDS accumulators (<= 512
// blocks) or the shards.
template <int DT, int MODE, int LF>
__device__ __forceinline__ void stats_tv(const TensorWork& wr, int64_t wg, TvStatsLds<MODE>& lds) {
    using T = typename Elem<DT>::T;
    using Acc = std::conditional_t<DT == F32, double, float>;
    const QTable* qt = wr.qt;
    if (threadIdx.x < kCodebookMax) lds.cbr[threadIdx.x] = *gbl(qt->cbr + threadIdx.x);
    if constexpr (MODE == 0) {
        for (int k = threadIdx.x; k < kWaves * kFactTileCols; k += kThreads) (&lds.colp[0][0])[k] = 0.0;
    }
    const float* s_cbr = lds.cbr;

    const T* g = static_cast<const T*>(wr.grad);
    const uint8_t* idxp = wr.idx;
    const float* mag_old = wr.mag;
    double* row_part = row_partials(wr);
    double* col_part = wr.col_part;
    const int64_t R = wr.R, C = wr.C, P = wr.P, ld = wr.gs1, nb = wr.nb;
    const double invP = wr.invP;
    const MomentumCoef mc = wr.mc;
    uint32_t* mb = wr.magbits + (wg % wr.shards) * nb;
    double* bsq = MODE == 1 ? wr.blk_sq + (wg % wr.shards) * nb : nullptr;
    const int64_t ctile = wg % wr.ct, rtile = wg / wr.ct;
    const int64_t c_begin = ctile * wr.tile_cols;
    const int64_t c_end = std::min<int64_t>(c_begin + wr.tile_cols, C);
    const int64_t r_begin = rtile * wr.tile_rows;
    const int64_t r_end = std::min<int64_t>(r_begin + wr.tile_rows, R);
    // blocks of the workgroup's region: few of them (large periods) reduce
    // in LDS and leave with one atomic per block and workgroup
    const int64_t b_wlo = div_floor(r_begin * C + c_begin, P, invP);
    const int64_t b_span = div_floor((r_end - 1) * C + (c_end - 1), P, invP) - b_wlo + 1;
    const bool lds_blk = b_span <= kTvLdsBlocks;
    if (lds_blk) {
        for (int k = threadIdx.x; k < b_span; k += kThreads) {
            lds.bmax[k] = 0u;
            if constexpr (MODE == 1) lds.bsum[k] = 0.0;
        }
    }
    const int lane = threadIdx.x & 63, la = lane & 7, lb = lane >> 3;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t cw0 = c_begin, cw1 = c_end;
    const int ncs = (int)((c_end - c_begin + kTv - 1) / kTv);
    const int64_t rw0 = r_begin + (int64_t)wave * kTv;
    const int ntile = rw0 < r_end ? ncs : 0;
    const int64_t dB = div_floor(C, P, invP);
    const int64_t dP = C - dB * P;
    __syncthreads();

    auto put_max = [&](int64_t b, uint32_t m) {
        if (m == 0u) return;
        if (lds_blk) atomicMax(&lds.bmax[b - b_wlo], m);
        else gatomic_max(mb + b, m);
    };
    auto put_sum = [&](int64_t b, double v) {
        if (v == 0.0) return;
        if (lds_blk) atomicAdd(&lds.bsum[b - b_wlo], v);
        else gatomic_add(bsq + b, v);
    };

    struct Tile {
        Raw8<DT> gv[kChunk];  // storage-row vectors: tile column 8b+k, rows 8a .. 8a+7
        RawIdx8 iv[kChunk];   // index chunks: row 8a+j, columns 8b .. 8b+7
    };
    // lanes outside the region read its last sub-block instead (the math
    // skips them)
    auto load_tile = [&](int s, Tile& t) {
        const int64_t r = rw0 + 8 * la;
        const int64_t c = cw0 + (int64_t)s * kTv + 8 * lb;
        const int64_t rl = r < r_end ? r : r_end - kChunk, cl = c < cw1 ? c : cw1 - kChunk;
#pragma unroll
        for (int k = 0; k < kChunk; ++k) load_raw8<DT>(g + (cl + k) * ld + rl, t.gv[k]);
#pragma unroll
        for (int j = 0; j < kChunk; ++j) t.iv[j] = load_raw_idx8_cached(idxp + (rl + j) * C + cl);
    };

    int left = (int)(wr.gran / kTv);  // 64-column tiles to the granule's end
    double rtot = 0.0;    // MODE 0: sum of row 8a + b over the granules so far
    double racc[kChunk];  // MODE 0: row sums of the lane's 8 rows over the granule's columns so far
#pragma unroll
    for (int j = 0; j < kChunk; ++j) racc[j] = 0.0;

    auto reduce_tile = [&](int s, const Tile& t) {
        const int cs = s;
        const int64_t r0 = rw0, c0 = cw0 + (int64_t)cs * kTv;
        const int64_t r = r0 + 8 * la, c = c0 + 8 * lb;
        const bool ok = r < r_end && c < cw1;
        const int64_t r_last = std::min<int64_t>(r0 + kTv, r_end) - 1;
        const int64_t c_last = std::min<int64_t>(c0 + kTv, cw1) - 1;
        const int64_t b_lo = uniform64(div_floor(r0 * C + c0, P, invP));
        const int64_t b_hi = uniform64(div_floor(r_last * C + c_last, P, invP));
        Acc colf[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) colf[k] = 0;
        // one chunk: max |u| bits, fp32 (MODE 0) or float64 (MODE 1) square sums
        auto chunk = [&](int j, float mo, uint32_t& m, Acc& rs, double& bs) {
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                const float gv = raw_elem<DT>(t.gv[k], j);
                const float uu = momentum_value<LF>(s_cbr[raw_idx(t.iv[j], k)], mo, gv, mc);
                const uint32_t ub = __float_as_uint(uu) & 0x7fffffffu;
                m = ub > m ? ub : m;
                if constexpr (MODE == 0) {
                    sq_add(rs, gv);
                    sq_add(colf[k], gv);
                } else {
                    float sq = gv * gv;
                    if constexpr (DT == BF16) sq = round_dt<BF16>(sq);
                    bs += (double)sq;
                }
            }
        };
        if (b_hi - b_lo < kTvFew) {
            float mo[kTvFew];
            tv_sload_few(mag_old, b_lo, nb, mo);
            uint32_t mx[kTvFew] = {0u, 0u, 0u, 0u};
            double bx[kTvFew] = {0.0, 0.0, 0.0, 0.0};
            if (ok) {
                int q[kChunk];
                tv_chunk_blocks(r, c, C, P, invP, dB, dP, b_lo, q);
#pragma unroll
                for (int j = 0; j < kChunk; ++j) {
                    uint32_t m = 0u;
                    Acc rs = 0;
                    double bs = 0.0;
                    chunk(j, tv_pick(q[j], mo), m, rs, bs);
                    if constexpr (MODE == 0) racc[j] += (double)rs;
#pragma unroll
                    for (int i = 0; i < kTvFew; ++i) {
                        if (q[j] == i) {
                            mx[i] = m > mx[i] ? m : mx[i];
                            if constexpr (MODE == 1) bx[i] += bs;
                        }
                    }
                }
            }
            const int nq = (int)(b_hi - b_lo) + 1;
#pragma unroll
            for (int i = 0; i < kTvFew; ++i) {
                if (i < nq) {
                    const uint32_t m = wave_max_u63(mx[i]);
                    double v = 0.0;
                    if constexpr (MODE == 1) v = wave_sum_d63(bx[i]);
                    if (lane == 63) {
                        put_max(b_lo + i, m);
                        if constexpr (MODE == 1) put_sum(b_lo + i, v);
                    }
                }
            }
        } else if (ok) {
            // many blocks in the tile (P small against C): per chunk
            const int64_t e = r * C + c;
            int64_t b = div_floor(e, P, invP);
            int64_t pin = e - b * P;
#pragma unroll
            for (int j = 0; j < kChunk; ++j) {
                uint32_t m = 0u;
                Acc rs = 0;
                double bs = 0.0;
                chunk(j, *gbl(mag_old + b), m, rs, bs);
                if constexpr (MODE == 0) racc[j] += (double)rs;
                put_max(b, m);
                if constexpr (MODE == 1) put_sum(b, bs);
                pin += dP;
                b += dB;
                if (pin >= P) { pin -= P; ++b; }
            }
        }
        if constexpr (MODE == 0) {
            // column 8b + a of this tile, over its rows
            double cv[kChunk];
#pragma unroll
            for (int k = 0; k < kChunk; ++k) cv[k] = (double)colf[k];
            const double col = tv_scatter_lo(cv, la);
            lds.colp[wave][cs * kTv + 8 * lb + la] = col;
            const bool last = cs == ncs - 1;
            if (--left == 0 || last) {
                left = (int)(wr.gran / kTv);
                rtot += tv_scatter_hi(racc, lb);
#pragma unroll
                for (int j = 0; j < kChunk; ++j) racc[j] = 0.0;
            }
            if (last) {
                const int64_t rr = r0 + 8 * la + lb;
                if (rr < r_end) *gbl(row_part + ctile * R + rr) = rtot;
            }
        }
    };

    if (ntile > 0) {
        // one tile in flight per wave: a second register set (the next
        // tile's loads issued before this one's math) measured no faster at
        // two waves per SIMD than one set at three
        Tile t;
        for (int s = 0; s < ntile; ++s) {
            load_tile(s, t);
            reduce_tile(s, t);
        }
    }
    __syncthreads();
    if constexpr (MODE == 0) {
        for (int64_t k = threadIdx.x; k < c_end - c_begin; k += kThreads) {
            double v = lds.colp[0][k];
#pragma unroll
            for (int ww = 1; ww < kWaves; ++ww) v += lds.colp[ww][k];
            *gbl(col_part + rtile * C + c_begin + k) = v;
        }
    }
    if (lds_blk) {
        for (int k = threadIdx.x; k < b_span; k += kThreads) {
            const uint32_t m = lds.bmax[k];
            if (m != 0u) gatomic_max(mb + b_wlo + k, m);
            if constexpr (MODE == 1) {
                const double v = lds.bsum[k];
                if (v != 0.0) gatomic_add(bsq + b_wlo + k, v);
            }
        }
    }
}

template <int DT, int MODE>
__device__ __forceinline__ void stats_tv_wg(const TensorWork& w, int64_t wg) {
    __shared__ TvStatsLds<MODE> lds;
    if (w.mc.small) stats_tv<DT, MODE, kLerpSmall>(w, wg, lds);
    else stats_tv<DT, MODE, kLerpLarge>(w, wg, lds);
}

// ====================================================================
// Block stats (block path): per-block sum of squared grads (rounded through
// bf16 for bf16 grads, gefen.py:180-190) and max |u|, summed in an order that
// does not depend on scheduling, so a run is bit-reproducible.
// Workgroup wg owns elements [wg*E, (wg+1)*E), E = kDetIters * 256 * EPL.  In
// iteration i, lane l of wave v takes the EPL elements of item
// j = i*256 + v*64 + l, all in one block (EPL = 8 needs P % 8 == 0 and
// N % 8 == 0; otherwise EPL = 1).  A wave's 64 items are combined per block
// by a segmented suffix sum (Hillis-Steele steps masked at block starts: a
// fixed schedule of float64 adds).  A block that starts and ends inside those
// 64 items is complete and is stored; the first and last block partials of
// each wave and iteration go to LDS, where wave 0 combines the workgroup's 64
// of them the same way.  The workgroup's own first and last block partials
// go to its record; finalize adds a block's stored sum and the records of
// the workgroups it spans, in workgroup order.  Max |u| takes one atomic max
// per block and wave (a max is exact in any order).
// ====================================================================
static_assert(kThreads == kCodebookMax, "one codebook entry per thread");
static_assert(2 * kDetIters * kWaves == 64, "the workgroup's run partials fill one wave");

// Flush a wave's running block max (wave-uniform key and value): one atomic
// into the workgroup's shard.
__device__ __forceinline__ void flush_det_max(uint32_t* mb, int64_t key, int64_t nb, uint32_t m) {
    if ((threadIdx.x & 63) == 0 && key >= 0 && key < nb && m != 0u) gatomic_max(mb + key, m);
}

// A workgroup whose elements all lie in one block (every block of at least
// E elements, most of them): no per-element block index and no segmented
// scans.  The old magnitude is one scalar load; each lane sums its items in
// iteration order, the waves combine by a fixed DPP pattern, then in wave
// order -- the same order on every run.  FULL: the workgroup's E elements
// all lie inside the tensor, so no load sits behind a branch.
template <int DT, int EPL, bool FULL>
__device__ __forceinline__ void stats_block_one(const TensorWork& w, int64_t wg, int64_t kb, float* s_cbr,
                                                double* s_sum) {
    using T = typename Elem<DT>::T;
    const T* g = static_cast<const T*>(w.grad);
    const int64_t N = w.N;
    const MomentumCoef mc = w.mc;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int64_t base = wg * (int64_t)(kDetIters * kThreads * EPL);
    const float mo = sload(w.mag + kb);
    // the codebook goes into a register first and into LDS after the element
    // loads are issued (loaded in this block, so the LDS write waits for it alone)
    const float cbr_v = *gbl(w.qt->cbr + threadIdx.x % kCodebookMax);
    Raw8<DT> gr[kDetIters];
    RawIdx8 ir[kDetIters];
    float graw[kDetIters];
    uint32_t iraw[kDetIters];
#pragma unroll
    for (int i = 0; i < kDetIters; ++i) {
        const int64_t e0 = base + ((int64_t)i * kThreads + threadIdx.x) * EPL;
        if (FULL || e0 < N) {
            if constexpr (EPL == kChunk) {
                if (w.det_vec) {
                    load_raw8<DT>(g + e0, gr[i]);
                    ir[i] = load_raw_idx8(w.idx + e0);
                } else {  // grad or indices not 16 / 8-byte aligned: the same items, element loads
                    load_raw8_elems<DT>(g + e0, gr[i]);
                    ir[i] = load_raw_idx8_elems(w.idx + e0);
                }
            } else {
                graw[i] = to_f32<DT>(*gbl(g + e0));
                iraw[i] = *gbl(w.idx + e0);
            }
        }
        if constexpr (FULL) __builtin_amdgcn_sched_barrier(0);  // iteration order kept: iteration i lands i-th
    }
    s_cbr[threadIdx.x % kCodebookMax] = cbr_v;  // every thread: no branch, so the waits stay exact
    __syncthreads();
    double lsum = 0.0;
    uint32_t lmax = 0u;
#pragma unroll
    for (int i = 0; i < kDetIters; ++i) {
        const int64_t e0 = base + ((int64_t)i * kThreads + threadIdx.x) * EPL;
        if (FULL || e0 < N) {
            double cs = 0.0;  // every square into float64, as the reference sums them
            if constexpr (EPL == kChunk) {
#pragma unroll
                for (int k = 0; k < kChunk; ++k) {
                    const float gv = raw_elem<DT>(gr[i], k);
                    const float u = momentum_value(s_cbr[raw_idx(ir[i], k)], mo, gv, mc);
                    const uint32_t ub = __float_as_uint(u) & 0x7fffffffu;
                    lmax = ub > lmax ? ub : lmax;
                    float sq = gv * gv;
                    if constexpr (DT == BF16) sq = round_dt<BF16>(sq);
                    cs += (double)sq;
                }
            } else {
                const float gv = graw[i];
                const float u = momentum_value(s_cbr[iraw[i]], mo, gv, mc);
                const uint32_t ub = __float_as_uint(u) & 0x7fffffffu;
                lmax = ub > lmax ? ub : lmax;
                float sq = gv * gv;
                if constexpr (DT == BF16) sq = round_dt<BF16>(sq);
                cs = (double)sq;
            }
            lsum += cs;
        }
    }
    lsum = wave_sum_d(lsum);
    const uint32_t wmax = wave_max_u63(lmax);  // in lane 63
    uint32_t* mb = w.magbits + (wg % w.shards) * w.nb;
    if (lane == 63 && wmax != 0u) gatomic_max(mb + kb, wmax);
    if (lane == 0) s_sum[wave] = lsum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int v = 0; v < kWaves; ++v) t += s_sum[v];
        DetRec* rec = w.det_rec + wg;
        rec->kf = kb;
        rec->sf = t;
        rec->kl = -1;
        rec->sl = 0.0;
    }
}

struct BlockStatsLds {
    float cbr[kCodebookMax];
    int64_t key[2 * kDetIters * kWaves];
    double sum[2 * kDetIters * kWaves];
};

template <int DT, int EPL>
__device__ __forceinline__ void stats_block_det(const TensorWork& w, int64_t wg, BlockStatsLds& lds) {
    using T = typename Elem<DT>::T;
    float* s_cbr = lds.cbr;
    int64_t* s_key = lds.key;
    double* s_sum = lds.sum;
    const int64_t N = w.N, P = w.P, nb = w.nb;
    constexpr int64_t E = (int64_t)kDetIters * kThreads * EPL;
    const int64_t base = wg * E;
    const int64_t wg_end = base + E < N ? base + E : N;
    const int64_t kfirst = div_floor(base, P, w.invP);
    if (kfirst == div_floor(wg_end - 1, P, w.invP)) {
        if (base + E <= N) stats_block_one<DT, EPL, true>(w, wg, kfirst, s_cbr, s_sum);
        else stats_block_one<DT, EPL, false>(w, wg, kfirst, s_cbr, s_sum);
        return;
    }
    const float cbr_v = *gbl(w.qt->cbr + threadIdx.x % kCodebookMax);  // to LDS after the element loads
    const T* g = static_cast<const T*>(w.grad);
    const MomentumCoef mc = w.mc;
    // max |u|: a wave carries the max of its current block across iterations
    // and flushes it into its workgroup's shard when the block changes, so a
    // block spanning many workgroups takes one atomic per wave, spread over
    // the shards (finalize takes the max over them)
    uint32_t* mb = w.magbits + (wg % w.shards) * nb;
    double* bsq = w.blk_sq;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    // every iteration's loads first
    Raw8<DT> gr[kDetIters];
    RawIdx8 ir[kDetIters];
    float graw[kDetIters];
    uint32_t iraw[kDetIters];
    float mo[kDetIters];
    int64_t keys[kDetIters];
#pragma unroll
    for (int i = 0; i < kDetIters; ++i) {
        const int64_t e0 = base + ((int64_t)i * kThreads + threadIdx.x) * EPL;
        keys[i] = nb;  // past the end: a sentinel key, never stored
        if (e0 < N) {
            keys[i] = div_floor(e0, P, w.invP);
            mo[i] = *gbl(w.mag + keys[i]);
            if constexpr (EPL == kChunk) {
                if (w.det_vec) {
                    load_raw8<DT>(g + e0, gr[i]);
                    ir[i] = load_raw_idx8(w.idx + e0);
                } else {  // grad or indices not 16 / 8-byte aligned: the same items, element loads
                    load_raw8_elems<DT>(g + e0, gr[i]);
                    ir[i] = load_raw_idx8_elems(w.idx + e0);
                }
            } else {
                graw[i] = to_f32<DT>(*gbl(g + e0));
                iraw[i] = *gbl(w.idx + e0);
            }
        }
    }
    s_cbr[threadIdx.x % kCodebookMax] = cbr_v;  // every thread: no branch, so the waits stay exact
    __syncthreads();  // s_cbr
    int64_t ck = -1;   // carried block and its running max (wave-uniform)
    uint32_t cm = 0u;
#pragma unroll
    for (int i = 0; i < kDetIters; ++i) {
        const int64_t e0 = base + ((int64_t)i * kThreads + threadIdx.x) * EPL;
        const int64_t key = keys[i];
        double val = 0.0;
        uint32_t mx = 0u;
        if (e0 < N) {
            double cs = 0.0;  // every square into float64, as the reference sums them
            if constexpr (EPL == kChunk) {
#pragma unroll
                for (int k = 0; k < kChunk; ++k) {
                    const float gv = raw_elem<DT>(gr[i], k);
                    const float u = momentum_value(s_cbr[raw_idx(ir[i], k)], mo[i], gv, mc);
                    const uint32_t ub = __float_as_uint(u) & 0x7fffffffu;
                    mx = ub > mx ? ub : mx;
                    float sq = gv * gv;
                    if constexpr (DT == BF16) sq = round_dt<BF16>(sq);
                    cs += (double)sq;
                }
            } else {
                const float gv = graw[i];
                const float u = momentum_value(s_cbr[iraw[i]], mo[i], gv, mc);
                mx = __float_as_uint(u) & 0x7fffffffu;
                float sq = gv * gv;
                if constexpr (DT == BF16) sq = round_dt<BF16>(sq);
                cs = (double)sq;
            }
            val = cs;
        }
        const uint64_t heads = run_heads(key);
        const double sv = seg_suffix_sum(val, heads);
        const uint32_t sm = seg_suffix_max(mx, heads);
        const bool start = (heads >> lane) & 1ull;
        const int last = 63 - __clzll((long long)heads);
        // max: the first run continues the carried block or flushes it; runs
        // strictly inside these 64 items are complete; the last run is carried
        const int64_t k0 = __shfl(key, 0, 64);
        const uint32_t m0 = (uint32_t)__shfl((int)sm, 0, 64);
        if (k0 == ck) {
            cm = m0 > cm ? m0 : cm;
        } else {
            flush_det_max(mb, ck, nb, cm);
            ck = k0;
            cm = m0;
        }
        if (last != 0) {
            flush_det_max(mb, ck, nb, cm);
            if (start && lane != last && lane != 0 && key < nb && sm != 0u) gatomic_max(mb + key, sm);
            ck = __shfl(key, last, 64);
            cm = (uint32_t)__shfl((int)sm, last, 64);
        }
        if (start && lane != 0 && lane != last && key < nb) bsq[key] = sv;  // complete inside these items
        const int q = 2 * (i * kWaves + wave);
        if (lane == 0) {
            s_key[q] = key;
            s_sum[q] = sv;
        }
        if (lane == last) {  // a single run: the second slot repeats the key with nothing to add
            s_key[q + 1] = key;
            s_sum[q + 1] = lane == 0 ? 0.0 : sv;
        }
    }
    flush_det_max(mb, ck, nb, cm);
    __syncthreads();
    if (wave == 0) {
        const int64_t key = s_key[lane];
        const uint64_t heads = run_heads(key);
        const double sv = seg_suffix_sum(s_sum[lane], heads);
        const bool start = (heads >> lane) & 1ull;
        const int last = 63 - __clzll((long long)heads);
        if (start && lane != 0 && lane != last && key < nb) bsq[key] = sv;
        DetRec* rec = w.det_rec + wg;
        if (lane == 0) {
            rec->kf = key < nb ? key : -1;
            rec->sf = sv;
            if (last == 0) {
                rec->kl = -1;
                rec->sl = 0.0;
            }
        }
        if (lane == last && last != 0) {
            rec->kl = key < nb ? key : -1;
            rec->sl = sv;
        }
    }
}

__device__ __forceinline__ bool block_stats_fast_ok(const TensorWork& w) {
    return w.det_epl == kChunk;
}

template <int DT>
__device__ __forceinline__ void stats_block_wg(const TensorWork& w, int64_t wg, BlockStatsLds& lds) {
    if (block_stats_fast_ok(w)) stats_block_det<DT, kChunk>(w, wg, lds);
    else stats_block_det<DT, 1>(w, wg, lds);
}

// ====================================================================
// General apply: any strides, C and P; grid-stride over logical chunks of 8
// elements with nwg workgroups, element loads and stores.
// MODE 0 factored, MODE 1 block.
// ====================================================================
__device__ __forceinline__ void load_vcol(const float* __restrict__ vc, float v[8]) {
    const GX_GLOBAL f32x4* q = gbl(reinterpret_cast<const f32x4*>(vc));
    const f32x4 v0 = q[0], v1 = q[1];
    v[0] = v0.x; v[1] = v0.y; v[2] = v0.z; v[3] = v0.w;
    v[4] = v1.x; v[5] = v1.y; v[6] = v1.z; v[7] = v1.w;
}

__device__ __forceinline__ void load_vcol_any(const float* __restrict__ vc, float v[8]) {
    const GX_GLOBAL f32x4_a4* q = GX_GLOBAL_AS(const f32x4_a4, vc);
    const f32x4 v0 = q[0], v1 = q[1];
    v[0] = v0.x; v[1] = v0.y; v[2] = v0.z; v[3] = v0.w;
    v[4] = v1.x; v[5] = v1.y; v[6] = v1.z; v[7] = v1.w;
}

struct ApplyCtx {
    float row_scale;  // (1 / mean(v_row)) * (1/bc2)
    float c1;         // (1/bc1) * lr
    RefStep ref;      // fp32 factored: the reference-order stepsize
    bool wd;
    StepScalars sc;
    uint32_t kmax;
    int kk;
    uint64_t seed;
};

template <int DT, int MODE, bool SR>
__device__ __forceinline__ void apply_phase(const TensorWork& w, int64_t wg, int64_t nwg,
                                            const SharedTables& st, const SharedSR& ssr) {
    using T = typename Elem<DT>::T;
    ApplyCtx cx;
    cx.sc = read_scalars(w);
    cx.kmax = (uint32_t)(w.qt->k - 1);
    cx.kk = w.qt->k;
    cx.seed = w.seed;
    if constexpr (SR) {
        if (w.seed_dev != nullptr) cx.seed = (uint64_t)w.seed_dev[0];
    }
    cx.row_scale = 0.0f;
    cx.ref.on = false;
    if constexpr (MODE == 0) {
        const float mean = stored_mean(w);
        cx.row_scale = (1.0f / mean) * cx.sc.inv_bc2;
        if constexpr (DT == F32) cx.ref = make_ref_step(w, cx.sc, mean);
    }
    cx.c1 = cx.sc.inv_bc1 * cx.sc.lr;
    cx.wd = cx.sc.wdf != 1.0f;

    T* p = static_cast<T*>(w.p);
    const T* g = static_cast<const T*>(w.grad);
    const int64_t nchunks = (w.N + kChunk - 1) / kChunk;
    int64_t ch = wg * kThreads + threadIdx.x;
    const int64_t stride = nwg * kThreads;
    for (; ch < nchunks; ch += stride) {
        const int64_t e0 = ch * kChunk;
        const int nvalid = (int)std::min<int64_t>(kChunk, w.N - e0);
        int64_t row = div_floor(e0, w.C, w.invC);
        int64_t col = e0 - row * w.C;
        int64_t blk = div_floor(e0, w.P, w.invP);
        int64_t pin = e0 - blk * w.P;
        float gv[kChunk], pv[kChunk];
        uint32_t ix[kChunk];
        {
            int64_t r = row, c = col;
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                if (k < nvalid) {
                    gv[k] = to_f32<DT>(g[r * w.gs0 + c * w.gs1]);
                    pv[k] = w.write_p ? to_f32<DT>(p[r * w.ps0 + c * w.ps1]) : 0.0f;
                    ix[k] = w.idx[e0 + k];
                    if (++c == w.C) { c = 0; ++r; }
                } else {
                    gv[k] = 0.0f;
                    pv[k] = 0.0f;
                    ix[k] = 0u;
                }
            }
        }
        float m_old = w.mag_old[blk];
        float m_new = w.mag[blk];
        float y = w.minv[blk];
        float bstep = 0.0f;
        if constexpr (MODE == 1) bstep = w.step[blk];
        float rs = 0.0f, vr = 0.0f;
        if constexpr (MODE == 0) {
            vr = w.v0[row];
            rs = vr * cx.row_scale;
        }
        int64_t r = row, c = col;
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (k < nvalid) {
                const float u = momentum_value(st.cbr[ix[k]], m_old, gv[k], w.mc);
                const float x = (m_new > 0.0f) ? div_by_block(u, m_new, y) : 0.0f;
                uint32_t ni;
                if constexpr (SR) ni = quant_stochastic(x, ssr.cb, ssr.lut, cx.kk, cx.seed, e0 + k);
                else ni = quant_nearest(x, st.bkt, st.thr, cx.kmax);
                ix[k] = ni;
                if (w.write_p) {
                    const float q = st.cbr[ni] * m_new;
                    float pw = pv[k];
                    if (cx.wd) pw = round_dt<DT>(pw * cx.sc.wdf);
                    if constexpr (MODE == 0) {
                        if (DT == F32 && cx.ref.on) {
                            pv[k] = pw - (q * ref_step(cx.ref, vr, w.v1[c])) * cx.sc.lr;
                        } else {
                            const float h = __builtin_amdgcn_sqrtf(rs * w.v1[c]) + w.eps;
                            pv[k] = pw - q * (__builtin_amdgcn_rcpf(h) * cx.c1);
                        }
                    } else {
                        pv[k] = pw - (q * bstep) * cx.sc.lr;
                    }
                }
                if (++c == w.C) {
                    c = 0;
                    ++r;
                    if constexpr (MODE == 0) {
                        if (k + 1 < nvalid) {
                            vr = w.v0[r];
                            rs = vr * cx.row_scale;
                        }
                    }
                }
                if (++pin == w.P) {
                    pin = 0;
                    ++blk;
                    if (k + 1 < nvalid) {
                        m_old = w.mag_old[blk];
                        m_new = w.mag[blk];
                        y = w.minv[blk];
                        if constexpr (MODE == 1) bstep = w.step[blk];
                    }
                }
            }
        }
        int64_t rr = row, cc = col;
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (k < nvalid) {
                w.idx[e0 + k] = (uint8_t)ix[k];
                if (w.write_p) p[rr * w.ps0 + cc * w.ps1] = from_f32<DT>(pv[k]);
                if (++cc == w.C) { cc = 0; ++rr; }
            }
        }
    }
}

// ====================================================================
// Fast apply (the hot path): contiguous p and grad of any alignment, P >= 8,
// nearest or stochastic rounding.  Per element the only LDS traffic of nearest
// rounding is the old codeword, one 8-byte quantiser entry {thr[base], base}
// and the new codeword (a table with several thresholds in one bucket takes
// the exact search instead); the step uses sqrt(v_col) precomputed by finalize
// and one sqrt(v_row * scale) per chunk.
// ====================================================================
struct FastTables {
    union {
        uint2 fq[kFqEntries];
        struct {  // a table with several thresholds in one bucket
            uint32_t bkt[kBuckets + 4];
            float thr[kCodebookMax + 4];
        } d;
    };
    float cbr[kCodebookMax];
};

// Buckets (the last one again past the end: x = 1 lands there) and thresholds
// (+inf past the end) for quant_dense.
__device__ __forceinline__ void stage_dense(FastTables& s, const QTable* __restrict__ t) {
    const GX_GLOBAL u32x4* src = gbl(reinterpret_cast<const u32x4*>(t->bucket));
    u32x4* dst = reinterpret_cast<u32x4*>(s.d.bkt);
#pragma unroll
    for (int j = 0; j < kBuckets / 4 / kThreads; ++j) dst[threadIdx.x + j * kThreads] = src[threadIdx.x + j * kThreads];
    s.d.thr[threadIdx.x] = *gbl(t->thr + threadIdx.x);
    s.cbr[threadIdx.x] = *gbl(t->cbr + threadIdx.x);
    if (threadIdx.x < 4) {
        s.d.bkt[kBuckets + threadIdx.x] = *gbl(t->bucket + kBuckets - 1);
        s.d.thr[kCodebookMax + threadIdx.x] = __builtin_inff();
    }
}

// Nearest index for x in [-1, 1] (never NaN).  Thresholds in later buckets
// are > x, so the first two from the bucket's base on are compared whatever
// their bucket; a bucket that holds more goes on with the rest.
__device__ __forceinline__ uint32_t quant_dense(float x, const FastTables& s) {
    int b = (int)__builtin_fmaf(x, (float)(kBuckets / 2), (float)(kBuckets / 2));
    b = b < 0 ? 0 : (b > kBuckets ? kBuckets : b);
    const uint32_t e = s.d.bkt[b];
    const uint32_t base = e & 0xffffu, cnt = e >> 16;
    uint32_t idx = base + (s.d.thr[base] < x ? 1u : 0u) + (s.d.thr[base + 1] < x ? 1u : 0u);
    for (uint32_t j = 2; j < cnt; ++j) idx += s.d.thr[base + j] < x ? 1u : 0u;
    return idx;
}

// All loads of a thread's share are issued before the first LDS write.
__device__ __forceinline__ void stage_fast(FastTables& s, const QTable* __restrict__ t) {
    constexpr int kVec = kFqEntries / 2;                   // uint4 per table
    constexpr int kPer = (kVec + kThreads - 1) / kThreads;
    const GX_GLOBAL u32x4* src = gbl(reinterpret_cast<const u32x4*>(t->fq));
    u32x4* dst = reinterpret_cast<u32x4*>(s.fq);
    u32x4 v[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = threadIdx.x + j * kThreads;
        if (i < kVec) v[j] = src[i];
    }
    const float c = threadIdx.x < kCodebookMax ? *gbl(t->cbr + threadIdx.x) : 0.0f;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = threadIdx.x + j * kThreads;
        if (i < kVec) dst[i] = v[j];
    }
    if (threadIdx.x < kCodebookMax) s.cbr[threadIdx.x] = c;
}

// Stochastic rounding.  Entry j (0..k) describes the codewords around insertion
// point j: r = min(j, k-1), l = max(r-1, 0), {cb[l], cb[r], RN(1 / (cb[r] -
// cb[l])) or 0 where that is not a normal number}; lut[b] packs the range of
// insertion points of bucket b, first | last << 16.
struct SrTables {
    float cbr[kCodebookMax];
    f32x4 e[kCodebookMax + 2];
    uint32_t lut[kBuckets];
};

__device__ __forceinline__ void stage_tabs(FastTables& s, const QTable* __restrict__ t) {
    if (t->max_cnt > 1) stage_dense(s, t);
    else stage_fast(s, t);
}
__device__ __forceinline__ void stage_tabs(SrTables& s, const QTable* __restrict__ t) {
    const int kk = t->k;
    for (int j = threadIdx.x; j < kCodebookMax + 2; j += kThreads) {
        const int r = j > kk - 1 ? kk - 1 : j, l = r - 1 < 0 ? 0 : r - 1;
        const float lv = *gbl(t->cb + l), hv = *gbl(t->cb + r);
        s.e[j] = f32x4{lv, hv, block_recip(hv - lv), 0.0f};
    }
    s.cbr[threadIdx.x % kCodebookMax] = *gbl(t->cbr + threadIdx.x % kCodebookMax);
#pragma unroll 4
    for (int b = threadIdx.x; b < kBuckets; b += kThreads) {
        int lo = *gbl(t->lut + b), hi = *gbl(t->lut + b + 1);
        lo = lo < 0 ? 0 : (lo > kk ? kk : lo);
        hi = hi < lo ? lo : (hi > kk ? kk : hi);
        s.lut[b] = (uint32_t)lo | ((uint32_t)hi << 16);
    }
}

// quant_stochastic, bit for bit, for two elements at a time (z0 + k dz: their
// hash inputs; four took 141 VGPRs in the apply): one LUT read, the entries of the bucket's first insertion point and
// of the next in one go (a bucket usually holds at most one codeword), the
// probability of rounding up through the span's reciprocal with one Markstein
// correction (exact where the offset and the quotient are at least 2^-100; a
// smaller one divides), and the hash's top 24 bits, which need neither its last
// xor-shift nor the low half of its last product.
__device__ __forceinline__ void quant_sr2(const float* xs, const SrTables& s, int kk, uint64_t z0, uint64_t dz,
                                          uint32_t* ix) {
    uint32_t pk[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        int b = (int)floorf((xs[k] + 1.0f) * (float)(kBuckets / 2));
        b = b < 0 ? 0 : (b > kBuckets - 1 ? kBuckets - 1 : b);
        pk[k] = s.lut[b];
    }
    f32x4 e0[2], e1[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        e0[k] = s.e[pk[k] & 0xffffu];
        e1[k] = s.e[(pk[k] & 0xffffu) + 1u];
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const float x = xs[k];
        uint32_t j = pk[k] & 0xffffu;
        const uint32_t hi = pk[k] >> 16;
        bool up = j < hi && e0[k].y < x;
        f32x4 e = e0[k];
        if (up) { e = e1[k]; ++j; }
        while (__any(up && j < hi)) {  // several codewords in one bucket
            up = up && j < hi && e.y < x;
            if (up) { ++j; e = s.e[j]; }
        }
        const uint32_t r = j > (uint32_t)(kk - 1) ? (uint32_t)(kk - 1) : j;
        const uint32_t l = r > 0u ? r - 1u : 0u;
        const float span = e.y - e.x;
        const float v = x < e.x ? e.x : (x > e.y ? e.y : x);
        const float d = v - e.x;
        const float q0 = d * e.z;
        float p_up = __builtin_fmaf(__builtin_fmaf(-q0, span, d), e.z, q0);
        const bool odd = span > 0.0f && (e.z == 0.0f || (d != 0.0f && !(q0 >= 0x1p-100f && d >= 0x1p-100f)));
        if (__builtin_expect(__any(odd), 0)) p_up = odd ? d / span : p_up;
        if (!(span > 0.0f)) p_up = 0.0f;
        uint64_t z = z0 + dz * (uint64_t)k;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
        z = z ^ (z >> 27);
        const uint32_t zl = (uint32_t)z, zh = (uint32_t)(z >> 32);
        const uint32_t h = __umulhi(zl, 0x133111EBu) + zl * 0x94D049BBu + zh * 0x133111EBu;
        const float u01 = (float)(h >> 8) * (1.0f / 16777216.0f);
        ix[k] = u01 < p_up ? r : l;  // one codeword (l == r): either
    }
}
constexpr uint64_t kSrStep = 0x9E3779B97F4A7C15ULL;  // hash input: seed + kSrStep * (element + 1)

struct Pos {
    int64_t blk, pin;  // block of an element and its offset there
};

// Everything the fast loop touches, copied out of the descriptor once: the
// stores to p / indices could alias the descriptor memory, so fields read
// through it would be re-fetched after every store.
template <int DT>
struct FastArgs {
    using T = typename Elem<DT>::T;
    T* p;
    const T* g;
    uint8_t* idx;
    const float* mag_old;
    const float* mag;
    const float* minv;
    const float* vrow;   // factored: v_row
    const float* vcs;    // factored: sqrt(v_col)
    const float* bstep;  // block: per-block stepsize
    const QTable* qt;
    int64_t P, fB, fP;
    float row_scale, c1, eps, wdf, lr;
    bool wd;
    int kk;              // codebook size
    uint64_t seed;       // stochastic rounding
    MomentumCoef mc;
    RefStep ref;         // fp32 factored: the reference-order stepsize (vcs then holds v_col itself)
};

// Inputs of one chunk, loaded one pipeline stage ahead of its math.
template <int DT>
struct ChunkIn {
    Raw8<DT> g, p;
    RawIdx8 i;
    float vc[kChunk];
    float m_old, m_new, y, rv;  // rv: v_row (factored) or the block stepsize (block)
};

template <int DT>
__device__ __forceinline__ Pos advance_flat(const FastArgs<DT>& a, Pos q) {
    q.pin += a.fP;
    q.blk += a.fB;
    if (q.pin >= a.P) { q.pin -= a.P; ++q.blk; }
    return q;
}

// Nearest index through the global threshold table (rare fallback).
__device__ __forceinline__ uint32_t quant_global(float x, const QTable* __restrict__ qt) {
    return quant_nearest(x, qt->bucket, qt->thr, (uint32_t)(qt->k - 1));
}

// Issue the loads of one chunk: the small per-row/per-block values first, so
// that waiting for them never waits for the streams issued after them.
template <int DT>
__device__ __forceinline__ void flat_load(const FastArgs<DT>& a, const Pos& ps, int64_t e0, ChunkIn<DT>& in) {
    in.m_old = *gbl(a.mag_old + ps.blk);
    in.m_new = *gbl(a.mag + ps.blk);
    in.y = *gbl(a.minv + ps.blk);
    in.rv = *gbl(a.bstep + ps.blk);
    load_raw8_any<DT>(a.g + e0, in.g);
    in.i = load_raw_idx8_any(a.idx + e0);
    load_raw8_any<DT>(a.p + e0, in.p);
}

// Requantise and apply one chunk: new indices in ix, new parameter values
// in pv.  g and p are the chunk's grads and parameters as floats, iv its old
// indices, vc its columns' sqrt(v_col) (v_col on the fp32 reference path),
// rv its v_row (factored) or block stepsize (block), e0 its first element
// (stochastic rounding).  general_q: the table may hold several thresholds per
// bucket (the fq entries do not describe it), so every element takes the exact
// search.
// LDSQ: ft was staged for a general_q table (else such elements search it in
// global memory).
template <int DT, int MODE, int LF, bool LDSQ = true, class Tabs>
__device__ __forceinline__ void chunk_math(const FastArgs<DT>& a, const Tabs& ft, const float g[kChunk],
                                           const float p[kChunk], const RawIdx8& iv, const float vc[kChunk],
                                           float m_old, float m_new, float y, float rv, bool general_q,
                                           int64_t e0, uint32_t ix[kChunk], float pv[kChunk]) {
    constexpr bool SR = std::is_same_v<Tabs, SrTables>;
    const float tb = 0x1.00001p-100f * fmaxf(m_new, 1.0f);
    float xs[kChunk];
    bool bad = (y == 0.0f) || (!LDSQ && general_q);
#pragma unroll
    for (int k = 0; k < kChunk; ++k) {
        const float u = momentum_value<LF>(ft.cbr[raw_idx(iv, k)], m_old, g[k], a.mc);
        const float q0 = u * y;
        const float r = __builtin_fmaf(-q0, m_new, u);
        xs[k] = __builtin_fmaf(r, y, q0);
        bad = bad || !(fabsf(u) >= tb);
    }
    if (__builtin_expect(__any(bad), 0)) {
        const bool nz = m_new > 0.0f;
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            const float u = momentum_value<LF>(ft.cbr[raw_idx(iv, k)], m_old, g[k], a.mc);
            const float x = nz ? div_by_block(u, m_new, y) : 0.0f;
            if constexpr (SR) xs[k] = x;
            else ix[k] = quant_global(x, a.qt);
        }
    } else if constexpr (!SR) {
        if (LDSQ && general_q) {
#pragma unroll
            for (int k = 0; k < kChunk; ++k) ix[k] = quant_dense(xs[k], ft);
        } else {
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                int b = (int)__builtin_fmaf(xs[k], (float)(kBuckets / 2), (float)(kBuckets / 2));
                b = b < 0 ? 0 : (b > kFqEntries - 1 ? kFqEntries - 1 : b);  // |x| <= 1 already (v_med3)
                const uint2 e = ft.fq[b];
                ix[k] = e.y + (__uint_as_float(e.x) < xs[k] ? 1u : 0u);
            }
        }
    }
    if constexpr (SR) {
        const uint64_t z0 = a.seed + kSrStep * ((uint64_t)e0 + 1ull);
#pragma unroll
        for (int k = 0; k < kChunk; k += 2) {
            quant_sr2(xs + k, ft, a.kk, z0 + (uint64_t)k * kSrStep, kSrStep, ix + k);
            __builtin_amdgcn_sched_barrier(0);  // two at a time: registers
        }
    }
    if constexpr (MODE == 0 && DT == F32) {
        if (a.ref.on) {  // reference order; vc holds v_col
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                const float q = ft.cbr[ix[k]] * m_new;
                float pw = p[k];
                if (a.wd) pw = round_dt<DT>(pw * a.wdf);
                pv[k] = pw - (q * ref_step(a.ref, rv, vc[k])) * a.lr;
            }
            return;
        }
    }
    float sr = 0.0f;
    if constexpr (MODE == 0) sr = __builtin_amdgcn_sqrtf(rv * a.row_scale);
#pragma unroll
    for (int k = 0; k < kChunk; ++k) {
        const float q = ft.cbr[ix[k]] * m_new;
        float pw = p[k];
        if (a.wd) pw = round_dt<DT>(pw * a.wdf);
        if constexpr (MODE == 0) {
            pv[k] = pw - q * (__builtin_amdgcn_rcpf(__builtin_fmaf(sr, vc[k], a.eps)) * a.c1);
        } else {
            pv[k] = pw - (q * rv) * a.lr;  // the reference's order (gefen.py:3806-3818)
        }
    }
}

template <int DT, int MODE, int LF, class Tabs>
__device__ __forceinline__ void fast_math(const FastArgs<DT>& a, const Tabs& ft, const ChunkIn<DT>& in,
                                          bool general_q, int64_t e0, uint32_t ix[kChunk], float pv[kChunk]) {
    float g[kChunk], p[kChunk];
#pragma unroll
    for (int k = 0; k < kChunk; ++k) {
        g[k] = raw_elem<DT>(in.g, k);
        p[k] = raw_elem<DT>(in.p, k);
    }
    chunk_math<DT, MODE, LF>(a, ft, g, p, in.i, in.vc, in.m_old, in.m_new, in.y, in.rv, general_q, e0,
                             ix, pv);
}

// Requantise and apply one chunk, then store its indices and parameters.
template <int DT, int MODE, int LF, class Tabs>
__device__ __forceinline__ void fast_compute(const FastArgs<DT>& a, const Tabs& ft, int64_t e0,
                                             const ChunkIn<DT>& in) {
    uint32_t ix[kChunk];
    float pv[kChunk];
    fast_math<DT, MODE, LF>(a, ft, in, false, e0, ix, pv);
    store_idx8(a.idx + e0, ix);
    store8<DT>(a.p + e0, pv);
}

template <int DT>
__device__ __forceinline__ FastArgs<DT> make_fast_args(const TensorWork& w, float row_scale) {
    FastArgs<DT> a;
    const StepScalars sc = read_scalars(w);
    a.p = static_cast<typename Elem<DT>::T*>(w.p);
    a.g = static_cast<const typename Elem<DT>::T*>(w.grad);
    a.idx = w.idx;
    a.mag_old = w.mag_old;
    a.mag = w.mag;
    a.minv = w.minv;
    a.vrow = w.v0;
    a.vcs = w.vcs;
    a.bstep = w.step;
    a.qt = w.qt;
    a.P = w.P; a.fB = w.fB; a.fP = w.fP;
    a.row_scale = row_scale;
    a.c1 = sc.inv_bc1 * sc.lr;
    a.eps = w.eps;
    a.wdf = sc.wdf;
    a.lr = sc.lr;
    a.wd = sc.wdf != 1.0f;
    a.kk = w.qt->k;
    a.seed = w.sr && w.seed_dev != nullptr ? (uint64_t)w.seed_dev[0] : w.seed;
    a.mc = w.mc;
    a.ref.on = false;
    if constexpr (DT == F32) {
        if (w.mode == 0 && w.bc2_div > 0.0f) {
            a.ref = make_ref_step(w, sc, stored_mean(w));
            a.vcs = w.v1;
        }
    }
    return a;
}

// One chunk of `nv` elements (8, or fewer at the end of a flat tensor) whose
// first `na` lie in block blk and the rest in the next: math and stores.  A
// lane whose chunk holds a border (na < nv) first stores what block blk gives
// for the whole chunk, then the elements of the next block over it (a wave's
// stores to one address stay in order, and no other wave touches the chunk):
// keeping the first results for a select instead cost the registers of the
// fourth wave per SIMD.
// BORDERS false: na and nv are 8.
template <int DT, int MODE, int LF, bool BORDERS, class Tabs>
__device__ __forceinline__ void chunk_step(const FastArgs<DT>& a, const Tabs& ft, ChunkIn<DT>& in, int64_t blk,
                                           int na, int nv, bool store, bool write_p, bool general_q, int64_t e0) {
    uint32_t ix[kChunk];
    float pv[kChunk];
    fast_math<DT, MODE, LF>(a, ft, in, general_q, e0, ix, pv);
    if (store && (!BORDERS || nv == kChunk)) {
        store_idx8_any(a.idx + e0, ix);
        if (write_p) store8_any<DT>(a.p + e0, pv);
    }
    if constexpr (!BORDERS) return;
    const bool border = na < nv;
    if (__builtin_expect(!__any(border || nv < kChunk), 1)) return;
    auto put = [&](int k0, int k1) {
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (k < k0 || k >= k1) continue;
            *gbl(a.idx + e0 + k) = (uint8_t)ix[k];
            if (write_p) *gbl(a.p + e0 + k) = from_f32<DT>(pv[k]);
        }
    };
    if (store && nv < kChunk) put(0, nv);
    if (!__any(border)) return;
    const int64_t b = border ? blk + 1 : blk;
    in.m_old = *gbl(a.mag_old + b);
    in.m_new = *gbl(a.mag + b);
    in.y = *gbl(a.minv + b);
    if constexpr (MODE == 1) in.rv = *gbl(a.bstep + b);
    fast_math<DT, MODE, LF>(a, ft, in, general_q, e0, ix, pv);
    if (store && border) put(na, nv);
}

// Block path, contiguous p and grad, a linear walk.  Workgroup wg owns chunks
// [wg*256*kApplyChunksPerThread, ...), thread t takes t, t+256, ... of them.
// HOT: P and N multiples of 8, everything aligned, nearest rounding.  Otherwise
// any alignment, N and P >= 8; two chunks are computed while the next two load.
template <int DT, int LF, bool HOT, class Tabs>
__device__ __forceinline__ void apply_flat(const TensorWork& w, int64_t wg, const Tabs& ft) {
    constexpr int MODE = 1;
    const FastArgs<DT> a = make_fast_args<DT>(w, 0.0f);
    const bool general_q = !std::is_same_v<Tabs, SrTables> && w.qt->max_cnt > 1;
    const bool write_p = w.write_p != 0;
    const int64_t N = w.N, nchunks = (N + kChunk - 1) / kChunk;
    const int64_t first = wg * (kThreads * kApplyChunksPerThread) + threadIdx.x;
    if (first >= nchunks) return;
    // chunks of this thread: first + i*256 for i < n (n >= 1)
    const int n = (int)std::min<int64_t>(kApplyChunksPerThread, (nchunks - first + kThreads - 1) / kThreads);
    Pos p0;
    {
        const int64_t e0 = first * kChunk;
        p0.blk = div_floor(e0, w.P, w.invP);
        p0.pin = e0 - p0.blk * w.P;
    }
    Pos p1 = advance_flat<DT>(a, p0);
    ChunkIn<DT> A, B;
    if constexpr (HOT) {
        if ((wg + 1) * (kThreads * kApplyChunksPerThread) <= nchunks && write_p && !general_q) {
            // A full workgroup: straight-line code with every load and store
            // unconditional, so each wait names exactly the chunk about to be
            // computed and the next two chunks stay in flight.  (A load or store
            // behind a branch makes the compiler assume, at the join, the path
            // with fewer operations in flight, and the waits then drain the
            // prefetched chunks as well.)
            flat_load<DT>(a, p0, first * kChunk, A);
            flat_load<DT>(a, p1, (first + kThreads) * kChunk, B);
#pragma unroll
            for (int i = 0; i < (int)kApplyChunksPerThread; i += 2) {
                const int64_t ea = (first + (int64_t)i * kThreads) * kChunk;
                const int64_t eb = ea + kThreads * kChunk;
                const Pos p2 = advance_flat<DT>(a, p1);
                const Pos p3 = advance_flat<DT>(a, p2);
                fast_compute<DT, MODE, LF>(a, ft, ea, A);
                if (i + 2 < (int)kApplyChunksPerThread) flat_load<DT>(a, p2, ea + 2 * kThreads * kChunk, A);
                fast_compute<DT, MODE, LF>(a, ft, eb, B);
                if (i + 3 < (int)kApplyChunksPerThread) flat_load<DT>(a, p3, eb + 2 * kThreads * kChunk, B);
                p1 = p3;
            }
            return;
        }
#pragma unroll 1
        for (int i = 0; i < n; ++i) {
            const int64_t e0 = (first + (int64_t)i * kThreads) * kChunk;
            flat_load<DT>(a, p0, e0, A);
            chunk_step<DT, MODE, LF, false>(a, ft, A, p0.blk, kChunk, kChunk, true, write_p, general_q, e0);
            p0 = advance_flat<DT>(a, p0);
        }
        return;
    }
    auto load = [&](const Pos& q, int64_t e0, ChunkIn<DT>& in) {
        if (e0 + kChunk <= N) {
            flat_load<DT>(a, q, e0, in);
            return;
        }
        // the tensor's last elements, one by one (the last one again past its end)
        in.m_old = *gbl(a.mag_old + q.blk);
        in.m_new = *gbl(a.mag + q.blk);
        in.y = *gbl(a.minv + q.blk);
        in.rv = *gbl(a.bstep + q.blk);
        const int64_t last = N - 1 - e0;
        auto at = [&](int k) { return e0 + (k < last ? k : last); };
        uint32_t lo = 0u, hi = 0u;
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            const uint32_t v = *gbl(a.idx + at(k));
            if (k < 4) lo |= v << (8 * k);
            else hi |= v << (8 * (k - 4));
        }
        in.i = RawIdx8{lo, hi};
        if constexpr (DT == F32) {
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                in.g.f[k] = *gbl(a.g + at(k));
                in.p.f[k] = *gbl(a.p + at(k));
            }
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                in.g.w[k] = (uint32_t)*gbl(a.g + at(2 * k)) | ((uint32_t)*gbl(a.g + at(2 * k + 1)) << 16);
                in.p.w[k] = (uint32_t)*gbl(a.p + at(2 * k)) | ((uint32_t)*gbl(a.p + at(2 * k + 1)) << 16);
            }
        }
    };
    auto compute = [&](const Pos& q, int64_t e0, ChunkIn<DT>& in) {
        const int na = (int)std::min<int64_t>(kChunk, a.P - q.pin);
        const int nv = (int)std::min<int64_t>(kChunk, N - e0);
        chunk_step<DT, MODE, LF, true>(a, ft, in, q.blk, na, nv, true, write_p, general_q, e0);
    };
    load(p0, first * kChunk, A);
    if (n > 1) load(p1, (first + kThreads) * kChunk, B);
#pragma unroll 1
    for (int i = 0; i < n; i += 2) {
        const int64_t ea = (first + (int64_t)i * kThreads) * kChunk;
        const int64_t eb = ea + kThreads * kChunk;
        const Pos p2 = advance_flat<DT>(a, p1);
        const Pos p3 = advance_flat<DT>(a, p2);
        compute(p0, ea, A);
        if (i + 2 < n) load(p2, ea + 2 * kThreads * kChunk, A);
        if (i + 1 < n) compute(p1, eb, B);
        if (i + 3 < n) load(p3, eb + 2 * kThreads * kChunk, B);
        p0 = p2;
        p1 = p3;
    }
}

// Factored apply, contiguous p and grad.  A row is cut into w.a_segs even
// segments of w.a_cols <= 512 columns; 1 << w.a_lg lanes take a segment, 8
// columns each, a wave 64 >> a_lg rows at a time.  A task is w.a_steps such row
// steps of one segment, segment-fastest; wave v of workgroup wg takes task 4*wg
// + v.  Lanes past the segment's last whole chunk repeat the segment's last 8
// columns: in each step every lane has loaded before any stores, and
// overlapping lanes store the same values, so no chunk needs a mask.  A lane
// keeps its 8 columns' sqrt(v_col) in registers.
// HOT (C >= 512, C and P multiples of 8, blocks of at least kShortPeriod,
// everything aligned, nearest rounding): a task whose segment lies inside one
// block in every row takes v_row and the block's magnitudes and reciprocal as
// scalar loads; per 8 elements the lane loads only g, p and the indices (the
// per-chunk v_col and block loads of a linear walk cost ~6% of the apply time).
// Two rows are in flight while two are computed.  Otherwise (any alignment, C >=
// 8, P >= 8, stochastic rounding) each lane loads its row's and block's values
// with its chunk (43M fp16 elements with stochastic rounding: 166 us + 81 for
// the odd-sized two through element loads -> 195 in one launch).  The two are kernels of their own: in one, the borders'
// registers cost the HOT tasks their fourth wave per SIMD (1.05e9 elements 1530
// -> 1592 us).
template <int DT, int LF, bool HOT, class Tabs>
__device__ __forceinline__ void apply_tasks(const TensorWork& w, int64_t wg, const Tabs& ft, float row_scale) {
    const FastArgs<DT> a = make_fast_args<DT>(w, row_scale);
    const bool general_q = !std::is_same_v<Tabs, SrTables> && w.qt->max_cnt > 1;
    const bool write_p = w.write_p != 0;
    const int64_t C = w.C, R = w.R, P = w.P;
    const int64_t t = wg * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t rt = t / w.a_segs;
    const int64_t cs = (t - rt * w.a_segs) * w.a_cols;
    const int64_t ce = std::min<int64_t>(cs + w.a_cols, C);
    const int lane = threadIdx.x & 63, lg = w.a_lg, rpw = 64 >> lg, steps = w.a_steps;
    const int64_t r0 = rt * steps * rpw;
    if (r0 >= R) return;
    const int64_t c = std::min<int64_t>(cs + (lane & ((1 << lg) - 1)) * kChunk, ce - kChunk);
    float vc[kChunk];
    load_vcol_any(a.vcs + c, vc);
    if (HOT && rpw == 1 && steps == kRowsPerTask && r0 + kRowsPerTask <= R && write_p && !general_q) {
        // block and offset of the segment's first element, row by row
        // (wave-uniform): one block per row when pin + seglen <= P
        int64_t bk[kRowsPerTask];
        bool uniform = true;
        {
            const int64_t e_first = r0 * C + cs;
            int64_t b = div_floor(e_first, P, w.invP);
            int64_t pin = e_first - b * P;
            const int64_t dB = div_floor(C, P, w.invP);
            const int64_t dP = C - dB * P;
#pragma unroll
            for (int i = 0; i < kRowsPerTask; ++i) {
                bk[i] = b;
                uniform = uniform && pin + (ce - cs) <= P;
                pin += dP;
                b += dB;
                if (pin >= P) { pin -= P; ++b; }
            }
        }
        if (uniform) {
            auto load_row = [&](int i, ChunkIn<DT>& in) {
                const int64_t r = r0 + i;
                const int64_t e0 = r * C + c;
                in.m_old = sload(a.mag_old + bk[i]);
                in.m_new = sload(a.mag + bk[i]);
                in.y = sload(a.minv + bk[i]);
                in.rv = sload(a.vrow + r);
                load_raw8<DT>(a.g + e0, in.g);
                in.i = load_raw_idx8(a.idx + e0);
                load_raw8<DT>(a.p + e0, in.p);
            };
            ChunkIn<DT> A, B;
            load_row(0, A);
            load_row(1, B);
#pragma unroll
            for (int i = 0; i < kRowsPerTask; i += 2) {
#pragma unroll
                for (int k = 0; k < kChunk; ++k) { A.vc[k] = vc[k]; B.vc[k] = vc[k]; }
                fast_compute<DT, 0, LF>(a, ft, (r0 + i) * C + c, A);
                if (i + 2 < kRowsPerTask) load_row(i + 2, A);
                fast_compute<DT, 0, LF>(a, ft, (r0 + i + 1) * C + c, B);
                if (i + 3 < kRowsPerTask) load_row(i + 3, B);
            }
            return;
        }
    }
    // rows of step i: r0 + i * rpw + sub; a lane past R loads row R - 1 and stores nothing
    const int sub = lane >> lg;
    const int n = (int)std::min<int64_t>(steps, (R - r0 + rpw - 1) / rpw);
    struct At {
        int64_t blk;
        int na;  // elements of the chunk in that block (8: all)
    };
    auto load = [&](int i, ChunkIn<DT>& in, At& at) {
        const int64_t r = std::min<int64_t>(r0 + (int64_t)i * rpw + sub, R - 1);
        const int64_t e0 = r * C + c;
        at.blk = div_floor(e0, P, w.invP);
        at.na = HOT ? kChunk : (int)std::min<int64_t>(kChunk, P - (e0 - at.blk * P));
        in.m_old = *gbl(a.mag_old + at.blk);
        in.m_new = *gbl(a.mag + at.blk);
        in.y = *gbl(a.minv + at.blk);
        in.rv = *gbl(a.vrow + r);
        load_raw8_any<DT>(a.g + e0, in.g);
        in.i = load_raw_idx8_any(a.idx + e0);
        load_raw8_any<DT>(a.p + e0, in.p);
    };
    auto compute = [&](int i, ChunkIn<DT>& in, const At& at) {
        const int64_t r = r0 + (int64_t)i * rpw + sub;
#pragma unroll
        for (int k = 0; k < kChunk; ++k) in.vc[k] = vc[k];
        chunk_step<DT, 0, LF, !HOT>(a, ft, in, at.blk, at.na, kChunk, r < R, write_p, general_q, r * C + c);
    };
    ChunkIn<DT> A, B;
    At pa, pb;
    if constexpr (HOT) {  // a block border inside the segment, or fewer rows: one row at a time
#pragma unroll 1
        for (int i = 0; i < n; ++i) {
            load(i, A, pa);
            compute(i, A, pa);
        }
    } else {
        load(0, A, pa);
        if (n > 1) load(1, B, pb);
#pragma unroll 1
        for (int i = 0; i < n; i += 2) {
            compute(i, A, pa);
            if (i + 2 < n) load(i + 2, A, pa);
            if (i + 1 < n) compute(i + 1, B, pb);
            if (i + 3 < n) load(i + 3, B, pb);
        }
    }
}

// Apply of a transposed view, MODE 0 factored / 1 block (nearest rounding; a
// table with several thresholds per bucket takes the exact search for every
// element).  Wave v of workgroup wg takes kTvTilesPerWave consecutive 64 x 64
// tiles in tile-row-fastest order, so a workgroup reads 1 KB runs of its 64
// storage rows.  (The other half of each 128-byte index line belongs to the
// next tile column and is fetched again; orders that read both halves in
// the same step shorten those runs and measured ~20% slower.)  Per tile a
// lane loads its sub-block's g and p
// vectors and index chunks, sqrt(v_col) of its 8 columns and v_row of its 8
// rows (factored) and the block values: scalar loads of the tile's first
// kTvFew blocks when it touches no more, else per chunk.  Then chunk by
// chunk it requantises and applies (indices stored per chunk) and collects
// the new parameters into storage-row vectors, stored at the end.
template <int DT, int MODE, int LF>
__device__ __forceinline__ void apply_tv(const TensorWork& w, int64_t wg, const FastTables& ft, float row_scale) {
    const FastArgs<DT> a = make_fast_args<DT>(w, row_scale);
    const int64_t R = w.R, C = w.C, P = w.P, ldg = w.gs1, ldp = w.ps1, nb = w.nb;
    const double invP = w.invP;
    const int64_t nrt = (R + kTv - 1) / kTv;
    const int64_t ntiles = nrt * ((C + kTv - 1) / kTv);
    const int lane = threadIdx.x & 63, la = lane & 7, lb = lane >> 3;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool general_q = w.qt->max_cnt > 1;
    const int64_t dB = div_floor(C, P, invP);
    const int64_t dP = C - dB * P;
    const int64_t t0 = (wg * kWaves + wave) * (int64_t)kTvTilesPerWave;
#pragma unroll 1
    for (int it = 0; it < kTvTilesPerWave; ++it) {
        const int64_t T = t0 + it;
        if (T >= ntiles) break;
        const int64_t r0 = (T % nrt) * kTv, c0 = (T / nrt) * kTv;
        const int64_t r = r0 + 8 * la, c = c0 + 8 * lb;
        const bool ok = r < R && c < C;
        // lanes outside the tensor load the last sub-block and store nothing
        const int64_t rl = r < R ? r : R - kChunk, cl = c < C ? c : C - kChunk;
        Raw8<DT> gv[kChunk], pv[kChunk];
        RawIdx8 iv[kChunk];
        float vc[kChunk], vr[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            load_raw8<DT>(a.g + (cl + k) * ldg + rl, gv[k]);
            load_raw8<DT>(a.p + (cl + k) * ldp + rl, pv[k]);
        }
#pragma unroll
        for (int j = 0; j < kChunk; ++j) iv[j] = load_raw_idx8_cached(a.idx + (rl + j) * C + cl);
        if constexpr (MODE == 0) {
            load_vcol(a.vcs + cl, vc);
            load_vcol(a.vrow + rl, vr);
        } else {
#pragma unroll
            for (int k = 0; k < kChunk; ++k) vc[k] = vr[k] = 0.0f;
        }
        // block values of the lane's chunks
        float mo[kChunk], mn[kChunk], y[kChunk], bs[kChunk];
        const int64_t r_last = std::min<int64_t>(r0 + kTv, R) - 1, c_last = std::min<int64_t>(c0 + kTv, C) - 1;
        const int64_t b_lo = uniform64(div_floor(r0 * C + c0, P, invP));
        const int64_t b_hi = uniform64(div_floor(r_last * C + c_last, P, invP));
        if (b_hi - b_lo < kTvFew) {
            float fo[kTvFew], fn[kTvFew], fy[kTvFew], fs[kTvFew];
            tv_sload_few(a.mag_old, b_lo, nb, fo);
            tv_sload_few(a.mag, b_lo, nb, fn);
            tv_sload_few(a.minv, b_lo, nb, fy);
            if constexpr (MODE == 1) tv_sload_few(a.bstep, b_lo, nb, fs);
            int q[kChunk];
            tv_chunk_blocks(rl, cl, C, P, invP, dB, dP, b_lo, q);
#pragma unroll
            for (int j = 0; j < kChunk; ++j) {
                mo[j] = tv_pick(q[j], fo);
                mn[j] = tv_pick(q[j], fn);
                y[j] = tv_pick(q[j], fy);
                bs[j] = MODE == 1 ? tv_pick(q[j], fs) : 0.0f;
            }
        } else {
            const int64_t e = rl * C + cl;
            int64_t b = div_floor(e, P, invP);
            int64_t pin = e - b * P;
#pragma unroll
            for (int j = 0; j < kChunk; ++j) {
                mo[j] = *gbl(a.mag_old + b);
                mn[j] = *gbl(a.mag + b);
                y[j] = *gbl(a.minv + b);
                bs[j] = MODE == 1 ? *gbl(a.bstep + b) : 0.0f;
                pin += dP;
                b += dB;
                if (pin >= P) { pin -= P; ++b; }
            }
        }
        float po[kChunk][kChunk];  // new parameters: po[k][j] = element (j, k)
#pragma unroll
        for (int j = 0; j < kChunk; ++j) {
            float gj[kChunk], pj[kChunk];
#pragma unroll
            for (int k = 0; k < kChunk; ++k) {
                gj[k] = raw_elem<DT>(gv[k], j);
                pj[k] = raw_elem<DT>(pv[k], j);
            }
            uint32_t ix[kChunk];
            float pn[kChunk];
            chunk_math<DT, MODE, LF, false>(a, ft, gj, pj, iv[j], vc, mo[j], mn[j], y[j], MODE == 0 ? vr[j] : bs[j],
                                     general_q, 0, ix, pn);
            if (ok) store_idx8(a.idx + (r + j) * C + c, ix);
#pragma unroll
            for (int k = 0; k < kChunk; ++k) po[k][j] = pn[k];
        }
        if (ok) {
#pragma unroll
            for (int k = 0; k < kChunk; ++k) store8<DT>(a.p + (c + k) * ldp + r, po[k]);
        }
    }
}

template <int DT, int MODE>
__device__ __forceinline__ void apply_tv_wg(const TensorWork& w, int64_t wg, FastTables& ft) {
    stage_fast(ft, w.qt);
    float row_scale = 0.0f;
    if constexpr (MODE == 0) {
        const StepScalars sc = read_scalars(w);
        row_scale = (1.0f / stored_mean(w)) * sc.inv_bc2;
    }
    __syncthreads();
    if (w.mc.small) apply_tv<DT, MODE, kLerpSmall>(w, wg, ft, row_scale);
    else apply_tv<DT, MODE, kLerpLarge>(w, wg, ft, row_scale);
}

// LDS of the apply kernels.
template <bool SR, int FAST>
struct ApplyLds {
    std::conditional_t<SR, SrTables, FastTables> f;
};
template <bool SR>
struct ApplyLds<SR, 0> {
    SharedTables st;
    SharedSR ssr;
};

// One apply workgroup.  FAST as w.fast_apply: 1 the HOT forms, 3 contiguous p
// and grad of any alignment, 0 any strides (grid-stride over all chunks).
template <int DT, int MODE, bool SR, int FAST>
__device__ __forceinline__ void apply_wg(const TensorWork& w, int64_t wg, int64_t nwg, ApplyLds<SR, FAST>& lds) {
    const QTable* qt = w.qt;
    if constexpr (FAST != 0) {
        constexpr bool HOT = FAST == 1;
        stage_tabs(lds.f, qt);
        float row_scale = 0.0f;
        if constexpr (MODE == 0) {
            const StepScalars sc = read_scalars(w);
            row_scale = (1.0f / stored_mean(w)) * sc.inv_bc2;
        }
        __syncthreads();
        if constexpr (MODE == 0) {
            if (w.mc.small) apply_tasks<DT, kLerpSmall, HOT>(w, wg, lds.f, row_scale);
            else apply_tasks<DT, kLerpLarge, HOT>(w, wg, lds.f, row_scale);
        } else {
            if (w.mc.small) apply_flat<DT, kLerpSmall, HOT>(w, wg, lds.f);
            else apply_flat<DT, kLerpLarge, HOT>(w, wg, lds.f);
        }
    } else {
        stage_tables(lds.st, qt);
        if constexpr (SR) stage_sr(lds.ssr, qt);
        __syncthreads();
        apply_phase<DT, MODE, SR>(w, wg, nwg, lds.st, lds.ssr);
    }
}

// ====================================================================
// Kernels.  Single parameter: descriptor by value.  Multi-tensor: a
// segment table maps launch workgroups to (descriptor, local workgroup).
// ====================================================================
// Workgroup b of a launch of G, renumbered so that each XCD (the hardware
// deals consecutive workgroups to the 8 XCDs in turn) runs one contiguous
// range of the launch's logical workgroups.
__device__ __forceinline__ int64_t xcd_contiguous(int64_t b, int64_t G) {
    const int64_t q = G / 8, r = G % 8, x = b % 8;
    return x * q + (x < r ? x : r) + b / 8;
}

// One LDS image for every form (each instantiation would otherwise declare its
// own): four workgroups per CU with it.
union StatsLds {
    FactStatsLds f;
    BlockStatsLds b;
};

template <int DT, bool FAST>
__device__ __forceinline__ void stats_factored_wg(const TensorWork& w, int64_t wg, FactStatsLds& lds) {
    if constexpr (FAST) {
        if (w.lg_lanes >= 0) {
            if (w.mc.small) stats_lanes<DT, kLerpSmall>(w, wg, lds);
            else stats_lanes<DT, kLerpLarge>(w, wg, lds);
            return;
        }
    }
    if (w.mc.small) stats_factored<DT, FAST, kLerpSmall>(w, wg, lds);
    else stats_factored<DT, FAST, kLerpLarge>(w, wg, lds);
}

template <int DT, bool FAST>
__global__ void __launch_bounds__(kThreads) k_factored_stats(TensorWork w) {
    __shared__ FactStatsLds lds;
    stats_factored_wg<DT, FAST>(w, blockIdx.x, lds);
}

template <int DT>
__global__ void __launch_bounds__(kThreads) k_factored_stats_tv(TensorWork w) {
    stats_tv_wg<DT, 0>(w, blockIdx.x);
}

template <int DT>
__global__ void __launch_bounds__(kThreads) k_apply_tv(TensorWork w) {
    __shared__ FastTables ft;
    apply_tv_wg<DT, 0>(w, blockIdx.x, ft);
}

template <int DT>
__global__ void __launch_bounds__(kThreads) k_block_stats(TensorWork w) {
    __shared__ BlockStatsLds lds;
    stats_block_wg<DT>(w, blockIdx.x, lds);
}

template <int DT, int MODE, bool SR, int FAST>
__global__ void __launch_bounds__(kThreads) k_apply(TensorWork w) {
    __shared__ ApplyLds<SR, FAST> lds;
    apply_wg<DT, MODE, SR, FAST>(w, blockIdx.x, gridDim.x, lds);
}

// Factored stats of a launch group; the group's block-path tensors of the
// same dtype (not transposed views) ride in the same launch.
template <int DT, bool FAST>
__global__ void __launch_bounds__(kThreads, FAST && DT != F32 ? 4 : 2) k_mt_factored_stats(const TensorWork* __restrict__ ws,
                                                                SegTable tb) {
    const Seg sg = find_seg(tb, blockIdx.x);
    const TensorWork& w = ws[sg.t];
    const int64_t local = (int64_t)blockIdx.x - sg.wg_begin;
    __shared__ StatsLds lds;
    if (w.mode != 0) {
        stats_block_wg<DT>(w, local, lds.b);
        return;
    }
    stats_factored_wg<DT, FAST>(w, local, lds.f);
}

template <int DT, int MODE>
__global__ void __launch_bounds__(kThreads) k_mt_stats_tv(const TensorWork* __restrict__ ws, SegTable tb) {
    const Seg sg = find_seg(tb, blockIdx.x);
    stats_tv_wg<DT, MODE>(ws[sg.t], (int64_t)blockIdx.x - sg.wg_begin);
}

template <int DT, int MODE>
// Workgroups in XCD-contiguous order: a tile's index chunks are the first or
// second half of 128-byte lines whose other half a workgroup a few places
// later reads, which then hits the same L2 (measured on the Qwen3-4B views:
// 2.07 -> 1.76 GB read per launch, the algorithmic bytes, at the same speed).
__global__ void __launch_bounds__(kThreads) k_mt_apply_tv(const TensorWork* __restrict__ ws, SegTable tb) {
    __shared__ FastTables ft;
    const int64_t L = xcd_contiguous(blockIdx.x, gridDim.x);
    const Seg sg = find_seg(tb, L);
    apply_tv_wg<DT, MODE>(ws[sg.t], L - sg.wg_begin, ft);
}

// Waves per SIMD of the apply.  Stochastic rounding is bound by its arithmetic and
// LDS reads: 4 waves in 128 VGPRs against 3 in 141 took the step of 4096 x 4096
// bf16 from 97 to 85 us (factored 103 to 91, 9001 x 4111 fp16 191 to 174).
template <bool SR, int FAST>
constexpr int kApplyWaves = FAST == 1 || (SR && FAST == 3) ? 4 : SR ? 2 : 3;

// Apply of a launch group; with MODE 0 the group's block-path tensors of the
// same dtype and variant (not transposed views) ride in the same launch.
template <int DT, int MODE, bool SR, int FAST>
// Each XCD runs a contiguous range of the launch's workgroups, i.e. streams
// its own part of each tensor (measured on the Llama-3-8B set: apply
// 11.51-11.61 -> 11.42-11.44 ms, with a smaller spread between processes).
__global__ void __launch_bounds__(kThreads, (kApplyWaves<SR, FAST>)) k_mt_apply(const TensorWork* __restrict__ ws,
                                                                                         SegTable tb) {
    __shared__ ApplyLds<SR, FAST> lds;
    const int64_t L = xcd_contiguous(blockIdx.x, gridDim.x);
    const Seg sg = find_seg(tb, L);
    const TensorWork& w = ws[sg.t];
    const int64_t local = L - sg.wg_begin;
    if (MODE == 0 && w.mode != 0) {
        apply_wg<DT, 1, SR, FAST>(w, local, w.apply_wgs, lds);
        return;
    }
    apply_wg<DT, MODE, SR, FAST>(w, local, w.apply_wgs, lds);
}

// ====================================================================
// Launchers
// ====================================================================
template <int DT>
void StepKernels<DT>::stats(const TensorWork& w, hipStream_t s) {
    const dim3 grid((unsigned)w.stats_wgs), block(kThreads);
    if (w.mode != 0) hipLaunchKernelGGL(k_block_stats<DT>, grid, block, 0, s, w);
    else if (w.fast_stats == 2) hipLaunchKernelGGL(k_factored_stats_tv<DT>, grid, block, 0, s, w);
    else if (w.fast_stats) hipLaunchKernelGGL((k_factored_stats<DT, true>), grid, block, 0, s, w);
    else hipLaunchKernelGGL((k_factored_stats<DT, false>), grid, block, 0, s, w);
}

template <int DT, int MODE>
static void launch_apply(const TensorWork& w, hipStream_t s) {
    const dim3 grid((unsigned)w.apply_wgs), block(kThreads);
    if (w.fast_apply == 1) {
        hipLaunchKernelGGL((k_apply<DT, MODE, false, 1>), grid, block, 0, s, w);
    } else if (w.fast_apply) {
        if (w.sr) hipLaunchKernelGGL((k_apply<DT, MODE, true, 3>), grid, block, 0, s, w);
        else hipLaunchKernelGGL((k_apply<DT, MODE, false, 3>), grid, block, 0, s, w);
    } else {
        if (w.sr) hipLaunchKernelGGL((k_apply<DT, MODE, true, 0>), grid, block, 0, s, w);
        else hipLaunchKernelGGL((k_apply<DT, MODE, false, 0>), grid, block, 0, s, w);
    }
}

template <int DT>
void StepKernels<DT>::apply(const TensorWork& w, hipStream_t s) {
    if (w.mode == 0 && w.fast_apply == 2)
        hipLaunchKernelGGL(k_apply_tv<DT>, dim3((unsigned)w.apply_wgs), dim3(kThreads), 0, s, w);
    else if (w.mode == 0) launch_apply<DT, 0>(w, s);
    else launch_apply<DT, 1>(w, s);
}

template <int DT>
void StepKernels<DT>::mt_stats(int key_mode, int fast, dim3 grid, hipStream_t s, const TensorWork* ws, SegTable sg) {
    const dim3 block(kThreads);
    if (key_mode != 0) hipLaunchKernelGGL((k_mt_stats_tv<DT, 1>), grid, block, 0, s, ws, sg);
    else if (fast == 2) hipLaunchKernelGGL((k_mt_stats_tv<DT, 0>), grid, block, 0, s, ws, sg);
    else if (fast) hipLaunchKernelGGL((k_mt_factored_stats<DT, true>), grid, block, 0, s, ws, sg);
    else hipLaunchKernelGGL((k_mt_factored_stats<DT, false>), grid, block, 0, s, ws, sg);
}

template <int DT>
void StepKernels<DT>::mt_apply(int key_mode, int fast, int sr, dim3 grid, hipStream_t s, const TensorWork* ws,
                               SegTable sg) {
    const dim3 block(kThreads);
    if (fast == 2) {
        if (key_mode == 0) hipLaunchKernelGGL((k_mt_apply_tv<DT, 0>), grid, block, 0, s, ws, sg);
        else hipLaunchKernelGGL((k_mt_apply_tv<DT, 1>), grid, block, 0, s, ws, sg);
    } else if (fast == 1) {
        // factored and block-path tensors together (the kernels branch per tensor)
        hipLaunchKernelGGL((k_mt_apply<DT, 0, false, 1>), grid, block, 0, s, ws, sg);
    } else if (fast) {
        if (sr) hipLaunchKernelGGL((k_mt_apply<DT, 0, true, 3>), grid, block, 0, s, ws, sg);
        else hipLaunchKernelGGL((k_mt_apply<DT, 0, false, 3>), grid, block, 0, s, ws, sg);
    } else {
        if (sr) hipLaunchKernelGGL((k_mt_apply<DT, 0, true, 0>), grid, block, 0, s, ws, sg);
        else hipLaunchKernelGGL((k_mt_apply<DT, 0, false, 0>), grid, block, 0, s, ws, sg);
    }
}

}  // namespace gx
