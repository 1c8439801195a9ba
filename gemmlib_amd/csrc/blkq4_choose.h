// Which kernel multiplies a given problem, and in which shape: the ONE place where the thresholds live.
// Host-only, plain C++ (no HIP headers): blkq4_api.cpp asks blkq4::choose(), hands the answer to the launchers
// inside blkq4_gemm_args, and the launchers (blkq4_gemm.hip, blkq4_skinny.hip) map it to a kernel instantiation
// without any threshold of their own.
//
// The reference switches kernels at m > 16 and knows two tile shapes (src/blkq4_f16_gemm_sm80.cu:343,
// src/mickey/blk_q4/f16_gemm_sm80.h:63-72); everything below is this library's own cost model, fitted to
// measurements on MI355X.

#pragma once

#include <stddef.h>
#include <stdint.h>

#include <initializer_list>
#include <limits>

#include "blkq4_device.h"

namespace blkq4 {

constexpr int kComputeUnits = 256;
constexpr size_t kMaxLdsBytes = 160 * 1024;
constexpr int kStreamingMaxRows = 1024;

// Where the streaming kernel's waves find their activation fragments.
constexpr int kRowsWholeInLds = 1;    // all rows, all of K, staged once per workgroup
constexpr int kRowsPerSlotInLds = 2;  // 16 * MT rows x 64 k staged per slice, private to the wave

constexpr int kFamilyStreaming = 0;  // weight-streaming kernel (blkq4_staged.hip; rows whole in LDS, by name: blkq4_skinny.hip)
constexpr int kFamilyTile = 1;       // MFMA tile kernel (blkq4_gemm.hip)
constexpr int kFamilyDecode = 2;     // decode kernel (blkq4_decode.hip)

using StreamingShape = blkq4_streaming_plan;  // see blkq4_device.h
using TileShape = blkq4_tile_plan;
using DecodeShape = blkq4_decode_plan;

struct Choice {
  int family;
  StreamingShape s;
  TileShape t;
  DecodeShape d;
};

// A kernel's identity as one number: what choose() picked and what a launcher started can be compared.
inline uint64_t streaming_id(int depth, int nt, int mt, int waves, int am, int split, bool refill) {
  return 1ull << 60 | static_cast<uint64_t>(depth) << 40 | static_cast<uint64_t>(nt) << 32 |
         static_cast<uint64_t>(mt) << 24 | static_cast<uint64_t>(waves) << 16 | static_cast<uint64_t>(am) << 12 |
         static_cast<uint64_t>(split) << 4 | (refill ? 1u : 0u);
}
inline uint64_t tile_id(int rt, int nt, int wm, int wn, int pw, bool split, int kw = 1) {
  return 2ull << 60 | static_cast<uint64_t>(rt) << 40 | static_cast<uint64_t>(nt) << 32 |
         static_cast<uint64_t>(wm) << 24 | static_cast<uint64_t>(wn) << 16 | static_cast<uint64_t>(pw) << 8 |
         static_cast<uint64_t>(kw) << 4 | (split ? 1u : 0u);
}
// the GEMV without MFMA (blkq4_gemv.hip; run only when asked for by name): rows kept (1, 2 or 4) and waves of a
// workgroup
inline int valu_gemv_rows(int m) { return m == 1 ? 1 : m == 2 ? 2 : 4; }
inline int valu_gemv_waves(int k) {
  // sixteen waves when every one of them gets at least two 128-deep slices, else eight, else four
  const int slices = (k / 32 + 3) / 4;
  return slices >= 32 ? 16 : slices >= 16 ? 8 : 4;
}
inline uint64_t valu_gemv_id(int rows, int waves) {
  return 3ull << 60 | static_cast<uint64_t>(rows) << 8 | static_cast<uint64_t>(waves);
}
inline uint64_t decode_id(bool row, int rows, int nt, int waves, int depth) {
  return 4ull << 60 | static_cast<uint64_t>(row ? 1 : 0) << 32 | static_cast<uint64_t>(rows) << 24 | static_cast<uint64_t>(nt) << 16 |
         static_cast<uint64_t>(waves) << 8 | static_cast<uint64_t>(depth);
}
// 64 x 128 tiles run one of two kernels: waves with columns of their own (blkq4_gemm.hip), or waves that are dealt whole k
// tiles (blkq4_kdeal.hip), which take a quarter to a third less per k tile and 1.1 us more in all (their first round is four
// k tiles, and they sum four tiles of accumulators at the end).  So by the k tiles of a workgroup, less two for every k tile
// that the last round of four lacks (its waves wait for the others).  Both were timed on 1160 shapes of every form, M = 17 ... 4096,
// N = 512 ... 50000, K = 1024 ... 20000, up to 4 parts, most with the weights in HBM; columns of their own against dealt k tiles, us:
//   fp16, from 36 on                M = 512, N = K = 4096 25.0 and 22.5, M = 256, N = 4096, K = 2560 13.5 and 12.7; but
//                                   M = 512, N = 3136, K = 2624 (41 k tiles, 44 in rounds) 13.7 and 14.1
//   along N                         from 24 on (M = 150, N = K = 4096 in 2 parts 18.2 and 16.5); without zero-points, where columns
//                                   of their own convert with less, from 32 on in every type
//   blocks of 16                    from 24 on (M = 512, N = K = 4096 26.9 and 25.1, M = 623, N = 2112, K = 3584 18.5 and 15.8); with
//                                   zero-points, whose ring is a k tile shorter, on more than 160 workgroups only where the last
//                                   round lacks no more than one (M = 190, N = 9792, K = 3968, 62 k tiles, 24.0 and 27.0), and along
//                                   N not at all (M = 205, N = 6976, K = 2112 14.5 and 15.3)
//   bf16                            from 20 on, blocks of 16 from 16 on (M = 256, N = 4096, K = 1536 11.5 and 10.8)
// By these lines 49 of 1159 plans that are dealt are slower by more than 2 % and 39 of 587 that are not by more than 5 %; 0.5 % in
// the mean over both.
inline bool tile_dealt_k_tiles(const TileShape& t, int k, bool column_wise, bool bf16, int block_size, bool has_zp) {
  if (!(t.kw == 1 && t.rt == 2 && t.nt == 1 && t.wm == 1 && t.wn == 4 && t.pw == 4)) return false;
  const int parts = t.split_k > 1 ? t.split_k : 1;
  const int workgroups = t.tiles + (parts - 1) * t.split_tiles;
  const int k_tiles = (k / 64 + parts - 1) / parts;
  const int lacking = (4 - k_tiles % 4) % 4, counted = k_tiles - 2 * lacking;
  if (!column_wise && !has_zp) return counted >= 32;
  if (bf16) return counted >= (block_size == 16 ? 16 : 20);
  if (block_size == 16) return counted >= 24 && (!has_zp || workgroups <= 160 || (column_wise && lacking <= 1));
  return counted >= (column_wise ? 36 : 24);
}
// The kernel with dealt k tiles in a plan: one wave covers the whole tile, four of them take the k tiles in turn.  (The same
// outputs per tile and the same workspace.)
inline bool tile_is_dealt(const TileShape& t) { return t.kw == 4 && t.rt == 2 && t.nt == 4 && t.wm == 1 && t.wn == 1; }
inline void deal_k_tiles(TileShape* t) {
  t->nt = 4;
  t->wn = 1;
  t->kw = 4;
}
inline uint64_t choice_id(const Choice& c) {
  if (c.family == kFamilyDecode) return decode_id(c.d.row != 0, c.d.rows, c.d.nt, c.d.waves, c.d.depth);
  return c.family == kFamilyStreaming
             ? streaming_id(c.s.depth, c.s.nt, c.s.mt, c.s.waves, c.s.am, c.s.split, c.s.refill != 0)
             : tile_id(c.t.rt, c.t.nt, c.t.wm, c.t.wn, c.t.pw, c.t.split_k > 1, c.t.kw);
}

// ---------------------------------------------------------------------------------------------------------
// Decode kernel
// ---------------------------------------------------------------------------------------------------------

constexpr int kDecodeMaxRows = 16;
constexpr int kDecodeMaxDepth = 8;
constexpr int kDecodeMaxDepthSixteenWaves = 14;  // up to four rows: K up to 28672

// LDS of a workgroup: the rows of every wave's slices (256 bytes per row and slice), then the waves' partial
// tiles (64 bytes per row and tile), then, with blocks along N, the scales and zero-points of every wave's slices
// (256 + 128 bytes per slice)
inline size_t decode_lds_bytes(bool row, int rows, int nt, int waves, int depth) {
  return static_cast<size_t>(waves) * depth * 256 * rows + static_cast<size_t>(waves) * nt * rows * 64 +
         (row ? static_cast<size_t>(waves) * depth * 384 : 0);
}

// Workgroups: one per group of nt column tiles, rounded up to whole sets of 64 groups (the kernel hands eight
// neighbouring groups to each of the 8 XCDs in turn)
inline uint32_t decode_grid(int n, int nt) {
  const int groups = (n / 16 + nt - 1) / nt;
  return static_cast<uint32_t>((groups + 63) / 64 * 64);
}

// Up to four rows on wide layers with long K: the streaming kernel's workgroups of four to seven tiles, all resident at
// once, beat the decode kernel's rounds of single tiles
//   - two to four rows, K >= 8192, 1376 to 3584 column tiles (same process, decode against streaming: M = 4, K = 8192:
//     N = 28672 27.6 -> 26.7 us, N = 57344 58.2 -> 52.2, blocks of 16 with zero-points, N = 24576 31.0 -> 25.9; the worst
//     case found, M = 3, N = 22016 without zero-points, 19.7 -> 20.5; one row: 23.1 against 24.3, stays);
//   - one to four rows, K > 8192 (where the decode kernel needs sixteen waves), 832 to 1792 column tiles (M = 1:
//     K = 16384, N = 28672 51.1 -> 45.5 us, N = 13312 29.7 -> 25.1; K = N = 28672 87.0 -> 75.8; K = 8256, N = 13312 18.4 ->
//     14.9; K = 11008, N = 28672 with zero-points 42.6 -> 37.7, N = 14336 without 19.0 -> 20.6, the one loss found; on
//     wider layers the decode kernel was ahead again: K = 11008, N = 36864 41.4 against 44.0).
// At K = 4096 and on wider layers the decode kernel won.  (Both against the streaming kernel of that time; what today's promises is
// weighed in decode_bar_us().)
// (The first case later, against the decode kernel's eight waves with eight slices each and one tile per workgroup:
// with blocks of 32 or 64 two and three rows are 2 - 7 % faster in the decode kernel up to 1792 tiles -- M = 2, K = 8192,
// N = 22016 21.3 against 23.0 us, N = 28672 26.0 against 27.7 -- four rows level, N = 57344 level to 8 % behind; with blocks
// of 16 the streaming kernel is 10 - 15 % ahead throughout, N = 24576, M = 4 28.9 against 33.1.)
inline bool streaming_takes_few_rows(int m, int n, int k, int block_size = 64) {
  const int tiles = n / 16;
  if (m > 4) return false;
  if (k > 8192 && tiles >= 832 && tiles <= 1792) return true;
  if (m >= 2 && k >= 8192 && tiles >= 1376 && tiles <= 3584) return block_size < 32 || m == 4 || tiles > 1792;
  return false;
}

// The decode kernel's shape for m rows, or false when it has none or the streaming kernel is expected to be
// faster: blocks along K, at most kDecodeMaxRows rows, K in whole 128-deep slices, few enough of them for the waves
// to request them all at once and for the rows to fit in LDS, and packed weights that 32-bit offsets reach.
//
// Waves.  Eight by default (measured on M = 1, rotating weights, against 4 and 16 waves: K = 2048, N = 2048: 2.62
// against 2.74 and 2.68 us; K = 4096, N = 11008: 6.54 against 6.64 and 7.06; N = 128256: 49.1 against 50.2 and 58.3;
// K = 8192, N = 4096: 5.41 against 16 waves' 5.40), four for short K, sixteen when eight would have to request more
// than eight slices each (up to four rows only).  (Four waves with eight slices each for one workgroup per compute
// unit, K = N = 4096, were the rule once: without zero-points the two are level, 3.71 against 3.70 us; with zero-points
// eight waves take 3.70 against 3.86, in bf16 3.91 against 4.07.)
//
// Column tiles per workgroup.  The busiest compute unit works through ceil(workgroups / 256) workgroups of nt
// tiles each, and every workgroup costs a fraction of a tile's work on top: staging the rows, the instructions
// before the first request, the sum across the waves.  That fraction, fitted to sweeps over N = 4096 .. 28672 at
// K = 4096 and 8192: 0.1 for one row, 0.5 for more.  Two tiles with more than six slices per wave take a tenth
// longer than that (registers: fewer workgroups fit a compute unit), with five or six a twenty-fifth (M = 2 ... 4, K = 5120,
// N = 27648: two tiles 15.5 - 16.1 us, one 16.6 - 17.6), and with eight two fifths longer when they need more than one
// round (K = 8192, M = 2: N = 14336 17.8 us against 15.2 with one tile, N = 28672 34.5 against 26.0; with seven slices,
// K = 7168, N = 32768, M = 3, two tiles take 24.2 us and one 27.6).
//
// Eight and sixteen rows keep 64 to 128 KiB of rows per workgroup, so one or two workgroups fit a compute unit and a
// second round of them starts from nothing; once there are more rounds than that the streaming kernel, whose
// workgroups keep their rows and walk over the column tiles, is faster (M = 16, K = 4096, N = 28672: 17.2 against
// 20.9 us; M = 8, K = 8192, N = 14336: 15.5 against 18.4; but M = 16, K = 4096, N = 11008: 9.2 against 7.9).  Sixteen rows
// take up to four tiles per workgroup (all of LDS at K = 4096), which keeps layers of 12304 ... 16384 columns in one round:
// M = 9 ... 16, K = 4096, N = 14336 9.1 - 9.9 us against the streaming kernel's 10.4 - 10.9, N = 16384 10.1 against 11.1 (at
// N = 11008 three tiles stay ahead, 8.7 against 9.4); with eight rows a fourth tile gains nothing (N = 14336 8.6 against
// 8.7 with two, N = 16384 9.6 against 9.0).
inline bool decode_shape(bool column_wise, int m, int n, int k, DecodeShape* d, int block_size = 64) {
  if (m < 1 || m > kDecodeMaxRows || (k % 128) != 0 || (n % 16) != 0 ||
      static_cast<uint64_t>(k) * static_cast<uint64_t>(n) > (uint64_t{1} << 32)) {
    return false;
  }
  if (!column_wise) {
    // Blocks along N: up to four rows, one column tile per workgroup, eight waves with up to eight slices each
    // (four waves for short K and, with one row, for one workgroup per compute unit at most with eight slices each); the scales
    // and zero-points of a wave's slices, one of each per k, come through LDS.  (M = 1, K = N = 4096: 4.3 against
    // the streaming kernel's 5.3 us.)
    const int slices = k / 128;
    const int tiles = n / 16;
    if (m > 4 || slices > 8 * kDecodeMaxDepth) return false;
    // (two to four rows: eight waves there too, M = 4, K = N = 4096 4.67 against 5.02 us; one row: level, 4.57 and 4.62)
    const int waves = (slices <= 8 || (m == 1 && slices > 28 && slices <= 32 && tiles <= kComputeUnits)) ? 4 : 8;
    d->row = 1;
    d->rows = m == 1 ? 1 : 4;
    d->nt = 1;
    d->waves = waves;
    d->depth = (slices + waves - 1) / waves;
    d->grid = decode_grid(n, 1);
    d->lds_bytes = static_cast<uint32_t>(decode_lds_bytes(true, d->rows, 1, waves, d->depth));
    return true;
  }
  const int slices = k / 128;
  const int tiles = n / 16;
  if (streaming_takes_few_rows(m, n, k, block_size)) return false;
  const int rows = m == 1 ? 1 : m <= 4 ? 4 : m <= 8 ? 8 : 16;
  int waves = 8;
  if (rows <= 4) {
    if (slices <= 8) waves = 4;
    if (slices > 8 * kDecodeMaxDepth) waves = 16;
    if (slices > 16 * kDecodeMaxDepthSixteenWaves) return false;
    // K = N = 8192 (512 tiles, 64 slices): sixteen waves with four slices each, two such workgroups per compute unit
    // and all 512 resident at once, against two rounds of eight waves with eight or one round of two tiles
    // (M = 1 8.53 against 8.84 us, M = 2 8.88 against 9.99, M = 4 9.38 against 9.78; with 320 ... 448 tiles, N = 5120 ... 7168,
    // the eight waves stay 0 - 8 % ahead, and so they do with blocks of 16, whose scales are four times as many:
    // M = 3 11.2 us with two tiles against 12.4)
    if (waves == 8 && block_size >= 32 && slices > 56 && slices <= 64 && tiles > 448 && tiles <= 2 * kComputeUnits) waves = 16;
  }
  const int depth = (slices + waves - 1) / waves;
  if (depth > ((rows == 16) ? 4 : (rows <= 4 && waves == 16) ? kDecodeMaxDepthSixteenWaves : kDecodeMaxDepth)) return false;
  const int max_nt = rows == 16 ? 4 : rows == 8 ? 3 : (waves == 8 ? 2 : 1);  // the instantiations that exist
  const float per_workgroup = rows == 1 ? 0.1f : 0.5f;
  int nt = 1;
  float best = 0.f;
  for (int t = 1; t <= max_nt; ++t) {
    if (decode_lds_bytes(false, rows, t, waves, depth) > kMaxLdsBytes) break;
    const int wgs = (tiles + t - 1) / t;
    float cost = static_cast<float>((wgs + kComputeUnits - 1) / kComputeUnits) * (static_cast<float>(t) + per_workgroup);
    if (rows <= 4 && t == 2 && depth > 4) cost *= depth <= 6 ? 1.04f : (depth < 8 || wgs <= kComputeUnits) ? 1.1f : 1.4f;
    if (t == 1 || cost < best) {
      best = cost;
      nt = t;
    }
  }
  d->row = 0;
  d->rows = rows;
  d->nt = nt;
  d->waves = waves;
  d->depth = depth;
  d->grid = decode_grid(n, nt);
  d->lds_bytes = static_cast<uint32_t>(decode_lds_bytes(false, rows, nt, waves, depth));
  if (d->lds_bytes > kMaxLdsBytes) return false;
  if (rows >= 8) {
    const int per_unit = static_cast<size_t>(d->lds_bytes) * 2 <= kMaxLdsBytes ? 2 : 1;  // workgroups a compute unit holds
    const int rounds = ((tiles + nt - 1) / nt + kComputeUnits * per_unit - 1) / (kComputeUnits * per_unit);
    // (eight rows: two rounds of one workgroup per unit still win while a wave requests five slices: M = 6 ... 8, K = 5120,
    // N = 13824 and 15360 11.4 - 12.1 us against 12.7 - 13.5, the streaming kernel's rings asking for a fifth more
    // slices than K = 5120 has; with six, K = 6144, N = 14336 and 16384, 13.8 - 14.7 against 13.0 - 14.1)
    if (rounds > per_unit && !(rounds == 2 && rows == 8 && depth == 5)) return false;
  }
  return true;
}

// ---------------------------------------------------------------------------------------------------------
// Streaming kernel
// ---------------------------------------------------------------------------------------------------------

// Neighbouring column groups that the streaming kernel gives to one XCD one after the other: four while a column
// group is narrower than a 128-byte line of scales (16 columns a tile), so that the line is fetched into one L2; one
// from four tiles per group on, which deals the column groups to the eight XCDs evenly also when there are few of them
// (80 groups of four tiles, three row groups: in fours XCDs 0 - 3 get 36 workgroups for their 32 compute units and the
// others 24, and the launch takes two rounds, 28.9 us at M = 96, K = N = 5120; singly every XCD gets 30).
constexpr int streaming_neighbours(int nt, int waves, int split) { return (split == waves && nt >= 4) ? 1 : 4; }
// Workgroups on the busiest XCD (the first one, which gets most of what is left over), one column group each; and
// those per compute unit of it, rounded up: the rounds a launch of resident workgroups takes.
inline int streaming_busiest_xcd(int row_groups, int col_groups, int neighbours) {
  const unsigned groups = static_cast<unsigned>(col_groups);  // (neighbours: 1 or 4)
  const int deals = static_cast<int>(neighbours == 1 ? groups / 8 : groups / 32);
  const int rest = static_cast<int>(neighbours == 1 ? groups % 8 : groups % 32);
  return (neighbours * deals + (rest < neighbours ? rest : neighbours)) * row_groups;
}
inline int streaming_rounds(int row_groups, int col_groups, int neighbours) {
  return (streaming_busiest_xcd(row_groups, col_groups, neighbours) + kComputeUnits / 8 - 1) / (kComputeUnits / 8);
}

// Rows staged per slice (blkq4_staged.hip): rows of a row group, dealt evenly ...
inline int staged_rows_per_group(int m, int row_groups) { return (m + row_groups - 1) / row_groups; }
// ... and the rounds of 64-deep slices that only the older half of eight waves takes, which a SIMD serves first (us with 0,
// 2 and 4 of them, K = N = 4096: M = 64 6.6, 6.5, 6.5, M = 128 8.9, 8.6, 8.4; M = 16, N = 28672, K = 8192 26.1, 25.9, 26.0;
// M = 12, N = 4096, K = 11008 11.3, 11.1, 11.3).
constexpr int staged_extra_rounds(int waves, int k) { return (waves == 8 && k >= 2048) ? 2 : 0; }

// Slices of a workgroup's busiest wave (without those rounds, which a shorter K does not have).
inline int staged_most_slices(int waves, int k) {
  const int slices = k / 64, rounds = slices / waves, rest = slices - rounds * waves;
  return rounds + (rest + waves / 2 - 1) / (waves / 2);
}

// Four column tiles, up to 16 rows: four waves or eight.  Eight while there is one workgroup per compute unit at most, which a unit
// with four waves only makes wait longer for its memory; four beyond, when a unit holds several small workgroups instead of a
// second round of large ones, and where eight waves would not have fewer slices each.  The faster of the two on 336 of the
// 338 shapes it decides out of 1563 (both blockings; none of the others by more than 2 %): M = 8, N = 18432, K = 4096 along N 12.9 with
// four and 16.2 us with eight waves, M = 6, N = 14336, K = 1216 along K 5.4 and 4.6, M = 4, N = 13824, K = 256 along N 2.89 and 3.03.
inline bool staged_four_waves(int n, int k) {
  return (n / 16 + 3) / 4 > kComputeUnits || staged_most_slices(4, k) <= staged_most_slices(8, k);
}

// LDS of a workgroup: per wave `depth` slots of 16 * mt rows x 128 bytes, 32 columns of packed weights at a time, scales and
// zero-points 256 bytes at a time; the waves' partial tiles take their place at the end.
constexpr int staged_lds_bytes(bool row, int block_size, bool has_zp, int nt, int mt, int waves, int depth) {
  const int columns = 16 * nt, groups = columns > block_size ? columns / block_size : 1;
  const int scale_words = row ? groups * 32 : 64 / block_size * columns / 2;
  const int zp_words = !has_zp ? 0 : row ? groups * 16 : 64 / block_size * columns / 4;
  const int slot = 16 * mt * 128 + (columns + 31) / 32 * 1024 + (scale_words + 63) / 64 * 256 + (zp_words + 63) / 64 * 256;
  const int partial = 16 * mt * (columns + 4) * 4;
  return waves * (depth * slot > partial ? depth * slot : partial);
}

// Blocks along N: one, two, four or eight column tiles (whole column groups, or a part of one).
// Five tiles of 48 rows fit in LDS unless a slice has four block rows of scales and of zero-points (blocks of 16 with them).
constexpr bool staged_shape_exists(bool row, int block_size, bool has_zp, int nt, int mt, int waves, int depth) {
  if (row && nt != 1 && nt != 2 && nt != 4 && nt != 8) return false;
  return static_cast<size_t>(staged_lds_bytes(row, block_size, has_zp, nt, mt, waves, depth)) <= kMaxLdsBytes;
}

// Launch geometry of one instantiation.  Many more workgroups than the chip holds at once: a workgroup then
// walks over several column groups (cg, cg + cg_stride, ...) and requests the first slices of the next one
// while it finishes the current one, so only the first column group of a workgroup waits for its weights with
// nothing else to do.  The partial tiles then get LDS of their own: the rows stay where they are for the next
// column group.  (not the sixteen-wave kernel for blocks along N: its walking variant does not fit in 128
// registers)
// (Rows staged per slice: one column group per workgroup, however many there are, and a kernel that knows its LDS itself.)
inline void streaming_geometry(StreamingShape* s, bool row, int n, int k) {
  if (s->am == kRowsPerSlotInLds) {
    const int groups = (n / 16 + s->nt - 1) / s->nt, deal = 8 * streaming_neighbours(s->nt, s->waves, s->split);
    s->cg_stride = (groups + deal - 1) / deal * deal;
    s->grid = static_cast<uint32_t>(s->cg_stride) * static_cast<uint32_t>(s->row_groups);
    return;
  }
  constexpr int kPersistentFactor = 2;  // column groups per workgroup from which on workgroups walk
  // partial tiles of the sum across waves: [wave][tile][row tile][row][16 columns] floats, rows that exist only
  const size_t rows = s->mt == 1 ? (size_t{1} << s->rows_log2) : 16;
  const size_t red_bytes = (s->split == 1) ? 0 : static_cast<size_t>(s->waves) * s->nt * s->mt * rows * 64;
  // the rows are copied 1 KiB at a time
  const size_t a_bytes = (((static_cast<size_t>(k) * 2) << s->rows_log2) + 1023) & ~size_t{1023};
  const int group_tiles = s->nt * (s->waves / s->split);
  const int col_groups = (n / 16 + group_tiles - 1) / group_tiles;
  const int per_xcd_round = 8 * streaming_neighbours(s->nt, s->waves, s->split);
  int cg_stride = (col_groups + per_xcd_round - 1) / per_xcd_round * per_xcd_round;  // one column group per workgroup
  // The partial tiles lie behind the rows when both fit (one barrier less: nobody has to wait until every wave
  // is done with the rows), else they reuse the rows' space.
  const bool separate = a_bytes + red_bytes <= kMaxLdsBytes;
  size_t lds_bytes = separate ? a_bytes + red_bytes : (a_bytes > red_bytes ? a_bytes : red_bytes);
  size_t red_offset = separate ? a_bytes : 0;
  const bool may_walk = !(row && s->waves == 16);
  if (may_walk && separate) {
    const int by_lds = static_cast<int>(kMaxLdsBytes / (a_bytes + red_bytes));
    const int by_waves = 32 / s->waves;
    const int resident = kComputeUnits * (by_lds < by_waves ? by_lds : by_waves);
    int stride = (resident / s->row_groups) / 32 * 32;
    if (stride < 32) stride = 32;
    if (cg_stride >= kPersistentFactor * stride) cg_stride = stride;
  }
  s->cg_stride = cg_stride;
  s->grid = static_cast<uint32_t>(cg_stride) * static_cast<uint32_t>(s->row_groups);
  s->lds_bytes = static_cast<uint32_t>(lds_bytes);
  s->red_offset = static_cast<uint32_t>(red_offset);
  // workgroups walk over several column groups, or waves stream all of K by themselves
  s->refill = (cg_stride < col_groups || s->split == 1) ? 1 : 0;
}

// What the cost of a workgroup depends on besides its shape.
enum CostForm { kCostPlain = 0, kCostBf16 = 1, kCostBlocksAlongN = 2, kCostBlocksOf16 = 4, kCostNoZeroPoints = 8 };  // bits
inline int cost_form(bool column_wise, bool bf16, int block_size, bool has_zp) {
  return (bf16 ? kCostBf16 : 0) | (!column_wise ? kCostBlocksAlongN : 0) | (block_size == 16 ? kCostBlocksOf16 : 0) |
         (has_zp ? 0 : kCostNoZeroPoints);
}

// Rows staged per slice (blkq4_staged.hip), one family of shapes per row tiles of a workgroup: up to 16 rows, row groups of 32
// and row groups of 48.  A launch takes, in us, a fixed part, the packed weights' way from HBM, and rounds of workgroups as
// the busiest XCD has them, each a fixed part and a part per 1024 k that grows with the rows and, per column tile, with the form.
// Least squares over plans up to 1.4 times their shape's fastest, four fifths of them with the weights in HBM, every form: up
// to 16 rows 20385 plans of 6100 shapes (N = 1024 ... 28672, along N 131072, K = 64 ... 16384; four tiles in the waves that
// staged_four_waves() gives them; a plan counts less the further it is behind its shape's fastest, half at a fifth; 6.5 % rms along
// K, 6.6 % along N), more rows 32072 plans of 9030 shapes (M = 17 ... 700; 5.2 - 5.9 %).  The shape with the smallest estimate takes
// 1.002 times the fastest one's time in the mean (at most 1.23) with more than 16 rows, 1.006 (1.16) along K and 1.005 (1.20) along N
// with fewer.
struct StagedShapeCost {
  int depth, nt, waves;
  double round, per_k;
};
struct StagedFamily {
  double base, from_hbm, from_hbm_blocks_of_16, rows, bf16, blocks_of_16, no_zero_points, fill;
  int count;
  StagedShapeCost shapes[9];
};
inline const StagedFamily& staged_family(bool row, int mt) {
  static constexpr StagedFamily kAlongK[3] = {
      {2.401, 2.500, 0.261, 0.555, 0.049, 0.042, -0.036, 0.046, 9,
       {{4, 1, 8, 0.314, 0.406}, {2, 1, 16, 0.544, 0.292}, {2, 2, 16, 0.620, 0.438}, {2, 3, 16, 0.823, 0.665}, {2, 4, 8, 0.717, 0.763},
        {2, 5, 8, 0.864, 1.074}, {2, 6, 8, 0.958, 1.304}, {2, 7, 8, 1.137, 1.562}, {2, 4, 4, 0.404, 0.801}}},
      {1.362, 3.678, 0.567, 0.418, 0.045, 0.036, -0.022, 0.031, 5,
       {{2, 1, 8, 1.302, 0.555}, {2, 2, 8, 1.419, 0.636}, {2, 4, 8, 1.949, 0.942}, {2, 6, 8, 2.441, 1.484}, {2, 8, 8, 2.739, 1.927}}},
      {1.210, 3.573, 0.721, 0.411, 0.039, 0.031, -0.032, 0.035, 5,
       {{2, 1, 8, 1.511, 0.608}, {2, 2, 8, 1.895, 0.779}, {2, 3, 8, 2.346, 0.973}, {2, 4, 8, 2.652, 1.145}, {2, 5, 8, 3.057, 1.477}}}};
  static constexpr StagedFamily kAlongN[3] = {
      {2.293, 2.893, 1.664, 0.398, 0.138, 0.016, -0.060, 0.004, 5,
       {{4, 1, 8, 0.433, 0.497}, {2, 1, 16, 0.686, 0.375}, {2, 2, 16, 0.804, 0.550}, {2, 4, 8, 0.820, 0.940}, {2, 4, 4, 0.451, 0.979}}},
      {1.476, 3.494, -0.106, 0.373, 0.128, 0.072, -0.044, 0.028, 4,
       {{2, 1, 8, 1.293, 0.547}, {2, 2, 8, 1.566, 0.643}, {2, 4, 8, 1.985, 1.077}, {2, 8, 8, 2.768, 2.310}}},
      {1.404, 3.637, -0.203, 0.344, 0.125, 0.073, -0.043, 0.047, 3,
       {{2, 1, 8, 1.440, 0.626}, {2, 2, 8, 1.872, 0.752}, {2, 4, 8, 2.479, 1.212}}}};
  return row ? kAlongN[mt - 1] : kAlongK[mt - 1];
}
inline double staged_estimate_us(const StagedFamily& f, const StagedShapeCost& c, int m, int n, int k, int row_groups, int form) {
  const int busiest = streaming_busiest_xcd(row_groups, (n / 16 + c.nt - 1) / c.nt, streaming_neighbours(c.nt, c.waves, c.waves));
  const int per_unit = kComputeUnits / 8;
  const double rounds = (busiest + per_unit - 1) / per_unit, fill = busiest / (rounds * per_unit);
  const double kk = static_cast<double>(k) / 1024.0, from_hbm = static_cast<double>(n) * kk / 100000.0;
  // up to 16 rows: what is copied of them, eight or sixteen
  const int rows = m <= 8 ? 8 : m <= 16 ? 16 : staged_rows_per_group(m, row_groups);
  const double per_tile = ((form & kCostBf16) ? f.bf16 : 0.0) + ((form & kCostBlocksOf16) ? f.blocks_of_16 : 0.0) +
                          ((form & kCostNoZeroPoints) ? f.no_zero_points : 0.0) + f.fill * fill;
  return f.base + from_hbm * (f.from_hbm + ((form & kCostBlocksOf16) ? f.from_hbm_blocks_of_16 : 0.0)) +
         rounds * (c.round + kk * (c.per_k + f.rows * rows / 32.0 + c.nt * per_tile));
}

// The streaming kernel's shape for any number of rows, and what it is expected to take: the smallest estimate of all shapes with rows
// staged per slice.  Rows whole in LDS (blkq4_skinny.hip), which used to run up to 16 rows and some row groups with blocks
// along N, start by name only: timed in turn on 715 drawn shapes of up to 16 rows that took them (70 of them with 28736 to 131072
// columns) the shape chosen here is slower by more than 2 % on none; along K it is 1.25 times as fast in the mean (M = 16, N = 4224, K = 2624
// 9.7 -> 5.7 us, M = 2, N = 13376, K = 5440 15.0 -> 10.1), along N 1.63 times (M = 11, N = 1536, K = 512 8.1 -> 3.2); in row groups,
// 113 shapes, it is faster on all (1.09 - 2.25 times, M = 57, N = 6080, K = 1856 10.7 -> 9.3).
//
// Row groups of 48 only where they are fewer than groups of 32: as many of them are never faster along N (1422 shapes), and along K
// on 29 of 1854 by 2 to 4 %, while their estimate, a twentieth off either way, chose them more often (253 drawn shapes: 113 are faster
// in groups of 32 by more than 2 %, 23 slower; M = 23, N = 20480, K = 8128 27.4 -> 24.2 us).  A single group (33 to 48 rows) along K
// that leaves an eighth of the compute units without a workgroup has to promise 4 % less than two groups of 32, whose workgroups
// hold twice the columns (269 drawn shapes: 207 faster, 8 slower, 1.05 in the mean; M = 35, N = 6016, K = 5120 11.2 -> 10.3); with every
// unit busy the estimates are level (M = 34, N = 8192, K = 4096 9.3 us, two groups of 32 11.2).
inline StreamingShape streaming_shape(bool row, int m, int n, int k, int block_size, int form, double* us) {
  StreamingShape s{};
  double best = 0.0;
  for (int mt = m <= 16 ? 1 : 2; mt <= (m <= 16 ? 1 : 3); ++mt) {
    const StagedFamily& f = staged_family(row, mt);
    const int row_groups = (m + 16 * mt - 1) / (16 * mt);
    for (int i = 0; i < f.count; ++i) {
      const StagedShapeCost& c = f.shapes[i];
      if (!staged_shape_exists(row, block_size, (form & kCostNoZeroPoints) == 0, c.nt, mt, c.waves, c.depth)) continue;
      if (mt == 1 && c.nt == 4 && (c.waves == 4) != staged_four_waves(n, k)) continue;
      if (mt == 3 && row_groups == (m + 31) / 32) continue;
      const double t = staged_estimate_us(f, c, m, n, k, row_groups, form);
      const bool one_group_bar = mt == 3 && row_groups == 1 && !row &&
                                 streaming_busiest_xcd(1, (n / 16 + c.nt - 1) / c.nt, streaming_neighbours(c.nt, c.waves, c.waves)) < 28;
      const double price = one_group_bar ? 1.04 * t : t;
      if (s.nt != 0 && price >= best) continue;
      best = price;
      *us = t;
      s.depth = c.depth; s.nt = c.nt; s.mt = mt; s.waves = c.waves; s.am = kRowsPerSlotInLds; s.split = c.waves;
      s.row_groups = row_groups;
    }
  }
  if (m <= 16 && !row && n > 28672) {
    // Beyond what the estimate was fitted on: the launch takes as long as the busiest compute unit's column tiles, a
    // twelfth more when that unit holds four waves only, a fifteenth with eight.  Four tiles and four waves (M = 12, N = 124800,
    // K = 2048 29.2 us, eight waves 44.2) unless five to seven tiles, all workgroups resident from the start, promise 3 % less.
    // (109 shapes, N = 28736 ... 131072: 1.02 times the fastest in the mean with four tiles alone.)
    auto busiest = [&](int nt, int waves, bool all_resident) -> double {
      const long resident = static_cast<long>(kMaxLdsBytes) /
                            staged_lds_bytes(false, block_size, (form & kCostNoZeroPoints) == 0, nt, 1, waves, 2);
      const long per_unit = ((n / 16 + nt - 1) / nt + kComputeUnits - 1) / kComputeUnits;
      if (all_resident && per_unit > resident) return -1.0;
      const long on_unit = per_unit * waves;
      return static_cast<double>(per_unit * nt) * (on_unit <= 4 ? 1.12 : on_unit <= 8 ? 1.07 : 1.0);
    };
    const double usual = busiest(4, 4, false);
    double least = 0.97 * usual;
    s.depth = 2; s.nt = 4; s.waves = 4; s.split = 4;
    for (const int w : {8, 4}) {
      for (const int t : {5, 6, 7}) {
        const double cost = busiest(t, w, true);
        if (cost > 0.0 && cost < least) {
          least = cost;
          s.nt = t;
          s.waves = w;
          s.split = w;
        }
      }
    }
  }
  // A single row group of 48 along K in two rounds of workgroups takes 8 % longer than its estimate where that lies near the one
  // of 64 x 128 tiles, 160 to 190 of which cover those layers (59 drawn shapes change for it: 40 are faster by more than 2 %, 9 slower,
  // 1.03 in the mean; M = 46, N = 20992, K = 7744, bf16 38.2 -> 35.1 us, M = 47, N = 22976, K = 3456 20.4 -> 18.7).  In more rounds
  // either may be ahead (24 shapes: 9 and 7; M = 33, N = 45120, K = 3008, bf16 is 7 % faster than tiles).
  if (s.mt == 3 && !row && s.row_groups == 1 &&
      streaming_rounds(1, (n / 16 + s.nt - 1) / s.nt, streaming_neighbours(s.nt, s.waves, s.split)) == 2) {
    *us *= 1.08;
  }
  streaming_geometry(&s, row, n, k);
  return s;
}

// ---------------------------------------------------------------------------------------------------------
// Tile kernel
// ---------------------------------------------------------------------------------------------------------

inline long ceil_div(int a, int b) { return (static_cast<uint32_t>(a) + static_cast<uint32_t>(b) - 1u) / static_cast<uint32_t>(b); }

// The tile shapes, (rt, nt, wm, wn, pw): 64 x 128, 128 x 128 and 128 x 256 tiles of four computing waves
// (64 x 32, 128 x 32, 128 x 64 each) plus four producer waves that only issue copies, and 256 x 256 tiles of
// four waves of 256 x 64 (every register of a SIMD belongs to the one wave, which leaves no room for producer
// waves).  Larger tiles convert fewer weights per MFMA; smaller ones fill the chip with smaller problems.
// Between the last two, 160 x 256 and 192 x 256 tiles of the same kind as 256 x 256, never split: for row counts, and tile counts, that
// 128-row tiles cover in a round and a bit and 256-row tiles with a third of the rows, or of the chip, idle (M = 777,
// N = 11008, K = 4096: 215 tiles of 160 rows 66.4 us, 172 of 256 rows, which it replaced, 79.1, 301 of 128 rows with the
// last 45 in parts 87.0; bf16 67.0, 79.4, 87.6; M = 320, N = 28672, K = 8192: 224 tiles 129.2, 336 of 128 rows with the last
// 80 in 3 parts, which it replaced, 158.7).
constexpr int kTileShapes[6][5] = {{2, 1, 1, 4, 4}, {4, 1, 1, 4, 4}, {4, 2, 1, 4, 4}, {5, 2, 1, 4, 0}, {6, 2, 1, 4, 0}, {8, 2, 1, 4, 0}};
constexpr bool tile_has_split_form(int rt) { return rt != 5 && rt != 6; }

// Arrival counters first (one per split tile), then the fp32 partial tiles of the split tiles.
constexpr size_t kCounterBytes = 16 * 1024;  // room for 4096 split tiles
constexpr int kMinKTilesPerPart = 4;         // a part of a split tile is at least this many 64-deep k tiles
constexpr int kMaxSplit = 4;                 // the workgroup that arrives last reads all the parts by itself

inline size_t tile_workspace_bytes(const TileShape& t) {
  if (t.split_k <= 1) return 0;
  const size_t tile_elems = static_cast<size_t>(32 * t.rt * t.wm) * (32 * t.nt * t.wn);
  return kCounterBytes + static_cast<size_t>(t.split_tiles) * t.split_k * tile_elems * 4;
}

// Tile order inside a whole round of 256 unsplit tiles.  Workgroup w of a round runs on XCD w % 8 (round-robin
// dispatch), each XCD with an L2 of its own.  In the column-major tile order an XCD gets every eighth tile: with 8 or
// more tile rows that is m_tiles / 8 rows x ALL the round's columns.  xcd_rows = 1, 2, 4 or 8 cuts the round's
// m_tiles x (256 / m_tiles) rectangle into xcd_rows row bands x (8 / xcd_rows) column bands instead, one block per
// XCD.  Needs m_tiles to be a power of two between xcd_rows and 32 * xcd_rows.  The kernel's argument: log2 of
// xcd_rows, of the block's rows and of the round's columns, 4 bits each.
inline int log2_exact(int v) {
  int l = 0;
  while ((1 << l) < v) ++l;
  return (1 << l) == v ? l : -1;
}
inline bool xcd_tile_map(int m_tiles, int xcd_rows, int* map) {
  const int ml = log2_exact(m_tiles), xl = log2_exact(xcd_rows);
  if (ml < 0 || xl < 0 || ml > 8 || xl > 3 || xl > ml || ml - xl > 5) return false;
  *map = xl | (ml - xl) << 4 | (8 - ml) << 8 | 1 << 12;
  return true;
}

// Which cut to use: per k, the 32 tiles of an XCD make its L2 fetch (block rows) x 2 BM + (block columns) x BN / 2
// bytes.  Blocks are used when they fetch at most 0.8 of what every-eighth-tile fetches (the large tiles' time does
// not depend on it, the traffic through the fabric does: C4 fetches 66 instead of 83 MB).  Measured with forced plans
// (same process, us; 0 = every eighth tile, else xcd_rows): M = 512, K = N = 4096 in 64 x 128 tiles (8 tile rows: a whole
// row of 32 tiles per XCD, 71 MB through the fabric; 2 row bands make it 33 MB) 23.4 | 1: 22.6, 2: 21.6, 4: 22.3, 8: 23.0;
// nothing else moves by more than 1 %: M = 1024 in 128 x 128 tiles 33.6 | 33.5 - 33.9, C4 58.0 | 58.2 - 59.0,
// M = 512, N = 11008 in 128 x 128 tiles 53.9 | 53.1 - 54.2, M = 1024, K = N = 8192 114.0 | 112.6 - 114.0, C5 1500 - 1527 |
// 1500 - 1516.
inline int xcd_rows_for(const TileShape& t, int m) {
  const int bm = 32 * t.rt * t.wm, bn = 32 * t.nt * t.wn;
  const int m_tiles = static_cast<int>(ceil_div(m, bm));
  const int ml = log2_exact(m_tiles);
  if (ml < 0 || ml > 8 || t.tiles - t.split_tiles < kComputeUnits) return 0;
  auto fetched = [&](int xcd_rows) {
    const int rows = m_tiles / xcd_rows;
    return rows * bm * 4 + (32 / rows) * bn;
  };
  const int as_is = fetched(m_tiles < 8 ? m_tiles : 8);
  int best = 0, best_bytes = as_is;
  for (int xr = 1; xr <= 8 && xr <= m_tiles; xr *= 2) {
    if (m_tiles / xr > 32) continue;
    if (fetched(xr) < best_bytes) {
      best = xr;
      best_bytes = fetched(xr);
    }
  }
  return best_bytes * 10 <= as_is * 8 ? best : 0;
}

// Microseconds of a workgroup: `fixed` outside its main loop, and per 64-deep k tile `idle` while at most half the compute
// units have one, rising with the load on the memory system and the clock that the chip holds to `full` with all of them (fp16,
// blocks of 32 or 64 along K); a split tile's exchange (two more barriers, the invalidate, the count, and what grows with
// the number of workgroups that exchange; the parts' bytes are counted apart); what 51 MB of packed weights from HBM add.
// The other forms convert with more instructions per weight, which counts where the conversion is what a workgroup waits
// for: factors on `idle` and `full` for bf16, blocks along N and blocks of 16, which multiply; blocks along N without
// zero-points are cheaper again.
// Least squares over 2700 shapes, M = 17 ... 4096, N = 512 ... 115000, K = 256 ... 20000, every form, every plan up to one and a half
// times the shape's fastest, six in seven with the weights in HBM, the others from the cache (those are 4 % faster; the
// constants lie between the two).  rms in the order of the table: 5.8, 4.6, 4.9, 5.2, 4.1, 3.9, 3.7, 3.3, 4.6, 3.9, 4.0 %.
// On 650 of them with M = 17 ... 800 and cold weights the plans taken by these are 0.3 % (blocks along K) and 0.5 %
// (along N) behind the fastest ones in the geometric mean, 11 by more than 5 %; by the constants before, which
// described kernels that had been replaced, 1.7 and 3.4 %, 83 by more than 5 %, up to twice the time (M = 148, N = 3264,
// K = 2368, blocks of 16 along N 29.1 -> 13.8 us; M = 298, N = 1408, K = 3264 13.3 -> 8.3; M = 256, N = K = 8192 54.2 -> 41.4).
struct TileCost {
  double fixed, idle, full, split, split_load, from_hbm;
  double form[3][2];  // bf16, blocks along N, blocks of 16: on idle, on full
  double along_n_without_zp;
};
inline const TileCost& tile_cost(const TileShape& t) {
  static constexpr TileCost kDealt = {4.50, 0.193, 0.258, 0.8, 2.5, 2.0, {{1.36, 1.07}, {1.32, 1.07}, {1.05, 1.13}}, 0.87};
  static constexpr TileCost k64x128 = {3.11, 0.253, 0.302, 1.3, 2.1, 1.4, {{1.38, 1.16}, {1.25, 1.15}, {1.07, 1.14}}, 0.82};
  static constexpr TileCost k128x32 = {3.48, 0.199, 0.206, 0.0, 0.0, 10.8, {{1.02, 0.99}, {1.0, 1.0}, {1.0, 1.02}}, 1.0};
  static constexpr TileCost k128x128 = {2.83, 0.340, 0.472, 1.5, 2.1, 2.0, {{1.25, 1.09}, {1.14, 1.09}, {1.08, 1.07}}, 0.92};
  static constexpr TileCost k128x256 = {4.02, 0.586, 0.847, 0.0, 4.7, 1.0, {{1.16, 1.04}, {1.08, 1.08}, {1.09, 1.06}}, 0.95};
  static constexpr TileCost k160x256 = {5.75, 0.714, 1.043, 0.0, 0.0, 1.2, {{1.09, 1.01}, {1.09, 1.06}, {1.11, 1.08}}, 0.95};
  static constexpr TileCost k192x256 = {6.44, 0.822, 1.211, 0.0, 0.0, 0.3, {{1.06, 1.02}, {1.04, 1.07}, {1.08, 1.06}}, 0.96};
  static constexpr TileCost k256x256 = {7.23, 1.063, 1.504, 5.0, 0.0, 1.7, {{1.02, 1.01}, {1.03, 1.04}, {1.07, 1.05}}, 0.96};
  static constexpr TileCost k32x128 = {3.39, 0.228, 0.228, 0.0, 0.0, 0.3, {{1.27, 1.10}, {1.0, 1.0}, {1.14, 1.14}}, 1.0};
  static constexpr TileCost k32x256 = {3.81, 0.292, 0.292, 0.0, 0.0, 3.7, {{1.25, 1.10}, {1.0, 1.0}, {1.19, 1.10}}, 1.0};
  static constexpr TileCost k64x256 = {4.10, 0.347, 0.357, 0.0, 0.0, 5.1, {{1.35, 1.10}, {1.0, 1.0}, {1.22, 1.20}}, 1.0};
  if (tile_is_dealt(t)) return kDealt;
  if (t.kw > 1) return k128x32;
  switch (t.rt) {
    case 1: return t.wn == 4 ? k32x128 : k32x256;
    case 2: return t.wn == 4 ? k64x128 : k64x256;
    case 4: return t.nt == 1 ? k128x128 : k128x256;
    case 5: return k160x256;
    case 6: return k192x256;
    default: return k256x256;
  }
}
// The same for one form of the problem and its rows: `full` - `idle` spread over the compute units beyond half of them.
struct TileStep {
  double fixed, idle, slope;
  bool dealt;  // whole rounds of four k tiles
  double round_us(int k_tiles, int busy) const {
    constexpr int kHalf = kComputeUnits / 2;
    const int load = busy < kComputeUnits ? busy : kComputeUnits;
    return fixed + (dealt ? (k_tiles + 3) / 4 * 4 : k_tiles) * (idle + (load > kHalf ? (load - kHalf) * slope : 0.0));
  }
};
inline TileStep tile_step(const TileShape& t, int m, int form) {
  const TileCost& c = tile_cost(t);
  double idle = c.idle, full = c.full, both = 1.0;
  for (int bit = 0; (form & 7) >> bit; ++bit) {
    if (form & (1 << bit)) {
      idle *= c.form[bit][0];
      full *= c.form[bit][1];
    }
  }
  if ((form & kCostBlocksAlongN) && (form & kCostNoZeroPoints)) both = c.along_n_without_zp;
  // rows past the last one repeat it, which takes less energy per k tile
  const int tile_rows = 32 * t.rt * t.wm;
  if (t.rt > 1) both *= 1.0 - 0.11 * (1.0 - static_cast<double>(m) / static_cast<double>(ceil_div(m, tile_rows) * tile_rows));
  return {c.fixed, both * idle, full > idle ? both * (full - idle) / (kComputeUnits / 2) : 0.0, tile_is_dealt(t)};
}

// A split tile's partial tile written once and all parts read by the workgroup that arrives last, about 67 GB/s.  (256 x 256:
// the accumulators fill the registers and the workgroup that adds the parts up has one request in flight at a time, 30 us per
// part -- by timestamps 118.6 us for four parts where a 128 x 256 tile's take 7.6; M = 1280, N = 14336, K = 8192 in 256 x 256
// tiles with the last 24 in 4 parts 366 us, unsplit 331, in 128 x 256 tiles with the last 48 in 4 parts 260)
inline double split_exchange_us(const TileShape& t, int parts) {
  return (1 + parts) * (4 * 32 * 32) * (t.rt * t.wm * t.nt * t.wn) / (t.rt == 8 ? 9e3 : 66.7e3);
}

// Estimated time of the tile kernel with shape t (split or not): whole rounds of unsplit tiles, a last round of what is left
// of them, then one round of parts: their share of the k tiles, the exchange and the partial tiles.
inline double tile_estimate_us(const TileShape& t, const TileStep& step, int n, int k) {
  const TileCost& c = tile_cost(t);
  const int kt = k / 64, whole = t.tiles - (t.split_k > 1 ? t.split_tiles : 0);
  double us = c.from_hbm * static_cast<double>(n) * static_cast<double>(k) / 102400000.0;
  if (whole / kComputeUnits) us += (whole / kComputeUnits) * step.round_us(kt, kComputeUnits);
  if (whole % kComputeUnits) us += step.round_us(kt, whole % kComputeUnits);
  if (t.split_k > 1) {
    const int units = t.split_tiles * t.split_k;
    us += ((units + kComputeUnits - 1) / kComputeUnits) *
          (step.round_us((kt + t.split_k - 1) / t.split_k, units) + c.split + c.split_load * units / kComputeUnits +
           split_exchange_us(t, t.split_k));
  }
  return us;
}

// The tile kernel's plan: the shape with the smallest estimate; when its last round of tiles would leave most of the chip
// idle, those last `split_tiles` tiles may each be shared out over split_k workgroups.  Up to 32 rows with blocks along K also
// tiles of one row tile (128 columns with four waves and four producer waves, or 256 columns with eight waves), up to 64 rows
// 64 x 256 tiles.  us: in, what another kernel is expected to take (a plan that cannot be faster is not looked at further); out,
// the plan's estimate, if a plan was faster (else rt is 0).
inline TileShape tile_plan(bool column_wise, int m, int n, int k, size_t workspace_capacity, bool bf16, int block_size, bool has_zp,
                           double* us) {
  const int form = cost_form(column_wise, bf16, block_size, has_zp);
  TileShape best{};
  auto shape = [&](int rt, int nt, int wm, int wn, int pw) {
    TileShape t{};
    t.rt = rt; t.nt = nt; t.wm = wm; t.wn = wn; t.pw = pw;
    t.kw = 1;
    t.split_k = 1;
    t.tiles = static_cast<int>(ceil_div(m, 32 * rt * wm) * ceil_div(n, 32 * nt * wn));
    return t;
  };
  auto consider = [&](TileShape t, TileStep step) {
    if (tile_dealt_k_tiles(t, k, column_wise, bf16, block_size, has_zp)) {
      deal_k_tiles(&t);
      step = tile_step(t, m, form);
    }
    const double t_us = tile_estimate_us(t, step, n, k);
    if (t_us < *us) {
      best = t;
      *us = t_us;
    }
  };
  const int kt = k / 64;
  for (const auto& sh : kTileShapes) {
    TileShape t = shape(sh[0], sh[1], sh[2], sh[3], sh[4]);
    // (160 and 192 rows also in several rounds, where the estimate, fitted to one, holds too: of 800 shapes of 300 to 4096 rows 97
    // get them there instead of 128 or 256 rows, two of those slower by more than 2 %, all 800 1.003 times their fastest plan in the
    // mean where one round only makes it 1.011.  M = 944, N = 21184, K = 4992 193 -> 165 us, M = 3647, N = 4544, K = 1856, blocks
    // of 16 82 -> 71, bf16, M = 1708, N = 21696, K = 10880 780 -> 648; the other way M = 2048, N = 11008, K = 4096 162 -> 164.)
    const TileStep step = tile_step(t, m, form);
    // (dealt k tiles, which the shape may turn into, take three quarters of a step)
    const auto at_least = [&](int k_tiles) { return step.fixed + 0.75 * step.idle * k_tiles; };
    if (at_least(kt) < *us) consider(t, step);
    const int rem = t.tiles % kComputeUnits;
    if (rem == 0 || !tile_has_split_form(sh[0])) continue;
    for (int split = 2; split <= kMaxSplit; ++split) {
      if (rem * split > kComputeUnits || kt / split < kMinKTilesPerPart) break;
      if (at_least(kt / split) + split_exchange_us(t, split) >= *us) continue;
      // A fourth part that fills the chip pays only with a long K: of 86 problems measured with 64 tiles in 4 parts, three
      // parts are faster for most below K = 8192 (median 6 %), four by 3 - 13 % at K = 11008; and with every compute unit
      // busy the last workgroups' invalidates hit the others' operands (M = 256, K = N = 4096, blocks along N, 128 x 128
      // tiles: 25 - 27 us in 4 parts on one machine, 20.6 on the others, 20.2 in 3 parts on all).
      if (split == 4 && rem * 4 > 224 && kt < 128) continue;
      t.split_k = split;
      t.split_tiles = rem;
      t.workspace_bytes = tile_workspace_bytes(t);
      if (t.workspace_bytes > workspace_capacity || static_cast<size_t>(rem) * sizeof(int) > kCounterBytes) continue;
      consider(t, step);
    }
  }
  if (column_wise) {
    // 128 x 32 tiles of four waves that split the k tile, when one round of them covers the problem
    TileShape t = shape(4, 1, 1, 1, 4);
    t.kw = 4;
    if (t.tiles <= kComputeUnits) consider(t, tile_step(t, m, form));
    const TileShape narrow = shape(1, 1, 1, 4, 4), wide = shape(m <= 32 ? 1 : 2, 1, 1, 8, 0);
    if (m <= 32) consider(narrow, tile_step(narrow, m, form));
    if (m <= 64) consider(wide, tile_step(wide, m, form));
  }
  if (best.rt != 0) best.xcd_rows = xcd_rows_for(best, m);
  return best;
}

// The streaming kernels' offsets into the packed weights (K N / 2 bytes) are 32 bits wide (so are the other kernels': the entry
// points refuse such problems before any kernel is chosen).
constexpr uint64_t kStreamingMaxWeights = uint64_t{1} << 33;

// What the streaming kernel has to promise to take a shape from the decode kernel, in us; 0: it does not.  Blocks along N, where the
// decode kernel has one column tile per workgroup: less than 0.92 of its own estimate (523 shapes, K up to 8192: 7.5 % rms;
// M = 2, N = 28416, K = 7936 42.6 -> 25.2 us, M = 3, N = 27072, K = 1152 10.3 -> 6.6), 0.87 up to K = 1152 (of 55 shapes there between
// 0.87 and 0.92 of it 26 are faster and 18 slower by more than 2 %, below it 48 and 4; with a longer K 137 and 12).  Of 215 measured
// shapes that it gives to the streaming kernel 185 are faster and 16 slower, 1.19 in the mean.  Blocks along K, K > 8192, where it
// needs sixteen waves, up to 28672 columns: less than its estimate (90 shapes, M = 4, N = 10496, K = 8704 17.9 -> 13.2, M = 2, N = 7680,
// K = 8448 15.3 -> 11.7).  On wider layers, which neither estimate was fitted on, whatever decode_shape() takes stays with the decode
// kernel, although it is behind on most: of 84 shapes with N = 28736 ... 57344, K = 8448 ... 16384 the streaming kernel is faster on 81,
// by 1.02 to 1.73 times with two to four rows, with one row from 0.88 to 1.53.
inline double decode_bar_us(const DecodeShape& d, int n, int k, int form) {
  const double kk = static_cast<double>(k) / 1024.0, t = static_cast<double>(n) / 4096.0;
  const double full = static_cast<double>((n + 4095) / 4096);
  const double bf = (form & kCostBf16) ? 1.0 : 0.0, no_zp = (form & kCostNoZeroPoints) ? 1.0 : 0.0, more = d.rows > 1 ? 1.0 : 0.0;
  if (d.row != 0) return (k <= 1152 ? 0.87 : 0.92) * (2.522 + 0.155 * t + kk * (full * (0.337 + 0.048 * more) + t * (0.188 + 0.208 * bf - 0.213 * no_zp)));
  if (d.waves == 16 && k > 8192 && n <= 28672) {
    return 1.777 + 2.259 * t + kk * (full * (0.345 + 0.060 * more) + t * (0.045 * bf - 0.022 * no_zp - 0.061));
  }
  return 0.0;
}

// The whole decision.  workspace_capacity: bytes of workspace the caller could hand to a split tile kernel
// (0: none, no split).
inline Choice choose(bool column_wise, bool bf16, int m, int n, int k, size_t workspace_capacity, int block_size, bool has_zp) {
  Choice c{};
  const int form = cost_form(column_wise, bf16, block_size, has_zp);
  // few rows, a K that a workgroup can request at once: the decode kernel, unless there is a bar that the streaming kernel clears
  const bool decodes = decode_shape(column_wise, m, n, k, &c.d, block_size);
  const double bar = decodes ? decode_bar_us(c.d, n, k, form) : 0.0;
  if (decodes && bar == 0.0) {
    c.family = kFamilyDecode;
    return c;
  }
  const bool streams = m <= kStreamingMaxRows && static_cast<uint64_t>(k) * static_cast<uint64_t>(n) < kStreamingMaxWeights;
  double us = std::numeric_limits<double>::infinity();
  if (streams) c.s = streaming_shape(!column_wise, m, n, k, block_size, form, &us);
  if (decodes && !(us < bar)) {
    c.family = kFamilyDecode;
    return c;
  }
  c.d = DecodeShape{};
  // The reference switches at m > 16 (src/blkq4_f16_gemm_sm80.cu:343, f16_gemm_sm80.h:63-72).  Here the weight-streaming
  // kernel keeps going, in row groups of 32 or 48, for as long as it is expected to be faster than the tile kernel, whose grid
  // cannot fill the chip when m is small.
  c.family = kFamilyTile;
  if (streams) {
    c.family = kFamilyStreaming;
    if (m <= 16) return c;
  }
  c.t = tile_plan(column_wise, m, n, k, workspace_capacity, bf16, block_size, has_zp, &us);
  if (c.t.rt != 0) c.family = kFamilyTile;
  return c;
}

}  // namespace blkq4
