// Tile kernel whose waves are dealt whole k tiles (gfx950): 64 x 128 outputs per workgroup.
//
// Four computing waves each own ALL of the tile's outputs and every fourth 64-deep k tile; four producer waves, one per
// computing wave, do nothing but copy.  The waves' accumulators are summed through LDS in wave order (every call the same
// bits), and all eight waves store the result.
//   - A computing wave reads its k tile once: 64 rows and 128 columns from LDS for 32 MFMAs, where four waves with columns of
//     their own read the rows four times, and the barrier comes once per 32 MFMAs instead of once per 8.
//   - Producer p copies for computing wave p: rows (16-byte chunks XOR-swizzled with bits 1..3 of the row, so that fragment
//     reads are free of bank conflicts), packed weights as they lie in memory, scales and zero-points four bytes a lane.
//     A ring of three k tiles per wave (two with blocks of 16), requested two rounds, about 3300 cycles, before they are read.
//   - Registers are refilled in place: a fragment's packed words, scales and zero-points are read for the next k tile as soon
//     as they have been converted, the rows of a 16-deep step as soon as its last MFMA has been issued.  So the slot of a
//     k tile is free early in the round in which it is multiplied, and a round's one barrier publishes the next k tile and
//     gives back the slot of this one.  (Blocks along N: 64 bytes of scales and zero-points per 16 k, read two words
//     ahead, so their ring is one k tile longer.)
//   - The conversion of word y + 1 and the first stage of word y + 2 are issued in the shadow of word y's MFMAs.
//
// What bounds it: instruction issue, one computing wave per SIMD.  A round of 32 MFMAs and 235 vector instructions takes 1650
// cycles (1420 with nothing but the MFMAs, 1830 - 1950 along N), which is what an MFMA's 18 cycles and 4.4 per vector
// instruction behind it come to; without the copies it is 30 cycles less, without the reads of the rows 80.  With every compute
// unit busy the clock falls to 1.8 - 2.0 GHz under the power limit (2.4 with half of them).  Beside the rounds 2 us until the
// first four k tiles (52 KB a workgroup) are there and 1 us for the sum through LDS (128 KB in, 128 KB out, at 128 bytes a
// cycle).  Tried instead of producer waves: eight computing waves, pairs that share a k tile and copy for themselves, 2290
// cycles a round (1730 without their copies).
// Layers launched one after the other, against waves with columns of their own: fp16, blocks of 64, M = 512, N = K = 4096
// 22.9 -> 21.4 us, M = 256 (unsplit) 18.8 -> 16.9; bf16, blocks of 32, M = 256 24.4 -> 19.7; blocks along N, blocks of 32,
// M = 150 in two parts 18.2 -> 16.5.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "blkq4_choose.h"
#include "blkq4_dequant.h"
#include "blkq4_device.h"
#include "blkq4_launch.h"
#include "blkq4_gemm_common.h"

// This file is compiled twice: as it is for fp16, and through blkq4_kdeal_bf16.hip, which defines BLKQ4_KDEAL_BF16 before
// including it, for bf16 activations, scales and outputs.
#ifdef BLKQ4_KDEAL_BF16
#define BLKQ4_KDEAL_ENTRY blkq4_dev_kdeal_bf16
#else
#define BLKQ4_KDEAL_ENTRY blkq4_dev_kdeal
#endif

namespace {

using namespace blkq4;

#ifdef BLKQ4_KDEAL_BF16
constexpr bool kBF = true;
#else
constexpr bool kBF = false;
#endif

constexpr int kDealt = 4;  // k tiles of a round: computing waves, and as many producer waves
constexpr int kThreads = 64 * 2 * kDealt;

// RT, NT: 32-row and 32-column fragments of the tile.
template <int BS, bool HAS_ZP, int RT, int NT, bool ROW>
struct Layout {
  static constexpr int kRows = 32 * RT;
  static constexpr int kCols = 32 * NT;
  static constexpr int kBlocks = 64 / BS;       // blocks along K: quantization block rows of a k tile
  static constexpr int kGroups = kCols / BS;    // blocks along N: column groups of the tile, 64 scales and zero-points each
  static constexpr int kSWords = ROW ? kGroups * 32 : kBlocks * kCols / 2;
  static constexpr int kZWords = !HAS_ZP ? 0 : ROW ? kGroups * 16 : kBlocks * kCols / 4;
  static constexpr int kSOps = (kSWords + 63) / 64;
  static constexpr int kZOps = (kZWords + 63) / 64;
  static constexpr int kAOps = 4 * RT;
  static constexpr int kOps = kAOps + NT + kSOps + kZOps;  // copies of a k tile
  // a wave's LDS: a ring of slots for rows and packed weights, then one for scales and zero-points
  static constexpr int kSlotBytes = RT * 4096 + NT * 1024;
  // (blocks along N: the producer turns the zero-points, 64 bytes a group, into the 128 bytes of pairs the conversion adds)
  static constexpr int kMetaBytes = kSOps * 256 + (ROW && HAS_ZP ? kGroups * 128 : kZOps * 256);
  static constexpr int kMetaAhead = ROW ? 1 : 0;
  static constexpr int wave_bytes(int ring) { return ring * kSlotBytes + (ring + kMetaAhead) * kMetaBytes; }
  static constexpr int kRing = kDealt * wave_bytes(3) <= static_cast<int>(kMaxLdsBytes) ? 3 : 2;
  static constexpr int kMetaRing = kRing + kMetaAhead;
  static constexpr int kWaveBytes = wave_bytes(kRing);
  static constexpr int kRowWords = kCols + 4;  // of a partial tile's row: rows start four banks apart
  static constexpr int kPartBytes = kRows * kRowWords * 4;
  static constexpr int kLdsBytes = kDealt * (kWaveBytes > kPartBytes ? kWaveBytes : kPartBytes);
  static_assert(kLdsBytes <= static_cast<int>(kMaxLdsBytes), "does not fit in LDS");
  static_assert((kRing - 1) * kOps <= 63, "the counter of outstanding requests");
};

// (BF repeats kBF so that the two compilations' kernels carry different names in a trace)
// SK: the last `split_tiles` tiles are computed by `split_k` workgroups each, exactly as in the tile kernel: partial tiles in
// `partials`, an arrival counter per tile, the last to arrive adds the parts in order.
template <int BS, bool HAS_ZP, int RT, int NT, bool ROW, bool SK, bool BF = kBF>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void kdeal_mfma_kernel(
    const uint8_t* __restrict__ A, const uint8_t* __restrict__ W, const uint8_t* __restrict__ S, const uint8_t* __restrict__ Z,
    uint16_t* __restrict__ C, const uint16_t* __restrict__ bias, int M, int N, int K, int m_tiles, int whole_tiles,
    int split_tiles, int split_k, float* __restrict__ partials, int* __restrict__ counters, int xcd_map) {
  using L = Layout<BS, HAS_ZP, RT, NT, ROW>;
  constexpr int kRing = L::kRing;
  constexpr int kMeta = (BS == 16) ? 2 : 1;  // quantization blocks inside a lane's 32-deep unit
  constexpr int kWords = 4 * NT;             // packed words of a lane per k tile
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)(smem)));

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int deal = wave & (kDealt - 1);  // which k tiles of four: the computing wave's, and its producer's

  // ---- workgroup -> tile (and part), as in the tile kernel ----
  int tile = blockIdx.x, part = 0, parts = 1;
  if (SK && tile >= whole_tiles) {
    const int u = tile - whole_tiles;
    tile = whole_tiles + u % split_tiles;
    part = u / split_tiles;
    parts = split_k;
  }
  int bm = tile % m_tiles, bn = tile / m_tiles;
  if (xcd_map != 0 && tile < (whole_tiles & ~255)) {
    // a round of 256 tiles in blocks per XCD (encoding: xcd_tile_map())
    const int xm = xcd_map & 15, rp = (xcd_map >> 4) & 15, cl = (xcd_map >> 8) & 15;
    const int wl = tile & 255, x = wl & 7, j = wl >> 3;
    bm = ((x & ((1 << xm) - 1)) << rp) + (j & ((1 << rp) - 1));
    bn = ((tile >> 8) << cl) + ((x >> xm) << (5 - rp)) + (j >> rp);
  }
  const int m0 = bm * L::kRows, c0 = bn * L::kCols;
  const int kt_first = SK ? static_cast<int>(static_cast<long>(K >> 6) * part / parts) : 0;
  const int KT = (SK ? static_cast<int>(static_cast<long>(K >> 6) * (part + 1) / parts) : (K >> 6)) - kt_first;
  const int rounds = (KT + kDealt - 1) / kDealt;
  const int mine = (KT - deal + kDealt - 1) / kDealt;  // this wave's k tiles: rounds, or one less
  const uint32_t slots = lds0 + deal * L::kWaveBytes;
  const uint32_t metas = slots + kRing * L::kSlotBytes;

  const int i = lane & 31;  // column of a weight fragment / row of an activation fragment
  const int h = lane >> 5;  // the 32-deep unit of the k tile that the lane multiplies
  float16_t acc[NT][RT];

  if (wave >= kDealt) {
    // ---- producer wave ----
    uint32_t a_voff[L::kAOps];
#pragma unroll
    for (int p = 0; p < L::kAOps; ++p) {  // eight rows a copy (a row past the last one: the last one)
      const int r8 = lane >> 3;
      a_voff[p] = static_cast<uint32_t>(min(m0 + 8 * p + r8, M - 1)) * (2u * K) + ((lane & 7) ^ (4 * (p & 1) + (r8 >> 1))) * 16u;
    }
    uint32_t w_voff[NT], s_voff[L::kSOps], z_voff[L::kZOps > 0 ? L::kZOps : 1];
#pragma unroll
    for (int t = 0; t < NT; ++t) {  // (a column past the matrix' last one: the last one)
      w_voff[t] = (h * static_cast<uint32_t>(N) + min(c0 + 32 * t + i, N - 1)) * 16u;
    }
    // 32-bit word d of the k tile's scales (two in a word) or zero-points (four): the index of its first element
    auto meta_index = [&](int d, int elems, int words) -> uint32_t {
      d = min(d, words - 1);
      if (ROW) {  // (a group past the matrix' last one: the last one)
        const int per_group = 64 / elems;
        return static_cast<uint32_t>(min(c0 / BS + d / per_group, N / BS - 1)) * K + (d % per_group) * elems;
      }
      const int per_row = L::kCols / elems;
      return static_cast<uint32_t>(d / per_row) * N + min(c0 + (d % per_row) * elems, N - elems);
    };
#pragma unroll
    for (int p = 0; p < L::kSOps; ++p) s_voff[p] = meta_index(64 * p + lane, 2, L::kSWords) * 2;
#pragma unroll
    for (int p = 0; p < L::kZOps; ++p) z_voff[p] = meta_index(64 * p + lane, 4, L::kZWords);
    const bool once = m_tiles == 1;  // every packed weight is read once per launch
    auto request = [&](int r, int slot, int meta) __attribute__((always_inline)) {
      const int kt = kt_first + kDealt * r + deal;
      const uint32_t dst = slots + slot * L::kSlotBytes;
      const uint32_t mdst = metas + meta * L::kMetaBytes;
      const uint8_t* const wb = W + static_cast<size_t>(kt) * N * 32;
      const size_t meta0 = static_cast<size_t>(kt) * (ROW ? 64 : L::kBlocks * N);
      if (once) {
#pragma unroll
        for (int t = 0; t < NT; ++t) async_copy_16_once(dst + RT * 4096 + t * 1024, wb, w_voff[t]);
      } else {
#pragma unroll
        for (int t = 0; t < NT; ++t) async_copy_16(dst + RT * 4096 + t * 1024, wb, w_voff[t]);
      }
#pragma unroll
      for (int p = 0; p < L::kSOps; ++p) async_copy_4(mdst + p * 256, S + meta0 * 2, s_voff[p]);
#pragma unroll
      for (int p = 0; p < L::kZOps; ++p) async_copy_4(mdst + (L::kSOps + p) * 256, Z + meta0, z_voff[p]);
      const uint8_t* const ab = A + static_cast<size_t>(kt) * 128;
#pragma unroll
      for (int p = 0; p < L::kAOps; ++p) async_copy_16(dst + p * 1024, ab, a_voff[p]);
    };
    // Blocks along N: the zero-points of a k tile, where they landed, become the pairs -(1024 + zp) or -(64 + zp) that the
    // conversion adds, for word j of a lane's unit sixteen bytes at 16 j.  Word w of a group's zero-points holds pair w % 4
    // of the two words of 16-row group w / 4 (see row_neg_c()).  Seven vector instructions per packed word that a computing
    // wave would issue beside its MFMAs.
    auto make_pairs = [&](int meta) __attribute__((always_inline)) {
      const RowMetaMasks rmasks = RowMetaMasks::make();
      const uint32_t base = metas + meta * L::kMetaBytes + L::kSOps * 256;
      constexpr int kEach = L::kZOps;
      uint32_t z[kEach > 0 ? kEach : 1];
#pragma unroll
      for (int p = 0; p < kEach; ++p) z[p] = lds_read_u32(base + (64 * p + lane) * 4);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the first is written over
#pragma unroll
      for (int p = 0; p < kEach; ++p) {
        const int d = 64 * p + lane, e = d & 3;
        const uint32_t lo = (e & 1) == 0 ? as_u32(row_neg_c<true>(z[p], 0, 0, rmasks)) : as_u32(row_neg_c<true>(z[p], 1, 0, rmasks));
        const uint32_t hi = (e & 1) == 0 ? as_u32(row_neg_c<true>(z[p], 0, 1, rmasks)) : as_u32(row_neg_c<true>(z[p], 1, 1, rmasks));
        if (d < L::kZWords) {
          const uint32_t at = base + (d >> 2) * 32 + e * 4;
          lds_write_4(at, 0, lo);
          lds_write_4(at, 16, hi);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
#pragma unroll
    for (int d = 0; d < kRing; ++d) {
      if (d < mine) request(d, d, d);
    }
    // k tile 0 has landed: everything but the requests behind it
    if (kRing == 3 && mine > 2) wait_vmcnt<(kRing - 1) * L::kOps>();
    else if (mine > 1) wait_vmcnt<L::kOps>();
    else wait_vmcnt<0>();
    if (ROW && HAS_ZP && mine > 0) make_pairs(0);
    block_barrier();
    int slot = 0, meta = kRing % L::kMetaRing;  // of k tile r + kRing
    int next_meta = 1;                          // of k tile r + 1
    for (int r = 0; r < rounds; ++r) {
      // k tile r + 1 has landed: behind it only r + 2 has been requested
      if (kRing == 3 && r + 2 < mine) wait_vmcnt<L::kOps>();
      else wait_vmcnt<0>();
      if (ROW && HAS_ZP && r + 1 < mine) make_pairs(next_meta);
      block_barrier();  // also: the slot of k tile r has been read
      if (r + kRing < mine) request(r + kRing, slot, meta);
      slot = slot + 1 < kRing ? slot + 1 : 0;
      meta = meta + 1 < L::kMetaRing ? meta + 1 : 0;
      next_meta = next_meta + 1 < L::kMetaRing ? next_meta + 1 : 0;
    }
  } else {
    // ---- computing wave ----
    uint32_t a_rd[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) a_rd[j] = slots + i * 128 + (((4 * h + j) ^ ((i >> 1) & 7)) * 16);
    const uint32_t w_rd = slots + RT * 4096 + lane * 16;
    const int block = (BS == 64) ? 0 : (BS == 32) ? h : 2 * h;
    // blocks along N: the lane's 32 rows are two 16-row groups, 32 bytes of scales and 32 of zero-point pairs each
    const uint32_t s_rd = metas + (ROW ? (BS < 32 ? (i / BS) * 128 : 0) + h * 64 : (block * L::kCols + i) * 2);
    const uint32_t z_rd = metas + L::kSOps * 256 + (ROW ? (BS < 32 ? (i / BS) * 128 : 0) + h * 64 : block * L::kCols + i);
    const DequantMasks masks = DequantMasks::make();

    half8_t af[4][RT];
    uint32_t words[NT][4];
    uint32_t sc[NT][kMeta], zp[NT][kMeta];
    uint4 rs[2][2], rn[2][2];  // blocks along N: the two 16-row groups of the fragment being converted
    half2_t pt[2][4];       // words on their way through the conversion
    half2_t wf[2][4];       // converted words
    DequantConsts dc[2];
    Bf16Consts bc[2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int x = 0; x < RT; ++x) acc[t][x] = float16_t(0.f);

    auto read_weights = [&](int t, uint32_t so, uint32_t mo) __attribute__((always_inline)) {
      const uint4 v = lds_read_16(w_rd + so, t * 1024);
      words[t][0] = v.x;
      words[t][1] = v.y;
      words[t][2] = v.z;
      words[t][3] = v.w;
      if constexpr (!ROW) {
#pragma unroll
        for (int q = 0; q < kMeta; ++q) {
          sc[t][q] = lds_read_u16(s_rd + mo, (q * L::kCols + 32 * t) * 2);
          zp[t][q] = HAS_ZP ? lds_read_u8(z_rd + mo, q * L::kCols + 32 * t) : 8u;
        }
      }
    };
    auto read_row_meta = [&](int t, int g, uint32_t mo) __attribute__((always_inline)) {
      rs[g][0] = lds_read_16(s_rd + mo, (32 * t / BS) * 128 + g * 32);
      rs[g][1] = lds_read_16(s_rd + mo, (32 * t / BS) * 128 + g * 32 + 16);
      if (HAS_ZP) {
        rn[g][0] = lds_read_16(z_rd + mo, (32 * t / BS) * 128 + g * 32);
        rn[g][1] = lds_read_16(z_rd + mo, (32 * t / BS) * 128 + g * 32 + 16);
      }
    };
    auto read_rows = [&](int j, uint32_t so) __attribute__((always_inline)) {
#pragma unroll
      for (int x = 0; x < RT; ++x) af[j][x] = as_half8(lds_read_16(a_rd[j] + so, x * 4096));
    };
    // The conversion of word y (fragment y / 4, word y % 4) in three stages.  y counts on into the next k tile.
    // Blocks along N: word j is rows 8 (j & 1) .. + 7 of 16-row group j / 2.
    auto set_of = [](int y) { return (y / (4 / kMeta)) & 1; };
    auto stage0 = [&](int y) __attribute__((always_inline)) {
      const int t = (y % kWords) / 4, j = y % 4;
      if (!ROW && j % (4 / kMeta) == 0) {
        if constexpr (kBF) bc[set_of(y)] = make_bf16_consts(sc[t][j / (4 / kMeta)], zp[t][j / (4 / kMeta)]);
        else dc[set_of(y)] = make_dequant_consts(sc[t][j / (4 / kMeta)], zp[t][j / (4 / kMeta)]);
      }
      const uint32_t w = words[t][j], ws = w >> 8;
      pt[y & 1][0] = as_half2((w & masks.lo_mask) | masks.magic_1024);
      pt[y & 1][1] = as_half2((w & masks.hi_mask) | masks.magic_64);
      pt[y & 1][2] = as_half2((ws & masks.lo_mask) | masks.magic_1024);
      pt[y & 1][3] = as_half2((ws & masks.hi_mask) | masks.magic_64);
    };
    float pf[4][2];
    auto stage1 = [&](int y) __attribute__((always_inline)) {
      const int g = (y % 4) >> 1, hh = y & 1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (ROW) {
          pt[y & 1][e] = pt[y & 1][e] + (HAS_ZP ? as_half2(vec_word(rn[g][hh], e)) : as_half2((e & 1) == 0 ? 0xE408E408u : 0xD480D480u));
        } else if constexpr (kBF) {
          const Bf16Consts& b = bc[set_of(y)];
          pf[e][0] = __builtin_fmaf(static_cast<float>(pt[y & 1][e][0]), b.scale, (e & 1) == 0 ? b.neg_c0 : b.neg_c1);
          pf[e][1] = __builtin_fmaf(static_cast<float>(pt[y & 1][e][1]), b.scale, (e & 1) == 0 ? b.neg_c0 : b.neg_c1);
        } else {
          pt[y & 1][e] = pt[y & 1][e] + ((e & 1) == 0 ? dc[set_of(y)].neg_c0 : dc[set_of(y)].neg_c1);
        }
      }
    };
    auto stage2 = [&](int y) __attribute__((always_inline)) {
      const int g = (y % 4) >> 1, hh = y & 1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (ROW) {
          const uint32_t pair = vec_word(rs[g][(2 * e + hh) >> 2], (2 * e + hh) & 3);
          if constexpr (kBF) wf[y & 1][e] = as_half2(row_pair_bf16(pt[y & 1][e], pair));
          else wf[y & 1][e] = pt[y & 1][e] * as_half2(pair);
        } else if constexpr (kBF) {
          typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
          bf16x2_t v;
          v[0] = static_cast<__bf16>(pf[e][0]);
          v[1] = static_cast<__bf16>(pf[e][1]);
          wf[y & 1][e] = __builtin_bit_cast(half2_t, v);
        } else {
          wf[y & 1][e] = pt[y & 1][e] * dc[set_of(y)].scale2;
        }
      }
    };
    struct half2x4_t { half2_t a, b, c, d; };

    block_barrier();  // k tile 0 has landed
    if (mine > 0) {
#pragma unroll
      for (int t = 0; t < NT; ++t) read_weights(t, 0, 0);
      if (ROW) {
        read_row_meta(0, 0, 0);
        read_row_meta(0, 1, 0);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) read_rows(j, 0);
      stage0(0);
      stage1(0);
      stage2(0);
      stage0(1);
    }
    // offsets of the next k tile's slots, and of this one's scales and zero-points
    uint32_t next = L::kSlotBytes, next_meta = L::kMetaBytes, meta = 0;
    for (int r = 0; r < rounds; ++r) {
      if (r < mine) {
        BLKQ4_PIN();
#pragma unroll
        for (int y = 0; y < kWords; ++y) {
          const int t = y / 4, j = y % 4;
#pragma unroll
          for (int x = 0; x < RT; ++x) {
            const half8_t w = __builtin_bit_cast(half8_t, half2x4_t{wf[y & 1][0], wf[y & 1][1], wf[y & 1][2], wf[y & 1][3]});
            if constexpr (kBF) {
              acc[t][x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, af[j][x]), acc[t][x], 0, 0, 0);
            } else {
              acc[t][x] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, af[j][x], acc[t][x], 0, 0, 0);
            }
            BLKQ4_PIN();
            if (x == 0) {
              stage1(y + 1);
              stage2(y + 1);
            }
            if (x == RT - 1) {
              stage0(y + 2);
              // refills for the next k tile (past the last one: whatever lies there, and nothing uses it)
              if (t == NT - 1) read_rows(j, next);
              if (y >= 4 && j == 0) read_weights(t - 1, next, next_meta);
              if (y == kWords - 1) read_weights(NT - 1, next, next_meta);
              // blocks along N: the next fragment's, each 16-row group once this fragment's last word of it is converted
              if (ROW && (j == 0 || j == 2)) read_row_meta((t + 1) % NT, j / 2, t + 1 < NT ? meta : next_meta);
            }
            BLKQ4_PIN();
          }
          if (y == 3) {
            // the slot of this k tile has been read, its producer may refill it; the next k tile has landed
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            block_barrier();
          }
        }
        next = next + L::kSlotBytes < kRing * L::kSlotBytes ? next + L::kSlotBytes : 0;
        meta = next_meta;
        next_meta = next_meta + L::kMetaBytes < L::kMetaRing * L::kMetaBytes ? next_meta + L::kMetaBytes : 0;
      } else {
        block_barrier();
      }
    }
  }

  // ---- the waves' partial tiles, [wave][row][columns + 4 of padding] floats, where the ring was ----
  block_barrier();
  if (wave < kDealt) {
    const uint32_t wr = lds0 + wave * L::kPartBytes + (i * L::kRowWords + 4 * h) * 4;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int x = 0; x < RT; ++x)
#pragma unroll
        for (int g = 0; g < 4; ++g) {  // elements 4 g .. 4 g + 3: row i, columns 8 g + 4 h .. + 3
          const float e0 = acc[t][x][4 * g], e1 = acc[t][x][4 * g + 1], e2 = acc[t][x][4 * g + 2], e3 = acc[t][x][4 * g + 3];
          lds_write_16(wr, (32 * x * L::kRowWords + 32 * t + 8 * g) * 4, __float_as_uint(e0), __float_as_uint(e1),
                       __float_as_uint(e2), __float_as_uint(e3));
        }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  block_barrier();
  constexpr int kChunks = L::kCols / 8;                      // eight columns of a row
  constexpr int kPasses = L::kRows * kChunks / kThreads;
  static_assert(L::kRows * kChunks % kThreads == 0, "whole passes");
  constexpr int kRowsPerPass = kThreads / kChunks;
  const int chunk = tid % kChunks, row0 = tid / kChunks;
  const int col = c0 + chunk * 8;
  float sum[kPasses][8];
#pragma unroll
  for (int v = 0; v < kPasses; ++v) {
    const uint32_t rd = lds0 + ((row0 + v * kRowsPerPass) * L::kRowWords + chunk * 8) * 4;
#pragma unroll
    for (int w = 0; w < kDealt; ++w) {
      const uint4 lo = lds_read_16(rd, w * L::kPartBytes), hi = lds_read_16(rd, w * L::kPartBytes + 16);
      const float f[8] = {__uint_as_float(lo.x), __uint_as_float(lo.y), __uint_as_float(lo.z), __uint_as_float(lo.w),
                          __uint_as_float(hi.x), __uint_as_float(hi.y), __uint_as_float(hi.z), __uint_as_float(hi.w)};
#pragma unroll
      for (int e = 0; e < 8; ++e) sum[v][e] = (w == 0) ? f[e] : sum[v][e] + f[e];
    }
  }
  if (SK && parts > 1) {
    // The exchange between workgroups on different XCDs, as in the tile kernel: device-scope accesses, stores acknowledged
    // when the device can see them, and one acquire in the workgroup that arrives last, which has its own part in registers.
    constexpr int kPairs = kPasses * 4 * kThreads;  // 8-byte pairs of a partial tile
    const int st = tile - whole_tiles;
    uint64_t* const tile_parts = reinterpret_cast<uint64_t*>(partials) + static_cast<size_t>(st) * parts * kPairs + tid;
    uint64_t* const own = tile_parts + static_cast<size_t>(part) * kPairs;
#pragma unroll
    for (int v = 0; v < kPasses; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint64_t pair = static_cast<uint64_t>(__float_as_uint(sum[v][2 * e])) |
                              static_cast<uint64_t>(__float_as_uint(sum[v][2 * e + 1])) << 32;
        __hip_atomic_store(own + (4 * v + e) * kThreads, pair, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    wait_vmcnt<0>();  // this wave's stores have been acknowledged
    block_barrier();  // every wave's have
    if (tid == 0) {
      const int arrived = __hip_atomic_fetch_add(&counters[st], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (arrived == parts - 1) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        // nobody else touches this counter any more in this launch: back to zero for the next one
        __hip_atomic_store(&counters[st], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      lds_write_8(lds0, 0, static_cast<uint32_t>(arrived), 0u);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    block_barrier();
    const int arrived = static_cast<int>(lds_read_u32(lds0));
    if (arrived != parts - 1) return;  // somebody else finishes this tile
    float total[kPasses][8];
    for (int p = 0; p < parts; ++p) {  // fixed order, whoever arrived last: part 0 + part 1 + ...
      float in[kPasses][8];
      if (p == part) {
#pragma unroll
        for (int y = 0; y < kPasses * 8; ++y) in[y / 8][y % 8] = sum[y / 8][y % 8];
      } else {
        const uint64_t* src = tile_parts + static_cast<size_t>(p) * kPairs;
        uint64_t pair[kPasses * 4];
#pragma unroll
        for (int y = 0; y < kPasses * 4; ++y) pair[y] = __hip_atomic_load(src + y * kThreads, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int y = 0; y < kPasses * 4; ++y) {
          in[y / 4][2 * (y % 4)] = __uint_as_float(static_cast<uint32_t>(pair[y]));
          in[y / 4][2 * (y % 4) + 1] = __uint_as_float(static_cast<uint32_t>(pair[y] >> 32));
        }
      }
#pragma unroll
      for (int y = 0; y < kPasses * 8; ++y) total[y / 8][y % 8] = (p == 0) ? in[y / 8][y % 8] : total[y / 8][y % 8] + in[y / 8][y % 8];
    }
#pragma unroll
    for (int y = 0; y < kPasses * 8; ++y) sum[y / 8][y % 8] = total[y / 8][y % 8];
  }
  uint4 bias8 = make_uint4(0, 0, 0, 0);
  if (bias != nullptr && col < N) bias8 = *reinterpret_cast<const uint4*>(bias + col);
#pragma unroll
  for (int v = 0; v < kPasses; ++v) {
    uint4 o = make_uint4(float_to_bits<kBF>(sum[v][0]) | (float_to_bits<kBF>(sum[v][1]) << 16),
                         float_to_bits<kBF>(sum[v][2]) | (float_to_bits<kBF>(sum[v][3]) << 16),
                         float_to_bits<kBF>(sum[v][4]) | (float_to_bits<kBF>(sum[v][5]) << 16),
                         float_to_bits<kBF>(sum[v][6]) | (float_to_bits<kBF>(sum[v][7]) << 16));
    if (bias != nullptr) {
      o = make_uint4(add_bias_pair_t<kBF>(o.x, bias8.x), add_bias_pair_t<kBF>(o.y, bias8.y),
                     add_bias_pair_t<kBF>(o.z, bias8.z), add_bias_pair_t<kBF>(o.w, bias8.w));
    }
    const int m = m0 + row0 + v * kRowsPerPass;
    if (m < M && col < N) {  // written once, not read again by this launch
      __builtin_nontemporal_store(uint4_t{o.x, o.y, o.z, o.w}, reinterpret_cast<uint4_t*>(C + static_cast<size_t>(m) * N + col));
    }
  }
}

template <int BS, bool HAS_ZP, bool ROW, bool SK>
int launch_one(const blkq4_gemm_args* a) {
  constexpr int RT = 2, NT = 4;
  using L = Layout<BS, HAS_ZP, RT, NT, ROW>;
  const blkq4_tile_plan& t = a->tile;
  // as the choice names the tile, or by this kernel's own name
  if (t.wm != 1 || t.pw != 4 || !((t.rt == RT && t.nt == 1 && t.wn == 4 && t.kw == 1) || (t.rt == RT && t.nt == NT && t.wn == 1 && t.kw == kDealt))) {
    return static_cast<int>(hipErrorInvalidValue);
  }
  const int m_tiles = (a->m + L::kRows - 1) / L::kRows;
  const int tiles = m_tiles * ((a->n + L::kCols - 1) / L::kCols);
  if (a->launched_id != nullptr) *a->launched_id = tile_id(t.rt, t.nt, t.wm, t.wn, t.pw, SK, t.kw);
  int whole = tiles, split_tiles = 0, split_k = 1;
  float* partials = nullptr;
  int* counters = nullptr;
  if (SK) {
    // what the kernel assumes about the workspace, checked here: counters first, then the partial tiles
    split_tiles = t.split_tiles;
    split_k = t.split_k;
    whole = tiles - split_tiles;
    const size_t need = kCounterBytes + static_cast<size_t>(split_tiles) * split_k * L::kRows * L::kCols * 4;
    if (split_tiles < 1 || split_tiles > tiles || split_k < 2 || split_k > a->k / 64 ||
        static_cast<size_t>(split_tiles) * sizeof(int) > kCounterBytes || t.workspace_bytes != need) {
      return static_cast<int>(hipErrorInvalidValue);
    }
    if (a->dry_run) return 0;  // the plan has passed every check a launch makes but those of the buffer itself
    if (a->workspace == nullptr || a->workspace_bytes < need || (reinterpret_cast<uintptr_t>(a->workspace) & 255u) != 0) {
      return static_cast<int>(hipErrorInvalidValue);
    }
    counters = static_cast<int*>(a->workspace);
    partials = reinterpret_cast<float*>(static_cast<char*>(a->workspace) + kCounterBytes);
  }
  if (t.tiles != tiles) return static_cast<int>(hipErrorInvalidValue);
  int xcd_map = 0;
  if (t.xcd_rows != 0 && !xcd_tile_map(m_tiles, t.xcd_rows, &xcd_map)) return static_cast<int>(hipErrorInvalidValue);
  if (a->dry_run) return 0;
  constexpr auto kernel = kdeal_mfma_kernel<BS, HAS_ZP, RT, NT, ROW, SK>;
  const hipError_t attr = raise_lds_limit_once(reinterpret_cast<const void*>(kernel), kMaxLdsBytes, &lds_limit_flags<kernel>());
  if (attr != hipSuccess) return static_cast<int>(attr);
  const dim3 grid(static_cast<unsigned>(whole + split_tiles * split_k));
  // the launch's own status: a sticky error of an earlier, unrelated call stays where it is
  return static_cast<int>(launch_status(kernel, grid, dim3(kThreads), L::kLdsBytes, a->stream,
                                        static_cast<const uint8_t*>(a->a), static_cast<const uint8_t*>(a->packed_w),
                                        static_cast<const uint8_t*>(a->scales), static_cast<const uint8_t*>(a->zero_points),
                                        static_cast<uint16_t*>(a->c), static_cast<const uint16_t*>(a->bias), a->m, a->n, a->k,
                                        m_tiles, whole, split_tiles, split_k, partials, counters, xcd_map));
}

template <int BS, bool HAS_ZP>
int launch_plan(const blkq4_gemm_args* a) {
  const bool sk = a->tile.split_k > 1;
  if (a->column_wise) return sk ? launch_one<BS, HAS_ZP, false, true>(a) : launch_one<BS, HAS_ZP, false, false>(a);
  return sk ? launch_one<BS, HAS_ZP, true, true>(a) : launch_one<BS, HAS_ZP, true, false>(a);
}

template <int BS>
int launch_bs(const blkq4_gemm_args* a) {
  return a->zero_points ? launch_plan<BS, true>(a) : launch_plan<BS, false>(a);
}

}  // namespace

extern "C" int BLKQ4_KDEAL_ENTRY(const blkq4_gemm_args* a) {
  if (a->m < 1 || (a->n % 32) != 0 || a->n < 32 || (a->k % 64) != 0 || a->k < 64 || (!a->column_wise && (a->n % a->block_size) != 0)) return static_cast<int>(hipErrorInvalidValue);
  // scales and zero-points are copied four bytes at a time
  if ((reinterpret_cast<uintptr_t>(a->scales) & 3u) != 0 || (reinterpret_cast<uintptr_t>(a->zero_points) & 3u) != 0) {
    return static_cast<int>(hipErrorInvalidValue);
  }
  // the async copies address A and W with 32-bit byte offsets
  if (static_cast<uint64_t>(a->m) * a->k * 2 >= (1ull << 32) || static_cast<uint64_t>(a->k) * a->n / 2 >= (1ull << 32)) {
    return static_cast<int>(hipErrorInvalidValue);
  }
  switch (a->block_size) {
    case 16: return launch_bs<16>(a);
    case 32: return launch_bs<32>(a);
    case 64: return launch_bs<64>(a);
    default: return static_cast<int>(hipErrorInvalidValue);
  }
}
