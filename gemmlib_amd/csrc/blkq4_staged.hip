// Weight-streaming kernel for gfx950, rows staged slice by slice: up to 16 rows wherever the decode kernel does not take them, and
// more rows in groups of 32 or 48, both blockings.
//
// A workgroup of 16, 8 or 4 waves owns 16 * NT output columns, up to 16, 32 or 48 rows and all of K.  The waves split K into
// 64-deep slices; a wave multiplies all the workgroup's rows with all its columns over its slices, and the waves' partial
// tiles are summed through LDS in wave order: no barrier before that sum, every call the same bits.
//   - Everything a slice needs goes HBM / L2 -> LDS by asynchronous copies, private to the wave: the rows' 128 bytes each
//     (16-byte chunks XOR-swizzled with bits 1..3 of the row, so that fragment reads are free of bank conflicts), the packed
//     weights in the order they lie in memory, scales and zero-points four bytes a lane.  A wave has DEPTH slices of LDS.  It
//     waits for a slice by the count of requests behind it, reads all of it into registers at once, requests the slice
//     DEPTH further on into the same LDS, and only then converts and multiplies.  The waits are exact because the compiler
//     issues no vector memory request of its own in the loop.
//   - Row groups of 32: fragments of 32 columns x 16 k and v_mfma_f32_32x32x16, one conversion for 32 rows; a lane reads its
//     16-byte unit back whole.  16 or 48 rows, 16 columns, blocks along N: v_mfma_f32_16x16x32, a lane takes half a unit (two of
//     its four words), which keeps the slice 64 deep.  64 because K is a multiple of that: there is no partial slice.
//   - Row groups of 48: 33 to 48 rows are one group instead of two, so every weight is fetched and converted once: 40 rows,
//     N = 14336, K = 4096 16.9 -> 13.0 us, M = 48, N = 11008 14.7 -> 12.7, M = 144, N = 4096 12.9 -> 12.1.  (64 rows a group
//     were tried on one shape, along K: M = 64, N = 8192, K = 4096 11.1 in two groups, 12.4 in one.)
//   - Blocks along N: with one column tile a workgroup fetches the rows again for every 16 columns and builds the zero-point
//     constants of its 16-row groups (half of a word's instructions) for one tile.  Two, four or eight tiles share both: K = N = 4096,
//     M = 150 11.7 us (tiles, which ran there, 16.3), M = 48, N = 8192, K = 2048 11.7 -> 7.0, M = 12, N = 53440, K = 3584 45.5 -> 28.8.
//   - The copies' lane offsets never change, the slice moves a scalar base: a request costs no vector instruction.
//   - Rows are dealt evenly to the row groups (64 rows: two groups of 32); the row groups of a column group run on one
//     XCD and share its weights there.  With a single row group the weights are read once per launch: non-temporal.
//   - A SIMD serves its older wave first, also its memory requests: of eight waves the younger four get their first slice
//     1.8 us after the others (M = 48, N = 11008) and finish last.  So the older half takes extra rounds of slices
//     (staged_extra_rounds() in blkq4_choose.h): M = 128, K = N = 4096 8.9 -> 8.5 us.
//   - A wave's slice is a chain (wait, read LDS, request, convert, multiply) of 850 cycles whatever its depth, and two waves a
//     SIMD do not cover it: with eight rows or less on a long K, and with blocks along N, sixteen waves with half the depth
//     each.  M = 3, N = 2048, K = 23360 20.1 -> 15.7 us, M = 6, N = 960, K = 16320 13.0 -> 11.1 (five slices in flight for
//     eight waves: 12.8), blocks along N, M = 8, N = 8192, K = 7552 9 % less.
//
// What bounds it, from a copy of this kernel that does nothing but its requests -- rows alone, weights with scales and
// zero-points alone, both -- and the kernel, weights from HBM, us (about 2 of each are launching and the first answer):
//   M = 16, N = 28672, K = 8192    5.1, 22.4, 22.4   25.5   the weight stream, 5.9 TB/s; the rows cost nothing beside it
//   M = 12, N = 128256, K = 4096   10.9, 46.5, 50.0  54.7   the same
//   M = 48, N = 11008, K = 4096    5.2, 9.0, 11.5    14.0   two groups of 24 rows: rows and weights overlap in part; conversion,
//                                                           twice per weight (one group of 48 rows: -, 7.2, 11.6, 13.1)
//   M = 128, N = K = 4096          4.9, 5.0, 7.1     8.9    the same, four times per weight
// Why rows and weights do not overlap better, as far as it is understood: a compute unit's vector cache returns what it was asked for
// in order, and what is asked for occupies its 32 KB until then.  Rows alone, or weights that lie in L2, come at 126 - 150 bytes a ns
// (64 a cycle); with weights from HBM (950 cycles, L2 236) between them 32 KB per HBM answer would be 70 bytes a ns; 48 rows
// see 53, whatever the order of the slices over the workgroups, and also when the rows have been brought into every L2 beforehand
// (both tried).
// What the conversion adds shares its issue port with the MFMAs, at 1.6 (M = 512) to 2.0 GHz (M = 48): the chip is power limited.
// fp16, blocks of 64, K = 4096, us, against the kernel before (128-deep slices, weights in registers, refilled after use), a few
// weight sets in turn that the Infinity Cache holds:
//   M = 64, N = 4096 8.4 -> 6.5; M = 128, N = 4096 11.4 -> 8.6; M = 48, N = 11008 15.9 -> 13.2; M = 32, N = 11008 12.7 ->
//   11.1; M = 12, N = 128256 58.7 -> 55.8; M = 12, N = 4096, K = 11008 11.8 -> 11.0; M = 16, N = 28672, K = 8192 27.9 -> 25.9.
// From HBM (600 MB of weight sets in turn): M = 64, N = 4096 8.3 -> 8.2; M = 128, N = 4096 11.3 -> 10.4; M = 48, N = 11008
//   15.9 -> 13.7; M = 16, N = 28672, K = 8192 27.3 -> 26.2.

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "blkq4_choose.h"
#include "blkq4_dequant.h"
#include "blkq4_device.h"
#include "blkq4_launch.h"
#include "blkq4_gemm_common.h"

// This file is compiled twice: as it is for fp16, and through blkq4_staged_bf16.hip, which defines BLKQ4_STAGED_BF16 before
// including it, for bf16 activations, scales and outputs.
#ifdef BLKQ4_STAGED_BF16
#define BLKQ4_STAGED_ENTRY blkq4_dev_staged_bf16
#else
#define BLKQ4_STAGED_ENTRY blkq4_dev_staged
#endif

namespace {

using namespace blkq4;

#ifdef BLKQ4_STAGED_BF16
constexpr bool kBF = true;
#else
constexpr bool kBF = false;
#endif

// NT: 16-column tiles of a workgroup; MT: 16-row tiles (1, 2 or 3).
template <int BS, bool HAS_ZP, int NT, int MT, int kWaves, int DEPTH, bool ROW>
struct Layout {
  static constexpr int F = (MT == 2 && NT % 2 == 0 && !ROW) ? 32 : 16;  // columns and rows of a fragment
  static constexpr int kFrags = 16 * NT / F;       // column fragments
  static constexpr int kRowFrags = 16 * MT / F;    // row fragments
  static constexpr int kRows = 16 * MT;
  static constexpr int kCols = 16 * NT;
  static constexpr int kABytes = kRows * 128;
  static constexpr int kWPieces = (kCols + 31) / 32;  // copies of 32 columns x 64 k
  static constexpr int kBlocks = 64 / BS;             // blocks along K: quantization block rows of a slice
  // blocks along N: the 64 scales and zero-points of each of the column groups that the workgroup's columns lie in
  static constexpr int kGroups = kCols > BS ? kCols / BS : 1;
  static constexpr int kSWords = ROW ? kGroups * 32 : kBlocks * kCols / 2;
  static constexpr int kZWords = !HAS_ZP ? 0 : ROW ? kGroups * 16 : kBlocks * kCols / 4;
  static constexpr int kSOps = (kSWords + 63) / 64;
  static constexpr int kZOps = (kZWords + 63) / 64;
  static constexpr int kWOps = kWPieces + kSOps + kZOps;
  static constexpr int kWOff = kABytes;  // a slot: rows, packed weights, scales, zero-points
  static constexpr int kSOff = kWOff + kWPieces * 1024;
  static constexpr int kZOff = kSOff + kSOps * 256;
  static constexpr int kSlotBytes = kZOff + kZOps * 256;
  static constexpr int kWaveBytes = DEPTH * kSlotBytes;
  static constexpr int kRowWords = kCols + 4;  // of a partial tile's row: rows start four banks apart
  static constexpr int kPartBytes = kRows * kRowWords * 4;
  static constexpr int kLdsBytes = kWaves * (kWaveBytes > kPartBytes ? kWaveBytes : kPartBytes);
  static_assert(kLdsBytes <= static_cast<int>(kMaxLdsBytes), "does not fit in LDS");
  static_assert(kLdsBytes == staged_lds_bytes(ROW, BS, HAS_ZP, NT, MT, kWaves, DEPTH), "what the choice counts with");
  static_assert(!ROW || BS % kCols == 0 || kCols % BS == 0, "blocks along N: whole column groups, or a part of one");
  static_assert(MT >= 1 && MT <= 3, "up to 48 rows");
  static_assert((DEPTH - 1) * (kWOps + kRows / 8) <= 63, "the counter of outstanding requests");
};

template <int F>
struct AccOf { typedef float4_t type; };
template <>
struct AccOf<32> { typedef float16_t type; };

// waits until at most n * per requests are outstanding, n <= N
template <int N, int per>
__device__ __forceinline__ void wait_slices(int n) {
  if constexpr (N == 0) {
    wait_vmcnt<0>();
  } else {
    if (n >= N) wait_vmcnt<N * per>();
    else wait_slices<N - 1, per>(n);
  }
}

// (BF repeats kBF so that the two compilations' kernels carry different names in a trace)
// The arguments that the first requests need come first: the 14 registers' worth of them arrive with the wave (kernel argument
// preload, as in the decode kernel), where a load of them was waited for before the first address could be computed: M = 64,
// N = K = 4096 6.41 -> 6.15 us, M = 128 8.68 -> 8.45, M = 48, N = 11008 12.0 -> 11.75, wide layers and long K 0.1 us.
template <int BS, bool HAS_ZP, int NT, int MT, int kWaves, int DEPTH, bool ROW, bool BF = kBF>
__global__ __launch_bounds__(64 * kWaves)
    __attribute__((amdgpu_waves_per_eu(kWaves == 8 ? 2 : 4, kWaves == 8 ? 2 : 4))) void staged_mfma_kernel(
        const uint8_t* __restrict__ A, const uint8_t* __restrict__ W, const uint8_t* __restrict__ S,
        const uint8_t* __restrict__ Z, int M_total, int N, int K, int row_groups, int rows_per_group, uint32_t row_groups_inv,
        uint16_t* __restrict__ C, const uint16_t* __restrict__ bias) {
  using L = Layout<BS, HAS_ZP, NT, MT, kWaves, DEPTH, ROW>;
  constexpr int F = L::F;
  typedef typename AccOf<F>::type acc_t;
  constexpr int kSteps = F == 32 ? 4 : 2;               // MFMA steps of a slice: words of a unit that a lane multiplies
  constexpr int kMeta = (BS == 16 && F == 32) ? 2 : 1;  // quantization blocks those words lie in
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)(smem)));

  // Workgroup -> (row group, column group), as streaming_geometry() deals them: workgroup w runs on XCD w % 8, an XCD takes
  // the row groups of a column group, then the next of a few neighbouring column groups.
  // (q / row_groups by a multiplication: the division takes 30 instructions in front of the first request)
  const int col_groups = static_cast<uint32_t>(N + L::kCols - 1) / L::kCols;
  const uint32_t q = blockIdx.x >> 3;
  const uint32_t cq = row_groups == 1 ? q : __umulhi(q, row_groups_inv);
  const uint32_t rg = q - cq * row_groups;
  constexpr int kNeighbours = streaming_neighbours(NT, kWaves, kWaves);
  const int cg = kNeighbours * ((blockIdx.x & 7) + 8 * (cq / kNeighbours)) + (cq % kNeighbours);
  const int m0 = static_cast<int>(rg) * rows_per_group;
  if (cg >= col_groups || m0 >= M_total) return;
  const int M = min(rows_per_group, M_total - m0);
  const int c0 = cg * L::kCols;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int i = lane & (F - 1);                    // column of a weight fragment / row of an activation fragment
  const int g = lane / F;
  const int unit = g & 1;                          // which 32-deep unit of the slice the lane multiplies
  const int word0 = (F == 32) ? 0 : 2 * (g >> 1);  // and from which of its four words on

  // This wave's slices: rounds of one per wave, then rounds for the older half of the waves only.
  constexpr int kOld = kWaves / 2;
  const int slices = K >> 6;
  const int rounds = static_cast<uint32_t>(max(slices - staged_extra_rounds(kWaves, K) * kOld, 0)) / kWaves;
  const int rest = slices - rounds * kWaves;
  const int mine = rounds + (wave < kOld ? static_cast<uint32_t>(rest - wave + kOld - 1) / kOld : 0);
  auto slice_of = [&](int li) { return li < rounds ? wave + kWaves * li : rounds * kWaves + wave + kOld * (li - rounds); };

  // ---- lane offsets of the copies ----
  const uint32_t slots = lds0 + wave * L::kWaveBytes;
  const int r8 = lane >> 3;
  const int row_copies = (rows_per_group + 7) >> 3;  // of eight rows; the same in every row group
  uint32_t a_voff[L::kRows / 8];
#pragma unroll
  for (int p = 0; p < L::kRows / 8; ++p) {  // (a row past the last one: the last one)
    a_voff[p] = static_cast<uint32_t>(min(8 * p + r8, M - 1)) * (2u * K) + ((lane & 7) ^ (4 * (p & 1) + (r8 >> 1))) * 16u;
  }
  uint32_t w_voff[L::kWPieces], s_voff[L::kSOps], z_voff[L::kZOps > 0 ? L::kZOps : 1];
#pragma unroll
  for (int p = 0; p < L::kWPieces; ++p) {  // (a column past the workgroup's, or the matrix', last one: the last one)
    w_voff[p] = ((lane >> 5) * static_cast<uint32_t>(N) + min(c0 + min(32 * p + (lane & 31), L::kCols - 1), N - 1)) * 16u;
  }
  // 32-bit word d of the slice's scales (two in a word) or zero-points (four): the index of its first element
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
  const uint8_t* const a_base = A + static_cast<size_t>(m0) * K * 2;
  const bool once = row_groups == 1;
  auto request = [&](int s, int slot) __attribute__((always_inline)) {
    const uint32_t dst = slots + slot * L::kSlotBytes;
    const uint8_t* const wb = W + static_cast<size_t>(s) * N * 32;
    const size_t meta0 = ROW ? static_cast<size_t>(s) * 64 : static_cast<size_t>(s) * L::kBlocks * N;
#pragma unroll
    for (int p = 0; p < L::kSOps; ++p) async_copy_4(dst + L::kSOff + p * 256, S + meta0 * 2, s_voff[p]);
#pragma unroll
    for (int p = 0; p < L::kZOps; ++p) async_copy_4(dst + L::kZOff + p * 256, Z + meta0, z_voff[p]);
    if (once) {
#pragma unroll
      for (int p = 0; p < L::kWPieces; ++p) async_copy_16_once(dst + L::kWOff + p * 1024, wb, w_voff[p]);
    } else {
#pragma unroll
      for (int p = 0; p < L::kWPieces; ++p) async_copy_16(dst + L::kWOff + p * 1024, wb, w_voff[p]);
    }
    const uint8_t* const ab = a_base + static_cast<size_t>(s) * 128;
#pragma unroll
    for (int p = 0; p < L::kRows / 8; ++p) {
      if (p == 0 || p < row_copies) async_copy_16(dst + p * 1024, ab, a_voff[p]);
    }
  };
  // the slice after which `later` (0 .. DEPTH - 1) slices have been requested has landed
  auto wait = [&](int later) __attribute__((always_inline)) {
    if constexpr (MT >= 3) {
      if (row_copies >= 6) return wait_slices<DEPTH - 1, L::kWOps + 6>(later);
      if (row_copies == 5) return wait_slices<DEPTH - 1, L::kWOps + 5>(later);
    }
    if constexpr (MT >= 2) {
      if (row_copies >= 4) return wait_slices<DEPTH - 1, L::kWOps + 4>(later);
      if (row_copies == 3) return wait_slices<DEPTH - 1, L::kWOps + 3>(later);
    }
    if (row_copies >= 2) return wait_slices<DEPTH - 1, L::kWOps + 2>(later);
    wait_slices<DEPTH - 1, L::kWOps + 1>(later);
  };

  // The first requests, before anything that they do not need (with the division gone: M = 12, N = 1024, K = 1088 3.34 -> 3.24 us,
  // M = 24, N = K = 2048 4.60 -> 4.53, M = 48, N = 11008 13.06 -> 12.79; M = 64 and 128, N = 4096, and wide layers level).
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    if (d < mine) request(slice_of(d), d);
  }

  // ---- LDS addresses of this lane's reads ----
  uint32_t a_rd[kSteps];
#pragma unroll
  for (int j = 0; j < kSteps; ++j) a_rd[j] = slots + i * 128 + (((4 * unit + word0 + j) ^ ((i >> 1) & 7)) * 16);
  const uint32_t w_rd = slots + L::kWOff + unit * 512 + i * 16 + word0 * 4;
  const int block = (BS == 64) ? 0 : (BS == 32) ? unit : 2 * unit + (F == 32 ? 0 : g >> 1);
  const uint32_t s_rd = slots + L::kSOff + (ROW ? (2 * unit + (g >> 1)) * 32 : (block * L::kCols + i) * 2);
  const uint32_t z_rd = slots + L::kZOff + (ROW ? (2 * unit + (g >> 1)) * 16 : block * L::kCols + i);

  const DequantMasks masks = DequantMasks::make();
  const RowMetaMasks rmasks = ROW ? RowMetaMasks::make() : RowMetaMasks{};
  acc_t acc[L::kFrags][L::kRowFrags];
#pragma unroll
  for (int t = 0; t < L::kFrags; ++t)
#pragma unroll
    for (int mt = 0; mt < L::kRowFrags; ++mt) acc[t][mt] = acc_t(0.f);

  auto step = [&](int li, auto slot_tag) __attribute__((always_inline)) {
    constexpr int slot = decltype(slot_tag)::value;
    constexpr int off = slot * L::kSlotBytes;
    wait(mine - 1 - li);
    uint4 af[L::kRowFrags][kSteps];
    uint32_t words[L::kFrags][kSteps];
    uint32_t sc[L::kFrags][kMeta], zp[L::kFrags][kMeta];
    uint4 rs[L::kGroups][2] = {}, rz[L::kGroups] = {};  // blocks along N: 16 scales and zero-points in the packed order
#pragma unroll
    for (int t = 0; t < L::kFrags; ++t) {
      if constexpr (F == 32) {
        const uint4 v = lds_read_16(w_rd, off + t * 1024);
        words[t][0] = v.x;
        words[t][1] = v.y;
        words[t][2] = v.z;
        words[t][3] = v.w;
      } else {
        const uint2 v = lds_read_8(w_rd, off + (t >> 1) * 1024 + (t & 1) * 256);
        words[t][0] = v.x;
        words[t][1] = v.y;
      }
      if constexpr (!ROW) {
#pragma unroll
        for (int b = 0; b < kMeta; ++b) {
          sc[t][b] = lds_read_u16(s_rd, off + (b * L::kCols + t * F) * 2);
          zp[t][b] = HAS_ZP ? lds_read_u8(z_rd, off + b * L::kCols + t * F) : 8u;
        }
      }
    }
    if constexpr (ROW) {
#pragma unroll
      for (int b = 0; b < L::kGroups; ++b) {
        rs[b][0] = lds_read_16(s_rd, off + b * 128);
        rs[b][1] = lds_read_16(s_rd, off + b * 128 + 16);
        if (HAS_ZP) rz[b] = lds_read_16(z_rd, off + b * 64);
      }
    }
#pragma unroll
    for (int j = 0; j < kSteps; ++j)
#pragma unroll
      for (int mt = 0; mt < L::kRowFrags; ++mt) af[mt][j] = lds_read_16(a_rd[j], off + mt * F * 128);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot has been read
    if (li + DEPTH < mine) request(slice_of(li + DEPTH), slot);

    DequantConsts dc[kMeta];
    Bf16Consts bc[kMeta];
    auto convert = [&](const int t, const int j) -> half8_t {
      const uint32_t word = words[t][j], y = word >> 8;
      if constexpr (ROW) {
        // word word0 + j is rows 8 j .. 8 j + 7 of the lane's 16-row group; the fragments of a column group share what is
        // built from its zero-points
        const int b = t * F / BS;
        half2_t p[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t src = (e >= 2) ? y : word;
          const half2_t d = (((e & 1) == 0) ? as_half2((src & masks.lo_mask) | masks.magic_1024)
                                            : as_half2((src & masks.hi_mask) | masks.magic_64)) +
                            row_neg_c<HAS_ZP>(vec_word(rz[b], e), e, j, rmasks);
          const uint32_t pair = vec_word(rs[b][(2 * e + j) >> 2], (2 * e + j) & 3);
          if constexpr (kBF) p[e] = as_half2(row_pair_bf16(d, pair));
          else p[e] = d * as_half2(pair);
        }
        return half8_t{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
      } else {
        if (j == 0) {
#pragma unroll
          for (int b = 0; b < kMeta; ++b) {
            if constexpr (kBF) bc[b] = make_bf16_consts(sc[t][b], zp[t][b]);
            else dc[b] = make_dequant_consts(sc[t][b], zp[t][b]);
          }
        }
        const int b = (kMeta == 2) ? (j >> 1) : 0;
        if constexpr (kBF) {
          return __builtin_bit_cast(half8_t, dequant_word_bf16(word, bc[b], masks));
        } else {
          const half2_t p0 = dequant_pair(word, 0, dc[b], masks), p1 = dequant_pair(word, 1, dc[b], masks);
          const half2_t p2 = dequant_pair(y, 2, dc[b], masks), p3 = dequant_pair(y, 3, dc[b], masks);
          return half8_t{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
        }
      }
    };
    // the next word is converted before this one's MFMAs are issued: an MFMA right behind the instruction that makes its
    // operand would wait for it
    half8_t wf = convert(0, 0);
#pragma unroll
    for (int y = 0; y < kSteps * L::kFrags; ++y) {
      const int t = y / kSteps, j = y % kSteps;
      half8_t next = wf;
      if (y + 1 < kSteps * L::kFrags) next = convert((y + 1) / kSteps, (y + 1) % kSteps);
      BLKQ4_PIN();
#pragma unroll
      for (int mt = 0; mt < L::kRowFrags; ++mt) {
        const half8_t a = as_half8(af[mt][j]);
        if constexpr (F == 16 && kBF) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf), __builtin_bit_cast(bf16x8_t, a), acc[t][mt], 0, 0, 0);
        else if constexpr (F == 16) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf, a, acc[t][mt], 0, 0, 0);
        else if constexpr (kBF) acc[t][mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wf), __builtin_bit_cast(bf16x8_t, a), acc[t][mt], 0, 0, 0);
        else acc[t][mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf, a, acc[t][mt], 0, 0, 0);
      }
      wf = next;
    }
  };

  for (int li = 0; li < mine; li += DEPTH) {
    step(li, std::integral_constant<int, 0>{});
    if (li + 1 < mine) step(li + 1, std::integral_constant<int, 1>{});
    if constexpr (DEPTH == 4) {
      if (li + 2 < mine) step(li + 2, std::integral_constant<int, 2>{});
      if (li + 3 < mine) step(li + 3, std::integral_constant<int, 3>{});
    }
  }
  static_assert(DEPTH == 2 || DEPTH == 4, "unrolled by hand for these depths");

  // ---- the waves' partial tiles, [wave][row][16 * NT columns + 4 of padding] floats, where the slots were ----
  __syncthreads();
  const uint32_t wr = lds0 + wave * L::kPartBytes + (i * L::kRowWords + 4 * g) * 4;
#pragma unroll
  for (int t = 0; t < L::kFrags; ++t)
#pragma unroll
    for (int mt = 0; mt < L::kRowFrags; ++mt)
#pragma unroll
      for (int b = 0; b < (F == 16 ? 1 : 4); ++b) {
        // elements 4 b .. 4 b + 3: row i, columns 4 g .. + 3 (F = 16) or 8 b + 4 g .. + 3 (F = 32)
        const float e0 = acc[t][mt][4 * b], e1 = acc[t][mt][4 * b + 1], e2 = acc[t][mt][4 * b + 2], e3 = acc[t][mt][4 * b + 3];
        lds_write_16(wr, (mt * F * L::kRowWords + t * F + 8 * b) * 4, __float_as_uint(e0), __float_as_uint(e1),
                     __float_as_uint(e2), __float_as_uint(e3));
      }
  __syncthreads();
  constexpr int kChunks = L::kCols / 4;  // four columns of a row each
  for (int v = tid; v < M * kChunks; v += 64 * kWaves) {
    const int row = v / kChunks, col = c0 + (v % kChunks) * 4;
    const uint32_t rd = lds0 + (row * L::kRowWords + (v % kChunks) * 4) * 4;
    float sum[4];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const uint4 p = lds_read_16(rd, w * L::kPartBytes);
      const float f[4] = {__uint_as_float(p.x), __uint_as_float(p.y), __uint_as_float(p.z), __uint_as_float(p.w)};
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] = (w == 0) ? f[e] : sum[e] + f[e];
    }
    if (col < N) {
      uint32_t lo = float_to_bits<kBF>(sum[0]) | (float_to_bits<kBF>(sum[1]) << 16);
      uint32_t hi = float_to_bits<kBF>(sum[2]) | (float_to_bits<kBF>(sum[3]) << 16);
      if (bias != nullptr) {
        const uint2 b = *reinterpret_cast<const uint2*>(bias + col);
        lo = add_bias_pair_t<kBF>(lo, b.x);
        hi = add_bias_pair_t<kBF>(hi, b.y);
      }
      *reinterpret_cast<uint2*>(C + static_cast<size_t>(m0 + row) * N + col) = make_uint2(lo, hi);
    }
  }
}

// One instantiation with the launch geometry of the plan; what the kernel assumes about it is checked here.
template <int BS, bool HAS_ZP, bool ROW, int DEPTH, int NT, int MT, int kWaves>
int launch_kernel(const blkq4_gemm_args* a) {
  using L = Layout<BS, HAS_ZP, NT, MT, kWaves, DEPTH, ROW>;
  const blkq4_streaming_plan& p = a->streaming;
  if (a->launched_id != nullptr) *a->launched_id = streaming_id(DEPTH, NT, MT, kWaves, kRowsPerSlotInLds, kWaves, false);
  const int col_groups = (a->n + L::kCols - 1) / L::kCols;
  const int deal = 8 * streaming_neighbours(NT, kWaves, kWaves);  // column groups dealt to the XCDs at a time
  const int rows_per_group = staged_rows_per_group(a->m, p.row_groups);
  if (p.row_groups < 1 || rows_per_group > L::kRows || rows_per_group * p.row_groups < a->m || p.refill != 0 ||
      p.cg_stride < col_groups || (p.cg_stride % deal) != 0 ||
      p.grid != static_cast<uint32_t>(p.cg_stride) * static_cast<uint32_t>(p.row_groups)) {
    return static_cast<int>(hipErrorInvalidValue);
  }
  // q / row_groups = (q * inv) >> 32 with inv = floor(2^32 / row_groups) + 1 (unused with one row group): exact while q *
  // row_groups < 2^32 (inv * row_groups is at most row_groups over 2^32), q below the workgroups of an XCD.  At most 32 row
  // groups of weights below 4 GiB, K from 64 on, come to 2^30.
  const uint64_t groups = static_cast<uint32_t>(p.row_groups);
  if ((p.grid >> 3) * groups >= (uint64_t{1} << 32)) return static_cast<int>(hipErrorInvalidValue);
  const uint32_t row_groups_inv = static_cast<uint32_t>((uint64_t{1} << 32) / groups + 1);
  if (a->dry_run) return 0;  // the plan has passed every check a launch makes
  constexpr auto kernel = staged_mfma_kernel<BS, HAS_ZP, NT, MT, kWaves, DEPTH, ROW>;
  const hipError_t attr = raise_lds_limit_once(reinterpret_cast<const void*>(kernel), kMaxLdsBytes, &lds_limit_flags<kernel>());
  if (attr != hipSuccess) return static_cast<int>(attr);
  // the launch's own status: a sticky error of an earlier, unrelated call stays where it is
  return static_cast<int>(launch_status(kernel, dim3(p.grid), dim3(64 * kWaves), L::kLdsBytes, a->stream,
                                        static_cast<const uint8_t*>(a->a), static_cast<const uint8_t*>(a->packed_w),
                                        static_cast<const uint8_t*>(a->scales),
                                        static_cast<const uint8_t*>(a->zero_points), a->m, a->n, a->k, p.row_groups,
                                        rows_per_group, row_groups_inv,
                                        static_cast<uint16_t*>(a->c), static_cast<const uint16_t*>(a->bias)));
}

// The shapes that exist, (DEPTH, NT, MT, waves), where staged_shape_exists(): what blkq4::choose() may ask for.
#define BLKQ4_STAGED_SHAPES(X)                                                 \
  /* row groups of 32 */                                                       \
  X(2, 1, 2, 8) X(2, 2, 2, 8) X(2, 4, 2, 8) X(2, 6, 2, 8) X(2, 8, 2, 8)        \
  /* row groups of 48 */                                                       \
  X(2, 1, 3, 8) X(2, 2, 3, 8) X(2, 3, 3, 8) X(2, 4, 3, 8) X(2, 5, 3, 8)        \
  /* up to 16 rows: wide layers, long K */                                     \
  X(2, 4, 1, 4) X(2, 5, 1, 4) X(2, 6, 1, 4) X(2, 7, 1, 4)                      \
  X(2, 4, 1, 8) X(2, 5, 1, 8) X(2, 6, 1, 8) X(2, 7, 1, 8)                      \
  X(4, 1, 1, 8) X(4, 2, 1, 8) X(4, 3, 1, 8) X(2, 1, 1, 16) X(2, 2, 1, 16) X(2, 3, 1, 16)

template <int BS, bool HAS_ZP, bool ROW>
int launch_plan(const blkq4_gemm_args* a) {
  const blkq4_streaming_plan& p = a->streaming;
  if (p.am != kRowsPerSlotInLds || p.split != p.waves) return static_cast<int>(hipErrorInvalidValue);
#define BLKQ4_TRY(D_, NT_, MT_, W_)                                             \
  if (p.depth == D_ && p.nt == NT_ && p.mt == MT_ && p.waves == W_) {           \
    if constexpr (staged_shape_exists(ROW, BS, HAS_ZP, NT_, MT_, W_, D_)) {     \
      return launch_kernel<BS, HAS_ZP, ROW, D_, NT_, MT_, W_>(a);               \
    } else {                                                                    \
      return static_cast<int>(hipErrorInvalidValue);                            \
    }                                                                           \
  }
  BLKQ4_STAGED_SHAPES(BLKQ4_TRY)
#undef BLKQ4_TRY
  return static_cast<int>(hipErrorInvalidValue);  // a shape that does not exist
}

template <int BS>
int launch_bs(const blkq4_gemm_args* a) {
  if (a->column_wise) return a->zero_points ? launch_plan<BS, true, false>(a) : launch_plan<BS, false, false>(a);
  return a->zero_points ? launch_plan<BS, true, true>(a) : launch_plan<BS, false, true>(a);
}

}  // namespace

extern "C" int BLKQ4_STAGED_ENTRY(const blkq4_gemm_args* a) {
  if (a->m < 1 || a->m > kStreamingMaxRows || (a->n % 32) != 0 || (a->k % 64) != 0) return static_cast<int>(hipErrorInvalidValue);
  // a wave's offsets inside a slice are 32 bits wide, as are the streaming kernel's over the whole matrix
  if (static_cast<uint64_t>(a->k) * static_cast<uint64_t>(a->n) >= kStreamingMaxWeights) return static_cast<int>(hipErrorInvalidValue);
  // scales and zero-points are copied four bytes at a time, the output is stored eight bytes at a time
  if ((reinterpret_cast<uintptr_t>(a->scales) & 3u) != 0 || (reinterpret_cast<uintptr_t>(a->zero_points) & 3u) != 0 ||
      (reinterpret_cast<uintptr_t>(a->c) & 7u) != 0 || (reinterpret_cast<uintptr_t>(a->bias) & 7u) != 0) {
    return static_cast<int>(hipErrorInvalidValue);
  }
  if (!a->column_wise && (a->n % a->block_size) != 0) return static_cast<int>(hipErrorInvalidValue);
  switch (a->block_size) {
    case 16: return launch_bs<16>(a);
    case 32: return launch_bs<32>(a);
    case 64: return launch_bs<64>(a);
    default: return static_cast<int>(hipErrorInvalidValue);
  }
}
