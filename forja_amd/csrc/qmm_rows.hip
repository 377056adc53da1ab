// MLX affine quantised products over a middling number of activation rows per weight: dense decode
// batches of more rows (or longer K) than the K-split kernels hold in registers, f32 activations
// of prompt chunks, and the routed products of a batch with tens of routes per expert.  Same
// arithmetic as qmm_ksplit.hip: a weight operand is exact, a 64-value group is contracted in f32 on the
// matrix cores and scaled once,
//   y[m,n] = sum_g scale[n,g] * (sum_{k in g} x[m,k] * (q - c)[n,k]) + (bias + c * scale)[n,g] * sum_{k in g} x[m,k]
// (affine_quant_dot, crates/forja-cpu/src/lib.rs:1277-1310).  bf16 rows meet 16 + q in bf16 (c = -16);
// f32 rows, brought into f16's range by a power of two per row and group, go in as three f16 pieces of
// eleven bits that make up each value (to 2^-38 of the group's largest), against q - 8 (4 bits) or q - 128 (8 bits) in f16: centred,
// because what 16 + q adds to a group's sum only to be taken off again costs f32 results their last
// bits.  Error of 512 x 512 x 2048 on f32 N(0,1) rows against 64 bits (2-norm): 1.0e-7, on rows of mean 1
// 2.7e-7 (the vector-ALU kernels, value by value: 2.9e-7 both; bf16 pieces against 16 + q: 5.2e-7, 2.5e-6).
//
// No one unit bounds such a product (48 x 34816 x 5120, counters: while two waves share a SIMD, its vector ALU is
// busy 0.57 of the cycles and its matrix cores 0.26, and a wave issues for 0.41 of its life, is ready but not issued for
// 0.40 and waits for the rest).  A weight is used for 16 to 64 rows, so its unpacking (8
// instructions a word) and its share of activation traffic have to be spread over all of them.  A wave therefore owns 64 weight columns and every row of the tile: the weights go
// straight from memory to the wave's registers, 16 rows x 64 bytes per load, a pair of groups ahead of
// the arithmetic, and are unpacked once; the activations, which the column waves of a workgroup share,
// are staged through LDS in operand order (one ds_read_b128 per operand, few bank conflicts),
// split and summed per group on the way in.  K is divided over WK waves of a workgroup and, where the
// output has too few tiles for the device, over workgroups whose f32 partial sums a second launch
// adds in order.
// Measured, before (streaming, tile-product and vector-ALU kernels) and now: bf16 48 x 34816 x 5120 101 ->
// 56 us, 48 x 5120 x 17408 75 -> 30; f32 512 x 5120 x 2048 284 -> 52, 512 x 2048 x 4096 231 -> 42, 8 bits 512 x 128 x 2048
// 93 -> 12; routed, 128 experts of 768 x 2048, gate/up and down together: bf16 16640 routes 435 -> 294, f32 4096 routes
// 1027 -> 232 (in steps, where their weights come from memory).
//
// The activations come in by rows, eight lanes to a row's 128 bytes of a group: sixteen bytes of another row in every lane
// (operand order) cost the compute unit's address unit 65 cycles a load against 18, and a third of all loads were of
// that kind; the chunks find their operand places on the way into LDS, and a group's sum is three exchanges within eight
// lanes.  A lane quarter reads the scales and biases of one column tile for all four, by global loads: through pointers
// that may point to LDS every wait for LDS waited for them and for all loads before (48 x 34816 x 5120 57.7 us for 56.1,
// 8 bits 512 x 128 x 2048 13.5 for 12.3).  Against operand-order loads by every quarter: bf16 48 x 34816 x 5120 63 -> 56 us,
// 48 x 151936 x 5120 183 -> 164, 64 x 34816 x 5120 75 -> 70, 20 x 34816 x 5120 49 -> 47; f32 512 x 5120 x 2048 57 -> 52, 8 bits
// 512 x 128 x 2048 12.7 -> 12.3 (back to back, weights from memory).
//
// The bias term rides on the matrix cores too: the group sums are split into their three exact
// bf16 pieces, one per lane quarter, and the operand against them is the column's scales and
// biases as they lie in memory (both exact in bf16), so that one instruction per 16 x 16 block and
// four groups does the whole term.
#include <type_traits>

#include "fast_kernels.hpp"

namespace fh {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

constexpr uint32_t kGroup = 64, kQuad = 4 * kGroup;   // K advances by four groups: whole 128-byte lines of 4-bit weights
constexpr uint32_t kNoBlock = 0xffffffffu;
constexpr int kColTiles = 4;                          // 16-column tiles of a wave (both projections of a pair together)

struct RowsArgs {
  const void *x;            // bf16 or f32 rows, innermost axis contiguous
  uint64_t x_row_stride;    // elements
  const uint32_t *packed[2];
  const uint16_t *scales[2], *biases[2];
  uint64_t expert_words, expert_groups;   // per expert matrix; 0 for dense
  void *out;                // bf16 or f32; the partial sums [splits][rows][columns] when splits > 1
  uint64_t out_row_stride;
  uint32_t out_f32, out_aligned;   // out_aligned: four results of a row make one aligned store
  const void *residual;     // dense, splits == 1: rows of the activations' dtype
  uint64_t residual_row_stride;
  uint32_t rows, inner, columns;
  uint32_t col_blocks, row_blocks, splits;
  const uint32_t *sorted_routes, *blocks, *n_blocks;   // routed: tiles (expert, first, count)
  uint32_t route_div;
};

__device__ inline float low_bf16(uint32_t word) { return __uint_as_float(word << 16); }
__device__ inline float high_bf16(uint32_t word) { return __uint_as_float(word & 0xffff0000u); }

__device__ inline uint32_t pack_bf16(float lo, float hi) {
  bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// Eight nibbles as bf16 (16 + q), slot order (0,4)(1,5)(2,6)(3,7); see qmm_ksplit.hip.
__device__ inline bf16x8 unpack_nibbles(uint32_t w) {
  uint32_t mask = 0x00780078u, magic = 0x41804180u;
  asm("" : "+s"(mask), "+v"(magic));   // no instruction: keeps the two constants in registers
  uint4 r;
  r.x = ((w << 3) & mask) | magic;
  r.y = ((w >> 1) & mask) | magic;
  r.z = ((w >> 5) & mask) | magic;
  r.w = ((w >> 9) & mask) | magic;
  return __builtin_bit_cast(bf16x8, r);
}

// Eight nibbles as f16 q - 8, the same slots: a nibble in the low mantissa bits of 1024 is 1024 + q, in
// the next four 1024 + 16 q; one packed instruction takes either to q - 8, exactly.
__device__ inline f16x8 unpack_nibbles_f16(uint32_t w) {
  uint32_t low = 0x000f000fu, high = 0x00f000f0u, magic = 0x64006400u;
  asm("" : "+s"(low), "+s"(high), "+v"(magic));
  const f16x2 minus_low = {(_Float16)-1032.0f, (_Float16)-1032.0f}, minus_high = {(_Float16)-72.0f, (_Float16)-72.0f};
  const f16x2 sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
  const uint32_t shifted = w >> 8;
  const f16x2 pairs[4] = {
      __builtin_bit_cast(f16x2, (w & low) | magic) + minus_low,
      __builtin_elementwise_fma(__builtin_bit_cast(f16x2, (w & high) | magic), sixteenth, minus_high),
      __builtin_bit_cast(f16x2, (shifted & low) | magic) + minus_low,
      __builtin_elementwise_fma(__builtin_bit_cast(f16x2, (shifted & high) | magic), sixteenth, minus_high)};
  return __builtin_shufflevector(__builtin_shufflevector(pairs[0], pairs[1], 0, 1, 2, 3),
                                 __builtin_shufflevector(pairs[2], pairs[3], 0, 1, 2, 3), 0, 1, 2, 3, 4, 5, 6, 7);
}

// Eight bytes as f16 q - 128, in order: a byte under the high byte of 1024 is 1024 + q.
__device__ inline f16x8 unpack_bytes_f16(uint32_t lo, uint32_t hi) {
  const f16x2 minus = {(_Float16)-1152.0f, (_Float16)-1152.0f};
  auto pair = [&](uint32_t w, uint32_t select) {
    return __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, w, select)) + minus;
  };
  return __builtin_shufflevector(__builtin_shufflevector(pair(lo, 0x04010400u), pair(lo, 0x04030402u), 0, 1, 2, 3),
                                 __builtin_shufflevector(pair(hi, 0x04010400u), pair(hi, 0x04030402u), 0, 1, 2, 3),
                                 0, 1, 2, 3, 4, 5, 6, 7);
}

__device__ inline uint4 permute_slots(const uint4 &v) {
  uint4 p;
  p.x = __builtin_amdgcn_perm(v.z, v.x, 0x05040100u);  // (x0, x4)
  p.y = __builtin_amdgcn_perm(v.z, v.x, 0x07060302u);  // (x1, x5)
  p.z = __builtin_amdgcn_perm(v.w, v.y, 0x05040100u);  // (x2, x6)
  p.w = __builtin_amdgcn_perm(v.w, v.y, 0x07060302u);  // (x3, x7)
  return p;
}

// The same pointer, kept in scalar registers: the lane's part of an address is then one 32-bit
// offset for all of a wave's loads.  (Left to itself the compiler adds the two once, outside the
// loop, and keeps a 64-bit vector address per load: a hundred registers here, which spill.)
typedef const __attribute__((address_space(1))) char *global_bytes;
__device__ inline global_bytes uniform(const char *base) {
  global_bytes p = (global_bytes)base;
  asm("" : "+s"(p));
  return p;
}
template <typename T>
__device__ inline T load_at(global_bytes base, uint32_t offset) {
  asm volatile("" : "+v"(offset));   // ... and the 32-bit offset must not be widened outside the loop either
  return *(const __attribute__((address_space(1))) T *)(base + offset);
}

// Bytes of LDS: the staged activations of a pair of groups and their sums, per K part, twice (so that
// one barrier per pair of groups is enough).  f32 rows: and the factor of each row and group.
template <int XP, int RT>
constexpr uint32_t part_bytes() { return XP * RT * 4 * 1024 + RT * 1024 + (XP == 1 ? 0 : RT * 128); }
template <int XP, int RT, int WK>
constexpr uint32_t staged_bytes() { return 2u * WK * part_bytes<XP, RT>(); }

// The value of another lane of the same eight: its neighbour, of the other pair of its four, of the other four (any of them:
// for sums that the four already share).
constexpr int kOther = 0xb1, kOtherPair = 0x4e, kOtherFour = 0x141;   // quad_perm 1,0,3,2 and 2,3,0,1; row_half_mirror
template <int kWay>
__device__ inline int across(int v) { return __builtin_amdgcn_update_dpp(0, v, kWay, 0xf, 0xf, true); }

// XP: pieces of an activation (1: bf16 rows as they are, 3: f32 rows in f16).  BITS: 4 or 8 (f32 rows only).  RT: 16-row tiles.
// WC waves side by side (64 columns each; of a pair 32 of either projection), WK waves along K.
template <int XP, int BITS, int RT, int WC, int WK, bool kPair, bool kRouted>
__global__ __launch_bounds__(64 * WC * WK, 2) void qmm_rows_kernel(RowsArgs a) {
  static_assert(!kRouted || WK == 1, "routed tiles are not split along K");
  constexpr int P = kPair ? 2 : 1, CT = kColTiles / P;
  constexpr uint32_t kBlockCols = 16u * CT * WC;
  constexpr int kTasks = RT * 2 / WC;            // (row tile, group) pieces a wave stages per pair of groups
  static_assert(kTasks * WC == RT * 2, "whole pieces per wave");
  constexpr int XW = XP == 1 ? 4 : 8;            // registers of eight activations
  constexpr uint32_t kFragments = XP * RT * 4;   // 1 KiB operands of a pair: [piece][row tile][group][half]
  constexpr uint32_t kPartBytes = part_bytes<XP, RT>();
  extern __shared__ __attribute__((aligned(16))) char staged[];   // [2][WK]{operands, sums}
  const uint32_t lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t wc = wave % WC, wk = wave / WC;

  // Workgroups are dealt round-robin to the eight XCDs.  Dense: those that share weights (row
  // blocks of the same columns) follow each other on one XCD; routed: an XCD takes a contiguous
  // run of tiles, so that the tiles of an expert and the column blocks of a tile meet in its L2.
  uint32_t tile_first, tile_count, col_block, split = 0;
  uint64_t expert = 0;
  const uint32_t xcd = blockIdx.x % 8, position = blockIdx.x / 8;
  if constexpr (kRouted) {
    const uint32_t tiles = __builtin_amdgcn_readfirstlane(a.n_blocks[0]), share = (tiles + 7) / 8;
    const uint32_t local = position / a.col_blocks, tile = xcd * share + local;
    if (local >= share || tile >= tiles) return;
    const uint32_t id = __builtin_amdgcn_readfirstlane(a.blocks[3 * tile]);
    if (id == kNoBlock) return;
    expert = id;
    tile_first = __builtin_amdgcn_readfirstlane(a.blocks[3 * tile + 1]);
    tile_count = __builtin_amdgcn_readfirstlane(a.blocks[3 * tile + 2]);
    col_block = position % a.col_blocks;
  } else {
    const uint32_t unit = position / a.row_blocks * 8 + xcd;
    if (unit >= a.col_blocks * a.splits) return;
    tile_first = position % a.row_blocks * (16 * RT);
    tile_count = min(16u * RT, a.rows - tile_first);
    col_block = unit % a.col_blocks;
    split = unit / a.col_blocks;
  }
  uint32_t *row_ids = (uint32_t *)(staged + staged_bytes<XP, RT, WK>());   // routed: the tile's output rows
  if (kRouted && threadIdx.x < 16 * RT) row_ids[threadIdx.x] = a.sorted_routes[tile_first + min(threadIdx.x, tile_count - 1)];
  const uint32_t quads = a.inner / kQuad;
  const uint32_t first_quad = split * quads / a.splits, last_quad = (split + 1) * quads / a.splits;
  const uint32_t rounds = (last_quad - first_quad + WK - 1) / WK;

  // ---- the activations this wave stages: for each of its pieces, lane (row e, chunk c) brings values [8c, 8c+8) of
  // rows e and 8 + e of one group: neighbouring lanes read neighbouring addresses.  (Sixteen bytes of another row
  // in every lane take the address unit 65 cycles a load, whole lines of a row 18.)
  const uint32_t chunk = lane & 7, e = lane >> 3;
  constexpr uint32_t kValue = XP == 1 ? 2 : 4;
  // Bytes.  Dense: one lane offset for every row, from a buffer that ends with the last row (past it zeros, never
  // stored); routed: each row's own.  (Tiles of 64 dense rows, too: there the buffers' scalars push nine registers out, 85
  // us against 76 for 64 x 34816 x 5120; of 48 rows the offsets do, 66 against 61 for 48 x 34816 x 5120.)
  constexpr bool kOwnOffsets = kRouted || RT == 4;
  uint32_t x_lane[kOwnOffsets ? kTasks : 1][2];
  const uint32_t x_bytes = (uint32_t)(((uint64_t)(a.rows - 1) * a.x_row_stride + a.inner) * kValue);
  if constexpr (kOwnOffsets) {
#pragma unroll
    for (int t = 0; t < kTasks; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t task = wc + t * WC, row = 16 * (task / 2) + 8 * i + e;
        const uint32_t safe = row < tile_count ? row : 0;     // rows past the tile: computed, never stored
        const uint64_t in_row = kRouted ? a.sorted_routes[tile_first + safe] / a.route_div : tile_first + safe;
        x_lane[t][i] = (uint32_t)(in_row * a.x_row_stride + kGroup * (task % 2) + 8 * chunk) * kValue;
      }
  } else {
    x_lane[0][0] = (uint32_t)(e * a.x_row_stride + 8 * chunk) * kValue;
  }
  uint32_t xr[kTasks][2][XW];
  auto load_rows = [&](uint32_t quad, int pair) {   // (a quad past the end reads the last one)
    const uint64_t at = (uint64_t)min(quad, quads - 1) * kQuad + 2 * kGroup * pair;
#pragma unroll
    for (int t = 0; t < kTasks; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        u32x4 eight[XW / 4];
        if constexpr (kOwnOffsets) {
          const global_bytes from = uniform((const char *)a.x + at * kValue);
#pragma unroll
          for (int v = 0; v < XW / 4; ++v) eight[v] = load_at<u32x4>(from, x_lane[t][i] + 16 * v);
        } else {
          const uint32_t task = wc + t * WC;
          const uint64_t skip = ((tile_first + 16 * (task / 2) + 8 * i) * a.x_row_stride + at + kGroup * (task % 2)) * kValue;
          const auto rows = __builtin_amdgcn_make_buffer_rsrc((char *)const_cast<void *>(a.x) + skip, 0,
                                                              (int)(skip < x_bytes ? x_bytes - (uint32_t)skip : 0u), 0x27000);
#pragma unroll
          for (int v = 0; v < XW / 4; ++v) eight[v] = __builtin_amdgcn_raw_buffer_load_b128(rows, (int)x_lane[0][0] + 16 * v, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < XW / 4; ++v) {
          const u32x4 four = eight[v];
          xr[t][i][4 * v] = four.x, xr[t][i][4 * v + 1] = four.y;
          xr[t][i][4 * v + 2] = four.z, xr[t][i][4 * v + 3] = four.w;
        }
      }
  };
  // Where a chunk of eight values lies in operand order: chunk c of a group belongs to quarter
  // c / 2 of the lanes and operand half c % 2; with 4-bit weights the half-wave swaps leave
  // quarter q of the lanes holding the nibbles of values [16 q', 16 q' + 16), q' = (0,2,1,3)[q].
  // A row's place within its quarter is turned by twice the quarter and half, so that the sixteen lanes of a store,
  // two rows of eight chunks, meet different banks.
  auto turn_of = [](uint32_t at, uint32_t half) { return 2 * (2 * at + half); };
  const uint32_t quarter = chunk / 2, at_quarter = BITS == 4 ? 2 * (quarter & 1) + (quarter >> 1) : quarter;
  const uint32_t slot0 = (chunk % 2) * 1024 + (16 * at_quarter + (e ^ turn_of(at_quarter, chunk % 2))) * 16;
  const uint32_t slot[2] = {slot0, slot0 ^ 128};   // rows e and 8 + e
  uint32_t sum_mask[3];
#pragma unroll
  for (int piece = 0; piece < 3; ++piece) {
    sum_mask[piece] = chunk % 4 == (uint32_t)piece ? 0xffffffffu : 0u;
    asm("" : "+v"(sum_mask[piece]));
  }
  // `parity`: which of the two sets of group sums (by quad)
  auto stage_rows = [&](uint32_t buffer, uint32_t parity, int pair) {
    char *part = staged + (buffer * WK + wk) * kPartBytes;
    char *sums = staged + (parity * WK + wk) * kPartBytes + kFragments * 1024;
#pragma unroll
    for (int t = 0; t < kTasks; ++t) {
      const uint32_t task = wc + t * WC, row_tile = task / 2, group = task % 2;
      float s[2] = {0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if constexpr (XP == 1) {
          const uint4 v = make_uint4(xr[t][i][0], xr[t][i][1], xr[t][i][2], xr[t][i][3]);
          const uint32_t words[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int w = 0; w < 4; ++w)
            s[i] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, words[w]), __builtin_bit_cast(bf16x2, 0x3f803f80u), s[i], false);
          *(uint4 *)(part + (row_tile * 4 + group * 2) * 1024 + slot[i]) = permute_slots(v);
        } else {
          // A power of two takes the largest of the row's group into [2^14, 2^15); then three f16
          // pieces, each the leading eleven bits of what the ones before left, make up every value to
          // 2^-38 of that largest: the smallest step of f16 is 2^-24 (pieces are cut off, not rounded, so that
          // the rest is exact).
          uint32_t largest = 0;
#pragma unroll
          for (int v = 0; v < 8; ++v) {
            s[i] += __uint_as_float(xr[t][i][v]);
            largest = max(largest, xr[t][i][v] & 0x7fffffffu);
          }
          largest = max(largest, (uint32_t)across<kOther>((int)largest));
          largest = max(largest, (uint32_t)across<kOtherPair>((int)largest));
          largest = max(largest, (uint32_t)across<kOtherFour>((int)largest));
          const uint32_t exponent = max(largest >> 23, 15u);
          const float up = __uint_as_float((268u - exponent) << 23);   // exponent - 127 + 14, undone: 141 - exponent + 127
          if (chunk == 0) ((float *)(part + kFragments * 1024 + RT * 1024))[group * 16 * RT + 16 * row_tile + 8 * i + e] = __uint_as_float((exponent - 14u) << 23);
          float value[8];
#pragma unroll
          for (int v = 0; v < 8; ++v) value[v] = __uint_as_float(xr[t][i][v]) * up;
#pragma unroll
          for (int piece = XP - 1; piece >= 0; --piece) {   // piece 0 holds the low bits, added first
            uint4 packed;
            uint32_t *words = (uint32_t *)&packed;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const auto two = __builtin_amdgcn_cvt_pkrtz(value[2 * v], value[2 * v + 1]);
              value[2 * v] -= (float)two[0];
              value[2 * v + 1] -= (float)two[1];
              words[v] = __builtin_bit_cast(uint32_t, two);
            }
            *(uint4 *)(part + ((piece * RT + row_tile) * 4 + group * 2) * 1024 + slot[i]) =
                BITS == 4 ? permute_slots(packed) : packed;
          }
        }
        // the eight chunks of the row's group
        s[i] += __int_as_float(across<kOther>(__float_as_int(s[i])));
        s[i] += __int_as_float(across<kOtherPair>(__float_as_int(s[i])));
        s[i] += __int_as_float(across<kOtherFour>(__float_as_int(s[i])));
      }
      // Chunks 0..3 store the four pieces of row e's sum (high, middle, low, nothing), 4..7 those of row 8 + e: slots
      // 0..3 of a lane quarter's operand stand against the quad's four scales, 4..7 against its biases.
      const float sum = chunk < 4 ? s[0] : s[1];
      const float high = __uint_as_float(__float_as_uint(sum) & 0xffff0000u);
      const float rest = sum - high, middle = __uint_as_float(__float_as_uint(rest) & 0xffff0000u);
      const float low = rest - middle;
      // (by masks: written as a choice it becomes branches, which the contraction would be split by)
      const float mine = __uint_as_float((__float_as_uint(high) & sum_mask[0]) | (__float_as_uint(middle) & sum_mask[1]) |
                                         (__float_as_uint(low) & sum_mask[2]));
      const float offset = (XP == 1 ? -16.0f : BITS == 4 ? 8.0f : 128.0f) * mine;
      uint16_t *to = (uint16_t *)(sums + row_tile * 1024 + (16 * (chunk % 4) + 8 * (chunk / 4) + e) * 16) + 2 * pair + group;
      to[0] = (uint16_t)(__float_as_uint(offset) >> 16);
      to[4] = (uint16_t)(__float_as_uint(mine) >> 16);
    }
  };

  // ---- the weights: lane (column n, quarter g) reads 16 bytes of a pair of groups (4 bits) or of
  // each group (8 bits) of each of the wave's columns.
  const uint32_t words_per_row = a.inner / (32 / BITS), groups_per_row = a.inner / kGroup;
  constexpr int LPP = BITS / 4;                  // loads per pair of groups and column tile
  // The tile's base address is uniform and stays in scalar registers (a tile past the last column
  // reads the last one); one offset per lane serves every tile.
  const char *w_from[kColTiles];
  const uint32_t w_lane = (n * words_per_row + 4 * g) * 4;
#pragma unroll
  for (int tp = 0; tp < kColTiles; ++tp) {
    const int pj = tp / CT, ct = tp % CT;
    const uint32_t column = min(col_block * kBlockCols + (wc * CT + ct) * 16, a.columns - 16);
    w_from[tp] = (const char *)(a.packed[pj] + expert * a.expert_words + (uint64_t)column * words_per_row);
  }
  // Scales and biases: lane (n, g) reads those of column n of tile g, one load for the four tiles.
  global_bytes s_from, b_from;
  {
    const uint32_t column = min(col_block * kBlockCols + (wc * CT + g % CT) * 16, a.columns - 16) + n;
    const uint64_t at = expert * a.expert_groups + (uint64_t)column * groups_per_row;
    // (uniform: chosen from registers, not loaded by lane; and known to be global: a load from a pointer that may
    // point to LDS waits for, and is waited for with, every access to LDS)
    const global_bytes s0 = uniform((const char *)a.scales[0]), s1 = uniform((const char *)a.scales[P - 1]);
    const global_bytes b0 = uniform((const char *)a.biases[0]), b1 = uniform((const char *)a.biases[P - 1]);
    s_from = (g / CT ? s1 : s0) + 2 * at;
    b_from = (g / CT ? b1 : b0) + 2 * at;
  }
  // Requested ahead: the weights one pair of groups, the scales one quad, the biases from the
  // start of their quad to its end.
  u32x4 w[kColTiles][LPP];
  u32x2 scale4[kColTiles], next_scales, biases;
  auto load_weights = [&](uint32_t quad, int pair) {
    const uint32_t at = (min(quad, quads - 1) * 2 + pair) * (LPP * 64);
#pragma unroll
    for (int tp = 0; tp < kColTiles; ++tp)
#pragma unroll
      for (int l = 0; l < LPP; ++l) w[tp][l] = load_at<u32x4>(uniform(w_from[tp] + at), w_lane + 64 * l);
  };
  auto load_params = [&](global_bytes from, uint32_t quad) {
    return *(const __attribute__((address_space(1))) u32x2 *)(from + min(quad, quads - 1) * 8);
  };
  // Tile t's values from lane quarter t to all four quarters.
  auto spread = [](uint32_t v, uint32_t (&to)[kColTiles]) {
    const auto even_odd = __builtin_amdgcn_permlane16_swap(v, v, false, false);   // quarters 0 0 2 2 and 1 1 3 3
    const uint32_t even = even_odd[0], odd = even_odd[1];
    const auto low = __builtin_amdgcn_permlane32_swap(even, even, false, false);
    const auto high = __builtin_amdgcn_permlane32_swap(odd, odd, false, false);
    to[0] = low[0], to[1] = high[0], to[2] = low[1], to[3] = high[1];
  };
  static_assert(kColTiles == 4, "a tile for each quarter of the lanes");

  f32x4 acc[kColTiles][RT];
#pragma unroll
  for (int tp = 0; tp < kColTiles; ++tp)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[tp][rt] = f32x4{0.f, 0.f, 0.f, 0.f};

  using Operand = typename std::conditional<XP == 1, bf16x8, f16x8>::type;
  auto multiply = [](const Operand &rows, const Operand &weights, const f32x4 &sum) {
    if constexpr (XP == 1)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(rows, weights, sum, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(rows, weights, sum, 0, 0, 0);
  };
  const uint32_t read_slot[2] = {(16 * g + (n ^ turn_of(g, 0))) * 16, (16 * g + (n ^ turn_of(g, 1))) * 16};
  auto contract = [&](uint32_t buffer, int pair, uint32_t next_quad) {
    const char *part = staged + (buffer * WK + wk) * kPartBytes;
    const char *factors = staged + (buffer * WK + wk) * kPartBytes + kFragments * 1024 + RT * 1024 + 16 * g;   // rows 4g..4g+3
    u32x2 first[kColTiles], second[kColTiles];
    if constexpr (BITS == 4) {
#pragma unroll
      for (int tp = 0; tp < kColTiles; ++tp) {
        const u32x4 v = w[tp][0];
        first[tp] = __builtin_amdgcn_permlane32_swap(v.x, v.z, false, false);
        second[tp] = __builtin_amdgcn_permlane32_swap(v.y, v.w, false, false);
      }
      load_weights(next_quad, pair ^ 1);
    }
    constexpr int kAhead = XP == 1 ? 1 : 0;   // row tiles whose operands are read ahead of their use (registers)
    Operand rows[2][XP][2];
    auto read_rows = [&](int unit) {
#pragma unroll
      for (int piece = 0; piece < XP; ++piece)
#pragma unroll
        for (int half = 0; half < 2; ++half)
          rows[unit % 2][piece][half] = *(const Operand *)(part + read_slot[half] + ((piece * RT + unit % RT) * 4 + unit / RT * 2 + half) * 1024);
    };
    if (kAhead) read_rows(0);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      Operand b[kColTiles][2];
      float scale[kColTiles];
#pragma unroll
      for (int tp = 0; tp < kColTiles; ++tp) {
        if constexpr (BITS == 4) {
          if constexpr (XP == 1) {
            b[tp][0] = unpack_nibbles(first[tp][j]);
            b[tp][1] = unpack_nibbles(second[tp][j]);
          } else {
            b[tp][0] = unpack_nibbles_f16(first[tp][j]);
            b[tp][1] = unpack_nibbles_f16(second[tp][j]);
          }
        } else {
          const u32x4 v = w[tp][j % LPP];
          b[tp][0] = unpack_bytes_f16(v.x, v.y);
          b[tp][1] = unpack_bytes_f16(v.z, v.w);
        }
        const uint32_t word = pair ? scale4[tp].y : scale4[tp].x;
        scale[tp] = j ? high_bf16(word) : low_bf16(word);
      }
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const int unit = j * RT + rt;
        if (unit + kAhead < 2 * RT) read_rows(unit + kAhead);
        f32x4 sum[kColTiles];
#pragma unroll
        for (int tp = 0; tp < kColTiles; ++tp) sum[tp] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int piece = 0; piece < XP; ++piece)
#pragma unroll
          for (int half = 0; half < 2; ++half) {
#pragma unroll
            for (int tp = 0; tp < kColTiles; ++tp)
              sum[tp] = multiply(rows[unit % 2][piece][half], b[tp][half], sum[tp]);
          }
        f32x4 factor = {1.0f, 1.0f, 1.0f, 1.0f};
        if constexpr (XP > 1) factor = *(const f32x4 *)(factors + (j * 16 * RT + 16 * rt) * 4);
#pragma unroll
        for (int tp = 0; tp < kColTiles; ++tp)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float by = XP == 1 ? scale[tp] : scale[tp] * factor[i];
            acc[tp][rt][i] = __builtin_fmaf(by, sum[tp][i], acc[tp][rt][i]);
          }
        // No instruction: the group's sums are used up here.  (Free to choose, the compiler keeps all of
        // them and does the scaling where the round ends, in registers that it does not have.)
#pragma unroll
        for (int tp = 0; tp < kColTiles; ++tp) asm volatile("" : "+v"(acc[tp][rt]));
      }
    }
  };
  auto add_bias = [&](uint32_t parity, uint32_t keep) {
    const char *sums = staged + (parity * WK + wk) * kPartBytes + kFragments * 1024 + lane * 16;
    uint32_t bias_x[kColTiles], bias_y[kColTiles];
    spread(biases.x & keep, bias_x);
    spread(biases.y & keep, bias_y);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const bf16x8 rows = *(const bf16x8 *)(sums + rt * 1024);
#pragma unroll
      for (int tp = 0; tp < kColTiles; ++tp) {
        const uint4 params = make_uint4(scale4[tp].x, scale4[tp].y, bias_x[tp], bias_y[tp]);
        acc[tp][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rows, __builtin_bit_cast(bf16x8, params), acc[tp][rt], 0, 0, 0);
      }
    }
  };

  const uint32_t my_first = first_quad + wk;
  load_rows(my_first, 0);
  next_scales = load_params(s_from, my_first);
  load_weights(my_first, 0);
  uint32_t buffer = 0;
  for (uint32_t round = 0; round < rounds; ++round) {
    const uint32_t quad = my_first + round * WK;
    const uint32_t parity = round & 1;
    biases = load_params(b_from, quad);   // (requested before the scales are waited for)
    // A wave whose part of the range is a quad short contracts a quad of another range with all
    // scales and biases zero: under a branch its loads would be waited for where the paths meet.
    const uint32_t keep = WK == 1 || quad < last_quad ? 0xffffffffu : 0u;
    {
      uint32_t x[kColTiles], y[kColTiles];
      spread(next_scales.x & keep, x);
      spread(next_scales.y & keep, y);
#pragma unroll
      for (int tp = 0; tp < kColTiles; ++tp) scale4[tp] = u32x2{x[tp], y[tp]};
    }
    next_scales = load_params(s_from, quad + WK);
#pragma unroll
    for (int pair = 0; pair < 2; ++pair) {
      stage_rows(buffer, parity, pair);
      load_rows(pair ? quad + WK : quad, pair ^ 1);
      __syncthreads();
      contract(buffer, pair, pair ? quad + WK : quad);
      if (pair == 1) add_bias(parity, keep);
      if (BITS == 8) load_weights(pair ? quad + WK : quad, pair ^ 1);
      buffer ^= 1;
    }
  }

  // ---- results: lane (column n, quarter g) holds rows 4g..4g+3 of each 16 x 16 block.  Through LDS
  // they are turned into pieces of four columns of a row per lane (whole lines per store, one short
  // loop of code), and the K parts meet there, added in order, each part finishing its share of the rows.
  constexpr uint32_t kLine = 16 * kColTiles + 4;          // floats of a row of a wave's block: no bank conflicts
  constexpr uint32_t kBlock = 16 * kLine;                 // ... of one row tile
  constexpr int kBlocks = WK > 1 ? RT : 1;                // row tiles in LDS at a time
  static_assert(WC * WK * kBlocks * kBlock * 4 <= staged_bytes<XP, RT, WK>(), "the results fit the staging buffers");
  constexpr uint32_t kOutCols = 16 * CT, kLanes = kOutCols / 4, kRows = 64 / kLanes;   // of a piece of 64 lanes
  __syncthreads();
  float *blocks = (float *)staged;
  // (counted anew: the thread's index need not stay in a register through the loop)
  const uint32_t out_lane = __builtin_amdgcn_mbcnt_hi(0xffffffffu, __builtin_amdgcn_mbcnt_lo(0xffffffffu, 0u));
  const uint32_t piece_row = out_lane / kLanes, piece_column = out_lane % kLanes * 4;
  const uint32_t column = col_block * kBlockCols + wc * kOutCols + piece_column;
  auto put_block = [&](int rt) {
    float *mine = blocks + ((wk * WC + wc) * kBlocks + rt % kBlocks) * kBlock + 4 * (out_lane >> 4) * kLine + (out_lane & 15);
#pragma unroll
    for (int tp = 0; tp < kColTiles; ++tp)
#pragma unroll
      for (int i = 0; i < 4; ++i) mine[i * kLine + 16 * tp] = acc[tp][rt][i];
  };
  auto swiglu = [](f32x4 &value, const f32x4 &up) {
#pragma unroll
    for (int i = 0; i < 4; ++i) value[i] = value[i] * (1.0f / (1.0f + __expf(-value[i]))) * up[i];
  };
  auto store = [&](uint32_t row, f32x4 value) {
    if (!kRouted && a.splits > 1) {
      *(f32x4 *)((float *)a.out + ((uint64_t)split * a.rows + tile_first + row) * a.columns + column) = value;
      return;
    }
    if (!kRouted && a.residual) {
      const uint64_t at = (uint64_t)(tile_first + row) * a.residual_row_stride + column;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        value[i] += XP == 1 ? low_bf16(((const uint16_t *)a.residual)[at + i]) : ((const float *)a.residual)[at + i];
    }
    const uint64_t at = (uint64_t)(kRouted ? row_ids[row] : tile_first + row) * a.out_row_stride + column;
    if (a.out_f32) {
      float *to = (float *)a.out + at;
      if (a.out_aligned)
        *(f32x4 *)to = value;
      else
        for (int i = 0; i < 4; ++i) to[i] = value[i];
    } else {
      uint16_t *to = (uint16_t *)a.out + at;
      const u32x2 packed = {pack_bf16(value[0], value[1]), pack_bf16(value[2], value[3])};
      if (a.out_aligned)
        *(u32x2 *)to = packed;
      else
        for (int i = 0; i < 4; ++i) to[i] = (uint16_t)(packed[i / 2] >> (16 * (i % 2)));
    }
  };
  // Results that are computed again value by value, after the others (one copy of the code), a bit for each
  // four that are no numbers: a row that holds an infinity has it subtracted from itself by its pieces and
  // by its group sum, and values next to f32's largest overflow on the way (a group sum by 128 of them).
  // What the products themselves give is the reference's infinity, or NaN.
  // So too results of f32 rows that are next to nothing, all four below 2^-80: where every value of a row is
  // below 2^-104 or so, the pieces of the group sums and the products of factor and scale lose bits below the
  // smallest normal number, and only such rows (or weights no larger than 2^-40) end there.  (Rows of 4096
  // values at 2^-126: error 3e-4 through the pieces, 4e-7 value by value.  Looking at the values instead of
  // the results costs the loop 2 % of the time.)
  constexpr uint32_t kSteps = 16 / kRows;
  uint32_t again = 0;
  auto is_number = [](const f32x4 &value) {
    uint32_t largest = 0;   // bits of the largest of the four; a NaN's are above an infinity's
#pragma unroll
    for (int i = 0; i < 4; ++i) largest = max(largest, __float_as_uint(value[i]) & 0x7fffffffu);
    return XP == 1 ? largest < 0x7f800000u : largest - (47u << 23) < 0x7f800000u - (47u << 23) || largest == 0;
  };
  auto finish_block = [&](int rt) {
    const float *from = blocks + (wc * kBlocks + rt % kBlocks) * kBlock + piece_column;
#pragma unroll 1
    for (uint32_t step = wk; step < kSteps; step += WK) {
      const uint32_t in_tile = step * kRows + piece_row, row = 16 * rt + in_tile;
      f32x4 value = *(const f32x4 *)(from + in_tile * kLine);
#pragma unroll
      for (int part = 1; part < WK; ++part)
        value += *(const f32x4 *)(from + part * WC * kBlocks * kBlock + in_tile * kLine);
      bool number = is_number(value);
      if constexpr (kPair) {
        const f32x4 up = *(const f32x4 *)(from + in_tile * kLine + kOutCols);
        number &= is_number(up);
        swiglu(value, up);
      }
      if (row >= tile_count || column >= a.columns) continue;
      if (!number) again |= 1u << (rt * kSteps + step);
      store(row, value);
    }
  };
  auto by_value = [&](int pj, uint32_t row) -> f32x4 {
    const uint64_t in_row = kRouted ? row_ids[row] / a.route_div : tile_first + row;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (uint32_t k = first_quad * kQuad; k < last_quad * kQuad; ++k) {
      const uint64_t x_at = in_row * a.x_row_stride + k;
      const float x = XP == 1 ? low_bf16(((const uint16_t *)a.x)[x_at]) : ((const float *)a.x)[x_at];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint64_t group = expert * a.expert_groups + (uint64_t)(column + i) * groups_per_row + k / kGroup;
        const uint32_t word = a.packed[pj][expert * a.expert_words + (uint64_t)(column + i) * words_per_row + k / (32 / BITS)];
        const float q = (float)(word >> (k % (32 / BITS) * BITS) & ((1u << BITS) - 1));
        sum[i] += x * (low_bf16(a.scales[pj][group]) * q + low_bf16(a.biases[pj][group]));
      }
    }
    return sum;
  };
  if constexpr (WK > 1) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) put_block(rt);
    __syncthreads();
#pragma unroll 1
    for (int rt = 0; rt < RT; ++rt) finish_block(rt);
  } else {   // (a wave's own block, written and read by that wave: its LDS accesses are in order)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      put_block(rt);
      __builtin_amdgcn_wave_barrier();
      finish_block(rt);
      __builtin_amdgcn_wave_barrier();
    }
  }
#pragma unroll 1
  for (; again; again &= again - 1) {
    const uint32_t bit = (uint32_t)__ffs((int)again) - 1, row = 16 * (bit / kSteps) + bit % kSteps * kRows + piece_row;
    f32x4 value = by_value(0, row);
    if constexpr (kPair) swiglu(value, by_value(1, row));
    store(row, value);
  }
}

// out[r, c..c+4) = residual? + the K ranges' partial sums, added in order.  Bound by its bytes, and of few rows by the
// launch: what a thread reads it asks for at once, and its four results are one store where rows and residual are
// `aligned` to four elements (four ranges of 512 x 5120: 10.3 -> 9.1 us).
__global__ __launch_bounds__(256) void sum_ranges_kernel(const float *partials, uint32_t splits, uint32_t rows,
                                                         uint32_t columns, void *out, uint64_t out_row_stride,
                                                         uint32_t out_f32, const void *residual,
                                                         uint64_t residual_row_stride, uint32_t residual_f32,
                                                         uint32_t aligned) {
  const uint64_t at = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 4, plane = (uint64_t)rows * columns;
  if (at >= plane) return;
  const uint64_t row = plane <= 0xffffffffull ? (uint32_t)at / columns : at / columns, column = at - row * columns;
  f32x4 added = {0.0f, 0.0f, 0.0f, 0.0f};
  if (residual) {
    const uint64_t from = row * residual_row_stride + column;
    if (aligned && residual_f32) {
      added = *(const f32x4 *)((const float *)residual + from);
    } else if (aligned) {
      const uint2 words = *(const uint2 *)((const uint16_t *)residual + from);
      added = f32x4{low_bf16(words.x), high_bf16(words.x), low_bf16(words.y), high_bf16(words.y)};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        added[i] = residual_f32 ? ((const float *)residual)[from + i] : low_bf16(((const uint16_t *)residual)[from + i]);
    }
  }
  f32x4 total = *(const f32x4 *)(partials + at);
#pragma unroll 4
  for (uint32_t s = 1; s < splits; ++s) total += *(const f32x4 *)(partials + s * plane + at);
  if (residual) total += added;
  const uint64_t to = row * out_row_stride + column;
  if (aligned && out_f32) {
    *(f32x4 *)((float *)out + to) = total;
  } else if (aligned) {
    *(uint2 *)((uint16_t *)out + to) = make_uint2(pack_bf16(total[0], total[1]), pack_bf16(total[2], total[3]));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (out_f32)
        ((float *)out)[to + i] = total[i];
      else
        ((uint16_t *)out)[to + i] = (uint16_t)pack_bf16(total[i], 0.0f);
    }
  }
}

template <int XP, int BITS, int RT, int WC, int WK, bool kPair, bool kRouted>
void launch_rows(hipStream_t stream, const RowsArgs &a, uint32_t grid) {
  constexpr uint32_t lds = staged_bytes<XP, RT, WK>() + (kRouted ? 64 * RT : 0);
  const void *kernel = reinterpret_cast<const void *>(&qmm_rows_kernel<XP, BITS, RT, WC, WK, kPair, kRouted>);
  static const hipError_t configured =
      hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);   // once per process
  (void)configured;
  qmm_rows_kernel<XP, BITS, RT, WC, WK, kPair, kRouted><<<dim3(grid), 64 * WC * WK, lds, stream>>>(a);
}

}  // namespace

bool launch_rows_dense(fh_backend *backend, const RowsDense &d) {
  if (d.rows == 0 || d.columns == 0 || d.columns % 16 != 0 || d.inner == 0 || d.inner % kQuad != 0) return false;
  if (d.bits != 4 && !(d.bits == 8 && d.wide)) return false;
  if (d.rows * d.x_row_stride * (d.wide ? 4 : 2) > 0xffffffffull) return false;   // a lane's row offset is 32 bits
  // Row tiles: of bf16 rows as few times 16 as divide the rows evenly, 64 at most; of f32 rows, whose
  // operands take three times the registers, 32 (64 measured the same at 512 rows and up to a fifth
  // slower below 128).
  const uint32_t most_rows = d.wide ? 32 : 64, row_blocks = (d.rows + most_rows - 1) / most_rows;
  const uint32_t tile_rows = d.wide ? 32 : ((d.rows + row_blocks - 1) / row_blocks + 15) / 16 * 16;
  const uint32_t block_cols = d.wide ? 256 : 128;
  RowsArgs a{};
  a.x = d.x;
  a.x_row_stride = d.x_row_stride;
  a.packed[0] = d.packed;
  a.scales[0] = d.scales;
  a.biases[0] = d.biases;
  a.out = d.out;
  a.out_row_stride = d.out_row_stride;
  a.out_f32 = d.out_f32;
  a.out_aligned = (uintptr_t)d.out % (d.out_f32 ? 16 : 8) == 0 && d.out_row_stride % 4 == 0;
  a.residual = d.residual;
  a.residual_row_stride = d.residual_row_stride;
  a.rows = d.rows;
  a.inner = d.inner;
  a.columns = d.columns;
  a.row_blocks = row_blocks;
  a.col_blocks = (d.columns + block_cols - 1) / block_cols;
  a.splits = 1;
  // K over workgroups where that shortens the launch, estimated for the XCD that gets the most of them (units go round
  // the eight: 220 tiles of 350 x 5120 put 33 on each of four XCDs, which take a third longer than 32 would).  In microseconds:
  // a workgroup alone on its compute unit takes `alone` per quad of its longest K wave (measured, K = 17408: rows of
  // 16, 32, 48 and 64 2.0, 2.5, 2.9 and 3.5; f32 rows 4.4), two that share one `shared`, a round of those 2 besides;
  // splits cost their partial sums and the launch that adds them.  What is not measured by itself is chosen so that of 109
  // products of 9 to 128 bf16 rows (K 2048 to 17408) and 63 of 33 to 1024 f32 rows, each timed with one to ten splits, the
  // chosen number is 0.14 and 0.6 % off the fastest on average, 4 and 7 % at most.  (Counted for the whole device, with
  // constants from operand-order loads: 1.0 and 4 %, 13 and 40 % at most; 95 x 5120 x 17408 51 -> 46 us with six splits
  // for three, 330 f32 rows x 5120 x 2048 58 -> 41 with two for one.)
  const uint32_t quads = d.inner / kQuad, waves_k = d.wide ? 1 : 2;
  const uint64_t places = 2 * std::max<uint32_t>(1, backend_compute_units(backend) / 8);   // of an XCD
  const uint64_t plane = (uint64_t)d.rows * d.columns * sizeof(float);
  if (d.columns % 4 == 0) {
    const double alone = d.wide ? 4.4 : 1.45 + 0.5 * tile_rows / 16, shared = (d.wide ? 1.55 : 1.65) * alone;
    const double bytes_per_us = d.wide ? 4.5e6 : 3e6;
    const uint64_t most = std::min<uint64_t>(std::max<uint32_t>(1, quads / waves_k), backend_workspace_limit(backend) / plane);
    uint64_t best = 1;
    double best_us = 0.0;
    for (uint64_t splits = 1; splits == 1 || splits <= most; ++splits) {
      const uint64_t range = (quads + splits - 1) / splits, rounds = (range + waves_k - 1) / waves_k;
      const uint64_t groups = (a.col_blocks * splits + 7) / 8 * a.row_blocks, whole = groups / places, rest = groups % places;
      double us = (whole + (2 * rest > places)) * (rounds * shared + 2.0);
      if (rest && 2 * rest <= places) us += rounds * alone;
      if (splits > 1) us += splits * plane / bytes_per_us + 3.0;
      if (splits == 1 || us < best_us) best = splits, best_us = us;
    }
    if (best > 1) {
      float *partials = (float *)backend_workspace(backend, best * plane);
      if (partials) {
        a.splits = (uint32_t)best;
        a.out = partials;
        a.residual = nullptr;
      }
    }
  }
  const uint64_t units = ((uint64_t)a.col_blocks * a.splits + 7) / 8 * 8;
  if (units * a.row_blocks > 0x7fffffffull) return false;
  const uint32_t grid = (uint32_t)(units * a.row_blocks);
  hipStream_t stream = backend_stream(backend);
  KernelTimer timer(backend, FH_KC_QMM_KERNEL);
  if (d.wide) {
    if (d.bits == 4)
      launch_rows<3, 4, 2, 4, 1, false, false>(stream, a, grid);
    else
      launch_rows<3, 8, 2, 4, 1, false, false>(stream, a, grid);
  } else {
    switch (tile_rows / 16) {
    case 1: launch_rows<1, 4, 1, 2, 2, false, false>(stream, a, grid); break;
    case 2: launch_rows<1, 4, 2, 2, 2, false, false>(stream, a, grid); break;
    case 3: launch_rows<1, 4, 3, 2, 2, false, false>(stream, a, grid); break;
    default: launch_rows<1, 4, 4, 2, 2, false, false>(stream, a, grid); break;
    }
  }
  const bool residual_aligned = !d.residual || ((uintptr_t)d.residual % (d.wide ? 16 : 8) == 0 && d.residual_row_stride % 4 == 0);
  if (a.splits > 1)
    sum_ranges_kernel<<<dim3((unsigned)(((uint64_t)d.rows * d.columns / 4 + 255) / 256)), 256, 0, stream>>>(
        (const float *)a.out, a.splits, d.rows, d.columns, d.out, d.out_row_stride, d.out_f32, d.residual,
        d.residual_row_stride, d.wide, a.out_aligned && residual_aligned);
  return true;
}

uint32_t rows_route_tile(bool wide) { return wide ? 32 : 64; }

bool rows_routed_supports(uint32_t inner, uint32_t columns) {
  return columns != 0 && columns % 16 == 0 && inner != 0 && inner % kQuad == 0;
}

bool launch_rows_routed(fh_backend *backend, const KsplitRouted &r) {
  if (r.tile_rows != rows_route_tile(r.wide) || (r.wide && !r.out_f32)) return false;
  if (!rows_routed_supports(r.inner, r.columns)) return false;
  RowsArgs a{};
  a.x = r.x;
  a.x_row_stride = r.x_row_stride;
  for (int pj = 0; pj < (r.pair ? 2 : 1); ++pj) {
    a.packed[pj] = r.packed[pj];
    a.scales[pj] = r.scales[pj];
    a.biases[pj] = r.biases[pj];
  }
  a.expert_words = (uint64_t)r.columns * r.inner / 8;
  a.expert_groups = (uint64_t)r.columns * r.inner / kGroup;
  a.out = r.out;
  a.out_row_stride = r.columns;
  a.out_f32 = r.out_f32;
  a.out_aligned = (uintptr_t)r.out % (r.out_f32 ? 16 : 8) == 0;   // (columns are a multiple of 16)
  a.inner = r.inner;
  a.columns = r.columns;
  a.splits = 1;
  a.sorted_routes = r.sorted_routes;
  a.blocks = r.blocks;
  a.n_blocks = r.n_blocks;
  a.route_div = r.route_div;
  const uint32_t block_cols = r.pair ? 128 : 256;
  a.col_blocks = (r.columns + block_cols - 1) / block_cols;
  const uint64_t blocks = ((uint64_t)r.max_blocks + 7) / 8 * 8 * a.col_blocks;
  if (blocks > 0x7fffffffull) return false;
  const uint32_t grid = (uint32_t)blocks;
  hipStream_t stream = backend_stream(backend);
  if (r.wide)
    r.pair ? launch_rows<3, 4, 2, 4, 1, true, true>(stream, a, grid)
           : launch_rows<3, 4, 2, 4, 1, false, true>(stream, a, grid);
  else
    r.pair ? launch_rows<1, 4, 4, 4, 1, true, true>(stream, a, grid)
           : launch_rows<1, 4, 4, 4, 1, false, true>(stream, a, grid);
  return true;
}

}  // namespace fh
