// GPU-side token->expert packing for routed (MoE) projections.
//
// Behavioural reference: count_expert_routes / plan_expert_routes / arrange_expert_routes
// (crates/forja-metal/src/quant_matmul.metal:1217-1357): per-expert counts, exclusive offsets,
// and `sorted_routes` = route ids r*k+s grouped by expert with ascending route id inside an
// expert (a stable counting sort), plus (expert,start,count<=tile_rows) row blocks for a grouped
// GEMM.  Pure integer work: results are bit-exact against the closed form.
#include "kernels.hpp"

namespace fh {

namespace {

// One workgroup of 16 waves does the whole plan in a single launch: what matters is the number of dependent memory
// round trips.  Up to 1024 routes each thread has one (route_pack_round_kernel).  Beyond, each wave takes a
// contiguous run of routes, 64 at a time: it counts them per expert in its own row of LDS, the rows are scanned over
// the experts and waves once, and the wave walks its run again with its own cursors, so that the number of barriers
// does not grow with the routes.  The sorted routes are put together in LDS where they fit (kStaged; 16 bits
// each) and leave in whole lines.  16640 routes of 128 experts 22.5 us, 4096 9.7 (in rounds of 1024, five barriers each, 42
// and 13; 1024 routes 6.8 in the round, 8.5 by runs).
constexpr uint32_t kPackThreads = 1024, kPackWaves = kPackThreads / 64;
constexpr int kPackAhead = 4;   // steps whose expert ids are requested together (more unrolled steps cost more to fetch than to run)

// At most 1024 routes, one to a thread.
__global__ __launch_bounds__(1024) void route_pack_round_kernel(
    View indices, uint32_t rows, uint32_t k, uint32_t experts, uint32_t tile_rows, uint32_t *counts,
    uint32_t *offsets, uint32_t *sorted_routes, uint32_t *blocks, uint32_t max_blocks,
    uint32_t *n_blocks, uint32_t *zero_rows, uint32_t zero_row_words, ErrorSlot *error) {
  extern __shared__ uint32_t lds[];
  uint32_t *lds_counts = lds;                    // [experts]
  uint32_t *lds_cursor = lds + experts;          // [experts] first position of the expert
  uint32_t *wave_counts = lds + 2 * experts;     // [kPackWaves][experts]
  uint32_t *scan = lds + (2 + kPackWaves) * experts;  // [kPackWaves + 1]
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t routes = rows * k;
  auto expert_of = [&](uint32_t route) {
    return load_u32_at(indices, indices.offset + (uint64_t)(route / k) * indices.stride[0] +
                                    (uint64_t)(route % k) * indices.stride[1]);
  };
  for (uint32_t e = tid; e < experts; e += kPackThreads) lds_counts[e] = 0;
  __syncthreads();
  const uint32_t route = tid, expert = route < routes ? expert_of(route) : 0xffffffffu;
  const bool valid = route < routes && expert < experts;
  if (valid) {
    atomicAdd(&lds_counts[expert], 1u);
  } else if (route < routes) {
    report_error(error, expert);
    // a bad route is never packed: its output row (if the caller has one) is cleared here
    if (zero_rows)
      for (uint32_t w = 0; w < zero_row_words; ++w) zero_rows[(uint64_t)route * zero_row_words + w] = 0;
  }
  __syncthreads();
  // Exclusive scans over the experts of the route counts (-> offsets) and of the tile counts
  // (-> first row block of each expert): one expert per thread per round, wave scans stitched
  // through LDS.
  uint32_t running = 0, block_running = 0;
  for (uint32_t base = 0; base < experts; base += kPackThreads) {
    const uint32_t e = base + tid;
    const uint32_t c = e < experts ? lds_counts[e] : 0;
    const uint32_t tiles = (c + tile_rows - 1) / tile_rows;
    uint32_t inclusive = c, inclusive_tiles = tiles;
    for (int offset = 1; offset < 64; offset <<= 1) {
      const uint32_t other = __shfl_up(inclusive, offset, 64);
      const uint32_t other_tiles = __shfl_up(inclusive_tiles, offset, 64);
      if ((int)lane >= offset) {
        inclusive += other;
        inclusive_tiles += other_tiles;
      }
    }
    if (lane == 63) {
      scan[wave] = inclusive;
      scan[kPackWaves + 1 + wave] = inclusive_tiles;
    }
    __syncthreads();
    uint32_t before = running, before_tiles = block_running, total = 0, total_tiles = 0;
    for (uint32_t w = 0; w < kPackWaves; ++w) {
      if (w < wave) {
        before += scan[w];
        before_tiles += scan[kPackWaves + 1 + w];
      }
      total += scan[w];
      total_tiles += scan[kPackWaves + 1 + w];
    }
    if (e < experts) {
      const uint32_t start = before + inclusive - c;
      counts[e] = c;
      offsets[e] = start;
      lds_cursor[e] = start;
      const uint32_t first = before_tiles + inclusive_tiles - tiles;
      for (uint32_t t = 0; t < tiles; ++t) {
        const uint32_t b = first + t;
        if (b >= max_blocks) break;
        const uint32_t remaining = c - t * tile_rows;
        blocks[3 * b + 0] = e;
        blocks[3 * b + 1] = start + t * tile_rows;
        blocks[3 * b + 2] = remaining < tile_rows ? remaining : tile_rows;
      }
    }
    running += total;
    block_running += total_tiles;
    __syncthreads();
  }
  if (tid == 0) {
    offsets[experts] = running;
    n_blocks[0] = block_running < max_blocks ? block_running : max_blocks;
  }
  for (uint32_t b = block_running + tid; b < max_blocks; b += kPackThreads) {
    blocks[3 * b + 0] = 0xffffffffu;
    blocks[3 * b + 1] = 0;
    blocks[3 * b + 2] = 0;
  }
  // Stable: a route's position is its expert's first + the routes of the same expert in lower waves + its rank among
  // the lower lanes of its own wave.
  for (uint32_t i = tid; i < kPackWaves * experts; i += kPackThreads) wave_counts[i] = 0;
  unsigned long long same = __ballot(valid);
  for (uint32_t bit = 0; (experts - 1) >> bit; ++bit) {
    const unsigned long long set = __ballot(valid && ((expert >> bit) & 1u));
    same &= ((expert >> bit) & 1u) ? set : ~set;
  }
  const uint32_t rank = __popcll(same & ((1ull << lane) - 1ull));
  __syncthreads();  // wave_counts cleared
  if (valid && rank == 0) wave_counts[wave * experts + expert] = __popcll(same);
  __syncthreads();
  if (valid) {
    uint32_t position = lds_cursor[expert] + rank;
    for (uint32_t w = 0; w < wave; ++w) position += wave_counts[w * experts + expert];
    sorted_routes[position] = route;
  }
}

template <bool kStaged>
__global__ __launch_bounds__(1024) void route_pack_kernel(
    View indices, uint32_t rows, uint32_t k, uint32_t experts, uint32_t tile_rows, uint32_t *counts,
    uint32_t *offsets, uint32_t *sorted_routes, uint32_t *blocks, uint32_t max_blocks,
    uint32_t *n_blocks, uint32_t *zero_rows, uint32_t zero_row_words, ErrorSlot *error) {
  extern __shared__ uint32_t lds[];
  uint32_t *cursors = lds;                                   // [kPackWaves][experts]: a wave's counts, then its next places
  uint32_t *scan = lds + kPackWaves * experts;               // [2][kPackWaves]
  uint16_t *staged = (uint16_t *)(scan + 2 * kPackWaves);    // [routes]
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t routes = rows * k;
  const uint32_t run = (routes + kPackThreads - 1) / kPackThreads * 64;   // routes of a wave
  const uint32_t first = min(wave * run, routes), last = min(first + run, routes);
  const bool dense = indices.stride[1] == 1 && indices.stride[0] == k;
  auto expert_of = [&](uint32_t route) {   // (a route past the end reads the last one)
    const uint64_t r = min(route, routes - 1);
    return load_u32_at(indices, indices.offset + (dense ? r : r / k * indices.stride[0] + r % k * indices.stride[1]));
  };
  // the lanes of the wave that hold the same expert
  auto same_expert = [&](uint32_t expert, bool valid) {
    unsigned long long same = __ballot(valid);
    for (uint32_t bit = 0; (experts - 1) >> bit; ++bit) {
      const unsigned long long set = __ballot(valid && ((expert >> bit) & 1u));
      same &= ((expert >> bit) & 1u) ? set : ~set;
    }
    return same;
  };
  uint32_t *mine = cursors + wave * experts;
  for (uint32_t i = tid; i < kPackWaves * experts; i += kPackThreads) cursors[i] = 0;
  __syncthreads();
  // Calls step(route, expert, valid) for the wave's routes in order, 64 at a time.
  auto walk = [&](auto step) {
    uint32_t next[kPackAhead];
#pragma unroll
    for (int i = 0; i < kPackAhead; ++i) next[i] = expert_of(first + 64 * i + lane);
#pragma unroll 1
    for (uint32_t base = first; base < last; base += 64 * kPackAhead) {
      uint32_t now[kPackAhead];
#pragma unroll
      for (int i = 0; i < kPackAhead; ++i) {
        now[i] = next[i];
        next[i] = expert_of(base + 64 * (kPackAhead + i) + lane);
      }
#pragma unroll
      for (int i = 0; i < kPackAhead; ++i) {
        const uint32_t route = base + 64 * i + lane;
        if (base + 64 * i < last) step(route, now[i], route < last && now[i] < experts);
      }
    }
  };
  walk([&](uint32_t route, uint32_t expert, bool valid) {
    if (valid) {
      atomicAdd(&mine[expert], 1u);
    } else if (route < last) {
      report_error(error, expert);
      // a bad route is never packed: its output row (if the caller has one) is cleared here
      if (zero_rows)
        for (uint32_t w = 0; w < zero_row_words; ++w) zero_rows[(uint64_t)route * zero_row_words + w] = 0;
    }
  });
  __syncthreads();
  // Exclusive scans over the experts of the route counts (-> offsets) and of the tile counts
  // (-> first row block of each expert): one expert per thread per round, wave scans stitched
  // through LDS.
  uint32_t running = 0, block_running = 0;
  for (uint32_t base = 0; base < experts; base += kPackThreads) {
    const uint32_t e = base + tid;
    uint32_t of_wave[kPackWaves], c = 0;
#pragma unroll
    for (uint32_t w = 0; w < kPackWaves; ++w) of_wave[w] = e < experts ? cursors[w * experts + e] : 0;
#pragma unroll
    for (uint32_t w = 0; w < kPackWaves; ++w) c += of_wave[w];
    const uint32_t tiles = (c + tile_rows - 1) / tile_rows;
    uint32_t inclusive = c, inclusive_tiles = tiles;
    for (int offset = 1; offset < 64; offset <<= 1) {
      const uint32_t other = __shfl_up(inclusive, offset, 64);
      const uint32_t other_tiles = __shfl_up(inclusive_tiles, offset, 64);
      if ((int)lane >= offset) {
        inclusive += other;
        inclusive_tiles += other_tiles;
      }
    }
    if (lane == 63) {
      scan[wave] = inclusive;
      scan[kPackWaves + wave] = inclusive_tiles;
    }
    __syncthreads();
    uint32_t before = running, before_tiles = block_running, total = 0, total_tiles = 0;
    for (uint32_t w = 0; w < kPackWaves; ++w) {
      if (w < wave) {
        before += scan[w];
        before_tiles += scan[kPackWaves + w];
      }
      total += scan[w];
      total_tiles += scan[kPackWaves + w];
    }
    if (e < experts) {
      const uint32_t start = before + inclusive - c;
      counts[e] = c;
      offsets[e] = start;
      uint32_t place = start;   // of the wave's first route of this expert
#pragma unroll
      for (uint32_t w = 0; w < kPackWaves; ++w) {
        cursors[w * experts + e] = place;
        place += of_wave[w];
      }
      const uint32_t first_tile = before_tiles + inclusive_tiles - tiles;
      for (uint32_t t = 0; t < tiles; ++t) {
        const uint32_t b = first_tile + t;
        if (b >= max_blocks) break;
        const uint32_t remaining = c - t * tile_rows;
        blocks[3 * b + 0] = e;
        blocks[3 * b + 1] = start + t * tile_rows;
        blocks[3 * b + 2] = remaining < tile_rows ? remaining : tile_rows;
      }
    }
    running += total;
    block_running += total_tiles;
    __syncthreads();
  }
  if (tid == 0) {
    offsets[experts] = running;
    n_blocks[0] = block_running < max_blocks ? block_running : max_blocks;
  }
  for (uint32_t b = block_running + tid; b < max_blocks; b += kPackThreads) {
    blocks[3 * b + 0] = 0xffffffffu;
    blocks[3 * b + 1] = 0;
    blocks[3 * b + 2] = 0;
  }
  // Stable: a route's place is its expert's cursor in this wave + its rank among the step's lower lanes.
  walk([&](uint32_t route, uint32_t expert, bool valid) {
    const unsigned long long same = same_expert(expert, valid);
    const uint32_t rank = __popcll(same & ((1ull << lane) - 1ull));
    uint32_t place = 0;
    if (valid) place = mine[expert] + rank;
    __builtin_amdgcn_wave_barrier();   // (LDS accesses of a wave are in order)
    if (valid && rank == 0) mine[expert] = place + __popcll(same);
    __builtin_amdgcn_wave_barrier();
    if (valid) {
      if (kStaged)
        staged[place] = (uint16_t)route;
      else
        sorted_routes[place] = route;
    }
  });
  if (kStaged) {
    __syncthreads();
    for (uint32_t i = tid; i < running; i += kPackThreads) sorted_routes[i] = staged[i];
  }
}

}  // namespace

void launch_route_pack(hipStream_t s, const View &indices, uint32_t rows, uint32_t k,
                       uint32_t experts, uint32_t tile_rows, uint32_t *counts, uint32_t *offsets,
                       uint32_t *sorted_routes, uint32_t *blocks, uint32_t max_blocks,
                       uint32_t *n_blocks, ErrorSlot *error, uint32_t *zero_rows,
                       uint32_t zero_row_words) {
  if ((uint64_t)rows * k <= kPackThreads) {
    const size_t lds = ((size_t)experts * (2 + kPackWaves) + 2 * (kPackWaves + 1)) * sizeof(uint32_t);
    route_pack_round_kernel<<<dim3(1), kPackThreads, lds, s>>>(indices, rows, k, experts, tile_rows, counts, offsets,
                                                               sorted_routes, blocks, max_blocks, n_blocks, zero_rows,
                                                               zero_row_words, error);
    return;
  }
  size_t lds = ((size_t)experts * kPackWaves + 2 * kPackWaves) * sizeof(uint32_t);
  const size_t staged = (size_t)rows * k * sizeof(uint16_t);
  const bool fits = (uint64_t)rows * k <= 65536 && lds + staged <= 64 * 1024;
  auto *kernel = fits ? route_pack_kernel<true> : route_pack_kernel<false>;
  kernel<<<dim3(1), kPackThreads, lds + (fits ? staged : 0), s>>>(indices, rows, k, experts, tile_rows, counts, offsets,
                                                                 sorted_routes, blocks, max_blocks, n_blocks, zero_rows,
                                                                 zero_row_words, error);
}

}  // namespace fh
