// searchsorted of many values in a long array: the values go to the part of the array that holds their answers, the array is
// read once, and the answers come back, all in tiles of values that stay where they are in memory.
//
// Stands where SearchSortedTask's GPU variant runs one search per thread over the array
// (src/cupynumeric/sort/searchsorted.cu:27-116).  The array is cut into up to 2048 parts of equal length.
//   group   a workgroup puts a tile of 16384 values into the order of their parts (part: a search among the parts' first
//           elements, in LDS); a table says where each part starts in the tile, and each value keeps its place (16 bits)
//   plan    how many values every part has, and from that one piece of work per 8704 of them
//   search  a workgroup per piece collects its values from all tiles, sorts them by the windows of the part, and goes through
//           the windows: one coalesced read of 32 KiB of the array each, the searches in LDS.  Windows without a value
//           are not read.  The answers go back to the values' places in their tiles.
//   return  a workgroup per tile puts the answers of its values into the order that the values came in.
//
// Bound by the read of the array and by latency: for 2^24 float32 values in 2^28, group 52 us, plan 11, search 335 (the read at
// the rate of a copy: 173), return 47.  The other way, a sort of the values with their positions, costs four passes over them (for
// 8-byte keys up to eight) and one 8-byte store per value at a place of its own, 64 bytes of memory traffic each: of the
// 503 us that its search took for 2^24 float32 values in 2^28, 248 went into these stores.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sort_driver.h"

namespace cpn {

constexpr int FIND_PARTS    = 2048;
constexpr int FIND_BLOCK    = 1024;  // group, return
constexpr int FIND_ITEMS    = 16;
constexpr int FIND_AT_ONCE  = 4;     // searches of a lane in flight
constexpr int FIND_TILE     = FIND_BLOCK * FIND_ITEMS;
constexpr int FIND_TILES    = 1024;  // of a batch of values
constexpr int FIND_SEARCHERS = 512;  // a workgroup of the search
constexpr int FIND_LANES    = 8;     // lanes that copy a tile's values of a part (8 of them in the mean)
constexpr int FIND_GATHER   = 8;     // tiles of which a lane has a value in flight
// Values of a part in a tile that the whole workgroup copies (8 lanes alone: half of 2^24 values in a thousandth of 2^28,
// 1342 -> 725 us a call).
constexpr int FIND_CROWD    = 64;
constexpr int FIND_WINDOW   = 32768; // bytes
constexpr int FIND_WINDOWS  = 64;    // of a part, at most
constexpr int FIND_EACH     = 17;    // values of a piece, per lane: a part of a full batch has 8192 in the mean
// Waves per SIMD: as many workgroups as LDS has room for (4-byte keys, two or three of them a CU: 369 / 346 us).
constexpr int find_waves(int key_bytes) { return key_bytes == 4 ? 6 : 4; }

struct FindPlan {  // at the head of the workspace
  uint32_t items;
};

template <int CODEC, bool LEFT, typename KeyT>
__device__ __forceinline__ bool before_answer(KeyT element, KeyT value)
{
  return LEFT ? element < value : element <= value;
}

// What is computed from the result is not kept over the steps of a kernel: places and conditions of twenty values would
// take all registers.
__device__ __forceinline__ uint32_t find_opaque(uint32_t x)
{
  asm volatile("" : "+v"(x));
  return x;
}

// The steps of a search look at elements that are a power of two apart, which would lie in one bank of LDS: a gap after every
// 256 bytes of them moves them to different ones (2^24 float32 values in 2^28, group 129 -> 72 us, search 394 -> 375).  With
// a table filled up to a power of two the steps need no test of the bound: 72 -> 52 and 375 -> 369.
__device__ constexpr uint32_t find_pivot_at(uint32_t j) { return j + (j >> 6); }
__device__ constexpr uint32_t find_pack_at(uint32_t p) { return p + (p >> 4); }
template <typename KeyT>
__device__ constexpr uint32_t find_key_at(uint32_t i)
{
  constexpr uint32_t PACK = 16 / sizeof(KeyT);
  return i + i / (16 * PACK) * PACK;
}

// 16 bytes of the array
template <int CODEC, typename KeyT>
__device__ __forceinline__ uint4 ordered_pack(uint4 q)
{
  if constexpr (sizeof(KeyT) == 4) {
    return uint4{ordered_bits<CODEC, KeyT>(q.x), ordered_bits<CODEC, KeyT>(q.y), ordered_bits<CODEC, KeyT>(q.z),
                 ordered_bits<CODEC, KeyT>(q.w)};
  } else {
    const uint64_t a = ordered_bits<CODEC, KeyT>(q.x | static_cast<uint64_t>(q.y) << 32);
    const uint64_t b = ordered_bits<CODEC, KeyT>(q.z | static_cast<uint64_t>(q.w) << 32);
    return uint4{static_cast<uint32_t>(a), static_cast<uint32_t>(a >> 32), static_cast<uint32_t>(b), static_cast<uint32_t>(b >> 32)};
  }
}

// The first elements of all parts but the first.
template <typename KeyT, int CODEC>
__global__ __launch_bounds__(256) void find_pivots_kernel(const KeyT* __restrict__ sorted, uint64_t n, uint64_t part, uint32_t parts,
                                                          KeyT* __restrict__ pivots)
{
  const uint32_t j = blockIdx.x * 256 + threadIdx.x;
  if (j + 1 < parts) {  // (then (j + 1) * part < n)
    pivots[j] = ordered_bits<CODEC, KeyT>(sorted[(j + 1) * part]);
  }
}

template <typename KeyT, int CODEC, bool LEFT>
__global__ __launch_bounds__(FIND_BLOCK) void find_group_kernel(const KeyT* __restrict__ values, uint64_t num_values,
                                                                const KeyT* __restrict__ pivots, uint32_t parts,
                                                                KeyT* __restrict__ grouped, uint16_t* __restrict__ places,
                                                                uint16_t* __restrict__ starts, FindPlan* __restrict__ plan)
{
  // first the pivots, then the tile, 8-byte keys one half after the other: two workgroups share a CU
  __shared__ __align__(16) union {
    KeyT pivot[find_pivot_at(FIND_PARTS)];
    uint32_t word[FIND_TILE];
  } s;
  __shared__ uint32_t s_start[FIND_PARTS];
  __shared__ uint32_t s_wave[FIND_BLOCK / WAVE];
  const uint32_t tid   = threadIdx.x;
  const uint32_t lane  = tid & (WAVE - 1);
  const uint64_t first = static_cast<uint64_t>(blockIdx.x) * FIND_TILE;
  const uint32_t len   = num_values - first < FIND_TILE ? static_cast<uint32_t>(num_values - first) : FIND_TILE;
  KeyT key[FIND_ITEMS];
#pragma unroll
  for (int i = 0; i < FIND_ITEMS; ++i) {
    const uint32_t o = i * FIND_BLOCK + tid;
    key[i]           = values[first + (o < len ? o : len - 1)];
  }
  for (uint32_t j = tid; j < FIND_PARTS; j += FIND_BLOCK) {
    s_start[j] = 0;
    s.pivot[find_pivot_at(j)] = j + 1 < parts ? pivots[j] : ~KeyT{};  // (left of no answer, or see below)
  }
  if (blockIdx.x == 0 && tid == 0) {
    plan->items = 0;
  }
  __syncthreads();
  uint32_t where[FIND_ITEMS];
#pragma unroll
  for (int i = 0; i < FIND_ITEMS; ++i) {
    key[i]   = ordered_bits<CODEC, KeyT>(key[i]);
    where[i] = 0;
  }
  // (`where` counts gaps as well until the last step: it is a multiple of 2 * step, so that they add up)
#pragma unroll
  for (int i0 = 0; i0 < FIND_ITEMS; i0 += FIND_AT_ONCE) {
#pragma unroll
    for (uint32_t step = FIND_PARTS / 2; step != 0; step >>= 1) {
#pragma unroll
      for (int i = i0; i < i0 + FIND_AT_ONCE; ++i) {
        where[i] += before_answer<CODEC, LEFT>(s.pivot[where[i] + find_pivot_at(step - 1)], key[i]) ? find_pivot_at(step) : 0u;
      }
    }
#pragma unroll
    for (int i = i0; i < i0 + FIND_AT_ONCE; ++i) {
      where[i] -= where[i] / 65;
      where[i] = where[i] < parts ? where[i] : parts - 1;  // (the largest key of all is not left of those that fill the table up)
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < FIND_ITEMS; ++i) {
    if (i * FIND_BLOCK + tid < len) {
      where[i] |= atomicAdd(&s_start[where[i]], 1u) << 16;  // part, and in the upper half which of its values
    }
  }
  static_assert(FIND_TILE <= 32768 && FIND_PARTS <= 65536, "both halves");
  __syncthreads();
  // two parts per thread
  static_assert(FIND_PARTS == 2 * FIND_BLOCK, "two parts per thread");
  const uint32_t c0 = s_start[2 * tid], c1 = s_start[2 * tid + 1];
  const uint32_t incl = wave_inclusive_sum_dpp(c0 + c1);
  if (lane == WAVE - 1) {
    s_wave[tid / WAVE] = incl;
  }
  __syncthreads();
  uint32_t run = incl - c0 - c1;
#pragma unroll
  for (uint32_t w = 0; w < FIND_BLOCK / WAVE; ++w) {
    run += w < tid / WAVE ? s_wave[w] : 0u;
  }
  uint16_t* const row = starts + static_cast<uint64_t>(blockIdx.x) * (FIND_PARTS + 1);
  s_start[2 * tid]     = run;
  s_start[2 * tid + 1] = run + c0;
  row[2 * tid]         = static_cast<uint16_t>(run);
  row[2 * tid + 1]     = static_cast<uint16_t>(run + c0);
  if (tid == FIND_BLOCK - 1) {
    row[FIND_PARTS] = static_cast<uint16_t>(len);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < FIND_ITEMS; ++i) {
    const uint32_t o = i * FIND_BLOCK + tid;
    if (o < len) {
      where[i]          = s_start[where[i] & 0xFFFFu] + (where[i] >> 16);
      s.word[where[i]]  = static_cast<uint32_t>(key[i]);
      places[first + o] = static_cast<uint16_t>(where[i]);
    }
  }
  __syncthreads();
  if constexpr (sizeof(KeyT) == 4) {
#pragma unroll
    for (int i = 0; i < FIND_ITEMS; ++i) {
      const uint32_t o = i * FIND_BLOCK + tid;
      if (o < len) {
        grouped[first + o] = s.word[o];
      }
    }
  } else {
    uint32_t low[FIND_ITEMS];
#pragma unroll
    for (int i = 0; i < FIND_ITEMS; ++i) {
      low[i] = s.word[i * FIND_BLOCK + tid];  // (past the last value: not used)
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < FIND_ITEMS; ++i) {
      if (i * FIND_BLOCK + tid < len) {
        s.word[where[i]] = static_cast<uint32_t>(static_cast<uint64_t>(key[i]) >> 32);
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < FIND_ITEMS; ++i) {
      const uint32_t o = i * FIND_BLOCK + tid;
      if (o < len) {
        grouped[first + o] = low[i] | static_cast<uint64_t>(s.word[o]) << 32;
      }
    }
  }
}

// 64 parts per workgroup: their values in all tiles, and a piece of work for every `room` of them: part, and in the upper
// half which piece of the part.
__global__ __launch_bounds__(FIND_BLOCK) void find_plan_kernel(const uint16_t* __restrict__ starts, uint32_t tiles, uint32_t room,
                                                               FindPlan* __restrict__ plan, uint32_t* __restrict__ items)
{
  __shared__ uint32_t s_sum[FIND_BLOCK / WAVE][WAVE];
  __shared__ uint32_t s_at;
  const uint32_t lane = threadIdx.x & (WAVE - 1);
  const uint32_t wave = threadIdx.x / WAVE;
  const uint32_t part = blockIdx.x * WAVE + lane;
  uint32_t sum        = 0;
#pragma unroll 8
  for (uint32_t t = wave; t < tiles; t += FIND_BLOCK / WAVE) {
    const uint16_t* const row = starts + static_cast<uint64_t>(t) * (FIND_PARTS + 1) + part;
    sum += static_cast<uint32_t>(row[1]) - row[0];
  }
  s_sum[wave][lane] = sum;
  __syncthreads();
  if (wave != 0) {
    return;
  }
  sum = 0;
#pragma unroll
  for (int w = 0; w < FIND_BLOCK / WAVE; ++w) {
    sum += s_sum[w][lane];
  }
  const uint32_t pieces = (sum + room - 1) / room;
  const uint32_t incl   = wave_inclusive_sum_dpp(pieces);
  if (lane == WAVE - 1) {
    s_at = atomicAdd(&plan->items, incl);
  }
  __builtin_amdgcn_wave_barrier();
  const uint32_t at = *static_cast<volatile uint32_t*>(&s_at) + incl - pieces;
  for (uint32_t j = 0; j < pieces; ++j) {
    items[at + j] = part | (j << 16);
  }
}

template <typename KeyT, int CODEC, bool LEFT>
__global__ __launch_bounds__(FIND_SEARCHERS, find_waves(sizeof(KeyT))) void find_search_kernel(const KeyT* __restrict__ sorted, uint64_t n, uint64_t part_len,
                                                                     const KeyT* __restrict__ grouped,
                                                                     const uint16_t* __restrict__ starts, uint32_t tiles,
                                                                     const FindPlan* __restrict__ plan,
                                                                     const uint32_t* __restrict__ items,
                                                                     uint32_t* __restrict__ answers)
{
  constexpr int EACH     = FIND_EACH;
  constexpr int ROOM     = FIND_SEARCHERS * EACH;
  constexpr int WINDOW   = FIND_WINDOW / sizeof(KeyT);
  constexpr int PACK     = 16 / sizeof(KeyT);
  constexpr int PACKS    = FIND_WINDOW / 16 / FIND_SEARCHERS;
  constexpr int WAVES    = FIND_SEARCHERS / WAVE;
  constexpr int GROUPS   = FIND_SEARCHERS / FIND_LANES;
  constexpr int PER_SCAN = FIND_TILES / FIND_SEARCHERS;
  // the piece's values, its windows one after the other, its answers
  __shared__ __align__(16) union {
    KeyT key[ROOM];
    uint4 pack[find_pack_at(FIND_WINDOW / 16)];
    uint32_t word[ROOM];
  } s;
  __shared__ uint32_t s_base[FIND_TILES + 1];  // of the part's values in all tiles, those before a tile's
  __shared__ uint16_t s_from[FIND_TILES];      // where they are in the tile
  __shared__ uint32_t s_count[FIND_WINDOWS + WAVE];
  __shared__ uint32_t s_first[FIND_WINDOWS + 1];
  __shared__ KeyT s_pivot[FIND_WINDOWS];
  __shared__ uint32_t s_wave[WAVES];
  __shared__ uint32_t s_crowds;
  __shared__ uint16_t s_crowd[ROOM / FIND_CROWD];  // tiles with more values of the part
  // workgroups of one XCD take neighbouring parts: they share the cache lines of the tiles' table and of the tiles
  const uint32_t all  = plan->items;
  const uint32_t per  = (all + 7) / 8;
  const uint32_t mine = blockIdx.x % 8 * per + blockIdx.x / 8;
  if (blockIdx.x / 8 >= per || mine >= all) {
    return;
  }
  const uint32_t tid  = threadIdx.x;
  const uint32_t lane = tid & (WAVE - 1);
  const uint32_t part = items[mine] & 0xFFFFu;
  const uint32_t lo   = (items[mine] >> 16) * ROOM;  // of the part's values, the piece's first
  const uint64_t origin = part * part_len;
  const uint32_t extent = n - origin < part_len ? static_cast<uint32_t>(n - origin) : static_cast<uint32_t>(part_len);
  const uint32_t windows = (extent + WINDOW - 1) / WINDOW;
  const KeyT* const elements = sorted + origin;

  // ---- where the values are ----
  uint32_t len[PER_SCAN], own = 0;
#pragma unroll
  for (int k = 0; k < PER_SCAN; ++k) {
    const uint32_t t = tid * PER_SCAN + k;
    uint32_t from    = 0;
    len[k]           = 0;
    if (t < tiles) {
      const uint16_t* const row = starts + static_cast<uint64_t>(t) * (FIND_PARTS + 1) + part;
      from                      = row[0];
      len[k]                    = row[1] - from;
    }
    s_from[t] = static_cast<uint16_t>(from);
    own += len[k];
  }
  const uint32_t incl = wave_inclusive_sum_dpp(own);
  if (lane == WAVE - 1) {
    s_wave[tid / WAVE] = incl;
  }
  if (tid == 0) {
    s_crowds = 0;
  }
  if (tid < FIND_WINDOWS) {
    s_count[tid] = 0;
    s_pivot[tid] = tid + 1 < windows ? ordered_bits<CODEC, KeyT>(elements[(tid + 1) * WINDOW]) : ~KeyT{};
  }
  __syncthreads();
  uint32_t run = incl - own, total = 0;
#pragma unroll
  for (uint32_t w = 0; w < WAVES; ++w) {
    run += w < tid / WAVE ? s_wave[w] : 0u;
    total += s_wave[w];
  }
#pragma unroll
  for (int k = 0; k < PER_SCAN; ++k) {
    s_base[tid * PER_SCAN + k] = run;
    run += len[k];
  }
  if (tid == 0) {
    s_base[FIND_TILES] = total;
  }
  __syncthreads();
  const uint32_t count = total - lo < ROOM ? total - lo : ROOM;  // (a piece is not empty)
  const uint32_t hi    = lo + count;

  // ---- the values, `FIND_LANES` lanes per tile and `FIND_GATHER` tiles of theirs at once ----
  const uint32_t sub = tid % FIND_LANES;
  for (uint32_t t0 = tid / FIND_LANES; t0 < tiles; t0 += FIND_GATHER * GROUPS) {
    uint32_t at[FIND_GATHER], end[FIND_GATHER];
    uint32_t from[FIND_GATHER];  // (a batch has 2^24 values)
    KeyT k[FIND_GATHER];
#pragma unroll
    for (int j = 0; j < FIND_GATHER; ++j) {
      const uint32_t t = t0 + j * GROUPS < tiles ? t0 + j * GROUPS : tiles - 1;
      const uint32_t b = s_base[t], e = s_base[t + 1];
      at[j]   = (b > lo ? b : lo) + sub;
      end[j]  = t0 + j * GROUPS < tiles ? (e < hi ? e : hi) : 0u;
      from[j] = t * FIND_TILE + s_from[t] + at[j] - b;
      k[j]    = KeyT{};
      if (at[j] < end[j]) {
        k[j] = grouped[from[j]];
      }
    }
#pragma unroll
    for (int j = 0; j < FIND_GATHER; ++j) {
      if (at[j] < end[j]) {
        s.key[at[j] - lo] = k[j];
      }
      if (end[j] > at[j] - sub + FIND_CROWD) {  // the same for the lanes of a tile
        if (sub == 0) {
          s_crowd[atomicAdd(&s_crowds, 1u)] = static_cast<uint16_t>(t0 + j * GROUPS);
        }
        continue;
      }
      for (uint32_t o = FIND_LANES; at[j] + o < end[j]; o += FIND_LANES) {
        s.key[at[j] + o - lo] = grouped[from[j] + o];
      }
    }
  }
  __syncthreads();
  const uint32_t crowds = s_crowds;
  for (uint32_t c = 0; c < crowds; ++c) {  // uniform
    const uint32_t t = s_crowd[c];
    const uint32_t b = s_base[t], e = s_base[t + 1];
    const uint32_t from = b > lo ? b : lo, to = e < hi ? e : hi;
    const KeyT* const in = grouped + static_cast<uint64_t>(t) * FIND_TILE + s_from[t];
#pragma unroll 4
    for (uint32_t at = from + tid; at < to; at += FIND_SEARCHERS) {
      s.key[at - lo] = in[at - b];
    }
  }
  __syncthreads();

  // ---- in the order of their windows ----
  uint32_t me = tid;
  KeyT key[EACH];
  uint32_t where[EACH];
  if (windows == 1) {  // uniform: they are
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      where[k] = k * FIND_SEARCHERS + me;
      key[k]   = s.key[where[k]];
    }
    if (tid == 0) {
      s_first[0] = 0;
      s_first[1] = count;
    }
    __syncthreads();
  } else {
    me = find_opaque(tid);
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      const uint32_t o = k * FIND_SEARCHERS + me;
      key[k]           = s.key[o];  // (past the last value: whatever is there, and not used)
      uint32_t w       = 0;
#pragma unroll
      for (uint32_t step = FIND_WINDOWS / 2; step != 0; step >>= 1) {
        w += before_answer<CODEC, LEFT>(s_pivot[w + step - 1], key[k]) ? step : 0u;
      }
      // (branches around parts of this loop make it spill; past the last value a lane counts for itself)
      w        = o < count ? (w < windows ? w : windows - 1) : FIND_WINDOWS + lane;
      where[k] = w | (atomicAdd(&s_count[w], 1u) << 8);
      if (k % FIND_AT_ONCE == FIND_AT_ONCE - 1) {
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
    if (tid < WAVE) {
      const uint32_t c = s_count[tid];
      const uint32_t i = wave_inclusive_sum_dpp(c);
      s_first[tid + 1] = i;
      if (tid == 0) {
        s_first[0] = 0;
      }
    }
    static_assert(FIND_WINDOWS == WAVE, "a lane per window");
    __syncthreads();
    me = find_opaque(tid);
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      const uint32_t o = k * FIND_SEARCHERS + me;
      const uint32_t w = where[k] & 0xFFu;
      where[k]         = w < FIND_WINDOWS ? s_first[w < FIND_WINDOWS ? w : 0] + (where[k] >> 8) : o;
      s.key[where[k]]  = key[k];
    }
    __syncthreads();
    me = find_opaque(tid);
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      key[k] = s.key[k * FIND_SEARCHERS + me];
    }
    __syncthreads();
    me = find_opaque(tid);
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      s.word[where[k]] = k * FIND_SEARCHERS + me;
    }
    __syncthreads();
    me = find_opaque(tid);
#pragma unroll
    for (int k = 0; k < EACH; ++k) {
      where[k] = s.word[k * FIND_SEARCHERS + me];  // which of the piece's values key[k] is
    }
    __syncthreads();
  }

  // ---- window by window, the next one on its way ----
  const auto next_of = [&](uint32_t w) {
    while (w < windows && s_first[w + 1] == s_first[w]) {
      ++w;
    }
    return w;
  };
  uint4 p[PACKS];
  const auto request = [&](uint32_t w) {  // whole packs; what is left of the array's last window is read when it is its turn
    const uint32_t width = extent - w * WINDOW < WINDOW ? extent - w * WINDOW : WINDOW;
    const uint32_t whole = width / PACK;
    if (whole == 0) {
      return;
    }
    const uint4* __restrict__ q = reinterpret_cast<const uint4*>(elements + w * WINDOW);
#pragma unroll
    for (int j = 0; j < PACKS; ++j) {
      const uint32_t o = j * FIND_SEARCHERS + tid;
      p[j]             = q[o < whole ? o : whole - 1];
    }
  };
  uint32_t w = next_of(0);
  if (w < windows) {
    request(w);
  }
  while (w < windows) {  // uniform
    const uint32_t width = extent - w * WINDOW < WINDOW ? extent - w * WINDOW : WINDOW;
    const uint32_t begin = s_first[w], end = s_first[w + 1];
    const uint32_t whole = width / PACK;
#pragma unroll
    for (int j = 0; j < PACKS; ++j) {
      const uint32_t o = j * FIND_SEARCHERS + tid;
      if (o != whole) {  // (behind the array's end: keys that are left of no answer, or of too many, see below)
        s.pack[find_pack_at(o)] = o < whole ? ordered_pack<CODEC, KeyT>(p[j]) : uint4{~0u, ~0u, ~0u, ~0u};
      }
    }
    if (whole < FIND_WINDOW / 16 && tid < PACK) {
      const uint32_t i               = whole * PACK + tid;
      s.key[find_key_at<KeyT>(i)] = i < width ? ordered_bits<CODEC, KeyT>(elements[w * WINDOW + i]) : ~KeyT{};
    }
    __syncthreads();
    const uint32_t follows = next_of(w + 1);
    if (follows < windows) {
      request(follows);
    }
    const auto search = [&](KeyT value) {
      uint32_t pos = 0;
#pragma unroll
      for (uint32_t step = WINDOW / 2; step != 0; step >>= 1) {  // (counts gaps as well, see find_group_kernel)
        pos += before_answer<CODEC, LEFT>(s.key[pos + find_key_at<KeyT>(step - 1)], value) ? find_key_at<KeyT>(step) : 0u;
      }
      pos += before_answer<CODEC, LEFT>(s.key[pos], value) ? 1u : 0u;
      pos -= pos / (17 * PACK) * PACK;
      return static_cast<KeyT>(w * WINDOW + (pos < width ? pos : width));  // (see find_group_kernel)
    };
    me = find_opaque(tid);
    if constexpr (sizeof(KeyT) == 4) {
#pragma unroll
      for (int k = 0; k < EACH; ++k) {
        if ((k + 1) * FIND_SEARCHERS > begin && k * FIND_SEARCHERS < end) {  // uniform
          const uint32_t o = k * FIND_SEARCHERS + me;
          if (o >= begin && o < end) {
            key[k] = search(key[k]);
          }
        }
      }
    } else {  // (registers are left for two searches of a lane side by side)
#pragma unroll
      for (int k = 0; k < EACH; k += 2) {
        if ((k + 2) * FIND_SEARCHERS > begin && k * FIND_SEARCHERS < end) {  // uniform
          const int k1      = k + 1 < EACH ? k + 1 : k;
          const uint32_t o  = k * FIND_SEARCHERS + me;
          const bool first  = o >= begin && o < end;
          const bool second = k1 != k && o + FIND_SEARCHERS >= begin && o + FIND_SEARCHERS < end;
          if (__ballot(first) != 0 && __ballot(second) != 0) {
            const KeyT a = search(key[k]), b = search(key[k1]);
            key[k]  = first ? a : key[k];
            key[k1] = second ? b : key[k1];
          } else if (first || second) {
            const KeyT a = search(first ? key[k] : key[k1]);
            key[k]       = first ? a : key[k];
            key[k1]      = second ? a : key[k1];
          }
        }
      }
    }
    __syncthreads();
    w = follows;
  }

  // ---- the answers, back to the places of the values ----
  me = find_opaque(tid);
#pragma unroll
  for (int k = 0; k < EACH; ++k) {
    if (k * FIND_SEARCHERS + me < count) {
      s.word[where[k]] = static_cast<uint32_t>(origin) + static_cast<uint32_t>(key[k]);
    }
  }
  __syncthreads();
  for (uint32_t t = tid / FIND_LANES; t < tiles; t += GROUPS) {
    const uint32_t b = s_base[t], e = s_base[t + 1];
    const uint32_t end = e < hi ? e : hi;
    const uint32_t from = b > lo ? b : lo;
    if (end > from + FIND_CROWD) {
      continue;
    }
    uint32_t* const to = answers + static_cast<uint64_t>(t) * FIND_TILE + s_from[t];
    for (uint32_t at = from + sub; at < end; at += FIND_LANES) {
      to[at - b] = s.word[at - lo];
    }
  }
  for (uint32_t c = 0; c < crowds; ++c) {
    const uint32_t t = s_crowd[c];
    const uint32_t b = s_base[t], e = s_base[t + 1];
    const uint32_t from = b > lo ? b : lo, end = e < hi ? e : hi;
    uint32_t* const to  = answers + static_cast<uint64_t>(t) * FIND_TILE + s_from[t];
    for (uint32_t at = from + tid; at < end; at += FIND_SEARCHERS) {
      to[at - b] = s.word[at - lo];
    }
  }
}

// Bound by memory: 14 bytes per value.
__global__ __launch_bounds__(FIND_BLOCK) void find_return_kernel(const uint32_t* __restrict__ answers,
                                                                 const uint16_t* __restrict__ places, uint64_t num_values,
                                                                 int64_t* __restrict__ out)
{
  __shared__ uint32_t s_answer[FIND_TILE];
  const uint32_t tid   = threadIdx.x;
  const uint64_t first = static_cast<uint64_t>(blockIdx.x) * FIND_TILE;
  const uint32_t len   = num_values - first < FIND_TILE ? static_cast<uint32_t>(num_values - first) : FIND_TILE;
  uint16_t place[FIND_ITEMS];
#pragma unroll
  for (int i = 0; i < FIND_ITEMS; ++i) {
    const uint32_t o = i * FIND_BLOCK + tid;
    place[i]         = places[first + (o < len ? o : len - 1)];
  }
#pragma unroll
  for (int i = 0; i < FIND_ITEMS; ++i) {
    const uint32_t o = i * FIND_BLOCK + tid;
    if (o < len) {
      s_answer[o] = answers[first + o];
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < FIND_ITEMS; ++i) {
    const uint32_t o = i * FIND_BLOCK + tid;
    if (o < len) {
      out[first + o] = static_cast<int64_t>(s_answer[place[i]]);
    }
  }
}

struct FindLayout {
  uint64_t part;  // elements
  uint32_t parts, items;
  uint64_t batch;  // values
  uint64_t off_pivots, off_items, off_starts, off_grouped, off_places, off_answers, total;
};

static FindLayout find_layout(int key_bytes, uint64_t n, uint64_t num_values)
{
  FindLayout L{};
  const uint64_t window = FIND_WINDOW / key_bytes;
  const uint64_t even   = align_up((n + FIND_PARTS - 1) / FIND_PARTS, 16);  // (parts start on 16-byte boundaries)
  L.part                = even > window ? even : window;
  L.parts               = static_cast<uint32_t>((n + L.part - 1) / L.part);
  L.batch               = num_values < static_cast<uint64_t>(FIND_TILES) * FIND_TILE ? num_values : static_cast<uint64_t>(FIND_TILES) * FIND_TILE;
  const uint64_t tiles  = (L.batch + FIND_TILE - 1) / FIND_TILE;
  L.items               = static_cast<uint32_t>(FIND_PARTS + L.batch / (FIND_SEARCHERS * FIND_EACH));
  L.off_pivots          = WORKSPACE_ALIGN;
  L.off_items           = L.off_pivots + FIND_PARTS * static_cast<uint64_t>(key_bytes);
  L.off_starts          = L.off_items + align_up(L.items * 4ull, WORKSPACE_ALIGN);
  L.off_grouped         = L.off_starts + align_up(tiles * (FIND_PARTS + 1) * 2, WORKSPACE_ALIGN);
  L.off_places          = L.off_grouped + align_up(L.batch * key_bytes, WORKSPACE_ALIGN);
  L.off_answers         = L.off_places + align_up(L.batch * 2, WORKSPACE_ALIGN);
  L.total               = L.off_answers + align_up(L.batch * 4, WORKSPACE_ALIGN);
  return L;
}

// From 8 MiB of array and 2^16 values on (a caller that can choose takes searchsorted_few_kernel, without a workspace, up to 2^19):
// below, the five launches and parts too few for all CUs (a part has a window at
// least) cost more than direct probes of the caches; and not for values so sparse that reading the whole array for them is the
// larger part.  us per call of `searchsorted`, probes or sorted values / this way, values spread as the array / half of
// them in a thousandth of it:
//   float32    4 MiB,   2^20 values    74 / 94    70 / 82       8 MiB   87 / 77    79 / 71
//              8 MiB,   2^16           75 / 44    57 / 58      32 MiB, 2^24   2267 / 260   914 / 302
//            512 MiB,   2^16          156 / 150  159 / 144     2^20   260 / 164   224 / 180    2^24    752 / 338  1046 / 418
//              1 GiB,   2^20          277 / 264  240 / 273     2^21   360 / 273   322 / 282    2^24    897 / 440  1096 / 492
//   float64    2 MiB,   2^20           60 / 82    55 / 104      8 MiB, 2^16     77 / 50    64 / 60
//              1 GiB,   2^18          272 / 277  264 / 300     2^20   383 / 289   351 / 321    2^24   1552 / 534  1725 / 622
static bool find_pays(int key_bytes, uint64_t n, uint64_t num_values)
{
  const uint64_t bytes = n * key_bytes;
  return bytes >= (8ull << 20) && num_values >= (1ull << 16) &&
         bytes <= num_values * (bytes > (512ull << 20) ? 128 * key_bytes : 4096);
}

template <typename KeyT, int CODEC, bool LEFT>
static int run(const void* sorted_v, uint64_t n, const void* values_v, uint64_t num_values, int64_t* out, unsigned char* ws,
               hipStream_t stream)
{
  const FindLayout L = find_layout(sizeof(KeyT), n, num_values);
  const KeyT* sorted = static_cast<const KeyT*>(sorted_v);
  FindPlan* plan     = reinterpret_cast<FindPlan*>(ws);
  KeyT* pivots       = reinterpret_cast<KeyT*>(ws + L.off_pivots);
  uint32_t* items    = reinterpret_cast<uint32_t*>(ws + L.off_items);
  uint16_t* starts   = reinterpret_cast<uint16_t*>(ws + L.off_starts);
  KeyT* grouped      = reinterpret_cast<KeyT*>(ws + L.off_grouped);
  uint16_t* places   = reinterpret_cast<uint16_t*>(ws + L.off_places);
  uint32_t* answers  = reinterpret_cast<uint32_t*>(ws + L.off_answers);
  {
    ProfileScope prof("find_pivots", stream);
    hipLaunchKernelGGL((find_pivots_kernel<KeyT, CODEC>), dim3(FIND_PARTS / 256), dim3(256), 0, stream, sorted, n, L.part, L.parts,
                       pivots);
  }
  CPN_HIP_TRY(hipGetLastError());
  for (uint64_t first = 0; first < num_values; first += L.batch) {
    const KeyT* values   = static_cast<const KeyT*>(values_v) + first;
    const uint64_t count = num_values - first < L.batch ? num_values - first : L.batch;
    const uint32_t tiles = static_cast<uint32_t>((count + FIND_TILE - 1) / FIND_TILE);
    {
      ProfileScope prof("find_group", stream);
      hipLaunchKernelGGL((find_group_kernel<KeyT, CODEC, LEFT>), dim3(tiles), dim3(FIND_BLOCK), 0, stream, values, count, pivots,
                         L.parts, grouped, places, starts, plan);
    }
    CPN_HIP_TRY(hipGetLastError());
    {
      ProfileScope prof("find_plan", stream);
      hipLaunchKernelGGL(find_plan_kernel, dim3(FIND_PARTS / WAVE), dim3(FIND_BLOCK), 0, stream, starts, tiles,
                         static_cast<uint32_t>(FIND_SEARCHERS * FIND_EACH), plan, items);
    }
    CPN_HIP_TRY(hipGetLastError());
    {
      ProfileScope prof("find_search", stream);
      hipLaunchKernelGGL((find_search_kernel<KeyT, CODEC, LEFT>), dim3((L.items + 7) / 8 * 8), dim3(FIND_SEARCHERS), 0, stream,
                         sorted, n, L.part, grouped, starts, tiles, plan, items, answers);
    }
    CPN_HIP_TRY(hipGetLastError());
    {
      ProfileScope prof("find_return", stream);
      hipLaunchKernelGGL(find_return_kernel, dim3(tiles), dim3(FIND_BLOCK), 0, stream, answers, places, count, out + first);
    }
    CPN_HIP_TRY(hipGetLastError());
  }
  return CPN_OK;
}

template <typename KeyT, int CODEC>
static int run_side(const void* sorted, uint64_t n, const void* values, uint64_t num_values, bool left, int64_t* out,
                    unsigned char* ws, hipStream_t stream)
{
  return left ? run<KeyT, CODEC, true>(sorted, n, values, num_values, out, ws, stream)
              : run<KeyT, CODEC, false>(sorted, n, values, num_values, out, ws, stream);
}

}  // namespace cpn

extern "C" uint64_t cpn_searchsorted_grouped_temp_bytes(int dtype, const void* sorted, uint64_t n, uint64_t num_values)
{
  using namespace cpn;
  const KeyKind k = key_kind(dtype);
  if ((k.bytes != 4 && k.bytes != 8) || k.codec < 0 || k.codec == CODEC_COMPLEX || n >= (1ull << 32) ||
      reinterpret_cast<uintptr_t>(sorted) % 16 != 0 || !find_pays(k.bytes, n, num_values)) {
    return 0;
  }
  const FindLayout L = find_layout(k.bytes, n, num_values);
  return L.part > static_cast<uint64_t>(FIND_WINDOWS) * (FIND_WINDOW / k.bytes) ? 0 : L.total;
}

extern "C" int cpn_searchsorted_grouped(int dtype, const void* sorted, uint64_t n, const void* values, uint64_t num_values, int left,
                                        int64_t* positions_out, void* temp, uint64_t temp_bytes, void* stream)
{
  using namespace cpn;
  const KeyKind k = key_kind(dtype);
  if (k.bytes == 0 || k.codec < 0) {
    return CPN_ERR_DTYPE;
  }
  const uint64_t need = cpn_searchsorted_grouped_temp_bytes(dtype, sorted, n, num_values);
  if (need == 0) {
    return CPN_ERR_UNSUPPORTED;
  }
  if (sorted == nullptr || values == nullptr || positions_out == nullptr) {
    return CPN_ERR_NULL;
  }
  if ((reinterpret_cast<uintptr_t>(values) % static_cast<uint64_t>(k.bytes)) != 0 ||
      (reinterpret_cast<uintptr_t>(positions_out) % 8) != 0) {
    return CPN_ERR_ALIGN;
  }
  if (temp == nullptr || temp_bytes < need || (reinterpret_cast<uintptr_t>(temp) % WORKSPACE_ALIGN) != 0) {
    return CPN_ERR_TEMP;
  }
  unsigned char* ws = static_cast<unsigned char*>(temp);
  hipStream_t s     = static_cast<hipStream_t>(stream);
  const bool l      = left != 0;
  switch (k.codec) {
    case CODEC_UNSIGNED:
      return k.bytes == 8 ? run_side<uint64_t, CODEC_UNSIGNED>(sorted, n, values, num_values, l, positions_out, ws, s)
                          : run_side<uint32_t, CODEC_UNSIGNED>(sorted, n, values, num_values, l, positions_out, ws, s);
    case CODEC_SIGNED:
      return k.bytes == 8 ? run_side<uint64_t, CODEC_SIGNED>(sorted, n, values, num_values, l, positions_out, ws, s)
                          : run_side<uint32_t, CODEC_SIGNED>(sorted, n, values, num_values, l, positions_out, ws, s);
    default:
      return k.bytes == 8 ? run_side<uint64_t, CODEC_FLOAT>(sorted, n, values, num_values, l, positions_out, ws, s)
                          : run_side<uint32_t, CODEC_FLOAT>(sorted, n, values, num_values, l, positions_out, ws, s);
  }
}
