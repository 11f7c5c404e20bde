// Equalised digits: long rows sorted by two scatter passes and one sort in LDS.
//
// The byte digits of a key say little about where it belongs: eight-byte keys take eight passes over
// memory of which two would do if the digits split the keys evenly.  Here a sample of the row makes
// such digits.  The range of the ordered images is cut into cells of equal width (2^k, so that a cell
// is found with a shift), every cell gets a share of 65 536 buckets in proportion to the sampled keys
// in it, and a key's place inside its cell selects one of them:
//
//     bucket(u) = base[cell(u)] + floor(width[cell(u)] * (u's place inside the cell, in [0, 1)))
//
// which never decreases with u, whatever the sample held.  Two stable passes of the scatter kernel
// (onesweep.h) on the low and the high byte of the bucket put the buckets in order; groups of whole
// buckets that fit the LDS of a CU are then sorted by the per-row kernel (lds_row_sort.h).  Buckets
// too large for it are in order already when all their keys are equal (that is what makes most of
// them large: a value that occurs often).
//
// When the sample shows buckets that are too large and hold different keys, or keys so close that the sort in LDS would
// not take them (eq_limits), the row keeps the byte passes.  When that is seen only after the two passes, the byte passes run on what those left, which
// is a stable arrangement of the input and therefore sorts to the same result.
//
// The reference's cub::DeviceRadixSort (src/cupynumeric/sort/cub_sort.cuh:60-182) always runs
// sizeof(key) passes of 8 bits.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "radix_common.h"

namespace cpn {

constexpr uint32_t EQ_BUCKETS = 65536;
// Cells of the table: what the LDS of a CU has left beside the tiles of the scatter pass.
__host__ __device__ constexpr int eq_cell_bits(int key_bytes) { return key_bytes == 8 ? 11 : 10; }
constexpr int EQ_MAX_CELLS      = 2048;
constexpr int EQ_SAMPLE_BLOCK   = 1024;
constexpr int EQ_SAMPLE_ITEMS   = 16;
constexpr uint32_t EQ_SAMPLE    = EQ_SAMPLE_BLOCK * EQ_SAMPLE_ITEMS;
// Buckets every cell gets whatever the sample says: keys in cells that the sample missed (there are about
// n / EQ_SAMPLE of them beyond either end) are spread over that many.
constexpr uint32_t EQ_CELL_MIN = 4;

struct EqualPlan {
  uint32_t mode;     // 1: the row is sorted by equalised digits
  uint32_t failed;   // a bucket too large to be sorted holds different keys: the byte passes take over
  uint32_t n_large;  // entries of the list of large buckets
  uint32_t n_extra;  // further pieces for the LDS sort
  uint32_t n_list;   // pieces for the general LDS sort
  uint32_t lshift;   // left shift that brings the cell number to the top of the word
  uint32_t per_xcd;  // the passes deal their tiles per XCD
  uint64_t origin;   // image where cell 0 starts
  uint64_t last;     // largest distance from the origin inside the table
  alignas(16) uint32_t table[EQ_MAX_CELLS];  // base (low 16 bits) and width (high 16 bits) of every cell
};
// The second word of a sort's workspace says whether the sort deals its tiles per XCD (claim_tile, onesweep.h).  One of a
// device's sorts at a time may: the first launch takes the device's word `order` (null: the sort is not to), the
// last one gives it back.  (Should a launch in between be refused, it stays taken, and later sorts do without.)
constexpr uint64_t HEADER_PER_XCD = 4;
__device__ __forceinline__ uint32_t take_xcd_order(uint32_t* order)
{
  return (order != nullptr && atomicCAS(order, 0u, 1u) == 0u) ? 1u : 0u;
}
__device__ __forceinline__ bool eq_sorted(const EqualPlan* eq) { return eq != nullptr && eq->mode != 0 && eq->failed == 0; }
__device__ __forceinline__ bool eq_failed(const EqualPlan* eq) { return eq != nullptr && eq->mode != 0 && eq->failed != 0; }

// The bucket of an ordered image, with the first `bits` bits of its fraction (at most 15) behind it.  U: uint32_t
// or uint64_t.
template <typename U>
__device__ __forceinline__ uint32_t eq_bucket(U u, U origin, U last, uint32_t lshift, const uint32_t* table, int bits)
{
  constexpr int CB = eq_cell_bits(sizeof(U));
  U v              = u > origin ? static_cast<U>(u - origin) : static_cast<U>(0);
  v                = v < last ? v : last;
  const U w        = static_cast<U>(v << lshift);
  uint32_t cell, frac;
  if constexpr (sizeof(U) == 8) {
    const uint32_t hi = static_cast<uint32_t>(w >> 32);
    cell              = hi >> (32 - CB);
    frac              = static_cast<uint32_t>(w >> (32 - CB));
  } else {
    cell = w >> (32 - CB);
    frac = w << CB;
  }
  const uint32_t e = table[cell];
  return ((e & 0xFFFFu) << bits) + __umulhi(frac, (e >> 16) << bits);
}

// A copy of the plan's scalars in registers and of its table in LDS (made visible by the caller's barrier).
template <typename U>
struct EqualDigits {
  U origin, last;
  uint32_t lshift;
  const uint32_t* table;
  __device__ __forceinline__ uint32_t bucket(U image) const { return eq_bucket<U>(image, origin, last, lshift, table, 0); }
  // with `bits` more of the bucket's fraction
  __device__ __forceinline__ uint32_t fine(U image, int bits) const { return eq_bucket<U>(image, origin, last, lshift, table, bits); }
};
template <typename U>
__device__ __forceinline__ EqualDigits<U> eq_load(const EqualPlan* eq, uint32_t* s_table, int tid, int block)
{
  constexpr int CELLS = 1 << eq_cell_bits(sizeof(U));
  for (int j = tid; j < CELLS / 4; j += block) {
    reinterpret_cast<uint4*>(s_table)[j] = reinterpret_cast<const uint4*>(eq->table)[j];
  }
  return EqualDigits<U>{static_cast<U>(eq->origin), static_cast<U>(eq->last), eq->lshift, s_table};
}

// ---- the sample ---------------------------------------------------------------------------
// EQ_RANGE_SAMPLE keys, one at a pseudo-random place in each of as many equal stretches of the row: every
// workgroup leaves the range of its keys, and every EQ_RANGE_SAMPLE / EQ_SAMPLE-th key is kept.  (One workgroup
// that reads EQ_SAMPLE keys from all over the row by itself takes 46 us: a CU has too few misses in flight.
// Nothing depends on the clearing of the workspace, so this launch does that as well.)
// ranges: lowest and highest image of every workgroup; sample: EQ_SAMPLE images.
constexpr int EQ_GATHER_BLOCK       = 256;
constexpr int EQ_GATHER_GRID        = 1024;
constexpr uint32_t EQ_RANGE_SAMPLE  = EQ_GATHER_BLOCK * EQ_GATHER_GRID;
constexpr uint32_t EQ_SAMPLE_THREADS = EQ_GATHER_BLOCK / (EQ_RANGE_SAMPLE / EQ_SAMPLE);  // of a workgroup
template <typename KeyT, int CODEC>
__global__ __launch_bounds__(EQ_GATHER_BLOCK) void eq_gather_kernel(const KeyT* __restrict__ keys,
                                                                    uint64_t seg,
                                                                    KeyT* __restrict__ ranges,
                                                                    KeyT* __restrict__ sample,
                                                                    uint4* __restrict__ clear,
                                                                    uint64_t n_clear,
                                                                    uint4* __restrict__ clear2,
                                                                    uint64_t n_clear2,
                                                                    uint32_t* order)
{
  constexpr int WAVES = EQ_GATHER_BLOCK / WAVE;
  __shared__ KeyT s_lo[WAVES], s_hi[WAVES];
  const uint32_t tid   = threadIdx.x;
  const uint32_t s     = blockIdx.x * EQ_GATHER_BLOCK + tid;
  const uint64_t begin = (static_cast<uint64_t>(s) * seg) / EQ_RANGE_SAMPLE;
  const uint64_t end   = (static_cast<uint64_t>(s + 1) * seg) / EQ_RANGE_SAMPLE;
  uint32_t h           = s * 0x9E3779B1u;
  h ^= h >> 15;
  h *= 0x85EBCA6Bu;
  h ^= h >> 13;
  // seg >= EQ_RANGE_SAMPLE: no stretch is empty
  const KeyT u = ordered_bits<CODEC, KeyT>(keys[begin + ((static_cast<uint64_t>(h) * (end - begin)) >> 32)]);
  for (uint64_t i = s; i < n_clear; i += EQ_RANGE_SAMPLE) {
    clear[i] = make_uint4(0u, i == 0 ? take_xcd_order(order) : 0u, 0u, 0u);  // (the workspace, from its head on)
  }
  for (uint64_t i = s; i < n_clear2; i += EQ_RANGE_SAMPLE) {
    clear2[i] = make_uint4(0u, 0u, 0u, 0u);
  }
  KeyT lo = u, hi = u;
#pragma unroll
  for (int d = 1; d < WAVE; d <<= 1) {
    const KeyT a = static_cast<KeyT>(__shfl_xor(static_cast<unsigned long long>(lo), d, WAVE));
    const KeyT b = static_cast<KeyT>(__shfl_xor(static_cast<unsigned long long>(hi), d, WAVE));
    lo           = a < lo ? a : lo;
    hi           = b > hi ? b : hi;
  }
  if (tid % WAVE == 0) {
    s_lo[tid / WAVE] = lo;
    s_hi[tid / WAVE] = hi;
  }
  // (neighbouring threads' keys come from neighbouring stretches: every 16th is spread over the row as all are)
  if (tid % (EQ_GATHER_BLOCK / EQ_SAMPLE_THREADS) == 0) {
    sample[s / (EQ_GATHER_BLOCK / EQ_SAMPLE_THREADS)] = u;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < WAVES; ++w) {
      lo = s_lo[w] < lo ? s_lo[w] : lo;
      hi = s_hi[w] > hi ? s_hi[w] : hi;
    }
    ranges[2 * blockIdx.x]     = lo;
    ranges[2 * blockIdx.x + 1] = hi;
  }
}

// ---- the plan -----------------------------------------------------------------------------
// One workgroup: the range, the cells, the shares, and whether the row is one for equalised digits.  What the LDS
// sort cannot take costs far more than the two passes save (a row whose pieces all go to the general sort 1.6 times
// the byte passes, one that fails when it has been sorted as much), so the row keeps the byte passes
//   - when fewer than EQ_MIN_BYTES bytes of the sampled images vary (that many byte passes are as fast);
//   - when a bucket that `crowd` and more of the sampled keys fall into holds different ones;
//   - when such a bucket holds one key, and its cell other keys as well that do not crowd theirs (a value that
//     occurs often among keys that are close to it: some are bound to share its bucket);
//   - when the cells of floats are half an octave or wider: rows that span zero, or hold one, whose images reach over
//     the magnitudes that do not occur (2050 octaves for both signs, cells of two).  A density that falls off inside such
//     a cell leaves a few buckets too large, and those of the tails hold too few sampled keys to show it: of 2^26 normal
//     keys a bucket at 2.0 holds 11 100, and 45 10^6 keys of three times that spread failed in 15 of 16 rows, of a
//     logistic distribution in 2, 2^26 of the latter in 15; accepted and then sorted again they took 1.65 times the byte
//     passes (which 2^25 normal keys, that would fit, keep as well: 1290 us instead of 740);
//   - when `dense` and more sampled keys outside such buckets fall into 2^group_log2 neighbouring buckets: the density
//     varies too much inside a cell;
//   - when `close` and more ordered pairs of sampled keys share a bucket (16384 evenly spread keys: 4700): the keys
//     stand in clusters narrower than a bucket, e.g. a few thousand groups of neighbouring numbers;
//   - when `equal` and more sampled keys find one in their bucket that would share a bin of the LDS sort with them:
//     values repeat, or stand in clusters so narrow, that they crowd the bins.
// (No sample sees a handful of neighbours of a value that occurs often: such a row fails after its two passes.)
// `veto`: a word that says (non-zero) that the sort runs otherwise.
struct EqualLimits {
  uint32_t crowd, group_log2, dense, close, equal;
};
// n: length of the row; fits / tile: keys of a bucket that the general sort and the LDS sort can take.
inline EqualLimits eq_limits(uint64_t n, uint32_t fits, uint32_t tile)
{
  EqualLimits l{};
  // A bucket that just fits holds `mean` sampled keys on average (5 of 2^25 keys, 2.5 of 2^26), and one of evenly
  // spread keys 0.29: three and a half standard deviations above the former are a crowd, and never fewer than seven
  // (which one row in 700 of the latter has in some bucket).
  const double mean = static_cast<double>(fits) * EQ_SAMPLE / static_cast<double>(n);
  l.crowd           = static_cast<uint32_t>(mean + 3.5 * __builtin_sqrt(mean));
  l.crowd           = l.crowd > 7 ? l.crowd : 7;
  // Windows of as many buckets (n / 2^21, a power of two) as hold 60 to 120 sampled keys at three quarters of what fits,
  // and 4.6 to 9.1 of evenly spread ones.
  l.group_log2 = 4;
  while (l.group_log2 < 7 && (1ull << (21 + l.group_log2)) < n) {
    ++l.group_log2;
  }
  l.dense = static_cast<uint32_t>(((3ull * fits * EQ_SAMPLE / 4) << l.group_log2) / n) + 1;
  // the bucket of an average key: four fifths of the tile, but nine twentieths of a sampled key, which evenly spread ones
  // stay well below
  const uint64_t share = 4ull * tile * EQ_SAMPLE * EQ_SAMPLE / (5 * n);
  l.close              = static_cast<uint32_t>(share > EQ_SAMPLE * 9 / 20 ? share : EQ_SAMPLE * 9 / 20);
  // Every key one of 32 equal ones, or a smaller share of them one of more (a pair counts once; of three keys in a bucket,
  // two of them equal, it depends on the third, so that rows near the limit may go either way).
  l.equal = static_cast<uint32_t>((16ull * EQ_SAMPLE * EQ_SAMPLE) / n) + 1;
  return l;
}
constexpr int EQ_MIN_BYTES = 5;
// Cells of half an octave (2^52 images of 8-byte floats) and wider: see above.
constexpr uint32_t EQ_MAX_FLOAT_SHIFT = 51;
constexpr int EQ_MARK_BITS = 11;  // a bucket of evenly spread keys is 910 (2^25 keys) or 1820 bins (2^26) of the LDS sort
template <typename KeyT, int CODEC>
__global__ __launch_bounds__(EQ_SAMPLE_BLOCK) void eq_plan_kernel(const KeyT* __restrict__ ranges,
                                                                  const KeyT* __restrict__ sample,
                                                                  const EqualLimits limits,
                                                                  const uint32_t* __restrict__ veto,
                                                                  const uint32_t* __restrict__ per_xcd,
                                                                  EqualPlan* __restrict__ eq)
{
  constexpr int CB           = eq_cell_bits(sizeof(KeyT));
  constexpr int CELLS        = 1 << CB;
  constexpr uint32_t EXTRA   = CELLS / 16;  // cells beyond the sampled range, at either end
  constexpr int WAVES        = EQ_SAMPLE_BLOCK / WAVE;
  constexpr int CELLS_THREAD = CELLS / EQ_SAMPLE_BLOCK;
  static_assert(CELLS % EQ_SAMPLE_BLOCK == 0 && CELLS <= EQ_MAX_CELLS, "whole cells per thread");
  static_assert(EQ_GATHER_GRID == EQ_SAMPLE_BLOCK, "one range per thread");
  __shared__ __align__(16) uint32_t s_count[EQ_BUCKETS / 2];  // sampled keys per bucket, two counters per word
  __shared__ uint32_t s_table[CELLS];
  __shared__ uint64_t s_lo[WAVES], s_hi[WAVES], s_and[WAVES], s_or[WAVES];
  __shared__ uint32_t s_wsum[WAVES];
  __shared__ uint32_t s_cells_crowded[CELLS / 32], s_cells_other[CELLS / 32];  // one bit per cell
  __shared__ uint32_t s_group[EQ_BUCKETS / 16 / 2];  // sampled keys per window of buckets, two counters per word
  __shared__ uint32_t s_dense, s_close, s_equal;
  if (veto != nullptr && *veto != 0) {
    return;  // (the plan is cleared: mode 0)
  }
  const int tid  = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wave = tid / WAVE;

  KeyT u[EQ_SAMPLE_ITEMS];
#pragma unroll
  for (int i = 0; i < EQ_SAMPLE_ITEMS; ++i) {
    u[i] = sample[i * EQ_SAMPLE_BLOCK + tid];
  }
  uint64_t lo = ranges[2 * tid], hi = ranges[2 * tid + 1];
  for (int j = tid; j < static_cast<int>(EQ_BUCKETS / 8); j += EQ_SAMPLE_BLOCK) {
    reinterpret_cast<uint4*>(s_count)[j] = make_uint4(0u, 0u, 0u, 0u);
  }
  for (int j = tid; j < CELLS; j += EQ_SAMPLE_BLOCK) {
    s_table[j] = 0;
  }
  if (tid < CELLS / 32) {
    s_cells_crowded[tid] = 0;
    s_cells_other[tid]   = 0;
  }
  for (int j = tid; j < static_cast<int>(EQ_BUCKETS / 32); j += EQ_SAMPLE_BLOCK) {
    s_group[j] = 0;
  }
  if (tid == 0) {
    s_dense = 0;
    s_close = 0;
    s_equal = 0;
  }
  KeyT bits_and = static_cast<KeyT>(~static_cast<KeyT>(0)), bits_or = 0;
#pragma unroll
  for (int i = 0; i < EQ_SAMPLE_ITEMS; ++i) {
    bits_and &= u[i];
    bits_or |= u[i];
  }
  bits_and = wave_reduce_and_dpp(bits_and);
  bits_or  = wave_reduce_or_dpp(bits_or);
#pragma unroll
  for (int d = 1; d < WAVE; d <<= 1) {
    const uint64_t a = __shfl_xor(static_cast<unsigned long long>(lo), d, WAVE);
    const uint64_t b = __shfl_xor(static_cast<unsigned long long>(hi), d, WAVE);
    lo               = a < lo ? a : lo;
    hi               = b > hi ? b : hi;
  }
  if (lane == 0) {
    s_lo[wave]  = lo;
    s_hi[wave]  = hi;
    s_and[wave] = bits_and;
    s_or[wave]  = bits_or;
  }
  __syncthreads();
  uint64_t all_and = ~0ull, all_or = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    lo = s_lo[w] < lo ? s_lo[w] : lo;
    hi = s_hi[w] > hi ? s_hi[w] : hi;
    all_and &= s_and[w];
    all_or |= s_or[w];
  }
  int busy = 0;
#pragma unroll
  for (int p = 0; p < static_cast<int>(sizeof(KeyT)); ++p) {
    busy += (((all_and ^ all_or) >> (8 * p)) & 0xFFu) != 0 ? 1 : 0;
  }
  if (busy < EQ_MIN_BYTES) {
    return;  // uniform; mode 0
  }
  // The smallest cells with which the sampled range and EXTRA cells at either end (one more for the
  // rounding of the origin) fit the table.
  uint32_t shift = 0;
  while (((hi - lo) >> shift) > static_cast<uint64_t>(CELLS - 2 * EXTRA - 2)) {
    ++shift;
  }
  if (CODEC == CODEC_FLOAT && shift >= EQ_MAX_FLOAT_SHIFT) {
    return;  // uniform; mode 0
  }
  constexpr uint32_t TOP  = 8 * sizeof(KeyT) - CB;  // (shift <= TOP: the whole range is CELLS cells then)
  const uint64_t below    = static_cast<uint64_t>(EXTRA) << shift;
  const uint64_t origin   = (lo > below ? lo - below : 0ull) >> shift << shift;
  const uint64_t all      = sizeof(KeyT) == 8 ? ~0ull : 0xFFFFFFFFull;
  const uint64_t last     = shift >= TOP ? all : (static_cast<uint64_t>(CELLS) << shift) - 1;
  const uint32_t lshift   = shift >= TOP ? 0u : TOP - shift;

#pragma unroll
  for (int i = 0; i < EQ_SAMPLE_ITEMS; ++i) {
    const uint64_t v = static_cast<uint64_t>(u[i]) - origin;  // lo >= origin
    atomicAdd(&s_table[static_cast<uint32_t>((v < last ? v : last) >> (TOP - lshift))], 1u);
  }
  __syncthreads();
  // base[c] = EQ_CELL_MIN * c + (sampled keys before cell c) * (the remaining buckets) / EQ_SAMPLE
  {
    uint32_t c[CELLS_THREAD], sum = 0;
#pragma unroll
    for (int j = 0; j < CELLS_THREAD; ++j) {
      c[j] = s_table[tid * CELLS_THREAD + j];
      sum += c[j];
    }
    const uint32_t incl = wave_inclusive_scan(sum, lane);
    if (lane == WAVE - 1) {
      s_wsum[wave] = incl;
    }
    __syncthreads();
    uint32_t run = incl - sum;
    for (int w = 0; w < wave; ++w) {
      run += s_wsum[w];
    }
    constexpr uint32_t SHARED = EQ_BUCKETS - EQ_CELL_MIN * CELLS;
    static_assert(EQ_SAMPLE == 16384 && SHARED < (1u << 17), "products of 32 bits");
#pragma unroll
    for (int j = 0; j < CELLS_THREAD; ++j) {
      const uint32_t cell = static_cast<uint32_t>(tid * CELLS_THREAD + j);
      const uint32_t base = EQ_CELL_MIN * cell + (run * SHARED) / EQ_SAMPLE;
      run += c[j];
      const uint32_t next = EQ_CELL_MIN * (cell + 1) + (run * SHARED) / EQ_SAMPLE;
      s_table[cell]       = base | ((next - base) << 16);  // (the widest cell: 65536 - 4 * (CELLS - 1))
      eq->table[cell]     = s_table[cell];
    }
  }
  __syncthreads();
  // ---- buckets that look too large: do they hold one key each? ----
  uint32_t bucket[EQ_SAMPLE_ITEMS];  // and, behind it, EQ_MARK_BITS bits of the place in it
  uint32_t second = 0;  // bit i: key i was the second to arrive in its bucket
#pragma unroll
  for (int i = 0; i < EQ_SAMPLE_ITEMS; ++i) {
    bucket[i] = eq_bucket<KeyT>(u[i], static_cast<KeyT>(origin), static_cast<KeyT>(last), lshift, s_table, EQ_MARK_BITS);
    const uint32_t b    = bucket[i] >> EQ_MARK_BITS;
    const uint32_t half = 16 * (b % 2);
    const uint32_t was  = atomicAdd(&s_count[b / 2], 1u << half);  // (EQ_SAMPLE < 2^16: no carry)
    second |= ((was >> half) & 0xFFFFu) == 1 ? 1u << i : 0u;
  }
  __syncthreads();
  uint32_t crowded = 0, shared = 0, pairs = 0;
#pragma unroll
  for (int i = 0; i < EQ_SAMPLE_ITEMS; ++i) {
    const uint32_t b = bucket[i] >> EQ_MARK_BITS;
    const uint32_t c = (s_count[b / 2] >> (16 * (b % 2))) & 0xFFFFu;
    if (c >= limits.crowd) {
      crowded |= 1u << i;
    } else {
      const uint32_t g = b >> limits.group_log2;
      atomicAdd(&s_group[g / 2], 1u << (16 * (g % 2)));
      shared |= c >= 2 ? 1u << i : 0u;
      pairs += c - 1;
    }
    const uint64_t v    = static_cast<uint64_t>(u[i]) - origin;
    const uint32_t cell = static_cast<uint32_t>((v < last ? v : last) >> (TOP - lshift));
    uint32_t* const map = c >= limits.crowd ? s_cells_crowded : s_cells_other;
    if (((map[cell / 32] >> (cell % 32)) & 1u) == 0) {  // (most find the bit set)
      atomicOr(&map[cell / 32], 1u << (cell % 32));
    }
  }
  __syncthreads();
  // (some key of a bucket leaves a mark there; the others compare: 16 bits of the key itself in a crowded bucket, the
  // place in the others)
  uint16_t* const s_mark = reinterpret_cast<uint16_t*>(s_count);
  auto mark_of           = [&](int i) -> uint16_t {
    return ((crowded >> i) & 1u) != 0 ? static_cast<uint16_t>((static_cast<uint64_t>(u[i]) * 0x9E3779B97F4A7C15ull) >> 48)
                                      : static_cast<uint16_t>(bucket[i] & ((1u << EQ_MARK_BITS) - 1));
  };
#pragma unroll
  for (int i = 0; i < EQ_SAMPLE_ITEMS; ++i) {
    if (((crowded | shared) >> i) & 1u) {
      s_mark[bucket[i] >> EQ_MARK_BITS] = mark_of(i);
    }
  }
  uint32_t most = 0;
  for (int j = tid; j < static_cast<int>(EQ_BUCKETS / 32); j += EQ_SAMPLE_BLOCK) {
    const uint32_t two = s_group[j];
    most               = (two & 0xFFFFu) > most ? (two & 0xFFFFu) : most;
    most               = (two >> 16) > most ? (two >> 16) : most;
  }
  __syncthreads();
  // Keys with another one of their place in the bucket: those that find their own mark, but for one in every bucket of several
  // (whose mark it is), i.e. for as many as arrived second.
  int no         = 0;
  uint32_t equal = 0;
#pragma unroll
  for (int i = 0; i < EQ_SAMPLE_ITEMS; ++i) {
    const bool same = s_mark[bucket[i] >> EQ_MARK_BITS] == mark_of(i);
    no |= (((crowded >> i) & 1u) != 0 && !same) ? 1 : 0;
    equal += (((shared >> i) & 1u) != 0 && same) ? 1u : 0u;
  }
  equal -= __popc(shared & second);  // (of the thread: modulo 2^32)
  if (tid < CELLS / 32 && (s_cells_crowded[tid] & s_cells_other[tid]) != 0) {
    no = 1;
  }
  equal = static_cast<uint32_t>(__shfl(wave_inclusive_sum_dpp(equal), WAVE - 1, WAVE));
  pairs = static_cast<uint32_t>(__shfl(wave_inclusive_sum_dpp(pairs), WAVE - 1, WAVE));
  if (lane == 0) {
    atomicAdd(&s_equal, equal);
    atomicAdd(&s_close, pairs);
  }
  if (most >= limits.dense) {
    s_dense = 1;
  }
  const int any   = __syncthreads_or(no);  // (a statement of its own: the words below are read behind the barrier)
  const int mixed = any | (s_dense != 0 ? 1 : 0) | (s_close >= limits.close ? 1 : 0) | (s_equal >= limits.equal ? 1 : 0);
  if (tid == 0) {
    eq->origin  = origin;
    eq->last    = last;
    eq->lshift  = lshift;
    eq->per_xcd = *per_xcd;
    eq->mode    = mixed != 0 ? 0u : 1u;
  }
}

// ---- histograms of the two digits: hist[0..255] low byte, hist[256..511] high byte of the bucket ----
// (A launch of its own makes offsets of them: the fences with which the last of these workgroups could do it
// write the L2s back 2048 times, 0.14 -> 0.45 ms for 2^26 keys.)
// SPECIALS as in histogram_kernel: float keys of keys-only sorts, is there a NaN or a -0.0?
// grid: chunks of `chunk` keys (a multiple of EQ_HIST_BLOCK * 16 bytes).
constexpr int EQ_HIST_BLOCK  = 256;
constexpr int EQ_HIST_COPIES = 8;
template <typename KeyT, int CODEC, bool SPECIALS>
__global__ __launch_bounds__(EQ_HIST_BLOCK) void eq_histogram_kernel(const KeyT* __restrict__ keys,
                                                                     uint32_t* __restrict__ hist,
                                                                     uint64_t seg,
                                                                     uint64_t chunk,
                                                                     const EqualPlan* __restrict__ eq,
                                                                     uint32_t* __restrict__ specials)
{
  constexpr int VEC   = 16 / sizeof(KeyT);
  constexpr int CELLS = 1 << eq_cell_bits(sizeof(KeyT));
  __shared__ uint32_t s_hist[2 * RADIX * EQ_HIST_COPIES];
  __shared__ __align__(16) uint32_t s_table[CELLS];
  if (eq->mode == 0) {
    return;
  }
  const int tid = threadIdx.x;
  for (int j = tid; j < 2 * RADIX * EQ_HIST_COPIES; j += EQ_HIST_BLOCK) {
    s_hist[j] = 0;
  }
  const EqualDigits<KeyT> digits = eq_load<KeyT>(eq, s_table, tid, EQ_HIST_BLOCK);
  __syncthreads();
  const uint64_t begin = static_cast<uint64_t>(blockIdx.x) * chunk;
  const uint64_t end   = begin + chunk < seg ? begin + chunk : seg;
  const uint32_t copy  = tid % EQ_HIST_COPIES;
  bool special         = false;
  auto count           = [&](KeyT raw) {
    const KeyT image = ordered_bits<CODEC, KeyT>(raw);
    if constexpr (SPECIALS) {
      special |= image != sign_flip(raw);
    }
    const uint32_t b = digits.bucket(image);
    atomicAdd(&s_hist[(b & 0xFFu) * EQ_HIST_COPIES + copy], 1u);
    atomicAdd(&s_hist[(RADIX + (b >> 8)) * EQ_HIST_COPIES + copy], 1u);
  };
  if (begin < end) {
    // elements before the first 16-byte boundary, 128-bit loads over the middle, elements after it
    const KeyT* p        = keys;
    const uintptr_t addr = reinterpret_cast<uintptr_t>(p + begin);
    uint64_t head        = ((16u - (addr & 15u)) & 15u) / sizeof(KeyT);
    head                 = head < end - begin ? head : end - begin;
    if (static_cast<uint64_t>(tid) < head) {
      count(p[begin + tid]);
    }
    const uint64_t vbegin = begin + head;
    const uint64_t nvec   = (end - vbegin) / VEC;
    const uint4* vp       = reinterpret_cast<const uint4*>(p + vbegin);
    uint64_t v            = tid;
    for (; v + 3 * EQ_HIST_BLOCK < nvec; v += 4 * EQ_HIST_BLOCK) {
      const uint4 q0 = vp[v], q1 = vp[v + EQ_HIST_BLOCK], q2 = vp[v + 2 * EQ_HIST_BLOCK], q3 = vp[v + 3 * EQ_HIST_BLOCK];
      KeyT k[4 * VEC];
      __builtin_memcpy(k, &q0, 16);
      __builtin_memcpy(k + VEC, &q1, 16);
      __builtin_memcpy(k + 2 * VEC, &q2, 16);
      __builtin_memcpy(k + 3 * VEC, &q3, 16);
#pragma unroll
      for (int j = 0; j < 4 * VEC; ++j) {
        count(k[j]);
      }
    }
    for (; v < nvec; v += EQ_HIST_BLOCK) {
      const uint4 q = vp[v];
      KeyT k[VEC];
      __builtin_memcpy(k, &q, 16);
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        count(k[j]);
      }
    }
    for (uint64_t i = vbegin + nvec * VEC + tid; i < end; i += EQ_HIST_BLOCK) {
      count(p[i]);
    }
  }
  if constexpr (SPECIALS) {
    const int any = __syncthreads_or(special ? 1 : 0);
    if (any != 0 && tid == 0) {
      __hip_atomic_store(specials, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  } else {
    __syncthreads();
  }
  for (int j = tid; j < 2 * RADIX; j += EQ_HIST_BLOCK) {
    uint32_t c = 0;
#pragma unroll
    for (int r = 0; r < EQ_HIST_COPIES; ++r) {
      c += s_hist[j * EQ_HIST_COPIES + r];
    }
    if (c != 0) {
      __hip_atomic_fetch_add(&hist[j], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// ---- what the LDS sort is given -----------------------------------------------------------
// Segment w of the row is the buckets that start in [w * stride, (w + 1) * stride).  One that fits
// `capacity` keys is one piece of work, segs[w] (first element, length; 0: none).  Of a longer one everything but
// the last bucket is (no other bucket of it reaches past the stretch), and the last bucket is another one, in
// extras[]; or, when it does not fit either, an entry of the general sort's list, which takes up to `medium` keys,
// or of the list of large buckets, in parts.
constexpr int EQ_SEGMENT_BLOCK    = 64;
constexpr uint32_t EQ_LARGE_PART  = 16384;  // elements of a part
struct EqualLarge {
  uint32_t begin, length, first;  // a part of a bucket, and the bucket's first element
};
// Entries that the list can need: a part per EQ_LARGE_PART elements and one more per bucket.
__host__ __device__ constexpr uint64_t eq_large_entries(uint64_t seg, uint64_t capacity)
{
  return seg / EQ_LARGE_PART + seg / capacity + 2;  // (of more than `capacity` keys each)
}

// A thread per segment start: four probes 256 elements apart at once, then bisection (about a dozen dependent
// reads; a wavefront per start, probing 16 and then 64 places, reads so many more lines that it took 70 us
// instead of 25 for 2^26 keys).  The last thread of a workgroup finds the end of the last segment.
constexpr int EQ_SEGMENT_GROUP = EQ_SEGMENT_BLOCK - 1;
template <typename KeyT, int CODEC>
__global__ __launch_bounds__(EQ_SEGMENT_BLOCK) void eq_segments_kernel(const KeyT* __restrict__ keys,
                                                                       uint32_t n,
                                                                       uint32_t segments,
                                                                       uint32_t stride,
                                                                       uint32_t capacity,
                                                                       uint32_t medium,
                                                                       uint32_t max_entries,
                                                                       const uint32_t* __restrict__ status,
                                                                       EqualPlan* __restrict__ eq,
                                                                       uint2* __restrict__ segs,
                                                                       uint2* __restrict__ extras,
                                                                       uint2* __restrict__ list,
                                                                       EqualLarge* __restrict__ large)
{
  constexpr int CELLS = 1 << eq_cell_bits(sizeof(KeyT));
  __shared__ __align__(16) uint32_t s_table[CELLS];
  __shared__ uint32_t s_start[EQ_SEGMENT_BLOCK];
  if (eq->mode == 0 || *status != 0) {
    return;  // (a pass that gave up leaves keys in no order)
  }
  const EqualDigits<KeyT> digits = eq_load<KeyT>(eq, s_table, threadIdx.x, EQ_SEGMENT_BLOCK);
  __syncthreads();
  const uint32_t tid = threadIdx.x;
  auto bucket_at     = [&](uint32_t i) { return digits.bucket(ordered_bits<CODEC, KeyT>(keys[i])); };
  // The first element in (lo, hi] whose bucket is not below b, given that lo's is and that hi's is not (or
  // hi == n).  The keys are in bucket order.
  auto first_not_below = [&](uint32_t b, uint32_t lo, uint32_t hi) -> uint32_t {
    for (uint32_t step = 256; hi - lo > step; step *= 4) {
      bool below[4];
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) {
        const uint64_t at = lo + static_cast<uint64_t>(k + 1) * step;
        below[k]          = at < hi && bucket_at(static_cast<uint32_t>(at < hi ? at : hi - 1)) < b;
      }
      const uint32_t k = below[0] ? (below[1] ? (below[2] ? (below[3] ? 4u : 3u) : 2u) : 1u) : 0u;
      if (k < 4) {
        const uint64_t top = lo + static_cast<uint64_t>(k + 1) * step;
        hi                 = top < hi ? static_cast<uint32_t>(top) : hi;
        lo += k * step;
        break;
      }
      lo += 4 * step;
    }
    while (hi - lo > 1) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (bucket_at(mid) < b) {
        lo = mid;
      } else {
        hi = mid;
      }
    }
    return hi;
  };
  const uint32_t w = blockIdx.x * EQ_SEGMENT_GROUP + tid;
  const uint64_t p = static_cast<uint64_t>(w) * stride;
  uint32_t begin   = p < n ? static_cast<uint32_t>(p) : n;  // the first bucket start at or after p
  if (begin != 0 && begin != n) {
    begin = first_not_below(bucket_at(begin - 1) + 1, begin - 1, n);
  }
  s_start[tid] = begin;
  __syncthreads();
  if (tid == EQ_SEGMENT_GROUP || w >= segments) {
    return;
  }
  const uint32_t p1  = n - static_cast<uint32_t>(p) <= stride ? n : static_cast<uint32_t>(p) + stride;
  const uint32_t end = s_start[tid + 1];
  uint2 first        = make_uint2(begin, end > begin ? end - begin : 0u);
  if (first.y > capacity) {
    // the last bucket: it starts before p1, and everything before it ends there
    const uint32_t b    = bucket_at(end - 1);
    const uint32_t from = bucket_at(begin) >= b ? begin : first_not_below(b, begin, p1 < end ? p1 : end);
    first.y             = from - begin;
    const uint2 second  = make_uint2(from, end - from);
    if (second.y <= medium) {  // (no more than one per segment: the lists cannot overflow)
      const bool fits   = second.y <= capacity;
      const uint32_t at = __hip_atomic_fetch_add(fits ? &eq->n_extra : &eq->n_list, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      (fits ? extras : list)[at] = second;
    } else {
      const uint32_t parts = (second.y + EQ_LARGE_PART - 1) / EQ_LARGE_PART;
      const uint32_t at    = __hip_atomic_fetch_add(&eq->n_large, parts, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      for (uint32_t j = 0; j < parts && at + j < max_entries; ++j) {
        const uint32_t off = j * EQ_LARGE_PART;
        large[at + j] = EqualLarge{from + off, second.y - off < EQ_LARGE_PART ? second.y - off : EQ_LARGE_PART, from};
      }
    }
  }
  segs[w] = first;
}

// ---- the LDS sort -------------------------------------------------------------------------
// The pieces, dealt to the workgroups in turn.  A piece is split into EQ_BINS bins that cover its buckets evenly
// (the bucket's fraction goes on where its number ends) and every key is put into its bin in the order in which
// the counting atomic saw it; then the thread that owns a bin puts the few keys of it in order.  Equal keys go
// by place (plain sorts: they are the same bits) or by position.  Bins of more than EQ_BIN_LIMIT keys (values that
// repeat) are put in order by a wave each, larger ones by the whole workgroup one after the other: a thread compares
// its key with all of the bin.
// Pieces that hold a NaN or a -0.0, more than a workgroup's worth of keys in a bin, or too many bins for the workgroup, go
// on the general sort's list.
// Bound by vector instructions: 2^26 float64 keys 0.40 ms (1.07 GB).  Comparing every key with the others of its bin, as
// lds_row_sort_kernel does, takes 156 of them per key (0.50 ms in that kernel when this one took 0.46, with a grid that
// did not fit at once).
constexpr int EQ_SORT_BLOCK       = 512;
constexpr int EQ_SORT_ITEMS       = 6;
// Waves per SIMD, and with them workgroups per CU (three).  At 80 registers a dozen values are spilled, addresses and
// bounds of the loop over the pieces for the most part; without that (108 registers, two workgroups) 2^26 float64 keys
// take 1409 us instead of 1368, with positions 1748 instead of 1672.
constexpr int EQ_SORT_WAVES       = 6;
constexpr int EQ_SORT_GROUPS      = EQ_SORT_WAVES * 4 / (EQ_SORT_BLOCK / WAVE);
constexpr int EQ_SORT_TILE        = EQ_SORT_BLOCK * EQ_SORT_ITEMS;
constexpr int EQ_BINS             = 4096;  // two 16-bit counters per word
// (Evenly spread keys: 0.56 in a bin on average.  With 24, 2^26 float64 keys of which half occur 20 times each took 4.2 ms
// with positions, whose order the counting atomic leaves mixed; 2.3 now, the byte passes 3.2.)
constexpr uint32_t EQ_BIN_LIMIT   = 8;
// Bins for the whole workgroup, one after the other: with more of them the general sort is the faster one.  (Pieces of
// many sparse buckets and a full one, whose keys share a few bins: 2^25 keys with a dozen such pieces took 802 us
// without this limit, 742 with it.)
constexpr uint32_t EQ_LARGE_BINS  = 6;
constexpr int EQ_FRACTION_BITS    = 14;    // of a bucket, for the bins

template <typename KeyT, int CODEC, bool HAS_IDX>
struct EqualSort {
  static constexpr int BLOCK = EQ_SORT_BLOCK;
  static constexpr int WAVES = BLOCK / WAVE;
  static constexpr int WORDS = EQ_BINS / 2 / BLOCK;  // words of counters per thread
  static_assert(WORDS == 4, "one 16-byte access");
  static constexpr uint32_t CROWDED = EQ_SORT_TILE / (EQ_BIN_LIMIT + 1);  // bins of more than EQ_BIN_LIMIT keys, at most
  struct Shared {
    alignas(16) KeyT keys[EQ_SORT_TILE];
    alignas(16) uint32_t bins[EQ_BINS / 2 + 4];
    uint16_t idx[HAS_IDX ? EQ_SORT_TILE : 1];
    uint32_t wsum[WAVES];
    uint32_t n_crowded, n_large;
    uint16_t crowded[CROWDED];  // bins for a wave, and from the end on those for the workgroup
  };
  // The image of a key that is neither a NaN nor a -0.0, and back.
  static __device__ __forceinline__ KeyT image(KeyT k)
  {
    return CODEC == CODEC_FLOAT ? sign_flip<KeyT>(k) : ordered_bits<CODEC == CODEC_FLOAT ? CODEC_UNSIGNED : CODEC, KeyT>(k);
  }
  static __device__ __forceinline__ KeyT unimage(KeyT u)
  {
    return CODEC == CODEC_FLOAT ? sign_unflip<KeyT>(u) : ordered_bits<CODEC == CODEC_FLOAT ? CODEC_UNSIGNED : CODEC, KeyT>(u);
  }
  // Returns whether the piece has been sorted; `len` in (BLOCK * (R - 1), BLOCK * R].
  template <int R>
  static __device__ __forceinline__ bool piece(Shared& sh, const KeyT* keys, KeyT* out, const uint32_t* pos, int64_t* idx_out,
                                               int64_t offset, uint32_t len, const EqualDigits<KeyT>& eq)
  {
    const uint32_t tid  = threadIdx.x;
    const uint32_t lane = tid % WAVE;
    auto has            = [&](int i) { return i < R - 1 || i * BLOCK + tid < len; };
    KeyT u[R];
    int odd = 0;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const uint32_t o = i * BLOCK + tid;
      u[i]             = keys[i < R - 1 || o < len ? o : len - 1];
    }
    // the buckets of the first and the last key bound those of the piece
    const uint32_t b0 = eq.bucket(ordered_bits<CODEC, KeyT>(keys[0]));
    const uint32_t b1 = eq.bucket(ordered_bits<CODEC, KeyT>(keys[len - 1]));
    const uint32_t origin = b0 << EQ_FRACTION_BITS;
    // fine steps of the piece (at least 2^EQ_FRACTION_BITS > EQ_BINS) to bins, rounded down: below EQ_BINS for all
    static_assert((1 << EQ_FRACTION_BITS) > EQ_BINS, "the scale is a fraction");
    const uint32_t scale =
      static_cast<uint32_t>((static_cast<uint64_t>(EQ_BINS) << 32) / (static_cast<uint64_t>(b1 - b0 + 1) << EQ_FRACTION_BITS));
    uint4* const my_bins = reinterpret_cast<uint4*>(sh.bins) + tid;
    *my_bins             = make_uint4(0u, 0u, 0u, 0u);
    if (tid == 0) {
      sh.n_crowded = 0;
      sh.n_large   = 0;
    }
    uint32_t at[R];  // bin, and above it how many keys of the bin were counted before
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if constexpr (CODEC == CODEC_FLOAT) {
        odd |= is_nan_or_negative_zero(u[i]) ? 1 : 0;
      }
      u[i]             = image(u[i]);
      const uint32_t f = eq.fine(u[i], EQ_FRACTION_BITS);
      at[i]            = __umulhi(f - origin, scale);
      at[i]            = at[i] < EQ_BINS ? at[i] : EQ_BINS - 1;  // (a NaN, a -0.0: any number, not used)
    }
    if (__syncthreads_or(odd) != 0) {
      return false;
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (has(i)) {
        const uint32_t half = 16 * (at[i] % 2);
        const uint32_t was  = atomicAdd(&sh.bins[at[i] / 2], 1u << half);
        at[i] |= (was >> half) << 16;
      }
    }
    __syncthreads();
    const uint4 c4            = *my_bins;
    const uint32_t counts[4]  = {c4.x, c4.y, c4.z, c4.w};
    uint32_t pairs = 0, most = 0;  // both halves of the words summed at once: a piece has fewer than 2^16 keys
    uint32_t several = 0;          // bit j: bin j of this thread holds more than one key (and not too many)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      pairs += counts[k];
      const uint32_t a = counts[k] & 0xFFFFu, b = counts[k] >> 16;
      most = a > most ? a : most;
      most = b > most ? b : most;
      several |= (a > 1 ? 1u << (2 * k) : 0u) | (b > 1 ? 2u << (2 * k) : 0u);
    }
    if (most > EQ_BIN_LIMIT) {  // (rare)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t c = (counts[k / 2] >> (16 * (k % 2))) & 0xFFFFu;
        if (c > EQ_BIN_LIMIT) {
          several &= ~(1u << k);
          const uint32_t entry = c <= WAVE ? atomicAdd(&sh.n_crowded, 1u) : CROWDED - 1 - atomicAdd(&sh.n_large, 1u);
          sh.crowded[entry]    = static_cast<uint16_t>(tid * (2 * WORDS) + k);
        }
      }
    }
    const uint32_t sum  = (pairs & 0xFFFFu) + (pairs >> 16);
    const uint32_t incl = wave_inclusive_sum_dpp(sum);
    if (lane == WAVE - 1) {
      sh.wsum[tid / WAVE] = incl;
    }
    if (__syncthreads_or(most > BLOCK ? 1 : 0) != 0 || sh.n_large > EQ_LARGE_BINS) {
      return false;
    }
    uint32_t run = incl - sum;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      run += w < static_cast<int>(tid / WAVE) ? sh.wsum[w] : 0u;
    }
    uint32_t starts_of[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t a = counts[k] & 0xFFFFu, b = counts[k] >> 16;
      starts_of[k] = run | ((run + a) << 16);
      run += a + b;
    }
    *my_bins = make_uint4(starts_of[0], starts_of[1], starts_of[2], starts_of[3]);
    if (tid == BLOCK - 1) {
      sh.bins[EQ_BINS / 2] = run;  // the end of the last bin
    }
    __syncthreads();
    const uint16_t* const starts = reinterpret_cast<const uint16_t*>(sh.bins);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      at[i] = starts[at[i] & 0xFFFFu] + (at[i] >> 16);
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (has(i)) {
        sh.keys[at[i]] = u[i];
        if constexpr (HAS_IDX) {
          sh.idx[at[i]] = static_cast<uint16_t>(i * BLOCK + tid);
        }
      }
    }
    __syncthreads();
    while (several != 0) {
      const uint32_t bin  = tid * (2 * WORDS) + static_cast<uint32_t>(__builtin_ctz(several));
      const uint32_t from = starts[bin], to = starts[bin + 1];
      several &= several - 1;
      // insertion; the greatest key so far stays in registers (most bins hold two)
      KeyT last          = sh.keys[from];
      uint32_t last_idx  = HAS_IDX ? sh.idx[from] : 0u;
      for (uint32_t p = from + 1; p < to; ++p) {
        const KeyT k         = sh.keys[p];
        const uint32_t k_idx = HAS_IDX ? sh.idx[p] : 0u;
        if (k < last || (HAS_IDX && k == last && k_idx < last_idx)) {
          uint32_t q = p;  // the place of k: everything from there on moves up by one
          KeyT x = last;
          uint32_t x_idx = last_idx;
          while (true) {
            sh.keys[q] = x;
            if constexpr (HAS_IDX) {
              sh.idx[q] = static_cast<uint16_t>(x_idx);
            }
            --q;
            if (q == from) {
              break;
            }
            x = sh.keys[q - 1];
            if constexpr (HAS_IDX) {
              x_idx = sh.idx[q - 1];
            }
            if (!(k < x || (HAS_IDX && k == x && k_idx < x_idx))) {
              break;
            }
          }
          sh.keys[q] = k;
          if constexpr (HAS_IDX) {
            sh.idx[q] = static_cast<uint16_t>(k_idx);
          }
        } else {
          last     = k;
          last_idx = k_idx;
        }
      }
    }
    // (the lists are complete: there have been barriers since)
    auto rank_in_bin = [&](uint32_t from, uint32_t to, KeyT k, uint32_t k_idx) -> uint32_t {
      uint32_t place = from;
#pragma unroll 4
      for (uint32_t p = from; p < to; ++p) {
        const KeyT x         = sh.keys[p];
        const uint32_t x_idx = HAS_IDX ? sh.idx[p] : p;
        place += (x < k || (x == k && x_idx < k_idx)) ? 1u : 0u;
      }
      return place;
    };
    const uint32_t n_crowded = sh.n_crowded, n_large = sh.n_large;
    for (uint32_t c = tid / WAVE; c < n_crowded; c += WAVES) {  // uniform in a wave
      const uint32_t bin  = sh.crowded[c];
      const uint32_t from = starts[bin], to = starts[bin + 1];
      const uint32_t mine = from + lane < to ? from + lane : from;
      const KeyT k         = sh.keys[mine];
      const uint32_t k_idx = HAS_IDX ? sh.idx[mine] : mine;
      const uint32_t place = rank_in_bin(from, to, k, k_idx);
      __builtin_amdgcn_wave_barrier();  // (every lane has read the bin)
      if (from + lane < to) {
        sh.keys[place] = k;
        if constexpr (HAS_IDX) {
          sh.idx[place] = static_cast<uint16_t>(k_idx);
        }
      }
    }
    for (uint32_t c = 0; c < n_large; ++c) {  // uniform
      const uint32_t bin  = sh.crowded[CROWDED - 1 - c];
      const uint32_t from = starts[bin], to = starts[bin + 1];
      const bool in        = from + tid < to;
      const uint32_t mine  = in ? from + tid : from;
      const KeyT k         = sh.keys[mine];
      const uint32_t k_idx = HAS_IDX ? sh.idx[mine] : mine;
      const uint32_t place = rank_in_bin(from, in ? to : from, k, k_idx);
      __syncthreads();
      if (in) {
        sh.keys[place] = k;
        if constexpr (HAS_IDX) {
          sh.idx[place] = static_cast<uint16_t>(k_idx);
        }
      }
    }
    __syncthreads();
    if (out != nullptr) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        u[i] = sh.keys[i * BLOCK + tid];  // (BLOCK * R <= the tile)
      }
#pragma unroll
      for (int i = 0; i < R; ++i) {
        if (has(i)) {
          out[i * BLOCK + tid] = unimage(u[i]);
        }
      }
    }
    if constexpr (HAS_IDX) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        at[i] = has(i) ? sh.idx[i * BLOCK + tid] : 0u;
      }
#pragma unroll
      for (int i = 0; i < R; ++i) {
        at[i] = pos[at[i]];
      }
#pragma unroll
      for (int i = 0; i < R; ++i) {
        if (has(i)) {
          idx_out[i * BLOCK + tid] = static_cast<int64_t>(at[i]) + offset;
        }
      }
    }
    return true;
  }
};

template <typename KeyT, int CODEC, bool HAS_IDX>
__global__ __launch_bounds__(EQ_SORT_BLOCK) __attribute__((amdgpu_waves_per_eu(EQ_SORT_WAVES)))
void eq_sort_kernel(const KeyT* __restrict__ keys,
                                                                KeyT* __restrict__ keys_out,
                                                                const uint32_t* __restrict__ pos,
                                                                int64_t* __restrict__ idx_out,
                                                                int64_t index_offset,
                                                                uint32_t segments,
                                                                const uint32_t* __restrict__ status,
                                                                const uint2* __restrict__ segs,
                                                                const uint2* __restrict__ extras,
                                                                uint2* __restrict__ list,
                                                                const EqualLarge* __restrict__ large,
                                                                uint32_t max_large,
                                                                EqualPlan* __restrict__ eq)
{
  using Sort = EqualSort<KeyT, CODEC, HAS_IDX>;
  __shared__ typename Sort::Shared sh;
  if (eq->mode == 0 || *status != 0) {
    return;
  }
  // (the table stays in memory: a piece's keys lie in a few neighbouring cells)
  const EqualDigits<KeyT> digits{static_cast<KeyT>(eq->origin), static_cast<KeyT>(eq->last), eq->lshift, eq->table};
  const uint32_t pieces = segments + (eq->n_extra < segments ? eq->n_extra : segments);
  for (uint32_t e = blockIdx.x; e < pieces; e += gridDim.x) {
    const uint2 p = e < segments ? segs[e] : extras[e - segments];
    if (p.y == 0) {
      continue;  // uniform
    }
    const KeyT* in        = keys + p.x;
    KeyT* out             = keys_out != nullptr ? keys_out + p.x : nullptr;
    const uint32_t* pos_p = HAS_IDX ? pos + p.x : nullptr;
    int64_t* idx_p        = HAS_IDX ? idx_out + p.x : nullptr;
    bool done;
    switch ((p.y - 1) / EQ_SORT_BLOCK) {
      case 0: done = Sort::template piece<1>(sh, in, out, pos_p, idx_p, index_offset, p.y, digits); break;
      case 1: done = Sort::template piece<2>(sh, in, out, pos_p, idx_p, index_offset, p.y, digits); break;
      case 2: done = Sort::template piece<3>(sh, in, out, pos_p, idx_p, index_offset, p.y, digits); break;
      case 3: done = Sort::template piece<4>(sh, in, out, pos_p, idx_p, index_offset, p.y, digits); break;
      case 4: done = Sort::template piece<5>(sh, in, out, pos_p, idx_p, index_offset, p.y, digits); break;
      default: done = Sort::template piece<6>(sh, in, out, pos_p, idx_p, index_offset, p.y, digits); break;
    }
    static_assert(EQ_SORT_ITEMS == 6, "one case per count of rounds");
    if (!done && threadIdx.x == 0) {
      list[__hip_atomic_fetch_add(&eq->n_list, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)] = p;
    }
    __syncthreads();  // the next piece reuses the shared memory
  }
  // Large buckets: their keys have to be equal, or the byte passes are needed; equal keys are where they belong.
  const uint32_t parts = eq->n_large < max_large ? eq->n_large : max_large;
  for (uint32_t e = blockIdx.x; e < parts; e += gridDim.x) {
    const EqualLarge part = large[e];
    const KeyT want       = ordered_bits<CODEC, KeyT>(keys[part.first]);
    bool differs          = false;
    for (uint32_t i = threadIdx.x; i < part.length; i += EQ_SORT_BLOCK) {
      const KeyT k = keys[part.begin + i];
      differs |= ordered_bits<CODEC, KeyT>(k) != want;
      if (keys_out != nullptr) {
        keys_out[part.begin + i] = k;
      }
      if constexpr (HAS_IDX) {
        idx_out[part.begin + i] = static_cast<int64_t>(pos[part.begin + i]) + index_offset;
      }
    }
    if (differs) {
      __hip_atomic_store(&eq->failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

}  // namespace cpn
