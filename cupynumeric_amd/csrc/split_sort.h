// Rows of ten thousand to a few million real keys of 4 and 8 bytes: split once by sampled keys, every part sorted in LDS.
//
// Two launches that depend on each other, whatever the key's width and the distribution of the values:
//   split_tile_kernel   a workgroup takes one tile of the row, sorts a sample of the whole row (every workgroup the same
//                       one, in its own LDS: a launch of its own would take longer than sorting it does), takes every
//                       eighth sampled key as a splitter, and puts the keys of its tile in the order of the buckets between
//                       them, stably.  They stay together in memory; where each bucket starts goes into a table.
//   split_bucket_kernel a workgroup takes one bucket: its parts of all tiles are gathered, in the order of the tiles, and
//                       sorted in LDS.  Where the bucket goes follows from the table as well.
// Nothing is counted ahead, nothing has to be cleared, no workgroup waits for another.  The passes that rows of this length
// went through before (one per key byte, onesweep.h, or levels of merging, merge_rows.h) are chains of 5 to 12 dependent
// launches, each of them a few us long whatever it does.
//
// A splitter is a pair of a key and its place in the row, so that equal keys are divided as well as any others: the sizes
// of the buckets do not depend on how the values are distributed, only on which places are sampled, and
// these are drawn from a hash of their number.  A bucket lies between eight sampled keys; the room in LDS is four times
// the mean.  (Of a bucket with more there is one in ten million; only a row that was made for the purpose has many.)
// Such a bucket is sorted by its workgroup in memory, one byte after another (oversized_bucket): slow, and still right.
//
// Stands where the reference calls cub's radix sort or thrust's merge sort of one row
// (src/cupynumeric/sort/cub_sort.cuh:60-151, src/cupynumeric/sort/thrust_sort.cuh:37-66).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "bitonic_row_sort.h"
#include "radix_common.h"

namespace cpn {

constexpr int SPLIT_BLOCK       = 1024;
constexpr int SPLIT_BUCKET_BLOCK = 512;
constexpr int SPLIT_BUCKET_ITEMS = 8;
constexpr int SPLIT_WAVES       = SPLIT_BLOCK / WAVE;
constexpr int SPLIT_TILE_ITEMS  = 4;                       // keys per thread of a tile
constexpr int SPLIT_SAMPLE_E    = 8;                       // sampled keys per lane of a wave that sorts them
constexpr int SPLIT_MAX_BUCKETS = 1024;
constexpr int SPLIT_MAX_TILES   = 256;
constexpr uint32_t SPLIT_CROWD  = 64;  // most sampled keys of a bin

// A mixed 32-bit word: which key of its stretch sample i takes.
__host__ __device__ __forceinline__ uint32_t split_hash(uint32_t x)
{
  x ^= x >> 16;
  x *= 0x7FEB352Du;
  x ^= x >> 15;
  x *= 0x846CA68Bu;
  x ^= x >> 16;
  return x;
}
// The place in a row of n keys that sample i of `samples` is taken from: one place of each of `samples` equal stretches.
__host__ __device__ __forceinline__ uint32_t split_sample_place(uint32_t i, uint32_t samples, uint32_t n)
{
  const uint32_t from = static_cast<uint32_t>(static_cast<uint64_t>(i) * n / samples);
  const uint32_t to   = static_cast<uint32_t>(static_cast<uint64_t>(i + 1) * n / samples);
  return from + static_cast<uint32_t>((static_cast<uint64_t>(split_hash(i)) * (to - from)) >> 32);
}

// Stable rank of a lane's bucket among those of its wave (radix_common.h's wave_match_rank, for as many bits as a
// bucket's number has and counters of 16 bits).
template <int BITS>
__device__ __forceinline__ uint32_t split_match_rank(uint32_t bucket, bool valid, uint16_t* wctr)
{
  const uint64_t vmask = __builtin_amdgcn_ballot_w64(valid);
  uint32_t mis_lo = 0, mis_hi = 0;
#pragma unroll
  for (int b = 0; b < BITS; ++b) {
    int32_t own = __builtin_amdgcn_sbfe(static_cast<int32_t>(bucket), b, 1);
    asm volatile("" : "+v"(own));
    const uint64_t bal = __builtin_amdgcn_ballot_w64(own != 0);
    mis_lo = __builtin_amdgcn_bitop3_b32(mis_lo, static_cast<uint32_t>(bal), static_cast<uint32_t>(own), 0xF6);
    mis_hi = __builtin_amdgcn_bitop3_b32(mis_hi, static_cast<uint32_t>(bal >> 32), static_cast<uint32_t>(own), 0xF6);
  }
  const uint32_t peers_lo = static_cast<uint32_t>(vmask) & ~mis_lo;
  const uint32_t peers_hi = static_cast<uint32_t>(vmask >> 32) & ~mis_hi;
  const uint32_t lower    = __builtin_amdgcn_mbcnt_hi(peers_hi, __builtin_amdgcn_mbcnt_lo(peers_lo, 0u));
  const uint32_t total    = static_cast<uint32_t>(__builtin_popcount(peers_lo) + __builtin_popcount(peers_hi));
  const uint32_t old      = wctr[bucket];
  __builtin_amdgcn_wave_barrier();
  if (valid && lower + 1 == total) {
    wctr[bucket] = static_cast<uint16_t>(old + total);
  }
  __builtin_amdgcn_wave_barrier();
  return old + lower;
}

// Exchange of the sample between waves: word r of thread t lies at r * THREADS + t.
template <typename W>
struct SplitExchange;
template <>
struct SplitExchange<F64Word> {
  static constexpr int BYTES = 8;
  static __device__ __forceinline__ void put(unsigned char* s, int, int slot, const F64Word& w) { reinterpret_cast<double*>(s)[slot] = w.v; }
  static __device__ __forceinline__ F64Word get(const unsigned char* s, int, int slot) { return F64Word{reinterpret_cast<const double*>(s)[slot]}; }
};
template <>
struct SplitExchange<ImagePos> {
  static constexpr int BYTES = 12;
  static __device__ __forceinline__ void put(unsigned char* s, int slots, int slot, const ImagePos& w)
  {
    reinterpret_cast<uint64_t*>(s)[slot]             = w.image;
    reinterpret_cast<uint32_t*>(s + 8 * slots)[slot] = static_cast<uint32_t>(w.pos);
  }
  static __device__ __forceinline__ ImagePos get(const unsigned char* s, int slots, int slot)
  {
    return ImagePos{reinterpret_cast<const uint64_t*>(s)[slot], reinterpret_cast<const uint32_t*>(s + 8 * slots)[slot]};
  }
};

// Merges the sorted runs of single waves into one of SW waves (the steps of bitonic_row_sort.h's network that cross
// waves, through LDS).  Every thread of the workgroup calls; those of the first SW waves hold keys.
template <int RUN, int SW, typename W>
__device__ __forceinline__ void split_merge_waves(W (&w)[SPLIT_SAMPLE_E], unsigned char* s, uint32_t tid)
{
  if constexpr (RUN <= SW) {
    constexpr int THREADS = SW * WAVE, SLOTS = THREADS * SPLIT_SAMPLE_E;
    using X            = SplitExchange<W>;
    const bool holds   = tid < THREADS;
    const uint32_t sub = tid % (RUN * WAVE);
#pragma unroll
    for (int d = RUN; d >= 2; d /= 2) {  // d == RUN: the mirror image in the run; then lanes at distance d * WAVE / 2
      const bool mirror = d == RUN;
      __syncthreads();
      if (holds) {
#pragma unroll
        for (int r = 0; r < SPLIT_SAMPLE_E; ++r) {
          X::put(s, SLOTS, r * THREADS + tid, w[r]);
        }
      }
      __syncthreads();
      if (holds) {
        const uint32_t other = mirror ? tid ^ (RUN * WAVE - 1) : tid ^ (d * WAVE / 2);
        const bool keep_min  = mirror ? sub < RUN * WAVE / 2 : (tid & (d * WAVE / 2)) == 0;
#pragma unroll
        for (int r = 0; r < SPLIT_SAMPLE_E; ++r) {
          const W o = X::get(s, SLOTS, (mirror ? SPLIT_SAMPLE_E - 1 - r : r) * THREADS + other);
          w[r]      = word_select(word_less(w[r], o) == keep_min, w[r], o);
        }
      }
    }
    if (holds) {
      cross_steps<WAVE / 2>(w, tid & (WAVE - 1));
      lane_sort_bitonic(w);
    }
    split_merge_waves<2 * RUN, SW>(w, s, tid);
  }
}

// A number that does not decrease with the key (32 bits are enough to spread a sample); NaNs: +infinity.
template <int CODEC, typename KeyT>
__device__ __forceinline__ float split_value(KeyT raw)
{
  if constexpr (CODEC == CODEC_FLOAT) {
    float f;
    if constexpr (sizeof(KeyT) == 8) {
      f = static_cast<float>(__longlong_as_double(static_cast<long long>(raw)));
    } else {
      f = __uint_as_float(raw);
    }
    return f != f ? __builtin_huge_valf() : f;
  } else if constexpr (CODEC == CODEC_SIGNED) {
    return static_cast<float>(static_cast<std::conditional_t<sizeof(KeyT) == 8, int64_t, int32_t>>(raw));
  } else {
    return static_cast<float>(raw);
  }
}

// The sum of the words of the waves before this one, and of all.  (All reads at once: in a loop that ends at the wave's own
// number they wait for each other.)
__device__ __forceinline__ uint32_t split_waves_before(const uint32_t* s_wave, uint32_t wave)
{
  uint32_t before = 0;
#pragma unroll
  for (uint32_t v = 0; v < SPLIT_WAVES; ++v) {
    before += v < wave ? s_wave[v] : 0u;
  }
  return before;
}

// What a workgroup needs in LDS to find the splitters of a row, PER_THREAD sampled keys each: a word per sampled key, and
// room for the network's exchanges (the keys in the order of their bins, and their numbers, take less).
template <typename KeyT, int PER_THREAD, int PER_BUCKET>
struct SplitSample {
  using W                        = std::conditional_t<sizeof(KeyT) == 8, ImagePos, F64Word>;
  static constexpr int SAMPLES   = PER_THREAD * SPLIT_BLOCK;
  static constexpr int SORTERS   = SAMPLES / SPLIT_SAMPLE_E;  // threads of the network
  static constexpr int SPLITTERS = SAMPLES / PER_BUCKET;
  static constexpr int BYTES     = SAMPLES * SplitExchange<W>::BYTES;
  static_assert(SPLIT_SAMPLE_E % PER_BUCKET == 0, "the first of a lane's sampled keys is a splitter");
};

// The bin of a value: subtraction, scaling and truncation do not decrease with it.  (Clamped before the conversion, NaN to
// 0: all that an infinite span leaves in one bin, or in two, is crowded.)
struct SplitBins {
  float lowest, scale;
};
template <int SAMPLES>
__device__ __forceinline__ uint32_t split_bin(const SplitBins& b, float value)
{
  return static_cast<uint32_t>(__builtin_fminf(__builtin_fmaxf((value - b.lowest) * b.scale, 0.0f), static_cast<float>(SAMPLES - 1)));
}
// How many splitters lie in the bins before one that starts behind `from` sampled keys (splitter 0 does not count).
template <int PER_BUCKET>
__device__ __forceinline__ uint32_t split_splitters_before(uint32_t from)
{
  return from != 0 ? (from - 1) / PER_BUCKET : 0;
}

// Splitter j of a row is the smallest of the j-th PER_BUCKET sampled keys: put(j, image, place) for every j; s_bins is left
// with the number of sampled keys before each bin.  The whole workgroup calls.  The sample is spread over as many bins of equal width in the value as it has keys; one atomic per key
// says which of its bin it is, a scan where the bin starts, and a walk over the bin how many of its keys come before.  A
// sample that crowds its bins (few different values, values of many magnitudes) goes through a sorting network.
template <int CODEC, int PER_THREAD, int PER_BUCKET, typename KeyT, typename Get, typename Put>
__device__ __forceinline__ SplitBins split_find_splitters(uint32_t n, unsigned char* s_mem, uint32_t* s_bins, uint32_t* s_wave, uint32_t* s_low,
                                                          const KeyT (&got)[PER_THREAD], Get get, Put put)
{
  using S                = SplitSample<KeyT, PER_THREAD, PER_BUCKET>;
  using W                = typename S::W;
  constexpr int SAMPLES  = S::SAMPLES;
  const uint32_t tid     = threadIdx.x;
  const uint32_t lane    = tid & (WAVE - 1);
  const uint32_t wave    = tid / WAVE;
  KeyT* const s_image     = reinterpret_cast<KeyT*>(s_mem);
  uint16_t* const s_which = reinterpret_cast<uint16_t*>(s_mem + SAMPLES * sizeof(KeyT));
#pragma unroll
  for (int r = 0; r < PER_THREAD; ++r) {
    s_bins[r * SPLIT_BLOCK + tid] = 0;
  }
  uint32_t low = 0, high = 0;  // of the finite values: the complement of the smallest image, the largest
#pragma unroll
  for (int r = 0; r < PER_THREAD; ++r) {
    const float value    = split_value<CODEC, KeyT>(got[r]);
    const bool finite    = __builtin_fabsf(value) < __builtin_huge_valf();
    const uint32_t image = sign_flip<uint32_t>(__float_as_uint(value));
    high                 = finite && image > high ? image : high;
    low                  = finite && ~image > low ? ~image : low;
  }
  high = wave_inclusive_max_dpp(high);
  low  = wave_inclusive_max_dpp(low);
  if (lane == WAVE - 1) {
    s_wave[wave] = high;
    s_low[wave]  = low;
  }
  __syncthreads();
#pragma unroll
  for (int v = 0; v < SPLIT_WAVES; ++v) {
    high = s_wave[v] > high ? s_wave[v] : high;
    low  = s_low[v] > low ? s_low[v] : low;
  }
  SplitBins bins;
  bins.lowest      = __uint_as_float(sign_unflip<uint32_t>(~low));
  const float span = __uint_as_float(sign_unflip<uint32_t>(high)) - bins.lowest;
  bins.scale       = span > 0.0f ? static_cast<float>(SAMPLES) / span : 0.0f;
  uint32_t bin[PER_THREAD];  // and, in the upper half, which of it
#pragma unroll
  for (int r = 0; r < PER_THREAD; ++r) {
    bin[r] = split_bin<SAMPLES>(bins, split_value<CODEC, KeyT>(got[r]));
    bin[r] |= atomicAdd(&s_bins[bin[r]], 1u) << 16;
  }
  __syncthreads();
  uint32_t count[PER_THREAD], sum = 0, most = 0;
#pragma unroll
  for (int r = 0; r < PER_THREAD; ++r) {
    count[r] = s_bins[tid * PER_THREAD + r];
    sum += count[r];
    most = count[r] > most ? count[r] : most;
  }
  const uint32_t sums = wave_inclusive_sum_dpp(sum);
  if (lane == WAVE - 1) {
    s_wave[wave] = sums;
  }
  uint32_t number = tid;
  asm volatile("" : "+v"(number));  // (or the places of all sampled keys are kept from the loads on, and spilled)
  const int crowded = __syncthreads_or(most > SPLIT_CROWD ? 1 : 0);
  uint32_t run      = sums - sum + split_waves_before(s_wave, wave);
#pragma unroll
  for (int r = 0; r < PER_THREAD; ++r) {
    s_bins[tid * PER_THREAD + r] = run;
    run += count[r];
  }
  __syncthreads();
  if (crowded == 0) {
#pragma unroll
    for (int r = 0; r < PER_THREAD; ++r) {
      const uint32_t to = s_bins[bin[r] & 0xFFFFu] + (bin[r] >> 16);
      s_image[to]       = ordered_bits<CODEC, KeyT>(got[r]);
      s_which[to]       = static_cast<uint16_t>(r * SPLIT_BLOCK + tid);
    }
    __syncthreads();
    // (all walks of a thread in step: their reads do not wait for each other; bins that no splitter lies in are not walked)
    uint32_t from[PER_THREAD], len[PER_THREAD], before[PER_THREAD], longest = 0;
    KeyT image[PER_THREAD];
#pragma unroll
    for (int r = 0; r < PER_THREAD; ++r) {
      const uint32_t b = bin[r] & 0xFFFFu;
      from[r]          = s_bins[b];
      len[r]           = (b + 1 < SAMPLES ? s_bins[b + 1] : static_cast<uint32_t>(SAMPLES)) - from[r];
      image[r]         = s_image[from[r] + (bin[r] >> 16)];
      before[r]        = from[r];
      if ((from[r] + PER_BUCKET - 1) / PER_BUCKET * PER_BUCKET >= from[r] + len[r]) {
        len[r] = 0;
      }
      longest = len[r] > longest ? len[r] : longest;
    }
    for (uint32_t j = 0; j < longest; ++j) {
#pragma unroll
      for (int r = 0; r < PER_THREAD; ++r) {
        const uint32_t at = from[r] + (j < len[r] ? j : 0u);
        const KeyT other  = s_image[at];
        const bool first  = (other < image[r]) | ((other == image[r]) & (s_which[at] < r * SPLIT_BLOCK + number));
        before[r] += (first & (j < len[r])) ? 1u : 0u;
      }
    }
#pragma unroll
    for (int r = 0; r < PER_THREAD; ++r) {
      if (len[r] != 0 && before[r] % PER_BUCKET == 0) {
        put(before[r] / PER_BUCKET, image[r], split_sample_place(r * SPLIT_BLOCK + number, SAMPLES, n));
      }
    }
  } else {
    W w[SPLIT_SAMPLE_E];
    if (tid < S::SORTERS) {
#pragma unroll
      for (int r = 0; r < SPLIT_SAMPLE_E; ++r) {
        const uint32_t i = number * SPLIT_SAMPLE_E + r;
        const KeyT image = ordered_bits<CODEC, KeyT>(get(i));
        if constexpr (sizeof(KeyT) == 8) {
          w[r] = ImagePos{image, i};
        } else {
          w[r] = pack_image_pos(image, i);
        }
      }
      blocked_sort<WAVE>(w, lane);
    }
    split_merge_waves<2, S::SORTERS / WAVE>(w, s_mem, tid);
    if (tid < S::SORTERS) {
#pragma unroll
      for (int r = 0; r < SPLIT_SAMPLE_E; r += PER_BUCKET) {
        KeyT image;
        if constexpr (sizeof(KeyT) == 8) {
          image = w[r].image;
        } else {
          image = static_cast<KeyT>(static_cast<uint64_t>(__double_as_longlong(w[r].v)) >> 20);
        }
        put((tid * SPLIT_SAMPLE_E + r) / PER_BUCKET, image, split_sample_place(word_pos(w[r]), SAMPLES, n));
      }
    }
  }
  return bins;
}

// The sampled keys of the row, gathered by many workgroups: one alone reads a thousand scattered keys in 2.5 us, and so
// does each of the workgroups that need all of them.
template <typename KeyT>
__global__ __launch_bounds__(256) void split_gather_kernel(const KeyT* __restrict__ keys_in, uint32_t n, uint32_t samples,
                                                           KeyT* __restrict__ out)
{
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;  // (`samples` is a multiple of the workgroup)
  out[i]           = keys_in[split_sample_place(i, samples, n)];
}

// One tile of a row into the order of its buckets.
//   grouped, places   the keys of the tile, and where in the tile each was (16 bits), at the tile's own place in the row
//   starts            [tile][bucket]: where each bucket starts in its tile, and the tile's length
//   sample            the sampled keys, or nullptr: the workgroup gathers them
// HAS_POS: positions are asked for, and `places` written.  PER_THREAD, PER_BUCKET: sampled keys.
// Bound by its own chain (load the sample, sort it, search, rank, exchange, store), not by memory or arithmetic: 8 us for
// tiles of 1024 keys and 1024 sampled ones (2.5 of it their scattered reads), 12 with 2048, 26 for tiles of 4096 and 8192 sampled.
// The splitters by binary search among all of them took 18 us of such a tile; by the bin of the key's value, 13.
template <typename KeyT, int CODEC, bool HAS_POS, int PER_THREAD, int PER_BUCKET, int ITEMS>
__global__ __launch_bounds__(SPLIT_BLOCK) void split_tile_kernel(const KeyT* __restrict__ keys_in, uint32_t n,
                                                                 uint32_t tile_len, const KeyT* __restrict__ sample,
                                                                 KeyT* __restrict__ grouped, uint16_t* __restrict__ places,
                                                                 uint16_t* __restrict__ starts, uint32_t* __restrict__ status)
{
  using S                 = SplitSample<KeyT, PER_THREAD, PER_BUCKET>;
  constexpr int SAMPLES   = S::SAMPLES;
  constexpr int BUCKETS   = S::SPLITTERS;
  constexpr int BITS      = 31 - __builtin_clz(BUCKETS);
  constexpr int TILE      = SPLIT_BLOCK * ITEMS;
  constexpr int X_BYTES   = S::BYTES;
  constexpr int K_BYTES   = TILE * static_cast<int>(sizeof(KeyT));
  constexpr int CTR_BYTES = SPLIT_WAVES * BUCKETS * 2;
  static_assert(CTR_BYTES >= SAMPLES * 4, "a word per bin");
  static_assert(BUCKETS <= SPLIT_BLOCK, "a thread per bucket");
  static_assert(TILE <= 65535, "places and starts are 16 bits");
  __shared__ __align__(16) unsigned char s_mem[X_BYTES > K_BYTES ? X_BYTES : K_BYTES];  // the sample, then the tile
  __shared__ uint16_t s_place[HAS_POS ? TILE : 1];
  __shared__ __align__(16) uint16_t s_ctr[SPLIT_WAVES * BUCKETS];  // before: the words of the sampled keys
  __shared__ KeyT s_split[BUCKETS];
  __shared__ uint32_t s_split_at[BUCKETS];
  __shared__ uint16_t s_base[BUCKETS];
  __shared__ uint32_t s_wave[SPLIT_WAVES], s_low[SPLIT_WAVES];

  const uint32_t tid  = threadIdx.x;
  const uint32_t lane = tid & (WAVE - 1);
  const uint32_t wave = tid / WAVE;
  if (blockIdx.x == 0 && tid == 0) {
    *status = 0;  // (the workspace's status word: this sort cannot fail on the device)
  }
  const uint32_t first  = blockIdx.x * tile_len;
  const uint32_t len    = n - first < tile_len ? n - first : tile_len;  // (no tile is empty)
  const uint32_t rounds = (len + SPLIT_BLOCK - 1) / SPLIT_BLOCK;        // uniform; every wave takes that many 64 keys
  const uint32_t woff   = wave * rounds * WAVE + lane;

  // ---- the sample, and the tile's own keys: all loads first ----
  auto sampled = [&](uint32_t i) -> KeyT { return sample != nullptr ? sample[i] : keys_in[split_sample_place(i, SAMPLES, n)]; };
  KeyT got[PER_THREAD];
#pragma unroll
  for (int r = 0; r < PER_THREAD; ++r) {
    got[r] = sampled(r * SPLIT_BLOCK + tid);
  }
  KeyT key[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t o = woff + i * WAVE;
    key[i]           = keys_in[first + (o < len ? o : len - 1)];
  }
  uint32_t* const s_bins = reinterpret_cast<uint32_t*>(s_ctr);
  const SplitBins bins   = split_find_splitters<CODEC, PER_THREAD, PER_BUCKET>(n, s_mem, s_bins, s_wave, s_low, got, sampled,
                                                                             [&](uint32_t j, KeyT image, uint32_t place) {
                                                                               s_split[j]    = image;
                                                                               s_split_at[j] = place;
                                                                             });
  __syncthreads();

  // ---- the bucket of every key: how many splitters come before it.  The bin of its value leaves none or one of them to
  //      ask (all of them at most: a binary search over those of the bin) ----
  uint32_t bucket[ITEMS], left[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t bin = split_bin<SAMPLES>(bins, split_value<CODEC, KeyT>(key[i]));
    bucket[i]          = split_splitters_before<PER_BUCKET>(s_bins[bin]);
    left[i]            = split_splitters_before<PER_BUCKET>(bin + 1 < SAMPLES ? s_bins[bin + 1] : static_cast<uint32_t>(SAMPLES)) - bucket[i];
  }
  for (;;) {
    uint32_t most = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      most = left[i] > most ? left[i] : most;
    }
    if (__ballot(most != 0) == 0) {
      break;
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const uint32_t at   = first + woff + i * WAVE;
      const uint32_t half = (left[i] + 1) / 2;
      const uint32_t c    = bucket[i] + half;  // (left == 0: the splitter before, which is reached)
      const KeyT image    = ordered_bits<CODEC, KeyT>(key[i]);
      const KeyT split    = s_split[c];
      const bool reached  = (split < image) | ((split == image) & (s_split_at[c] <= at));
      bucket[i]           = reached ? c : bucket[i];
      left[i]             = left[i] == 0 ? 0 : (reached ? left[i] - half : half - 1);
    }
  }
  __syncthreads();
  for (uint32_t j = tid; j < CTR_BYTES / 16; j += SPLIT_BLOCK) {
    reinterpret_cast<uint4*>(s_ctr)[j] = make_uint4(0u, 0u, 0u, 0u);
  }
  __syncthreads();
  // ---- ranks: stable, wave by wave, then over the waves of the workgroup ----
  uint32_t rank[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    rank[i] = 0;
    if (i < static_cast<int>(rounds)) {  // uniform
      rank[i] = split_match_rank<BITS>(bucket[i], woff + i * WAVE < len, s_ctr + wave * BUCKETS);
    }
  }
  __syncthreads();
  uint32_t total = 0;
  if (tid < BUCKETS) {
    uint32_t c[SPLIT_WAVES];
#pragma unroll
    for (int v = 0; v < SPLIT_WAVES; ++v) {
      c[v] = s_ctr[v * BUCKETS + tid];
    }
#pragma unroll
    for (int v = 0; v < SPLIT_WAVES; ++v) {
      s_ctr[v * BUCKETS + tid] = static_cast<uint16_t>(total);
      total += c[v];
    }
  }
  const uint32_t incl = wave_inclusive_sum_dpp(total);
  if (lane == WAVE - 1) {
    s_wave[wave] = incl;
  }
  __syncthreads();
  if (tid < BUCKETS) {
    const uint32_t start = incl - total + split_waves_before(s_wave, wave);
    s_base[tid]          = static_cast<uint16_t>(start);
    uint16_t* const to   = starts + static_cast<uint64_t>(blockIdx.x) * (BUCKETS + 1);
    to[tid]              = static_cast<uint16_t>(start);
    if (tid == 0) {
      to[BUCKETS] = static_cast<uint16_t>(len);
    }
  }
  __syncthreads();
  KeyT* const s_keys = reinterpret_cast<KeyT*>(s_mem);
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t o = woff + i * WAVE;
    if (i < static_cast<int>(rounds) && o < len) {
      const uint32_t to = s_base[bucket[i]] + s_ctr[wave * BUCKETS + bucket[i]] + rank[i];
      s_keys[to]        = key[i];
      if constexpr (HAS_POS) {
        s_place[to] = static_cast<uint16_t>(o);
      }
    }
  }
  __syncthreads();
  KeyT* const out = grouped + first;
  for (uint32_t o = tid; o < len; o += SPLIT_BLOCK) {
    out[o] = s_keys[o];
    if constexpr (HAS_POS) {
      places[first + o] = s_place[o];
    }
  }
}

// What the workgroups of the buckets are given.
template <typename KeyT>
struct SplitBuckets {
  const KeyT* grouped;
  const uint16_t* places;
  const uint16_t* starts;
  uint32_t* ids;  // two words per key: what the slow way of an oversized bucket orders
  uint32_t n, tiles, tile_len, buckets;
};

// A bucket of more keys than LDS has room for, sorted by its workgroup alone: one stable pass per key byte over the
// numbers of its keys, which go back and forth between two arrays in memory.  A turn of BLOCK keys takes about 2 us.
//   s_from  [tiles]: where the part of a tile lies in `grouped`, less where it lies in the bucket (modulo 2^32)
//   s_slot  [tiles]: where it lies in the bucket
//   s_ctr   a counter per digit and wave, s_digit: one per digit
template <typename KeyT, int CODEC, bool HAS_IDX, int BLOCK>
__device__ __forceinline__ void oversized_bucket(const SplitBuckets<KeyT>& sb, uint32_t m, uint32_t base,
                                                 const uint32_t* s_from, const uint32_t* s_slot, uint32_t* s_ctr,
                                                 uint32_t* s_digit, KeyT* keys_out, int64_t* idx_out, int64_t index_offset)
{
  using KT             = KeyTraits<CODEC, KeyT>;
  constexpr int WAVES  = BLOCK / WAVE;
  const uint32_t tid   = threadIdx.x;
  const uint32_t wave  = tid / WAVE;
  auto tile_of = [&](uint32_t slot) -> uint32_t {  // the last tile whose part starts at or before the slot
    uint32_t lo = 0, hi = sb.tiles;
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) / 2;
      if (s_slot[mid] <= slot) {
        lo = mid;
      } else {
        hi = mid;
      }
    }
    return lo;
  };
  for (int pass = 0; pass < KT::PASSES; ++pass) {
    const uint32_t* const ids_in = sb.ids + base + (pass % 2 == 0 ? sb.n : 0u);
    uint32_t* const ids_out      = sb.ids + base + (pass % 2 == 0 ? 0u : sb.n);
    auto id_at    = [&](uint32_t i) -> uint32_t { return pass == 0 ? i : ids_in[i]; };
    auto digit_at = [&](uint32_t id) -> uint32_t { return KT::digit(sb.grouped[s_from[tile_of(id)] + id], pass); };
    if (tid < RADIX) {
      s_ctr[tid] = 0;
    }
    __syncthreads();
    for (uint32_t i = tid; i < m; i += BLOCK) {
      atomicAdd(&s_ctr[digit_at(id_at(i))], 1u);
    }
    __syncthreads();
    if (tid < WAVE) {  // four digits a lane
      uint32_t c[RADIX / WAVE], sum = 0;
#pragma unroll
      for (int k = 0; k < RADIX / WAVE; ++k) {
        c[k] = s_ctr[tid * (RADIX / WAVE) + k];
        sum += c[k];
      }
      uint32_t run = wave_inclusive_sum_dpp(sum) - sum;
#pragma unroll
      for (int k = 0; k < RADIX / WAVE; ++k) {
        s_digit[tid * (RADIX / WAVE) + k] = run;
        run += c[k];
      }
    }
    for (uint32_t from = 0; from < m; from += BLOCK) {
      __syncthreads();
      for (uint32_t j = tid; j < WAVES * RADIX; j += BLOCK) {
        s_ctr[j] = 0;
      }
      __syncthreads();
      const uint32_t i   = from + tid;
      const bool valid   = i < m;
      const uint32_t id  = id_at(valid ? i : m - 1);
      const uint32_t d   = digit_at(id);
      const uint32_t rnk = wave_match_rank(d, valid, s_ctr + wave * RADIX);
      __syncthreads();
      if (tid < RADIX) {
        uint32_t run = s_digit[tid];
#pragma unroll
        for (int v = 0; v < WAVES; ++v) {
          const uint32_t c       = s_ctr[v * RADIX + tid];
          s_ctr[v * RADIX + tid] = run;
          run += c;
        }
        s_digit[tid] = run;
      }
      __syncthreads();
      if (valid) {
        ids_out[s_ctr[wave * RADIX + d] + rnk] = id;
      }
    }
    __threadfence_block();
    __syncthreads();
  }
  const uint32_t* const ids = sb.ids + base + (KT::PASSES % 2 == 0 ? sb.n : 0u);
  for (uint32_t i = tid; i < m; i += BLOCK) {
    const uint32_t id = ids[i], t = tile_of(id), at = s_from[t] + id;
    if (keys_out != nullptr) {
      keys_out[base + i] = sb.grouped[at];
    }
    if constexpr (HAS_IDX) {
      idx_out[base + i] = static_cast<int64_t>(t * sb.tile_len + sb.places[at]) + index_offset;
    }
  }
}

// The arithmetic type of a real key of 4 or 8 bytes, whose order is that of its images where there is no NaN.
template <int CODEC, int BYTES>
struct SplitNative {
  using type = uint32_t;
};
template <> struct SplitNative<CODEC_UNSIGNED, 8> { using type = uint64_t; };
template <> struct SplitNative<CODEC_SIGNED, 4> { using type = int32_t; };
template <> struct SplitNative<CODEC_SIGNED, 8> { using type = int64_t; };
template <> struct SplitNative<CODEC_FLOAT, 4> { using type = float; };
template <> struct SplitNative<CODEC_FLOAT, 8> { using type = double; };

constexpr uint32_t SPLIT_BIN_LIMIT = 24;  // most keys of a bin that are compared with each other

// One bucket of a row: its parts of all tiles gathered, sorted, stored.
//   a bucket of equal images is in order: it was gathered in the order of the row
//   others are spread over four bins per thread, of equal width between their smallest and their largest key; one atomic per key
//     says which of its bin it is, a scan where the bin starts, a walk over the bin how many of its keys come before
//   buckets with a NaN or a crowded bin: passes over the bytes of the images, of which numbers of keys move and the keys
//     stay where they are in LDS.  One pass where there are two values, else the four leading bytes that vary and, where
//     that does not put them in order, all
// Ties go by the place in the gathered order.
// Bound by its chain where every bucket has a compute unit (7 to 8 us for buckets of 400 keys; as one more mode of
// lds_row_sort_kernel, with two reductions and two atomics per key, 11), else by the workgroups that fit, two to a unit of
// 512 threads with 8-byte keys, three with 4-byte keys.
template <typename KeyT, int CODEC, bool HAS_IDX, int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) void split_bucket_kernel(const SplitBuckets<KeyT> sb, KeyT* __restrict__ keys_out,
                                                             int64_t* __restrict__ idx_out, int64_t index_offset)
{
  constexpr int WAVES = BLOCK / WAVE;
  constexpr int TILE  = BLOCK * ITEMS;
  constexpr int BINS  = 4 * BLOCK;
  constexpr int OWN   = BINS / BLOCK;  // bins a thread scans
  static_assert(OWN % 4 == 0, "whole vectors");
  static_assert(BLOCK >= SPLIT_MAX_TILES && BLOCK >= RADIX, "a thread per tile, and per digit");
  static_assert(TILE <= 65536 && BINS <= 65536, "numbers of 16 bits");
  constexpr int WORDS0 = BINS > WAVES * RADIX ? BINS : WAVES * RADIX;
  constexpr int WORDS  = WORDS0 > TILE / 2 ? WORDS0 : TILE / 2;
  using Native         = typename SplitNative<CODEC, sizeof(KeyT)>::type;
  using Scale          = std::conditional_t<sizeof(KeyT) == 4, float, double>;
  __shared__ __align__(16) KeyT s_keys[TILE + SPLIT_BIN_LIMIT];
  __shared__ uint16_t s_num[TILE + SPLIT_BIN_LIMIT];
  __shared__ __align__(16) uint32_t s_ctr[WORDS];  // marks of tiles, bins, counters of digits
  __shared__ uint32_t s_from[SPLIT_MAX_TILES], s_slot[SPLIT_MAX_TILES];
  __shared__ uint64_t s_red[2 * WAVES];
  __shared__ uint32_t s_wave[WAVES];
  __shared__ uint32_t s_digit[RADIX];

  const uint32_t tid    = threadIdx.x;
  const uint32_t lane   = tid & (WAVE - 1);
  const uint32_t wave   = tid / WAVE;
  const uint32_t bucket = blockIdx.x;

  // ---- the bucket's part of every tile; m keys in all, `base` keys of the row before them ----
  uint32_t start = 0, len = 0;
  if (tid < sb.tiles) {
    const uint16_t* const at = sb.starts + static_cast<uint64_t>(tid) * (sb.buckets + 1) + bucket;
    start                    = at[0];
    len                      = at[1] - start;
  }
  const uint32_t incl_len   = wave_inclusive_sum_dpp(len);
  const uint32_t incl_start = wave_inclusive_sum_dpp(start);
  if (lane == WAVE - 1) {
    s_red[wave] = (static_cast<uint64_t>(incl_start) << 32) | incl_len;
  }
  for (uint32_t j = tid; j < TILE / 8; j += BLOCK) {
    reinterpret_cast<uint4*>(s_ctr)[j] = make_uint4(0u, 0u, 0u, 0u);
  }
  __syncthreads();
  uint32_t slot = incl_len - len, m = 0, base = 0;
#pragma unroll
  for (uint32_t w = 0; w < WAVES; ++w) {
    const uint64_t sums = s_red[w];
    slot += w < wave ? static_cast<uint32_t>(sums) : 0u;
    m += static_cast<uint32_t>(sums);
    base += static_cast<uint32_t>(sums >> 32);
  }
  if (m == 0) {
    return;  // uniform
  }
  if (tid < sb.tiles) {
    s_from[tid] = tid * sb.tile_len + start - slot;
    s_slot[tid] = slot;
  }
  if (m > TILE) {  // uniform
    __syncthreads();
    oversized_bucket<KeyT, CODEC, HAS_IDX, BLOCK>(sb, m, base, s_from, s_slot, s_ctr, s_digit, keys_out, idx_out, index_offset);
    return;
  }
  // the number of a tile, plus one, at the first slot of its part
  uint16_t* const marks = reinterpret_cast<uint16_t*>(s_ctr);
  if (len != 0) {
    marks[slot] = static_cast<uint16_t>(tid + 1);
  }
  __syncthreads();

  // ---- gather: wave w holds slots [64 rounds w, 64 rounds (w + 1)) ----
  const uint32_t rounds = (m + BLOCK - 1) / BLOCK;  // uniform
  const uint32_t first  = wave * rounds * WAVE + lane;
  auto runs             = [&](int i) -> bool { return i < static_cast<int>(rounds); };  // uniform
  auto holds            = [&](int i) -> bool { return runs(i) && first + i * WAVE < m; };
  KeyT key[ITEMS];
  uint32_t pos[HAS_IDX ? ITEMS : 1];
  {
    uint32_t tile[ITEMS], last = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {  // the last mark at or before a slot: in the wave's slots, then in the waves before
      tile[i] = 0;
      if (runs(i)) {
        const uint32_t o = first + i * WAVE;
        tile[i]          = wave_inclusive_max_dpp(o < m ? marks[o] : 0u);
        tile[i]          = tile[i] > last ? tile[i] : last;
        last             = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(tile[i]), WAVE - 1));
      }
    }
    if (lane == 0) {
      s_wave[wave] = last;
    }
    __syncthreads();
    last = 0;
#pragma unroll
    for (uint32_t w = 0; w < WAVES; ++w) {
      last = (w < wave && s_wave[w] > last) ? s_wave[w] : last;
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      key[i] = KeyT{};
      if (runs(i)) {
        const uint32_t o = first + i * WAVE;
        tile[i]          = (tile[i] > last ? tile[i] : last) - 1u;
        const uint32_t a = s_from[tile[i]] + (o < m ? o : m - 1);
        key[i]           = sb.grouped[a];
        if constexpr (HAS_IDX) {
          pos[i] = sb.places[a];
        }
      }
    }
    if constexpr (HAS_IDX) {
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        pos[i] += runs(i) ? tile[i] * sb.tile_len : 0u;
      }
    }
  }
  // ---- the extremes, on the images ----
  KeyT low = 0, high = 0;  // the complement of the smallest, the largest
  int special = 0;         // a NaN or a -0.0 (with positions, ties go by the place in any case)
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    if (holds(i)) {
      const KeyT image = ordered_bits<CODEC, KeyT>(key[i]);
      high             = image > high ? image : high;
      low              = static_cast<KeyT>(~image) > low ? static_cast<KeyT>(~image) : low;
      if constexpr (CODEC == CODEC_FLOAT && !HAS_IDX) {
        special |= is_nan_or_negative_zero(key[i]) ? 1 : 0;
      }
    }
  }
  high = wave_max_dpp(high);
  low  = wave_max_dpp(low);
  __syncthreads();  // (all have read the marks)
  if (lane == 0) {
    s_red[2 * wave]     = static_cast<uint64_t>(high);
    s_red[2 * wave + 1] = static_cast<uint64_t>(low);
  }
  for (uint32_t j = tid; j < BINS / 4; j += BLOCK) {
    reinterpret_cast<uint4*>(s_ctr)[j] = make_uint4(0u, 0u, 0u, 0u);
  }
  special = __syncthreads_or(special);
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const KeyT h = static_cast<KeyT>(s_red[2 * w]), l = static_cast<KeyT>(s_red[2 * w + 1]);
    high = h > high ? h : high;
    low  = l > low ? l : low;
  }
  low = static_cast<KeyT>(~low);
  if (low == high) {  // uniform
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        const uint32_t o = base + first + i * WAVE;
        if (keys_out != nullptr) {
          keys_out[o] = key[i];
        }
        if constexpr (HAS_IDX) {
          idx_out[o] = static_cast<int64_t>(pos[i]) + index_offset;
        }
      }
    }
    return;
  }
  uint32_t to[ITEMS];  // where a key belongs; until then its bin and, in the upper half, which of the bin it is
  bool placed = false;
  if (special == 0 && (CODEC != CODEC_FLOAT || high != static_cast<KeyT>(~KeyT{0}))) {  // uniform
    auto native = [](KeyT k) -> Native {
      Native v;
      __builtin_memcpy(&v, &k, sizeof(Native));
      return v;
    };
    Scale origin = 0, scale = 0;
    int shift = 0;
    if constexpr (CODEC == CODEC_FLOAT) {
      origin = native(sign_unflip<KeyT>(low));
      scale  = static_cast<Scale>(BINS) / (native(sign_unflip<KeyT>(high)) - origin);
    } else {
      const int bits = 64 - __builtin_clzll(static_cast<unsigned long long>(high - low));
      constexpr int LOG2 = 31 - __builtin_clz(BINS);
      shift          = bits > LOG2 ? bits - LOG2 : 0;
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      to[i] = 0;
      if (holds(i)) {
        if constexpr (CODEC == CODEC_FLOAT) {
          // (subtraction, scaling and truncation do not decrease with the key; clamped before the conversion, NaN to 0: an
          // infinite extreme or span crowds a bin)
          const Scale t = (native(key[i]) - origin) * scale;
          if constexpr (sizeof(Scale) == 4) {
            to[i] = static_cast<uint32_t>(__builtin_fminf(__builtin_fmaxf(t, 0.0f), static_cast<float>(BINS - 1)));
          } else {
            to[i] = static_cast<uint32_t>(__builtin_fmin(__builtin_fmax(t, 0.0), static_cast<double>(BINS - 1)));
          }
        } else {
          to[i] = static_cast<uint32_t>(static_cast<KeyT>(ordered_bits<CODEC, KeyT>(key[i]) - low) >> shift);
        }
        to[i] |= atomicAdd(&s_ctr[to[i]], 1u) << 16;
      }
    }
    __syncthreads();
    uint32_t cnt[OWN], total = 0, largest = 0;
#pragma unroll
    for (int c = 0; c < OWN / 4; ++c) {
      const uint4 q  = reinterpret_cast<const uint4*>(s_ctr)[tid * (OWN / 4) + c];
      cnt[4 * c] = q.x, cnt[4 * c + 1] = q.y, cnt[4 * c + 2] = q.z, cnt[4 * c + 3] = q.w;
    }
#pragma unroll
    for (int j = 0; j < OWN; ++j) {
      total += cnt[j];
      largest = cnt[j] > largest ? cnt[j] : largest;
    }
    const uint32_t incl = wave_inclusive_sum_dpp(total);
    if (lane == WAVE - 1) {
      s_wave[wave] = incl;
    }
    placed = __syncthreads_or(largest > SPLIT_BIN_LIMIT ? 1 : 0) == 0;
    if (placed) {
      uint32_t run = incl - total;
#pragma unroll
      for (uint32_t w = 0; w < WAVES; ++w) {
        run += w < wave ? s_wave[w] : 0u;
      }
#pragma unroll
      for (int c = 0; c < OWN / 4; ++c) {
        uint4 e;
        e.x = run, run += cnt[4 * c];
        e.y = run, run += cnt[4 * c + 1];
        e.z = run, run += cnt[4 * c + 2];
        e.w = run, run += cnt[4 * c + 3];
        reinterpret_cast<uint4*>(s_ctr)[tid * (OWN / 4) + c] = e;
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        if (holds(i)) {
          const uint32_t went = s_ctr[to[i] & 0xFFFFu] + (to[i] >> 16);
          s_keys[went]        = key[i];
          if constexpr (HAS_IDX) {
            s_num[went] = static_cast<uint16_t>(first + i * WAVE);
          }
        }
      }
      __syncthreads();
      // (four walks of a thread in step: their reads do not wait for each other.  One past the end of a bin fetches a key of
      // a later bin, or of the padding, and is not counted)
      constexpr int GROUP = 4;
      static_assert(ITEMS % GROUP == 0, "whole groups");
#pragma unroll
      for (int g = 0; g < ITEMS; g += GROUP) {
        if (!runs(g)) {
          break;  // uniform
        }
        uint32_t from[GROUP], length[GROUP], before[GROUP], longest = 0;
#pragma unroll
        for (int k = 0; k < GROUP; ++k) {
          from[k] = 0, length[k] = 0, before[k] = 0;
          if (holds(g + k)) {
            const uint32_t b = to[g + k] & 0xFFFFu;
            from[k]          = s_ctr[b];
            length[k]        = (b + 1 < BINS ? s_ctr[b + 1] : m) - from[k];
            longest          = length[k] > longest ? length[k] : longest;
          }
        }
        for (uint32_t j = 0; j < longest; ++j) {
          KeyT other[GROUP];
          uint32_t number[HAS_IDX ? GROUP : 1];
#pragma unroll
          for (int k = 0; k < GROUP; ++k) {
            other[k] = s_keys[from[k] + j];
            if constexpr (HAS_IDX) {
              number[k] = s_num[from[k] + j];
            }
          }
#pragma unroll
          for (int k = 0; k < GROUP; ++k) {
            const Native a = native(other[k]), b = native(key[g + k]);
            bool earlier;
            if constexpr (HAS_IDX) {
              earlier = (a < b) | ((a == b) & (number[k] < first + (g + k) * WAVE));
            } else {
              earlier = (a < b) | ((a == b) & (j < (to[g + k] >> 16)));
            }
            before[k] += (earlier & (j < length[k])) ? 1u : 0u;
          }
        }
#pragma unroll
        for (int k = 0; k < GROUP; ++k) {
          to[g + k] = from[k] + before[k];
        }
      }
    }
  }
  if (!placed) {
    // ---- the passes: number o of the order so far is s_num[o] ----
    int other_value = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        const KeyT image = ordered_bits<CODEC, KeyT>(key[i]);
        other_value |= (image != low && image != high) ? 1 : 0;
        s_keys[first + i * WAVE] = key[i];
        s_num[first + i * WAVE]  = static_cast<uint16_t>(first + i * WAVE);
      }
    }
    const bool two_values = __syncthreads_or(other_value) == 0;
    const int top         = 64 - __builtin_clzll(static_cast<unsigned long long>(static_cast<KeyT>(low ^ high)));  // bits that vary: below it
    int from_bit          = (!two_values && top > 32) ? top - 32 : 0;
    for (;;) {
      for (int bit = from_bit; bit < top; bit += RADIX_BITS) {
        for (uint32_t j = tid; j < WAVES * RADIX; j += BLOCK) {
          s_ctr[j] = 0;
        }
        __syncthreads();
        uint32_t packed[ITEMS];  // number, digit
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
          if (runs(i)) {
            const uint32_t o = first + i * WAVE;
            const bool valid = o < m;
            const uint32_t k = s_num[valid ? o : m - 1];
            const KeyT image = ordered_bits<CODEC, KeyT>(s_keys[k]);
            const uint32_t d = two_values ? (image == high ? 1u : 0u) : static_cast<uint32_t>(image >> bit) & (RADIX - 1);
            packed[i]        = (k << 8) | d;
            to[i]            = wave_match_rank(d, valid, s_ctr + wave * RADIX);
          }
        }
        __syncthreads();
        uint32_t total = 0;
        if (tid < RADIX) {
#pragma unroll
          for (int w = 0; w < WAVES; ++w) {
            const uint32_t c       = s_ctr[w * RADIX + tid];
            s_ctr[w * RADIX + tid] = total;
            total += c;
          }
        }
        const uint32_t incl = wave_inclusive_sum_dpp(total);
        if (lane == WAVE - 1) {
          s_wave[wave] = incl;
        }
        __syncthreads();
        if (tid < RADIX) {
          uint32_t run = incl - total;
#pragma unroll
          for (uint32_t w = 0; w < RADIX / WAVE; ++w) {
            run += w < wave ? s_wave[w] : 0u;
          }
          s_digit[tid] = run;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
          if (holds(i)) {
            const uint32_t d = packed[i] & (RADIX - 1);
            s_num[s_digit[d] + s_ctr[wave * RADIX + d] + to[i]] = static_cast<uint16_t>(packed[i] >> 8);
          }
        }
        __syncthreads();
        if (two_values) {
          break;
        }
      }
      if (from_bit == 0) {
        break;
      }
      int bad = 0;
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        const uint32_t o = first + i * WAVE;
        if (runs(i) && o + 1 < m) {
          bad |= ordered_bits<CODEC, KeyT>(s_keys[s_num[o]]) > ordered_bits<CODEC, KeyT>(s_keys[s_num[o + 1]]) ? 1 : 0;
        }
      }
      if (__syncthreads_or(bad) == 0) {
        break;
      }
      from_bit = 0;
    }
    // as the walk leaves it: where each key of this thread belongs
    uint32_t number[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        number[i] = s_num[first + i * WAVE];
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        s_num[number[i]] = static_cast<uint16_t>(first + i * WAVE);
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        to[i]  = s_num[first + i * WAVE];
        key[i] = s_keys[first + i * WAVE];
      }
    }
  }
  // ---- out, through LDS, so that neighbouring lanes store neighbouring elements ----
  if (keys_out != nullptr) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        s_keys[to[i]] = key[i];
      }
    }
    __syncthreads();
    for (uint32_t o = tid; o < m; o += BLOCK) {
      keys_out[base + o] = s_keys[o];
    }
  }
  if constexpr (HAS_IDX) {
    uint32_t* const s_pos = reinterpret_cast<uint32_t*>(s_keys);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        s_pos[to[i]] = pos[i];
      }
    }
    __syncthreads();
    for (uint32_t o = tid; o < m; o += BLOCK) {
      idx_out[base + o] = static_cast<int64_t>(s_pos[o]) + index_offset;
    }
  }
}

}  // namespace cpn
