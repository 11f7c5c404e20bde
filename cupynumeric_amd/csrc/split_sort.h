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
// these are drawn from a hash of their number.  A bucket lies between four to 128 sampled keys; the room in LDS is four times
// the mean or more, in the longest rows 1.6 times and more, with as many more sampled keys (split_plan.h).  (Of a bucket with more there is
// one in a million or fewer; only a row that was made for the purpose has many.)
// Such a bucket is sorted by its workgroup in memory, one byte after another (oversized_bucket): slow, and still right.
//
// Stands where the reference calls cub's radix sort or thrust's merge sort of one row
// (src/cupynumeric/sort/cub_sort.cuh:60-151, src/cupynumeric/sort/thrust_sort.cuh:37-66).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "radix_common.h"

namespace cpn {

constexpr int SPLIT_BLOCK       = 1024;
constexpr int SPLIT_BUCKET_BLOCK = 512;
constexpr int SPLIT_BUCKET_ITEMS = 8;
constexpr int SPLIT_WAVES       = SPLIT_BLOCK / WAVE;
constexpr int SPLIT_TILE_ITEMS  = 4;                       // keys per thread of a tile
constexpr int SPLIT_MAX_TILES   = 256;
// rows whose splitters are found ahead (split_wide_tile_kernel)
constexpr int SPLIT_WIDE_MAX_TILES = 1280;
constexpr int SPLIT_WIDE_ITEMS     = 14;
constexpr int SPLIT_WIDE_BINS      = 2;  // per splitter
// Most sampled keys of a bin that are compared with each other (64: 10^6 int32 keys of 200 values, 41 of them in every bin, take 80 us, of
// which the walks are half).
constexpr uint32_t SPLIT_CROWD  = 24;
// Threads with a bin that is not empty: at most so many, and the keys are of a few values (of a bucket, of the sample).
constexpr int SPLIT_FEW         = 12;
constexpr int SPLIT_FEW_SAMPLED = 256;

// A mixed 32-bit word: which key of its stretch sample i takes.  (Chris Wellons' "lowbias32", published with his search for
// integer hashes of 32 bits, constants and shifts.)
__host__ __device__ __forceinline__ uint32_t split_hash(uint32_t x)
{
  x ^= x >> 16;
  x *= 0x7FEB352Du;
  x ^= x >> 15;
  x *= 0x846CA68Bu;
  x ^= x >> 16;
  return x;
}
// The place in a row of n keys that sample i of `samples`, a power of two, is taken from: one place of each of `samples` equal
// stretches.  (By a shift: with two divisions of 64 bits the 524 288 keys that 10^7 are sampled with took 10.9 us to gather.)
__host__ __device__ __forceinline__ uint32_t split_sample_place(uint32_t i, uint32_t samples, uint32_t n)
{
  const int log2      = __builtin_ctz(samples);
  const uint32_t from = static_cast<uint32_t>((static_cast<uint64_t>(i) * n) >> log2);
  const uint32_t to   = static_cast<uint32_t>((static_cast<uint64_t>(i + 1) * n) >> log2);
  return from + static_cast<uint32_t>((static_cast<uint64_t>(split_hash(i)) * (to - from)) >> 32);
}

// The head of the workspace of a row that byte passes may have sorted ahead (split_plan.h, narrow): the status word,
// HEADER_NARROW bytes on whether they did (PlanRequest::narrow, onesweep.h), and, HEADER_WIDE bytes on, what the look at the row
// found (any_wide).  Null: no passes.
constexpr uint64_t HEADER_NARROW     = 8;
constexpr uint64_t HEADER_WIDE       = 64;
constexpr uint32_t SPLIT_WIDE_FLAGS  = 16;
__device__ __forceinline__ bool split_done(const uint32_t* head)
{
  return head != nullptr && head[HEADER_NARROW / 4] != 0 && head[0] == 0;
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

// Puts the numbers of m keys in LDS in the order of their images' bits [from_bit, top), stably: passes of 8 bits, of which
// the numbers move and the keys stay where they are.  num: in, any order; ctr: a counter per wave and digit.  Every thread
// of the workgroup calls, with the same arguments.
template <int CODEC, int BLOCK, int ITEMS, typename KeyT>
__device__ __forceinline__ void split_order_passes(const KeyT* keys, uint16_t* num, uint16_t* ctr, uint32_t* s_wave, uint32_t m, int from_bit,
                                                   int top)
{
  constexpr int WAVES   = BLOCK / WAVE;
  const uint32_t tid    = threadIdx.x;
  const uint32_t lane   = tid & (WAVE - 1);
  const uint32_t wave   = tid / WAVE;
  const uint32_t rounds = (m + BLOCK - 1) / BLOCK;  // uniform
  // (ranks count in the order of waves, rounds and lanes: wave w has numbers [64 rounds w, 64 rounds (w + 1)))
  uint32_t first = wave * rounds * WAVE + lane;
  for (int bit = from_bit; bit < top; bit += RADIX_BITS) {
    asm volatile("" : "+v"(first));  // (or every address below is worked out ahead of the loop, into 160 registers)
    for (uint32_t j = tid; j < WAVES * RADIX / 2; j += BLOCK) {
      reinterpret_cast<uint32_t*>(ctr)[j] = 0;
    }
    __syncthreads();
    uint32_t packed[ITEMS], rank[ITEMS];  // number and digit
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      packed[i] = 0, rank[i] = 0;
      if (i < static_cast<int>(rounds)) {
        const uint32_t o = first + i * WAVE;
        const bool valid = o < m;
        const uint32_t k = num[valid ? o : m - 1];
        const uint32_t d = static_cast<uint32_t>(ordered_bits<CODEC, KeyT>(keys[k]) >> bit) & (RADIX - 1);
        packed[i]        = (k << 8) | d;
        rank[i]          = split_match_rank<RADIX_BITS>(d, valid, ctr + wave * RADIX);
      }
    }
    __syncthreads();
    uint32_t total = 0;
    if (tid < RADIX) {
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        const uint32_t c     = ctr[w * RADIX + tid];
        ctr[w * RADIX + tid] = static_cast<uint16_t>(total);
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
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        ctr[w * RADIX + tid] = static_cast<uint16_t>(ctr[w * RADIX + tid] + run);
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (i < static_cast<int>(rounds) && first + i * WAVE < m) {
        num[ctr[wave * RADIX + (packed[i] & (RADIX - 1))] + rank[i]] = static_cast<uint16_t>(packed[i] >> 8);
      }
    }
    __syncthreads();
  }
}
// The same for all bits that vary (`vary` has those in which any key's image differs from another's).  The leading 40 put almost
// every row in order, the leading 16 one of a few values that repeat: passes over them, a look at every pair of neighbours,
// and more passes if one is not in order.  (Every pass is stable, and so is what follows another.)  Nothing is done for low bits that
// all keys share, as those of whole numbers held as floats do.  us a sort, 40 bits of any key at first / this: 10^7 float64 of 20 000
// whole numbers 370 / 250, 10^6 int64 of 100 values 70 / 55; with 16 bits first for all, normal float64 with 1 % zeros lost 5 %.
template <int CODEC, int BLOCK, int ITEMS, typename KeyT>
__device__ __forceinline__ void split_order(const KeyT* keys, uint16_t* num, uint16_t* ctr, uint32_t* s_wave, uint32_t m, uint64_t vary,
                                            bool few)
{
  const int top    = vary != 0 ? 64 - __builtin_clzll(vary) : 0;
  const int bottom = vary != 0 ? __builtin_ctzll(vary) : 0;
  for (int bits = few ? 16 : 40;; bits = bits == 16 ? 40 : 64) {
    const int from_bit = top - bits > bottom ? top - bits : bottom;
    split_order_passes<CODEC, BLOCK, ITEMS>(keys, num, ctr, s_wave, m, from_bit, top);
    if (from_bit == bottom) {
      return;
    }
    int bad = 0;
    for (uint32_t o = threadIdx.x; o + 1 < m; o += BLOCK) {
      bad |= ordered_bits<CODEC, KeyT>(keys[num[o]]) > ordered_bits<CODEC, KeyT>(keys[num[o + 1]]) ? 1 : 0;
    }
    if (__syncthreads_or(bad) == 0) {
      return;
    }
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
// room for their images, their numbers, and the counters of passes over them.
template <typename KeyT, int PER_THREAD, int PER_BUCKET>
struct SplitSample {
  static constexpr int SAMPLES   = PER_THREAD * SPLIT_BLOCK;
  static constexpr int SPLITTERS = SAMPLES / PER_BUCKET;
  static constexpr int WHICH     = SAMPLES * static_cast<int>(sizeof(KeyT));
  static constexpr int COUNTERS  = WHICH + SAMPLES * 2;
  static constexpr int EXTREMES  = COUNTERS + SPLIT_WAVES * RADIX * 2;
  static constexpr int BYTES     = EXTREMES + 2 * SPLIT_WAVES * static_cast<int>(sizeof(KeyT));
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
// sample that crowds its bins (few different values, values of many magnitudes) goes through passes over its bytes.
template <int CODEC, int PER_THREAD, int PER_BUCKET, typename KeyT, typename Put>
__device__ __forceinline__ SplitBins split_find_splitters(uint32_t n, unsigned char* s_mem, uint32_t* s_bins, uint32_t* s_wave, uint32_t* s_low,
                                                          const KeyT (&got)[PER_THREAD], Put put)
{
  using S                = SplitSample<KeyT, PER_THREAD, PER_BUCKET>;
  constexpr int SAMPLES  = S::SAMPLES;
  const uint32_t tid     = threadIdx.x;
  const uint32_t lane    = tid & (WAVE - 1);
  const uint32_t wave    = tid / WAVE;
  KeyT* const s_image     = reinterpret_cast<KeyT*>(s_mem);
  uint16_t* const s_which = reinterpret_cast<uint16_t*>(s_mem + S::WHICH);
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
    KeyT* const s_ext = reinterpret_cast<KeyT*>(s_mem + S::EXTREMES);
    const bool few = __syncthreads_count(sum != 0 ? 1 : 0) <= SPLIT_FEW_SAMPLED;
    KeyT any = 0, all = static_cast<KeyT>(~KeyT{0});  // OR and AND of the images
#pragma unroll
    for (int r = 0; r < PER_THREAD; ++r) {
      const KeyT image                 = ordered_bits<CODEC, KeyT>(got[r]);
      any |= image;
      all &= image;
      s_image[r * SPLIT_BLOCK + tid]   = image;
      s_which[r * SPLIT_BLOCK + tid]   = static_cast<uint16_t>(r * SPLIT_BLOCK + tid);
    }
    any = wave_reduce_or_dpp(any);
    all = wave_reduce_and_dpp(all);
    if (lane == 0) {
      s_ext[wave]               = any;
      s_ext[SPLIT_WAVES + wave] = all;
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < SPLIT_WAVES; ++v) {
      any |= s_ext[v];
      all &= s_ext[SPLIT_WAVES + v];
    }
    split_order<CODEC_UNSIGNED, SPLIT_BLOCK, PER_THREAD>(s_image, s_which, reinterpret_cast<uint16_t*>(s_mem + S::COUNTERS), s_wave,
                                                         static_cast<uint32_t>(SAMPLES), static_cast<uint64_t>(any ^ all), few);
    for (uint32_t j = number; j < S::SPLITTERS; j += SPLIT_BLOCK) {
      const uint32_t i = s_which[j * PER_BUCKET];
      put(j, s_image[i], split_sample_place(i, SAMPLES, n));
    }
  }
  return bins;
}

// The sampled keys of the row, gathered by many workgroups: one alone reads a thousand scattered keys in 2.5 us, and so
// does each of the workgroups that need all of them.
template <typename KeyT>
__global__ __launch_bounds__(256) void split_gather_kernel(const KeyT* __restrict__ keys_in, uint32_t n, uint32_t samples,
                                                           KeyT* __restrict__ out, const uint32_t* __restrict__ head)
{
  if (split_done(head)) {
    return;
  }
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;  // (`samples` is a multiple of the workgroup)
  out[i]           = keys_in[split_sample_place(i, samples, n)];
}
// The same as the first launch of a row that may be narrow.  It also gathers what the sample's own sort samples (`again` keys of
// it; 10^7 keys 2 us less than by a launch), clears what the passes count with, from the head of the workspace on, and the first
// SPLIT_WIDE_FLAGS workgroups look at the keys that they gather, 4096 in all: where these differ in no bit of `outside`, the passes are
// to try.  (One workgroup that looks at 4096 keys of its own takes 5 us longer than all the others.)
template <typename KeyT, int CODEC>
__global__ __launch_bounds__(256) void split_front_kernel(const KeyT* __restrict__ keys_in, uint32_t n, uint32_t samples,
                                                          KeyT* __restrict__ out, uint32_t again, KeyT* __restrict__ out_again,
                                                          uint4* __restrict__ clear, uint32_t n_clear, KeyT outside)
{
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  const KeyT own   = keys_in[split_sample_place(i, samples, n)];
  if (i < again) {
    out_again[i] = keys_in[split_sample_place(split_sample_place(i, again, samples), samples, n)];
  }
  for (uint32_t v = i; v < n_clear; v += samples) {
    if (v < HEADER_WIDE / 16 || v >= HEADER_WIDE / 16 + SPLIT_WIDE_FLAGS / 4) {
      clear[v] = make_uint4(0u, 0u, 0u, 0u);
    }
  }
  if (blockIdx.x < SPLIT_WIDE_FLAGS) {
    const KeyT vary = ordered_bits<CODEC, KeyT>(own) ^ ordered_bits<CODEC, KeyT>(keys_in[0]);
    const int wide  = __syncthreads_or((vary & outside) != 0 ? 1 : 0);
    if (threadIdx.x == 0) {
      (reinterpret_cast<uint32_t*>(clear) + HEADER_WIDE / 4)[blockIdx.x] = wide != 0 ? 1u : 0u;
    }
  }
  out[i] = own;
}
// What passes leave undone: a row of equal keys, and a row sorted in place, which they leave in a buffer.
template <typename KeyT>
struct SplitLeft {
  const KeyT* sorted;  // null: not in place
  KeyT* keys_out;      // may be null
  int64_t* idx_out;    // may be null
  int64_t index_offset;
};
template <typename KeyT>
__device__ __forceinline__ void split_finish(const SplitLeft<KeyT>& left, const KeyT* keys_in, bool equal, uint32_t first, uint32_t len)
{
  const KeyT* const from = equal ? keys_in : left.sorted;
  if (left.keys_out != nullptr && from != nullptr && from != left.keys_out) {
    for (uint32_t o = first + threadIdx.x; o < first + len; o += SPLIT_BLOCK) {
      left.keys_out[o] = from[o];
    }
  }
  if (equal && left.idx_out != nullptr) {
    for (uint32_t o = first + threadIdx.x; o < first + len; o += SPLIT_BLOCK) {
      left.idx_out[o] = static_cast<int64_t>(o) + left.index_offset;
    }
  }
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
                                                                 uint16_t* __restrict__ starts, uint32_t* __restrict__ status,
                                                                 const uint32_t* __restrict__ head)
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
  if (split_done(head)) {
    return;  // uniform
  }
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
  const SplitBins bins   = split_find_splitters<CODEC, PER_THREAD, PER_BUCKET>(n, s_mem, s_bins, s_wave, s_low, got,
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

// ---- rows whose splitters are found ahead ----
// Longer rows take more buckets and more sampled keys than a tile's workgroup can sort by the way: the sample is gathered,
// sorted as a row of its own (by the kernels above and below), and every (samples / buckets)-th key of it is a splitter.

// Where the sort of a sample leaves the splitters.
template <typename KeyT>
struct SplitPicks {
  KeyT* images;
  uint32_t* places;
  float* values;
  uint32_t log2_step;   // of 2^log2_step sampled keys one is a splitter
  uint32_t samples, n;  // of a row of n keys
};

// The bins of the splitters' values, and how many splitters come before each (one workgroup).
template <int BITS>
__global__ __launch_bounds__(SPLIT_BLOCK) void split_table_kernel(const float* __restrict__ values, uint16_t* __restrict__ before,
                                                                  SplitBins* __restrict__ bins_out, const uint32_t* __restrict__ passes,
                                                                  uint32_t* __restrict__ head)
{
  constexpr int BUCKETS = 1 << BITS;
  constexpr int BINS    = BUCKETS * SPLIT_WIDE_BINS;
  constexpr int OWN     = BUCKETS / SPLIT_BLOCK;  // splitters of a thread
  constexpr int SPAN    = BINS / SPLIT_BLOCK;     // bins of a thread
  __shared__ uint32_t s_bins[BINS];
  __shared__ uint32_t s_wave[SPLIT_WAVES], s_low[SPLIT_WAVES];
  const uint32_t tid  = threadIdx.x;
  const uint32_t lane = tid & (WAVE - 1);
  const uint32_t wave = tid / WAVE;
  if (split_done(passes)) {
    return;
  }
  float value[OWN];
  uint32_t low = 0, high = 0;  // as in split_find_splitters
#pragma unroll
  for (int r = 0; r < OWN; ++r) {
    value[r]             = values[r * SPLIT_BLOCK + tid];
    const bool finite    = __builtin_fabsf(value[r]) < __builtin_huge_valf();
    const uint32_t image = sign_flip<uint32_t>(__float_as_uint(value[r]));
    high                 = finite && image > high ? image : high;
    low                  = finite && ~image > low ? ~image : low;
  }
  high = wave_inclusive_max_dpp(high);
  low  = wave_inclusive_max_dpp(low);
  if (lane == WAVE - 1) {
    s_wave[wave] = high;
    s_low[wave]  = low;
  }
#pragma unroll
  for (int r = 0; r < SPAN; ++r) {
    s_bins[r * SPLIT_BLOCK + tid] = 0;
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
  bins.scale       = span > 0.0f ? static_cast<float>(BINS) / span : 0.0f;
#pragma unroll
  for (int r = 0; r < OWN; ++r) {
    if (r * SPLIT_BLOCK + tid != 0) {  // (splitter 0 does not count)
      atomicAdd(&s_bins[split_bin<BINS>(bins, value[r])], 1u);
    }
  }
  __syncthreads();
  uint32_t count[SPAN], sum = 0;
#pragma unroll
  for (int r = 0; r < SPAN; ++r) {
    count[r] = s_bins[tid * SPAN + r];
    sum += count[r];
  }
  const uint32_t sums = wave_inclusive_sum_dpp(sum);
  if (lane == WAVE - 1) {
    s_wave[wave] = sums;
  }
  __syncthreads();
  uint32_t run = sums - sum + split_waves_before(s_wave, wave);
#pragma unroll
  for (int r = 0; r < SPAN; ++r) {
    before[tid * SPAN + r] = static_cast<uint16_t>(run);
    run += count[r];
  }
  if (tid == 0) {
    *bins_out = bins;
    // (also where passes have given up, see split_done: this sort cannot fail on the device)
    head[HEADER_NARROW / 4] = 0;
    head[0]                 = 0;
  }
}

// split_tile_kernel for these rows: tiles of up to 14 336 keys, 1024 to 4096 buckets.  The splitters, then the counters of
// the ranks (a 16-bit word per wave and bucket), then the tile itself take turns in the same 140 KiB.
template <typename KeyT, int CODEC, bool HAS_POS, int BITS>
__global__ __launch_bounds__(SPLIT_BLOCK) void split_wide_tile_kernel(const KeyT* __restrict__ keys_in, uint32_t n, uint32_t tile_len,
                                                                      const KeyT* __restrict__ images,
                                                                      const uint32_t* __restrict__ split_places,
                                                                      const uint16_t* __restrict__ before,
                                                                      const SplitBins* __restrict__ bins_in,
                                                                      KeyT* __restrict__ grouped, uint16_t* __restrict__ places,
                                                                      uint16_t* __restrict__ starts, const uint32_t* __restrict__ head,
                                                                      const SplitLeft<KeyT> left)
{
  constexpr int ITEMS    = SPLIT_WIDE_ITEMS;
  constexpr int BUCKETS  = 1 << BITS;
  constexpr int BINS     = BUCKETS * SPLIT_WIDE_BINS;
  constexpr int TILE     = SPLIT_BLOCK * ITEMS;
  constexpr int OWN      = BUCKETS / SPLIT_BLOCK;  // buckets a thread scans
  constexpr int S_BYTES  = BUCKETS * (static_cast<int>(sizeof(KeyT)) + 4) + BINS * 2;
  constexpr int C_BYTES  = SPLIT_WAVES * BUCKETS * 2 + BUCKETS * 2;
  constexpr int K_BYTES  = TILE * (static_cast<int>(sizeof(KeyT)) + (HAS_POS ? 2 : 0));
  constexpr int SC_BYTES = S_BYTES > C_BYTES ? S_BYTES : C_BYTES;
  static_assert(OWN == 1 || OWN == 2 || OWN == 4, "a thread's buckets are one word of the counters");
  using Word = std::conditional_t<OWN == 1, uint16_t, std::conditional_t<OWN == 2, uint32_t, uint64_t>>;
  __shared__ __align__(16) unsigned char s_mem[SC_BYTES > K_BYTES ? SC_BYTES : K_BYTES];
  __shared__ uint32_t s_wave[SPLIT_WAVES];

  const uint32_t tid    = threadIdx.x;
  const uint32_t lane   = tid & (WAVE - 1);
  const uint32_t wave   = tid / WAVE;
  const uint32_t first  = blockIdx.x * tile_len;
  const uint32_t len    = n - first < tile_len ? n - first : tile_len;  // (no tile is empty)
  const uint32_t rounds = (len + SPLIT_BLOCK - 1) / SPLIT_BLOCK;        // uniform
  const uint32_t woff   = wave * rounds * WAVE + lane;
  auto runs             = [&](int i) -> bool { return i < static_cast<int>(rounds); };  // uniform
  if (split_done(head)) {
    split_finish(left, keys_in, head[HEADER_NARROW / 4] == 2, first, len);
    return;
  }

  KeyT key[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t o = woff + i * WAVE;
    key[i]           = KeyT{};
    if (runs(i)) {
      key[i] = keys_in[first + (o < len ? o : len - 1)];
    }
  }
  KeyT* const s_split        = reinterpret_cast<KeyT*>(s_mem);
  uint32_t* const s_split_at = reinterpret_cast<uint32_t*>(s_mem + BUCKETS * sizeof(KeyT));
  uint16_t* const s_before   = reinterpret_cast<uint16_t*>(s_mem + BUCKETS * (sizeof(KeyT) + 4));
#pragma unroll
  for (int r = 0; r < OWN; ++r) {
    s_split[r * SPLIT_BLOCK + tid]    = images[r * SPLIT_BLOCK + tid];
    s_split_at[r * SPLIT_BLOCK + tid] = split_places[r * SPLIT_BLOCK + tid];
  }
#pragma unroll
  for (int r = 0; r < BINS / 2 / SPLIT_BLOCK; ++r) {
    reinterpret_cast<uint32_t*>(s_before)[r * SPLIT_BLOCK + tid] = reinterpret_cast<const uint32_t*>(before)[r * SPLIT_BLOCK + tid];
  }
  const SplitBins bins = *bins_in;
  __syncthreads();
  // ---- buckets, as in split_tile_kernel, GROUP keys of a thread at a time ----
  uint32_t where[ITEMS];  // bucket; later, in the upper half, the rank; then where the key goes
  constexpr int GROUP = 7;
  static_assert(ITEMS % GROUP == 0, "whole groups");
#pragma unroll
  for (int g = 0; g < ITEMS; g += GROUP) {
    uint32_t left[GROUP];
#pragma unroll
    for (int k = 0; k < GROUP; ++k) {
      const uint32_t bin = split_bin<BINS>(bins, split_value<CODEC, KeyT>(key[g + k]));
      where[g + k]       = s_before[bin];
      left[k]            = (bin + 1 < BINS ? s_before[bin + 1] : static_cast<uint32_t>(BUCKETS - 1)) - where[g + k];
    }
    for (;;) {
      uint32_t most = 0;
#pragma unroll
      for (int k = 0; k < GROUP; ++k) {
        most = left[k] > most ? left[k] : most;
      }
      if (__ballot(most != 0) == 0) {
        break;
      }
#pragma unroll
      for (int k = 0; k < GROUP; ++k) {
        const uint32_t at   = first + woff + (g + k) * WAVE;
        const uint32_t half = (left[k] + 1) / 2;
        const uint32_t c    = where[g + k] + half;
        const KeyT image    = ordered_bits<CODEC, KeyT>(key[g + k]);
        const KeyT split    = s_split[c];
        const bool reached  = (split < image) | ((split == image) & (s_split_at[c] <= at));
        where[g + k]        = reached ? c : where[g + k];
        left[k]             = left[k] == 0 ? 0 : (reached ? left[k] - half : half - 1);
      }
    }
  }
  __syncthreads();
  // ---- ranks ----
  uint16_t* const s_ctr  = reinterpret_cast<uint16_t*>(s_mem);
  uint16_t* const s_base = s_ctr + SPLIT_WAVES * BUCKETS;
  for (uint32_t j = tid; j < SPLIT_WAVES * BUCKETS * 2 / 16; j += SPLIT_BLOCK) {
    reinterpret_cast<uint4*>(s_mem)[j] = make_uint4(0u, 0u, 0u, 0u);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    if (runs(i)) {
      where[i] |= split_match_rank<BITS>(where[i], woff + i * WAVE < len, s_ctr + wave * BUCKETS) << 16;
    }
  }
  __syncthreads();
  uint64_t totals = 0;  // of the thread's buckets, 16 bits each (a tile has fewer than 2^16 keys)
  {
    Word* const own = reinterpret_cast<Word*>(s_ctr) + tid;
#pragma unroll
    for (int v = 0; v < SPLIT_WAVES; ++v) {
      const uint64_t c   = own[v * SPLIT_BLOCK];
      own[v * SPLIT_BLOCK] = static_cast<Word>(totals);
      totals += c;
    }
  }
  uint32_t sum = 0;
#pragma unroll
  for (int r = 0; r < OWN; ++r) {
    sum += static_cast<uint32_t>(totals >> (16 * r)) & 0xFFFFu;
  }
  const uint32_t sums = wave_inclusive_sum_dpp(sum);
  if (lane == WAVE - 1) {
    s_wave[wave] = sums;
  }
  __syncthreads();
  {
    uint32_t run       = sums - sum + split_waves_before(s_wave, wave);
    uint16_t* const to = starts + static_cast<uint64_t>(blockIdx.x) * (BUCKETS + 1);
#pragma unroll
    for (int r = 0; r < OWN; ++r) {
      s_base[tid * OWN + r] = static_cast<uint16_t>(run);
      to[tid * OWN + r]     = static_cast<uint16_t>(run);
      run += static_cast<uint32_t>(totals >> (16 * r)) & 0xFFFFu;
    }
    if (tid == 0) {
      to[BUCKETS] = static_cast<uint16_t>(len);
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t b = where[i] & 0xFFFFu;
    where[i]         = s_base[b] + s_ctr[wave * BUCKETS + b] + (where[i] >> 16);
  }
  __syncthreads();
  // ---- the tile in the order of its buckets ----
  KeyT* const s_keys      = reinterpret_cast<KeyT*>(s_mem);
  uint16_t* const s_place = reinterpret_cast<uint16_t*>(s_mem + TILE * sizeof(KeyT));
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t o = woff + i * WAVE;
    if (runs(i) && o < len) {
      s_keys[where[i]] = key[i];
      if constexpr (HAS_POS) {
        s_place[where[i]] = static_cast<uint16_t>(o);
      }
    }
  }
  __syncthreads();
  for (uint32_t o = tid; o < len; o += SPLIT_BLOCK) {
    grouped[first + o] = s_keys[o];
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
  const uint32_t* head;
};

// A bucket of more keys than LDS has room for, sorted by its workgroup alone: one stable pass per key byte over the
// numbers of its keys, which go back and forth between two arrays in memory.  A turn of BLOCK keys takes about 2 us.
//   s_from  [tiles]: where the part of a tile lies in `grouped`, less where it lies in the bucket (modulo 2^32)
//   s_slot  [tiles]: where it lies in the bucket
//   s_ctr   a counter per digit and wave, s_digit: one per digit
//   put_key, put_pos  take the bucket's o-th key and its place in the row
template <typename KeyT, int CODEC, bool HAS_IDX, int BLOCK, typename PutKey, typename PutPos>
__device__ __forceinline__ void oversized_bucket(const SplitBuckets<KeyT>& sb, uint32_t m, uint32_t base,
                                                 const uint32_t* s_from, const uint32_t* s_slot, uint32_t* s_ctr,
                                                 uint32_t* s_digit, PutKey put_key, PutPos put_pos)
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
    put_key(i, sb.grouped[at]);
    if constexpr (HAS_IDX) {
      put_pos(i, t * sb.tile_len + sb.places[at]);
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

// Most keys of a bin that are compared with each other.  (192 of them: 10^5 keys of a hundred values 50 us instead of 19,
// 10^6 with a hundredth of NaNs and zeros 72 instead of 66: the longest walk of a wave is everyone's.)
constexpr uint32_t SPLIT_BIN_LIMIT = 24;

// One bucket of a row: its parts of all tiles gathered, sorted, stored.
//   a bucket of equal images is in order: it was gathered in the order of the row
//   others are spread over four bins per thread (WIDE: eight), of equal width between their smallest and their largest key; one atomic per key
//     says which of its bin it is, a scan where the bin starts, a walk over the bin how many of its keys come before
//   buckets with a crowded bin: passes over the bytes of the images, of which numbers of keys move and the keys
//     stay where they are in LDS.  One pass where there are two values
// Ties go by the place in the gathered order.
// Neighbouring buckets, whose parts of a tile share cache lines, go to neighbouring workgroups of one XCD.
// Bound by its chain where every bucket has a compute unit (7 to 8 us for buckets of 400 keys; as one more mode of
// lds_row_sort_kernel, with two reductions and two atomics per key, 11), else by the workgroups that fit, two to a unit of
// 512 threads with 8-byte keys, three with 4-byte keys.
// PICK: of a sample's sort nothing is kept but the splitters.  (A launch of its own that looked them up took 4 us.)
template <typename KeyT, int CODEC, bool HAS_IDX, bool WIDE, bool PICK>
__global__ __launch_bounds__(SPLIT_BUCKET_BLOCK) void split_bucket_kernel(const SplitBuckets<KeyT> sb, KeyT* __restrict__ keys_out,
                                                             int64_t* __restrict__ idx_out, int64_t index_offset,
                                                             const SplitPicks<KeyT> picks)
{
  constexpr int BLOCK = SPLIT_BUCKET_BLOCK;
  constexpr int ITEMS = SPLIT_BUCKET_ITEMS;
  constexpr int WAVES = BLOCK / WAVE;
  constexpr int TILE  = BLOCK * ITEMS;
  constexpr int BINS  = (WIDE ? 8 : 4) * BLOCK;
  constexpr int TILES = WIDE ? SPLIT_WIDE_MAX_TILES : SPLIT_MAX_TILES;
  constexpr int PARTS = (TILES + BLOCK - 1) / BLOCK;  // tiles per thread
  constexpr int OWN   = BINS / BLOCK;  // bins a thread scans
  static_assert(OWN % 4 == 0, "whole vectors");
  static_assert(PARTS * BLOCK >= TILES && BLOCK >= RADIX, "a thread per digit");
  static_assert(TILE <= 65536 && BINS <= 65536, "numbers of 16 bits");
  constexpr int WORDS0 = BINS > WAVES * RADIX ? BINS : WAVES * RADIX;
  constexpr int WORDS  = WORDS0 > TILE / 2 ? WORDS0 : TILE / 2;
  constexpr bool BY_PLACE = HAS_IDX || CODEC == CODEC_FLOAT;  // (integers that tie are the same bits)
  using Native         = typename SplitNative<CODEC, sizeof(KeyT)>::type;
  using Scale          = std::conditional_t<sizeof(KeyT) == 4, float, double>;
  __shared__ __align__(16) KeyT s_keys[TILE + SPLIT_BIN_LIMIT];
  __shared__ uint16_t s_num[TILE + SPLIT_BIN_LIMIT];
  __shared__ __align__(16) uint32_t s_ctr[WORDS];  // marks of tiles, bins, counters of digits
  __shared__ uint32_t s_from[TILES];
  uint32_t* const s_slot = reinterpret_cast<uint32_t*>(s_keys);  // (an oversized bucket's)
  static_assert(TILES * 4 <= TILE * sizeof(KeyT), "a word per tile");
  __shared__ uint64_t s_red[2 * WAVES];
  __shared__ uint32_t s_wave[WAVES];
  static_assert(ITEMS * WAVES <= WAVE, "a lane per wave and round");
  __shared__ uint32_t s_last[WAVE];
  uint32_t* const s_digit = reinterpret_cast<uint32_t*>(s_num);  // (an oversized bucket's)
  static_assert(RADIX * 4 <= TILE * 2 && RADIX <= TILES, "a word per digit");

  const uint32_t tid    = threadIdx.x;
  const uint32_t lane   = tid & (WAVE - 1);
  const uint32_t wave   = tid / WAVE;
  constexpr uint32_t XCDS = 8;  // workgroups go round them
  const uint32_t bucket   = blockIdx.x % XCDS * (sb.buckets / XCDS) + blockIdx.x / XCDS;
  if (split_done(sb.head)) {
    return;  // uniform
  }

  // ---- the bucket's part of every tile; m keys in all, `base` keys of the row before them ----
  uint32_t start[PARTS], len[PARTS], starts = 0, lens = 0;
#pragma unroll
  for (int k = 0; k < PARTS; ++k) {
    start[k] = 0, len[k] = 0;
    if (tid * PARTS + k < sb.tiles) {
      const uint16_t* const at = sb.starts + static_cast<uint64_t>(tid * PARTS + k) * (sb.buckets + 1) + bucket;
      start[k]                 = at[0];
      len[k]                   = at[1] - start[k];
    }
    starts += start[k];
    lens += len[k];
  }
  const uint32_t incl_len   = wave_inclusive_sum_dpp(lens);
  const uint32_t incl_start = wave_inclusive_sum_dpp(starts);
  if (lane == WAVE - 1) {
    s_red[wave] = (static_cast<uint64_t>(incl_start) << 32) | incl_len;
  }
  for (uint32_t j = tid; j < TILE / 8; j += BLOCK) {
    reinterpret_cast<uint4*>(s_ctr)[j] = make_uint4(0u, 0u, 0u, 0u);
  }
  __syncthreads();
  uint32_t slot = incl_len - lens, m = 0, base = 0;
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
  auto put_key = [&](uint32_t o, KeyT key) {
    if constexpr (PICK) {
      const uint32_t at = base + o;
      if ((at & ((1u << picks.log2_step) - 1)) == 0) {
        picks.images[at >> picks.log2_step] = ordered_bits<CODEC, KeyT>(key);
        picks.values[at >> picks.log2_step] = split_value<CODEC, KeyT>(key);
      }
    } else if (keys_out != nullptr) {
      keys_out[base + o] = key;
    }
  };
  auto put_pos = [&](uint32_t o, uint32_t pos) {
    if constexpr (PICK) {
      const uint32_t at = base + o;
      if ((at & ((1u << picks.log2_step) - 1)) == 0) {
        picks.places[at >> picks.log2_step] = split_sample_place(pos, picks.samples, picks.n);
      }
    } else {
      idx_out[base + o] = static_cast<int64_t>(pos) + index_offset;
    }
  };
  static_assert(HAS_IDX || !PICK, "splitters have places");
  uint32_t part_slot[PARTS];
#pragma unroll
  for (int k = 0; k < PARTS; ++k) {
    const uint32_t t = tid * PARTS + k;
    part_slot[k]     = slot;
    if (t < sb.tiles) {
      s_from[t] = t * sb.tile_len + start[k] - slot;
      if (m > TILE) {
        s_slot[t] = slot;
      }
    }
    slot += len[k];
  }
  if (m > TILE) {  // uniform
    __syncthreads();
    oversized_bucket<KeyT, CODEC, HAS_IDX, BLOCK>(sb, m, base, s_from, s_slot, s_ctr, s_digit, put_key, put_pos);
    return;
  }
  // the number of a tile, plus one, at the first slot of its part
  uint16_t* const marks = reinterpret_cast<uint16_t*>(s_ctr);
#pragma unroll
  for (int k = 0; k < PARTS; ++k) {
    if (len[k] != 0) {
      marks[part_slot[k]] = static_cast<uint16_t>(tid * PARTS + k + 1);
    }
  }
  __syncthreads();

  // ---- gather: slot number i * BLOCK + tid is a thread's i-th ----
  auto slot_of = [&](int i) -> uint32_t { return i * BLOCK + tid; };
  auto holds   = [&](int i) -> bool { return slot_of(i) < m; };
  KeyT key[ITEMS];
  uint32_t pos[HAS_IDX ? ITEMS : 1];
  {
    // the tile that a slot belongs to: the last mark at or before it, among the 64 slots of its wave and round, then in
    // those before
    uint32_t tile[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      tile[i] = wave_inclusive_max_dpp(holds(i) ? marks[slot_of(i)] : 0u);
      if (lane == WAVE - 1) {
        s_last[i * WAVES + wave] = tile[i];
      }
    }
    __syncthreads();
    const uint32_t lasts = wave_inclusive_max_dpp(lane < ITEMS * WAVES ? s_last[lane] : 0u);
    const int uwave      = __builtin_amdgcn_readfirstlane(static_cast<int>(wave));
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int e           = i * WAVES + uwave;
      const uint32_t before = e != 0 ? static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(lasts), e - 1)) : 0u;
      tile[i]               = (tile[i] > before ? tile[i] : before) - 1u;
      const uint32_t a      = s_from[tile[i]] + (holds(i) ? slot_of(i) : m - 1);
      key[i]                = sb.grouped[a];
      if constexpr (HAS_IDX) {
        pos[i] = sb.places[a];
      }
    }
    if constexpr (HAS_IDX) {
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        pos[i] += tile[i] * sb.tile_len;
      }
    }
  }
  // ---- the extremes, on the images ----
  constexpr KeyT NAN_IMAGE = static_cast<KeyT>(~KeyT{0});  // (float keys)
  KeyT low = 0, high = 0;  // the complement of the smallest, the largest that is no NaN
  int nans = 0;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    if (holds(i)) {
      const KeyT image = ordered_bits<CODEC, KeyT>(key[i]);
      const bool nan   = CODEC == CODEC_FLOAT && image == NAN_IMAGE;
      high             = !nan && image > high ? image : high;
      low              = static_cast<KeyT>(~image) > low ? static_cast<KeyT>(~image) : low;
      nans |= nan ? 1 : 0;
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
  nans = __syncthreads_or(nans);
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const KeyT h = static_cast<KeyT>(s_red[2 * w]), l = static_cast<KeyT>(s_red[2 * w + 1]);
    high = h > high ? h : high;
    low  = l > low ? l : low;
  }
  low = static_cast<KeyT>(~low);
  if (low == NAN_IMAGE ? (CODEC == CODEC_FLOAT || high == NAN_IMAGE) : (low == high && nans == 0)) {  // uniform: one image
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        put_key(slot_of(i), key[i]);
        if constexpr (HAS_IDX) {
          put_pos(slot_of(i), pos[i]);
        }
      }
    }
    return;
  }
  uint32_t to[ITEMS];  // where a key belongs; until then its bin and, in the upper half, which of the bin it is
  bool placed = false, few = false;
  {
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
          // (subtraction, scaling and truncation do not decrease with the key; clamped before the conversion: an infinite
          // extreme or span crowds a bin.  NaNs: the last bin)
          const Native v = native(key[i]);
          const Scale t  = (v - origin) * scale;
          if constexpr (sizeof(Scale) == 4) {
            to[i] = static_cast<uint32_t>(__builtin_fminf(__builtin_fmaxf(t, 0.0f), static_cast<float>(BINS - 1)));
          } else {
            to[i] = static_cast<uint32_t>(__builtin_fmin(__builtin_fmax(t, 0.0), static_cast<double>(BINS - 1)));
          }
          to[i] = v != v ? BINS - 1 : to[i];
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
    if (!placed) {
      few = __syncthreads_count(total != 0 ? 1 : 0) <= SPLIT_FEW;
    }
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
          s_keys[went]        = ordered_bits<CODEC, KeyT>(key[i]);
          if constexpr (BY_PLACE) {
            s_num[went] = static_cast<uint16_t>(slot_of(i));
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
          uint32_t number[BY_PLACE ? GROUP : 1];
#pragma unroll
          for (int k = 0; k < GROUP; ++k) {
            other[k] = s_keys[from[k] + j];
            if constexpr (BY_PLACE) {
              number[k] = s_num[from[k] + j];
            }
          }
#pragma unroll
          for (int k = 0; k < GROUP; ++k) {
            const KeyT image = ordered_bits<CODEC, KeyT>(key[g + k]);
            bool earlier;
            if constexpr (BY_PLACE) {
              earlier = (other[k] < image) | ((other[k] == image) & (number[k] < slot_of(g + k)));
            } else {
              earlier = (other[k] < image) | ((other[k] == image) & (j < (to[g + k] >> 16)));
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
    high = nans != 0 ? NAN_IMAGE : high;
    // ---- the passes: number o of the order so far is s_num[o] ----
    int other_value = 0;
    KeyT vary       = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        const KeyT image = ordered_bits<CODEC, KeyT>(key[i]);
        other_value |= (image != low && image != high) ? 1 : 0;
        vary |= image ^ low;
        s_keys[slot_of(i)] = key[i];
        s_num[slot_of(i)]  = static_cast<uint16_t>(slot_of(i));
      }
    }
    vary = wave_reduce_or_dpp(vary);
    if (lane == 0) {
      s_red[wave] = static_cast<uint64_t>(vary);  // (the extremes in it have been read)
    }
    uint16_t* const c = reinterpret_cast<uint16_t*>(s_ctr);
    if (__syncthreads_or(other_value) == 0) {
      const int top = 64 - __builtin_clzll(static_cast<unsigned long long>(static_cast<KeyT>(low ^ high)));
      split_order_passes<CODEC, BLOCK, ITEMS>(s_keys, s_num, c, s_wave, m, top - 1, top);  // two values: they differ in this bit
    } else {
      uint64_t all_vary = 0;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        all_vary |= s_red[w];
      }
      split_order<CODEC, BLOCK, ITEMS>(s_keys, s_num, c, s_wave, m, all_vary, few);
    }
    // as the walk leaves it: where each key of this thread belongs
    uint32_t number[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      number[i] = s_num[holds(i) ? slot_of(i) : 0u];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        s_num[number[i]] = static_cast<uint16_t>(slot_of(i));
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const uint32_t o = holds(i) ? slot_of(i) : 0u;
      to[i]            = s_num[o];
      key[i]           = s_keys[o];
    }
  }
  // ---- out, through LDS, so that neighbouring lanes store neighbouring elements ----
  if (PICK || keys_out != nullptr) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (holds(i)) {
        s_keys[to[i]] = key[i];
      }
    }
    __syncthreads();
    for (uint32_t o = tid; o < m; o += BLOCK) {
      put_key(o, s_keys[o]);
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
      put_pos(o, s_pos[o]);
    }
  }
}

}  // namespace cpn
