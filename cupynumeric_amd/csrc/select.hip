// Quantiles of one long unsorted vector: the few elements of the sorted order that the quantiles need
// are selected, without sorting the rest.
//
// Takes the place of sort + take in _quantile_impl (cupynumeric/_module/stats_order.py:249-337) when
// the axis is one long vector.  The elements are those that stand at the requested positions of
// this library's stable sort, bit for bit.
//
// Radix selection from the top: each round counts, for the keys that agree with a target in the bits
// resolved so far, the next 9 ... 12 bits of their ordered images, and the workgroup that finishes last
// finds every target's bin.  A round also learns in which lower bits the keys of every prefix agree: these
// take no round of their own (ids held in 64 bits, whole numbers held as floats).  Once no more than a
// quarter of the keys can still be asked for, a round copies them out as it counts them and the
// following rounds read the copy.
//
// Normal or uniform floats are read three times: the sign, exponent and first mantissa bits take two rounds, the
// third makes the copy; the later rounds are launches.  Five percentiles of 10^7 normal float64: rounds of 27, 35 and
// 36 us, bound by the counting (a read of the 80 MB takes 13 at the rate of a large copy), then 14, 10, 5 and 5, and four
// launches of 2 to 5.  Us per call against sort and take:
//   float64, normal   10^7 elements 127 / 551   2^26 432 / 2560   2^28 1500 / 9370
//   float64, 0 and 1  10^7 elements  81 / 285   2^26 336 /  771   2^28 1144 / 2538
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lerp.h"
#include "select_plan.h"
#include "sort_driver.h"

namespace cpn {

constexpr int SELECT_BLOCK      = 1024;
constexpr int SELECT_WAVES      = SELECT_BLOCK / WAVE;
constexpr int SELECT_STAGED     = 4;      // 16-byte loads per thread that the copy stages at a time
constexpr uint32_t SELECT_FIRST_SPREAD = 2;
static_assert((1 << (SELECT_FIRST_BITS + SELECT_FIRST_SPREAD)) == SELECT_BINS, "copies of the first round's counters");
constexpr uint32_t SELECT_SPREAD_MIN = 1u << 20;  // keys from which a round spreads its counters
constexpr int SELECT_CHUNKS     = 1024;   // select_count_class_kernel

struct SelectRanks {
  uint32_t rank[SELECT_MAX_RANKS];  // ascending, all different
  uint32_t n;
};
struct SelectQuantiles {
  uint32_t left[SELECT_MAX_Q], right[SELECT_MAX_Q];  // targets
  double gamma[SELECT_MAX_Q];
  uint32_t n;
};

template <typename T>
__device__ __forceinline__ T agent_load(const T* p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

static __global__ __launch_bounds__(256) void select_init_kernel(SelectPlan* plan, uint4* hist, uint32_t n_vec, uint32_t n,
                                                                 uint32_t bits, SelectRanks ranks)
{
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n_vec; i += gridDim.x * 256) {
    hist[i] = make_uint4(0u, 0u, 0u, 0u);
  }
  if (blockIdx.x == 0 && threadIdx.x < SELECT_MAX_RANKS) {
    plan->rank[threadIdx.x]  = ranks.rank[threadIdx.x];
    plan->which[threadIdx.x] = 0;
    plan->any[threadIdx.x]   = 0;
    plan->all[threadIdx.x]   = ~0ull;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    plan->prefix[0] = 0;
    plan->n_prefix  = 1;
    plan->bits_left = bits;
    plan->list_len  = n;
    plan->from_copy = plan->copy_now = plan->copied = plan->done = plan->ties = 0;
    for (int r = 0; r <= SELECT_MAX_ROUNDS; ++r) {
      plan->blocks_done[r] = 0;
    }
  }
}

// OR and AND of a set of images.
struct alignas(16) Agreement {
  uint64_t any, all;
};
static_assert(SELECT_WAVES <= SELECT_MAX_RANKS, "first round: one entry per wavefront");

// Is this the last workgroup of the launch to get here?  What the others have written with agent-scope
// atomics is then seen by agent-scope loads: every wavefront waits until its own are done.  (A fence
// instead writes the L2 back, from every wavefront of the grid: 140 us per round of 512 workgroups.)
__device__ __forceinline__ bool last_workgroup(uint32_t* counter, uint32_t* s_flag)
{
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *s_flag               = (before + 1 == gridDim.x) ? 1u : 0u;
  }
  __syncthreads();
  return *s_flag != 0;
}

// One round; 16-byte loads over the aligned middle of the list, the ends by the first workgroup.
template <typename KeyT, int CODEC, bool FIRST>
__global__ __launch_bounds__(SELECT_BLOCK) void select_round_kernel(const KeyT* __restrict__ values, KeyT* copy, uint32_t copy_cap,
                                                                    SelectPlan* plan, uint32_t* hist, uint32_t n_ranks, int round)
{
  constexpr int VEC = 16 / sizeof(KeyT);
  __shared__ uint32_t s_hist[SELECT_BINS];
  __shared__ __align__(16) KeyT s_stage[FIRST ? 1 : SELECT_STAGED * SELECT_BLOCK * VEC];
  __shared__ Agreement s_agree[SELECT_MAX_RANKS];  // per prefix; first round: per wavefront
  __shared__ uint64_t s_prefix[SELECT_MAX_RANKS];
  __shared__ uint32_t s_count[SELECT_MAX_RANKS], s_which[SELECT_MAX_RANKS], s_rank[SELECT_MAX_RANKS];
  __shared__ uint32_t s_staged, s_base, s_flag;

  if (plan->done != 0) {  // (written by earlier launches only: uniform)
    return;
  }
  const int tid            = threadIdx.x;
  const int lane           = tid & (WAVE - 1);
  const uint32_t n_prefix  = FIRST ? 1u : plan->n_prefix;
  const uint32_t bits_left = plan->bits_left;
  const uint32_t want      = FIRST ? static_cast<uint32_t>(SELECT_FIRST_BITS) : select_bits(n_prefix);
  const uint32_t w         = want < bits_left ? want : bits_left;
  const uint32_t shift     = bits_left - w;
  const uint32_t mask      = (1u << w) - 1u;
  const bool copy_now      = !FIRST && plan->copy_now != 0;
  const bool from_copy     = !FIRST && plan->from_copy != 0;
  const KeyT* list         = from_copy ? copy : values;
  const uint32_t len       = plan->list_len;
  // Copies of every counter, by lane: with few prefixes most keys may be of one value, and the lanes of a wave
  // that add to one counter wait for each other.  Median of 2^28 int64 of five values: 3.1 ms without, 2.7 with
  // copies; a short list is done before the copies are added up.
  uint32_t spread = FIRST ? SELECT_FIRST_SPREAD : 0u;  // logarithm of their number
  if (!FIRST && !from_copy && len >= SELECT_SPREAD_MIN) {
    while ((n_prefix << (w + spread + 1)) <= static_cast<uint32_t>(SELECT_BINS) && spread < SELECT_FIRST_SPREAD) {
      ++spread;
    }
  }
  const uint32_t own  = static_cast<uint32_t>(tid) & ((1u << spread) - 1u);
  const uint32_t bins = n_prefix << (w + spread);
  for (uint32_t j = tid; j < bins; j += SELECT_BLOCK) {
    s_hist[j] = 0;
  }
  if (tid < static_cast<int>(n_prefix)) {
    s_prefix[tid] = plan->prefix[tid];
    s_agree[tid]  = Agreement{0, ~0ull};
  }
  if (tid < static_cast<int>(n_ranks)) {
    s_which[tid] = plan->which[tid];
    s_rank[tid]  = plan->rank[tid];
  }
  if (tid == 0) {
    s_staged = 0;
  }
  __syncthreads();

  Agreement mine = {0, ~0ull};  // first round
  // counts the keys of an array; bit j of the result: key j can still be a target
  auto count = [&](const auto& k) -> uint32_t {
    constexpr int N = sizeof(k) / sizeof(KeyT);
    uint64_t image[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      image[j] = static_cast<uint64_t>(ordered_bits<CODEC, KeyT>(k[j]));
    }
    if constexpr (FIRST) {
#pragma unroll
      for (int j = 0; j < N; ++j) {
        mine.any |= image[j];
        mine.all &= image[j];
        atomicAdd(&s_hist[((static_cast<uint32_t>(image[j] >> shift) & mask) << spread) + own], 1u);
      }
      return ~0u;
    } else {
      uint32_t which[N];
      uint32_t hits = 0;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        which[j] = ~0u;
      }
      for (uint32_t t = 0; t < n_prefix; ++t) {
        const uint64_t p = s_prefix[t];
#pragma unroll
        for (int j = 0; j < N; ++j) {  // (bits_left < 64 after the first round)
          which[j] = (image[j] >> bits_left) == p ? t : which[j];
        }
      }
#pragma unroll
      for (int j = 0; j < N; ++j) {
        if (which[j] != ~0u) {
          atomicAdd(&s_hist[(((which[j] << w) + (static_cast<uint32_t>(image[j] >> shift) & mask)) << spread) + own], 1u);
          hits |= 1u << j;
          // Does the key add to its prefix's agreement?  After the first few keys hardly ever.  (An entry read while
          // another lane updates it has fewer bits set, or cleared: that costs an update, no bit is lost.)
          if (shift != 0) {
            const Agreement known = s_agree[which[j]];
            if (((image[j] & ~known.any) | (known.all & ~image[j])) != 0) {
              __hip_atomic_fetch_or(&s_agree[which[j]].any, image[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
              __hip_atomic_fetch_and(&s_agree[which[j]].all, image[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
          }
        }
      }
      return hits;
    }
  };
  // the keys of one iteration that go to the copy: staged, then stored side by side.  copy_cap is at least
  // the number of keys that match (the plan compares) unless the caller writes to the input meanwhile: keys
  // without room are dropped, and the next round reads no more than copy_cap (select_advance).
  auto flush = [&]() {
    __syncthreads();
    const uint32_t staged = s_staged;
    if (tid == 0 && staged != 0) {
      s_base = __hip_atomic_fetch_add(&plan->copied, staged, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (staged != 0) {
      const uint32_t base = s_base;
      for (uint32_t j = tid; j < staged; j += SELECT_BLOCK) {
        if (base + j < copy_cap) {
          copy[base + j] = s_stage[j];
        }
      }
    }
    __syncthreads();
    if (tid == 0) {
      s_staged = 0;
    }
    __syncthreads();
  };
  auto stage = [&](KeyT raw, bool keep) {  // called by all lanes of a wave
    const uint64_t bal = __builtin_amdgcn_ballot_w64(keep);
    if (bal != 0) {
      uint32_t at = 0;
      if (lane == 0) {
        at = atomicAdd(&s_staged, static_cast<uint32_t>(__builtin_popcountll(bal)));
      }
      at = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(at))) + lanes_below(bal);
      if (keep) {
        s_stage[at] = raw;
      }
    }
  };

  uint32_t head = static_cast<uint32_t>(((16u - (reinterpret_cast<uintptr_t>(list) & 15u)) & 15u) / sizeof(KeyT));
  if (head > len) {
    head = len;
  }
  const uint32_t nvec  = (len - head) / VEC;
  const uint32_t tail  = head + nvec * VEC;  // the elements from here on: fewer than VEC
  const uint4* vp      = reinterpret_cast<const uint4*>(list + head);
  const uint32_t step  = gridDim.x * SELECT_BLOCK;
  const uint32_t first = blockIdx.x * SELECT_BLOCK;
  if (blockIdx.x == 0) {
    const uint32_t ends = head + (len - tail);  // < 2 * VEC <= SELECT_BLOCK
    const bool mine     = static_cast<uint32_t>(tid) < ends;
    KeyT k[1]           = {};
    bool keep           = false;
    if (mine) {
      k[0] = list[static_cast<uint32_t>(tid) < head ? tid : tail + (tid - head)];
      keep = count(k) != 0;
    }
    if (copy_now) {
      stage(k[0], keep);
      flush();
    }
  }
  if (!FIRST && copy_now) {
    // four loads in flight and one flush for them, of four barriers and a global atomic: the median of 2^28 int64 of
    // five values 2.7 -> 1.5 ms against a flush per load, five percentiles of 10^7 normal float64 142 -> 132 us
    for (uint64_t v0 = first; v0 < nvec; v0 += static_cast<uint64_t>(SELECT_STAGED) * step) {  // uniform per workgroup
      uint4 q[SELECT_STAGED];
#pragma unroll
      for (int i = 0; i < SELECT_STAGED; ++i) {
        const uint64_t v = v0 + static_cast<uint64_t>(i) * step + tid;
        q[i]             = vp[v < nvec ? v : nvec - 1];
      }
#pragma unroll
      for (int i = 0; i < SELECT_STAGED; ++i) {
        const uint64_t v = v0 + static_cast<uint64_t>(i) * step + tid;
        KeyT k[VEC];
        __builtin_memcpy(k, &q[i], 16);
        const uint32_t hits = v < nvec ? count(k) : 0u;
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          stage(k[j], ((hits >> j) & 1u) != 0);
        }
      }
      flush();
    }
  } else {
    uint64_t v = first + tid;
    for (; v + 3ull * step < nvec; v += 4ull * step) {  // four loads in flight
      uint4 q[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        q[i] = vp[v + static_cast<uint64_t>(i) * step];
      }
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        KeyT k[2 * VEC];
        __builtin_memcpy(k, &q[i], 16);
        __builtin_memcpy(k + VEC, &q[i + 1], 16);
        count(k);
      }
    }
    for (; v < nvec; v += step) {
      KeyT k[VEC];
      const uint4 q = vp[v];
      __builtin_memcpy(k, &q, 16);
      count(k);
    }
  }
  if constexpr (FIRST) {
    mine.any = wave_reduce_or_dpp(mine.any);
    mine.all = wave_reduce_and_dpp(mine.all);
    __syncthreads();  // (entry 0 was set at the start)
    if (lane == 0) {
      s_agree[tid / WAVE] = mine;
    }
  }
  __syncthreads();
  if constexpr (FIRST) {
    if (tid == 0) {
      for (int i = 1; i < SELECT_WAVES; ++i) {
        mine.any |= s_agree[i].any;
        mine.all &= s_agree[i].all;
      }
    }
  } else if (tid < static_cast<int>(n_prefix)) {
    mine = s_agree[tid];
  }
  if (tid < static_cast<int>(n_prefix) && (mine.any | ~mine.all) != 0) {  // (a prefix none of whose keys are here adds nothing)
    __hip_atomic_fetch_or(&plan->any[tid], mine.any, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_fetch_and(&plan->all[tid], mine.all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  uint32_t* out = hist + static_cast<uint32_t>(round) * SELECT_BINS;
  for (uint32_t j = tid; j < (n_prefix << w); j += SELECT_BLOCK) {
    uint32_t c = 0;
    for (uint32_t i = 0; i < (1u << spread); ++i) {
      c += s_hist[(j << spread) + i];
    }
    if (c != 0) {
      __hip_atomic_fetch_add(&out[j], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (!last_workgroup(&plan->blocks_done[round], &s_flag)) {
    return;
  }

  // ---- the last workgroup: the counts into LDS, all loads in flight at once (one after the other they cost
  //      a memory round trip each), then every target's bin, one wavefront per target ----
  {
    constexpr int EACH = SELECT_BINS / SELECT_BLOCK;
    uint32_t c[EACH];
    if (tid < static_cast<int>(n_prefix)) {
      mine.any = agent_load(&plan->any[tid]);
      mine.all = agent_load(&plan->all[tid]);
    }
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const uint32_t j = i * SELECT_BLOCK + tid;
      c[i]             = j < (n_prefix << w) ? agent_load(&out[j]) : 0u;
    }
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      s_hist[i * SELECT_BLOCK + tid] = c[i];
    }
    if (tid < static_cast<int>(n_prefix)) {
      s_agree[tid]   = mine;
      plan->any[tid] = 0;  // for the next round
      plan->all[tid] = ~0ull;
    }
  }
  __syncthreads();
  __shared__ uint64_t s_new[SELECT_MAX_RANKS];
  for (uint32_t t = tid / WAVE; t < n_ranks; t += SELECT_WAVES) {
    const uint32_t which = s_which[t];
    const uint32_t rank  = s_rank[t];
    uint32_t run         = 0;
    if (which == SELECT_FINISHED) {  // uniform for the wavefront
      continue;
    }
    if (lane == 0) {  // (no key at this rank: only if the caller has written to the input during the call)
      s_new[t]   = 0;
      s_count[t] = 0;
    }
    for (uint32_t b0 = 0; b0 <= mask; b0 += WAVE) {  // uniform for the wavefront
      const uint32_t b    = b0 + lane;
      const uint32_t c    = b <= mask ? s_hist[(which << w) + b] : 0u;
      const uint32_t incl = run + wave_inclusive_sum_dpp(c);
      if (incl - c <= rank && rank < incl) {  // one lane of one step: the ranks of a prefix are below its count
        s_new[t]      = (s_prefix[which] << w) | b;
        s_count[t]    = c;
        plan->rank[t] = rank - (incl - c);
      }
      run = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), WAVE - 1));
      if (rank < run) {
        break;
      }
    }
  }
  __syncthreads();
  if (tid >= WAVE) {
    return;
  }
  // The plan of the next round by one wavefront, a lane per target (ascending: equal prefixes are neighbours).
  const uint32_t copied = copy_now ? agent_load(&plan->copied) : 0u;
  const bool target     = lane < static_cast<int>(n_ranks);
  const uint32_t before = target ? s_which[lane] : SELECT_FINISHED;
  const bool active     = before != SELECT_FINISHED;
  const SelectChild c   = active ? select_child(s_new[lane], shift, s_agree[before].any, s_agree[before].all) : SelectChild{0, 0};
  const uint32_t left   = select_bits_left(wave_reduce_or_dpp(c.varying));
  const bool goes_on    = active && c.varying != 0;
  const uint64_t prefix = c.image >> left;
  const uint64_t going  = __builtin_amdgcn_ballot_w64(goes_on);
  const uint64_t lower  = going & ((1ull << lane) - 1);  // the active target before this one
  const int neighbour   = lower != 0 ? 63 - __builtin_clzll(lower) : lane;
  const uint64_t theirs = __shfl(prefix, neighbour, WAVE);
  const bool opens      = goes_on && (lower == 0 || theirs != prefix);
  const uint64_t heads  = __builtin_amdgcn_ballot_w64(opens);
  const uint32_t which  = lanes_below(heads) + (opens ? 1u : 0u) - 1u;
  const uint32_t total  = wave_inclusive_sum_dpp(opens ? s_count[lane] : 0u);  // below 2^31: keys of different prefixes
  if (active) {
    plan->which[lane] = goes_on ? which : SELECT_FINISHED;
    if (!goes_on) {
      plan->image[lane] = c.image;
    }
  }
  if (opens) {
    plan->prefix[which] = prefix;
  }
  const uint32_t all_keys = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(total), WAVE - 1));
  if (lane == 0) {
    select_next_list(plan, copy_now, from_copy, static_cast<uint32_t>(__builtin_popcountll(heads)), left, all_keys, copied, copy_cap);
  }
  if constexpr (CODEC == CODEC_FLOAT) {
    // targets whose image keys of other bits share, now or in an earlier round
    const KeyT image = static_cast<KeyT>(active ? c.image : (target ? plan->image[lane] : 0));
    const bool whole = target && !goes_on;
    const uint64_t nans  = __builtin_amdgcn_ballot_w64(whole && image == static_cast<KeyT>(~static_cast<KeyT>(0)));
    const uint64_t zeros = __builtin_amdgcn_ballot_w64(whole && image == FloatLayout<KeyT>::sign);
    if (lane == 0) {
      plan->ties = (nans != 0 ? 1u : 0u) | (zeros != 0 ? 2u : 0u);
    }
  }
}

// ---- float targets among the NaNs or the zeros: keys of other bits share their image, and the sort keeps
// ---- them in the order of the input.  Which chunk of the input holds the one that is wanted?
template <typename KeyT>
__global__ __launch_bounds__(256) void select_count_class_kernel(const KeyT* __restrict__ values, uint32_t n, uint32_t chunk,
                                                                 SelectPlan* plan, uint32_t* counts, uint32_t n_ranks)
{
  __shared__ uint32_t s_wave[2][256 / WAVE];
  __shared__ uint32_t s_flag;
  if (plan->ties == 0) {
    return;
  }
  constexpr KeyT NAN_KEY = static_cast<KeyT>(~static_cast<KeyT>(0));
  const int tid          = threadIdx.x;
  const uint64_t begin   = static_cast<uint64_t>(blockIdx.x) * chunk;
  const uint64_t end     = begin + chunk < n ? begin + chunk : n;
  uint32_t nans = 0, zeros = 0;
#pragma unroll 8
  for (uint64_t i = begin + tid; i < end; i += 256) {
    const KeyT image = ordered_bits<CODEC_FLOAT, KeyT>(values[i]);
    nans += image == NAN_KEY ? 1u : 0u;
    zeros += image == FloatLayout<KeyT>::sign ? 1u : 0u;
  }
  nans  = wave_inclusive_sum_dpp(nans);
  zeros = wave_inclusive_sum_dpp(zeros);
  if ((tid & (WAVE - 1)) == WAVE - 1) {
    s_wave[0][tid / WAVE] = nans;
    s_wave[1][tid / WAVE] = zeros;
  }
  __syncthreads();
  if (tid < 2) {
    uint32_t c = 0;
    for (int i = 0; i < 256 / WAVE; ++i) {
      c += s_wave[tid][i];
    }
    __hip_atomic_store(&counts[tid * SELECT_CHUNKS + blockIdx.x], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (!last_workgroup(&plan->blocks_done[SELECT_MAX_ROUNDS], &s_flag)) {
    return;
  }
  constexpr uint32_t EACH = SELECT_CHUNKS / WAVE;
  const uint32_t lane     = tid & (WAVE - 1);
  for (uint32_t t = tid / WAVE; t < n_ranks; t += 256 / WAVE) {
    const KeyT image    = static_cast<KeyT>(plan->image[t]);
    const uint32_t rank = plan->rank[t];
    if (image != NAN_KEY && image != FloatLayout<KeyT>::sign) {
      continue;
    }
    const uint32_t* c = counts + (image == NAN_KEY ? 0 : SELECT_CHUNKS);
    uint32_t here[EACH];
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t i = 0; i < EACH; ++i) {
      here[i] = lane * EACH + i < gridDim.x ? agent_load(&c[lane * EACH + i]) : 0u;
    }
#pragma unroll
    for (uint32_t i = 0; i < EACH; ++i) {
      sum += here[i];
    }
    const uint32_t incl = wave_inclusive_sum_dpp(sum);
    uint32_t run        = incl - sum;
#pragma unroll
    for (uint32_t i = 0; i < EACH; ++i) {
      if (run <= rank && rank < run + here[i]) {  // one lane, one step
        plan->chunk[t] = lane * EACH + i;
        plan->rank[t]  = rank - run;
      }
      run += here[i];
    }
  }
}

// One workgroup per target: its element into selected[t].
template <typename KeyT, int CODEC>
__global__ __launch_bounds__(SELECT_BLOCK) void select_fetch_kernel(const KeyT* __restrict__ values, uint32_t n, uint32_t chunk,
                                                                    const SelectPlan* __restrict__ plan, KeyT* __restrict__ selected)
{
  const uint32_t t = blockIdx.x;
  const KeyT image = static_cast<KeyT>(plan->image[t]);
  const int tid    = threadIdx.x;
  if constexpr (CODEC == CODEC_FLOAT) {
    __shared__ uint32_t s_wave[SELECT_WAVES];
    if (image == static_cast<KeyT>(~static_cast<KeyT>(0)) || image == FloatLayout<KeyT>::sign) {
      const uint64_t begin = static_cast<uint64_t>(plan->chunk[t]) * chunk;
      const uint64_t end   = begin + chunk < n ? begin + chunk : n;
      uint32_t rank        = plan->rank[t];
      for (uint64_t i0 = begin; i0 < end; i0 += SELECT_BLOCK) {
        const uint64_t i   = i0 + tid;
        const KeyT raw     = i < end ? values[i] : KeyT{};
        const bool hit     = i < end && ordered_bits<CODEC_FLOAT, KeyT>(raw) == image;
        const uint64_t bal = __builtin_amdgcn_ballot_w64(hit);
        if ((tid & (WAVE - 1)) == 0) {
          s_wave[tid / WAVE] = static_cast<uint32_t>(__builtin_popcountll(bal));
        }
        __syncthreads();
        uint32_t before = 0, total = 0;
#pragma unroll
        for (int j = 0; j < SELECT_WAVES; ++j) {
          before += j < tid / WAVE ? s_wave[j] : 0u;
          total += s_wave[j];
        }
        if (hit && before + lanes_below(bal) == rank) {
          selected[t] = raw;
        }
        if (rank < total) {
          return;  // uniform
        }
        rank -= total;
        __syncthreads();
      }
      return;
    }
    if (tid == 0) {
      selected[t] = sign_unflip<KeyT>(image);
    }
  } else if (tid == 0) {
    selected[t] = CODEC == CODEC_SIGNED ? static_cast<KeyT>(image ^ (static_cast<KeyT>(1) << (sizeof(KeyT) * 8 - 1))) : image;
  }
}

template <typename T, bool INTERPOLATE>
__global__ __launch_bounds__(WAVE) void select_eval_kernel(const T* __restrict__ selected, SelectQuantiles q, void* __restrict__ out)
{
  const uint32_t i = threadIdx.x;
  if (i < q.n) {
    if constexpr (INTERPOLATE) {
      static_cast<double*>(out)[i] = Lerp<T>::eval(selected[q.left[i]], selected[q.right[i]], q.gamma[i]);
    } else {
      static_cast<T*>(out)[i] = selected[q.left[i]];
    }
  }
}

struct SelectLayout {
  uint64_t off_hist, off_counts, off_selected, off_copy, copy_cap, total;
};
static SelectLayout select_layout(int key_bytes, uint64_t n)
{
  SelectLayout L{};
  L.off_hist     = SELECT_PLAN_BYTES;
  L.off_counts   = L.off_hist + SELECT_MAX_ROUNDS * SELECT_BINS * 4ull;
  L.off_selected = L.off_counts + 2ull * SELECT_CHUNKS * 4;
  L.off_copy     = L.off_selected + align_up(SELECT_MAX_RANKS * 8ull, WORKSPACE_ALIGN);
  L.copy_cap     = n / 4;
  L.total        = L.off_copy + align_up(L.copy_cap * key_bytes + 16, WORKSPACE_ALIGN);
  return L;
}

template <typename KeyT, int CODEC, typename T>
static int select_typed(const void* values_v, uint32_t n, const SelectRanks& ranks, const SelectQuantiles& q, int interpolate,
                        void* out, unsigned char* ws, hipStream_t s)
{
  const KeyT* values   = static_cast<const KeyT*>(values_v);
  const SelectLayout L = select_layout(sizeof(KeyT), n);
  SelectPlan* plan     = reinterpret_cast<SelectPlan*>(ws);
  uint32_t* hist       = reinterpret_cast<uint32_t*>(ws + L.off_hist);
  uint32_t* counts     = reinterpret_cast<uint32_t*>(ws + L.off_counts);
  KeyT* selected       = reinterpret_cast<KeyT*>(ws + L.off_selected);
  KeyT* copy           = reinterpret_cast<KeyT*>(ws + L.off_copy);
  const int bits       = static_cast<int>(sizeof(KeyT)) * 8;
  const int rounds     = select_rounds(bits, ranks.n);
  {
    ProfileScope prof("select_init", s);
    const uint32_t n_vec = static_cast<uint32_t>(rounds) * SELECT_BINS / 4;
    hipLaunchKernelGGL(select_init_kernel, dim3((n_vec + 255) / 256), dim3(256), 0, s, plan, reinterpret_cast<uint4*>(hist), n_vec, n,
                       static_cast<uint32_t>(bits), ranks);
  }
  CPN_HIP_TRY(hipGetLastError());
  // the workgroups that fit on the CUs (two each, one with the staging area of the copy), with at least two 16-byte loads per thread
  uint64_t grid      = (static_cast<uint64_t>(n) * sizeof(KeyT) + 32 * SELECT_BLOCK - 1) / (32 * SELECT_BLOCK);
  const uint64_t cus = static_cast<uint64_t>(compute_units());
  grid               = grid < 1 ? 1 : (grid > 2 * cus ? 2 * cus : grid);
  for (int r = 0; r < rounds; ++r) {
    ProfileScope prof("select_round", s);
    if (r == 0) {
      hipLaunchKernelGGL((select_round_kernel<KeyT, CODEC, true>), dim3(static_cast<uint32_t>(grid)), dim3(SELECT_BLOCK), 0, s, values,
                         copy, static_cast<uint32_t>(L.copy_cap), plan, hist, ranks.n, r);
    } else {
      hipLaunchKernelGGL((select_round_kernel<KeyT, CODEC, false>), dim3(static_cast<uint32_t>(grid < cus ? grid : cus)), dim3(SELECT_BLOCK), 0, s, values,
                         copy, static_cast<uint32_t>(L.copy_cap), plan, hist, ranks.n, r);
    }
    CPN_HIP_TRY(hipGetLastError());
  }
  const uint32_t chunk  = (n + SELECT_CHUNKS - 1) / SELECT_CHUNKS;
  const uint32_t chunks = (n + chunk - 1) / chunk;
  if constexpr (CODEC == CODEC_FLOAT) {
    ProfileScope prof("select_count_class", s);
    hipLaunchKernelGGL((select_count_class_kernel<KeyT>), dim3(chunks), dim3(256), 0, s, values, n, chunk, plan, counts, ranks.n);
    CPN_HIP_TRY(hipGetLastError());
  }
  {
    ProfileScope prof("select_fetch", s);
    hipLaunchKernelGGL((select_fetch_kernel<KeyT, CODEC>), dim3(ranks.n), dim3(SELECT_BLOCK), 0, s, values, n, chunk, plan, selected);
  }
  CPN_HIP_TRY(hipGetLastError());
  {
    ProfileScope prof("select_eval", s);
    if (interpolate != 0) {
      hipLaunchKernelGGL((select_eval_kernel<T, true>), dim3(1), dim3(WAVE), 0, s, reinterpret_cast<const T*>(selected), q, out);
    } else {
      hipLaunchKernelGGL((select_eval_kernel<T, false>), dim3(1), dim3(WAVE), 0, s, reinterpret_cast<const T*>(selected), q, out);
    }
  }
  CPN_HIP_TRY(hipGetLastError());
  return CPN_OK;
}

}  // namespace cpn

extern "C" uint64_t cpn_quantile_select_temp_bytes(int dtype, uint64_t n, uint64_t num_q)
{
  const cpn::KeyKind k = cpn::key_kind(dtype);
  if (k.bytes < 4 || k.codec == cpn::CODEC_COMPLEX || n == 0 || n >= (1ull << 31) || num_q == 0 ||
      num_q > static_cast<uint64_t>(cpn::SELECT_MAX_Q)) {
    return 0;
  }
  return cpn::select_layout(k.bytes, n).total;
}

extern "C" int cpn_quantile_select(int dtype, const void* values, uint64_t n, uint64_t num_q, const int64_t* left,
                                   const int64_t* right, const double* gamma, int interpolate, void* out, void* temp,
                                   uint64_t temp_bytes, void* stream)
{
  using namespace cpn;
  const KeyKind k = key_kind(dtype);
  if (k.bytes == 0 || k.codec == CODEC_COMPLEX) {
    return CPN_ERR_DTYPE;
  }
  if (num_q == 0) {
    return CPN_OK;
  }
  if (n == 0) {
    return CPN_ERR_SHAPE;  // no element to take
  }
  const uint64_t need = cpn_quantile_select_temp_bytes(dtype, n, num_q);
  if (need == 0) {
    return CPN_ERR_UNSUPPORTED;
  }
  if (values == nullptr || left == nullptr || out == nullptr || (interpolate != 0 && (right == nullptr || gamma == nullptr))) {
    return CPN_ERR_NULL;
  }
  if (temp == nullptr || temp_bytes < need || (reinterpret_cast<uintptr_t>(temp) % WORKSPACE_ALIGN) != 0) {
    return CPN_ERR_TEMP;
  }
  const uintptr_t out_mask = interpolate != 0 ? 7u : static_cast<uintptr_t>(k.bytes - 1);
  if ((reinterpret_cast<uintptr_t>(values) & static_cast<uintptr_t>(k.bytes - 1)) != 0 ||
      (reinterpret_cast<uintptr_t>(out) & out_mask) != 0) {
    return CPN_ERR_ALIGN;
  }
  // the different positions, ascending
  SelectRanks ranks{};
  SelectQuantiles q{};
  uint32_t pos[SELECT_MAX_RANKS];
  uint32_t m = 0;
  for (uint64_t i = 0; i < num_q; ++i) {
    for (int side = 0; side < (interpolate != 0 ? 2 : 1); ++side) {
      const int64_t p = side == 0 ? left[i] : right[i];
      if (p < 0 || static_cast<uint64_t>(p) >= n) {
        return CPN_ERR_SHAPE;
      }
      uint32_t at = 0;
      while (at < m && pos[at] < static_cast<uint32_t>(p)) {
        ++at;
      }
      if (at == m || pos[at] != static_cast<uint32_t>(p)) {
        for (uint32_t j = m; j > at; --j) {
          pos[j] = pos[j - 1];
        }
        pos[at] = static_cast<uint32_t>(p);
        ++m;
      }
    }
  }
  auto target_of = [&](int64_t p) {
    uint32_t at = 0;
    while (pos[at] != static_cast<uint32_t>(p)) {
      ++at;
    }
    return at;
  };
  ranks.n = m;
  for (uint32_t j = 0; j < m; ++j) {
    ranks.rank[j] = pos[j];
  }
  q.n = static_cast<uint32_t>(num_q);
  for (uint64_t i = 0; i < num_q; ++i) {
    q.left[i]  = target_of(left[i]);
    q.right[i] = interpolate != 0 ? target_of(right[i]) : q.left[i];
    q.gamma[i] = interpolate != 0 ? gamma[i] : 0.0;
  }
  unsigned char* ws = static_cast<unsigned char*>(temp);
  hipStream_t s     = static_cast<hipStream_t>(stream);
  const uint32_t n32 = static_cast<uint32_t>(n);
  switch (dtype) {
    case CPN_INT32: return select_typed<uint32_t, CODEC_SIGNED, int32_t>(values, n32, ranks, q, interpolate, out, ws, s);
    case CPN_INT64: return select_typed<uint64_t, CODEC_SIGNED, int64_t>(values, n32, ranks, q, interpolate, out, ws, s);
    case CPN_UINT32: return select_typed<uint32_t, CODEC_UNSIGNED, uint32_t>(values, n32, ranks, q, interpolate, out, ws, s);
    case CPN_UINT64: return select_typed<uint64_t, CODEC_UNSIGNED, uint64_t>(values, n32, ranks, q, interpolate, out, ws, s);
    case CPN_FLOAT32: return select_typed<uint32_t, CODEC_FLOAT, float>(values, n32, ranks, q, interpolate, out, ws, s);
    case CPN_FLOAT64: return select_typed<uint64_t, CODEC_FLOAT, double>(values, n32, ranks, q, interpolate, out, ws, s);
    default: return CPN_ERR_UNSUPPORTED;
  }
}
