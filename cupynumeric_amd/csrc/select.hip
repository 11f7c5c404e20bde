// Quantiles of one long unsorted vector: the few elements of the sorted order that the quantiles need
// are selected, without sorting the rest.
//
// Takes the place of sort + take in _quantile_impl (cupynumeric/_module/stats_order.py:249-337) when
// the axis is one long vector.  The elements are those that stand at the requested positions of
// this library's stable sort, bit for bit.
//
// Radix selection from the top: each round counts, for the keys that agree with a target in the bits
// resolved so far, the next 9 ... 12 bits of their ordered images, and the workgroup that finishes last
// finds every target's bin.  The first round also learns which bits vary at all and later rounds
// start below the others (ids held in 64 bits).  Once no more than a quarter of the keys can still be
// asked for, a round copies them out as it counts them and the following rounds read the copy.
//
// Bound by reading the vector: three times for normal or uniform floats (the sign, exponent and first
// mantissa bits take two rounds, the third makes the copy); the later rounds are launches.
// Five percentiles of 10^7 normal float64 values: rounds of 35, 34 and 46 us (the copy), then 6 to 16 us
// each, 152 us per call where the sort took 552; one read of the 80 MB at the rate of a large copy is 15 us.
// 2^26 float64: 484 us against 2556 (one read: 103 us).
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lerp.h"
#include "select_plan.h"
#include "sort_driver.h"

namespace cpn {

constexpr int SELECT_BLOCK      = 1024;
constexpr int SELECT_WAVES      = SELECT_BLOCK / WAVE;
constexpr int SELECT_COPIES     = SELECT_BINS >> SELECT_FIRST_BITS;  // first round: copies of every counter, by lane
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
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    plan->key_or    = 0;
    plan->key_and   = ~0ull;
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
  __shared__ __align__(16) KeyT s_stage[FIRST ? 1 : SELECT_BLOCK * VEC];
  __shared__ uint64_t s_or[SELECT_WAVES], s_and[SELECT_WAVES];
  __shared__ uint64_t s_prefix[SELECT_MAX_RANKS];
  __shared__ uint32_t s_count[SELECT_MAX_RANKS];
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
  const uint32_t bins      = FIRST ? static_cast<uint32_t>(SELECT_BINS) : (n_prefix << w);
  for (uint32_t j = tid; j < bins; j += SELECT_BLOCK) {
    s_hist[j] = 0;
  }
  if (tid < static_cast<int>(n_prefix)) {
    s_prefix[tid] = plan->prefix[tid];
  }
  if (tid == 0) {
    s_staged = 0;
  }
  __syncthreads();

  uint64_t k_or = 0, k_and = ~0ull;
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
        k_or |= image[j];
        k_and &= image[j];
        atomicAdd(&s_hist[(static_cast<uint32_t>(image[j] >> shift) & mask) * SELECT_COPIES + (tid % SELECT_COPIES)], 1u);
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
          atomicAdd(&s_hist[(which[j] << w) + (static_cast<uint32_t>(image[j] >> shift) & mask)], 1u);
          hits |= 1u << j;
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
    for (uint32_t v0 = first; v0 < nvec; v0 += step) {  // uniform per workgroup
      const uint32_t v = v0 + tid;
      KeyT k[VEC] = {};
      uint32_t hits = 0;
      if (v < nvec) {
        const uint4 q = vp[v];
        __builtin_memcpy(k, &q, 16);
        hits = count(k);
      }
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        stage(k[j], ((hits >> j) & 1u) != 0);
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
    k_or  = wave_reduce_or_dpp(k_or);
    k_and = wave_reduce_and_dpp(k_and);
    if (lane == 0) {
      s_or[tid / WAVE]  = k_or;
      s_and[tid / WAVE] = k_and;
    }
  }
  __syncthreads();
  if constexpr (FIRST) {
    if (tid == 0) {
      for (int i = 1; i < SELECT_WAVES; ++i) {
        k_or |= s_or[i];
        k_and &= s_and[i];
      }
      __hip_atomic_fetch_or(&plan->key_or, k_or, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_and(&plan->key_and, k_and, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  uint32_t* out = hist + static_cast<uint32_t>(round) * SELECT_BINS;
  for (uint32_t j = tid; j < (n_prefix << w); j += SELECT_BLOCK) {
    uint32_t c = 0;
    if constexpr (FIRST) {
#pragma unroll
      for (int i = 0; i < SELECT_COPIES; ++i) {
        c += s_hist[j * SELECT_COPIES + i];
      }
    } else {
      c = s_hist[j];
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
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const uint32_t j = i * SELECT_BLOCK + tid;
      c[i]             = j < (n_prefix << w) ? agent_load(&out[j]) : 0u;
    }
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      s_hist[i * SELECT_BLOCK + tid] = c[i];
    }
  }
  __syncthreads();
  __shared__ uint64_t s_new[SELECT_MAX_RANKS];
  for (uint32_t t = tid / WAVE; t < n_ranks; t += SELECT_WAVES) {
    const uint32_t which = plan->which[t];
    const uint32_t rank  = plan->rank[t];
    uint32_t run         = 0;
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
  if (tid == 0) {
    uint64_t common = 0, varying = 0;
    if constexpr (FIRST) {
      common  = agent_load(&plan->key_and);
      varying = common ^ agent_load(&plan->key_or);
    }
    select_advance(plan, s_new, s_count, n_ranks, shift, FIRST, common, varying, copy_now ? agent_load(&plan->copied) : 0u, copy_cap);
    if (plan->done != 0) {
      uint32_t ties = 0;
      for (uint32_t t = 0; t < n_ranks; ++t) {
        if constexpr (CODEC == CODEC_FLOAT) {
          ties |= static_cast<KeyT>(s_new[t]) == static_cast<KeyT>(~static_cast<KeyT>(0)) ? 1u : 0u;
          ties |= static_cast<KeyT>(s_new[t]) == FloatLayout<KeyT>::sign ? 2u : 0u;
        }
      }
      plan->ties = ties;
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
