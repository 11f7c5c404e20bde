// The distinct values of a long integer array that has few of them for its length, in no order: what `unique` sorts
// instead of the array.
//
// Stands where UniqueTask's GPU variant sorts the whole array and drops the repetitions afterwards
// (src/cupynumeric/set/unique.cu:137-204).  A sample of 8192 keys says how many values to expect (one workgroup, hashed in
// LDS: the values seen once and twice give Chao's estimate of those not seen), and with it the way, on the device:
//   few   up to 3000 values: every workgroup reads a share of the array into a hash table in LDS that starts with the
//         sample's values, and enters those that are new into one in memory.  Bound by the read.
//   many  up to 2^21 values (of 8-byte keys 2^20), a quarter of the keys at most: every workgroup puts a tile of the array in the
//         order of 256 classes of a hash of the key (split_sort.h does so with the keys' order: the tile stays together, a table
//         says where each class starts), then a workgroup per class reads its part of every tile into a hash table in LDS.
//         Values that the sample has at least eight times are known by then and leave the array with the first step, so that
//         a frequent value does not fill a class.  The first step is bound by its two passes over memory (85 us for 2^26
//         int32), the second by the vector and LDS instructions of the look-ups (146 us, 41 of them the reads of LDS alone; 151
//         before the next eight tiles were asked for first).
//   none  the caller sorts (cpn_unique).
// A table that fills up, where the estimate was wrong (values of very unlike frequency: Chao's is a lower bound), ends the
// attempt the same way.
//
// us per call of `unique`, sorted / this way: 2^26 int32 of 16 values 868 / 119, of 2^20 923 / 330, of 2^26 1016 / 1036; 2^25 int64
// of 1000 values 834 / 120, of 2^18 849 / 290, of 2^25 935 / 963.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sort_driver.h"
#include "split_sort.h"

namespace cpn {

constexpr int COLLECT_SAMPLES     = 8192;
constexpr int COLLECT_BLOCK       = 1024;
constexpr int COLLECT_WAVES       = COLLECT_BLOCK / WAVE;
constexpr int COLLECT_SLOTS       = 16384;  // of the sample's table, and of the one in memory
constexpr int collect_class_slots(int key_bytes) { return key_bytes == 4 ? 32768 : 16384; }  // (128 KiB)
constexpr int COLLECT_FEW_SLOTS   = 8192;   // of a workgroup's table of few values
constexpr int COLLECT_HEAVY_SLOTS = 2048;
constexpr int COLLECT_HEAVY       = 8;      // times in the sample
constexpr int COLLECT_HEAVY_MAX   = COLLECT_SAMPLES / COLLECT_HEAVY;
constexpr int COLLECT_KNOWN_MAX   = 3072;   // few: values of the sample; many: heavy ones
constexpr int COLLECT_CLASSES     = 256;
constexpr int COLLECT_ITEMS       = 14;     // a class has 56 keys of a tile, one load of a wave, in the mean
constexpr int COLLECT_TILE        = COLLECT_BLOCK * COLLECT_ITEMS;
// A table is closed with a quarter of it free.  (A wave looks before every step, of one key per lane: all waves of a
// workgroup together are at most 1024 keys past the line.)
constexpr uint32_t collect_class_full(int key_bytes) { return collect_class_slots(key_bytes) / 4 * 3; }
constexpr uint32_t COLLECT_FEW_FULL = 6144;
static_assert(collect_class_full(8) + COLLECT_BLOCK < collect_class_slots(8) && COLLECT_FEW_FULL + COLLECT_BLOCK < COLLECT_FEW_SLOTS, "never full");
// In the table in memory, a fifth full if the estimate is right.  (Every one is a round trip: in a full table, of 2^23 int32 keys with 20 000
// different values whose frequencies fall as the power of 1.7 of their rank, `unique` took 890 us with 512 for each value of each
// workgroup; 480 with 128 until one of a wave has found no place; 250 sorted.)
constexpr int COLLECT_FEW_PROBES = 128;
constexpr double COLLECT_FEW_MAX  = 3000.0;
constexpr double collect_many_max(int key_bytes) { return 64.0 * collect_class_slots(key_bytes); }  // a quarter of the tables
// Few values of like frequencies, up to 3000, are seen twice more often than once, and so are 2500 whose frequencies fall as the 7/8th power
// of their rank by a third as often; of those that fall as its power of 1.7, without end, the sample sees a fifth as many twice.  Of these
// the sample foretells 9000 to 35 000 for 2^23 keys, of which 20 000 are there, and nine in ten samples of them more than the table has places;
// of the power of 2 one in twenty for 2^25 keys, where the table still does.  us per call of `unique` tried / not, 2^25 int64 of the power of
// 1.5 3300 / 860, of 1.7 1160 / 850, of 2 214 / 860.
constexpr double COLLECT_FEW_ONCE   = 3.6;
constexpr double COLLECT_FEW_GROWTH = COLLECT_SLOTS;
constexpr double collect_tail_max(int key_bytes) { return 0.9 * COLLECT_CLASSES * collect_class_full(key_bytes); }
// An array that turns out to be sorted after all has waited for the sample, 28 us.  (Less than one copy for count and status in place of
// two, and shorter scans, save: 2^22 int64 of as many values 226 before both, 206 since; 2^23 int32 250 / 230, 2^26 1037 / 1001.)  us per
// call of `unique`, sorted / asked first: 2^23 int32 of 1000 values 222 / 91, of 2^18 223 / 144, of 2^23 243 / 270; 2^22 int64 of 1000 values 200 / 87, of 2^18
// 196 / 150, of 2^22 206 / 235; and 2^22 int32 180 / 94, 180 / 144, 187 / 212: too much for what it gives.
constexpr uint64_t collect_min_volume(int key_bytes) { return 1ull << (key_bytes == 4 ? 23 : 22); }

static_assert(COLLECT_FEW_MAX <= COLLECT_KNOWN_MAX && COLLECT_HEAVY_MAX <= COLLECT_KNOWN_MAX, "room for them");

enum : uint32_t { COLLECT_NONE = 0, COLLECT_FEW = 1, COLLECT_MANY = 2 };
// The head of the workspace; the caller reads the first three words and the last.
struct CollectPlan {
  uint32_t mode;
  uint32_t failed;
  uint32_t count;      // of the list
  uint32_t saw_empty;  // the key that stands for an empty slot is in the array
  uint32_t n_known;
  uint32_t doubt;      // there may be far more values than the mode is for
};

template <typename KeyT>
__device__ constexpr KeyT collect_empty()
{
  return static_cast<KeyT>(0x9E3779B97F4A7C15ull);
}
// (one multiplication, which takes as long as four other instructions)
__device__ __forceinline__ uint32_t collect_hash(uint32_t k) { return (k ^ (k >> 15)) * 0x9E3779B1u; }
__device__ __forceinline__ uint32_t collect_hash(uint64_t k)
{
  const uint32_t lo = static_cast<uint32_t>(k), hi = static_cast<uint32_t>(k >> 32);
  return collect_hash(lo ^ __builtin_rotateleft32(hi, 13) ^ (hi >> 7));
}
// (classes take the upper 8 bits of a hash, tables those below)
__device__ __forceinline__ uint32_t collect_class(uint32_t hash) { return hash >> 24; }
// Where a key's slots begin: at one of those that a 16-byte read starts with.
template <int SLOTS, typename KeyT>
__device__ __forceinline__ uint32_t collect_slot(uint32_t hash)
{
  constexpr uint32_t PER_READ = 16 / sizeof(KeyT);
  return (hash >> 9) & (SLOTS - PER_READ);
}
template <typename KeyT>
__device__ __forceinline__ KeyT collect_cas(KeyT* p, KeyT expected, KeyT key)
{
  if constexpr (sizeof(KeyT) == 8) {
    return static_cast<KeyT>(atomicCAS(reinterpret_cast<unsigned long long*>(p), static_cast<unsigned long long>(expected),
                                       static_cast<unsigned long long>(key)));
  } else {
    return static_cast<KeyT>(atomicCAS(p, expected, key));
  }
}
// Enters a key per lane into a table in LDS that has room for all of them; true where it was not there.
template <int SLOTS, typename KeyT>
__device__ __forceinline__ bool collect_enter(KeyT* table, KeyT key, bool valid)
{
  constexpr KeyT EMPTY = collect_empty<KeyT>();
  uint32_t slot        = collect_slot<SLOTS, KeyT>(collect_hash(key));
  bool added           = false;
  bool todo            = valid;
  for (int step = 0; step < SLOTS && __ballot(todo) != 0; ++step) {
    if (todo) {
      KeyT there = table[slot];
      if (there == EMPTY) {
        there = collect_cas<KeyT>(&table[slot], EMPTY, key);
        added = there == EMPTY;
        todo  = !added && there != key;
      } else {
        todo = there != key;
      }
      slot = (slot + 1) & (SLOTS - 1);
    }
  }
  return added;
}
// Is the key in the slots of its first read?
template <int SLOTS, typename KeyT>
__device__ __forceinline__ bool collect_known(const KeyT* table, KeyT key)
{
  constexpr int PER_READ = 16 / sizeof(KeyT);
  const uint4 q          = *reinterpret_cast<const uint4*>(table + collect_slot<SLOTS, KeyT>(collect_hash(key)));
  KeyT there[PER_READ];
  __builtin_memcpy(there, &q, 16);
  bool known = false;
#pragma unroll
  for (int j = 0; j < PER_READ; ++j) {
    known |= there[j] == key;
  }
  return known & (key != collect_empty<KeyT>());
}

// A workgroup's table in LDS.  Nearly every key is a repetition and found by the one read of collect_known; the others of a
// wave wait in a queue until a wave's worth of them is entered together (one by one, with most lanes idle, entering took
// four fifths of the time: 2^26 keys of 2^20 values 336 us, the step over the classes).
template <typename KeyT, int SLOTS, uint32_t FULL>
struct CollectTable {
  KeyT* table;
  KeyT* queue;     // of the wave, two wave's worths
  uint32_t* count;  // values in the table, of the workgroup
  uint32_t* empty;  // has the key that stands for an empty slot come up?
  uint32_t queued = 0;
  bool failed     = false;

  __device__ __forceinline__ void drain(uint32_t keep)
  {
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    while (queued > keep) {  // uniform
      failed = failed || *static_cast<volatile uint32_t*>(count) > FULL;
      if (failed) {
        queued = 0;
        return;
      }
      const uint32_t take = queued < WAVE ? queued : WAVE;
      const KeyT k        = queue[lane < take ? queued - take + lane : 0];
      const bool valid    = lane < take && k != collect_empty<KeyT>();
      if (lane < take && !valid) {
        *empty = 1;
      }
      const bool added    = collect_enter<SLOTS>(table, k, valid);
      const uint64_t bal  = __ballot(added);
      if (bal != 0 && lane == 0) {
        atomicAdd(count, static_cast<uint32_t>(__builtin_popcountll(bal)));
      }
      queued -= take;
      __builtin_amdgcn_wave_barrier();
    }
  }
  // N keys of every lane
  template <int N>
  __device__ __forceinline__ void add(const KeyT (&k)[N], const bool (&valid)[N])
  {
    bool known[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      known[j] = collect_known<SLOTS>(table, k[j]);
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const bool wait    = valid[j] && !known[j];
      const uint64_t bal = __ballot(wait);
      if (bal != 0) {  // uniform
        if (wait) {
          queue[queued + lanes_below(bal)] = k[j];
        }
        queued += static_cast<uint32_t>(__builtin_popcountll(bal));
        __builtin_amdgcn_wave_barrier();  // (LDS operations of a wave execute in order)
        if (queued >= WAVE) {
          drain(WAVE - 1);
        }
      }
    }
  }
};

// Values of very unlike frequency make Chao's estimate, a lower bound, far too low: of 2^25 keys spread evenly over the logarithm of
// 2^24 it sees 47 000 values where there are 5.2 million, and the tables fill up after all the work (`unique` 1088 us sorted, 1360
// this way and then sorted).  Values of like frequencies are seen once, twice and three times as a Poisson law has it, f1 f3 /
// f2^2 = 2/3 if they are many; a tail of rarer and rarer ones shows in a larger f3.  Then the sample is read as one of
// values whose frequencies fall with their rank: c / x^2 dx of them are expected x times in the sample, from some least x on, which f1 =
// c (ln(1 / x) - 0.577) and f2 = c / 2 give, and so many of them are expected in n keys.  (A few frequent values beside very many
// rare ones of one frequency show in nothing: those still fail.)  2^23 keys over the logarithm of 2^22, 1.4 million values, are still
// tried: 310 sorted, 209.
__device__ __forceinline__ double collect_tail(double f1, double f2, double f3, uint64_t n)
{
  const double like = f2 * f2 / 1.5 / (f1 > 1.0 ? f1 : 1.0);  // f3 of like frequencies
  if (f3 <= 3.0 + 2.0 * like + 3.0 * sqrt(like)) {
    return 0.0;
  }
  const double c    = 2.0 * (f2 > 1.0 ? f2 : 1.0);
  const double x    = exp(-f1 / c - 0.5772);
  const double more = static_cast<double>(n) / COLLECT_SAMPLES;
  return x * more < 0.3 ? c * more * (0.4228 - log(x * more)) : c / x;
}
// The same for few values: where frequencies fall as a power of the rank without end, n keys have c n^a of them, with an a that is the share
// of the sample's that it has once.
__device__ __forceinline__ double collect_growth(double seen, double f1, uint64_t n)
{
  return seen * exp2(f1 / seen * log2(static_cast<double>(n) / COLLECT_SAMPLES));
}

// The plan, from the sampled keys, by one workgroup.  Their hashes stand for them: two values of one hash count as one, which
// only the estimate notices.
template <typename KeyT>
__global__ __launch_bounds__(COLLECT_BLOCK) void collect_plan_kernel(const KeyT* __restrict__ sample, uint64_t n, CollectPlan* plan,
                                                                       KeyT* __restrict__ list, KeyT* __restrict__ heavy,
                                                                       KeyT* __restrict__ table)
{
  constexpr int EACH = COLLECT_SAMPLES / COLLECT_BLOCK;
  __shared__ uint32_t s_hash[COLLECT_SLOTS];       // 0: empty
  __shared__ uint32_t s_count[COLLECT_SLOTS / 2];  // 16 bits each
  __shared__ uint16_t s_first[COLLECT_SLOTS];      // a sampled key of the value
  __shared__ uint32_t s_sum[4];
  __shared__ uint32_t s_heavy, s_mode, s_empty;
  const uint32_t tid = threadIdx.x;
  KeyT key[EACH];
#pragma unroll
  for (int r = 0; r < EACH; ++r) {
    key[r] = sample[r * COLLECT_BLOCK + tid];
  }
  for (uint32_t j = tid; j < COLLECT_SLOTS; j += COLLECT_BLOCK) {
    s_hash[j] = 0;
    if (j < COLLECT_SLOTS / 2) {
      s_count[j] = 0;
    }
  }
  if (tid < 4) {
    s_sum[tid] = 0;
  }
  if (tid == 0) {
    s_heavy = 0;
    s_empty = 0;
  }
  __syncthreads();
  uint32_t slot[EACH], f[EACH], there[EACH];
#pragma unroll
  for (int r = 0; r < EACH; ++r) {
    const uint32_t h = collect_hash(key[r]);
    f[r]             = h != 0 ? h : 1u;
    slot[r]          = (h >> 9) & (COLLECT_SLOTS - 1);
    there[r]         = atomicCAS(&s_hash[slot[r]], 0u, f[r]);
  }
#pragma unroll
  for (int r = 0; r < EACH; ++r) {
    for (int step = 0; step < COLLECT_SLOTS && there[r] != 0u && there[r] != f[r]; ++step) {  // (8192 keys in 16 384 slots: one is free)
      slot[r]  = (slot[r] + 1) & (COLLECT_SLOTS - 1);
      there[r] = atomicCAS(&s_hash[slot[r]], 0u, f[r]);
    }
    if (there[r] == 0u) {
      s_first[slot[r]] = static_cast<uint16_t>(r * COLLECT_BLOCK + tid);
    }
    atomicAdd(&s_count[slot[r] / 2], slot[r] % 2 != 0 ? 0x10000u : 1u);
  }
  __syncthreads();
  uint32_t once = 0, twice = 0, thrice = 0, values = 0;
  for (uint32_t j = tid; j < COLLECT_SLOTS; j += COLLECT_BLOCK) {
    const uint32_t c = (s_count[j / 2] >> (j % 2 * 16)) & 0xFFFFu;
    values += c != 0 ? 1u : 0u;
    once += c == 1 ? 1u : 0u;
    twice += c == 2 ? 1u : 0u;
    thrice += c == 3 ? 1u : 0u;
  }
  values = wave_inclusive_sum_dpp(values);
  once   = wave_inclusive_sum_dpp(once);
  twice  = wave_inclusive_sum_dpp(twice);
  thrice = wave_inclusive_sum_dpp(thrice);
  if (tid % WAVE == WAVE - 1) {
    atomicAdd(&s_sum[0], values);
    atomicAdd(&s_sum[1], once);
    atomicAdd(&s_sum[2], twice);
    atomicAdd(&s_sum[3], thrice);
  }
  __syncthreads();
  if (tid == 0) {
    const double seen = s_sum[0], f1 = s_sum[1], f2 = s_sum[2];
    const double all  = seen + f1 * f1 / (2.0 * (f2 > 1.0 ? f2 : 1.0));
    uint32_t mode     = COLLECT_NONE;
    if (all <= COLLECT_FEW_MAX) {
      mode = COLLECT_FEW;
    } else if (all <= collect_many_max(sizeof(KeyT)) && all * 4.0 <= static_cast<double>(n)) {
      mode = COLLECT_MANY;
    }
    const double room = collect_tail_max(sizeof(KeyT)), quarter = static_cast<double>(n) / 4.0;
    const bool tail   = mode == COLLECT_MANY && collect_tail(f1, f2, s_sum[3], n) > (room < quarter ? room : quarter);
    plan->doubt       = tail || (mode == COLLECT_FEW && f1 > COLLECT_FEW_ONCE * f2 + 4.0 && collect_growth(seen, f1, n) > COLLECT_FEW_GROWTH) ? 1u : 0u;
    s_mode            = mode;
  }
  __syncthreads();
  const uint32_t mode = s_mode;
  if (mode != COLLECT_NONE) {
    const uint32_t least = mode == COLLECT_FEW ? 1u : static_cast<uint32_t>(COLLECT_HEAVY);
    for (uint32_t j = tid; j < COLLECT_SLOTS; j += COLLECT_BLOCK) {
      if (((s_count[j / 2] >> (j % 2 * 16)) & 0xFFFFu) >= least) {
        const uint32_t at = atomicAdd(&s_heavy, 1u);  // (at most COLLECT_KNOWN_MAX)
        const KeyT k      = sample[s_first[j]];
        heavy[at]         = k;
        list[at]          = k;
        if (k == collect_empty<KeyT>()) {
          s_empty = 1;
        }
      }
    }
  }
  if (mode == COLLECT_FEW) {
    for (uint32_t j = tid; j < COLLECT_SLOTS; j += COLLECT_BLOCK) {
      table[j] = collect_empty<KeyT>();
    }
  }
  __syncthreads();
  if (tid == 0) {
    plan->mode      = mode;
    plan->failed    = 0;
    plan->count     = s_heavy;
    plan->saw_empty = s_empty;
    plan->n_known   = s_heavy;
  }
}

__device__ __forceinline__ void collect_refuse(CollectPlan* plan)
{
  if (threadIdx.x == 0) {
    plan->failed = 1;
  }
}

// The key that stands for empty slots, by the first workgroup that has met it.
template <typename KeyT>
__device__ __forceinline__ void collect_list_empty(CollectPlan* plan, KeyT* list, uint32_t room)
{
  if (atomicExch(&plan->saw_empty, 1u) == 0) {
    const uint32_t at = atomicAdd(&plan->count, 1u);
    if (at < room) {
      list[at] = collect_empty<KeyT>();
    }
  }
}

template <typename KeyT>
__global__ __launch_bounds__(COLLECT_BLOCK) void collect_few_kernel(const KeyT* __restrict__ values, uint64_t n, CollectPlan* plan,
                                                                     const KeyT* __restrict__ known, KeyT* __restrict__ list,
                                                                     uint32_t room, KeyT* __restrict__ table)
{
  constexpr KeyT EMPTY = collect_empty<KeyT>();
  constexpr int VEC    = 16 / sizeof(KeyT);
  __shared__ __align__(16) KeyT s_table[COLLECT_FEW_SLOTS];
  __shared__ KeyT s_queue[COLLECT_WAVES * 2 * WAVE];
  __shared__ uint64_t s_listed[COLLECT_FEW_SLOTS / WAVE];  // a bit per slot: a value of the sample
  __shared__ uint32_t s_count, s_empty;
  if (plan->mode != COLLECT_FEW) {  // (the host was told another mode)
    collect_refuse(plan);
    return;
  }
  const uint32_t tid = threadIdx.x;
  for (uint32_t j = tid; j < COLLECT_FEW_SLOTS; j += COLLECT_BLOCK) {
    s_table[j] = EMPTY;
  }
  if (tid == 0) {
    s_count = 0;
    s_empty = 0;
  }
  __syncthreads();
  const uint32_t n_known = plan->n_known;
  for (uint32_t j0 = 0; j0 < n_known; j0 += COLLECT_BLOCK) {  // uniform
    const uint32_t j = j0 + tid;
    const KeyT k     = known[j < n_known ? j : 0];
    collect_enter<COLLECT_FEW_SLOTS>(s_table, k, j < n_known && k != EMPTY);
  }
  if (tid == 0) {
    s_count = n_known;
  }
  __syncthreads();
  for (uint32_t j = tid; j < COLLECT_FEW_SLOTS; j += COLLECT_BLOCK) {
    const uint64_t bal = __ballot(s_table[j] != EMPTY);
    if (j % WAVE == 0) {
      s_listed[j / WAVE] = bal;
    }
  }
  __syncthreads();
  CollectTable<KeyT, COLLECT_FEW_SLOTS, COLLECT_FEW_FULL> t{s_table, s_queue + tid / WAVE * 2 * WAVE, &s_count, &s_empty};
  // 16-byte loads over the aligned middle, the ends by the first workgroup
  uint64_t head = ((16u - (reinterpret_cast<uintptr_t>(values) & 15u)) & 15u) / sizeof(KeyT);
  head          = head < n ? head : n;
  const uint64_t nvec = (n - head) / VEC;
  const uint64_t tail = head + nvec * VEC;
  const uint4* vp     = reinterpret_cast<const uint4*>(values + head);
  if (blockIdx.x == 0) {
    const uint64_t ends = head + (n - tail);  // fewer than 2 * VEC
    const KeyT k[1]     = {tid < ends ? values[tid < head ? tid : tail + (tid - head)] : KeyT{}};
    const bool valid[1] = {tid < ends};
    t.add(k, valid);
  }
  const uint64_t step = static_cast<uint64_t>(gridDim.x) * COLLECT_BLOCK;
  for (uint64_t v0 = static_cast<uint64_t>(blockIdx.x) * COLLECT_BLOCK; v0 < nvec && !t.failed; v0 += 4 * step) {  // uniform per wave
    uint4 q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint64_t v = v0 + i * step + tid;
      q[i]             = vp[v < nvec ? v : nvec - 1];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      KeyT k[VEC];
      bool valid[VEC];
      __builtin_memcpy(k, &q[i], 16);
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        valid[j] = v0 + i * step + tid < nvec;
      }
      t.add(k, valid);
    }
  }
  t.drain(0);
  __syncthreads();
  if (s_count > COLLECT_FEW_FULL) {
    if (tid == 0) {
      plan->failed = 1;
    }
    return;
  }
  if (tid == 0 && s_empty != 0) {
    collect_list_empty<KeyT>(plan, list, room);
  }
  // The workgroup's values into the table in memory, and those that are new to it into the list, a wave's worth with one addition
  // to the one counter.  A wave that finds no place gives up.
  for (uint32_t j0 = 0; j0 < COLLECT_FEW_SLOTS; j0 += COLLECT_BLOCK) {  // uniform
    const uint32_t j = j0 + tid;
    const KeyT k     = s_table[j];
    bool todo        = k != EMPTY && ((s_listed[j / WAVE] >> (j % WAVE)) & 1u) == 0;
    bool added       = false;
    uint32_t slot    = collect_slot<COLLECT_SLOTS, KeyT>(collect_hash(k));
    for (int probe = 0; probe < COLLECT_FEW_PROBES && todo; ++probe) {
      KeyT there = __hip_atomic_load(&table[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (there == EMPTY) {
        there = collect_cas<KeyT>(&table[slot], EMPTY, k);
        added = there == EMPTY;
      }
      todo = !added && there != k;
      slot = (slot + 1) & (COLLECT_SLOTS - 1);
    }
    const uint64_t bal = __ballot(added);
    if (bal != 0) {
      uint32_t at = 0;
      if (tid % WAVE == 0) {
        at = atomicAdd(&plan->count, static_cast<uint32_t>(__builtin_popcountll(bal)));
      }
      at = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(at))) + lanes_below(bal);
      if (added && at < room) {
        list[at] = k;
      }
    }
    if (__ballot(todo) != 0) {
      if (tid % WAVE == 0) {
        plan->failed = 1;
      }
      break;
    }
  }
}

// A tile into the order of its classes, heavy values left out.  The order inside a class is whatever the atomics make it.
template <typename KeyT>
__global__ __launch_bounds__(COLLECT_BLOCK) void collect_group_kernel(const KeyT* __restrict__ values, uint64_t n,
                                                                        const CollectPlan* __restrict__ plan,
                                                                        const KeyT* __restrict__ heavy, KeyT* __restrict__ grouped,
                                                                        uint16_t* __restrict__ starts)
{
  constexpr KeyT EMPTY = collect_empty<KeyT>();
  __shared__ __align__(16) KeyT s_keys[COLLECT_TILE];
  __shared__ uint32_t s_start[COLLECT_CLASSES];
  __shared__ uint32_t s_wave[COLLECT_CLASSES / WAVE];
  static_assert(COLLECT_HEAVY_SLOTS <= COLLECT_TILE, "the heavy values' table is read before the keys take its place");
  if (plan->mode != COLLECT_MANY) {
    return;
  }
  const uint32_t tid     = threadIdx.x;
  const uint32_t lane    = tid & (WAVE - 1);
  const uint32_t n_heavy = plan->n_known;
  const uint64_t first   = static_cast<uint64_t>(blockIdx.x) * COLLECT_TILE;
  const uint32_t len     = n - first < COLLECT_TILE ? static_cast<uint32_t>(n - first) : COLLECT_TILE;
  const KeyT* const in   = values + first;
  KeyT key[COLLECT_ITEMS];
#pragma unroll
  for (int i = 0; i < COLLECT_ITEMS; ++i) {
    const uint32_t o = i * COLLECT_BLOCK + tid;
    key[i]           = in[o < len ? o : len - 1];
  }
  if (tid < COLLECT_CLASSES) {
    s_start[tid] = 0;
  }
  if (n_heavy != 0) {  // uniform
    for (uint32_t j = tid; j < COLLECT_HEAVY_SLOTS; j += COLLECT_BLOCK) {
      s_keys[j] = EMPTY;
    }
    __syncthreads();
    const KeyT k = tid < n_heavy ? heavy[tid] : EMPTY;
    collect_enter<COLLECT_HEAVY_SLOTS>(s_keys, k, k != EMPTY);
  }
  static_assert(COLLECT_HEAVY_MAX <= COLLECT_BLOCK && 2 * COLLECT_HEAVY_MAX <= COLLECT_HEAVY_SLOTS, "a thread per heavy value, half a table");
  __syncthreads();
  uint32_t where[COLLECT_ITEMS];  // class, and in the upper half which of it; ~0: left out
#pragma unroll
  for (int i = 0; i < COLLECT_ITEMS; ++i) {
    const uint32_t h = collect_hash(key[i]);
    bool keep        = i * COLLECT_BLOCK + tid < len;
    if (n_heavy != 0) {
      uint32_t slot = collect_slot<COLLECT_HEAVY_SLOTS, KeyT>(h);
      for (int step = 0; step < COLLECT_HEAVY_SLOTS; ++step) {
        const KeyT there = s_keys[slot];
        keep             = keep && there != key[i];
        if (there == EMPTY || there == key[i]) {
          break;
        }
        slot = (slot + 1) & (COLLECT_HEAVY_SLOTS - 1);
      }
      keep = keep || (key[i] == EMPTY && i * COLLECT_BLOCK + tid < len);  // (its own flag says whether it is listed)
    }
    where[i] = ~0u;
    if (keep) {
      const uint32_t c = collect_class(h);
      where[i]         = c | (atomicAdd(&s_start[c], 1u) << 16);
    }
  }
  __syncthreads();
  uint32_t count = 0, incl = 0;
  if (tid < COLLECT_CLASSES) {
    count = s_start[tid];
    incl  = wave_inclusive_sum_dpp(count);
    if (lane == WAVE - 1) {
      s_wave[tid / WAVE] = incl;
    }
  }
  __syncthreads();
  uint16_t* const to = starts + static_cast<uint64_t>(blockIdx.x) * (COLLECT_CLASSES + 1);
  if (tid < COLLECT_CLASSES) {
    uint32_t run = incl - count;
#pragma unroll
    for (uint32_t w = 0; w < COLLECT_CLASSES / WAVE; ++w) {
      run += w < tid / WAVE ? s_wave[w] : 0u;
    }
    s_start[tid] = run;
    to[tid]      = static_cast<uint16_t>(run);
    if (tid == COLLECT_CLASSES - 1) {
      to[COLLECT_CLASSES] = static_cast<uint16_t>(run + count);
    }
  }
  __syncthreads();
  const uint32_t kept = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
  static_assert(COLLECT_CLASSES / WAVE == 4, "four waves of classes");
#pragma unroll
  for (int i = 0; i < COLLECT_ITEMS; ++i) {
    if (where[i] != ~0u) {
      s_keys[s_start[where[i] & 0xFFFFu] + (where[i] >> 16)] = key[i];
    }
  }
  __syncthreads();
  for (uint32_t o = tid; o < kept; o += COLLECT_BLOCK) {
    grouped[first + o] = s_keys[o];
  }
}

// One class: its part of every tile into a table in LDS, the table into the list.
template <typename KeyT>
__global__ __launch_bounds__(COLLECT_BLOCK) void collect_class_kernel(const KeyT* __restrict__ grouped,
                                                                        const uint16_t* __restrict__ starts, uint32_t tiles,
                                                                        CollectPlan* plan, KeyT* __restrict__ list, uint32_t room)
{
  constexpr KeyT EMPTY    = collect_empty<KeyT>();
  constexpr int SLOTS     = collect_class_slots(sizeof(KeyT));
  constexpr uint32_t FULL = collect_class_full(sizeof(KeyT));
  __shared__ __align__(16) KeyT s_table[SLOTS];
  __shared__ KeyT s_queue[COLLECT_WAVES * 2 * WAVE];
  __shared__ uint32_t s_count, s_empty, s_base, s_next;
  if (plan->mode != COLLECT_MANY) {
    collect_refuse(plan);
    return;
  }
  const uint32_t tid  = threadIdx.x;
  const uint32_t lane = tid & (WAVE - 1);
  const uint32_t wave = tid / WAVE;
  for (uint32_t j = tid; j < SLOTS; j += COLLECT_BLOCK) {
    s_table[j] = EMPTY;
  }
  if (tid == 0) {
    s_count = 0;
    s_empty = 0;
    s_next  = 0;
  }
  __syncthreads();
  CollectTable<KeyT, SLOTS, FULL> table{s_table, s_queue + wave * 2 * WAVE, &s_count, &s_empty};
  constexpr int AHEAD = 8;  // segments in flight
  for (uint32_t t0 = wave * WAVE; t0 < tiles && !table.failed; t0 += COLLECT_WAVES * WAVE) {  // uniform per wave
    // a lane per tile looks up the class's part of it
    uint32_t from = 0, len = 0;
    if (t0 + lane < tiles) {
      const uint16_t* const at = starts + static_cast<uint64_t>(t0 + lane) * (COLLECT_CLASSES + 1) + blockIdx.x;
      from                     = at[0];
      len                      = at[1] - from;
    }
    const uint32_t here = tiles - t0 < WAVE ? tiles - t0 : WAVE;
    KeyT next[AHEAD];
    const auto request = [&](uint32_t j0) {  // (lanes past the last tile hold a length of 0)
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) {
        const uint32_t f = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(from), j0 + j));
        const uint32_t l = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(len), j0 + j));
        next[j]          = KeyT{};
        if (lane < l) {
          next[j] = grouped[static_cast<uint64_t>(t0 + j0 + j) * COLLECT_TILE + f + lane];
        }
      }
    };
    request(0);
    for (uint32_t j0 = 0; j0 < here; j0 += AHEAD) {
      KeyT k[AHEAD];
      uint32_t l[AHEAD], f[AHEAD];
      bool valid[AHEAD];
      uint32_t longest = 0;
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) {
        k[j]     = next[j];
        f[j]     = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(from), j0 + j));
        l[j]     = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(len), j0 + j));
        valid[j] = lane < l[j];
        longest  = l[j] > longest ? l[j] : longest;
      }
      if (j0 + AHEAD < here) {
        request(j0 + AHEAD);
      }
      table.add(k, valid);
      for (uint32_t more = WAVE; more < longest; more += WAVE) {  // uniform: what is left of segments longer than a wave
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
          valid[j] = more + lane < l[j];
          k[j]     = valid[j] ? grouped[static_cast<uint64_t>(t0 + j0 + j) * COLLECT_TILE + f[j] + more + lane] : KeyT{};
        }
        table.add(k, valid);
      }
    }
  }
  table.drain(0);
  static_assert(WAVE % AHEAD == 0, "whole groups of lanes");
  __syncthreads();
  if (s_count > FULL) {  // (uniform; a wave that stopped has seen the same)
    if (tid == 0) {
      plan->failed = 1;
    }
    return;
  }
  if (tid == 0) {
    s_base = atomicAdd(&plan->count, s_count);
    if (s_empty != 0) {
      collect_list_empty<KeyT>(plan, list, room);
    }
  }
  __syncthreads();
  const uint32_t base = s_base;
  for (uint32_t j = tid; j < SLOTS; j += COLLECT_BLOCK) {
    const KeyT k       = s_table[j];
    const uint64_t bal = __ballot(k != EMPTY);
    uint32_t at        = 0;
    if (lane == 0 && bal != 0) {
      at = atomicAdd(&s_next, static_cast<uint32_t>(__builtin_popcountll(bal)));
    }
    at = base + static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(at))) + lanes_below(bal);
    if (k != EMPTY && at < room) {
      list[at] = k;
    }
  }
}

struct CollectLayout {
  uint64_t off_sample, off_known, off_table, off_list, off_starts, off_grouped, total;
  uint32_t tiles, room;
};
static CollectLayout collect_layout(int key_bytes, uint64_t n)
{
  CollectLayout L{};
  L.tiles       = static_cast<uint32_t>((n + COLLECT_TILE - 1) / COLLECT_TILE);
  L.room        = COLLECT_CLASSES * (collect_class_full(key_bytes) + COLLECT_BLOCK) + COLLECT_HEAVY_MAX + 1;
  L.room        = n < L.room ? static_cast<uint32_t>(n) : L.room;
  L.off_sample  = WORKSPACE_ALIGN;
  L.off_known   = L.off_sample + COLLECT_SAMPLES * static_cast<uint64_t>(key_bytes);
  L.off_table   = L.off_known + align_up(COLLECT_KNOWN_MAX * static_cast<uint64_t>(key_bytes), WORKSPACE_ALIGN);
  L.off_list    = L.off_table + COLLECT_SLOTS * static_cast<uint64_t>(key_bytes);
  L.off_starts  = L.off_list + align_up(static_cast<uint64_t>(L.room) * key_bytes, WORKSPACE_ALIGN);
  L.off_grouped = L.off_starts + align_up(static_cast<uint64_t>(L.tiles) * (COLLECT_CLASSES + 1) * sizeof(uint16_t), WORKSPACE_ALIGN);
  L.total       = L.off_grouped + align_up(n * key_bytes, WORKSPACE_ALIGN);
  return L;
}
static_assert(sizeof(CollectPlan) <= WORKSPACE_ALIGN, "the plan has the head of the workspace");

template <typename KeyT>
static int collect_plan_typed(const void* values_v, uint64_t n, unsigned char* ws, hipStream_t s)
{
  const CollectLayout L = collect_layout(sizeof(KeyT), n);
  const KeyT* values    = static_cast<const KeyT*>(values_v);
  KeyT* sample          = reinterpret_cast<KeyT*>(ws + L.off_sample);
  {
    ProfileScope prof("collect_sample", s);
    hipLaunchKernelGGL((split_gather_kernel<KeyT>), dim3(COLLECT_SAMPLES / 256), dim3(256), 0, s, values, static_cast<uint32_t>(n),
                       static_cast<uint32_t>(COLLECT_SAMPLES), sample, static_cast<const uint32_t*>(nullptr));
  }
  CPN_HIP_TRY(hipGetLastError());
  {
    ProfileScope prof("collect_plan", s);
    hipLaunchKernelGGL((collect_plan_kernel<KeyT>), dim3(1), dim3(COLLECT_BLOCK), 0, s, sample, n, reinterpret_cast<CollectPlan*>(ws),
                       reinterpret_cast<KeyT*>(ws + L.off_list), reinterpret_cast<KeyT*>(ws + L.off_known),
                       reinterpret_cast<KeyT*>(ws + L.off_table));
  }
  CPN_HIP_TRY(hipGetLastError());
  return CPN_OK;
}

template <typename KeyT>
static int collect_typed(const void* values_v, uint64_t n, uint32_t mode, unsigned char* ws, hipStream_t s)
{
  const CollectLayout L = collect_layout(sizeof(KeyT), n);
  const KeyT* values    = static_cast<const KeyT*>(values_v);
  CollectPlan* plan     = reinterpret_cast<CollectPlan*>(ws);
  KeyT* known           = reinterpret_cast<KeyT*>(ws + L.off_known);
  KeyT* list            = reinterpret_cast<KeyT*>(ws + L.off_list);
  if (mode == COLLECT_FEW) {
    // as many workgroups as fit at once
    const uint32_t grid = static_cast<uint32_t>((sizeof(KeyT) == 4 ? 2 : 1) * compute_units());
    ProfileScope prof("collect_few", s);
    hipLaunchKernelGGL((collect_few_kernel<KeyT>), dim3(grid), dim3(COLLECT_BLOCK), 0, s, values, n, plan, known, list, L.room,
                       reinterpret_cast<KeyT*>(ws + L.off_table));
    CPN_HIP_TRY(hipGetLastError());
    return CPN_OK;
  }
  uint16_t* starts = reinterpret_cast<uint16_t*>(ws + L.off_starts);
  KeyT* grouped    = reinterpret_cast<KeyT*>(ws + L.off_grouped);
  {
    ProfileScope prof("collect_group", s);
    hipLaunchKernelGGL((collect_group_kernel<KeyT>), dim3(L.tiles), dim3(COLLECT_BLOCK), 0, s, values, n, plan, known, grouped, starts);
  }
  CPN_HIP_TRY(hipGetLastError());
  {
    ProfileScope prof("collect_class", s);
    hipLaunchKernelGGL((collect_class_kernel<KeyT>), dim3(COLLECT_CLASSES), dim3(COLLECT_BLOCK), 0, s, grouped, starts, L.tiles, plan,
                       list, L.room);
  }
  CPN_HIP_TRY(hipGetLastError());
  return CPN_OK;
}

static int collect_check(int dtype, const void* values, uint64_t volume, const void* temp, uint64_t temp_bytes)
{
  const KeyKind k     = key_kind(dtype);
  const uint64_t need = cpn_distinct_temp_bytes(dtype, volume, nullptr);
  if (k.bytes == 0 || k.codec < 0) {
    return CPN_ERR_DTYPE;
  }
  if (need == 0) {
    return CPN_ERR_UNSUPPORTED;
  }
  if (values == nullptr) {
    return CPN_ERR_NULL;
  }
  if (temp == nullptr || temp_bytes < need || (reinterpret_cast<uintptr_t>(temp) % WORKSPACE_ALIGN) != 0) {
    return CPN_ERR_TEMP;
  }
  if ((reinterpret_cast<uintptr_t>(values) & static_cast<uintptr_t>(k.bytes - 1)) != 0) {
    return CPN_ERR_ALIGN;
  }
  return CPN_OK;
}

}  // namespace cpn

extern "C" uint64_t cpn_distinct_temp_bytes(int dtype, uint64_t volume, uint64_t* list_offset)
{
  using namespace cpn;
  const KeyKind k = key_kind(dtype);
  if ((k.bytes != 4 && k.bytes != 8) || (k.codec != CODEC_UNSIGNED && k.codec != CODEC_SIGNED) || volume < collect_min_volume(k.bytes) ||
      volume >= (1ull << 31)) {
    return 0;
  }
  const CollectLayout L = collect_layout(k.bytes, volume);
  if (list_offset != nullptr) {
    *list_offset = L.off_list;
  }
  return L.total;
}

extern "C" int cpn_distinct_plan(int dtype, const void* values, uint64_t volume, void* temp, uint64_t temp_bytes, void* stream)
{
  using namespace cpn;
  const int bad = collect_check(dtype, values, volume, temp, temp_bytes);
  if (bad != CPN_OK) {
    return bad;
  }
  unsigned char* ws = static_cast<unsigned char*>(temp);
  hipStream_t s     = static_cast<hipStream_t>(stream);
  return key_kind(dtype).bytes == 4 ? collect_plan_typed<uint32_t>(values, volume, ws, s)
                                    : collect_plan_typed<uint64_t>(values, volume, ws, s);
}

extern "C" int cpn_distinct(int dtype, const void* values, uint64_t volume, int mode, void* temp, uint64_t temp_bytes, void* stream)
{
  using namespace cpn;
  const int bad = collect_check(dtype, values, volume, temp, temp_bytes);
  if (bad != CPN_OK) {
    return bad;
  }
  if (mode != static_cast<int>(COLLECT_FEW) && mode != static_cast<int>(COLLECT_MANY)) {
    return CPN_ERR_UNSUPPORTED;
  }
  unsigned char* ws = static_cast<unsigned char*>(temp);
  hipStream_t s     = static_cast<hipStream_t>(stream);
  return key_kind(dtype).bytes == 4 ? collect_typed<uint32_t>(values, volume, static_cast<uint32_t>(mode), ws, s)
                                    : collect_typed<uint64_t>(values, volume, static_cast<uint32_t>(mode), ws, s);
}
