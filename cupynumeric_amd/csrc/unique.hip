// unique: the sorted distinct values of an array.
//
// Replaces UniqueTask's GPU variant on one processor (src/cupynumeric/set/unique.cu:137-204:
// copy into a buffer, thrust::sort, thrust::unique, result handed back as an unbound store of
// the distinct count; the tree reduction over ranks :49-135 belongs to the multi-GPU case).
// Here: the library's own stable sort into the workspace, then a compaction that keeps the
// first element of every run of equal keys.  Equality is equality of the ordered keys of
// key_codec.h: all NaNs are one value, -0.0 and +0.0 are one value, and every complex number
// with a NaN part is one value, as for numpy.unique (equal_nan=True), whereas thrust::unique
// compares with == and keeps every NaN.
//
// Compaction in three launches: the run heads of every 4096-element tile as one bit per
// element, an exclusive scan of the tile counts by one workgroup, and the heads to their places.
// The sorted buffer is read once and then only at the heads, the output is written once; the
// number of distinct values ends up in device memory and the caller reads it.  Measured on 2^26
// int32 with 2^20 distinct values: the whole call 1055 -> 938 us against two full reads of the sorted
// buffer (heads counted, then found again and scattered: 88 + 110 us, and 24 us in a scan that
// took 1024 tiles per round).  The scan reads two bytes per tile and writes a sum per sixteen tiles, which the
// scatter's workgroups complete: with eight bytes of both per tile it took 18.6 us for 2^26 elements, and takes 4.9.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sort_driver.h"

namespace cpn {

constexpr int UNIQUE_BLOCK = 256;
constexpr int UNIQUE_ITEMS = 16;
constexpr int UNIQUE_TILE  = UNIQUE_BLOCK * UNIQUE_ITEMS;
constexpr int UNIQUE_WAVES = UNIQUE_BLOCK / WAVE;
constexpr int HEADS_BLOCK  = 1024;
constexpr int HEADS_ITEMS  = 16;

template <typename KeyT, int CODEC>
__device__ __forceinline__ bool keys_differ(const KeyT& key, const KeyT& before)
{
  using KT = KeyTraits<CODEC, KeyT>;
  uint64_t a[KT::NWORDS], b[KT::NWORDS];
  KT::words(key, a);
  KT::words(before, b);
  bool differ = false;
#pragma unroll
  for (int k = 0; k < KT::NWORDS; ++k) {
    differ = differ || (a[k] != b[k]);
  }
  if constexpr (CODEC == CODEC_COMPLEX) {
    // the most significant word is the NaN class (0 = no NaN part): the NaN classes sort last
    // and form one value
    if (a[KT::NWORDS - 1] != 0 && b[KT::NWORDS - 1] != 0) {
      differ = false;
    }
  }
  return differ;
}

// marks[64 * b ..] = one bit per element of tile b, set where a run starts; counts[b] = their number.
// Word it * UNIQUE_WAVES + wave holds the 64 elements that this wave tests in round it, so the
// words of a tile are in element order.
//
// Bound by the read of the sorted buffer: the loads of a batch are issued together, without a
// branch around them (an element past the end repeats the last one).  The bits cost a 32nd of a 4-byte key and leave the
// second pass with the heads alone to read.
template <typename KeyT, int CODEC>
__global__ __launch_bounds__(UNIQUE_BLOCK) void unique_mark_kernel(const KeyT* __restrict__ sorted,
                                                                   uint64_t n,
                                                                   uint64_t* __restrict__ marks,
                                                                   uint16_t* __restrict__ counts)
{
  __shared__ uint64_t s_mark[WAVE];
  const int lane      = threadIdx.x & (WAVE - 1);
  const int wave      = threadIdx.x / WAVE;
  const uint64_t base = static_cast<uint64_t>(blockIdx.x) * UNIQUE_TILE;
  constexpr int BATCH = sizeof(KeyT) <= 4 ? UNIQUE_ITEMS : (sizeof(KeyT) == 8 ? 8 : 4);
#pragma unroll
  for (int start = 0; start < UNIQUE_ITEMS; start += BATCH) {
    // A batch past the end is a round trip to memory for nothing (1000 complex128 values: 71 us a call with them,
    // 68 without).  The first batch, all there is for keys of up to 4 bytes, is not asked.
    if (start != 0 && base + static_cast<uint64_t>(start) * UNIQUE_BLOCK >= n) {
      if (lane < BATCH) {
        s_mark[(start + lane) * UNIQUE_WAVES + wave] = 0;
      }
      continue;
    }
    KeyT key[BATCH], before[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; ++k) {
      const uint64_t i = base + static_cast<uint64_t>(start + k) * UNIQUE_BLOCK + threadIdx.x;
      const uint64_t j = i < n ? i : n - 1;
      key[k]           = sorted[j];
      before[k]        = sorted[j != 0 ? j - 1 : 0];
    }
#pragma unroll
    for (int k = 0; k < BATCH; ++k) {
      const uint64_t i   = base + static_cast<uint64_t>(start + k) * UNIQUE_BLOCK + threadIdx.x;
      const bool differ  = keys_differ<KeyT, CODEC>(key[k], before[k]);
      const uint64_t bal = __builtin_amdgcn_ballot_w64(i < n && (i == 0 || differ));
      if (lane == 0) {
        s_mark[(start + k) * UNIQUE_WAVES + wave] = bal;
      }
    }
  }
  __syncthreads();
  if (wave == 0) {
    const uint64_t mark = s_mark[lane];
    uint32_t cnt        = static_cast<uint32_t>(__builtin_popcountll(mark));
#pragma unroll
    for (int delta = WAVE / 2; delta > 0; delta >>= 1) {
      cnt += __shfl_xor(cnt, delta, WAVE);
    }
    marks[static_cast<uint64_t>(blockIdx.x) * WAVE + lane] = mark;
    if (lane == 0) {
      counts[blockIdx.x] = static_cast<uint16_t>(cnt);
    }
  }
}

// sums[g] = heads in the tiles before group g of sixteen; sums[groups] and *total_out = all of them.  One workgroup, a group
// per thread: a round is a chain of a load, a scan and two barriers, and this way 2^26 elements are one round.  (The
// counts lie on a 16-byte boundary with room for a whole group behind the last one.)
__global__ __launch_bounds__(HEADS_BLOCK) void unique_scan_kernel(const uint16_t* __restrict__ counts, uint64_t tiles,
                                                                  uint64_t* __restrict__ sums, uint64_t* total_out)
{
  __shared__ uint32_t s_wave[HEADS_BLOCK / WAVE];
  const int lane        = threadIdx.x & (WAVE - 1);
  const int wave        = threadIdx.x / WAVE;
  const uint64_t groups = (tiles + HEADS_ITEMS - 1) / HEADS_ITEMS;
  uint64_t carry        = 0;
  for (uint64_t start = 0; start < groups; start += HEADS_BLOCK) {
    const uint64_t group = start + threadIdx.x;
    uint32_t own         = 0;  // (a round's sum is at most 2^26)
    if (group < groups) {
      uint4 q[2];
      q[0] = reinterpret_cast<const uint4*>(counts)[2 * group];
      q[1] = reinterpret_cast<const uint4*>(counts)[2 * group + 1];
      uint16_t c[HEADS_ITEMS];
      __builtin_memcpy(c, q, sizeof(c));
#pragma unroll
      for (int k = 0; k < HEADS_ITEMS; ++k) {
        own += group * HEADS_ITEMS + k < tiles ? c[k] : 0u;
      }
    }
    const uint32_t incl = wave_inclusive_sum_dpp(own);
    if (lane == WAVE - 1) {
      s_wave[wave] = incl;
    }
    __syncthreads();
    uint64_t before = carry + incl - own;
#pragma unroll
    for (int w = 0; w < HEADS_BLOCK / WAVE; ++w) {
      const uint32_t t = s_wave[w];
      before += (w < wave) ? t : 0u;
      carry += t;
    }
    if (group < groups) {
      sums[group] = before;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (sums != nullptr) {
      sums[groups] = carry;
    }
    *total_out = carry;
  }
}

// The heads of a tile go to their places in the output.  Their indexes are gathered in LDS
// first, so that a tile with few heads is one load and one store per lane and not sixteen
// rounds of a load, a wait and a store under a nearly empty mask.
template <typename KeyT>
__global__ __launch_bounds__(UNIQUE_BLOCK) void unique_scatter_kernel(const KeyT* __restrict__ sorted,
                                                                      const uint64_t* __restrict__ marks,
                                                                      const uint64_t* __restrict__ sums,
                                                                      const uint16_t* __restrict__ counts,
                                                                      KeyT* __restrict__ out)
{
  __shared__ uint64_t s_mark[WAVE];
  __shared__ uint32_t s_before[WAVE];
  __shared__ uint16_t s_head[UNIQUE_TILE];
  const int lane       = threadIdx.x & (WAVE - 1);
  const int wave       = threadIdx.x / WAVE;
  const uint64_t base  = static_cast<uint64_t>(blockIdx.x) * UNIQUE_TILE;
  const int heads      = counts[blockIdx.x];
  if (heads == 0) {
    return;  // the same for every lane
  }
  // the tiles of the group before this one, a lane each
  const uint32_t in_group = blockIdx.x % HEADS_ITEMS;
  const uint32_t others   = static_cast<uint32_t>(lane) < in_group ? counts[blockIdx.x - in_group + lane] : 0u;
  const uint32_t before   = static_cast<uint32_t>(
    __builtin_amdgcn_readlane(static_cast<int>(wave_inclusive_sum_dpp(others)), WAVE - 1));
  const uint64_t begin = sums[blockIdx.x / HEADS_ITEMS] + before;
  if (wave == 0) {
    const uint64_t mark = marks[static_cast<uint64_t>(blockIdx.x) * WAVE + lane];
    const uint32_t c    = static_cast<uint32_t>(__builtin_popcountll(mark));
    s_mark[lane]        = mark;
    s_before[lane]      = wave_inclusive_scan(c, lane) - c;
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < UNIQUE_ITEMS; ++it) {
    const int word      = it * UNIQUE_WAVES + wave;
    const uint64_t mark = s_mark[word];
    if ((mark >> lane) & 1u) {
      s_head[s_before[word] + lanes_below(mark)] = static_cast<uint16_t>(word * WAVE + lane);
    }
  }
  __syncthreads();
#pragma unroll 4
  for (int t = threadIdx.x; t < heads; t += UNIQUE_BLOCK) {
    out[begin + t] = sorted[base + s_head[t]];
  }
}
static_assert(UNIQUE_ITEMS * UNIQUE_WAVES == WAVE, "one wave scans the words of a tile");

struct UniqueLayout {
  uint64_t sort_bytes;
  uint64_t off_sorted;
  uint64_t off_counts;  // the sums of the groups of tiles, then the counts of the tiles
  uint64_t off_marks;
  uint64_t total;
  uint64_t tiles;
};

// Of the sums of the groups of tiles and the counts of the tiles behind them, and of the bits.
static uint64_t sums_bytes(uint64_t tiles) { return align_up((tiles + 1) * 8, WORKSPACE_ALIGN); }
static uint64_t marks_bytes(uint64_t tiles) { return align_up(tiles * WAVE * 8, WORKSPACE_ALIGN); }

// With `least`, the sort's workspace is what it can do with instead of what it asks for (callers that kept a size).
static UniqueLayout unique_layout(int dtype, uint64_t volume, bool least)
{
  UniqueLayout L{};
  const KeyKind k = key_kind(dtype);
  L.sort_bytes    = workspace_bytes(k.bytes, key_passes(k.bytes, k.codec), k.codec, volume, volume, true, false, false, least);
  L.tiles         = (volume + UNIQUE_TILE - 1) / UNIQUE_TILE;
  L.off_sorted    = align_up(L.sort_bytes, WORKSPACE_ALIGN);
  L.off_counts    = L.off_sorted + align_up(volume * static_cast<uint64_t>(k.bytes), WORKSPACE_ALIGN);
  L.off_marks     = L.off_counts + sums_bytes(L.tiles);
  L.total         = L.off_marks + marks_bytes(L.tiles);
  return L;
}

template <typename KeyT, int CODEC>
static int compact(const void* sorted, uint64_t n, uint64_t* marks, uint64_t* sums, uint64_t tiles, void* out,
                   uint64_t* count_out, hipStream_t stream)
{
  if (tiles >= (1ull << 31)) {
    return CPN_ERR_UNSUPPORTED;
  }
  // Behind the sums, a 16-byte boundary further on.  (2.5 bytes per tile and fewer than 64 to round up: the room is for
  // 8 bytes per tile and one more, rounded up to WORKSPACE_ALIGN.)
  uint16_t* counts = reinterpret_cast<uint16_t*>(sums + align_up((tiles + HEADS_ITEMS - 1) / HEADS_ITEMS + 1, 2));
  {
    ProfileScope prof("unique_mark", stream);
    hipLaunchKernelGGL((unique_mark_kernel<KeyT, CODEC>), dim3(static_cast<uint32_t>(tiles)), dim3(UNIQUE_BLOCK), 0,
                       stream, static_cast<const KeyT*>(sorted), n, marks, counts);
  }
  CPN_HIP_TRY(hipGetLastError());
  {
    ProfileScope prof("unique_scan", stream);
    hipLaunchKernelGGL(unique_scan_kernel, dim3(1), dim3(HEADS_BLOCK), 0, stream, counts, tiles, sums, count_out);
  }
  CPN_HIP_TRY(hipGetLastError());
  {
    ProfileScope prof("unique_scatter", stream);
    hipLaunchKernelGGL((unique_scatter_kernel<KeyT>), dim3(static_cast<uint32_t>(tiles)), dim3(UNIQUE_BLOCK), 0,
                       stream, static_cast<const KeyT*>(sorted), marks, sums, counts, static_cast<KeyT*>(out));
  }
  CPN_HIP_TRY(hipGetLastError());
  return CPN_OK;
}

static int compact_keys(const KeyKind& k, const void* sorted, uint64_t volume, uint64_t* marks, uint64_t* sums, uint64_t tiles,
                        void* out, uint64_t* count_out, hipStream_t stream)
{
#define CPN_UNIQUE_CASE(T, C) return compact<T, C>(sorted, volume, marks, sums, tiles, out, count_out, stream)
  switch (k.codec) {
    case CODEC_UNSIGNED:
      switch (k.bytes) {
        case 1: CPN_UNIQUE_CASE(uint8_t, CODEC_UNSIGNED);
        case 2: CPN_UNIQUE_CASE(uint16_t, CODEC_UNSIGNED);
        case 4: CPN_UNIQUE_CASE(uint32_t, CODEC_UNSIGNED);
        case 8: CPN_UNIQUE_CASE(uint64_t, CODEC_UNSIGNED);
      }
      break;
    case CODEC_SIGNED:
      // equality of signed keys is equality of their bits
      switch (k.bytes) {
        case 1: CPN_UNIQUE_CASE(uint8_t, CODEC_UNSIGNED);
        case 2: CPN_UNIQUE_CASE(uint16_t, CODEC_UNSIGNED);
        case 4: CPN_UNIQUE_CASE(uint32_t, CODEC_UNSIGNED);
        case 8: CPN_UNIQUE_CASE(uint64_t, CODEC_UNSIGNED);
      }
      break;
    case CODEC_FLOAT:
      switch (k.bytes) {
        case 2: CPN_UNIQUE_CASE(uint16_t, CODEC_FLOAT);
        case 4: CPN_UNIQUE_CASE(uint32_t, CODEC_FLOAT);
        case 8: CPN_UNIQUE_CASE(uint64_t, CODEC_FLOAT);
      }
      break;
    case CODEC_COMPLEX:
      switch (k.bytes) {
        case 8: CPN_UNIQUE_CASE(uint64_t, CODEC_COMPLEX);
        case 16: CPN_UNIQUE_CASE(U128, CODEC_COMPLEX);
      }
      break;
  }
#undef CPN_UNIQUE_CASE
  return CPN_ERR_DTYPE;
}

}  // namespace cpn

extern "C" uint64_t cpn_unique_temp_bytes(int dtype, uint64_t volume)
{
  const cpn::KeyKind k = cpn::key_kind(dtype);
  if (k.bytes == 0 || k.codec < 0) {
    return 0;
  }
  if (volume == 0) {
    return cpn::HEADER_BYTES;
  }
  const cpn::UniqueLayout L = cpn::unique_layout(dtype, volume, false);
  return L.sort_bytes == 0 ? 0 : L.total;
}

extern "C" int cpn_unique(int dtype, const void* values_in, void* values_out, uint64_t volume, uint64_t* count_out,
                          void* temp, uint64_t temp_bytes, void* stream)
{
  using namespace cpn;
  const KeyKind k = key_kind(dtype);
  if (k.bytes == 0 || k.codec < 0) {
    return CPN_ERR_DTYPE;
  }
  if (count_out == nullptr) {
    return CPN_ERR_NULL;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (volume == 0) {
    // *count_out = 0 through the fill kernel (the word may be captured into a graph)
    if ((reinterpret_cast<uintptr_t>(count_out) % 8) != 0) {
      return CPN_ERR_ALIGN;
    }
    hipLaunchKernelGGL(unique_scan_kernel, dim3(1), dim3(HEADS_BLOCK), 0, s, static_cast<const uint16_t*>(nullptr), uint64_t{0},
                       static_cast<uint64_t*>(nullptr), count_out);
    CPN_HIP_TRY(hipGetLastError());
    return CPN_OK;
  }
  if (values_in == nullptr || values_out == nullptr) {
    return CPN_ERR_NULL;
  }
  UniqueLayout L = unique_layout(dtype, volume, false);
  if (L.sort_bytes == 0) {
    return CPN_ERR_UNSUPPORTED;
  }
  if (temp_bytes < L.total) {
    L = unique_layout(dtype, volume, true);
  }
  if (temp == nullptr || temp_bytes < L.total || (reinterpret_cast<uintptr_t>(temp) % WORKSPACE_ALIGN) != 0) {
    return CPN_ERR_TEMP;
  }
  if ((reinterpret_cast<uintptr_t>(count_out) % 8) != 0) {
    return CPN_ERR_ALIGN;
  }
  unsigned char* ws = static_cast<unsigned char*>(temp);
  void* sorted      = ws + L.off_sorted;
  uint64_t* sums    = reinterpret_cast<uint64_t*>(ws + L.off_counts);
  uint64_t* marks   = reinterpret_cast<uint64_t*>(ws + L.off_marks);
  int rc = cpn_local_sort(dtype, values_in, sorted, nullptr, volume, volume, 0, 1, ws, L.sort_bytes, stream);
  if (rc != CPN_OK) {
    return rc;
  }
  return compact_keys(k, sorted, volume, marks, sums, L.tiles, values_out, count_out, s);
}

extern "C" uint64_t cpn_unique_sorted_temp_bytes(int dtype, uint64_t volume)
{
  using namespace cpn;
  const KeyKind k = key_kind(dtype);
  if (k.bytes == 0 || k.codec < 0 || volume == 0) {
    return 0;
  }
  const uint64_t tiles = (volume + UNIQUE_TILE - 1) / UNIQUE_TILE;
  return sums_bytes(tiles) + marks_bytes(tiles);
}

extern "C" int cpn_unique_sorted(int dtype, const void* sorted, void* values_out, uint64_t volume, uint64_t* count_out,
                                 void* temp, uint64_t temp_bytes, void* stream)
{
  using namespace cpn;
  const KeyKind k = key_kind(dtype);
  if (k.bytes == 0 || k.codec < 0) {
    return CPN_ERR_DTYPE;
  }
  if (volume == 0) {
    return CPN_ERR_UNSUPPORTED;  // (cpn_unique has an answer)
  }
  if (sorted == nullptr || values_out == nullptr || count_out == nullptr) {
    return CPN_ERR_NULL;
  }
  const uint64_t tiles = (volume + UNIQUE_TILE - 1) / UNIQUE_TILE;
  if (temp == nullptr || temp_bytes < sums_bytes(tiles) + marks_bytes(tiles) ||
      (reinterpret_cast<uintptr_t>(temp) % WORKSPACE_ALIGN) != 0) {
    return CPN_ERR_TEMP;
  }
  const uintptr_t mask = static_cast<uintptr_t>(k.bytes - 1);
  if ((reinterpret_cast<uintptr_t>(sorted) & mask) != 0 || (reinterpret_cast<uintptr_t>(values_out) & mask) != 0 ||
      (reinterpret_cast<uintptr_t>(count_out) % 8) != 0) {
    return CPN_ERR_ALIGN;
  }
  unsigned char* ws = static_cast<unsigned char*>(temp);
  return compact_keys(k, sorted, volume, reinterpret_cast<uint64_t*>(ws + sums_bytes(tiles)), reinterpret_cast<uint64_t*>(ws), tiles,
                      values_out, count_out, static_cast<hipStream_t>(stream));
}
