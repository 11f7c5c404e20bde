// searchsorted: for every value, the leftmost ('left') or rightmost ('right') position at
// which it can be inserted into a sorted 1-D array without breaking the order.
//
// Replaces SearchSortedTask's GPU variant (src/cupynumeric/sort/searchsorted.cu:27-116: one
// thread per value, cub::LowerBound / cub::UpperBound over the sorted array, the position
// folded into the output with a MIN / MAX reduction because the sorted array may be split
// over several processors; on one GPU the bound itself is the answer).  Comparisons use the
// ordered keys of key_codec.h, i.e. the order the sort kernels produce (NaN last and equal to
// itself, -0.0 == +0.0, complex by NumPy's rule), where the reference compares with `<`.
//
// A probe of the sorted array is a dependent load, so the first eleven steps of every search
// run over a table of up to 2048 evenly spaced elements that each workgroup stages in LDS;
// the remaining steps stay inside one stride of the array.
//
// Every remaining probe of an unordered value is a sector of its own from HBM.  When the
// array is too large for the caches and there are many values, the values are therefore
// sorted first (with their positions, by the library's own sort, in the caller's workspace):
// neighbouring lanes then search for neighbouring values, their probes fall into the same
// cache lines, and the array is read about once instead of once per probe.  The answers go
// back to the positions the values came from.  Where the values are dense in the array the sorted
// values are served in tiles: the part of the array between the answers of two tiles' first
// values goes to LDS in one coalesced read, and the search runs there.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sort_driver.h"

namespace cpn {

constexpr int SEARCH_BLOCK  = 256;
constexpr int SEARCH_PIVOTS = 2048;
__device__ constexpr uint32_t search_pivot_at(uint32_t j) { return j + (j >> 6); }
// Up to so many values in an array of n every lane has one (searchsorted_few_kernel); past it the table that each workgroup loads
// first costs more than the lanes give.  us per call of `searchsorted`, sixteen values per lane / one:
//   float32 in 8192   2048 values 18 / 11  250 000  30 / 11  700 000  27 / 11  1 600 000  30 / 18  3 10^6  35 / 30  2^22  40 / 41
//        in 16 384    2^19            12   700 000  30 / 16  786 432  30 / 17  1 048 576  31 / 22  1 572 864  34 / 30  2^21  35 / 39
//        in 65 536    2048        22 / 11  250 000  38 / 18  700 000  37 / 36  786 432    37 / 39  900 000  38 / 45
//        in 2^18                           700 000  44 / 43  786 432    44 / 47
//        in 2^20      2048        27 / 11  250 000  61 / 23  700 000  65 / 48  786 432    66 / 54  900 000  66 / 62  2^20  66 / 71
//        in 4 10^6                         600 000  83 / 65  700 000  85 / 72  786 432    86 / 79  900 000  91 / 90
//        in 3 10^7                         600 000 112 / 107 700 000 122 / 124 786 432   126 / 137
//        in 2^28                           2^19    149 / 149 600 000 168 / 175 786 432   188 / 223
//   float64 in 16 384                      600 000  33 / 19  786 432  34 / 22  1 310 720  37 / 34  1 572 864  37 / 39
//        in 65 536                         600 000  41 / 33  786 432  42 / 41  900 000    42 / 47
//        in 2^20      2048        31 / 11  250 000  79 / 26  786 432  80 / 61  2^20       83 / 81  1 310 720  99 / 100
//        in 3 10^7                         600 000 127 / 119 786 432 146 / 148 900 000   160 / 167
constexpr uint64_t search_few(uint64_t n) { return n <= 16384 ? 3ull << 19 : (n <= (1ull << 24) ? 11ull << 16 : 1ull << 19); }

constexpr uint32_t WINDOW_BYTES    = 40960;
constexpr uint32_t WINDOW_TILE_MAX = 1024;
constexpr uint64_t WINDOW_WIDE_MAX = 1ull << 26;  // 8-byte keys of an array with the lower limit of values per tile
constexpr int BOUNDS_BLOCK         = 256;

template <int NW>
__device__ __forceinline__ bool words_less(const uint64_t (&a)[NW], const uint64_t (&b)[NW])
{
  bool lt = false, eq = true;  // most significant word last in the array
#pragma unroll
  for (int n = NW - 1; n >= 0; --n) {
    lt = lt || (eq && a[n] < b[n]);
    eq = eq && (a[n] == b[n]);
  }
  return lt;
}

// true when the search has to continue to the right of an element with key `a`
template <bool LEFT, int NW>
__device__ __forceinline__ bool go_right(const uint64_t (&a)[NW], const uint64_t (&v)[NW])
{
  return LEFT ? words_less<NW>(a, v) : !words_less<NW>(v, a);
}

template <typename KeyT, int CODEC, bool LEFT>
__global__ __launch_bounds__(SEARCH_BLOCK) void searchsorted_kernel(const KeyT* __restrict__ sorted,
                                                                    uint64_t n,
                                                                    const KeyT* __restrict__ values,
                                                                    uint64_t num_values,
                                                                    int64_t* __restrict__ out,
                                                                    const int64_t* __restrict__ origin,
                                                                    uint64_t step,
                                                                    uint32_t num_pivots)
{
  using KT         = KeyTraits<CODEC, KeyT>;
  constexpr int NW = KT::NWORDS;
  __shared__ uint64_t s_pivot[NW][SEARCH_PIVOTS];

  // pivot j is element j*step of the sorted array (num_pivots == 0: table not used)
  for (uint32_t j = threadIdx.x; j < num_pivots; j += SEARCH_BLOCK) {
    uint64_t w[NW];
    KT::words(sorted[static_cast<uint64_t>(j) * step], w);
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      s_pivot[k][j] = w[k];
    }
  }
  __syncthreads();

  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * SEARCH_BLOCK;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * SEARCH_BLOCK + threadIdx.x; i < num_values; i += stride) {
    uint64_t v[NW];
    KT::words(values[i], v);
    uint64_t lo = 0, hi = n;
    if (num_pivots != 0) {
      // first pivot at which the search would not continue to the right
      uint32_t pl = 0, ph = num_pivots;
      while (pl < ph) {
        const uint32_t pm = (pl + ph) / 2;
        uint64_t a[NW];
#pragma unroll
        for (int k = 0; k < NW; ++k) {
          a[k] = s_pivot[k][pm];
        }
        if (go_right<LEFT, NW>(a, v)) {
          pl = pm + 1;
        } else {
          ph = pm;
        }
      }
      // elements up to pivot pl-1 are to the left of the answer, pivot pl is not
      lo = (pl == 0) ? 0 : static_cast<uint64_t>(pl - 1) * step + 1;
      hi = (pl == num_pivots) ? n : static_cast<uint64_t>(pl) * step;
    }
    while (lo < hi) {
      const uint64_t mid = lo + (hi - lo) / 2;
      uint64_t a[NW];
      KT::words(sorted[mid], a);
      if (go_right<LEFT, NW>(a, v)) {
        lo = mid + 1;
      } else {
        hi = mid;
      }
    }
    // `origin` (values sorted beforehand): the position the value had in the caller's array
    out[origin != nullptr ? static_cast<uint64_t>(origin[i]) : i] = static_cast<int64_t>(lo);
  }
}

// The same for real keys and fewer values than the chip has lanes: a lane has one, where the kernel above gives sixteen to each
// of a few workgroups.  Bound by the chain of dependent loads.  A gap after every 64 elements in LDS keeps elements a power
// of two apart out of one bank, and what fills the table up saves the test of the bound.
template <typename KeyT, int CODEC, bool LEFT>
__global__ __launch_bounds__(SEARCH_BLOCK) void searchsorted_few_kernel(const KeyT* __restrict__ sorted, uint64_t n,
                                                                        const KeyT* __restrict__ values, uint64_t num_values,
                                                                        int64_t* __restrict__ out, const int64_t* __restrict__ origin,
                                                                        uint64_t step, uint32_t num_pivots)
{
  constexpr int EACH = SEARCH_PIVOTS / SEARCH_BLOCK;
  __shared__ KeyT s_pivot[search_pivot_at(SEARCH_PIVOTS)];
  const uint32_t tid = threadIdx.x;
  const uint64_t i   = static_cast<uint64_t>(blockIdx.x) * SEARCH_BLOCK + tid;
  const KeyT v       = ordered_bits<CODEC, KeyT>(values[i < num_values ? i : num_values - 1]);
  KeyT pivot[EACH];
#pragma unroll
  for (int k = 0; k < EACH; ++k) {
    const uint32_t j = k * SEARCH_BLOCK + tid;
    pivot[k]         = sorted[j < num_pivots ? j * step : 0];  // (the last pivot is element (num_pivots - 1) * step < n)
  }
#pragma unroll
  for (int k = 0; k < EACH; ++k) {
    const uint32_t j            = k * SEARCH_BLOCK + tid;
    s_pivot[search_pivot_at(j)] = j < num_pivots ? ordered_bits<CODEC, KeyT>(pivot[k]) : static_cast<KeyT>(~KeyT{0});
  }
  __syncthreads();
  // (`at` counts gaps as well until the last step: it is a multiple of 2 * half, so that they add up)
  uint32_t at = 0;
#pragma unroll
  for (uint32_t half = SEARCH_PIVOTS / 2; half != 0; half >>= 1) {
    const KeyT a = s_pivot[at + search_pivot_at(half - 1)];
    at += (LEFT ? a < v : a <= v) ? search_pivot_at(half) : 0u;
  }
  const KeyT last   = s_pivot[at];
  const uint32_t on = at - at / 65 + ((LEFT ? last < v : last <= v) ? 1u : 0u);
  const uint32_t c  = on < num_pivots ? on : num_pivots;  // (the largest key of all is not left of what fills the table up)
  uint64_t lo       = c == 0 ? 0 : static_cast<uint64_t>(c - 1) * step + 1;
  uint64_t hi       = c == num_pivots ? n : c * step;
  while (lo < hi) {
    const uint64_t mid = lo + (hi - lo) / 2;
    const KeyT a       = ordered_bits<CODEC, KeyT>(sorted[mid]);
    if (LEFT ? a < v : a <= v) {
      lo = mid + 1;
    } else {
      hi = mid;
    }
  }
  if (i < num_values) {
    out[origin != nullptr ? static_cast<uint64_t>(origin[i]) : i] = static_cast<int64_t>(lo);
  }
}

// bounds[b] = answer for the first value of tile b (values sorted, `tile` of them per tile); bounds[tiles] = answer for
// the last value.  Few searches, each a chain of dependent loads: evenly spaced elements in LDS take the first eleven.
template <typename KeyT, int CODEC, bool LEFT>
__global__ __launch_bounds__(BOUNDS_BLOCK) void window_bounds_kernel(const KeyT* __restrict__ sorted,
                                                                     uint64_t n,
                                                                     const KeyT* __restrict__ values,
                                                                     uint64_t num_values,
                                                                     uint32_t tile,
                                                                     uint64_t tiles,
                                                                     uint64_t* __restrict__ bounds)
{
  __shared__ KeyT s_pivot[SEARCH_PIVOTS];
  const uint64_t step = (n + SEARCH_PIVOTS - 1) / SEARCH_PIVOTS;
  constexpr int EACH  = SEARCH_PIVOTS / BOUNDS_BLOCK;
  KeyT pivot[EACH];
#pragma unroll
  for (int k = 0; k < EACH; ++k) {
    const uint64_t i = (k * BOUNDS_BLOCK + threadIdx.x) * step;
    pivot[k]         = sorted[i < n ? i : n - 1];
  }
  const uint64_t b = static_cast<uint64_t>(blockIdx.x) * BOUNDS_BLOCK + threadIdx.x;
  const uint64_t j = b < tiles ? b * tile : num_values - 1;
  const KeyT v     = ordered_bits<CODEC, KeyT>(values[j]);
#pragma unroll
  for (int k = 0; k < EACH; ++k) {
    s_pivot[k * BOUNDS_BLOCK + threadIdx.x] = ordered_bits<CODEC, KeyT>(pivot[k]);
  }
  __syncthreads();
  if (b > tiles) {
    return;
  }
  const uint32_t pivots = static_cast<uint32_t>((n + step - 1) / step);
  uint32_t right        = 0;  // pivots left of the answer
  for (uint32_t at = SEARCH_PIVOTS; at != 0; at >>= 1) {
    if (right + at <= pivots) {
      const KeyT a = s_pivot[right + at - 1];
      if (LEFT ? a < v : a <= v) {
        right += at;
      }
    }
  }
  uint64_t lo = right == 0 ? 0 : (right - 1) * step + 1;
  uint64_t hi = right == pivots ? n : right * step;
  while (lo < hi) {
    const uint64_t mid = lo + (hi - lo) / 2;
    const KeyT a       = ordered_bits<CODEC, KeyT>(sorted[mid]);
    if (LEFT ? a < v : a <= v) {
      lo = mid + 1;
    } else {
      hi = mid;
    }
  }
  bounds[b] = lo;
}

// One tile of sorted values per workgroup.  The answers of the tile lie in [bounds[b], bounds[b + 1]]; if that
// window of the array fits, its ordered keys go to LDS and the search runs there, else (values
// sparse in this part of the array) it runs in the array.
//
// Bound by the read of the array, once, and by the 8-byte stores at the values' own positions.
// 40 KB of window let four workgroups share a CU, so that one searches while others load; the
// loads of the whole window, 16 bytes each, are issued together.  Two values per lane search side by side,
// with a step count that is the same for all lanes.  2^24 float32 values in 2^28: 504 us + 25 us for the
// windows' bounds, against 837 us for probes of the array by lanes with neighbouring values.
// The stores stay ordinary ones: with non-temporal stores, which the L2 does not gather, the whole call
// took 1395 us instead of 891.
template <typename KeyT, int CODEC, bool LEFT>
__global__ __launch_bounds__(SEARCH_BLOCK) void searchsorted_window_kernel(const KeyT* __restrict__ sorted,
                                                                           uint64_t n,
                                                                           const KeyT* __restrict__ values,
                                                                           uint64_t num_values,
                                                                           int64_t* __restrict__ out,
                                                                           const int64_t* __restrict__ origin,
                                                                           uint32_t tile,
                                                                           const uint64_t* __restrict__ bounds)
{
  constexpr uint32_t CAPACITY = WINDOW_BYTES / sizeof(KeyT);
  constexpr uint32_t PACK     = 16 / sizeof(KeyT);
  constexpr int PACKS         = WINDOW_BYTES / 16 / SEARCH_BLOCK;  // per lane
  struct alignas(16) Pack {
    KeyT key[PACK];
  };
  static_assert(PACKS * 16 * SEARCH_BLOCK == WINDOW_BYTES, "one batch of loads covers the window");
  __shared__ Pack s_pack[CAPACITY / PACK];
  KeyT* s_key = s_pack[0].key;
  const uint64_t from   = bounds[blockIdx.x];
  const uint64_t extent = bounds[blockIdx.x + 1] - from;
  const uint64_t first  = static_cast<uint64_t>(blockIdx.x) * tile;
  const uint32_t count  = static_cast<uint32_t>(num_values - first < tile ? num_values - first : tile);
  // elements between the 16-byte boundary below the window and the window
  const uint32_t head = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(sorted + from) % 16 / sizeof(KeyT));
  if constexpr (sizeof(KeyT) <= 2) {
    const uint64_t to = from + extent;
    if (to <= from) {  // one answer for all, most often a value that ends or misses a run
      for (uint32_t t = threadIdx.x; t < count; t += SEARCH_BLOCK) {
        out[origin[first + t]] = static_cast<int64_t>(from);
      }
      return;
    }
    // An array this long has runs of 512 equal elements and more, and a window is mostly the run that the tile's first
    // value begins.  A value that equals the first one of this tile or of the next has that bound for an answer: if
    // there is no other, nothing of the array is read.  2^22 float16 values in 2^29: 162 us a call, 244 when the
    // window is searched all the same, 219 by probes of the array.  (Any lane?  The flag lies in the window's LDS: with
    // more of it per workgroup only three workgroups share a CU.)
    const KeyT v_from   = ordered_bits<CODEC, KeyT>(values[first]);
    const KeyT v_to     = ordered_bits<CODEC, KeyT>(values[first + tile < num_values ? first + tile : num_values - 1]);
    uint32_t* s_between = reinterpret_cast<uint32_t*>(s_pack);
    bool between        = false;
    for (uint32_t t = threadIdx.x; t < count; t += SEARCH_BLOCK) {
      const KeyT v = ordered_bits<CODEC, KeyT>(values[first + t]);
      between      = between || (v != v_from && v != v_to);
    }
    if (threadIdx.x == 0) {
      *s_between = 0;
    }
    __syncthreads();
    if (__builtin_amdgcn_ballot_w64(between) != 0 && threadIdx.x % WAVE == 0) {
      *s_between = 1;
    }
    __syncthreads();
    const bool search = *s_between != 0;
    __syncthreads();
    if (!search) {
      for (uint32_t t = threadIdx.x; t < count; t += SEARCH_BLOCK) {
        const KeyT v           = ordered_bits<CODEC, KeyT>(values[first + t]);
        out[origin[first + t]] = static_cast<int64_t>(v == v_from ? from : to);
      }
      return;
    }
  }
  // Room for whole packs at both ends.  An array that is not sorted can have bounds that fall: that
  // extent wraps to a large one and the search in the array ends at once.
  if (extent > CAPACITY - 2 * PACK) {  // the same for every lane of the workgroup
    for (uint32_t t = threadIdx.x; t < count; t += SEARCH_BLOCK) {
      uint64_t v[1];
      KeyTraits<CODEC, KeyT>::words(values[first + t], v);
      uint64_t lo = from, hi = from + extent;
      while (lo < hi) {
        const uint64_t mid = lo + (hi - lo) / 2;
        uint64_t a[1];
        KeyTraits<CODEC, KeyT>::words(sorted[mid], a);
        if (go_right<LEFT, 1>(a, v)) {
          lo = mid + 1;
        } else {
          hi = mid;
        }
      }
      out[origin[first + t]] = static_cast<int64_t>(lo);
    }
    return;
  }
  const uint32_t width = static_cast<uint32_t>(extent);
  const uint32_t packs = (head + width + PACK - 1) / PACK;
  uint32_t skip        = 0;  // elements in LDS before the window
  if (width != 0 && from >= head && from - head + static_cast<uint64_t>(packs) * PACK <= n) {
    // whole packs inside the array
    const Pack* __restrict__ source = reinterpret_cast<const Pack*>(sorted + (from - head));
    Pack p[PACKS];
    skip = head;
#pragma unroll
    for (int k = 0; k < PACKS; ++k) {
      const uint32_t j = k * SEARCH_BLOCK + threadIdx.x;
      p[k]             = source[j < packs ? j : packs - 1];
    }
#pragma unroll
    for (int k = 0; k < PACKS; ++k) {
#pragma unroll
      for (uint32_t e = 0; e < PACK; ++e) {
        p[k].key[e] = ordered_bits<CODEC, KeyT>(p[k].key[e]);
      }
      // (past the window: copies of its last pack; a store under a condition would pull its load along)
      s_pack[k * SEARCH_BLOCK + threadIdx.x] = p[k];
    }
  } else {  // the first or last window of an array that does not begin or end on a 16-byte boundary
    for (uint32_t j = threadIdx.x; j < width; j += SEARCH_BLOCK) {
      s_key[j] = ordered_bits<CODEC, KeyT>(sorted[from + j]);
    }
  }
  __syncthreads();
  const uint32_t largest_step = (width != 0) ? 1u << (31 - __builtin_clz(width)) : 0u;
  for (uint32_t start = 0; start < count; start += 2 * SEARCH_BLOCK) {
    KeyT v[2];
    uint32_t pos[2] = {0, 0};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t t = start + k * SEARCH_BLOCK + threadIdx.x;
      v[k]             = ordered_bits<CODEC, KeyT>(values[first + (t < count ? t : count - 1)]);
    }
    for (uint32_t step = largest_step; step != 0; step >>= 1) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const uint32_t to = pos[k] + step;  // every element before `to` is left of the answer?
        if (to <= width) {
          const KeyT a = s_key[skip + to - 1];
          if (LEFT ? a < v[k] : a <= v[k]) {
            pos[k] = to;
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t t = start + k * SEARCH_BLOCK + threadIdx.x;
      if (t < count) {
        out[origin[first + t]] = static_cast<int64_t>(from + pos[k]);
      }
    }
  }
}

// Values per tile of the window search for `key_bytes`-byte keys, 0 where it does not pay.  A window is
// planned to fill four fifths of its LDS, which leaves room for values that are not spread
// evenly.  Below 128 values per tile a value has more than 256 bytes of the array to itself, and reading
// all of it costs more than the cache lines that the probes of a value touch.  8-byte keys of an array past the 512 MiB
// need 256 values per tile: us per call by windows / by probes at 256 bytes per value, values spread as the
// array / half of them in a thousandth of it:
//   float64   512 MiB  387 / 446   390 / 407     1 GiB  582 / 603   577 / 552     4 GiB  2359 / 2375   2296 / 2160
//   float32   512 MiB  267 / 331   279 / 297     1 GiB  430 / 481   445 / 422     4 GiB  1744 / 1799   1545 / 1509
static uint32_t window_tile(int key_bytes, uint64_t n, uint64_t num_values)
{
  const double per_value = static_cast<double>(n) * key_bytes / static_cast<double>(num_values);
  const double fits      = 0.8 * WINDOW_BYTES / per_value;
  if (fits >= WINDOW_TILE_MAX) {
    return WINDOW_TILE_MAX;
  }
  const uint32_t least = key_bytes == 8 && n > WINDOW_WIDE_MAX ? 256 : 128;
  const uint32_t tile  = static_cast<uint32_t>(fits) / 128 * 128;
  return tile >= least ? tile : 0;
}

template <typename KeyT, int CODEC>
static int launch_window_search(const void* sorted, uint64_t n, const void* values, uint64_t num_values, bool left,
                                int64_t* out, const int64_t* origin, uint32_t tile, uint64_t* bounds,
                                hipStream_t stream)
{
  const uint64_t tiles = (num_values + tile - 1) / tile;
  const auto bounds_of = left ? &window_bounds_kernel<KeyT, CODEC, true> : &window_bounds_kernel<KeyT, CODEC, false>;
  const auto search =
    left ? &searchsorted_window_kernel<KeyT, CODEC, true> : &searchsorted_window_kernel<KeyT, CODEC, false>;
  {
    ProfileScope prof("window_bounds", stream);
    hipLaunchKernelGGL(bounds_of, dim3(static_cast<uint32_t>(tiles / BOUNDS_BLOCK + 1)), dim3(BOUNDS_BLOCK), 0, stream,
                       static_cast<const KeyT*>(sorted), n, static_cast<const KeyT*>(values), num_values, tile, tiles, bounds);
  }
  CPN_HIP_TRY(hipGetLastError());
  {
    ProfileScope prof("searchsorted", stream);
    hipLaunchKernelGGL(search, dim3(static_cast<uint32_t>(tiles)), dim3(SEARCH_BLOCK), 0, stream,
                       static_cast<const KeyT*>(sorted), n, static_cast<const KeyT*>(values), num_values, out, origin,
                       tile, bounds);
  }
  CPN_HIP_TRY(hipGetLastError());
  return CPN_OK;
}

template <typename KeyT, int CODEC>
static int launch_searchsorted(const void* sorted, uint64_t n, const void* values, uint64_t num_values, bool left,
                               int64_t* out, const int64_t* origin, uint64_t* bounds, hipStream_t stream)
{
  if constexpr (CODEC != CODEC_COMPLEX) {
    const uint32_t tile = window_tile(static_cast<int>(sizeof(KeyT)), n, num_values);
    if (bounds != nullptr && num_values / tile < (1ull << 31) - 1) {
      return launch_window_search<KeyT, CODEC>(sorted, n, values, num_values, left, out, origin, tile, bounds, stream);
    }
  }
  uint64_t step       = 0;
  uint32_t num_pivots = 0;
  if (n >= 8192 && num_values >= 2048) {
    step       = (n + SEARCH_PIVOTS - 1) / SEARCH_PIVOTS;
    num_pivots = static_cast<uint32_t>((n + step - 1) / step);
  }
  if constexpr (CODEC != CODEC_COMPLEX) {
    if (num_pivots != 0 && num_values <= search_few(n)) {
      const auto search = left ? &searchsorted_few_kernel<KeyT, CODEC, true> : &searchsorted_few_kernel<KeyT, CODEC, false>;
      ProfileScope prof("searchsorted", stream);
      hipLaunchKernelGGL(search, dim3(static_cast<uint32_t>((num_values + SEARCH_BLOCK - 1) / SEARCH_BLOCK)), dim3(SEARCH_BLOCK), 0,
                         stream, static_cast<const KeyT*>(sorted), n, static_cast<const KeyT*>(values), num_values, out, origin, step,
                         num_pivots);
      CPN_HIP_TRY(hipGetLastError());
      return CPN_OK;
    }
  }
  // with a pivot table every workgroup should serve a few thousand values
  const uint64_t per_block = (num_pivots != 0) ? 16 * SEARCH_BLOCK : SEARCH_BLOCK;
  uint64_t grid            = (num_values + per_block - 1) / per_block;
  if (grid > 16384) {
    grid = 16384;
  }
  ProfileScope prof("searchsorted", stream);
  if (left) {
    hipLaunchKernelGGL((searchsorted_kernel<KeyT, CODEC, true>), dim3(static_cast<uint32_t>(grid)), dim3(SEARCH_BLOCK),
                       0, stream, static_cast<const KeyT*>(sorted), n, static_cast<const KeyT*>(values), num_values, out,
                       origin, step, num_pivots);
  } else {
    hipLaunchKernelGGL((searchsorted_kernel<KeyT, CODEC, false>), dim3(static_cast<uint32_t>(grid)),
                       dim3(SEARCH_BLOCK), 0, stream, static_cast<const KeyT*>(sorted), n,
                       static_cast<const KeyT*>(values), num_values, out, origin, step, num_pivots);
  }
  CPN_HIP_TRY(hipGetLastError());
  return CPN_OK;
}

// Sorting the values first pays when the sorted array is far larger than the caches and the
// values are many; otherwise (and whenever the caller brings no workspace) values are searched
// in the order given.
static bool presort_pays(int key_bytes, uint64_t n, uint64_t num_values)
{
  return n * static_cast<uint64_t>(key_bytes) >= (64ull << 20) && num_values >= (1ull << 16);
}

// The windows' bounds lie behind the header of the sort's own workspace, which is done with by then and has room for them
// (a kilobyte of counters per 16384 values): a search by windows asks for no more than one by probes.
struct SearchLayout {
  uint64_t sort_bytes, off_values, off_origin, total;
};

// With `least`, the sort's workspace is what it can do with instead of what it asks for (callers that kept a size).
static SearchLayout search_layout(KeyKind k, uint64_t num_values, bool least)
{
  SearchLayout L{};
  L.sort_bytes = workspace_bytes(k.bytes, key_passes(k.bytes, k.codec), k.codec, num_values, num_values, true, true, false, least);
  L.off_values = align_up(L.sort_bytes, WORKSPACE_ALIGN);
  L.off_origin = L.off_values + align_up(num_values * static_cast<uint64_t>(k.bytes), WORKSPACE_ALIGN);
  L.total      = L.off_origin + align_up(num_values * 8, WORKSPACE_ALIGN);
  return L;
}

}  // namespace cpn

extern "C" uint64_t cpn_searchsorted_temp_bytes(int dtype, uint64_t n, uint64_t num_values)
{
  const cpn::KeyKind k = cpn::key_kind(dtype);
  if (k.bytes == 0 || k.codec < 0 || !cpn::presort_pays(k.bytes, n, num_values)) {
    return 0;
  }
  const cpn::SearchLayout L = cpn::search_layout(k, num_values, false);
  return L.sort_bytes == 0 ? 0 : L.total;
}

extern "C" int cpn_searchsorted(int dtype, const void* sorted, uint64_t n, const void* values, uint64_t num_values,
                                int left, int64_t* positions_out, void* temp, uint64_t temp_bytes, void* stream)
{
  using namespace cpn;
  const KeyKind k = key_kind(dtype);
  if (k.bytes == 0 || k.codec < 0) {
    return CPN_ERR_DTYPE;
  }
  if (num_values == 0) {
    return CPN_OK;
  }
  if (values == nullptr || positions_out == nullptr || (n != 0 && sorted == nullptr)) {
    return CPN_ERR_NULL;
  }
  const uint64_t align = static_cast<uint64_t>(k.bytes);
  if ((reinterpret_cast<uintptr_t>(sorted) % align) != 0 || (reinterpret_cast<uintptr_t>(values) % align) != 0 ||
      (reinterpret_cast<uintptr_t>(positions_out) % 8) != 0) {
    return CPN_ERR_ALIGN;
  }
  const int64_t* origin = nullptr;
  uint64_t* bounds      = nullptr;
  if (temp != nullptr && presort_pays(k.bytes, n, num_values)) {
    SearchLayout L = search_layout(k, num_values, false);
    if (temp_bytes < L.total) {
      L = search_layout(k, num_values, true);
    }
    if (L.sort_bytes != 0 && temp_bytes >= L.total) {
      if ((reinterpret_cast<uintptr_t>(temp) % WORKSPACE_ALIGN) != 0) {
        return CPN_ERR_TEMP;
      }
      unsigned char* ws = static_cast<unsigned char*>(temp);
      void* sorted_vals = ws + L.off_values;
      int64_t* where    = reinterpret_cast<int64_t*>(ws + L.off_origin);
      const int rc = cpn_local_sort(dtype, values, sorted_vals, where, num_values, num_values, 0, 1, ws, L.sort_bytes,
                                    stream);
      if (rc != CPN_OK) {
        return rc;
      }
      values = sorted_vals;
      origin = where;
      if (const uint32_t tile = window_tile(k.bytes, n, num_values);
          tile != 0 && L.sort_bytes >= HEADER_BYTES + ((num_values + tile - 1) / tile + 1) * 8) {
        bounds = reinterpret_cast<uint64_t*>(ws + HEADER_BYTES);
      }
    }
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool l  = left != 0;
#define CPN_SEARCH_CASE(T, C) \
  return launch_searchsorted<T, C>(sorted, n, values, num_values, l, positions_out, origin, bounds, s)
  switch (k.codec) {
    case CODEC_UNSIGNED:
      switch (k.bytes) {
        case 1: CPN_SEARCH_CASE(uint8_t, CODEC_UNSIGNED);
        case 2: CPN_SEARCH_CASE(uint16_t, CODEC_UNSIGNED);
        case 4: CPN_SEARCH_CASE(uint32_t, CODEC_UNSIGNED);
        case 8: CPN_SEARCH_CASE(uint64_t, CODEC_UNSIGNED);
      }
      break;
    case CODEC_SIGNED:
      switch (k.bytes) {
        case 1: CPN_SEARCH_CASE(uint8_t, CODEC_SIGNED);
        case 2: CPN_SEARCH_CASE(uint16_t, CODEC_SIGNED);
        case 4: CPN_SEARCH_CASE(uint32_t, CODEC_SIGNED);
        case 8: CPN_SEARCH_CASE(uint64_t, CODEC_SIGNED);
      }
      break;
    case CODEC_FLOAT:
      switch (k.bytes) {
        case 2: CPN_SEARCH_CASE(uint16_t, CODEC_FLOAT);
        case 4: CPN_SEARCH_CASE(uint32_t, CODEC_FLOAT);
        case 8: CPN_SEARCH_CASE(uint64_t, CODEC_FLOAT);
      }
      break;
    case CODEC_COMPLEX:
      switch (k.bytes) {
        case 8: CPN_SEARCH_CASE(uint64_t, CODEC_COMPLEX);
        case 16: CPN_SEARCH_CASE(U128, CODEC_COMPLEX);
      }
      break;
  }
#undef CPN_SEARCH_CASE
  return CPN_ERR_DTYPE;
}
