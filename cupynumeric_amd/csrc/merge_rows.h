// Rows too long for the per-row kernels: every row is cut into 2^levels pieces of equal length (the
// last one may be shorter), each sorted by the one-workgroup-per-row kernel (a piece fits the LDS of
// a CU), and neighbouring pieces are merged here, level by level, until the row is one run.
// One read and one write of HBM per element and step, against one pass per key byte, per-row
// histograms and tiles that end at every row on the global path.
//
// Stands, for these rows, where the reference runs cub::DeviceSegmentedRadixSort
// (src/cupynumeric/sort/cub_sort.cuh:81-105,153-182).
//
// The merge is stable: of two keys that tie, the one from the first piece of a pair (the lower
// positions of the row) comes first, and inside a piece the stable row sort has kept input order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "key_codec.h"
#include "radix_common.h"

namespace cpn {

#ifndef CPN_MERGE_ITEMS
#define CPN_MERGE_ITEMS 8
#endif
constexpr int MERGE_ITEMS = CPN_MERGE_ITEMS;
// Threads of a workgroup, which merges MERGE_ITEMS outputs per thread: 512 for keys alone (the
// kernel's time is trips to memory, so large chunks: 2^26 float32 keys in rows of 16 385 0.26 -> 0.23 ms
// against 256), 256 when int64 positions are staged beside the keys (56 KiB of LDS with 512 left two
// workgroups per CU: 0.37 -> 0.44 ms).
__host__ __device__ constexpr int merge_block(bool has_idx) { return has_idx ? 256 : 512; }
__host__ __device__ constexpr int merge_chunk(bool has_idx) { return merge_block(has_idx) * MERGE_ITEMS; }
constexpr int MERGE_CHUNK_MIN = 256 * MERGE_ITEMS;  // the smaller of the two: bounds the grid

// Where a workgroup of the merge starts: blockIdx.x -> row, pair of pieces in the row, chunk of the pair's outputs.
struct MergeChunk {
  uint64_t first;  // of the pair, in keys / idx and in the outputs
  uint32_t len_a, len_b;  // the two pieces (len_b == 0: nothing to merge with)
  uint32_t d0;            // first merged output of the chunk, counted inside the pair
};
__device__ inline MergeChunk merge_chunk_of(
  uint32_t block, uint32_t n, uint32_t piece, uint32_t chunks_per_pair, uint32_t pairs_per_row, uint32_t chunk_len)
{
  uint64_t row;
  uint32_t pair, chunk;
  if (pairs_per_row == 1) {
    row   = block / chunks_per_pair;
    pair  = 0;
    chunk = block - static_cast<uint32_t>(row * chunks_per_pair);
  } else {
    const uint32_t per_row = pairs_per_row * chunks_per_pair;
    row                    = block / per_row;
    const uint32_t rest    = block - static_cast<uint32_t>(row * per_row);
    pair                   = rest / chunks_per_pair;
    chunk                  = rest - pair * chunks_per_pair;
  }
  const uint64_t start = 2ull * pair * piece;  // of this pair in its row; start < n
  const uint32_t left  = n - static_cast<uint32_t>(start);
  MergeChunk c;
  c.first = row * n + start;
  c.len_a = left < piece ? left : piece;
  c.len_b = left - c.len_a < piece ? left - c.len_a : piece;
  c.d0    = chunk * chunk_len;
  return c;
}

// How many of the outputs before a chunk come from the first piece of its pair, for every chunk
// of the merge launch that follows (one thread each): the smallest i with !(a[i] <= b[d0 - 1 - i]).
// Done ahead of the merge because a search inside its workgroups, with one candidate per thread,
// touched a cache line per candidate, four times the lines of the chunk itself.
constexpr int MERGE_SPLIT_BLOCK = 256;
template <typename KeyT, int CODEC>
__global__ __launch_bounds__(MERGE_SPLIT_BLOCK) void merge_split_kernel(const KeyT* __restrict__ keys,
                                                                        uint32_t* __restrict__ splits,
                                                                        uint32_t n,
                                                                        uint32_t piece,
                                                                        uint32_t chunks_per_pair,
                                                                        uint32_t pairs_per_row,
                                                                        uint32_t chunk_len,
                                                                        uint32_t chunks_total)
{
  const uint32_t g = blockIdx.x * MERGE_SPLIT_BLOCK + threadIdx.x;
  if (g >= chunks_total) {
    return;
  }
  const MergeChunk c = merge_chunk_of(g, n, piece, chunks_per_pair, pairs_per_row, chunk_len);
  const uint32_t d   = c.d0 < c.len_a + c.len_b ? c.d0 : c.len_a + c.len_b;  // (chunks past the end of a short pair)
  const KeyT* a      = keys + c.first;
  const KeyT* b      = a + c.len_a;
  uint32_t lo = d > c.len_b ? d - c.len_b : 0u, hi = d < c.len_a ? d : c.len_a;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) / 2;
    if (ordered_bits<CODEC, KeyT>(a[mid]) <= ordered_bits<CODEC, KeyT>(b[d - 1 - mid])) {
      lo = mid + 1;
    } else {
      hi = mid;
    }
  }
  splits[g] = lo;
}

// keys / idx: the rows, [rows][n], every row in sorted pieces of `piece` elements: [0, piece),
// [piece, 2 piece), ... (the last one ends at n).  Pieces 2p and 2p + 1 of a row are merged into
// [2p piece, (2p + 2) piece) of the outputs; a piece without a partner is copied.
// idx holds the final int64 row positions of the elements (they count from the start of the row).
// keys_out may be nullptr (index-only sorts, last level), idx / idx_out are nullptr unless HAS_IDX.
// splits: merge_split_kernel's output for this launch.
// Grid: rows x pairs_per_row x chunks_per_pair workgroups, chunks_per_pair = ceil(2 piece / merge_chunk).
template <typename KeyT, int CODEC, bool HAS_IDX>
__global__ __launch_bounds__(merge_block(HAS_IDX)) void merge_halves_kernel(const KeyT* __restrict__ keys,
                                                                    const int64_t* __restrict__ idx,
                                                                    KeyT* __restrict__ keys_out,
                                                                    int64_t* __restrict__ idx_out,
                                                                    const uint32_t* __restrict__ splits,
                                                                    uint32_t n,
                                                                    uint32_t piece,
                                                                    uint32_t chunks_per_pair,
                                                                    uint32_t pairs_per_row)
{
  constexpr int MERGE_BLOCK = merge_block(HAS_IDX);
  constexpr int MERGE_CHUNK = merge_chunk(HAS_IDX);
  __shared__ KeyT s_key[MERGE_CHUNK];
  __shared__ int64_t s_idx[HAS_IDX ? MERGE_CHUNK : 1];
  __shared__ uint16_t s_src[HAS_IDX ? MERGE_CHUNK : 1];

  const int tid      = threadIdx.x;
  const MergeChunk c = merge_chunk_of(blockIdx.x, n, piece, chunks_per_pair, pairs_per_row, MERGE_CHUNK);
  const uint32_t len_a = c.len_a, len_b = c.len_b, d0 = c.d0;
  const uint32_t h = len_a;  // the second piece starts here
  if (d0 >= len_a + len_b) {
    return;  // (the whole workgroup: the last pair of a row may be short)
  }
  const bool ends      = d0 + MERGE_CHUNK >= len_a + len_b;  // the pair ends in this chunk
  const uint32_t d1    = ends ? len_a + len_b : d0 + MERGE_CHUNK;
  const uint64_t first = c.first;
  const KeyT* a        = keys + first;  // first piece, len_a keys

  auto image = [](KeyT k) { return ordered_bits<CODEC, KeyT>(k); };

  // how many of the outputs before the chunk, and before the next one, come from the first piece
  // (merge_split_kernel; the next chunk of the pair is the next workgroup)
  const uint32_t a0 = splits[blockIdx.x];
  const uint32_t a1 = ends ? len_a : splits[blockIdx.x + 1];
  const uint32_t b0 = d0 - a0, b1 = d1 - a1;
  const uint32_t na = a1 - a0, nb = b1 - b0, total = d1 - d0;

  // this chunk's keys of both halves, side by side in LDS (all loads of a thread first, from
  // positions clamped into the chunk, so that none waits for the one before it)
  {
    KeyT v[MERGE_ITEMS];
    int64_t p[HAS_IDX ? MERGE_ITEMS : 1];
#pragma unroll
    for (int k = 0; k < MERGE_ITEMS; ++k) {
      const uint32_t j   = static_cast<uint32_t>(tid) + k * MERGE_BLOCK;
      const uint32_t jj  = j < total ? j : total - 1;
      const uint32_t src = jj < na ? a0 + jj : h + b0 + (jj - na);
      v[k]               = a[src];
      if constexpr (HAS_IDX) {
        p[k] = idx[first + src];
      }
    }
#pragma unroll
    for (int k = 0; k < MERGE_ITEMS; ++k) {
      const uint32_t j = static_cast<uint32_t>(tid) + k * MERGE_BLOCK;
      if (j < total) {
        s_key[j] = v[k];
        if constexpr (HAS_IDX) {
          s_idx[j] = p[k];
        }
      }
    }
  }
  __syncthreads();

  // every thread merges MERGE_ITEMS consecutive outputs, from its own split of the chunk
  const uint32_t diag = static_cast<uint32_t>(tid) * MERGE_ITEMS < total ? static_cast<uint32_t>(tid) * MERGE_ITEMS : total;
  uint32_t tlo = diag > nb ? diag - nb : 0u, thi = diag < na ? diag : na;
  while (tlo < thi) {
    const uint32_t mid = (tlo + thi) / 2;
    if (image(s_key[mid]) <= image(s_key[na + (diag - 1 - mid)])) {
      tlo = mid + 1;
    } else {
      thi = mid;
    }
  }
  uint32_t ia = tlo, ib = diag - tlo;
  KeyT out_key[MERGE_ITEMS];
  uint32_t out_src[MERGE_ITEMS];
  // the heads of both runs stay in registers; a step reads only the successor of the key it took
  // (positions past the end of a run are clamped: their keys are read and never taken)
  KeyT head_a = s_key[ia < na ? ia : (na != 0 ? na - 1 : 0)];
  KeyT head_b = s_key[nb != 0 ? na + (ib < nb ? ib : nb - 1) : 0];
#pragma unroll
  for (int k = 0; k < MERGE_ITEMS; ++k) {
    out_key[k] = KeyT{};
    out_src[k] = 0;
    if (diag + k < total) {
      const bool take_a = ib >= nb || (ia < na && image(head_a) <= image(head_b));
      out_key[k]        = take_a ? head_a : head_b;
      out_src[k]        = take_a ? ia : na + ib;
      ia += take_a ? 1u : 0u;
      ib += take_a ? 0u : 1u;
      const uint32_t next = take_a ? (ia < na ? ia : ia - 1) : na + (ib < nb ? ib : ib - 1);
      const KeyT v        = s_key[next];
      head_a              = take_a ? v : head_a;
      head_b              = take_a ? head_b : v;
    }
  }
  __syncthreads();  // every thread has read what it needs of s_key
#pragma unroll
  for (int k = 0; k < MERGE_ITEMS; ++k) {
    if (diag + k < total) {
      s_key[diag + k] = out_key[k];
      if constexpr (HAS_IDX) {
        s_src[diag + k] = static_cast<uint16_t>(out_src[k]);
      }
    }
  }
  __syncthreads();
  const uint64_t out_base = first + d0;
#pragma unroll
  for (int k = 0; k < MERGE_ITEMS; ++k) {
    const uint32_t j = static_cast<uint32_t>(tid) + k * MERGE_BLOCK;
    if (j < total) {
      if (keys_out != nullptr) {
        keys_out[out_base + j] = s_key[j];
      }
      if constexpr (HAS_IDX) {
        idx_out[out_base + j] = s_idx[s_src[j]];
      }
    }
  }
}

// ---- short requests: all pieces of a row merged in one launch, by rank ----------------------------
// A key's place in the row is its place in its own piece plus, for every other piece, the number of that piece's
// keys that come before it.  A workgroup takes RANK_CHUNK neighbouring keys of one piece; what lies between the
// first and the last of them in another piece (about as many keys, where the pieces are alike) is copied into LDS
// and searched there by every key of the chunk.  The work grows with the number of pieces, so this is for
// requests that leave most of the chip idle, whose time is the chain of launches: 100 000 float64 keys with
// positions took 48 us for sorting eight pieces and three pairs of launches for merging them level by level, 59 us;
// now 22 us for thirteen pieces and 26 us for this kernel (which waits for memory and LDS in turn: the windows'
// ends, the windows, the searches).
constexpr int RANK_CHUNK      = 256;
constexpr int RANK_MAX_PIECES = 64;
// Keys of other pieces in LDS at a time (more are taken in turns), and how many of them a thread reads at once.
constexpr uint32_t RANK_STAGE = 8192;
constexpr int RANK_LOADS      = 8;
constexpr int RANK_ILP        = 4;  // pieces searched at once by a thread
// When the windows fill RANK_STAGE keys more often than this, those of more than RANK_WIDE keys are searched where they
// lie.  Where pieces are unlike (their values drift, or change halfway), neighbouring keys of one can have most of
// another between them, and a workgroup that copied all of that took as long as there was to copy: 262 144 float32
// keys, 8192 of them spread over the narrow range of the others, 366 us, now 68 (level by level: 88); the second half
// in a thousandth of the range of the first, 242 and 66 (88).  (Fewer keys are copied sooner than searched: a random walk
// of 9000 float64 keys, three pieces, 26 us against 32.)
constexpr uint32_t RANK_MAX_STAGES = 2;
constexpr uint32_t RANK_WIDE       = 4 * RANK_CHUNK;
constexpr int RANK_WIDE_ILP        = 8;  // windows searched at once

// keys / idx: the rows, [rows][n], in sorted pieces of `piece` elements (the last one of a row may be shorter); idx
// holds row positions.  Outputs may not alias them.  Grid: rows x pieces x chunks workgroups of RANK_CHUNK threads.
template <typename KeyT, int CODEC, bool HAS_IDX>
__global__ __launch_bounds__(RANK_CHUNK) void merge_ranks_kernel(const KeyT* __restrict__ keys,
                                                                 const int64_t* __restrict__ idx,
                                                                 KeyT* __restrict__ keys_out,
                                                                 int64_t* __restrict__ idx_out,
                                                                 uint32_t n,
                                                                 uint32_t piece,
                                                                 uint32_t pieces,
                                                                 uint32_t chunks)
{
  static_assert(2 * RANK_MAX_PIECES <= RANK_CHUNK, "a thread per end of a window");
  __shared__ KeyT s_keys[RANK_STAGE];                  // ordered images
  __shared__ uint32_t s_end[2][RANK_MAX_PIECES + RANK_ILP];  // of every piece: keys before the chunk's first / last key
  __shared__ uint32_t s_at[RANK_MAX_PIECES + 1];       // where its window starts, all copied ones one after the other
  __shared__ uint32_t s_wide;                          // is any window searched in memory?
  const uint32_t tid  = threadIdx.x;
  const uint32_t lane = tid % WAVE, wave = tid / WAVE;
  const uint32_t per_row = pieces * chunks;
  const uint64_t row     = blockIdx.x / per_row;
  const uint32_t rest    = blockIdx.x - static_cast<uint32_t>(row * per_row);
  const uint32_t mine    = rest / chunks;
  const uint32_t first   = (rest - mine * chunks) * RANK_CHUNK;  // of the chunk in its piece
  const KeyT* const row_keys = keys + row * n;
  auto length = [&](uint32_t j) { return n - j * piece < piece ? n - j * piece : piece; };
  if (first >= length(mine)) {
    return;  // (the whole workgroup: the last piece may be short)
  }
  const uint32_t count = length(mine) - first < RANK_CHUNK ? length(mine) - first : RANK_CHUNK;
  auto image           = [](KeyT k) { return ordered_bits<CODEC, KeyT>(k); };
  const uint64_t own   = row * n + static_cast<uint64_t>(mine) * piece + first;  // of the chunk
  const KeyT raw       = keys[own + (tid < count ? tid : count - 1)];
  const KeyT key       = image(raw);
  int64_t position     = 0;
  if constexpr (HAS_IDX) {
    position = idx[own + (tid < count ? tid : count - 1)];
  }
  // a key k of piece j comes before x of this chunk when it is smaller, or equal and j is the earlier piece:
  // k < x + (j < mine), where x + 1 may wrap, so as two comparisons
  auto before = [&](KeyT k, KeyT x, uint32_t j) { return k < x || (k == x && j < mine); };

  // ---- the windows: thread 2j + e counts the keys of piece j before the chunk's first (e = 0) or last key ----
  if (tid < 2 * pieces) {
    const uint32_t j = tid / 2;
    const KeyT x     = image(keys[own + ((tid & 1u) ? count - 1 : 0u)]);
    const KeyT* p    = row_keys + static_cast<uint64_t>(j) * piece;
    uint32_t lo = 0, hi = length(j);
    if (j == mine) {
      hi = 0;  // (not searched)
    }
    while (lo < hi) {  // three probes at once: half the dependent reads
      const uint32_t d = (hi - lo) / 4;
      const uint32_t m1 = lo + d, m2 = lo + (hi - lo) / 2, m3 = hi - 1 - d;
      const bool b1 = before(image(p[m1]), x, j), b2 = before(image(p[m2]), x, j), b3 = before(image(p[m3]), x, j);
      // m1 <= m2; m3 may stand before m2 in a short range, where the answers are still those of a sorted array
      uint32_t l = lo, h = hi;
      if (b1) { l = m1 + 1 > l ? m1 + 1 : l; } else { h = m1 < h ? m1 : h; }
      if (b2) { l = m2 + 1 > l ? m2 + 1 : l; } else { h = m2 < h ? m2 : h; }
      if (b3) { l = m3 + 1 > l ? m3 + 1 : l; } else { h = m3 < h ? m3 : h; }
      lo = l;
      hi = h;
    }
    s_end[tid & 1u][j] = lo;
  }
  __syncthreads();
  // window of piece j: keys [s_end[0][j], s_end[1][j]) of it; before a key of the chunk come s_end[0][j] of its keys
  // and some of the window
  uint32_t rank = first + tid;
  if (wave == 0) {
    static_assert(RANK_MAX_PIECES <= WAVE, "a lane per piece");
    const uint32_t window = lane < pieces ? s_end[1][lane] - s_end[0][lane] : 0u;
    const uint32_t sum    = wave_inclusive_sum_dpp(window);
    const uint32_t all    = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(sum), WAVE - 1));
    const bool in_memory  = all > RANK_MAX_STAGES * RANK_STAGE && window > RANK_WIDE;
    const uint32_t copied = in_memory ? 0u : window;
    const uint32_t incl   = wave_inclusive_sum_dpp(copied);
    if (lane < pieces) {
      s_at[lane] = incl - copied;
    }
    if (lane == WAVE - 1) {
      s_at[pieces] = incl;
    }
    const uint64_t wide = __ballot(in_memory);
    if (lane == 0) {
      s_wide = wide != 0 ? 1u : 0u;
    }
  }
  __syncthreads();
  for (uint32_t j = 0; j < pieces; ++j) {
    rank += s_end[0][j];
  }
  const uint32_t total = s_at[pieces];
  for (uint32_t from = 0; from < total; from += RANK_STAGE) {
    const uint32_t to = total - from < RANK_STAGE ? total : from + RANK_STAGE;
    // keys [from, to) of the windows laid end to end, RANK_LOADS of a thread's share in flight
    {
      uint32_t j = 0;
      for (uint32_t i0 = from + tid; i0 < to; i0 += RANK_LOADS * RANK_CHUNK) {
        KeyT k[RANK_LOADS];
#pragma unroll
        for (int l = 0; l < RANK_LOADS; ++l) {
          const uint32_t i = i0 + l * RANK_CHUNK < to ? i0 + l * RANK_CHUNK : to - 1;
          while (s_at[j + 1] <= i) {  // (s_at[pieces] == total > i)
            ++j;
          }
          k[l] = row_keys[static_cast<uint64_t>(j) * piece + s_end[0][j] + (i - s_at[j])];
        }
#pragma unroll
        for (int l = 0; l < RANK_LOADS; ++l) {
          if (i0 + l * RANK_CHUNK < to) {
            s_keys[i0 + l * RANK_CHUNK - from] = image(k[l]);
          }
        }
      }
    }
    __syncthreads();
    for (uint32_t j0 = 0; j0 < pieces; j0 += RANK_ILP) {
      uint32_t base[RANK_ILP], len[RANK_ILP], found[RANK_ILP], most = 0;
#pragma unroll
      for (int k = 0; k < RANK_ILP; ++k) {
        const uint32_t j = j0 + k < pieces ? j0 + k : pieces;
        const uint32_t a = s_at[j] > from ? s_at[j] : from;
        const uint32_t e = s_at[j < pieces ? j + 1 : j];
        const uint32_t b = e < to ? e : to;
        base[k]  = a - from;
        len[k]   = b > a ? b - a : 0u;
        found[k] = 0;
        most     = len[k] > most ? len[k] : most;
      }
      if (most == 0) {
        continue;  // uniform
      }
      for (uint32_t step = 1u << (31 - __builtin_clz(most)); step != 0; step >>= 1) {
#pragma unroll
        for (int k = 0; k < RANK_ILP; ++k) {
          const uint32_t at  = found[k] + step;
          const bool inside  = at <= len[k];
          const KeyT other   = s_keys[inside ? base[k] + at - 1 : 0u];
          const bool earlier = before(other, key, j0 + k);
          found[k]           = (inside && earlier) ? at : found[k];
        }
      }
#pragma unroll
      for (int k = 0; k < RANK_ILP; ++k) {
        rank += found[k];
      }
    }
    __syncthreads();
  }
  if (s_wide != 0) {
    for (uint32_t j0 = 0; j0 < pieces; j0 += RANK_WIDE_ILP) {
      uint32_t at[RANK_WIDE_ILP], len[RANK_WIDE_ILP], found[RANK_WIDE_ILP], most = 0;
#pragma unroll
      for (int k = 0; k < RANK_WIDE_ILP; ++k) {
        const uint32_t j = j0 + k < pieces ? j0 + k : pieces - 1;
        const uint32_t s = s_end[1][j] - s_end[0][j];
        at[k]            = j * piece + s_end[0][j];  // (n < 2^32)
        len[k]           = (j0 + k < pieces && s_at[j + 1] == s_at[j]) ? s : 0u;  // (none of it copied)
        found[k]         = 0;
        most             = len[k] > most ? len[k] : most;
      }
      if (most == 0) {
        continue;  // uniform
      }
      for (uint32_t step = 1u << (31 - __builtin_clz(most)); step != 0; step >>= 1) {
        KeyT other[RANK_WIDE_ILP];
#pragma unroll
        for (int k = 0; k < RANK_WIDE_ILP; ++k) {  // (all loads first; a place inside the row whatever is asked)
          other[k] = row_keys[found[k] + step <= len[k] ? at[k] + found[k] + step - 1 : 0u];
        }
#pragma unroll
        for (int k = 0; k < RANK_WIDE_ILP; ++k) {
          const bool earlier = before(image(other[k]), key, j0 + k);
          found[k]           = (found[k] + step <= len[k] && earlier) ? found[k] + step : found[k];
        }
      }
#pragma unroll
      for (int k = 0; k < RANK_WIDE_ILP; ++k) {
        rank += found[k];
      }
    }
  }
  if (tid < count) {
    if (keys_out != nullptr) {
      keys_out[row * n + rank] = raw;
    }
    if constexpr (HAS_IDX) {
      idx_out[row * n + rank] = position;
    }
  }
}

}  // namespace cpn
