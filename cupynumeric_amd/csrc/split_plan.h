// Which requests are split by sampled keys (split_sort.h), into what, and in which workspace.
#pragma once

#include "sort_driver.h"
#include "split_sort.h"

namespace cpn {

// Single rows split once by sampled keys (split_sort.h), real keys of 4 and 8 bytes.  buckets == 0: another way.
// (cpn_set_merge_rows: in the default mode only, and with the row kernels in use.)
struct SplitPlan {
  uint32_t buckets;     // a power of two
  uint32_t per_bucket;  // sampled keys
  uint32_t tiles, tile_len;
  bool gathered;        // the sample, by a launch of its own
  bool wide;            // the sample is sorted ahead, as a row of its own
};
// Where the lines lie (us per call, before / this way; normal float keys, sort and argsort):
//   from where one workgroup has more than 6144 8-byte or 8192 4-byte keys to sort (until 8 or 16 keys per thread, about 12
//   us, two launches cost as much): float64 6144 16, 19 / 15, 15, 8192 26, 21 / 15, 15, int64 6144 13, 15 / 14, 14, 8192 19, 18
//   / 14, 14, float32 8192 15, 19 / 13, 14, 9000 22, 21 / 14, 14, int32 8192 12, 16 / 13, 13, 9000 19, 18 / 13, 13.  Rows of few values
//   cost passes over the sample and in the buckets, where one workgroup skips the bytes that all keys share: of a hundred values 9000 float32 19, 22
//   / 19, 18, float64 34, 32 / 20, 20, int32 13, 13 / 17, 17, int64 14, 14 / 19, 19; of two 27, 25 / 20, 20, 29, 28 / 23, 23, 13,
//   13 / 20, 20, 15, 14 / 21, 21; of one 13 / 16 to 18
//   in between: 40 000 float32 29, 30 / 14, 15, float64 33, 34 / 16, 16; 100 000 41, 46 / 16, 17 and 53, 48 / 18, 18;
//   262 144 68, 75 / 23, 26 and 125, 115 / 26, 27; 524 288 65, 71 / 31, 34 and 152, 146 / 35, 37
//   to where 8192 sampled keys, which every tile's workgroup sorts, take half of its time: 10^6 float32 76, 86 / 48, 52,
//   float64 193, 176 / 54, 57, int64 148, 172 / 50, 52
constexpr uint64_t SPLIT_WIDE_ROW = SPLIT_MAX_TILES * SPLIT_BLOCK * SPLIT_TILE_ITEMS + 1;
constexpr uint64_t split_max_row(int key_bytes) { return key_bytes == 8 ? 4096 * 2560 : SPLIT_WIDE_ROW - 1; }
constexpr uint64_t split_min_row(int key_bytes) { return key_bytes == 8 ? 6145 : 8193; }
inline SplitPlan split_plan(int key_bytes, int passes, uint64_t volume, uint64_t seg, bool want_indices)
{
  SplitPlan p{};
  if (!merge_rows_default() || (key_bytes != 4 && key_bytes != 8) || passes != key_bytes || seg < split_min_row(key_bytes) ||
      seg > split_max_row(key_bytes) || volume != seg || lds_row_limit(key_bytes, want_indices) != lds_row_capacity(key_bytes, want_indices)) {
    return p;
  }
  if (seg >= SPLIT_WIDE_ROW) {
    // A bucket of 2560 keys at most (and room for 4096): the fuller, the more of them sampled, or rows with a bucket that does not
    // fit, which its workgroup sorts alone in about 0.2 ms, are no longer rare.  128 of 2560: none of 400 rows (simulated), 96 one,
    // 64 one in 15 (and 7 us of 225 less, 10^7 int64 ids); 64 of 2048: none, 32 one in 60 (7 us of 200 less); 16 of 1365: none.
    // Longer rows would need more buckets than a tile has room to count: of 12 10^6 keys, with 4096 buckets and 128 sampled
    // keys each, one row in 12 has such a bucket.  Tiles in whole rounds of the compute units.
    p.wide         = true;
    p.buckets      = seg <= (1ull << 21) ? 1024 : (seg <= (1ull << 22) ? 2048 : 4096);
    p.per_bucket   = seg <= p.buckets * 1365ull ? 16 : (seg <= p.buckets * 2048ull ? 64 : 128);
    uint64_t tiles = (seg + SPLIT_BLOCK * SPLIT_WIDE_ITEMS - 1) / (SPLIT_BLOCK * SPLIT_WIDE_ITEMS);
    tiles          = align_up(tiles, 256);
    p.tile_len     = static_cast<uint32_t>((seg + tiles - 1) / tiles);
    p.tiles        = static_cast<uint32_t>((seg + p.tile_len - 1) / p.tile_len);
    return p;
  }
  // A bucket of 1024 keys at most, eight of them sampled, or of 512, four of them sampled (and room for 4096).  A tile of as
  // few keys as leaves no compute unit without one.
  p.buckets      = seg <= 65536 ? 128 : (seg <= 262144 ? 256 : (seg <= 524288 ? 512 : 1024));
  p.per_bucket   = p.buckets == 256 && seg <= 131072 ? 4 : 8;
  p.gathered     = p.buckets * p.per_bucket >= 4096;
  uint64_t tiles = (seg + SPLIT_BLOCK - 1) / SPLIT_BLOCK;
  tiles          = tiles > SPLIT_MAX_TILES ? SPLIT_MAX_TILES : tiles;
  p.tile_len     = static_cast<uint32_t>((seg + tiles - 1) / tiles);
  p.tiles        = static_cast<uint32_t>((seg + p.tile_len - 1) / p.tile_len);
  return p;
}
static_assert(SPLIT_WIDE_FLAGS == WIDE_FLAGS && HEADER_WIDE + 4 * WIDE_FLAGS <= HEADER_TICKETS, "the flags have a place in the header");
// Byte passes that a wide row tries ahead of the split: the lowest of whole numbers, the highest of floats (signs, exponents and the
// leading bits of fractions; whole numbers that go below zero have busy upper bytes and do not try).  A row of which only those
// bytes vary is sorted by one read that counts and a pass for each byte that does; the split, which does not skip constant
// bytes, takes up to four times as long.  us a sort and an argsort, split / passes:
//   int64 of equal keys    2^22 122, 125 / 47, 45    10^7 223, 231 / 76, 66     below 200  114, 117 / 61, 67    207, 217 / 101, 117
//   below 20 000                119, 124 / 84, 93         232, 244 / 153, 180   below 300 000  131, 147 / 107, 119   244, 255 / 205, 258
//   float64 of two values       137, 141 / 92, 92         232, 241 / 168, 178
// Every other row pays for launches that find nothing to do: full int64 keys 2^21 + 1 83, 88 / 90, 96; 2^22 109, 118 / 117, 125;
// 10^7 217, 238 / 224, 243.  Up to 2^21 whole numbers a third pass wins nothing (2^21 below 300 000, three bytes: 78, 86 split, 91, 97
// in passes), nor do passes over floats (of two values 84, 85 / 81, 80; of three bytes, below 200: 2^23 195, 202 / 187, 202).
inline int narrow_passes(int codec, uint64_t n)
{
  if (codec == CODEC_FLOAT) {
    return n > (1ull << 21) ? 2 : 0;
  }
  return n > (1ull << 21) ? 3 : 2;
}
// Workspace: header, the sample, the keys in the order of the buckets of each tile, their places, the table, two words
// per key.  Wide: also the splitters (images, places, values), their table of bins, and the workspace of the sample's own sort.
struct SplitLayout {
  uint64_t off_hist, off_desc;                        // wide: the passes' histograms and descriptors,
  uint64_t off_key1, off_key2, off_idx1;              // and what they work on, where the split's own regions are
  uint64_t off_sample, off_images, off_at, off_values, off_before, off_bins, off_inner;
  uint64_t off_keys, off_places, off_starts, off_ids, total;
};
inline SplitLayout split_layout(const SplitPlan& p, int key_bytes, uint64_t n, bool want_indices)
{
  const uint64_t table = static_cast<uint64_t>(p.tiles) * (p.buckets + 1) * sizeof(uint16_t);
  SplitLayout L{};
  const uint64_t samples = static_cast<uint64_t>(p.buckets) * p.per_bucket;
  L.off_sample = HEADER_BYTES;
  if (p.wide) {
    L.off_hist   = HEADER_BYTES;
    L.off_desc   = L.off_hist + 8 * RADIX * sizeof(uint32_t);
    L.off_sample = L.off_desc + 3 * narrow_desc_bytes(n);
  }
  L.off_keys   = L.off_sample + (p.gathered || p.wide ? align_up(samples * key_bytes, WORKSPACE_ALIGN) : 0);
  if (p.wide) {
    L.off_images  = L.off_keys;
    L.off_at      = L.off_images + align_up(static_cast<uint64_t>(p.buckets) * key_bytes, WORKSPACE_ALIGN);
    L.off_values  = L.off_at + align_up(p.buckets * sizeof(uint32_t), WORKSPACE_ALIGN);
    L.off_before  = L.off_values + align_up(p.buckets * sizeof(float), WORKSPACE_ALIGN);
    L.off_bins    = L.off_before + align_up(p.buckets * SPLIT_WIDE_BINS * sizeof(uint16_t), WORKSPACE_ALIGN);
    L.off_inner   = L.off_bins + WORKSPACE_ALIGN;
    L.off_keys    = L.off_inner + split_layout(split_plan(key_bytes, key_bytes, samples, samples, true), key_bytes, samples, true).total;
  }
  L.off_places = L.off_keys + align_up(n * key_bytes, WORKSPACE_ALIGN);
  L.off_starts = L.off_places + (want_indices ? align_up(n * sizeof(uint16_t), WORKSPACE_ALIGN) : 0);
  L.off_ids    = L.off_starts + align_up(table, WORKSPACE_ALIGN);
  L.total      = L.off_ids + align_up(2 * n * sizeof(uint32_t), WORKSPACE_ALIGN);
  if (p.wide) {  // (the sample outlives the passes)
    L.off_key1         = L.off_images;
    L.off_key2         = L.off_key1 + align_up(n * key_bytes, WORKSPACE_ALIGN);
    L.off_idx1         = L.off_key2 + align_up(n * key_bytes, WORKSPACE_ALIGN);
    const uint64_t end = L.off_idx1 + (want_indices ? align_up(n * sizeof(uint32_t), WORKSPACE_ALIGN) : 0);
    L.total            = L.total > end ? L.total : end;
  }
  return L;
}

// (split_keys32.hip, split_keys64.hip: requests that split_plan accepts, with a workspace of split_layout)
int sort_split32(int codec, const SortRequest& r, const SplitPlan& plan);
int sort_split64(int codec, const SortRequest& r, const SplitPlan& plan);

}  // namespace cpn
