// Host side of split_sort.h: one call sorts the row of a request that split_plan (split_plan.h) accepts.
#pragma once

#include "split_plan.h"

namespace cpn {

// `head`: see split_done.  For a sample: whether what it is sampled with has been gathered, and where the splitters go.
template <typename KeyT, int CODEC, bool HAS_IDX>
inline int sort_row_split(const SortRequest& r, const SplitPlan& p, const uint32_t* head, bool sampled = false,
                          const SplitPicks<KeyT>* picks = nullptr);

// The launches ahead of a wide row's tiles, and these.
template <typename KeyT, int CODEC, bool HAS_IDX, int BITS>
inline int split_wide_tiles(const SortRequest& r, const SplitPlan& p, const SplitLayout& L)
{
  uint8_t* const ws      = static_cast<uint8_t*>(r.temp);
  const uint32_t n       = static_cast<uint32_t>(r.seg);
  const uint32_t samples = p.buckets * p.per_bucket;
  KeyT* sample           = reinterpret_cast<KeyT*>(ws + L.off_sample);
  KeyT* images           = reinterpret_cast<KeyT*>(ws + L.off_images);
  uint32_t* at           = reinterpret_cast<uint32_t*>(ws + L.off_at);
  float* values          = reinterpret_cast<float*>(ws + L.off_values);
  uint16_t* before       = reinterpret_cast<uint16_t*>(ws + L.off_before);
  SplitBins* bins        = reinterpret_cast<SplitBins*>(ws + L.off_bins);
  uint32_t* head         = static_cast<uint32_t*>(r.temp);
  const SplitPlan inner  = split_plan(sizeof(KeyT), sizeof(KeyT), samples, samples, true);
  const int count        = narrow_passes(CODEC, r.seg);
  uint32_t* passes       = count != 0 ? head : nullptr;
  SplitLeft<KeyT> left{nullptr, static_cast<KeyT*>(r.values_out), r.indices_out, r.index_offset};
  if (count == 0) {
    ProfileScope prof("split_gather", r.stream);
    hipLaunchKernelGGL((split_gather_kernel<KeyT>), dim3(samples / 256), dim3(256), 0, r.stream,
                       static_cast<const KeyT*>(r.values_in), n, samples, sample, static_cast<const uint32_t*>(nullptr));
    CPN_HIP_TRY(hipGetLastError());
  } else {
    const int first     = CODEC == CODEC_FLOAT ? static_cast<int>(sizeof(KeyT)) - count : 0;
    const KeyT launched = static_cast<KeyT>(((KeyT{1} << (8 * count)) - 1) << (8 * first));
    {
      ProfileScope prof("split_front", r.stream);
      hipLaunchKernelGGL((split_front_kernel<KeyT, CODEC>), dim3(samples / 256), dim3(256), 0, r.stream,
                         static_cast<const KeyT*>(r.values_in), n, samples, sample, inner.gathered ? inner.buckets * inner.per_bucket : 0u,
                         reinterpret_cast<KeyT*>(ws + L.off_inner + split_layout(inner, sizeof(KeyT), samples, true).off_sample),
                         reinterpret_cast<uint4*>(ws),
                         static_cast<uint32_t>((L.off_desc + count * narrow_desc_bytes(r.seg)) / 16), static_cast<KeyT>(~launched));
    }
    CPN_HIP_TRY(hipGetLastError());
    NarrowBuffers b{};
    b.head       = ws;
    b.narrow     = head + HEADER_NARROW / 4;
    b.wide       = reinterpret_cast<const uint4*>(ws + HEADER_WIDE);
    b.hist       = reinterpret_cast<uint32_t*>(ws + L.off_hist);
    b.desc       = ws + L.off_desc;
    b.key1       = ws + L.off_key1;
    b.key2       = ws + L.off_key2;
    b.idx1       = HAS_IDX ? reinterpret_cast<uint32_t*>(ws + L.off_idx1) : nullptr;
    const int rc = sort_narrow64(CODEC, r, b, first, count);
    if (rc != CPN_OK) {
      return rc;
    }
    left.sorted = r.values_out == r.values_in ? static_cast<const KeyT*>(b.key2) : nullptr;
  }
  {
    SortRequest c  = r;
    c.values_in    = sample;
    c.values_out   = nullptr;
    c.indices_out  = nullptr;
    c.volume       = samples;
    c.seg          = samples;
    c.index_offset = 0;
    c.temp         = ws + L.off_inner;
    const SplitPicks<KeyT> picks{images, at, values, static_cast<uint32_t>(__builtin_ctz(p.per_bucket)), samples, n};
    const int rc = sort_row_split<KeyT, CODEC, true>(c, inner, passes, count != 0, &picks);
    if (rc != CPN_OK) {
      return rc;
    }
  }
  {
    ProfileScope prof("split_table", r.stream);
    hipLaunchKernelGGL((split_table_kernel<BITS>), dim3(1), dim3(SPLIT_BLOCK), 0, r.stream, values, before, bins,
                       static_cast<const uint32_t*>(passes), head);
  }
  CPN_HIP_TRY(hipGetLastError());
  {
    ProfileScope prof("split_tiles", r.stream);
    hipLaunchKernelGGL((split_wide_tile_kernel<KeyT, CODEC, HAS_IDX, BITS>), dim3(p.tiles), dim3(SPLIT_BLOCK), 0, r.stream,
                       static_cast<const KeyT*>(r.values_in), n, p.tile_len, images, at, before, bins,
                       reinterpret_cast<KeyT*>(ws + L.off_keys), HAS_IDX ? reinterpret_cast<uint16_t*>(ws + L.off_places) : nullptr,
                       reinterpret_cast<uint16_t*>(ws + L.off_starts), static_cast<const uint32_t*>(passes), left);
  }
  CPN_HIP_TRY(hipGetLastError());
  return CPN_OK;
}

template <typename KeyT, int CODEC, bool HAS_IDX>
inline int sort_row_split(const SortRequest& r, const SplitPlan& p, const uint32_t* head, bool sampled, const SplitPicks<KeyT>* picks)
{
  // (float keys that tie need not be the same bits, but a bucket's keys stay in the order of the row on both ways, so
  // nothing but a request for positions needs their places)
  const SplitLayout L = split_layout(p, sizeof(KeyT), r.seg, HAS_IDX);
  uint8_t* const ws   = static_cast<uint8_t*>(r.temp);
  KeyT* grouped       = reinterpret_cast<KeyT*>(ws + L.off_keys);
  uint16_t* places    = HAS_IDX ? reinterpret_cast<uint16_t*>(ws + L.off_places) : nullptr;
  uint16_t* starts    = reinterpret_cast<uint16_t*>(ws + L.off_starts);
  const uint32_t n    = static_cast<uint32_t>(r.seg);
  KeyT* sample        = nullptr;
  if (p.wide) {
    int rc = CPN_ERR_UNSUPPORTED;
    if constexpr (sizeof(KeyT) == 8) {  // (split_max_row)
      switch (p.buckets) {
        case 1024: rc = split_wide_tiles<KeyT, CODEC, HAS_IDX, 10>(r, p, L); break;
        case 2048: rc = split_wide_tiles<KeyT, CODEC, HAS_IDX, 11>(r, p, L); break;
        case 4096: rc = split_wide_tiles<KeyT, CODEC, HAS_IDX, 12>(r, p, L); break;
      }
    }
    if (rc != CPN_OK) {
      return rc;
    }
    head = narrow_passes(CODEC, r.seg) != 0 ? static_cast<const uint32_t*>(r.temp) : nullptr;
  }
  if (p.gathered) {
    sample = reinterpret_cast<KeyT*>(ws + L.off_sample);
  }
  if (p.gathered && !sampled) {
    const uint32_t samples = p.buckets * p.per_bucket;
    ProfileScope prof("split_gather", r.stream);
    hipLaunchKernelGGL((split_gather_kernel<KeyT>), dim3(samples / 256), dim3(256), 0, r.stream,
                       static_cast<const KeyT*>(r.values_in), n, samples, sample, head);
    CPN_HIP_TRY(hipGetLastError());
  }
  if (!p.wide) {
    ProfileScope prof("split_tiles", r.stream);
    const dim3 grid(p.tiles);
    auto launch = [&](auto per_thread, auto per_bucket) {
      hipLaunchKernelGGL((split_tile_kernel<KeyT, CODEC, HAS_IDX, decltype(per_thread)::value, decltype(per_bucket)::value, SPLIT_TILE_ITEMS>),
                         grid, dim3(SPLIT_BLOCK), 0, r.stream, static_cast<const KeyT*>(r.values_in), n, p.tile_len,
                         sample, grouped, places, starts, static_cast<uint32_t*>(r.temp), head);
    };
    using C1 = std::integral_constant<int, 1>;
    using C8 = std::integral_constant<int, 8>;
    switch (p.buckets) {
      case 128: launch(C1{}, C8{}); break;
      case 256:
        if (p.per_bucket == 4) {
          launch(C1{}, std::integral_constant<int, 4>{});
        } else {
          launch(std::integral_constant<int, 2>{}, C8{});
        }
        break;
      case 512: launch(std::integral_constant<int, 4>{}, C8{}); break;
      case 1024: launch(C8{}, C8{}); break;
      default: return CPN_ERR_UNSUPPORTED;
    }
  }
  CPN_HIP_TRY(hipGetLastError());
  {
    SplitBuckets<KeyT> sb{};
    sb.grouped  = grouped;
    sb.places   = places;
    sb.starts   = starts;
    sb.ids      = reinterpret_cast<uint32_t*>(ws + L.off_ids);
    sb.n        = n;
    sb.tiles    = p.tiles;
    sb.tile_len = p.tile_len;
    sb.buckets  = p.buckets;
    sb.head     = head;
    ProfileScope prof("split_buckets", r.stream);
    auto launch = [&](auto wide, auto pick) {
      hipLaunchKernelGGL((split_bucket_kernel<KeyT, CODEC, HAS_IDX, decltype(wide)::value, decltype(pick)::value>), dim3(p.buckets),
                         dim3(SPLIT_BUCKET_BLOCK), 0, r.stream, sb, static_cast<KeyT*>(r.values_out), r.indices_out, r.index_offset,
                         picks != nullptr ? *picks : SplitPicks<KeyT>{});
    };
    bool launched = false;
    if constexpr (sizeof(KeyT) == 8) {
      if (p.wide) {
        launch(std::true_type{}, std::false_type{});
        launched = true;
      }
      if constexpr (HAS_IDX) {
        if (picks != nullptr) {
          launch(std::false_type{}, std::true_type{});
          launched = true;
        }
      }
    }
    if (!launched) {
      launch(std::false_type{}, std::false_type{});
    }
  }
  CPN_HIP_TRY(hipGetLastError());
  return CPN_OK;
}

template <typename KeyT>
inline int sort_split(int codec, const SortRequest& r, const SplitPlan& p)
{
  const bool idx = r.indices_out != nullptr;
  switch (codec) {
    case CODEC_UNSIGNED:
      return idx ? sort_row_split<KeyT, CODEC_UNSIGNED, true>(r, p, nullptr) : sort_row_split<KeyT, CODEC_UNSIGNED, false>(r, p, nullptr);
    case CODEC_SIGNED:
      return idx ? sort_row_split<KeyT, CODEC_SIGNED, true>(r, p, nullptr) : sort_row_split<KeyT, CODEC_SIGNED, false>(r, p, nullptr);
    case CODEC_FLOAT:
      return idx ? sort_row_split<KeyT, CODEC_FLOAT, true>(r, p, nullptr) : sort_row_split<KeyT, CODEC_FLOAT, false>(r, p, nullptr);
    default: return CPN_ERR_DTYPE;
  }
}

}  // namespace cpn
