// Instantiates the sort kernels for 64-bit keys (one translation unit per key width so
// that the hipcc runs proceed in parallel; the reference splits its instantiations per
// dtype for the same reason, src/cupynumeric/sort/cub_sort.h:21-115).
#include "sort_driver.h"

namespace cpn {

int sort_keys64(int codec, const SortRequest& r)
{
  switch (codec) {
    case CODEC_UNSIGNED: return sort_typed<uint64_t, CODEC_UNSIGNED>(r);
    case CODEC_SIGNED: return sort_typed<uint64_t, CODEC_SIGNED>(r);
    case CODEC_FLOAT: return sort_typed<uint64_t, CODEC_FLOAT>(r);
    case CODEC_COMPLEX: return sort_typed<uint64_t, CODEC_COMPLEX>(r);  // complex64
    default: return CPN_ERR_DTYPE;
  }
}

template <int CODEC>
static int narrow(const SortRequest& r, const NarrowBuffers& b, int first, int count)
{
  return r.indices_out != nullptr ? sort_narrow<uint64_t, CODEC, true>(r, b, first, count)
                                  : sort_narrow<uint64_t, CODEC, false>(r, b, first, count);
}

int sort_narrow64(int codec, const SortRequest& r, const NarrowBuffers& b, int first, int count)
{
  switch (codec) {
    case CODEC_UNSIGNED: return narrow<CODEC_UNSIGNED>(r, b, first, count);
    case CODEC_SIGNED: return narrow<CODEC_SIGNED>(r, b, first, count);
    case CODEC_FLOAT: return narrow<CODEC_FLOAT>(r, b, first, count);
    default: return CPN_ERR_DTYPE;
  }
}

}  // namespace cpn
