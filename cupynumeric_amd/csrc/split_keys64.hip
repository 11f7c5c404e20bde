// Instantiates the split of long rows for 64-bit keys (a translation unit of its own, as the sort kernels have per key width).
#include "split_driver.h"

namespace cpn {

int sort_split64(int codec, const SortRequest& r, const SplitPlan& plan) { return sort_split<uint64_t>(codec, r, plan); }

}  // namespace cpn
