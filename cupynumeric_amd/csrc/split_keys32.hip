// Instantiates the split of long rows for 32-bit keys (a translation unit of its own, as the sort kernels have per key width).
#include "split_driver.h"

namespace cpn {

int sort_split32(int codec, const SortRequest& r, const SplitPlan& plan) { return sort_split<uint32_t>(codec, r, plan); }

}  // namespace cpn
