// ozk_split_i8.hip -- split kernels with int8_t slices (one translation unit per
// slice dtype, compiled in parallel).
#include "ozk_split_kernels.h"

namespace ozk {

template struct SplitLaunch<int8_t>;

}  // namespace ozk
