// ozk_split_f16.hip -- split kernels with _Float16 slices (one translation unit per
// slice dtype, compiled in parallel).
#include "ozk_split_kernels.h"

namespace ozk {

template struct SplitLaunch<_Float16>;

}  // namespace ozk
