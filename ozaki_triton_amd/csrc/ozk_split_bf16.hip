// ozk_split_bf16.hip -- split kernels with __bf16 slices (one translation unit per
// slice dtype, compiled in parallel).
#include "ozk_split_kernels.h"

namespace ozk {

template struct SplitLaunch<__bf16>;

}  // namespace ozk
