// ozk_split_f32.hip -- split kernels with float slices (one translation unit per
// slice dtype, compiled in parallel).
#include "ozk_split_kernels.h"

namespace ozk {

template struct SplitLaunch<float>;

}  // namespace ozk
