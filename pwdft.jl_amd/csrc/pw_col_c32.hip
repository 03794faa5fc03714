// Column kernels: FP32 columns half spheres (pw_col.h).
#include "pw_col.h"

namespace pw {
template ColKernel<float> col_kernel<float, true>(int, bool, int*, size_t*);
}  // namespace pw
