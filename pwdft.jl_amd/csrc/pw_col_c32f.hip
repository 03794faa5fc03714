// Column kernels: FP32 columns any sphere (pw_col.h).
#include "pw_col.h"

namespace pw {
template ColKernel<float> col_kernel<float, false>(int, bool, int*, size_t*);
}  // namespace pw
