// Column kernels: FP64 columns half spheres (pw_col.h).
#include "pw_col.h"

namespace pw {
template ColKernel<double> col_kernel<double, true>(int, bool, int*, size_t*);
}  // namespace pw
