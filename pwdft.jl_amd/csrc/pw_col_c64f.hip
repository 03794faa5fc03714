// Column kernels: FP64 columns any sphere (pw_col.h).
#include "pw_col.h"

namespace pw {
template ColKernel<double> col_kernel<double, false>(int, bool, int*, size_t*);
}  // namespace pw
