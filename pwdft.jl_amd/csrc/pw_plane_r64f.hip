// Plane kernels: FP64 density planes, any sphere (pw_plane.h).
#include "pw_plane.h"

namespace pw {
template PlaneKernel<double> plane_kernel<double, MODE_RHO, false>(int, int);
}  // namespace pw
