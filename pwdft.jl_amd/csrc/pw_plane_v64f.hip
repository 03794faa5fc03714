// Plane kernels: FP64 local-potential planes, any sphere (pw_plane.h).
#include "pw_plane.h"

namespace pw {
template PlaneKernel<double> plane_kernel<double, MODE_VLOC, false>(int, int);
}  // namespace pw
