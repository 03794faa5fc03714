// Plane kernels: real fields from a sphere (pw_plane.h).
#include "pw_plane.h"

namespace pw {
template PlaneKernel<double> plane_kernel<double, MODE_REAL, false>(int, int);
}  // namespace pw
