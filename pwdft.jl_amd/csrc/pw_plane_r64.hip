// Plane kernels: FP64 density planes, half spheres (pw_plane.h).
#include "pw_plane.h"

namespace pw {
template PlaneKernel<double> plane_kernel<double, MODE_RHO, true>(int, int);
}  // namespace pw
