// Plane kernels: FP64 local-potential planes, half spheres (pw_plane.h).
#include "pw_plane.h"

namespace pw {
template PlaneKernel<double> plane_kernel<double, MODE_VLOC, true>(int, int);
}  // namespace pw
