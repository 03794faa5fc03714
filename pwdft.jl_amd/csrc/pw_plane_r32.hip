// Plane kernels: FP32 density planes, half spheres (pw_plane.h).
#include "pw_plane.h"

namespace pw {
template PlaneKernel<float> plane_kernel<float, MODE_RHO, true>(int, int);
}  // namespace pw
