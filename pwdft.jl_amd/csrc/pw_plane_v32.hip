// Plane kernels: FP32 local-potential planes, half spheres (pw_plane.h).
#include "pw_plane.h"

namespace pw {
template PlaneKernel<float> plane_kernel<float, MODE_VLOC, true>(int, int);
}  // namespace pw
