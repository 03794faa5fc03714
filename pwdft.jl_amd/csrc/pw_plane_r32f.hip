// Plane kernels: FP32 density planes, any sphere (pw_plane.h).
#include "pw_plane.h"

namespace pw {
template PlaneKernel<float> plane_kernel<float, MODE_RHO, false>(int, int);
}  // namespace pw
