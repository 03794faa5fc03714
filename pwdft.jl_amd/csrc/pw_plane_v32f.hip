// Plane kernels: FP32 local-potential planes, any sphere (pw_plane.h).
#include "pw_plane.h"

namespace pw {
template PlaneKernel<float> plane_kernel<float, MODE_VLOC, false>(int, int);
}  // namespace pw
