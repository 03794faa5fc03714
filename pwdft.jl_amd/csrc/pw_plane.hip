// Launches of the plane kernels (pw_plane.h).
#include <algorithm>
#include "pw_plane.h"

namespace pw {

// Lines of Yc a row of length n needs for its exchanges.
static int xch_lines_of(int n) {
  switch (n) {
#define PW_CASE(N_, R0_, R1_, L_) \
  case N_: return xch_lines<N_>();
    PW_LINE_PLANS(PW_CASE)
#undef PW_CASE
    default: return 0;
  }
}
// Wavefronts of the density kernel whose accumulators stay in registers (n1 = n2 = n), 0: the
// accumulators of length n live in global memory.
static int rho_waves_of(int n) {
  switch (n) {
#define PW_CASE(N_, R0_, R1_, L_) \
  case N_: return RhoPlan<N_>::reg ? RhoPlan<N_>::nw : 0;
    PW_LINE_PLANS(PW_CASE)
#undef PW_CASE
    default: return 0;
  }
}

// Fills what every mode shares; returns the LDS bytes, 0 when the plane kernels do not apply.
template <typename T>
static size_t plane_args(const pw_ctx* c, int maxx, PlaneArgs<T>& A) {
  if (c->plane_compressed != 0 || !line_plan_groups(c->n1) || !line_plan_groups(c->n2)) return 0;
  A.n1 = c->n1;
  A.n2 = c->n2;
  A.n3 = c->n3;
  A.N = c->N;
  A.twx = reinterpret_cast<const cplx<T>*>(sizeof(T) == 8 ? c->d_tw64[0] : c->d_tw32[0]);
  A.twy = reinterpret_cast<const cplx<T>*>(sizeof(T) == 8 ? c->d_tw64[1] : c->d_tw32[1]);
  A.lines = std::max(maxx, xch_lines_of(c->n1));
  const size_t lds = ((size_t)(A.lines + 1) * odd_stride(c->n2) + c->n1 + c->n2) * sizeof(cplx<T>) + (size_t)c->n1 * sizeof(int);
  return lds <= 160 * 1024 ? lds : 0;
}

// Wavefronts per workgroup.  A SIMD holds two or three of these register-heavy wavefronts, and
// the hardware deals a workgroup's wavefronts over the SIMDs from the first on, so workgroups
// of 1, 2 or 4 wavefronts pack and 5 or 6 do not (FP64 72^2, 160 bands: 338 us with 4, 353 with
// 2, 474 with 5).  A plane that leaves room for no second workgroup takes 8 (FP64 108^2).
static int plane_waves(const pw_ctx* c, size_t lds) {
  const int G = line_plan_groups(c->n1), rounds = (c->n2 + G - 1) / G;
  if (2 * lds > 160 * 1024) return 8;
  return rounds <= 1 ? 1 : rounds <= 4 ? 2 : 4;
}

template <typename T>
static PlaneKernel<T> vloc_kernel(const pw_ctx* c, bool half) {
  return half ? plane_kernel<T, MODE_VLOC, true>(c->n1, c->n2) : plane_kernel<T, MODE_VLOC, false>(c->n1, c->n2);
}

template <typename T>
bool plane_applies(const pw_ctx* c, int maxx) {
  PlaneArgs<T> A{};
  return plane_args<T>(c, maxx, A) != 0;
}
template bool plane_applies<double>(const pw_ctx*, int);
template bool plane_applies<float>(const pw_ctx*, int);

template <typename T>
void plane_vloc(pw_ctx* c, const KData& k, cplx<T>* W, const T* V, int nb) {
  PlaneArgs<T> A{};
  const size_t lds = plane_args<T>(c, k.nxact, A);
  const PlaneKernel<T> kern = lds ? vloc_kernel<T>(c, k.half) : nullptr;
  if (!kern) return;
  A.W = W;
  A.V = V;
  A.ctab = k.d_ctab;
  A.apos = k.d_apos;
  A.ncol = k.ncol;
  A.nxact = k.nxact;
  hipLaunchKernelGGL(kern, dim3(c->n3, nb), dim3(64 * plane_waves(c, lds)), lds, c->stream, A);
}

template <typename T>
void plane_vloc_batch(pw_ctx* c, const KBatch* dkb, int nk, int nb, int maxx, bool half, cplx<T>* W, const T* V) {
  PlaneArgs<T> A{};
  const size_t lds = plane_args<T>(c, maxx, A);
  const PlaneKernel<T> kern = lds ? vloc_kernel<T>(c, half) : nullptr;
  if (!kern) return;
  A.W = W;
  A.V = V;
  A.kb = dkb;
  A.nbk = nb;
  hipLaunchKernelGGL(kern, dim3(c->n3, nk * nb), dim3(64 * plane_waves(c, lds)), lds, c->stream, A);
}

template <typename T>
static int rho_waves(const pw_ctx* c, size_t lds) {
  const int reg = c->n1 == c->n2 ? rho_waves_of(c->n1) : 0;
  return reg ? reg : plane_waves(c, lds);
}

template <typename T>
int plane_rho_resident(const pw_ctx* c, int maxx) {
  PlaneArgs<T> A{};
  const size_t lds = plane_args<T>(c, maxx, A);
  if (!lds) return 1;
  // by LDS, and by registers about 12 wavefronts
  return std::max(1, std::min((int)(160 * 1024 / lds), 12 / rho_waves<T>(c, lds)));
}

template <typename T>
static void rho_launch(pw_ctx* c, PlaneArgs<T>& A, int maxx, bool half, cplx<T>* W, int nb, int bpg, int ngroup,
                       const double* d_w, double* rpart) {
  const size_t lds = plane_args<T>(c, maxx, A);
  if (!lds) return;
  const PlaneKernel<T> kern =
      half ? plane_kernel<T, MODE_RHO, true>(c->n1, c->n2) : plane_kernel<T, MODE_RHO, false>(c->n1, c->n2);
  if (!kern) return;
  A.W = W;
  A.nb = nb;
  A.bpg = bpg;
  A.wts = d_w;
  A.out = rpart;
  hipLaunchKernelGGL(kern, dim3(c->n3, ngroup), dim3(64 * rho_waves<T>(c, lds)), lds, c->stream, A);
}

template <typename T>
void plane_rho(pw_ctx* c, const KData& k, cplx<T>* W, int nb, int bpg, int ngroup, const double* d_w, double* rpart) {
  PlaneArgs<T> A{};
  A.ctab = k.d_ctab;
  A.apos = k.d_apos;
  A.ncol = k.ncol;
  A.nxact = k.nxact;
  rho_launch<T>(c, A, k.nxact, k.half, W, nb, bpg, ngroup, d_w, rpart);
}

template <typename T>
void plane_rho_batch(pw_ctx* c, const KBatch* dkb, int nbk, int nb, int maxx, bool half, cplx<T>* W, int bpg,
                     int ngroup, const double* d_w, double* rpart) {
  PlaneArgs<T> A{};
  A.kb = dkb;
  A.nbk = nbk;
  rho_launch<T>(c, A, maxx, half, W, nb, bpg, ngroup, d_w, rpart);
}

void plane_real(pw_ctx* c, const KData& k, cplx<double>* W, int nf, double* out, double scale, int acc) {
  PlaneArgs<double> A{};
  const size_t lds = plane_args<double>(c, k.nxact, A);
  const PlaneKernel<double> kern = lds ? plane_kernel<double, MODE_REAL, false>(c->n1, c->n2) : nullptr;
  if (!kern) return;
  A.W = W;
  A.ctab = k.d_ctab;
  A.apos = k.d_apos;
  A.ncol = k.ncol;
  A.nxact = k.nxact;
  A.out = out;
  A.scale = scale;
  A.acc = acc;
  hipLaunchKernelGGL(kern, dim3(c->n3, nf), dim3(64 * plane_waves(c, lds)), lds, c->stream, A);
}

template void plane_vloc<double>(pw_ctx*, const KData&, cplx<double>*, const double*, int);
template void plane_vloc<float>(pw_ctx*, const KData&, cplx<float>*, const float*, int);
template void plane_vloc_batch<double>(pw_ctx*, const KBatch*, int, int, int, bool, cplx<double>*, const double*);
template void plane_vloc_batch<float>(pw_ctx*, const KBatch*, int, int, int, bool, cplx<float>*, const float*);
template void plane_rho<double>(pw_ctx*, const KData&, cplx<double>*, int, int, int, const double*, double*);
template void plane_rho<float>(pw_ctx*, const KData&, cplx<float>*, int, int, int, const double*, double*);
template void plane_rho_batch<double>(pw_ctx*, const KBatch*, int, int, int, bool, cplx<double>*, int, int, const double*,
                                      double*);
template void plane_rho_batch<float>(pw_ctx*, const KBatch*, int, int, int, bool, cplx<float>*, int, int, const double*,
                                     double*);
template int plane_rho_resident<double>(const pw_ctx*, int);
template int plane_rho_resident<float>(const pw_ctx*, int);

}  // namespace pw
