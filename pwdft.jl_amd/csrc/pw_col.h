// Device code of the column kernels (pw_col.hip, pw_col_*.hip): the z-FFTs of the sphere's
// columns, with the gather of psi before the inverse one and the scatter into Hpsi after the
// forward one.
//
// A workgroup transforms a chunk of C columns of one band in LDS.  The passes of a line's
// two-pass plan hold their butterflies in registers: the inverse one reads psi through the slot
// table (ztab: row of psi at (column, z), or -1) straight into the first butterflies, the forward
// one leaves its last butterflies straight in Hpsi with the kinetic term, so the tile is neither
// cleared nor scattered into nor gathered from.  Only the W side, whose rows are contiguous over
// the columns, goes through the tile, in rows of C.
//
// What bounds it: HBM (psi, W and Hpsi once each).  Measured per launch, with the kernels before
// (scatter into a cleared tile, a division per element of W, 108 in three radix passes) in
// brackets: inverse 72^3, 160 bands FP64 61 us (65; 246 MB, 4.0 TB/s), FP32 35 (46); 108^3, 243
// bands FP32 226 (339); 27^3, 8 bands 3.6 (6.1).  Forward, only writing Hpsi: 44, 37 and 246 us;
// reading psi for the kinetic term and Hpsi to add to costs 75, 49 and 456 us more, because the
// rows of a column lie all over the band (pw_capi.hip: op_H_device puts both into the projector
// product where there is one).
#pragma once
#include "pw_fft_core.h"

namespace pw {

template <typename T>
struct ColArgs {
  const cplx<double>* psi;
  cplx<double>* hpsi;      // forward
  long ldpsi, ldh;
  int b0, nb;              // first band, bands of the launch
  cplx<T>* W;              // [band][z][ncol]
  const int* ztab;         // [ncol][n3]
  const double* gk2;
  int ncol;
  const KBatch* kb;        // several k-points (then psi .. ncol come from it, bands per k-point nb)
  int nk;
  const cplx<T>* tw;
  int kin, acc;            // forward: add 1/2 |G+k|^2 psi, add to hpsi
};

template <typename T, int N>
struct ColPlan {
  // 32 columns (W rows of 256 / 512 bytes) where four such tiles fit a CU, else 16
  static constexpr int C = 32 * odd_stride(N) * (int)sizeof(cplx<T>) <= 40 * 1024 ? 32 : 16;
  static constexpr int CS = odd_stride(N);
  static constexpr int NT = 256;
};

// The workgroup's columns: bands go round robin over the 8 XCDs and every chunk of a band stays
// on one, so the band's rows of psi / Hpsi share one L2.
template <typename T>
struct ColJob {
  const cplx<double>* p;
  cplx<double>* h;
  cplx<T>* w;
  const int* zt;
  const double* gk2;
  int ncol, c0, cn;
};
template <typename T, int N>
__device__ inline bool col_job(const ColArgs<T>& A, ColJob<T>& J) {
  constexpr int C = ColPlan<T, N>::C;
  int w = blockIdx.x;
  const KBatch* d = nullptr;
  J.ncol = A.ncol;
  if (A.kb) {
    int lo = 0, hi = A.nk - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (A.kb[mid].blk0 <= w) lo = mid; else hi = mid - 1;
    }
    d = A.kb + lo;
    w -= d->blk0;
    J.ncol = d->ncol;
  }
  const int nchunk = (J.ncol + C - 1) / C, s = w >> 3;
  const int bl = (w & 7) + 8 * (s / nchunk);
  J.c0 = (s % nchunk) * C;
  if (bl >= A.nb) return false;
  J.cn = min(C, J.ncol - J.c0);
  if (d) {
    J.p = d->psi + (long)bl * d->ldpsi;
    J.h = d->hpsi + (long)bl * d->ldh;
    J.w = A.W + d->woff + (long)bl * N * J.ncol;
    J.zt = d->ztab;
    J.gk2 = d->gk2;
  } else {
    J.p = A.psi + (long)(A.b0 + bl) * A.ldpsi;
    J.h = A.hpsi + (long)(A.b0 + bl) * A.ldh;
    J.w = A.W + (long)bl * N * J.ncol;
    J.zt = A.ztab;
    J.gk2 = A.gk2;
  }
  J.zt += (long)J.c0 * N;
  return true;
}

template <typename T, int N, bool HALF>
__global__ void __launch_bounds__(256) k_col_inv(ColArgs<T> A) {
  using P = LinePlan<N>;
  using W = Window<N, HALF>;
  using K = ColPlan<T, N>;
  extern __shared__ char smem_raw[];
  LDS_AS cplx<T>* lds = (LDS_AS cplx<T>*)smem_raw;
  LDS_AS cplx<T>* tw = lds + K::C * K::CS;
  ColJob<T> J;
  if (!col_job<T, N>(A, J)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int NW = K::NT / 64;
  const int g = lane / P::L, q = lane - g * P::L;
  for (int i = tid; i < N; i += K::NT) tw[i] = A.tw[i];
  for (int t0 = wave * P::G; t0 < J.cn; t0 += NW * P::G) {
    const int c = t0 + g;
    const bool act = g < P::G && c < J.cn;
    LDS_AS cplx<T>* line = lds + (act ? c : 0) * K::CS;
    const int* zt = J.zt + (act ? c : 0) * N;
#pragma unroll
    for (int s = 0; s < P::M0; ++s) {
      const int j = q + s * P::L;
      if (act && (P::M0 * P::L == P::R1 || j < P::R1)) {
        int row[W::NI];
        cplx<T> in[W::NI], v[P::R0];
#pragma unroll
        for (int i = 0; i < W::NI; ++i) row[i] = zt[j + P::R1 * W::r(i)];
#pragma unroll
        for (int i = 0; i < W::NI; ++i) {
          in[i] = mk((T)0, (T)0);
          if (row[i] >= 0) in[i] = cvt<T>(J.p[row[i]]);
        }
        dft_window<T, +1, N, HALF>(in, v);
#pragma unroll
        for (int r = 0; r < P::R0; ++r) line[j * P::R0 + r] = v[r];
      }
    }
  }
  __syncthreads();
  for (int t0 = wave * P::G; t0 < J.cn; t0 += NW * P::G) {
    const int c = t0 + g;
    const bool act = g < P::G && c < J.cn;
    LDS_AS cplx<T>* line = lds + (act ? c : 0) * K::CS;
#pragma unroll
    for (int s = 0; s < P::M1; ++s) {
      const int j = q + s * P::L;
      if (act && (P::M1 * P::L == P::R0 || j < P::R0)) {
        cplx<T> v[P::R1];
#pragma unroll
        for (int r = 0; r < P::R1; ++r) v[r] = line[j + P::R0 * r];
#pragma unroll
        for (int r = 1; r < P::R1; ++r) v[r] = cmul(v[r], tw[j * r]);
        DFT<T, +1, P::R1>::run(v);
#pragma unroll
        for (int r = 0; r < P::R1; ++r) line[j + P::R0 * r] = v[r];
      }
    }
  }
  __syncthreads();
  const int cl = tid % K::C;
  if (cl < J.cn)
#pragma unroll 4
    for (int z = tid / K::C; z < N; z += K::NT / K::C) J.w[(long)z * J.ncol + J.c0 + cl] = lds[cl * K::CS + z];
}

template <typename T, int N, bool HALF>
__global__ void __launch_bounds__(256) k_col_fwd(ColArgs<T> A) {
  using P = LinePlan<N>;
  using W = Window<N, HALF>;
  using K = ColPlan<T, N>;
  extern __shared__ char smem_raw[];
  LDS_AS cplx<T>* lds = (LDS_AS cplx<T>*)smem_raw;
  LDS_AS cplx<T>* tw = lds + K::C * K::CS;
  ColJob<T> J;
  if (!col_job<T, N>(A, J)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int NW = K::NT / 64;
  const int g = lane / P::L, q = lane - g * P::L;
  const int cl = tid % K::C;
  if (cl < J.cn)
#pragma unroll 8
    for (int z = tid / K::C; z < N; z += K::NT / K::C) lds[cl * K::CS + z] = J.w[(long)z * J.ncol + J.c0 + cl];
  for (int i = tid; i < N; i += K::NT) tw[i] = A.tw[i];
  __syncthreads();
  for (int t0 = wave * P::G; t0 < J.cn; t0 += NW * P::G) {
    const int c = t0 + g;
    const bool act = g < P::G && c < J.cn;
    LDS_AS cplx<T>* line = lds + (act ? c : 0) * K::CS;
    const int* zt = J.zt + (act ? c : 0) * N;
    cplx<T> u[P::M1][P::R1];
#pragma unroll
    for (int s = 0; s < P::M1; ++s) {
      const int j = q + s * P::L;
      if (act && (P::M1 * P::L == P::R0 || j < P::R0)) {
#pragma unroll
        for (int r = 0; r < P::R1; ++r) u[s][r] = line[j + P::R0 * r];
        DFT<T, -1, P::R1>::run(u[s]);
      }
    }
    wave_fence();
#pragma unroll
    for (int s = 0; s < P::M1; ++s) {
      const int j = q + s * P::L;
      if (act && (P::M1 * P::L == P::R0 || j < P::R0)) {
#pragma unroll
        for (int r = 0; r < P::R1; ++r) line[j * P::R1 + r] = u[s][r];
      }
    }
    wave_fence();
#pragma unroll
    for (int s = 0; s < P::M0; ++s) {
      const int j = q + s * P::L;
      if (act && (P::M0 * P::L == P::R1 || j < P::R1)) {
        int row[W::NI];
#pragma unroll
        for (int i = 0; i < W::NI; ++i) row[i] = zt[j + P::R1 * W::r(i)];
        cplx<T> v[P::R0];
#pragma unroll
        for (int r = 0; r < P::R0; ++r) v[r] = line[j + P::R1 * r];
#pragma unroll
        for (int r = 1; r < P::R0; ++r) v[r] = cmulc(v[r], tw[j * r]);
        DFT<T, -1, P::R0>::run(v);
#pragma unroll
        for (int i = 0; i < W::NI; ++i)
          if (row[i] >= 0) {
            cplx<double> o = cvt<double>(v[W::r(i)]);
            if (A.kin) o = o + scal(0.5 * J.gk2[row[i]], J.p[row[i]]);
            if (A.acc) o = o + J.h[row[i]];
            J.h[row[i]] = o;
          }
      }
    }
    wave_fence();
  }
}

template <typename T>
using ColKernel = void (*)(ColArgs<T>);
// The column kernels of length n (null without a plan); one translation unit per type.
template <typename T, bool HALF>
ColKernel<T> col_kernel(int n, bool fwd, int* chunk, size_t* lds) {
  switch (n) {
#define PW_CASE(N_, R0_, R1_, L_)                                                                         \
  case N_:                                                                                                \
    *chunk = ColPlan<T, N_>::C;                                                                           \
    *lds = (size_t)(ColPlan<T, N_>::C * ColPlan<T, N_>::CS + N_) * sizeof(cplx<T>);                       \
    return fwd ? k_col_fwd<T, N_, HALF> : k_col_inv<T, N_, HALF>;
    PW_LINE_PLANS(PW_CASE)
#undef PW_CASE
    default: return nullptr;
  }
}
extern template ColKernel<double> col_kernel<double, true>(int, bool, int*, size_t*);
extern template ColKernel<double> col_kernel<double, false>(int, bool, int*, size_t*);
extern template ColKernel<float> col_kernel<float, true>(int, bool, int*, size_t*);
extern template ColKernel<float> col_kernel<float, false>(int, bool, int*, size_t*);

// Host side (pw_col.hip).  col_chunk: columns per workgroup of the kernels for this context, 0
// where they do not apply (no plan for n3, PW_TUNE_COL_CHUNK or
// PW_TUNE_FFT_ORDER asking for the general kernels).  Launches go to the context stream.
template <typename T>
int col_chunk(const pw_ctx* c, bool zhalf);
template <typename T>
void col_inv(pw_ctx* c, const KData& k, const cplx<double>* psi, long ldpsi, int b0, int nb, cplx<T>* W);
template <typename T>
void col_fwd(pw_ctx* c, const KData& k, const cplx<double>* psi, long ldpsi, cplx<double>* hpsi, long ldh, int b0,
             int nb, const cplx<T>* W, int kin, int acc);
// blk: workgroups, KBatch::blk0 counted in chunks of col_chunk columns and bands rounded up to 8
template <typename T>
void col_inv_batch(pw_ctx* c, const KBatch* dkb, int nk, int nb, long blk, bool zhalf, cplx<T>* W);
template <typename T>
void col_fwd_batch(pw_ctx* c, const KBatch* dkb, int nk, int nb, long blk, bool zhalf, const cplx<T>* W, int kin, int acc);

}  // namespace pw
