// Device code of the plane kernels (pw_plane.hip, pw_plane_*.hip).
//
// The plane pass of the sphere-pruned 3-D FFT on compressed planes: per (z-plane, band) the
// inverse y-FFT of the active x lines, the x-FFT of every row, and what the caller wants of the
// row (times V(r)/N and back, |psi|^2 into the density, or a real field out).
//
// LDS holds the plane only at its active x (Yc: one y-line per active x, stride odd_stride(n2),
// and a line of zeros that stands for every inactive x).  Every line has a two-pass plan
// N = R0 R1 (LinePlan) whose butterflies stay in registers, so a pass costs one LDS read and
// one LDS write per element and the ends of the transforms need no LDS staging at all: the
// inverse y pass reads its inputs from W through the column table (-1: no column, a zero), the
// forward y pass writes its outputs to W, the x pass reads a row from Yc and writes only the
// active x back.  Between the x passes a row lives in its own slots of Yc, and V/N multiplies
// it in registers where the inverse transform ends and the forward one begins.  The plane needs
// two workgroup barriers.
//
// What bounds it (counters, 72^3, 160 bands): the LDS pipes, active for 65 % of the cycles in FP64
// and 71 % in FP32, about half of that bank conflicts; FP32 vector issue too (67 %; FP64 36 %), and
// in FP64 the two wavefronts per SIMD that its registers leave.  Per launch of 160 bands at 72^3 (a kernel with the whole padded plane in LDS, radix 9 x
// 8, before): FP64 338 us (498), FP32 176 us (203); 108^3, 243 bands: FP32 1.0 ms (3.4 ms with
// three radix passes), FP64 86 ns per plane.
#pragma once
#include "pw_fft_core.h"

namespace pw {

template <typename T>
struct PlaneArgs {
  cplx<T>* W;            // [band][z][ncol]
  const T* V;            // V(r) / N (MODE_VLOC)
  const int* ctab;       // [nxact][n2] column of (a, y), or -1
  const int* apos;       // [n1] active index of x, or -1
  const cplx<T>* twx;
  const cplx<T>* twy;
  const KBatch* kb;      // several k-points: their W, ctab, apos (band index = k nbk + band)
  double* out;           // MODE_RHO: partial planes per band group; MODE_REAL: fields
  const double* wts;     // MODE_RHO: band weights
  long N;
  double scale;          // MODE_REAL
  int n1, n2, n3, ncol, nxact;
  int nbk;               // bands per k-point (kb set)
  int nb, bpg;           // MODE_RHO: bands over all k-points, bands per group
  int acc;               // MODE_REAL: add to out
  int lines;             // lines of Yc in LDS before the zero line
};

enum { MODE_VLOC = 0, MODE_RHO = 1, MODE_REAL = 2, MODE_RHOREG = 3 };

// Inverse y-FFT of the active x lines, from the plane w (ncol entries) into Yc.
template <typename T, int N, bool HALF>
__device__ inline void plane_y_inv(LDS_AS cplx<T>* Yc, int nl, const cplx<T>* w, const int* ctab,
                                   const LDS_AS cplx<T>* tw) {
  constexpr int ys = odd_stride(N);
  using P = LinePlan<N>;
  using W = Window<N, HALF>;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
  const int g = lane / P::L, q = lane - g * P::L;
  for (int t0 = wave * P::G; t0 < nl; t0 += nwave * P::G) {
    const int a = t0 + g;
    const bool act = g < P::G && a < nl;
    LDS_AS cplx<T>* line = Yc + (act ? a : 0) * ys;
    const int* ct = ctab + (act ? a : 0) * N;
#pragma unroll
    for (int s = 0; s < P::M0; ++s) {
      const int j = q + s * P::L;
      if (act && (P::M0 * P::L == P::R1 || j < P::R1)) {
        cplx<T> in[W::NI], v[P::R0];
        int c[W::NI];
#pragma unroll
        for (int i = 0; i < W::NI; ++i) c[i] = ct[j + P::R1 * W::r(i)];
#pragma unroll
        for (int i = 0; i < W::NI; ++i) {
          const cplx<T> t = w[c[i] < 0 ? 0 : c[i]];
          in[i] = c[i] < 0 ? mk((T)0, (T)0) : t;
        }
        dft_window<T, +1, N, HALF>(in, v);
#pragma unroll
        for (int r = 0; r < P::R0; ++r) line[j * P::R0 + r] = v[r];
      }
    }
    wave_fence();
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
    wave_fence();
  }
}

// Forward y-FFT of the active x lines of Yc, the columns of the plane written to w.
template <typename T, int N, bool HALF>
__device__ inline void plane_y_fwd(LDS_AS cplx<T>* Yc, int nl, cplx<T>* w, const int* ctab,
                                   const LDS_AS cplx<T>* tw) {
  constexpr int ys = odd_stride(N);
  using P = LinePlan<N>;
  using W = Window<N, HALF>;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
  const int g = lane / P::L, q = lane - g * P::L;
  for (int t0 = wave * P::G; t0 < nl; t0 += nwave * P::G) {
    const int a = t0 + g;
    const bool act = g < P::G && a < nl;
    LDS_AS cplx<T>* line = Yc + (act ? a : 0) * ys;
    const int* ct = ctab + (act ? a : 0) * N;
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
        int c[W::NI];
#pragma unroll
        for (int i = 0; i < W::NI; ++i) c[i] = ct[j + P::R1 * W::r(i)];
        cplx<T> v[P::R0];
#pragma unroll
        for (int r = 0; r < P::R0; ++r) v[r] = line[j + P::R1 * r];
#pragma unroll
        for (int r = 1; r < P::R0; ++r) v[r] = cmulc(v[r], tw[j * r]);
        DFT<T, -1, P::R0>::run(v);
#pragma unroll
        for (int i = 0; i < W::NI; ++i)
          if (c[i] >= 0) w[c[i]] = v[W::r(i)];
      }
    }
    wave_fence();
  }
}

// A row between two passes lives in its own slots of Yc: the entries (a, y) of its y, which no
// other lane touches between the row's first reads and last writes.  Real and imaginary parts
// go one after the other, two reals per slot, so about N / 2 lines hold a row and the workgroup
// needs no row buffers (FP64 at 72^2: 45 KB, three workgroups per CU; with buffers two).
// From a pass of radix RA (RB butterflies) to one of radix RB (RA butterflies) output r of
// butterfly j is input j of butterfly r, a transpose; the pairing runs along an even radix, so
// that one side moves whole slots and every address is a lane base plus a constant.
template <int RA, int RB>
struct XchMap {
  static constexpr int HA = (RA + 1) / 2, HB = (RB + 1) / 2;
  static constexpr bool byA = RA % 2 == 0 || (RB % 2 != 0 && RB * HA <= RA * HB);
  static constexpr int lines = byA ? RB * HA : RA * HB;
};
template <typename T, int MA, int RA, int MB, int RB, int L>
__device__ inline void xch_split(LDS_AS cplx<T>* Yy, int ys, cplx<T> (&a)[MA][RA], cplx<T> (&b)[MB][RB], int q,
                                 bool act) {
  using X = XchMap<RA, RB>;
  const int ds = 2 * ys;
  LDS_AS T* d = (LDS_AS T*)Yy;
#pragma unroll
  for (int part = 0; part < 2; ++part) {
#pragma unroll
    for (int s = 0; s < MA; ++s) {
      const int j = q + s * L;
      if (act && (MA * L == RB || j < RB)) {
        LDS_AS T* dj = d + (X::byA ? j * (X::HA * ds) : (j >> 1) * ds + (j & 1));
#pragma unroll
        for (int r = 0; r < RA; ++r)
          dj[X::byA ? (r >> 1) * ds + (r & 1) : r * (X::HB * ds)] = part ? a[s][r].y : a[s][r].x;
      }
    }
    wave_fence();
#pragma unroll
    for (int s = 0; s < MB; ++s) {
      const int j = q + s * L;
      if (act && (MB * L == RA || j < RA)) {
        const LDS_AS T* dj = d + (X::byA ? (j >> 1) * ds + (j & 1) : j * (X::HB * ds));
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const T x = dj[X::byA ? r * (X::HA * ds) : (r >> 1) * ds + (r & 1)];
          if (part) b[s][r].y = x; else b[s][r].x = x;
        }
      }
    }
    wave_fence();
  }
}
// Lines of Yc a row needs for its two exchanges.
template <int N>
constexpr int xch_lines() {
  using P = LinePlan<N>;
  return XchMap<P::R0, P::R1>::lines > XchMap<P::R1, P::R0>::lines ? XchMap<P::R0, P::R1>::lines
                                                                   : XchMap<P::R1, P::R0>::lines;
}

// Every x-row of the plane.  off[x] (LDS): offset of x's line in Yc, the zero line for inactive
// x (zoff).  NY: n2 where it is known at compile time, else 0.  MODE_VLOC multiplies by V/N (vp)
// and transforms back; MODE_RHO puts scale |f|^2 into o, MODE_REAL scale Re f (added with acc, else
// stored); MODE_RHOREG adds scale |f|^2 to racc, whose entry (i, s, r) belongs to the
// wavefront's i-th round of rows.
template <typename T, int N, int NY, int MODE, bool HALF, int NR = 1>
__device__ inline void plane_x_rows(LDS_AS cplx<T>* Yc, const LDS_AS int* off, int zoff, int n2_, const LDS_AS cplx<T>* tw,
                                    const T* vp, double* o, double scale, int acc,
                                    double (*racc)[LinePlan<N>::M1][LinePlan<N>::R1] = nullptr) {
  using P = LinePlan<N>;
  using W = Window<N, HALF>;
  const int n2 = NY ? NY : n2_, ys = NY ? odd_stride(NY) : odd_stride(n2_);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
  const int g = lane / P::L, q = lane - g * P::L;
  int ox[P::M0][W::NI];
#pragma unroll
  for (int s = 0; s < P::M0; ++s) {
    const int j = q + s * P::L;
    const bool in = P::M0 * P::L == P::R1 || j < P::R1;
#pragma unroll
    for (int i = 0; i < W::NI; ++i) ox[s][i] = in ? off[j + P::R1 * W::r(i)] : zoff;
  }
  auto round = [&](int t0, int i) {
    const int y = t0 + g;
    const bool act = g < P::G && y < n2;
    const int yy = act ? y : 0;
    const long y0 = (long)yy * N;
    T vr[P::M1][P::R1];
    if (MODE == MODE_VLOC) {   // in flight during the inverse transform
#pragma unroll
      for (int s = 0; s < P::M1; ++s) {
        const int j = q + s * P::L;
        const bool in = act && (P::M1 * P::L == P::R0 || j < P::R0);
#pragma unroll
        for (int r = 0; r < P::R1; ++r) vr[s][r] = vp[in ? y0 + j + P::R0 * r : 0];
      }
    }
    // inverse, radix R0: butterfly j takes x = j + R1 r
    cplx<T> v[P::M0][P::R0], u[P::M1][P::R1];
#pragma unroll
    for (int s = 0; s < P::M0; ++s) {
      const int j = q + s * P::L;
      if (act && (P::M0 * P::L == P::R1 || j < P::R1)) {
        cplx<T> in[W::NI];
#pragma unroll
        for (int k = 0; k < W::NI; ++k) in[k] = Yc[ox[s][k] + y];
        dft_window<T, +1, N, HALF>(in, v[s]);
      }
    }
    wave_fence();
    xch_split<T, P::M0, P::R0, P::M1, P::R1, P::L>(Yc + yy, ys, v, u, q, act);
    // inverse, radix R1: butterfly j leaves x = j + R0 r, which is what the forward
    // transform's first pass (radix R1) takes
#pragma unroll
    for (int s = 0; s < P::M1; ++s) {
      const int j = q + s * P::L;
      if (act && (P::M1 * P::L == P::R0 || j < P::R0)) {
#pragma unroll
        for (int r = 1; r < P::R1; ++r) u[s][r] = cmul(u[s][r], tw[j * r]);
        DFT<T, +1, P::R1>::run(u[s]);
        if (MODE == MODE_VLOC) {
#pragma unroll
          for (int r = 0; r < P::R1; ++r) u[s][r] = scal(vr[s][r], u[s][r]);
          DFT<T, -1, P::R1>::run(u[s]);
        } else {
#pragma unroll
          for (int r = 0; r < P::R1; ++r) {
            double* d = o + y0 + j + P::R0 * r;
            const double re = (double)u[s][r].x, im = (double)u[s][r].y;
            if (MODE == MODE_RHOREG)
              racc[i][s][r] += scale * (re * re + im * im);
            else if (MODE == MODE_RHO)
              *d = acc ? *d + scale * (re * re + im * im) : scale * (re * re + im * im);
            else
              *d = acc ? *d + scale * re : scale * re;
          }
        }
      }
    }
    if (MODE == MODE_VLOC) {
      xch_split<T, P::M1, P::R1, P::M0, P::R0, P::L>(Yc + yy, ys, u, v, q, act);
      // forward, radix R0: butterfly j leaves x = j + R1 r
#pragma unroll
      for (int s = 0; s < P::M0; ++s) {
        const int j = q + s * P::L;
        if (act && (P::M0 * P::L == P::R1 || j < P::R1)) {
#pragma unroll
          for (int r = 1; r < P::R0; ++r) v[s][r] = cmulc(v[s][r], tw[j * r]);
          DFT<T, -1, P::R0>::run(v[s]);
#pragma unroll
          for (int k = 0; k < W::NI; ++k)
            if (ox[s][k] != zoff) Yc[ox[s][k] + y] = v[s][W::r(k)];
        }
      }
      wave_fence();
    }
  };
  if (MODE == MODE_RHOREG) {
#pragma unroll
    for (int i = 0; i < NR; ++i) round((i * nwave + wave) * P::G, i);
  } else {
    for (int t0 = wave * P::G; t0 < n2; t0 += nwave * P::G) round(t0, 0);
  }
}

// LDS: Yc (A.lines lines of stride odd_stride(n2), then the line of zeros, which no row's
// exchange reaches: it serves every band of a density group), twiddles, x offsets.
template <typename T>
struct PlaneLds {
  LDS_AS cplx<T>*Yc, *tx, *ty;
  LDS_AS int* off;
  int zoff;
};
template <typename T>
__device__ inline PlaneLds<T> plane_lds_of(const PlaneArgs<T>& A, int n1, int n2, char* smem) {
  PlaneLds<T> s;
  const int ys = odd_stride(n2);
  s.Yc = (LDS_AS cplx<T>*)smem;
  s.zoff = A.lines * ys;
  s.tx = s.Yc + (A.lines + 1) * ys;
  s.ty = s.tx + n1;
  s.off = (LDS_AS int*)(s.ty + n2);
  for (int i = threadIdx.x; i < n1; i += blockDim.x) s.tx[i] = A.twx[i];
  for (int i = threadIdx.x; i < n2; i += blockDim.x) s.ty[i] = A.twy[i];
  return s;
}
// The zero line and the x offsets of a k-point's active set.
template <typename T>
__device__ inline void plane_lds_k(const PlaneLds<T>& s, int n1, int n2, const int* apos) {
  const int ys = odd_stride(n2);
  for (int i = threadIdx.x; i < ys; i += blockDim.x) s.Yc[s.zoff + i] = mk((T)0, (T)0);
  for (int i = threadIdx.x; i < n1; i += blockDim.x) {
    const int a = apos[i];
    s.off[i] = a < 0 ? s.zoff : a * ys;
  }
}

// The kernel body over policies of the line lengths: Y::inv / Y::fwd / X::rows.
template <typename T, int MODE, typename L>
__device__ inline void plane_body(const PlaneArgs<T>& A, int n1, int n2) {
  extern __shared__ char smem_raw[];
  const PlaneLds<T> s = plane_lds_of<T>(A, n1, n2, smem_raw);
  const int z = blockIdx.x;
  if (MODE == MODE_RHO || MODE == MODE_RHOREG) {
    const int grp = blockIdx.y;
    double* o = A.out + (long)grp * A.N + (long)z * n1 * n2;
    typename L::Acc acc;
    if (MODE == MODE_RHOREG) L::zero(acc);
    const int bend = min(A.nb, (grp + 1) * A.bpg);
    int kk = -1, ncol = A.ncol, nxact = A.nxact;
    const int* ctab = A.ctab;
    cplx<T>* Wk = A.W;
    for (int i = grp * A.bpg; i < bend; ++i) {
      int b = i;
      if (!A.kb) {
        if (kk < 0) {
          kk = 0;
          plane_lds_k(s, n1, n2, A.apos);
          __syncthreads();
        }
      } else {
        const int k = i / A.nbk;
        b = i - k * A.nbk;
        if (k != kk) {
          kk = k;
          const KBatch& d = A.kb[k];
          ncol = d.ncol;
          nxact = d.nxact;
          ctab = d.ctab;
          Wk = A.W + d.woff;
          plane_lds_k(s, n1, n2, d.apos);
          __syncthreads();
        }
      }
      L::inv(s, nxact, Wk + ((long)b * A.n3 + z) * ncol, ctab, n2);
      __syncthreads();
      if (MODE == MODE_RHO)
        L::rho(s, n1, n2, o, A.wts[i], i != grp * A.bpg);
      else
        L::rhoreg(s, acc, A.wts[i]);
      __syncthreads();
    }
    if (MODE == MODE_RHOREG) L::store(acc, o);
    return;
  }
  int b = blockIdx.y, ncol = A.ncol, nxact = A.nxact;
  const int* ctab = A.ctab;
  const int* apos = A.apos;
  cplx<T>* W = A.W;
  if (A.kb) {
    const int k = b / A.nbk;
    const KBatch& d = A.kb[k];
    b -= k * A.nbk;
    ncol = d.ncol;
    nxact = d.nxact;
    ctab = d.ctab;
    apos = d.apos;
    W += d.woff;
  }
  plane_lds_k(s, n1, n2, apos);
  __syncthreads();
  cplx<T>* w = W + ((long)b * A.n3 + z) * ncol;
  L::inv(s, nxact, w, ctab, n2);
  __syncthreads();
  const long pl = (long)z * n1 * n2;
  if (MODE == MODE_VLOC) {
    L::vloc(s, n1, n2, A.V + pl);
    __syncthreads();
    L::fwd(s, nxact, w, ctab, n2);
  } else if (MODE == MODE_REAL) {
    L::real(s, n1, n2, A.out + (long)b * A.N + pl, A.scale, A.acc);
  }
}

// n1 = n2 = N, everything inlined.  Rounds of rows per wavefront of the density form, and its
// wavefronts: accumulators for at most three rounds stay in registers.
template <int N>
struct RhoPlan {
  static constexpr int G = LinePlan<N>::G;
  static constexpr int nw = N <= 6 * G ? 2 : N <= 12 * G ? 4 : 8;
  static constexpr int NR = (N + nw * G - 1) / (nw * G);
  static constexpr bool reg = NR <= 3;
};
template <typename T, int N, bool HALF, int NR>
struct LinesEq {
  using P = LinePlan<N>;
  struct Acc { double a[NR][P::M1][P::R1]; };
  __device__ static inline void inv(const PlaneLds<T>& s, int nl, const cplx<T>* w, const int* ctab, int) {
    plane_y_inv<T, N, HALF>(s.Yc, nl, w, ctab, s.ty);
  }
  __device__ static inline void fwd(const PlaneLds<T>& s, int nl, cplx<T>* w, const int* ctab, int) {
    plane_y_fwd<T, N, HALF>(s.Yc, nl, w, ctab, s.ty);
  }
  __device__ static inline void vloc(const PlaneLds<T>& s, int, int, const T* vp) {
    plane_x_rows<T, N, N, MODE_VLOC, HALF>(s.Yc, s.off, s.zoff, N, s.tx, vp, nullptr, 0.0, 0);
  }
  __device__ static inline void rho(const PlaneLds<T>& s, int, int, double* o, double w, int acc) {
    plane_x_rows<T, N, N, MODE_RHO, HALF>(s.Yc, s.off, s.zoff, N, s.tx, nullptr, o, w, acc);
  }
  __device__ static inline void real(const PlaneLds<T>& s, int, int, double* o, double scale, int acc) {
    plane_x_rows<T, N, N, MODE_REAL, HALF>(s.Yc, s.off, s.zoff, N, s.tx, nullptr, o, scale, acc);
  }
  __device__ static inline void zero(Acc& c) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int k = 0; k < P::M1; ++k)
#pragma unroll
        for (int r = 0; r < P::R1; ++r) c.a[i][k][r] = 0.0;
  }
  __device__ static inline void rhoreg(const PlaneLds<T>& s, Acc& c, double w) {
    plane_x_rows<T, N, N, MODE_RHOREG, HALF, NR>(s.Yc, s.off, s.zoff, N, s.tx, nullptr, nullptr, w, 0, c.a);
  }
  __device__ static inline void store(const Acc& c, double* o) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
    const int g = lane / P::L, q = lane - g * P::L;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int y = (i * nwave + wave) * P::G + g;
#pragma unroll
      for (int k = 0; k < P::M1; ++k) {
        const int j = q + k * P::L;
        if (g < P::G && y < N && (P::M1 * P::L == P::R0 || j < P::R0)) {
#pragma unroll
          for (int r = 0; r < P::R1; ++r) o[(long)y * N + j + P::R0 * r] = c.a[i][k][r];
        }
      }
    }
  }
};
template <typename T, int N, int MODE, bool HALF, int NR>
__global__ void __launch_bounds__(512) k_plane(PlaneArgs<T> A) {
  plane_body<T, MODE, LinesEq<T, N, HALF, NR>>(A, N, N);
}

// n1 != n2: the passes are functions called by line length.
template <typename T, int N, bool HALF>
__device__ __attribute__((noinline)) void call_inv(LDS_AS cplx<T>* Yc, int nl, const cplx<T>* w, const int* ctab,
                                                   const LDS_AS cplx<T>* tw) {
  plane_y_inv<T, N, HALF>(Yc, nl, w, ctab, tw);
}
template <typename T, int N, bool HALF>
__device__ __attribute__((noinline)) void call_fwd(LDS_AS cplx<T>* Yc, int nl, cplx<T>* w, const int* ctab,
                                                   const LDS_AS cplx<T>* tw) {
  plane_y_fwd<T, N, HALF>(Yc, nl, w, ctab, tw);
}
template <typename T, int N, int MODE, bool HALF>
__device__ __attribute__((noinline)) void call_rows(LDS_AS cplx<T>* Yc, const LDS_AS int* off, int zoff, int n2,
                                                    const LDS_AS cplx<T>* tw, const T* vp, double* o, double scale,
                                                    int acc) {
  plane_x_rows<T, N, 0, MODE, HALF>(Yc, off, zoff, n2, tw, vp, o, scale, acc);
}
template <typename T, bool HALF>
struct LinesAny {
  struct Acc {};
  template <int MODE>
  __device__ static inline void rows(const PlaneLds<T>& s, int n1, int n2, const T* vp, double* o, double scale,
                                     int acc) {
    switch (n1) {
#define PW_CASE(N_, R0_, R1_, L_) \
  case N_: call_rows<T, N_, MODE, HALF>(s.Yc, s.off, s.zoff, n2, s.tx, vp, o, scale, acc); break;
      PW_LINE_PLANS(PW_CASE)
#undef PW_CASE
      default: break;
    }
  }
  __device__ static inline void inv(const PlaneLds<T>& s, int nl, const cplx<T>* w, const int* ctab, int n2) {
    switch (n2) {
#define PW_CASE(N_, R0_, R1_, L_) \
  case N_: call_inv<T, N_, HALF>(s.Yc, nl, w, ctab, s.ty); break;
      PW_LINE_PLANS(PW_CASE)
#undef PW_CASE
      default: break;
    }
  }
  __device__ static inline void fwd(const PlaneLds<T>& s, int nl, cplx<T>* w, const int* ctab, int n2) {
    switch (n2) {
#define PW_CASE(N_, R0_, R1_, L_) \
  case N_: call_fwd<T, N_, HALF>(s.Yc, nl, w, ctab, s.ty); break;
      PW_LINE_PLANS(PW_CASE)
#undef PW_CASE
      default: break;
    }
  }
  __device__ static inline void vloc(const PlaneLds<T>& s, int n1, int n2, const T* vp) {
    rows<MODE_VLOC>(s, n1, n2, vp, nullptr, 0.0, 0);
  }
  __device__ static inline void rho(const PlaneLds<T>& s, int n1, int n2, double* o, double w, int acc) {
    rows<MODE_RHO>(s, n1, n2, nullptr, o, w, acc);
  }
  __device__ static inline void real(const PlaneLds<T>& s, int n1, int n2, double* o, double scale, int acc) {
    rows<MODE_REAL>(s, n1, n2, nullptr, o, scale, acc);
  }
  __device__ static inline void zero(Acc&) {}
  __device__ static inline void rhoreg(const PlaneLds<T>&, Acc&, double) {}
  __device__ static inline void store(const Acc&, double*) {}
};
// The kernel's registers are those of its heaviest callee (radix 15 and 16); FP32 is held to four
// wavefronts per SIMD, where only those callees spill (36 x 72 density planes, 41 bands: 29 -> 19 us).
template <typename T, int MODE, bool HALF>
__global__ void __launch_bounds__(512, sizeof(T) == 4 ? 4 : 2) k_plane_any(PlaneArgs<T> A) {
  plane_body<T, MODE, LinesAny<T, HALF>>(A, A.n1, A.n2);
}

template <typename T>
using PlaneKernel = void (*)(PlaneArgs<T>);
// The plane kernel of a mode for n1 x n2 planes, null when either length has no plan; half: the
// k-points' x and y lie in the windows of their plans.  One translation unit defines each.
// A sphere beyond the window (a grid smaller than twice the sphere) keeps the plane kernels, with
// every input read: sphere of radius 20 on 72^3, 160 bands, against the padded planes of pw_fft.hip:
// density 320 us (409) FP64, 200 (242) FP32, FP32 op_V_loc with its column kernels 308 (327).
template <typename T, int MODE, bool HALF>
PlaneKernel<T> plane_kernel(int n1, int n2) {
  if (!line_plan_groups(n1) || !line_plan_groups(n2)) return nullptr;
  if (n1 == n2) switch (n1) {
#define PW_CASE(N_, R0_, R1_, L_)                                                                      \
  case N_:                                                                                             \
    if constexpr (MODE == MODE_RHO && RhoPlan<N_>::reg)                                                \
      return k_plane<T, N_, MODE_RHOREG, HALF, RhoPlan<N_>::NR>;                                       \
    else                                                                                               \
      return k_plane<T, N_, MODE, HALF, 1>;
      PW_LINE_PLANS(PW_CASE)
#undef PW_CASE
      default: break;
    }
  return k_plane_any<T, MODE, HALF>;
}
extern template PlaneKernel<double> plane_kernel<double, MODE_VLOC, true>(int, int);
extern template PlaneKernel<double> plane_kernel<double, MODE_VLOC, false>(int, int);
extern template PlaneKernel<float> plane_kernel<float, MODE_VLOC, true>(int, int);
extern template PlaneKernel<float> plane_kernel<float, MODE_VLOC, false>(int, int);
extern template PlaneKernel<double> plane_kernel<double, MODE_RHO, true>(int, int);
extern template PlaneKernel<double> plane_kernel<double, MODE_RHO, false>(int, int);
extern template PlaneKernel<float> plane_kernel<float, MODE_RHO, true>(int, int);
extern template PlaneKernel<float> plane_kernel<float, MODE_RHO, false>(int, int);
extern template PlaneKernel<double> plane_kernel<double, MODE_REAL, false>(int, int);

// Host side (pw_plane.hip).  plane_applies: whether the plane kernels take planes with at most
// maxx active x (line lengths with plans, LDS, PW_TUNE_PLANE_COMPRESSED).
// The launches go to the context stream and are made only where it holds.
template <typename T>
bool plane_applies(const pw_ctx* c, int maxx);
template <typename T>
void plane_vloc(pw_ctx* c, const KData& k, cplx<T>* W, const T* V, int nb);
template <typename T>
void plane_vloc_batch(pw_ctx* c, const KBatch* dkb, int nk, int nb, int maxx, bool half, cplx<T>* W, const T* V);
// ngroup partial planes (rpart), bpg bands each, weights d_w per band; the batched form takes
// nb / nbk k-points of nbk bands each
template <typename T>
void plane_rho(pw_ctx* c, const KData& k, cplx<T>* W, int nb, int bpg, int ngroup, const double* d_w, double* rpart);
template <typename T>
void plane_rho_batch(pw_ctx* c, const KBatch* dkb, int nbk, int nb, int maxx, bool half, cplx<T>* W, int bpg,
                     int ngroup, const double* d_w, double* rpart);
// Workgroups of the density kernel that a CU holds at once, for at most maxx active x.
template <typename T>
int plane_rho_resident(const pw_ctx* c, int maxx);
void plane_real(pw_ctx* c, const KData& k, cplx<double>* W, int nf, double* out, double scale, int acc);

}  // namespace pw
