// Butterflies and line-FFT helpers shared by the FFT translation units (pw_fft.hip,
// pw_plane.hip).
#pragma once
#include "pw_internal.h"

namespace pw {

// ----------------------------------------------------------------------------- butterflies

template <typename T, int S, int R>
struct DFT;

template <typename T, int S>
struct DFT<T, S, 2> {
  __device__ static inline void run(cplx<T>* v) {
    cplx<T> a = v[0], b = v[1];
    v[0] = a + b;
    v[1] = a - b;
  }
};

template <typename T, int S>
struct DFT<T, S, 3> {
  __device__ static inline void run(cplx<T>* v) {
    const T c = (T)-0.5;
    const T d = (T)(S * 0.86602540378443864676);
    cplx<T> t1 = v[1] + v[2], t2 = v[1] - v[2];
    cplx<T> m = v[0] + scal(c, t1);
    cplx<T> q = mk(-d * t2.y, d * t2.x);  // i*d*t2
    v[0] = v[0] + t1;
    v[1] = m + q;
    v[2] = m - q;
  }
};

template <typename T, int S>
struct DFT<T, S, 4> {
  __device__ static inline void run(cplx<T>* v) {
    cplx<T> s02 = v[0] + v[2], d02 = v[0] - v[2];
    cplx<T> s13 = v[1] + v[3], d13 = mul_i<S>(v[1] - v[3]);
    v[0] = s02 + s13;
    v[2] = s02 - s13;
    v[1] = d02 + d13;
    v[3] = d02 - d13;
  }
};

template <typename T, int S>
struct DFT<T, S, 5> {
  __device__ static inline void run(cplx<T>* v) {
    const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
    const T s1 = (T)(S * 0.95105651629515357212), s2 = (T)(S * 0.58778525229247312917);
    cplx<T> t1 = v[1] + v[4], t2 = v[2] + v[3], t3 = v[1] - v[4], t4 = v[2] - v[3];
    cplx<T> a1 = v[0] + scal(c1, t1) + scal(c2, t2);
    cplx<T> a2 = v[0] + scal(c2, t1) + scal(c1, t2);
    cplx<T> b1 = scal(s1, t3) + scal(s2, t4);
    cplx<T> b2 = scal(s2, t3) - scal(s1, t4);
    cplx<T> ib1 = mk(-b1.y, b1.x), ib2 = mk(-b2.y, b2.x);
    v[0] = v[0] + t1 + t2;
    v[1] = a1 + ib1;
    v[4] = a1 - ib1;
    v[2] = a2 + ib2;
    v[3] = a2 - ib2;
  }
};

template <typename T, int S>
struct DFT<T, S, 8> {
  __device__ static inline void run(cplx<T>* v) {
    cplx<T> e[4] = {v[0], v[2], v[4], v[6]};
    cplx<T> o[4] = {v[1], v[3], v[5], v[7]};
    DFT<T, S, 4>::run(e);
    DFT<T, S, 4>::run(o);
    const T h = (T)0.70710678118654752440;
    // w^1 = (1 + S i)/sqrt2, w^2 = S i, w^3 = (-1 + S i)/sqrt2
    cplx<T> o1 = mk(h * (o[1].x - S * o[1].y), h * (o[1].y + S * o[1].x));
    cplx<T> o2 = mul_i<S>(o[2]);
    cplx<T> o3 = mk(h * (-o[3].x - S * o[3].y), h * (-o[3].y + S * o[3].x));
    v[0] = e[0] + o[0];
    v[4] = e[0] - o[0];
    v[1] = e[1] + o1;
    v[5] = e[1] - o1;
    v[2] = e[2] + o2;
    v[6] = e[2] - o2;
    v[3] = e[3] + o3;
    v[7] = e[3] - o3;
  }
};

template <typename T, int S>
struct DFT<T, S, 9> {
  __device__ static inline void run(cplx<T>* v) {
    // 9 = 3 x 3: inner DFT3 over p (r = 3p + q), twiddle w9^(q k1), outer DFT3 over q.
    cplx<T> y[3][3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      cplx<T> t[3] = {v[q], v[3 + q], v[6 + q]};
      DFT<T, S, 3>::run(t);
      y[q][0] = t[0];
      y[q][1] = t[1];
      y[q][2] = t[2];
    }
    const T c1 = (T)0.76604444311897803520, s1 = (T)(S * 0.64278760968653932632);  // w9^1
    const T c2 = (T)0.17364817766693034885, s2 = (T)(S * 0.98480775301220805936);  // w9^2
    const T c4 = (T)-0.93969262078590838405, s4 = (T)(S * 0.34202014332566873304); // w9^4
    y[1][1] = cmul(y[1][1], mk(c1, s1));
    y[1][2] = cmul(y[1][2], mk(c2, s2));
    y[2][1] = cmul(y[2][1], mk(c2, s2));
    y[2][2] = cmul(y[2][2], mk(c4, s4));
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      cplx<T> t[3] = {y[0][k1], y[1][k1], y[2][k1]};
      DFT<T, S, 3>::run(t);
      v[k1] = t[0];
      v[k1 + 3] = t[1];
      v[k1 + 6] = t[2];
    }
  }
};

// Coprime factors R = A B (Good's prime-factor map): no twiddles between the two stages.
__host__ __device__ constexpr int inv_mod(int a, int m) {
  for (int i = 0; i < m; ++i)
    if ((a * i) % m == 1 % m) return i;
  return 0;
}
template <typename T, int S, int A, int B>
struct DFTpfa {
  __device__ static inline void run(cplx<T>* v) {
    constexpr int R = A * B, CA = B * inv_mod(B % A, A), CB = A * inv_mod(A % B, B);
    cplx<T> y[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
      cplx<T> t[A];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) t[n1] = v[(B * n1 + A * n2) % R];
      DFT<T, S, A>::run(t);
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1) y[n2][k1] = t[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      cplx<T> t[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) t[n2] = y[n2][k1];
      DFT<T, S, B>::run(t);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[(CA * k1 + CB * k2) % R] = t[k2];
    }
  }
};
template <typename T, int S> struct DFT<T, S, 6> : DFTpfa<T, S, 2, 3> {};
template <typename T, int S> struct DFT<T, S, 10> : DFTpfa<T, S, 2, 5> {};
template <typename T, int S> struct DFT<T, S, 12> : DFTpfa<T, S, 4, 3> {};
template <typename T, int S> struct DFT<T, S, 15> : DFTpfa<T, S, 3, 5> {};

template <typename T, int S>
struct DFT<T, S, 16> {
  __device__ static inline void run(cplx<T>* v) {
    // 16 = 4 x 4: DFT4 over p (r = 4 p + q), twiddle w16^(q k1), DFT4 over q
    cplx<T> y[4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      cplx<T> t[4] = {v[q], v[4 + q], v[8 + q], v[12 + q]};
      DFT<T, S, 4>::run(t);
      y[q][0] = t[0];
      y[q][1] = t[1];
      y[q][2] = t[2];
      y[q][3] = t[3];
    }
    const T c = (T)0.92387953251128675613, s = (T)(S * 0.38268343236508977173), h = (T)0.70710678118654752440;
    y[1][1] = cmul(y[1][1], mk(c, s));
    y[1][2] = mk(h * (y[1][2].x - S * y[1][2].y), h * (y[1][2].y + S * y[1][2].x));
    y[1][3] = cmul(y[1][3], mk((T)(S * s), (T)(S * c)));
    y[2][1] = mk(h * (y[2][1].x - S * y[2][1].y), h * (y[2][1].y + S * y[2][1].x));
    y[2][2] = mul_i<S>(y[2][2]);
    y[2][3] = mk(h * (-y[2][3].x - S * y[2][3].y), h * (-y[2][3].y + S * y[2][3].x));
    y[3][1] = cmul(y[3][1], mk((T)(S * s), (T)(S * c)));
    y[3][2] = mk(h * (-y[3][2].x - S * y[3][2].y), h * (-y[3][2].y + S * y[3][2].x));
    y[3][3] = cmul(y[3][3], mk(-c, -s));
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
      cplx<T> t[4] = {y[0][k1], y[1][k1], y[2][k1], y[3][k1]};
      DFT<T, S, 4>::run(t);
      v[k1] = t[0];
      v[k1 + 4] = t[1];
      v[k1 + 8] = t[2];
      v[k1 + 12] = t[3];
    }
  }
};

// Wave-local Stockham FFT.  One line (length n, element r at lds[base + r*es]) is owned by
// a group of d.L lanes of one wavefront; a wavefront holds d.gpw groups.  Lane q of a group
// takes butterflies q, q + L, ... of each radix pass, so no workgroup barrier is needed
// between passes: the LDS operations of one wavefront complete in issue order, and the
// wavefront fence keeps the compiler from moving the next pass's reads above this pass's
// writes.  In-place: every lane reads all of its butterflies before any lane writes.
// Ns = product of the radices already applied; tw[t] = exp(+2 pi i t / n).
__device__ inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS pointers keep their address space across the (non-inlined) pass so that accesses
// compile to ds_read/ds_write rather than flat instructions.
#if defined(__HIP_DEVICE_COMPILE__)
#define LDS_AS __attribute__((address_space(3)))
#else
#define LDS_AS
#endif

// Two-pass line plans N = R0 R1 with every butterfly in registers: a line is owned by L lanes
// of one wavefront (G = 64 / L lines per wavefront).  A pass of radix R0 has R1 butterflies
// (M0 per lane), a pass of radix R1 has R0 (M1 per lane).  L is the lane count with the least
// arithmetic per line (idle lanes of a pass, lanes left over from 64 / L and twiddles
// counted) that keeps at most 16 elements per lane.
template <int N> struct LinePlan;
#define PW_LINE_PLANS(X)                                                                                     \
  X(12, 4, 3, 3) X(15, 5, 3, 3) X(16, 4, 4, 4) X(18, 6, 3, 3) X(20, 5, 4, 5) X(24, 8, 3, 3) X(25, 5, 5, 5)   \
  X(27, 9, 3, 3) X(30, 10, 3, 3) X(32, 8, 4, 4) X(36, 6, 6, 6) X(40, 10, 4, 4) X(45, 9, 5, 5)                \
  X(48, 12, 4, 4) X(50, 10, 5, 5) X(54, 9, 6, 6) X(60, 10, 6, 6) X(64, 8, 8, 8) X(72, 12, 6, 6)              \
  X(75, 15, 5, 5) X(80, 10, 8, 10) X(81, 9, 9, 9) X(90, 10, 9, 10) X(96, 12, 8, 12) X(100, 10, 10, 10)       \
  X(108, 12, 9, 12) X(120, 12, 10, 12) X(128, 16, 8, 8) X(135, 15, 9, 15) X(144, 12, 12, 12)                 \
  X(150, 15, 10, 15) X(160, 16, 10, 16) X(180, 15, 12, 15) X(192, 16, 12, 16)
#define PW_LINE_PLAN_DEF(N_, R0_, R1_, L_)                                                  \
  template <> struct LinePlan<N_> {                                                         \
    static_assert(R0_ * R1_ == N_ && L_ <= 16, "plan");                                     \
    static constexpr int R0 = R0_, R1 = R1_, L = L_, G = 64 / L_;                           \
    static constexpr int M0 = (R1_ + L_ - 1) / L_, M1 = (R0_ + L_ - 1) / L_;                \
  };
PW_LINE_PLANS(PW_LINE_PLAN_DEF)
#undef PW_LINE_PLAN_DEF

// Radices and lanes of the two-pass plan of length n (r0 = 0: there is none).
struct LinePlanInfo {
  int r0 = 0, r1 = 0, L = 0;
};
inline LinePlanInfo line_plan_of(int n) {
  LinePlanInfo p;
  switch (n) {
#define PW_LINE_PLAN_CASE(N_, R0_, R1_, L_) \
  case N_: p.r0 = R0_; p.r1 = R1_; p.L = L_; break;
    PW_LINE_PLANS(PW_LINE_PLAN_CASE)
#undef PW_LINE_PLAN_CASE
    default: break;
  }
  return p;
}
inline int line_plan_groups(int n) {
  const LinePlanInfo p = line_plan_of(n);
  return p.r0 ? 64 / p.L : 0;
}
// Inputs of a first pass (outputs of a last one) that the half-sphere window keeps on each side
// of zero: element x of a line may be non-zero only where x < nz R1 or x >= n - nz R1.
__host__ __device__ constexpr int line_window(int n, int r1) { return ((n - 1) / 4) / r1 + 1; }
// Whether x lies in the window of the plan of length n (false without a plan).
inline bool line_window_holds(int n, int x) {
  const LinePlanInfo p = line_plan_of(n);
  if (!p.r0) return false;
  const int nz = line_window(n, p.r1);
  return 2 * nz >= p.r0 || x < nz * p.r1 || x >= n - nz * p.r1;
}

// The inputs a first pass takes (and the outputs a last pass leaves): element j + R1 r for the
// r with live(r).  Spheres of half the grid's radius (wave functions) occupy |x| < N / 4 or so
// on each side of zero, so with HALF only the NZ lowest and the NZ highest r can be non-zero;
// the others are constants the butterflies fold away.
template <int N, bool HALF>
struct Window {
  using P = LinePlan<N>;
  static constexpr int NZ = line_window(N, P::R1);
  static constexpr bool all = !HALF || 2 * NZ >= P::R0;
  static constexpr int NI = all ? P::R0 : 2 * NZ;
  __host__ __device__ static constexpr int r(int i) { return all || i < NZ ? i : P::R0 - 2 * NZ + i; }
};

template <typename T, int S, int N, bool HALF>
__device__ inline void dft_window(const cplx<T>* in, cplx<T>* v) {
  using W = Window<N, HALF>;
#pragma unroll
  for (int r = 0; r < LinePlan<N>::R0; ++r) v[r] = mk((T)0, (T)0);
#pragma unroll
  for (int i = 0; i < W::NI; ++i) v[W::r(i)] = in[i];
  DFT<T, S, LinePlan<N>::R0>::run(v);
}

}  // namespace pw
