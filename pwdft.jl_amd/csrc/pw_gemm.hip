// Complex GEMM on real MFMA for the projector products of op_V_Ps_nloc
// (calc_betaNL_psi, PsPotNL.jl:242-254; beta * (D * proj), op_V_Ps_nloc.jl:59-76) and the
// Rayleigh-Ritz / Gram products of diag_LOBPCG (diag_LOBPCG.jl:85-203) and diag_davidson.
//
//   C (M x N) = alpha * op(A) * B + beta * C,  op(A) = A (M x K) or A^H (A is K x M)
//
// The 16x16x4 MFMA takes from lane l the A element of row l % 16 and the B element of column
// l % 16 at k = l / 16, so a lane's operands are whole complex numbers of A and B as they lie in
// memory: one 16-byte load per 16 x 4 complex entries of each, no LDS, no barrier.  A complex
// 16 x 16 tile is four real MFMAs per four k (re re, im im, re im, im re), 8 real flops per
// complex multiply-add with no wasted lanes.  Every wavefront runs on its own, its loads a ring
// of RING k-steps ahead of the MFMAs that use them.  What bounds it is MFMA issue (64 cycles per
// FP64 MFMA, 32 in FP32): a 32 x 32 tile needs four loads per 16 MFMAs.
//
// Long K (the Ngw-long inner products) is split into chunks; partial tiles are reduced by a
// second kernel in a fixed order, so results are bitwise repeatable.
#include "pw_internal.h"

namespace pw {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <typename TC>
struct Mfma;
template <>
struct Mfma<double> {
  typedef v4d acc_t;
  __device__ static inline acc_t run(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // row of D in register r of lane group g = l / 16 (the column is l % 16)
  __device__ static inline int row(int g, int r) { return g + 4 * r; }
};
template <>
struct Mfma<float> {
  typedef v4f acc_t;
  __device__ static inline acc_t run(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static inline int row(int g, int r) { return 4 * g + r; }
};

constexpr int GBK = 16;           // split-K chunks are multiples of this (and of every stage)

// Workgroup id -> (m tile, n tile, k chunk).  Consecutive workgroup ids land on different XCDs
// (round-robin over 8); XCD x takes the x-th contiguous eighth of the (chunk, n, m) order with
// split-K (the tiles of a chunk, which share its rows of A^H and B, meet in one L2) and of the
// (m, n) order without (the n tiles of one m tile, which share the rows of A).
__device__ inline bool tile_of(int w, int tm, int tn, int nz, int& mt, int& nt, int& z) {
  const int tiles = tm * tn, tot = tiles * nz, per = (tot + 7) >> 3;
  const int t = (w & 7) * per + (w >> 3);
  if ((w >> 3) >= per || t >= tot) return false;
  if (nz > 1) {
    z = t / tiles;
    const int r = t - z * tiles;
    nt = r / tm;
    mt = r - nt * tm;
  } else {
    z = 0;
    mt = t / tn;
    nt = t - mt * tn;
  }
  return true;
}

// A wavefront's T x T tiles of 16 x 16 complex outputs at (m0, n0), over the k-steps (4 k each)
// k0 + 4 (first + stride i) that lie wholly before kend, and the masked rest of K, which belongs
// to the wavefront with `tail`.
template <typename TC, typename TA, typename TB, int TRANSA, int TM, int TN>
struct WaveTile {
  typedef typename Mfma<TC>::acc_t acc_t;
  static constexpr int RING = TM * TN > 1 ? 4 : 8;   // k-steps in flight
  // FP32: an accumulator takes the products of RING k-steps only and is then added to a second
  // one, so that the rounding of a sum over K grows with K / (4 RING) + RING in place of K / 4
  // (error of A^H B against FP64, 320 x 160 x 23871: 1.5e-7, 5.7e-7 with one chain; 1080 x 480 x
  // 80797 with a tile per wavefront 4.2e-7, 4.2e-6).  The additions run beside other wavefronts'
  // MFMAs: 320 x 160 x 23871 170 us (174), 23871 x 160 x 320 128 (126).
  static constexpr bool WIDE = sizeof(TC) == 4;
  acc_t re[TM][TN], im[TM][TN];
  acc_t sre[TM][TN], sim[TM][TN];   // WIDE: the second accumulators

  __device__ inline void fold() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sre[i][j][r] += re[i][j][r];
          sim[i][j][r] += im[i][j][r];
          re[i][j][r] = im[i][j][r] = (TC)0;
        }
  }

  __device__ inline void mma(const cplx<TA> (&a)[TM], const cplx<TB> (&b)[TN]) {
    TC ar[TM], ai[TM], na[TM], br[TN], bi[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      ar[i] = (TC)a[i].x;
      ai[i] = (TC)a[i].y;
      na[i] = -ai[i];
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      br[j] = (TC)b[j].x;
      bi[j] = (TC)b[j].y;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        re[i][j] = Mfma<TC>::run(ar[i], br[j], re[i][j]);
        im[i][j] = Mfma<TC>::run(ar[i], bi[j], im[i][j]);
      }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        // A^H: re += im im, im -= im re; A: re -= im im, im += im re
        re[i][j] = Mfma<TC>::run(TRANSA ? ai[i] : na[i], bi[j], re[i][j]);
        im[i][j] = Mfma<TC>::run(TRANSA ? na[i] : ai[i], br[j], im[i][j]);
      }
  }

  __device__ inline void run(int M, int N, const cplx<TA>* __restrict__ A, long lda, const cplx<TB>* __restrict__ B,
                             long ldb, int m0, int n0, int kbeg, int kend, int first, int stride, bool tail) {
    const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          re[i][j][r] = im[i][j][r] = (TC)0;
          if constexpr (WIDE) sre[i][j][r] = sim[i][j][r] = (TC)0;
        }
    // rows and columns past the matrices take a valid one's data; their outputs are not stored
    const cplx<TA>* pa[TM];
    const cplx<TB>* pb[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = min(m0 + 16 * i + li, M - 1);
      pa[i] = TRANSA ? A + (long)m * lda + kbeg + lg : A + (long)(kbeg + lg) * lda + m;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) pb[j] = B + (long)min(n0 + 16 * j + li, N - 1) * ldb + kbeg + lg;
    const long sa = TRANSA ? 4 : 4 * lda;
    const int full = (kend - kbeg) >> 2;
    const int n = full > first ? (full - first + stride - 1) / stride : 0;
    cplx<TA> a[RING][TM];
    cplx<TB> b[RING][TN];
    auto load = [&](int d, int s) {
      const int k = first + s * stride;
#pragma unroll
      for (int i = 0; i < TM; ++i) a[d][i] = pa[i][k * sa];
#pragma unroll
      for (int j = 0; j < TN; ++j) b[d][j] = pb[j][4 * k];
    };
#pragma unroll
    for (int d = 0; d < RING; ++d)
      if (d < n) load(d, d);
    int s = 0;
    for (; s + 2 * RING <= n; s += RING) {
#pragma unroll
      for (int d = 0; d < RING; ++d) {
        mma(a[d], b[d]);
        load(d, s + RING + d);
      }
      if constexpr (WIDE) fold();
    }
    for (; s < n; s += RING) {
#pragma unroll
      for (int d = 0; d < RING; ++d) {
        if (s + d < n) mma(a[d], b[d]);
        if (s + RING + d < n) load(d, s + RING + d);
      }
      if constexpr (WIDE) fold();
    }
    if (tail && (kend - kbeg) & 3) {
      const bool ok = 4 * full + lg < kend - kbeg;
      cplx<TA> ta[TM];
      cplx<TB> tb[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) ta[i] = ok ? pa[i][full * sa] : mk((TA)0, (TA)0);
#pragma unroll
      for (int j = 0; j < TN; ++j) tb[j] = ok ? pb[j][4 * full] : mk((TB)0, (TB)0);
      mma(ta, tb);
    }
    if constexpr (WIDE) {
      fold();
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          re[i][j] = sre[i][j];
          im[i][j] = sim[i][j];
        }
    }
  }
};

struct GemmOut {
  cplx<double>* C;
  long ldc;
  cplx<double> alpha, beta;
  int direct, use_beta;
  cplx<double>* part;   // !direct: partial sums [z][n][m]
  GemmKin kin;          // kin.gk2 set: C += 1/2 gk2[m] psi[n][m]
};
__device__ inline void gemm_finish_one(const GemmOut& o, int m, int n, cplx<double> v) {
  cplx<double> r = cmul(o.alpha, v);
  if (o.use_beta) r = r + cmul(o.beta, o.C[(long)n * o.ldc + m]);
  if (o.kin.gk2) r = r + scal(0.5 * o.kin.gk2[m], o.kin.psi[(long)n * o.kin.ldpsi + m]);
  o.C[(long)n * o.ldc + m] = r;
}
__device__ inline void gemm_store(const GemmOut& o, int M, int N, int z, int m, int n, cplx<double> v) {
  if (m >= M || n >= N) return;
  if (o.direct) {
    gemm_finish_one(o, m, n, v);
  } else {
    o.part[((long)z * N + n) * M + m] = v;
  }
}

// WM x WN wavefronts, each with a 32 x 32 tile of its own.  (FP32: three wavefronts per SIMD in
// spite of the second accumulators; without the bound the compiler leaves two, A B 5 to 15 %
// slower.)
template <typename TC, typename TA, typename TB, int TRANSA, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN, sizeof(TC) == 4 && WM * WN <= 4 ? 3 : 1)
k_zgemm(int M, int N, int K, const cplx<TA>* __restrict__ A, long lda, const cplx<TB>* __restrict__ B,
        long ldb, int kchunk, GemmOut o, int tm, int tn, int nz) {
  int mt, nt, z;
  if (!tile_of(blockIdx.x, tm, tn, nz, mt, nt, z)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = mt * 32 * WM + 32 * (wave % WM), n0 = nt * 32 * WN + 32 * (wave / WM);
  if (m0 >= M || n0 >= N) return;
  WaveTile<TC, TA, TB, TRANSA, 2, 2> t;
  t.run(M, N, A, lda, B, ldb, m0, n0, z * kchunk, min(K, (z + 1) * kchunk), 0, 1, true);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        gemm_store(o, M, N, z, m0 + 16 * i + Mfma<TC>::row(lane >> 4, r), n0 + 16 * j + (lane & 15),
                   mk((double)t.re[i][j][r], (double)t.im[i][j][r]));
}

// WK wavefronts on one tile of (16 T) x (16 T) outputs, their k-steps interleaved, the partial
// tiles summed through LDS in wavefront order: products too small to fill the chip with 32 x 32
// tiles of their own.
template <typename TC, typename TA, typename TB, int TRANSA, int T, int WK>
__global__ void __launch_bounds__(64 * WK, sizeof(TC) == 4 && T == 2 ? 3 : 1)
k_zgemm_wk(int M, int N, int K, const cplx<TA>* __restrict__ A, long lda, const cplx<TB>* __restrict__ B,
           long ldb, int kchunk, GemmOut o, int tm, int tn, int nz) {
  __shared__ cplx<TC> red[WK][16][17];
  int mt, nt, z;
  if (!tile_of(blockIdx.x, tm, tn, nz, mt, nt, z)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = mt * 16 * T, n0 = nt * 16 * T;
  WaveTile<TC, TA, TB, TRANSA, T, T> t;
  t.run(M, N, A, lda, B, ldb, m0, n0, z * kchunk, min(K, (z + 1) * kchunk), wave, WK, wave == 0);
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j) {
      if (i + j > 0) __syncthreads();
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[wave][lane & 15][Mfma<TC>::row(lane >> 4, r)] = mk(t.re[i][j][r], t.im[i][j][r]);
      __syncthreads();
      for (int e = threadIdx.x; e < 256; e += 64 * WK) {
        const int n = e >> 4, m = e & 15;
        cplx<double> v = cvt<double>(red[0][n][m]);
#pragma unroll
        for (int w = 1; w < WK; ++w) v = v + cvt<double>(red[w][n][m]);
        gemm_store(o, M, N, z, m0 + 16 * i + m, n0 + 16 * j + n, v);
      }
    }
}

// FP32-accurate complex GEMM on BF16 MFMA (the mixed path's alternative to the FP32 MFMA
// kernel above).  Every real operand x is split into three BF16 parts x0 + x1 + x2 (x0 =
// bf16(x), x1 = bf16(x - x0), x2 = bf16(x - x0 - x1): 24 significant bits, as FP32), and
// a b = sum of the six products with a combined order above 2^-24 (a0 b0, a0 b1, a1 b0, a0 b2,
// a1 b1, a2 b0), accumulated in FP32 by v_mfma_f32_16x16x32_bf16.  The parts are formed
// once per element when a stage is written to LDS, with the 2x2 real form of op(A) already
// applied (no sign work in the MFMA loop).  Lane l feeds row (or column) l % 16 with the 8
// consecutive real k of slot block l / 16; the accumulator layout equals that of the FP32
// 16x16x4 MFMA, so the tiles, split-K and epilogue are those of k_zgemm.
// As in WaveTile an accumulator takes a short chain (one stage, two for A^H B, whose K is long)
// and is then added to a second one: error of A B 23871 x 160 x 320 1.0e-7 (3.8e-7 with one
// chain), of A^H B 1080 x 480 x 80797 3.7e-7 (1.9e-6), 67500 x 320 x 480 912 us (892).  A B in
// tiles of eight wavefronts keeps one chain over its short K: two of its workgroups share a CU at
// 128 registers, and with second accumulators one does (67500 x 480 x 320: 1103 us, 1489).
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
constexpr int HBK = 16;          // complex k per stage = 32 real k = one MFMA k step
constexpr int HKS = 2 * HBK + 8; // LDS row stride in bf16 (16-byte aligned rows, padded)

__device__ inline void split3(float x, __bf16& h0, __bf16& h1, __bf16& h2) {
  h0 = (__bf16)x;
  const float r1 = x - (float)h0;
  h1 = (__bf16)r1;
  h2 = (__bf16)(r1 - (float)h1);
}

template <typename TA, typename TB, int TRANSA, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN, WM * WN == 8 && !TRANSA ? 4 : 2)
k_zgemm_b3(int M, int N, int K, const cplx<TA>* __restrict__ A, long lda, const cplx<TB>* __restrict__ B,
           long ldb, int kchunk, GemmOut o, int tm, int tn, int nz) {
  constexpr int NT = 64 * WM * WN;
  constexpr int BMC = 32 * WM, BNC = 32 * WN;
  constexpr int NA = (BMC * HBK) / NT, NB = (BNC * HBK) / NT;
  constexpr bool WIDE = TRANSA || WM * WN < 8;
  constexpr int CHAIN = TRANSA ? 2 : 1;   // WIDE: stages whose products one FP32 accumulator takes
  static_assert(NA >= 1 && NB >= 1 && (BMC * HBK) % NT == 0 && (BNC * HBK) % NT == 0, "tile");
  __shared__ __attribute__((aligned(16))) __bf16 As[3][2 * BMC][HKS];  // [part][real row][real k]
  __shared__ __attribute__((aligned(16))) __bf16 Bs[3][BNC][HKS];      // [part][column][real k]
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave % WM, wn = wave / WM;
  int mt, nt, z;
  if (!tile_of(blockIdx.x, tm, tn, nz, mt, nt, z)) return;
  const int m0 = mt * BMC, n0 = nt * BNC;
  const int kbeg = z * kchunk;
  const int kend = min(K, kbeg + kchunk);
  v4f acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0f;
  v4f sum[4][2];   // WIDE: sums of the chains that are finished
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[i][j][r] = 0.0f;
  const int li = lane & 15, lg = lane >> 4;

  cplx<TA> ra[NA];
  cplx<TB> rb[NB];
  unsigned va = 0, vb = 0;
  auto a_idx = [&](int s, int& mm, int& kk) {
    if (TRANSA == 0) { mm = tid % BMC; kk = tid / BMC + (NT / BMC) * s; }
    else { kk = tid % HBK; mm = tid / HBK + (NT / HBK) * s; }
  };
  auto b_idx = [&](int s, int& kb, int& nn) { kb = tid % HBK; nn = tid / HBK + (NT / HBK) * s; };
  auto load_stage = [&](int k0) {
    va = 0;
    vb = 0;
#pragma unroll
    for (int s = 0; s < NA; ++s) {
      int mm, kk;
      a_idx(s, mm, kk);
      const int gm = m0 + mm, gk = k0 + kk;
      const bool ok = gm < M && gk < kend;
      ra[s] = A[ok ? (TRANSA == 0 ? (long)gk * lda + gm : (long)gm * lda + gk) : 0];
      va |= (unsigned)ok << s;
    }
#pragma unroll
    for (int s = 0; s < NB; ++s) {
      int kb, nn;
      b_idx(s, kb, nn);
      const int gkb = k0 + kb, gn = n0 + nn;
      const bool ok = gkb < kend && gn < N;
      rb[s] = B[ok ? (long)gn * ldb + gkb : 0];
      vb |= (unsigned)ok << s;
    }
  };
  // 2x2 real form of op(A)[m][k] = (x + i y): rows 2m, 2m+1, columns 2k, 2k+1 hold
  // [[x, -y], [y, x]] (x, y of A[m][k] for op = identity; of conj(A[k][m]) for op = ^H)
  auto store_stage = [&]() {
#pragma unroll
    for (int s = 0; s < NA; ++s) {
      int mm, kk;
      a_idx(s, mm, kk);
      float x = 0.0f, y = 0.0f;
      if ((va >> s) & 1u) {
        x = (float)ra[s].x;
        y = TRANSA == 0 ? (float)ra[s].y : -(float)ra[s].y;
      }
      // row 2m holds (x, -y), row 2m+1 holds (y, x) at columns 2k, 2k+1: one 4-byte write
      // per row and part
      __bf16 p0[2][2], p1[2][2], p2[2][2];
      split3(x, p0[0][0], p1[0][0], p2[0][0]);
      split3(-y, p0[0][1], p1[0][1], p2[0][1]);
      split3(y, p0[1][0], p1[1][0], p2[1][0]);
      p0[1][1] = p0[0][0];
      p1[1][1] = p1[0][0];
      p2[1][1] = p2[0][0];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
        bf16x2_t w0 = {p0[h][0], p0[h][1]}, w1 = {p1[h][0], p1[h][1]}, w2 = {p2[h][0], p2[h][1]};
        *reinterpret_cast<bf16x2_t*>(&As[0][2 * mm + h][2 * kk]) = w0;
        *reinterpret_cast<bf16x2_t*>(&As[1][2 * mm + h][2 * kk]) = w1;
        *reinterpret_cast<bf16x2_t*>(&As[2][2 * mm + h][2 * kk]) = w2;
      }
    }
#pragma unroll
    for (int s = 0; s < NB; ++s) {
      int kb, nn;
      b_idx(s, kb, nn);
      float x = 0.0f, y = 0.0f;
      if ((vb >> s) & 1u) {
        x = (float)rb[s].x;
        y = (float)rb[s].y;
      }
      typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
      __bf16 x0, x1, x2, y0, y1, y2;
      split3(x, x0, x1, x2);
      split3(y, y0, y1, y2);
      const bf16x2_t w0 = {x0, y0}, w1 = {x1, y1}, w2 = {x2, y2};
      *reinterpret_cast<bf16x2_t*>(&Bs[0][nn][2 * kb]) = w0;
      *reinterpret_cast<bf16x2_t*>(&Bs[1][nn][2 * kb]) = w1;
      *reinterpret_cast<bf16x2_t*>(&Bs[2][nn][2 * kb]) = w2;
    }
  };

  auto fold = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sum[i][j][r] += acc[i][j][r];
          acc[i][j][r] = 0.0f;
        }
  };

  if (kbeg < kend) load_stage(kbeg);
  for (int k0 = kbeg; k0 < kend; k0 += HBK) {
    store_stage();
    __syncthreads();
    if (k0 + HBK < kend) load_stage(k0 + HBK);  // in flight during the MFMA phase
    // six products, smallest first; the 8 accumulators interleave so that dependent MFMAs
    // on one accumulator are 8 instructions apart
    constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
    for (int ks = 0; ks < HBK / 16; ++ks) {
      bf16x8_t a[3][4], b[3][2];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
          a[p][rt] = *reinterpret_cast<const bf16x8_t*>(&As[p][wm * 64 + rt * 16 + li][32 * ks + 8 * lg]);
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
          b[p][ct] = *reinterpret_cast<const bf16x8_t*>(&Bs[p][wn * 32 + ct * 16 + li][32 * ks + 8 * lg]);
      }
#pragma unroll
      for (int pr = 0; pr < 6; ++pr)
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
          for (int ct = 0; ct < 2; ++ct)
            acc[rt][ct] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[PA[pr]][rt], b[PB[pr]][ct], acc[rt][ct], 0, 0, 0);
    }
    if constexpr (WIDE)
      if ((k0 - kbeg) / HBK % CHAIN == CHAIN - 1) fold();
    __syncthreads();
  }
  fold();
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int ip = wm * 64 + rt * 16 + 4 * lg + 2 * p;
        gemm_store(o, M, N, z, m0 + (ip >> 1), n0 + wn * 32 + ct * 16 + li,
                   mk((double)sum[rt][ct][2 * p], (double)sum[rt][ct][2 * p + 1]));
      }
}

__global__ void k_zgemm_reduce(int M, int N, int nz, GemmOut o) {
  const long tot = (long)M * N;
  for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < tot; t += (long)gridDim.x * blockDim.x) {
    const int m = (int)(t % M), n = (int)(t / M);
    cplx<double> s = mk(0.0, 0.0);
    for (int z = 0; z < nz; ++z) s = s + o.part[((long)z * N + n) * M + m];
    gemm_finish_one(o, m, n, s);
  }
}

// Complex multiply-adds from which the split-BF16 kernel takes FP32 products by default: Si216's
// projector and Gram products (4e10).  Where it pays depends on both columns and size; op_H with FP32
// products / with split ones, one after the other, us: 72^3, 320 projectors, 80 bands (6e8) 277 /
// 299, 120 bands 394 / 386, 160 bands (1.2e9) 520 / 495, 240 bands 796 / 723, 480 bands (3.7e9)
// 1618 / 1753; 108^3, 243 bands (5.3e9) 2562 / 2230, 480 bands (1e10) 4966 / 5097.  Its error on
// long sums is up to twice the FP32 kernels', so below the line it is left to the autotuner.
constexpr double GEMM_SPLIT_MIN = 8589934592.0;

// Split of K over `nz` chunks for about `slots` workgroups on `tiles` tiles (no chunk shorter
// than `kmin`, none longer than `kmax` where that is set: FP32 sums), the partial-sum workspace
// and the epilogue.
struct GemmSplit {
  int nz = 1, kchunk = GBK;
  long nwg = 0;
  GemmOut o{};
};
static int gemm_split(pw_ctx* c, int M, int N, int K, long tiles, long slots, int kmin, int kmax, cplx<double> alpha,
                      cplx<double> beta, cplx<double>* C, long ldc, const GemmKin& kin, GemmSplit& g) {
  const int ksteps = (K + GBK - 1) / GBK;
  long nz = std::min<long>(slots / std::max<long>(tiles, 1), K / std::max(kmin, GBK));
  nz = std::max<long>(nz, kmax > 0 ? (K + kmax - 1) / kmax : 1);
  nz = std::max<long>(nz, 1);
  // a no-allocation call splits K only as far as its fixed partial-sum array holds
  if (c->no_alloc && nz > 1) nz = std::max<long>(1, std::min<long>(nz, (long)(c->gpart_bytes / ((size_t)M * N * 16))));
  if (K > 0) {
    g.kchunk = (int)((ksteps + nz - 1) / nz) * GBK;
    nz = (K + g.kchunk - 1) / g.kchunk;
  }
  g.nz = (int)nz;
  g.nwg = 8 * ((tiles * nz + 7) / 8);   // ids past the work return at once
  g.o.C = C;
  g.o.ldc = ldc;
  g.o.alpha = alpha;
  g.o.beta = beta;
  g.o.use_beta = (beta.x != 0.0 || beta.y != 0.0) ? 1 : 0;
  g.o.direct = nz == 1 ? 1 : 0;
  g.o.kin = kin;
  if (nz > 1) {
    int rc = ensure(c, &c->d_gpart, &c->gpart_bytes, (size_t)nz * M * N * sizeof(cplx<double>));
    if (rc) return rc;
    g.o.part = reinterpret_cast<cplx<double>*>(c->d_gpart);
  }
  return PW_OK;
}
static int gemm_finish(pw_ctx* c, int M, int N, const GemmSplit& g) {
  if (g.nz > 1) {
    const long tot = (long)M * N;
    const int blocks = (int)std::min<long>((tot + 255) / 256, 2048);
    hipLaunchKernelGGL(k_zgemm_reduce, dim3(blocks), dim3(256), 0, c->stream, M, N, g.nz, g.o);
  }
  return hip_check(c, hipGetLastError(), "zgemm");
}

// One (WM x WN) instance of the kernels with 32 x 32 tiles per wavefront.
template <typename TC, typename TA, typename TB, int WM, int WN>
static int zgemm_launch(pw_ctx* c, int transa, int M, int N, int K, cplx<double> alpha, const cplx<TA>* A,
                        long lda, const cplx<TB>* B, long ldb, cplx<double> beta, cplx<double>* C, long ldc,
                        const GemmKin& kin, int target_wg) {
  constexpr int BMC = 32 * WM, BNC = 32 * WN;
  const int tm = (M + BMC - 1) / BMC, tn = (N + BNC - 1) / BNC;
  GemmSplit g;
  int rc = gemm_split(c, M, N, K, (long)tm * tn, target_wg, 128, sizeof(TC) == 4 ? 8192 : 0, alpha, beta, C, ldc,
                      kin, g);
  if (rc) return rc;
  bool split_bf16 = false;
  // the three-part operands of a 128 x 128 tile do not fit in LDS: that shape keeps FP32 MFMA
  if constexpr (sizeof(TC) == 4 && WM * WN < 16)
    split_bf16 = c->gemm_split_bf16 > 0 || (c->gemm_split_bf16 < 0 && (double)M * N * K >= GEMM_SPLIT_MIN);
  {
    ProfScope ps(c, transa ? PW_PROF_GEMM_CN : PW_PROF_GEMM_NN,
                 (double)M * K * sizeof(cplx<TA>) + (double)K * N * sizeof(cplx<TB>) +
                     (double)M * N * 16.0 * (g.o.use_beta ? 2 : 1));
    const dim3 grid((unsigned)g.nwg), blk(64 * WM * WN);
    if constexpr (sizeof(TC) == 4 && WM * WN < 16) {
      if (split_bf16) {
        if (transa)
          hipLaunchKernelGGL((k_zgemm_b3<TA, TB, 1, WM, WN>), grid, blk, 0, c->stream, M, N, K, A, lda, B, ldb,
                             g.kchunk, g.o, tm, tn, g.nz);
        else
          hipLaunchKernelGGL((k_zgemm_b3<TA, TB, 0, WM, WN>), grid, blk, 0, c->stream, M, N, K, A, lda, B, ldb,
                             g.kchunk, g.o, tm, tn, g.nz);
      }
    }
    if (!split_bf16) {
      if (transa)
        hipLaunchKernelGGL((k_zgemm<TC, TA, TB, 1, WM, WN>), grid, blk, 0, c->stream, M, N, K, A, lda, B, ldb, g.kchunk,
                           g.o, tm, tn, g.nz);
      else
        hipLaunchKernelGGL((k_zgemm<TC, TA, TB, 0, WM, WN>), grid, blk, 0, c->stream, M, N, K, A, lda, B, ldb, g.kchunk,
                           g.o, tm, tn, g.nz);
    }
    rc = gemm_finish(c, M, N, g);
  }
  return rc;
}

// The kernels whose WK wavefronts share one (16 T) x (16 T) tile.
template <typename TC, typename TA, typename TB, int T, int WK>
static int zgemm_wk_launch(pw_ctx* c, int transa, int M, int N, int K, cplx<double> alpha, const cplx<TA>* A,
                           long lda, const cplx<TB>* B, long ldb, cplx<double> beta, cplx<double>* C, long ldc,
                           const GemmKin& kin, int target_wg) {
  const int tm = (M + 16 * T - 1) / (16 * T), tn = (N + 16 * T - 1) / (16 * T);
  GemmSplit g;
  int rc = gemm_split(c, M, N, K, (long)tm * tn, target_wg, 16 * 4 * WK,
                      sizeof(TC) == 4 ? 512 * WK : 0, alpha, beta, C, ldc, kin, g);
  if (rc) return rc;
  ProfScope ps(c, transa ? PW_PROF_GEMM_CN : PW_PROF_GEMM_NN,
               (double)M * K * sizeof(cplx<TA>) + (double)K * N * sizeof(cplx<TB>) +
                   (double)M * N * 16.0 * (g.o.use_beta ? 2 : 1));
  const dim3 grid((unsigned)g.nwg), blk(64 * WK);
  if (transa)
    hipLaunchKernelGGL((k_zgemm_wk<TC, TA, TB, 1, T, WK>), grid, blk, 0, c->stream, M, N, K, A, lda, B, ldb, g.kchunk,
                       g.o, tm, tn, g.nz);
  else
    hipLaunchKernelGGL((k_zgemm_wk<TC, TA, TB, 0, T, WK>), grid, blk, 0, c->stream, M, N, K, A, lda, B, ldb, g.kchunk,
                       g.o, tm, tn, g.nz);
  return gemm_finish(c, M, N, g);
}

template <typename TC, typename TA, typename TB>
static int zgemm_t(pw_ctx* c, int transa, int M, int N, int K, cplx<double> alpha, const cplx<TA>* A,
                   long lda, const cplx<TB>* B, long ldb, cplx<double> beta, cplx<double>* C, long ldc,
                   const GemmKin& kin) {
  if (M <= 0 || N <= 0) return PW_OK;
  // tuning knobs (pw_tune_set): tile shape and the split-K target workgroup count
  const int slot = transa ? 0 : 1;
  int shape = c->tune_gemm_shape[slot], target = c->tune_gemm_wg[slot];
  const double work = (double)M * N * K;
  const long t32 = (long)((M + 31) / 32) * ((N + 31) / 32);
  // Measured (us; K chunks so that two wavefronts per SIMD run):
  //  - below 2^26 complex multiply-adds 32 x 32 tiles leave most of the chip idle: 16 x 16
  //    tiles, eight wavefronts along K (A^H B 40 x 20 x 4573: 14 against 19 with 32 x 32 tiles
  //    and 39 with LDS-staged 64 x 32 ones; 480 x 160 x 480: 17 against 32);
  //  - A^H B of few tiles (the Gram and projector products of one k-point): four wavefronts
  //    share a 32 x 32 tile's K, which quarters the partial sums (FP64 160 x 160 x 23871: 88
  //    against 114 with a tile per wavefront; FP32 320 x 160 x 23871: 136 against 145); from 64
  //    tiles on, in FP64, a tile per wavefront, whose neighbours share its loads in L1 (1080 x
  //    480 x 80797: 5470 with 8 wavefronts against 8290).  FP32 keeps the shared tile: a tile per
  //    wavefront is 9 % faster or slower by size (320 x 243 x 67500: 623 against 571, 700 x 400 x
  //    30000: 1056 against 1152, 500 x 300 x 9000: 213 against 196, 240 x 200 x 30000: 227
  //    against 242), its error half again as large;
  //  - A B that fills the chip: a tile per wavefront in FP64 (23871 x 160 x 160: 91 against
  //    105), four per tile in FP32, whose shorter MFMAs leave less time per load (23871 x 160 x
  //    320: 128 against 148).
  if constexpr (sizeof(TC) == 4) {
    if (shape < 0 && (c->gemm_split_bf16 > 0 || (c->gemm_split_bf16 < 0 && work >= GEMM_SPLIT_MIN))) {
      // the split-BF16 kernel's tiles
      const int pad64 = (N + 63) / 64 * 64, pad32 = (N + 31) / 32 * 32;
      shape = N >= 256 ? 1 : pad32 < pad64 && transa ? 5 : 0;
      if (!target) target = transa ? (N >= 256 ? 2048 : 1024) : 512;
    }
  }
  if (shape < 0) {
    if (work < 67108864.0) shape = 6;
    else if (transa) shape = t32 < 64 || sizeof(TC) == 4 ? 7 : t32 < 256 ? 0 : 1;
    else shape = t32 < 1024 || sizeof(TC) == 4 ? 7 : 4;
  }
  if (!target) target = shape == 2 || shape == 3 ? 256 : shape == 5 ? 1024 : 512;
  switch (shape) {
    case 1: return zgemm_launch<TC, TA, TB, 4, 2>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin, target);
    case 4: return zgemm_launch<TC, TA, TB, 4, 1>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin, target);
    case 5: return zgemm_launch<TC, TA, TB, 2, 1>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin, target);
    case 2: return zgemm_launch<TC, TA, TB, 2, 4>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin, target);
    case 3: return zgemm_launch<TC, TA, TB, 4, 4>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin, target);
    case 6: return zgemm_wk_launch<TC, TA, TB, 1, 8>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin, target);
    case 7: return zgemm_wk_launch<TC, TA, TB, 2, 4>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin, target);
    default: return zgemm_launch<TC, TA, TB, 2, 2>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin, target);
  }
}

int zgemm(pw_ctx* c, int transa, int M, int N, int K, cplx<double> alpha, const cplx<double>* A, long lda,
          const cplx<double>* B, long ldb, cplx<double> beta, cplx<double>* C, long ldc, int prec,
          const GemmKin& kin) {
  if (prec) return zgemm_t<float, double, double>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin);
  return zgemm_t<double, double, double>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin);
}

int zgemm_f32in(pw_ctx* c, int transa, int M, int N, int K, cplx<double> alpha, const cplx<float>* A,
                long lda, const cplx<double>* B, long ldb, cplx<double> beta, cplx<double>* C, long ldc,
                int prec, const GemmKin& kin) {
  (void)prec;
  return zgemm_t<float, float, double>(c, transa, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, kin);
}

}  // namespace pw
