// Small dense problems of the block eigensolvers (order n <= 64), one workgroup per matrix
// with the matrix in LDS, for many matrices in one launch: the Rayleigh-Ritz and Gram
// matrices of every k-point of a batched LOBPCG step (2 Nst, 3 Nst = 16, 24 at 8 bands), and
// those of small single k-point problems.  They replace the LAPACK calls of
// diag_LOBPCG.jl:106-118 (cholesky, inv) and :176-190 (eigen) for these orders, launch
// nothing else and need no library workspace, so a step that uses them can be captured
// into a graph whole.
//
//  - k_heev_jacobi: Hermitian eigenpairs by cyclic Jacobi rotations in tournament order
//    (n/2 disjoint rotations per round, all applied at once), a pair
//    rotated while |A_pq| > max(1e-15 sqrt|A_pp A_qq|, 2 eps ||A||_F), until no pair passes
//    that test (checked on every pair after each sweep, in place of a sweep that would only
//    confirm it); eigenvalues sorted ascending with their vectors.  Complex 2x2 step: the pair (p, q) with A_pq = |g| e^{i phi} is made
//    real by diag(1, e^{-i phi}) and diagonalised by the classical rotation
//    t = sign(tau) / (|tau| + sqrt(1 + tau^2)), tau = (A_qq - A_pp) / (2 |g|).
//  - k_chol_inv_small: inv(chol(Hermitian(A)).U) by right-looking elimination of [A | I], the
//    matrix held in registers and one barrier per step; the strict lower triangle zeroed.
//    Status: 0, or the index (1-based) of the first non-positive pivot.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "pw_internal.h"
#include "pw_fft_core.h"

namespace pw {

constexpr int SM_NT = 256;
constexpr int SM_NMAX = 64;
constexpr int SM_SWEEPS = 30;

__device__ inline double sm_block_sum(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int q = 0; q < SM_NT / 64; ++q) s += red[q];
  return s;
}

// Matrix b of the stack at A + b * stride (leading dimension lda): eigenvalues (ascending)
// into w + b * n, the nvec lowest eigenvectors into the matrix's first nvec columns.
// A <- J^H A J is applied per 2 x 2 block (rows of pair k, columns of pair k'; the pairs of
// a round are disjoint, so every element belongs to one block): the columns' rotation, then
// the rows', as a two-pass form would apply them, in one pass beside the update of V.
__device__ inline void jac_rot(cplx<double>& x0, cplx<double>& x1, double c, double s, cplx<double> ph) {
  // (x0, x1) <- (c x0 - s ph x1, s x0 + c ph x1)
  const cplx<double> xp = x0, xq = cmul(x1, ph);
  x0 = mk(c * xp.x - s * xq.x, c * xp.y - s * xq.y);
  x1 = mk(s * xp.x + c * xq.x, s * xp.y + c * xq.y);
}

__global__ void __launch_bounds__(SM_NT) k_heev_jacobi(cplx<double>* __restrict__ A, long lda, long stride, int n,
                                                    double* __restrict__ w, int nvec, int* __restrict__ info) {
  extern __shared__ char smem_raw[];
  cplx<double>* a = reinterpret_cast<cplx<double>*>(smem_raw);   // n x n
  cplx<double>* v = a + n * n;                                     // n x n
  __shared__ double rc[SM_NMAX / 2], rs[SM_NMAX / 2];
  __shared__ cplx<double> rph[SM_NMAX / 2];       // e^{-i phi} of each pair
  __shared__ int rp[SM_NMAX / 2], rq[SM_NMAX / 2];   // rq < 0: the index paired with the dummy player
  __shared__ double dsort[SM_NMAX];
  __shared__ int rank[SM_NMAX];
  cplx<double>* M = A + (long)blockIdx.x * stride;
  const int lane = threadIdx.x;
  const int nn = n * n;
  __shared__ double red[SM_NT / 64];
  __shared__ int flag, flag2;
  // Hermitian(M): upper triangle, real diagonal
  double fro = 0.0;
  for (int t = lane; t < nn; t += SM_NT) {
    const int i = t % n, j = t / n;
    cplx<double> x;
    if (i < j) x = M[(long)j * lda + i];
    else if (i == j) x = mk(M[(long)j * lda + i].x, 0.0);
    else { const cplx<double> u = M[(long)i * lda + j]; x = mk(u.x, -u.y); }
    a[i + n * j] = x;
    v[i + n * j] = mk(i == j ? 1.0 : 0.0, 0.0);
    fro += x.x * x.x + x.y * x.y;
  }
  fro = sm_block_sum(fro, red);
  // below 2 eps ||A||_F an off-diagonal entry is rounding noise of the rotations themselves
  // (rotating it changes eigenvalues by less than the backward error of the decomposition);
  // a tighter floor keeps pairs with small or disparate diagonals rotating on noise for
  // sweep after sweep
  const double gfloor = 2.0 * 2.220446049250313e-16 * sqrt(fro);
  const int m = (n + 1) / 2 * 2;     // players of the tournament (one dummy when n is odd)
  const int npair = m / 2;
  bool converged = false;
  for (int sweep = 0; sweep < SM_SWEEPS; ++sweep) {
    if (lane == 0) flag = 0;
    int nrot = 0;
    for (int r = 0; r < m - 1; ++r) {
      if (lane < npair) {
        int p, q;
        if (lane == 0) {
          p = m - 1;
          q = r;
        } else {
          // (r + lane) mod (m - 1) and (r - lane) mod (m - 1) by one conditional subtraction
          // each (both sums lie in [0, 2 (m - 1))): this runs on every round's critical path
          p = r + lane;
          if (p >= m - 1) p -= m - 1;
          q = r - lane + (m - 1);
          if (q >= m - 1) q -= m - 1;
        }
        if (p > q) { const int t = p; p = q; q = t; }
        double c = 1.0, s = 0.0;
        cplx<double> ph = mk(1.0, 0.0);
        if (q < n) {
          const cplx<double> g = a[p + n * q];
          const double ag2 = g.x * g.x + g.y * g.y;
          const double app = a[p + n * p].x, aqq = a[q + n * q].x;
          // the tests of |A_pq| on squares, and 1 / |A_pq| by one reciprocal square root: the
          // rotation parameters are a serial chain on every round's critical path
          if (ag2 > 1e-30 * fabs(app * aqq) && ag2 > gfloor * gfloor) {
            ++nrot;
            const double rag = rsqrt(ag2);   // 1 / |A_pq|
            const double tau = (aqq - app) * (0.5 * rag);
            const double t = (tau >= 0.0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
            c = rsqrt(1.0 + t * t);
            s = t * c;
            ph = mk(g.x * rag, -g.y * rag);   // e^{-i phi}
          }
        } else {
          q = -1;   // p meets the dummy: not rotated this round
        }
        rp[lane] = p;
        rq[lane] = q;
        rc[lane] = c;
        rs[lane] = s;
        rph[lane] = ph;
      }
      __syncthreads();
      // A <- J^H A J, block (rows of pair k, columns of pair k2), one block per thread (a
      // lane map on 32-wide rows of blocks idles most lanes at the batched orders 16 and 24)
      for (int t = lane; t < npair * npair; t += SM_NT) {
        const int k = t % npair, k2 = t / npair;
        const int p = rp[k], q = rq[k], p2 = rp[k2], q2 = rq[k2];
        const double s = rs[k], s2 = rs[k2];
        if (s == 0.0 && s2 == 0.0) continue;
        const bool qv = q >= 0, q2v = q2 >= 0;
        cplx<double> b00 = a[p + n * p2];
        cplx<double> b01 = q2v ? a[p + n * q2] : mk(0.0, 0.0);
        cplx<double> b10 = qv ? a[q + n * p2] : mk(0.0, 0.0);
        cplx<double> b11 = (qv && q2v) ? a[q + n * q2] : mk(0.0, 0.0);
        if (s2 != 0.0) {   // columns p2, q2
          const double c2 = rc[k2];
          const cplx<double> ph2 = rph[k2];
          jac_rot(b00, b01, c2, s2, ph2);
          jac_rot(b10, b11, c2, s2, ph2);
        }
        if (s != 0.0) {    // rows p, q: e^{i phi}
          const double c1 = rc[k];
          const cplx<double> phc = mk(rph[k].x, -rph[k].y);
          jac_rot(b00, b10, c1, s, phc);
          jac_rot(b01, b11, c1, s, phc);
        }
        a[p + n * p2] = b00;
        if (q2v) a[p + n * q2] = b01;
        if (qv) a[q + n * p2] = b10;
        if (qv && q2v) a[q + n * q2] = b11;
      }
      // V <- V J, columns of pair k2
      for (int t = lane; t < npair * n; t += SM_NT) {
        const int k2 = t / n, i = t % n;
        const int p2 = rp[k2], q2 = rq[k2];
        const double s2 = rs[k2];
        if (q2 < 0 || s2 == 0.0) continue;
        cplx<double> x0 = v[i + n * p2], x1 = v[i + n * q2];
        jac_rot(x0, x1, rc[k2], s2, rph[k2]);
        v[i + n * p2] = x0;
        v[i + n * q2] = x1;
      }
      __syncthreads();
    }
    if (nrot) flag = 1;   // any thread that rotated this sweep
    if (lane == 0) flag2 = 0;
    __syncthreads();
    const int more = flag;
    if (!more) {
      converged = true;
      break;
    }
    // would the next sweep rotate any pair?  The same test as the rotations', on every pair
    // of the matrix as it stands: when none passes, that sweep would change nothing, so the
    // sweep that only confirms convergence is skipped (the result is the same to the bit)
    for (int t = lane; t < nn; t += SM_NT) {
      const int i = t % n, j = t / n;
      if (i < j) {
        const cplx<double> g = a[i + n * j];
        const double ag2 = g.x * g.x + g.y * g.y;
        if (ag2 > 1e-30 * fabs(a[i + n * i].x * a[j + n * j].x) && ag2 > gfloor * gfloor) flag2 = 1;
      }
    }
    __syncthreads();
    const int again = flag2;
    __syncthreads();
    if (!again) {
      converged = true;
      break;
    }
  }
  // eigenvalues: the diagonal; sort ascending (ties by index) with the vectors
  if (lane < n) dsort[lane] = a[lane + n * lane].x;
  __syncthreads();
  if (lane < n) {
    const double d = dsort[lane];
    int r = 0;
    for (int j = 0; j < n; ++j) r += (dsort[j] < d || (dsort[j] == d && j < lane)) ? 1 : 0;
    rank[lane] = r;
    w[(long)blockIdx.x * n + r] = d;
  }
  __syncthreads();
  for (int t = lane; t < nn; t += SM_NT) {
    const int i = t % n, j = t / n;
    const int r = rank[j];
    if (r < nvec) M[(long)r * lda + i] = v[i + n * j];
  }
  if (lane == 0 && info) info[blockIdx.x] = converged ? 0 : 1;
}

// The same solver for n <= 32, built for the length of a round, which the rotation parameters'
// serial chain, the barriers and the instructions around them set (mean per solve over an SCF of
// Si2, n = 24: 186 us, 16: 76, 8: 17; 110 over the three orders with the kernel above, 78 now):
//  - A is updated from one buffer into another, so a round has one barrier: every wavefront
//    computes all rotation parameters for itself from the buffer nobody writes;
//  - a thread keeps one block of A or one pair of V for the whole solve (no index division per
//    round), A's blocks and V's pairs on different wavefronts side by side;
//  - tan(theta) starts from FP32 root and reciprocal; two Newton steps with the residual in FP64
//    bring it to FP64 accuracy (their slope may be FP32: it scales a correction).
__device__ inline void jac_pair(int r, int k, int m, int n, int& p, int& q) {
  if (k == 0) {
    p = m - 1;
    q = r;
  } else {
    p = r + k;
    if (p >= m - 1) p -= m - 1;
    q = r - k + (m - 1);
    if (q >= m - 1) q -= m - 1;
  }
  if (p > q) { const int t = p; p = q; q = t; }
  if (q >= n) q = -1;   // p meets the dummy: not rotated this round
}

constexpr int JLD = 33;   // column stride: odd, and a constant

template <int NT>
__global__ void __launch_bounds__(NT) k_heev_jacobi32(cplx<double>* __restrict__ A, long lda, long stride, int n,
                                                      double* __restrict__ w, int nvec, int* __restrict__ info) {
  constexpr int NW = NT / 64;
  extern __shared__ char smem_raw[];
  LDS_AS cplx<double>* cur = (LDS_AS cplx<double>*)smem_raw;   // n columns of JLD
  LDS_AS cplx<double>* nxt = cur + n * JLD;
  LDS_AS cplx<double>* v = nxt + n * JLD;
  __shared__ cplx<double> rcs[NW][16], rph[NW][16];   // (c, s) and e^{-i phi} of each pair
  __shared__ int pq[31 * 16];   // slot p | q << 8 of every pair of every round; q = 255: the dummy
  __shared__ double dsort[32];
  __shared__ int rank[32];
  __shared__ double red[NW];
  __shared__ int flag;
  cplx<double>* M = A + (long)blockIdx.x * stride;
  const int tid = threadIdx.x, wl = tid & 63, wave = tid >> 6;
  const int nn = n * n;
  double fro = 0.0;
  for (int t = tid; t < nn; t += NT) {
    const int i = t % n, j = t / n;
    cplx<double> x;
    if (i < j) x = M[(long)j * lda + i];
    else if (i == j) x = mk(M[(long)j * lda + i].x, 0.0);
    else { const cplx<double> u = M[(long)i * lda + j]; x = mk(u.x, -u.y); }
    cur[i + JLD * j] = x;
    v[i + JLD * j] = mk(i == j ? 1.0 : 0.0, 0.0);
    fro += x.x * x.x + x.y * x.y;
  }
  const int m = (n + 1) / 2 * 2, npair = m / 2;
  for (int t = tid; t < (m - 1) * 16; t += NT) {
    int p = 0, q = 255;
    if ((t & 15) < npair) jac_pair(t >> 4, t & 15, m, n, p, q);
    pq[t] = p | (q < 0 ? 255 : q) << 8;
  }
  for (int o = 32; o > 0; o >>= 1) fro += __shfl_xor(fro, o, 64);
  if (wl == 0) red[wave] = fro;
  __syncthreads();
  fro = 0.0;
  for (int q = 0; q < NW; ++q) fro += red[q];
  // the floor of the general kernel: below it an entry is the rotations' own rounding noise
  const double gfloor2 = 4.0 * 2.220446049250313e-16 * 2.220446049250313e-16 * fro;
  // this thread's work: A blocks (rows of pair k, columns of pair j), then V pairs (row j of V,
  // columns of pair k), the V items starting on a wavefront of their own
  const int na = npair * npair, v0 = (na + 63) / 64 * 64;
  const int kind = tid < na ? 1 : tid >= v0 && tid < v0 + npair * n ? 2 : 0;
  const int u0 = kind == 2 ? tid - v0 : tid, d0 = kind == 2 ? n : npair;
  const int j = kind == 2 ? u0 % d0 : u0 / d0, k = kind == 2 ? u0 / d0 : u0 % d0;
  bool converged = false;
  for (int sweep = 0; sweep < SM_SWEEPS; ++sweep) {
    if (tid == 0) flag = 0;
    // this round's pairs, read a round ahead: the wavefront's wl-th, and the item's two
    int ew = pq[wl & 15], ek = pq[k], ej = kind == 1 ? pq[j] : 0;
    for (int r = 0; r < m - 1; ++r) {
      const int cw = ew, ck = ek, cj = ej;
      const int rn = r + 1 < m - 1 ? (r + 1) * 16 : 0;
      ew = pq[rn + (wl & 15)];
      ek = pq[rn + k];
      if (kind == 1) ej = pq[rn + j];
      if (wl < npair) {
        const int p = cw & 255, q = cw >> 8;
        double c = 1.0, s = 0.0;
        cplx<double> ph = mk(1.0, 0.0);
        if (q != 255) {
          const cplx<double> g = cur[p + JLD * q];
          const double ag2 = g.x * g.x + g.y * g.y;
          const double app = cur[p + JLD * p].x, aqq = cur[q + JLD * q].x;
          if (ag2 > 1e-30 * fabs(app * aqq) && ag2 > gfloor2) {
            const double rag = rsqrt(ag2);   // 1 / |A_pq|
            const double tau = (aqq - app) * (0.5 * rag);   // |tau| < 1e16 by the floor
            const float tf = fabsf((float)tau);
            double t = (double)__builtin_amdgcn_rcpf(tf + __builtin_amdgcn_sqrtf(1.0f + tf * tf));
            const double at = fabs(tau);
            // t^2 + 2 |tau| t - 1 = 0; 4e-7 -> 1.2e-13 -> 1.7e-16 relative
            const double h = (double)__builtin_amdgcn_rcpf(2.0f * ((float)t + tf));
            t -= fma(t, t + 2.0 * at, -1.0) * h;
            t -= fma(t, t + 2.0 * at, -1.0) * h;
            if (tau < 0.0) t = -t;
            c = rsqrt(1.0 + t * t);
            s = t * c;
            ph = mk(g.x * rag, -g.y * rag);   // e^{-i phi}
          }
        }
        rcs[wave][wl] = mk(c, s);
        rph[wave][wl] = ph;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if (kind == 1) {
        const int p = ck & 255, q = ck >> 8, p2 = cj & 255, q2 = cj >> 8;
        const bool qv = q != 255, q2v = q2 != 255;
        const cplx<double> z = mk(0.0, 0.0);
        cplx<double> b00 = cur[p + JLD * p2];
        cplx<double> b01 = q2v ? cur[p + JLD * q2] : z;
        cplx<double> b10 = qv ? cur[q + JLD * p2] : z;
        cplx<double> b11 = (qv && q2v) ? cur[q + JLD * q2] : z;
        const cplx<double> cs = rcs[wave][k], cs2 = rcs[wave][j];
        if (cs2.y != 0.0) {   // columns p2, q2
          const cplx<double> ph2 = rph[wave][j];
          jac_rot(b00, b01, cs2.x, cs2.y, ph2);
          jac_rot(b10, b11, cs2.x, cs2.y, ph2);
        }
        if (cs.y != 0.0) {    // rows p, q: e^{i phi}
          const cplx<double> phc = mk(rph[wave][k].x, -rph[wave][k].y);
          jac_rot(b00, b10, cs.x, cs.y, phc);
          jac_rot(b01, b11, cs.x, cs.y, phc);
        }
        nxt[p + JLD * p2] = b00;
        if (q2v) nxt[p + JLD * q2] = b01;
        if (qv) nxt[q + JLD * p2] = b10;
        if (qv && q2v) nxt[q + JLD * q2] = b11;
      } else if (kind == 2) {
        const cplx<double> cs = rcs[wave][k];
        if (cs.y != 0.0) {
          const int p = ck & 255, q = ck >> 8;
          cplx<double> x0 = v[j + JLD * p], x1 = v[j + JLD * q];
          jac_rot(x0, x1, cs.x, cs.y, rph[wave][k]);
          v[j + JLD * p] = x0;
          v[j + JLD * q] = x1;
        }
      }
      __syncthreads();
      LDS_AS cplx<double>* t = cur;
      cur = nxt;
      nxt = t;
    }
    // would the next sweep rotate any pair?  (the rotations' own test on every pair)
    int any = 0;
    if (kind == 1) {
      // the blocks of round 0's pairs hold every entry once
      const int row[2] = {pq[k] & 255, pq[k] >> 8}, col[2] = {pq[j] & 255, pq[j] >> 8};
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int i = row[a], l = col[b];
          if (l != 255 && l > i) {
            const cplx<double> g = cur[i + JLD * l];
            const double ag2 = g.x * g.x + g.y * g.y;
            if (ag2 > 1e-30 * fabs(cur[i + JLD * i].x * cur[l + JLD * l].x) && ag2 > gfloor2) any = 1;
          }
        }
    }
    if (any) flag = 1;
    __syncthreads();
    const int again = flag;
    __syncthreads();
    if (!again) {
      converged = true;
      break;
    }
  }
  // eigenvalues: the diagonal; sort ascending (ties by index) with the vectors
  if (tid < n) dsort[tid] = cur[tid + JLD * tid].x;
  __syncthreads();
  if (tid < n) {
    const double d = dsort[tid];
    int r = 0;
    for (int j = 0; j < n; ++j) r += (dsort[j] < d || (dsort[j] == d && j < tid)) ? 1 : 0;
    rank[tid] = r;
    w[(long)blockIdx.x * n + r] = d;
  }
  __syncthreads();
  for (int t = tid; t < nn; t += NT) {
    const int i = t % n, j = t / n;
    const int r = rank[j];
    if (r < nvec) M[(long)r * lda + i] = v[i + JLD * j];
  }
  if (tid == 0 && info) info[blockIdx.x] = converged ? 0 : 1;
}

// Matrix b of the stack: inv(chol(Hermitian(A)).U) in place, strict lower triangle zeroed;
// info[b] (potrf) and info[nbatch + b] (trtri) as rocSOLVER would set them.
//
// Right-looking elimination on [A | I]: the row operations that bring A to upper triangular
// form turn I into L^-1, A = L D L^H, and inv(U) = L^-H D^-1/2.  A's part of row i is its
// columns j >= i and L^-1's the columns j < i (its diagonal is 1), so both share one n x n
// square, and one pass of n steps gives the inverse without U ever being stored.  Thread
// (ti, tj) of a 16 x 16 grid holds the entries (ti + 16 a, tj + 16 b) in registers from the
// load to the store; at step k the holders of row k publish it to an LDS row (two rows
// alternate), one barrier, then every thread updates its entries of the rows i > k in the
// columns j >= i and j <= k.  Both factors of a product are scaled by 1 / sqrt(A_kk), so
// nothing overflows that U and its inverse can hold.
//
// What bounds it is the chain of a step (LDS row, reciprocal root, update).  Separate passes
// for U and its inverse were 2 n steps; on 1024 threads, which one matrix above order 32
// took, a step also cost ~1 us in instructions issued for entries that are finished
// (a call with its
// synchronisation, n = 40: 83 us, now 48; n = 24: 58 us, now 33; the kernel alone 4.6 us to
// n = 16, 12.5 at n = 24).
template <int E>   // entries per thread along each axis, n <= 16 E
__global__ void __launch_bounds__(256) k_chol_inv_small(cplx<double>* __restrict__ A, long lda, long stride, int n,
                                                       int* __restrict__ info, int nbatch) {
  constexpr int G = 16;
  __shared__ cplx<double> rowbuf[2][SM_NMAX];
  __shared__ double rdiag[SM_NMAX];
  static_assert(G * E <= SM_NMAX, "row buffers");
  cplx<double>* M = A + (long)blockIdx.x * stride;
  const int tid = threadIdx.x, tj = tid % G, ti = tid / G;
  cplx<double> r[E][E];   // r[a][b]: entry (ti + G a, tj + G b)
#pragma unroll
  for (int a = 0; a < E; ++a)
#pragma unroll
    for (int b = 0; b < E; ++b) {
      const int i = ti + G * a, j = tj + G * b;
      cplx<double> v = mk(0.0, 0.0);
      if (j < n && i <= j) {
        v = M[(long)j * lda + i];
        if (i == j) v.y = 0.0;
      }
      r[a][b] = v;
    }
  int bad = 0;
  for (int k = 0; k < n; ++k) {
    const int buf = k & 1, ak = k / G;
    if (ti == k % G) {
#pragma unroll
      for (int a = 0; a < E; ++a)
        if (a == ak) {
#pragma unroll
          for (int b = 0; b < E; ++b) rowbuf[buf][tj + G * b] = r[a][b];
        }
    }
    __syncthreads();
    // the row reads are unconditional (every index is a valid LDS slot) so they issue together
    const double dkk = rowbuf[buf][k].x;
    cplx<double> m[E], x[E];
#pragma unroll
    for (int a = 0; a < E; ++a) m[a] = rowbuf[buf][ti + G * a];
#pragma unroll
    for (int b = 0; b < E; ++b) x[b] = rowbuf[buf][tj + G * b];
    if (!(dkk > 0.0)) {   // the same value on every thread: a uniform exit
      bad = k + 1;
      break;
    }
    const double rd = rsqrt(dkk);
    if (tid == 0) rdiag[k] = rd;
#pragma unroll
    for (int a = 0; a < E; ++a) m[a] = scal(rd, m[a]);
#pragma unroll
    for (int b = 0; b < E; ++b) x[b] = tj + G * b == k ? mk(rd, 0.0) : scal(rd, x[b]);
#pragma unroll
    for (int a = 0; a < E; ++a) {
      // tile rows wholly up to k are finished, tiles between k and the diagonal are zero:
      // skipped on every thread alike
      if (G * a + G - 1 <= k || G * a >= n) continue;
      const int i = ti + G * a;
#pragma unroll
      for (int b = 0; b < E; ++b) {
        if (b < a && G * b > k) continue;
        const int j = tj + G * b;
        if (i > k && (j >= i || j <= k)) {   // -= conj(m_i) x_j
          r[a][b].x = fma(-x[b].x, m[a].x, fma(-x[b].y, m[a].y, r[a][b].x));
          r[a][b].y = fma(-x[b].y, m[a].x, fma(x[b].x, m[a].y, r[a][b].y));
        }
      }
    }
  }
  const int bb = blockIdx.x;
  if (tid == 0) {
    info[bb] = bad;
    info[nbatch + bb] = 0;
  }
  if (bad) return;
  __syncthreads();   // rdiag
  // inv(U)_ji = conj(L^-1_ij) / sqrt(D_i), zeros below the diagonal
#pragma unroll
  for (int a = 0; a < E; ++a)
#pragma unroll
    for (int b = 0; b < E; ++b) {
      const int i = ti + G * a, j = tj + G * b;
      if (i >= n || j >= n) continue;
      const double rd = rdiag[i];
      M[(long)i * lda + j] = j < i ? mk(rd * r[a][b].x, -rd * r[a][b].y) : mk(j == i ? rd : 0.0, 0.0);
    }
}

int heev_small_batch(pw_ctx* c, int n, int nbatch, cplx<double>* A, long lda, long stride, double* d_w, int nvec,
                     int* d_info) {
  if (n < 1 || n > SM_NMAX || nbatch < 1) return set_error(c, PW_ERR_ARG, "heev_small_batch: order out of range");
  if (n <= 32) {
    // one thread per block of A and per pair of V
    const int npair = (n + 1) / 2, items = (npair * npair + 63) / 64 * 64 + npair * n;
    const size_t lds3 = 3 * (size_t)n * JLD * sizeof(cplx<double>);
    auto kern = items <= 128 ? k_heev_jacobi32<128> : items <= 192 ? k_heev_jacobi32<192>
              : items <= 512 ? k_heev_jacobi32<512> : k_heev_jacobi32<768>;
    const int nt = items <= 128 ? 128 : items <= 192 ? 192 : items <= 512 ? 512 : 768;
    hipLaunchKernelGGL(kern, dim3(nbatch), dim3(nt), lds3, c->stream, A, lda, stride, n, d_w, nvec, d_info);
    return hip_check(c, hipGetLastError(), "k_heev_jacobi32");
  }
  const size_t lds = 2 * (size_t)n * n * sizeof(cplx<double>);
  hipLaunchKernelGGL(k_heev_jacobi, dim3(nbatch), dim3(SM_NT), lds, c->stream, A, lda, stride, n, d_w, nvec, d_info);
  return hip_check(c, hipGetLastError(), "k_heev_jacobi");
}

int chol_inv_small_batch(pw_ctx* c, int n, int nbatch, cplx<double>* A, long lda, long stride, int* d_info) {
  if (n < 1 || n > SM_NMAX || nbatch < 1) return set_error(c, PW_ERR_ARG, "chol_inv_small_batch: order out of range");
  auto kern = n <= 16 ? k_chol_inv_small<1> : n <= 32 ? k_chol_inv_small<2>
            : n <= 48 ? k_chol_inv_small<3> : k_chol_inv_small<4>;
  hipLaunchKernelGGL(kern, dim3(nbatch), dim3(256), 0, c->stream, A, lda, stride, n, d_info, nbatch);
  return hip_check(c, hipGetLastError(), "k_chol_inv_small");
}

int small_dense_max_n() { return SM_NMAX; }

}  // namespace pw
