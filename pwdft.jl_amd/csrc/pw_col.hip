// Launches of the column kernels (pw_col.h).
#include "pw_col.h"

namespace pw {

template <typename T>
static ColKernel<T> kernel_of(const pw_ctx* c, bool zhalf, bool fwd, int* chunk, size_t* lds) {
  if (c->tune_col_chunk > 0 || c->fft_order != 0) return nullptr;
  return zhalf ? col_kernel<T, true>(c->n3, fwd, chunk, lds) : col_kernel<T, false>(c->n3, fwd, chunk, lds);
}

template <typename T>
int col_chunk(const pw_ctx* c, bool zhalf) {
  int chunk = 0;
  size_t lds = 0;
  return kernel_of<T>(c, zhalf, false, &chunk, &lds) ? chunk : 0;
}

template <typename T>
static void launch(pw_ctx* c, bool zhalf, bool fwd, ColArgs<T>& A, long blocks) {
  int chunk = 0;
  size_t lds = 0;
  const ColKernel<T> kern = kernel_of<T>(c, zhalf, fwd, &chunk, &lds);
  if (!kern) return;
  if (blocks <= 0) blocks = (long)((A.ncol + chunk - 1) / chunk) * ((A.nb + 7) / 8 * 8);
  A.tw = reinterpret_cast<const cplx<T>*>(sizeof(T) == 8 ? c->d_tw64[2] : c->d_tw32[2]);
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), lds, c->stream, A);
}

template <typename T>
void col_inv(pw_ctx* c, const KData& k, const cplx<double>* psi, long ldpsi, int b0, int nb, cplx<T>* W) {
  ColArgs<T> A{};
  A.psi = psi;
  A.ldpsi = ldpsi;
  A.b0 = b0;
  A.nb = nb;
  A.W = W;
  A.ztab = k.d_ztab;
  A.ncol = k.ncol;
  launch<T>(c, k.zhalf, false, A, 0);
}

template <typename T>
void col_fwd(pw_ctx* c, const KData& k, const cplx<double>* psi, long ldpsi, cplx<double>* hpsi, long ldh, int b0,
             int nb, const cplx<T>* W, int kin, int acc) {
  ColArgs<T> A{};
  A.psi = psi;
  A.ldpsi = ldpsi;
  A.hpsi = hpsi;
  A.ldh = ldh;
  A.b0 = b0;
  A.nb = nb;
  A.W = const_cast<cplx<T>*>(W);
  A.ztab = k.d_ztab;
  A.gk2 = k.d_gk2;
  A.ncol = k.ncol;
  A.kin = kin;
  A.acc = acc;
  launch<T>(c, k.zhalf, true, A, 0);
}

template <typename T>
void col_inv_batch(pw_ctx* c, const KBatch* dkb, int nk, int nb, long blk, bool zhalf, cplx<T>* W) {
  ColArgs<T> A{};
  A.kb = dkb;
  A.nk = nk;
  A.nb = nb;
  A.W = W;
  launch<T>(c, zhalf, false, A, blk);
}

template <typename T>
void col_fwd_batch(pw_ctx* c, const KBatch* dkb, int nk, int nb, long blk, bool zhalf, const cplx<T>* W, int kin,
                   int acc) {
  ColArgs<T> A{};
  A.kb = dkb;
  A.nk = nk;
  A.nb = nb;
  A.W = const_cast<cplx<T>*>(W);
  A.kin = kin;
  A.acc = acc;
  launch<T>(c, zhalf, true, A, blk);
}

#define PW_COL_INST(T)                                                                                            \
  template int col_chunk<T>(const pw_ctx*, bool);                                                                 \
  template void col_inv<T>(pw_ctx*, const KData&, const cplx<double>*, long, int, int, cplx<T>*);                 \
  template void col_fwd<T>(pw_ctx*, const KData&, const cplx<double>*, long, cplx<double>*, long, int, int,       \
                           const cplx<T>*, int, int);                                                             \
  template void col_inv_batch<T>(pw_ctx*, const KBatch*, int, int, long, bool, cplx<T>*);                         \
  template void col_fwd_batch<T>(pw_ctx*, const KBatch*, int, int, long, bool, const cplx<T>*, int, int);
PW_COL_INST(double)
PW_COL_INST(float)
#undef PW_COL_INST

}  // namespace pw
