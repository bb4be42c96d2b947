// Robust batched CholeskyQR in FP64 (see cholqr.hpp).
#include "cholqr.hpp"

#include <cstring>
#include <utility>

#include "gemm.hpp"
#include "small_dense.hpp"

namespace {

bool panels(const CholQrBlock& q) { return q.real && q.N <= WALKER_PANEL_NMAX; }

WalkerPanelArgs panel_args(const CholQrBlock& q, const void* W, const int* mask) {
  WalkerPanelArgs a;
  memset(&a, 0, sizeof(a));
  a.M = q.M; a.N = q.N; a.nw = q.nw;
  a.W = W; a.strideW = (long long)q.M * q.N;
  a.alive = mask;
  return a;
}

GemmArgs qr_gemm_base() {
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.alpha_re = 1.0;
  a.scale_group = 1;
  return a;
}

// S = W^H W (upper tiles only, Hermitian) for the walkers in mask
int gram(const CholQrBlock& q, const int* mask, hipStream_t s) {
  if (panels(q)) {
    WalkerPanelArgs a = panel_args(q, q.wf->p, mask);
    a.out = q.S; a.stride_out = (long long)q.N * q.N;
    return launch_walker_gram<double, double>(a, s);
  }
  GemmArgs a = qr_gemm_base();
  a.M = q.N; a.N = q.N; a.K = q.M; a.batch = q.nw;
  a.A = q.wf->p; a.lda = q.M; a.strideA = (long long)q.M * q.N;
  a.B = q.wf->p; a.ldb = q.M; a.strideB = (long long)q.M * q.N;
  a.C = q.S; a.ldc = q.N; a.strideC = (long long)q.N * q.N;
  a.alive = mask;
  a.herm = 1;
  // measured fastest for the Gram shapes: one 128x128 tile per matrix above 64 columns
  a.tile = q.N > 64 ? GEMM_TILE_128x128 : GEMM_TILE_64x64;
  return launch_cgemm<double>(OP_C, EPI_STORE, a, s);
}

// S <- R^{-1} with S = R^H R, ld = log sums, info = breakdown (or a Jacobi-scaled pivot <= pivot_tol),
// for the walkers in mask
int chol(const CholQrBlock& q, const int* mask, double pivot_tol, hipStream_t s) {
  SmallDenseArgs c;
  memset(&c, 0, sizeof(c));
  c.N = q.N; c.batch = q.nw; c.in = q.S; c.ld_in = q.N; c.stride_in = (long long)q.N * q.N;
  c.out = q.S; c.ld_out = q.N; c.stride_out = c.stride_in;
  c.logdet = q.ld; c.info = q.info; c.nsub = q.nsub; c.alive = mask; c.alive_div = 1;
  c.pivot_tol = pivot_tol;
  c.real = q.real;
  return launch_chol_inverse<double>(c, s);
}

// dst = src R^{-1} for the walkers in mask (R^{-1} upper triangular)
int times_rinv(const CholQrBlock& q, const void* src, void* dst, const int* mask, hipStream_t s) {
  if (panels(q)) {
    WalkerPanelArgs a = panel_args(q, src, mask);
    a.B = q.S; a.strideB = (long long)q.N * q.N; a.b_upper = 1;
    a.out = dst; a.stride_out = a.strideW;
    return launch_walker_times<double, double>(a, s);
  }
  GemmArgs g = qr_gemm_base();
  g.M = q.M; g.N = q.N; g.K = q.N; g.batch = q.nw;
  g.A = src; g.lda = q.M; g.strideA = (long long)q.M * q.N;
  g.B = q.S; g.ldb = q.N; g.strideB = (long long)q.N * q.N;
  g.C = dst; g.ldc = q.M; g.strideC = (long long)q.M * q.N;
  g.alive = mask;
  g.b_upper = 1;
  g.tile = GEMM_TILE_32x32;  // measured fastest for W R^{-1}
  return launch_cgemm<double>(OP_N, EPI_STORE, g, s);
}

// a further CholeskyQR of the walkers in `among` that are farther than tol from orthonormal:
// they are copied to tmp and multiplied back into wf (real ones in place), the others stay put
int refine(const CholQrBlock& q, const int* among, hipStream_t s) {
  int rc;
  if ((rc = gram(q, among, s))) return rc;
  if ((rc = launch_ortho_check(q.nw, q.N, q.S, among, q.tol, q.need, s))) return rc;
  if ((rc = chol(q, q.need, 0.0, s))) return rc;
  // an exactly zero column left after the shifted pass (Householder's R_kk = 0): the walker dies, and
  // leaves the shifted set so that the pass over it does not count the walker a second time
  if ((rc = launch_qr_kill(q.nw, q.need, q.flag, q.info, q.alive, q.sc, 0, s))) return rc;
  if (panels(q)) {  // in place
    if ((rc = times_rinv(q, q.wf->p, q.wf->p, q.need, s))) return rc;
  } else {
    if ((rc = launch_select_alive(q.nw, (long long)q.M * q.N, sizeof(zd), q.need, q.wf->p, q.tmp->p, s))) return rc;
    if ((rc = times_rinv(q, q.tmp->p, q.wf->p, q.need, s))) return rc;
  }
  return launch_logw_add_real(q.nw, q.logw, q.need, q.ld, nullptr, 0, q.m0, q.m1, s);
}

}  // namespace

int cholqr_f64(const CholQrBlock& q, hipStream_t s) {
  int rc;
  // pass 1, with the shifted Gram matrix for the walkers whose Cholesky broke down
  if ((rc = gram(q, q.alive, s))) return rc;
  // a scaled pivot below 1e-10 (condition number above about 1e5) takes the shifted pass
  if ((rc = chol(q, q.alive, 1e-10, s))) return rc;
  if ((rc = launch_qr_flag(q.nw, q.alive, q.info, q.flag, s))) return rc;
  if ((rc = gram(q, q.flag, s))) return rc;
  const double u = 1.1102230246251565e-16;  // 2^-53
  const double c = 11.0 * ((double)q.M * q.N + (double)q.N * (q.N + 1)) * u;
  if ((rc = launch_qr_shift(q.nw, q.N, q.S, q.flag, c, s))) return rc;
  if ((rc = chol(q, q.flag, 0.0, s))) return rc;
  // the shifted Gram matrix is positive definite unless the walker holds non-finite numbers
  if ((rc = launch_qr_kill(q.nw, q.flag, nullptr, q.info, q.alive, q.sc, 1, s))) return rc;
  if ((rc = times_rinv(q, q.wf->p, q.tmp->p, q.alive, s))) return rc;
  std::swap(*q.wf, *q.tmp);
  if ((rc = launch_logw_add_real(q.nw, q.logw, q.alive, q.ld, nullptr, 0, q.m0, q.m1, s))) return rc;
  // pass 2: every alive walker not yet orthonormal to tol; pass 3: shifted ones still not
  if (q.check_all && (rc = refine(q, q.alive, s))) return rc;
  return refine(q, q.flag, s);
}

// A block of 2048 walkers of 256 x 112: Gram matrix 186, factorisation 610, W R^-1 337, check 194 us, the
// passes over the masks (empty in an ordinary run) 5 us each: 1.4 ms (1024 walkers 0.75).  With FP64
// copies of all walkers and complex products 2048 of them took 4.2 ms.
int cholqr_real_f32(const CholQrBlock& q, const void* w32, void* out, void* gram32, int* mask, double check_tol,
                    hipStream_t s) {
  REQUIRE(panels(q), "real FP32 CholeskyQR: real walkers of at most %d columns", WALKER_PANEL_NMAX);
  const long long size = (long long)q.M * q.N, sq = (long long)q.N * q.N;
  int rc;
  // pass 1
  WalkerPanelArgs g = panel_args(q, w32, q.alive);
  g.out = q.S; g.stride_out = sq;
  if ((rc = launch_walker_gram<float, double>(g, s))) return rc;
  if ((rc = chol(q, q.alive, 1e-10, s))) return rc;
  if ((rc = launch_qr_flag(q.nw, q.alive, q.info, q.flag, s))) return rc;
  // flagged walkers: the shifted Gram matrix
  g.alive = q.flag;
  if ((rc = launch_walker_gram<float, double>(g, s))) return rc;
  const double c = 11.0 * ((double)q.M * q.N + (double)q.N * (q.N + 1)) * 1.1102230246251565e-16;
  if ((rc = launch_qr_shift(q.nw, q.N, q.S, q.flag, c, s))) return rc;
  if ((rc = chol(q, q.flag, 0.0, s))) return rc;
  if ((rc = launch_qr_kill(q.nw, q.flag, nullptr, q.info, q.alive, q.sc, 1, s))) return rc;
  // W R^-1 rounded to FP32
  WalkerPanelArgs t = panel_args(q, w32, q.alive);
  t.skip = q.flag;
  t.B = q.S; t.strideB = sq; t.b_upper = 1;
  t.out = out; t.stride_out = size;
  if ((rc = launch_walker_times<float, double>(t, s))) return rc;
  if ((rc = launch_logw_add_real(q.nw, q.logw, q.alive, q.ld, nullptr, 0, q.m0, q.m1, s))) return rc;
  // mask: the flagged walkers and those whose rounded result is beyond check_tol; they take W R^-1
  // on an FP64 copy (S still holds R^-1) and further passes there, and are rounded after those
  WalkerPanelArgs k = panel_args(q, out, q.alive);
  k.skip = q.flag;
  k.out = gram32; k.stride_out = sq;
  if ((rc = launch_walker_gram<float, float>(k, s))) return rc;
  if ((rc = launch_ortho_check_f32(q.nw, q.N, reinterpret_cast<const zf*>(gram32), q.alive, check_tol, mask, s,
                                   q.flag)))
    return rc;
  if ((rc = launch_convert_f32_f64_masked(w32, q.wf->p, size, q.nw, mask, s))) return rc;
  if ((rc = times_rinv(q, q.wf->p, q.wf->p, mask, s))) return rc;
  CholQrBlock r = q;
  r.flag = mask;  // a walker that dies leaves the mask
  for (int pass = 0; pass < 2; ++pass)
    if ((rc = refine(r, mask, s))) return rc;
  return launch_convert_f64_f32_masked(q.wf->p, out, size, q.nw, mask, s);
}

int cholqr_refine(const CholQrBlock& q, const int* among, hipStream_t s) { return refine(q, among, s); }
