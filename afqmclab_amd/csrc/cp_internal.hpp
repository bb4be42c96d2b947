// Internal state of the constraint-path propagator and its walker sets, and the batched GEMM /
// dense helpers that the step, the measurement and the adjoint share.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <complex>
#include <type_traits>
#include <cstring>
#include <vector>

#include "../../include/afqmc_mi355x.h"
#include "cp_kernels.hpp"
#include "gemm.hpp"
#include "group.hpp"
#include "real_gemm.hpp"
#include "runtime.hpp"
#include "small_dense.hpp"
#include "walker_panel.hpp"

using cd = std::complex<double>;

struct afqmc_cp_s {
  afqmc_ctx ctx = nullptr;
  int device = 0;  // destroy must not touch ctx, which may already be gone
  int L = 0, N = 0, Nup = 0, Ndn = 0, nblk = 1, dense = 1, fp32 = 0;
  int split_bf16 = 0;  // the propagation GEMM in split-BF16 products (precision 2)
  int Mb[2] = {0, 0}, Nb[2] = {0, 0}, row0[2] = {0, 0}, col0[2] = {0, 0};
  int decomp = 1, force_type = 0, diag_only = 1, maxw = 0;
  double dt = 0.01, cap = 1.5, log_half_L = 0.0, dtUSum = 0.0;
  zd trial_logw{0, 0};
  zd hop_logw[3];
  DevBuf<char> phiT[2], expK[3][2], wdkT[2];
  // Operators whose imaginary parts are all zero, found once at creation: the trial and the
  // propagators are then kept as real arrays too and their products take real_gemm.  real_ops: all
  // of them, K, gamma and the site constants are real, so that walkers stay real under every
  // operation of this propagator (afqmc_walkers_s::real).
  int real_phi = 0, real_expk[3] = {0, 0, 0}, real_ops = 0;
  DevBuf<char> real_buf;  // holds:
  char *phiTr[2] = {}, *expKr[3][2] = {}, *wdkTr[2] = {};
  DevBuf<zd> gamma, cdiag;
  DevBuf<double> U, mu, hx, hy, hz, cforce;
  DevBuf<DevScalars> sc;
  DevBuf<double> ubuf;
  // workspace
  DevBuf<char> ovl[2], scale[2], d2x2, qrS[2], qr64[2], qr64b[2];
  DevBuf<char> gjwork[2];  // FP64 working copies of the overlap matrices above 160 columns
  DevBuf<zd> ldet[2], qrld[2], logO, gpart[3][2], per_walker, site_acc, site_part, den;
  DevBuf<int> info[2], qrinfo[2], prefix, table, comb_num, qr_need, qr_flag, qr_mask;
  DevBuf<double> weight, comb_prob, force_rec;
  DevBuf<int> aux_rec, aux_in;
  int ntile[2] = {1, 1};
  int tile[3] = {GEMM_TILE_64x64, GEMM_TILE_64x64, GEMM_TILE_64x64};  // propagate, overlap, green
  std::vector<cd> h_gamma, h_cdiag;
  std::vector<cd> h_K;                                 // 2L x 2L, for energies from Green matrices
  std::vector<double> h_U, h_mu, h_hx, h_hy, h_hz;
  size_t esz() const { return fp32 ? sizeof(zf) : sizeof(zd); }
};

struct afqmc_walkers_s {
  afqmc_cp cp = nullptr;
  int device = 0;  // destroy must not touch cp, which may already be gone
  int nw = 0;
  DevBuf<char> wf[2], tmp[2];
  DevBuf<zd> logw, logw_tmp;
  DevBuf<int> alive;
  // the imaginary part of every walker element is zero: set where the host knows what it writes
  // (creation, upload, trial), kept by every operation of a propagator with real_ops
  int real = 0;
  long long wsize(int b) const { return (long long)cp->Mb[b] * cp->Nb[b]; }
};

// ------------------------------------------------------------------ helpers shared by the entry points
namespace cpi {

template <typename T>
void pack_block(const double* dense, int L2, int N, int r0, int c0, int Mb, int Nb, std::vector<cplx<T>>& out,
                long long off) {
  for (int j = 0; j < Nb; ++j)
    for (int i = 0; i < Mb; ++i) {
      const double* s = dense + 2 * ((long long)(r0 + i) + (long long)(c0 + j) * L2);
      out[off + i + (long long)j * Mb] = cmk<T>((T)s[0], (T)s[1]);
    }
}

// every imaginary part zero and every real part finite
template <typename T>
bool all_real(const cplx<T>* v, size_t n) {
  bool ok = true;
  for (size_t k = 0; k < n; ++k) ok = ok && v[k].im == (T)0 && std::isfinite(v[k].re);
  return ok;
}

template <typename T>
int upload_matrix_blocks(afqmc_cp cp, const double* dense, int cols, DevBuf<char>* dst, bool square) {
  const int L2 = 2 * cp->L;
  for (int b = 0; b < cp->nblk; ++b) {
    const int Mb = cp->Mb[b], Nb = square ? cp->Mb[b] : cp->Nb[b];
    const int c0 = square ? cp->row0[b] : cp->col0[b];
    std::vector<cplx<T>> h((size_t)Mb * Nb);
    pack_block<T>(dense, L2, cols, cp->row0[b], c0, Mb, Nb, h, 0);
    int rc = dst[b].alloc_bytes(h.size() * sizeof(cplx<T>));
    if (rc) return rc;
    HIP_TRY(hipMemcpy(dst[b].p, h.data(), h.size() * sizeof(cplx<T>), hipMemcpyHostToDevice));
  }
  return 0;
}

template <typename T>
GemmArgs gemm_base() {
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.alpha_re = 1.0;
  a.scale_group = 1;
  return a;
}

template <typename T>
int cp_gemm(afqmc_cp cp, int opa, int epi, const GemmArgs& a) {
  return launch_cgemm<T>(opa, epi, a, cp->ctx->stream);
}

// the matrix blocks' real parts appended to `out` (each block at a multiple of 16 bytes, its offset
// in off[b]) when every imaginary part is zero and every real part finite in T; else nothing
template <typename T>
bool append_real_blocks(afqmc_cp cp, const double* dense, int cols, bool square, std::vector<T>& out, size_t* off) {
  const int L2 = 2 * cp->L;
  std::vector<cplx<T>> h[2];
  for (int b = 0; b < cp->nblk; ++b) {
    const int Mb = cp->Mb[b], Nb = square ? cp->Mb[b] : cp->Nb[b];
    h[b].resize((size_t)Mb * Nb);
    pack_block<T>(dense, L2, cols, cp->row0[b], square ? cp->row0[b] : cp->col0[b], Mb, Nb, h[b], 0);
    if (!all_real(h[b].data(), h[b].size())) return false;
  }
  for (int b = 0; b < cp->nblk; ++b) {
    out.resize((out.size() + 3) / 4 * 4);
    off[b] = out.size();
    for (const cplx<T>& v : h[b]) out.push_back(v.re);
  }
  return true;
}

// The real copies of the trial, the propagators and (phiT^H K)^T, in one device buffer; sets real_phi,
// real_expk and *real_wdk.
template <typename T>
int upload_real_operators(afqmc_cp cp, const double* phiT, const double* const* mats, const double* wdkT, bool* real_wdk) {
  std::vector<T> h;
  size_t off[5][2] = {};
  cp->real_phi = append_real_blocks<T>(cp, phiT, cp->N, false, h, off[0]);
  for (int k = 0; k < 3; ++k) cp->real_expk[k] = append_real_blocks<T>(cp, mats[k], 2 * cp->L, true, h, off[1 + k]);
  *real_wdk = append_real_blocks<T>(cp, wdkT, cp->N, false, h, off[4]);
  if (h.empty()) return 0;
  int rc = cp->real_buf.alloc_bytes(h.size() * sizeof(T));
  if (rc) return rc;
  HIP_TRY(hipMemcpy(cp->real_buf.p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
  for (int b = 0; b < cp->nblk; ++b) {
    auto at = [&](int k) { return cp->real_buf.p + off[k][b] * sizeof(T); };
    cp->phiTr[b] = at(0);
    for (int k = 0; k < 3; ++k) cp->expKr[k][b] = at(1 + k);
    cp->wdkTr[b] = at(4);
  }
  return 0;
}

// Which of block b's products take a real kernel.  real: the imaginary parts of wf are zero.  The
// kernels of the others take the tile shapes afqmc_cp_s::tile.
template <typename T>
bool real_overlap(afqmc_cp cp, afqmc_walkers w, DevBuf<char>* wf, int b, int real, RealGemmArgs* r) {
  memset(r, 0, sizeof(*r));
  r->M = cp->Nb[b]; r->N = cp->Nb[b] * w->nw; r->K = cp->Mb[b]; r->op_t = 1; r->alpha = 1.0; r->b_real = real;
  r->A = cp->phiTr[b]; r->lda = cp->Mb[b];
  r->B = wf[b].p; r->ldb = cp->Mb[b];
  r->C = cp->ovl[b].p; r->ldc = cp->Nb[b];
  return cp->real_phi && real_gemm_ok<T>(*r);
}
template <typename T>
bool real_propagate(afqmc_cp cp, afqmc_walkers w, int which, DevBuf<char>* in, DevBuf<char>* out, bool scaled, int b,
                    int real, RealGemmArgs* r) {
  memset(r, 0, sizeof(*r));
  r->M = cp->Mb[b]; r->N = cp->Nb[b] * w->nw; r->K = cp->Mb[b]; r->alpha = 1.0; r->b_real = real;
  r->A = cp->expKr[which][b]; r->lda = cp->Mb[b];
  r->B = in[b].p; r->ldb = cp->Mb[b];
  r->C = out[b].p; r->ldc = cp->Mb[b];
  if (scaled) { r->scale = cp->scale[b].p; r->scale_group = cp->Nb[b]; r->scale_strideG = cp->Mb[b]; }
  return cp->real_expk[which] && !(std::is_same<T, float>::value && cp->split_bf16) && real_gemm_ok<T>(*r);
}
inline bool real_green(afqmc_cp cp, int b, int real) { return real && cp->Nb[b] <= WALKER_PANEL_NMAX; }

// overlap O_b = phiT_b^H W_b for all walkers ("giant" GEMM with shared A).  real: the imaginary
// parts of wf are zero.  A real trial takes real products (two per complex B element, one per
// real one, against three in FP32 and four in FP64).
template <typename T>
int overlap_gemm(afqmc_cp cp, afqmc_walkers w, DevBuf<char>* wf, int real = 0) {
  GroupFork fork;  // the blocks are independent: a grouped call launches them together
  for (int b = 0; b < cp->nblk; ++b) {
    fork.branch();
    RealGemmArgs r;
    if (real_overlap<T>(cp, w, wf, b, real, &r)) {
      int rc = launch_real_gemm<T>(r, cp->ctx->stream);
      if (rc) return rc;
      continue;
    }
    GemmArgs a = gemm_base<T>();
    a.M = cp->Nb[b]; a.N = cp->Nb[b] * w->nw; a.K = cp->Mb[b]; a.batch = 1;
    a.A = cp->phiT[b].p; a.lda = cp->Mb[b]; a.strideA = 0;
    a.B = wf[b].p; a.ldb = cp->Mb[b]; a.strideB = 0;
    a.C = cp->ovl[b].p; a.ldc = cp->Nb[b]; a.strideC = 0;
    a.tile = cp->tile[1];
    int rc = cp_gemm<T>(cp, OP_C, EPI_STORE, a);
    if (rc) return rc;
  }
  return 0;
}

// (real: the imaginary parts of the overlaps are zero)
template <typename T>
int gj_blocks(afqmc_cp cp, afqmc_walkers w, bool write_inverse, const int* alive, int real = 0) {
  GroupFork fork;  // the blocks are independent: a grouped call launches them together
  for (int b = 0; b < cp->nblk; ++b) {
    fork.branch();
    SmallDenseArgs s;
    memset(&s, 0, sizeof(s));
    s.N = cp->Nb[b]; s.batch = w->nw;
    s.in = cp->ovl[b].p; s.ld_in = cp->Nb[b]; s.stride_in = (long long)cp->Nb[b] * cp->Nb[b];
    s.out = cp->ovl[b].p; s.ld_out = s.ld_in; s.stride_out = s.stride_in;
    s.logdet = cp->ldet[b].p; s.info = cp->info[b].p; s.write_inverse = write_inverse ? 1 : 0;
    s.alive = alive; s.alive_div = 1;
    s.work = cp->gjwork[b].p;
    s.real = real;
    int rc = launch_gj_inverse<T>(s, cp->ctx->stream);
    if (rc) return rc;
  }
  return 0;
}

// X_b = W_b O_b^{-1} with green row-dot epilogue.  real: the imaginary parts of wf are zero and the
// operators are real (real_ops), so everything here is.
template <typename T>
int green_gemm(afqmc_cp cp, afqmc_walkers w, DevBuf<char>* wf, const int* alive, bool kinetic, int real = 0) {
  GroupFork fork;  // the blocks are independent: a grouped call launches them together
  for (int b = 0; b < cp->nblk; ++b) {
    fork.branch();
    if (real_green(cp, b, real)) {
      WalkerPanelArgs g;
      memset(&g, 0, sizeof(g));
      g.M = cp->Mb[b]; g.N = cp->Nb[b]; g.nw = w->nw;
      g.W = wf[b].p; g.strideW = w->wsize(b);
      g.B = cp->ovl[b].p; g.strideB = (long long)cp->Nb[b] * cp->Nb[b];
      g.alive = alive;
      g.P0 = cp->phiTr[b]; g.P2 = kinetic ? cp->wdkTr[b] : nullptr;
      g.partner_half = cp->dense ? cp->L : 0;
      g.out0 = cp->gpart[0][b].p; g.out1 = cp->dense ? cp->gpart[1][b].p : nullptr;
      g.out2 = kinetic ? cp->gpart[2][b].p : nullptr;
      int rc = launch_walker_green<T>(g, cp->ctx->stream);
      if (rc) return rc;
      continue;
    }
    GemmArgs a = gemm_base<T>();
    a.M = cp->Mb[b]; a.N = cp->Nb[b]; a.K = cp->Nb[b]; a.batch = w->nw;
    a.A = wf[b].p; a.lda = cp->Mb[b]; a.strideA = w->wsize(b);
    a.B = cp->ovl[b].p; a.ldb = cp->Nb[b]; a.strideB = (long long)cp->Nb[b] * cp->Nb[b];
    a.P0 = cp->phiT[b].p; a.P2 = kinetic ? cp->wdkT[b].p : nullptr; a.ldp = cp->Mb[b];
    a.partner_half = cp->dense ? cp->L : 0;
    a.out0 = cp->gpart[0][b].p; a.out1 = cp->dense ? cp->gpart[1][b].p : nullptr;
    a.out2 = kinetic ? cp->gpart[2][b].p : nullptr;
    a.alive = alive;
    a.tile = cp->tile[2];
    int rc = cp_gemm<T>(cp, OP_N, EPI_GREEN, a);
    if (rc) return rc;
  }
  return 0;
}

// W'_b = B_b diag(s) W_b  (all walkers, one GEMM per block).  real: the imaginary parts of the
// input are zero (and, where scaled, those of the scale: real_ops).  A real B_b takes real products.
template <typename T>
int propagate_gemm(afqmc_cp cp, afqmc_walkers w, int which, DevBuf<char>* in, DevBuf<char>* out, bool scaled,
                   int real = 0) {
  GroupFork fork;  // the blocks are independent: a grouped call launches them together
  for (int b = 0; b < cp->nblk; ++b) {
    fork.branch();
    RealGemmArgs r;
    if (real_propagate<T>(cp, w, which, in, out, scaled, b, real, &r)) {
      int rc = launch_real_gemm<T>(r, cp->ctx->stream);
      if (rc) return rc;
      continue;
    }
    GemmArgs a = gemm_base<T>();
    a.M = cp->Mb[b]; a.N = cp->Nb[b] * w->nw; a.K = cp->Mb[b]; a.batch = 1;
    a.A = cp->expK[which][b].p; a.lda = cp->Mb[b];
    a.B = in[b].p; a.ldb = cp->Mb[b];
    a.C = out[b].p; a.ldc = cp->Mb[b];
    if (scaled) {
      a.scale = cp->scale[b].p; a.scale_group = cp->Nb[b]; a.scale_strideG = cp->Mb[b]; a.scale_strideB = 0;
    }
    a.tile = cp->tile[0];
    a.split_bf16 = std::is_same<T, float>::value ? cp->split_bf16 : 0;
    int rc = cp_gemm<T>(cp, OP_N, EPI_STORE, a);
    if (rc) return rc;
  }
  return 0;
}

// the walker step with each alive walker's aux fields written to aux_dev ([nw][L], device)
int step_record(afqmc_cp cp, afqmc_walkers w, int* aux_dev);
// cp->den[w] = the mixed-estimator weight of walker w (all walkers; dead ones are masked by the user)
int mixed_weight(afqmc_cp cp, afqmc_walkers w);
// SD::stabilize of every alive walker, enqueued without synchronising
int stabilize(afqmc_cp cp, afqmc_walkers w);

}  // namespace cpi
