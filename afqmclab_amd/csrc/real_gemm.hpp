// GEMM with a real A and complex or real B on MFMA (gfx950):
//
//   C = alpha * op(A) * diag(s_g) * B  (+ C)        op in {N, T}
//
// A is a plain real array (element type T), shared by every column of B.  B and C hold complex
// numbers; with b_real every imaginary part of B (and of the scale) is zero, so only the real parts
// are multiplied and C gets zero imaginary parts.  Used wherever an operator of the model is real:
// exp(-dt K) of a real hopping matrix, a real trial, real half-rotated Cholesky vectors.
#pragma once
#include "common.hpp"

struct RealGemmArgs {
  int M, N, K, op_t;                // op_t: A is K x M column-major (op T), else M x K
  const void* A; long long lda;
  const void* B; long long ldb;
  void* C; long long ldc;
  double alpha;
  int beta_one;
  int b_real;
  // optional row scaling of B: s = scale + (n / scale_group) * scale_strideG (complex T)
  const void* scale; long long scale_strideG; int scale_group;
  int n_fastest;                    // as GemmArgs::n_fastest
};

// whether the kernel takes these operands (its byte offsets from a tile's operand bases are 32-bit)
template <typename T>
bool real_gemm_ok(const RealGemmArgs& a);
template <typename T>
int launch_real_gemm(const RealGemmArgs& a, hipStream_t s);
