// Per-walker products of real walkers (complex storage whose imaginary parts are all zero): each
// workgroup works on one walker's M x N matrix W, with the N x N factor in LDS.
//
//   walker_green   row dots of X = W B with the trial, as the Green epilogue of gemm.hpp writes them
//   walker_times   W' = W B (B optionally upper triangular; W' may be W)
//   walker_gram    S = W^T W
//
// TS is the walkers' storage type, TC the type of the products and sums.
#pragma once
#include "common.hpp"

constexpr int WALKER_PANEL_NMAX = 128;  // columns; wider walkers take the general kernels

struct WalkerPanelArgs {
  int M, N, nw;
  const void* W; long long strideW;  // cplx<TS>, M x N column-major per walker
  const void* B; long long strideB;  // cplx<TB>, N x N column-major per walker
  int b_upper;
  const int* alive;                  // walkers with alive[w] == 0 are skipped (nullptr: none)
  const int* skip;                   // and those with skip[w] != 0 (nullptr: none)
  // walker_times / walker_gram
  void* out; long long stride_out;   // cplx<TS> M x N, or cplx<TC> N x N
  // walker_green: real partners (element type TS, M x N) and partial sums as GemmArgs::P0, P2,
  // partner_half, out0, out1, out2
  const void* P0; const void* P2;
  int partner_half;
  zd* out0; zd* out1; zd* out2;
};

template <typename T> int launch_walker_green(const WalkerPanelArgs& a, hipStream_t s);
// TB: storage type of B; the products are formed in TB
template <typename TS, typename TB> int launch_walker_times(const WalkerPanelArgs& a, hipStream_t s);
template <typename TS, typename TC> int launch_walker_gram(const WalkerPanelArgs& a, hipStream_t s);
