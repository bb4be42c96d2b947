// Exchange and background traces of the mixed estimator for real half-rotated Cholesky vectors.
#pragma once
#include "common.hpp"

struct PhExchangeArgs {
  int nw, L, Ns, G;
  const void* A;      // real T, [G][Ns][L]: A_g, L x Ns column-major
  const void* X;      // complex T, [nw][Ns][L]: X_w, L x Ns column-major
  zd* ex;             // [nw][G]
  void* bg;           // complex T, [nw][G]
  int accumulate;     // add to ex and bg (the second spin)
};
// D = A_g^T X_w:  ex[w][g] (+)= tr(D D), bg[w][g] (+)= tr(D), without D in memory.
// Takes any L and G and Ns <= 48 where X_w and a block of D fit the LDS (see the source file).
template <typename T>
bool ph_exchange_ok(int L, int Ns);
template <typename T>
int launch_ph_exchange(const PhExchangeArgs& a, hipStream_t s);
