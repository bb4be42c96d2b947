// Several fixed-field steps of real walkers in one launch, forward and reverse.
#pragma once
#include "cp_kernels.hpp"

struct FfFusedArgs {
  int s0, s1;                // steps s0 .. s1-1 (reverse: from s1-1 down)
  int nw, M, N;              // one spin block, M x N per walker
  unsigned long long key;    // of the field stream
  double sigma, dt;          // +1 up, -1 down
  const zd* gamma;           // [M], real
  const zd* cdiag;           // [M] of the spin, real
  const double* B;           // M x M column-major: exp(-dt K)
  zd* W;                     // [nw][N][M]: forward: W; reverse: the adjoint of W
  double* Q;                 // forward: W before step s goes to Q + (s - q0) nw M N (nullptr: not kept); reverse reads
  int q0;
  // reverse only
  const zd* gprime;          // [M] d gamma / d U
  double* bpart;             // [slots][M][M] += sum over the slot's walkers and the steps of Wbar (D Q)^T
  double* upart;             // [slots][M] += Ubar
};
constexpr int FF_SLOTS = 512;  // partial sums of a reverse launch (as many as workgroups)
bool ff_fused_ok(int M, int N);
int launch_ff_forward(const FfFusedArgs& a, hipStream_t s);
int launch_ff_reverse(const FfFusedArgs& a, hipStream_t s);
// out[e] (+)= sum over slots of part[slot][e], as complex numbers without imaginary part
int launch_ff_sum(int slots, int per, const double* part, zd* out, int accumulate, hipStream_t s);
