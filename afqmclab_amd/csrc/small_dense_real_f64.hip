// The small dense kernels on real working matrices (SmallDenseArgs::real), FP64 storage: a quarter
// of the complex multiply-adds and half of the registers and LDS, so more matrices share a CU.
#include "small_dense_kernels.hpp"

template <>
int small_dense_real<double>(int kind, const SmallDenseArgs& a, hipStream_t s) {
  return dispatch_registers<double, double>(kind, a, s);
}
