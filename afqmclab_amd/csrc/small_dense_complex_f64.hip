// The small dense kernels on complex working matrices, FP64 storage.
#include "small_dense_kernels.hpp"

template <>
int small_dense_complex<double>(int kind, const SmallDenseArgs& a, hipStream_t s) {
  return dispatch_registers<double, zd>(kind, a, s);
}
