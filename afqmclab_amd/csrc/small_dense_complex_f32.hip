// The small dense kernels on complex working matrices, FP32 storage.
#include "small_dense_kernels.hpp"

template <>
int small_dense_complex<float>(int kind, const SmallDenseArgs& a, hipStream_t s) {
  return dispatch_registers<float, zd>(kind, a, s);
}
