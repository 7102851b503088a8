// The type in which a kernel's activations lie in memory: float, or with CP4_IO16 a 16-bit
// type (1: bfloat16, 2: IEEE half precision), widened exactly as it is read and rounded to
// nearest even as it is written.  FwdArgs::x and y then point at 16-bit elements.
#ifndef CP4_ACT_IO_H
#define CP4_ACT_IO_H

#include <hip/hip_runtime.h>

namespace cp4 {
namespace {

#ifdef CP4_IO16
using io_t = unsigned short;
__device__ __forceinline__ float from_io(io_t v) {
#if CP4_IO16 == 2
  return (float)__builtin_bit_cast(_Float16, v);
#else
  return __uint_as_float((unsigned)v << 16);
#endif
}
__device__ __forceinline__ io_t to_io(float v) {
#if CP4_IO16 == 2
  return __builtin_bit_cast(unsigned short, static_cast<_Float16>(v));
#else
  return __builtin_bit_cast(unsigned short, static_cast<__bf16>(v));
#endif
}
__device__ __forceinline__ unsigned io_pair(float a, float b) {
  return (unsigned)to_io(a) | ((unsigned)to_io(b) << 16);
}
#else
using io_t = float;
__device__ __forceinline__ float from_io(io_t v) { return v; }
__device__ __forceinline__ io_t to_io(float v) { return v; }
#endif
constexpr int kIoBytes = (int)sizeof(io_t);

}  // namespace
}  // namespace cp4
#endif  // CP4_ACT_IO_H
