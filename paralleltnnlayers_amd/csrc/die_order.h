// One order of the work over the chip's eight dies for kernels that read the same operands one after
// the other: die d (workgroup index & 7, where the grid's first dimension is a multiple of eight) takes the
// d-th contiguous eighth of the images.  What a kernel has read stays in its die's L2 for the next one, up to
// 32 MB on all dies (24 MB read again by the same die 2.1 us, by another 4.8; written data is not
// found again either way).
#ifndef CP4_DIE_ORDER_H
#define CP4_DIE_ORDER_H

#include <hip/hip_runtime.h>

namespace cp4 {

// The first dimension of a grid for `count` workgroups.
inline unsigned die_grid(long count) { return (unsigned)((count + 7) / 8 * 8); }
// The place of workgroup `wg` of such a grid among the `count`; -1: none.
__device__ __forceinline__ int die_place(int wg, int count) {
  const int die = wg & 7, j = wg >> 3, base = count >> 3, rest = count & 7;
  if (j >= base + (die < rest)) return -1;
  return die * base + (die < rest ? die : rest) + j;
}


// The same with the order chosen by the host, without a branch: four numbers that one scalar load brings.
struct DieOrder {
  int mask, shift, base, rest;                           // {0, 0, count, 0}: in turn
};
inline DieOrder die_order(long count, bool dies) {
  return dies ? DieOrder{7, 3, (int)(count >> 3), (int)(count & 7)} : DieOrder{0, 0, (int)count, 0};
}
__device__ __forceinline__ int die_place(int wg, const DieOrder& o) {
  const int die = wg & o.mask, j = wg >> o.shift;
  return j < o.base + (die < o.rest) ? die * o.base + (die < o.rest ? die : o.rest) + j : -1;
}

}  // namespace cp4
#endif
