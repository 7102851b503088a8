// Shared by the tile kernels of the dense filter gradient (bwd_filter_dense_tiles.hip,
// bwd_filter_dense_direct.hip).
#ifndef CP4_DENSE_TILES_H
#define CP4_DENSE_TILES_H

#include "cp4_internal.h"

namespace cp4 {

// A workgroup's tiles.  Workgroups go to the chip's eight dies in turn (blockIdx & 7), each die
// with an L2 of its own: a die takes one contiguous eighth of the tiles and its workgroups
// stride through it, so that tiles which share halo rows and columns run on the same die at
// about the same time (tile t, t + 1 on neighbouring dies: every halo cell is fetched once
// per die that needs it, 1.7 - 1.9 times the input in all).
struct TileRange {
  int first, end, step;
};
__device__ __forceinline__ TileRange tiles_of_workgroup(int ntiles) {
  const int dies = gridDim.x < 8 ? (int)gridDim.x : 8;            // (fewer than eight workgroups: a range each)
  const int die = blockIdx.x % dies, slot = blockIdx.x / dies;
  const int on_die = ((int)gridDim.x - die + dies - 1) / dies;     // workgroups on this die
  TileRange r;
  r.first = (int)((long)ntiles * die / dies) + slot;
  r.end = (int)((long)ntiles * (die + 1) / dies);
  r.step = on_die;
  return r;
}

// The tile kernel that takes dy straight from memory: workgroups (partial sets) for a shape, 0 if it
// does not take it; aligned16: x, dy and act_y on 16-byte boundaries.
int dense_direct_sets(const cp4_shape&, bool aligned16);
// `sets` of them; act_y, act_bits, dbias, bias_part as in the masked builds of the other.
hipError_t dense_direct_launch(const BwdFilterArgs&, float* partial, int sets, hipStream_t);

}  // namespace cp4
#endif
