// out[i] = sum over the partial sets s of part[s][i], up to five segments in one launch: the last step
// of the factor gradients, alone (bwd_filter_mfma.hip) or beside the input gradient's expansion
// (rank_expand.hip).
#ifndef CP4_REDUCE_SETS_H
#define CP4_REDUCE_SETS_H

#include "cp4_internal.h"

namespace cp4 {

struct ReduceArgs {
  const float* part[5];
  float* out[5];
  int count[5], S[5];
};

// A workgroup owns 64 consecutive outputs of segment `seg`, from 64 * block on; its `waves` waves (4 or
// 16) each sum a part of the S partials in index order (sixteen loads in flight, eight added as a tree), then the
// parts are added in wave order: the result does not depend on timing.  part: 64 floats a wave.
__device__ __forceinline__ void reduce_sets_block(const ReduceArgs& a, int seg, int block, int waves,
                                                  float (*part)[64]) {
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int i = block * 64 + lane;
  const int count = a.count[seg], S = a.S[seg];
  if (block * 64 >= count) return;                         // whole workgroup
  const int shift = waves == 4 ? 2 : 4;                    // (a division is a third of a small sum's time)
  const int k0 = (int)((unsigned)S * q >> shift), k1 = (int)((unsigned)S * (q + 1) >> shift);
  float s = 0.f;
  if (i < count) {
    const float* p = a.part[seg] + i;
    const size_t stride = count;
    int k = k0;
    float s1 = 0.f;                                        // (two chains of sums, each half as long)
    for (; k + 16 <= k1; k += 16) {
      float v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = p[(size_t)(k + u) * stride];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        v[u] += v[u + 4];
        v[u + 8] += v[u + 12];
      }
      s += (v[0] + v[2]) + (v[1] + v[3]);
      s1 += (v[8] + v[10]) + (v[9] + v[11]);
    }
    for (; k + 8 <= k1; k += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = p[(size_t)(k + u) * stride];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] += v[u + 4];
      s += (v[0] + v[2]) + (v[1] + v[3]);
    }
    s += s1;
    // (the rest together too, the last set in place of those past it; none left: the same for a wave)
    if (k < k1) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = p[(size_t)(k + u < k1 ? k + u : k1 - 1) * stride];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += k + u < k1 ? v[u] : 0.f;
    }
  }
  part[q][lane] = s;
  __syncthreads();
  if (q == 0 && i < count) {
    float t = part[0][lane];
    if (waves == 4) t = (t + part[1][lane]) + (part[2][lane] + part[3][lane]);
    else for (int w = 1; w < waves; ++w) t += part[w][lane];
    a.out[seg][i] = t;
  }
}

// dst[n,c,p] = sum_r F[c,r] Z[n,r,p] (ranks up to 64), dst of a cp4_dtype, and the sums beside it in the same
// launch, in workgroups of their own.
hipError_t rank_expand_reduce_launch(const float* F, const float* Z, void* dst, int dtype, int N, int C,
                                     int HW, int R, const ReduceArgs&, hipStream_t);

}  // namespace cp4
#endif
