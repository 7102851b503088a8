// Rank -> channel expansion of planes in memory, dst[n,c,p] = sum_r F[c,r] Z[n,r,p]: the input
// gradient of a layer whose backward pass has G1 (the adjoint taps of FK^T dy) at hand, as the
// factor gradients do.  dx = FC G1 then reads R planes an image instead of contracting T
// channels of dy again.
//
// Bound by the stores of dst: C channels out against R ranks in.  A wave takes 32 * PX
// consecutive pixels (across images) and a slice of the channels; the lane that is column l of a
// matrix block holds PX neighbouring pixels, one in each of PX blocks, so that every store
// of a channel row is 16 bytes a lane, 512 contiguous bytes (PX = 4).  Z's pieces are loaded and
// split once per wave (exact products from three bf16 parts, like every contraction here), F's
// come from the cache and are split per block of 32 channels: no LDS, no barrier.  Waves of a
// workgroup share the pixels and differ in the channel slice where there are slices, and
// workgroups of one die (blockIdx & 7) take a contiguous range of the pixels, so that cache
// lines that two blocks share meet in one L2.
// N32 C256 56x56 R32 fp32 (103 MB written, 13 MB read): 26 us in a training step; the backward-data
// pass from dy takes 56.  dx goes to memory by store_policy.h: its training step 210.7 us with it
// streamed, 214.2 with plain stores; N32 C128 28x28 R16 bf16 5.3 -> 4.2 going through the L2.
// The factor gradients' four-launch variant and its strided and 16-bit siblings bring dx along
// wherever they run: 100 layers (fp32 and bf16, C and T 16-256, R 8-64 also beyond C and T, filters
// 1-5, stride 1 and 2) took 0.99 to 1.82 times as long with the pass of its own (C = T = 16, R 64,
// N16 160x160 bf16: 539 us against 316).
#include <cstdint>

#include "cp4_internal.h"
#include "reduce_sets.h"
#include "split_bf16.h"
#include "store_policy.h"

namespace cp4 {
namespace {

using split::f32x16;
using split::u32x4;

constexpr int kThreads = 256;

struct ExpandArgs {
  const float *F, *Z;          // [C][R], [N][R][HW]
  void* dst;                   // [N][C][HW]
  int C, R, HW;
  int cblocks;                 // blocks of 32 channels a wave takes
  int slices;                  // waves a block of pixels is shared by
  long pixels, items;          // N * HW; blocks of pixels * slices
  int rblocks;                 // workgroups in front that add partial sets up (a multiple of eight)
};

int reduce_blocks(const ReduceArgs& r) {
  int n = 0;
  for (int i = 0; i < 5; ++i) n += (r.count[i] + 63) / 64;
  return n;
}

struct ToF32 {
  using raw = float;
  static __device__ __forceinline__ raw down(float v) { return v; }
};
struct ToBF16 {
  using raw = unsigned short;
  static __device__ __forceinline__ raw down(float v) {
    return __builtin_bit_cast(raw, static_cast<__bf16>(v));
  }
};
struct ToF16 {
  using raw = unsigned short;
  static __device__ __forceinline__ raw down(float v) {
    return __builtin_bit_cast(raw, static_cast<_Float16>(v));
  }
};

// KC chunks of 16 ranks.  VEC: HW a multiple of PX and dst on a PX-element boundary, a lane's PX
// pixels are neighbours and move in one access; else they are 32 apart and move one by one
// (planes start at any address then, and a wider access off its own boundary is the slower:
// N16 C128 55x55 R32 28 us against 10.7).
template <class Out, int KC, int PX, bool VEC, int STORE>
__global__ __launch_bounds__(kThreads, 2) void rank_expand_kernel(ExpandArgs a, ReduceArgs sums) {
  // The factor gradients' partial sets, which the GEMM before left: in a launch of their own they waited for
  // loads while nothing else ran (us, expansion + sums, and both together: N32 C256 56x56 R32 26.5 + 6.8,
  // 28.7; N16 C128 T256 55x55 R32 stride 2 12.0 + 4.0, 13.1; N32 C128 28x28 R16 bf16 4.2 + 4.2, 4.5).
  __shared__ float part[kThreads / 64][64];
  if ((int)blockIdx.x < a.rblocks) {
    int block = blockIdx.x;
    for (int seg = 0; seg < 5; ++seg) {
      const int n = (sums.count[seg] + 63) >> 6;
      if (block < n) {
        reduce_sets_block(sums, seg, block, kThreads / 64, part);
        return;
      }
      block -= n;
    }
    return;
  }
  using raw = typename Out::raw;
  typedef float ZV __attribute__((ext_vector_type(PX)));
  typedef raw OV __attribute__((ext_vector_type(PX)));
  typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
  constexpr int NP = VEC ? 1 : PX;                           // accesses a row takes
  const int lane = threadIdx.x & 63, l32 = lane & 31, hi = lane >> 5;
  // workgroups of a die: consecutive ones
  const unsigned bid = blockIdx.x - a.rblocks, grid = gridDim.x - a.rblocks;
  const unsigned die = bid & 7, per = grid >> 3, rest = grid & 7;
  const unsigned wg = die * per + (die < rest ? die : rest) + (bid >> 3);
  const long item = (long)wg * (kThreads / 64) + (threadIdx.x >> 6);
  if (item >= a.items) return;
  const int slice = (int)(item % a.slices);
  const long g = item / a.slices * (32 * PX) + (VEC ? PX : 1) * l32;   // this lane's first pixel
  const int HW = a.HW, R = a.R, C = a.C;
  // (lanes past the last pixel keep a valid one for their loads and store nothing)
  bool live[NP];
  size_t zat[NP], oat[NP];
  {
    long n = (g < a.pixels ? g : a.pixels - 1) / HW;
    long p = (g < a.pixels ? g : a.pixels - 1) - n * HW;
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      live[q] = g + 32 * q < a.pixels;
      if (live[q])
        while (p >= HW) {
          p -= HW;
          ++n;
        }
      else {
        n = (a.pixels - 1) / HW;
        p = HW - (VEC ? PX : 1);
      }
      zat[q] = (size_t)n * R * HW + p;
      oat[q] = (size_t)n * C * HW + p;
      p += 32;
    }
  }
  // ---- this lane's pixels, split: B operands [chunk][pixel][part] ----
  u32x4 bh[KC][PX], bm[KC][PX], bl[KC][PX];
#pragma unroll
  for (int ch = 0; ch < KC; ++ch) {
    float v[PX][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int r = 16 * ch + 8 * hi + e;
      const float* z = a.Z + (size_t)(r < R ? r : R - 1) * HW;
      if constexpr (VEC) {
        const ZV t = *reinterpret_cast<const ZV*>(z + zat[0]);
#pragma unroll
        for (int q = 0; q < PX; ++q) v[q][e] = t[q];
      } else {
#pragma unroll
        for (int q = 0; q < PX; ++q) v[q][e] = z[zat[q]];
      }
    }
#pragma unroll
    for (int q = 0; q < PX; ++q) split::split8(v[q], bh[ch][q], bm[ch][q], bl[ch][q]);
  }
  // ---- channel blocks: F's rows are the A operand (zero past the last rank) ----
  auto load_f = [&](float (&f)[KC][8], int c0) {
    const int c = c0 + l32 < C ? c0 + l32 : C - 1;
    const float* fp = a.F + (size_t)c * R;
#pragma unroll
    for (int ch = 0; ch < KC; ++ch) {
      const int r0 = 16 * ch + 8 * hi;
      if (r0 + 8 <= R) {
        const f32x4u t0 = *reinterpret_cast<const f32x4u*>(fp + r0);
        const f32x4u t1 = *reinterpret_cast<const f32x4u*>(fp + r0 + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { f[ch][e] = t0[e]; f[ch][4 + e] = t1[e]; }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[ch][e] = r0 + e < R ? fp[r0 + e] : 0.f;
      }
    }
  };
  const int first = slice * a.cblocks * 32;
  const int last = first + a.cblocks * 32 < C ? first + a.cblocks * 32 : C;
  if (first >= last) return;
  raw* dst = static_cast<raw*>(a.dst);
  const __amdgpu_buffer_rsrc_t drs = __builtin_amdgcn_make_buffer_rsrc(
      a.dst, 0, STORE == kStoreThrough ? (int)(a.pixels * C * sizeof(raw)) : 0, 0x00020000);
  float f[KC][8];
  load_f(f, first);
  for (int c0 = first; c0 < last; c0 += 32) {
    f32x16 acc[PX];
#pragma unroll
    for (int q = 0; q < PX; ++q) acc[q] = (f32x16)(0.f);
    u32x4 ah[KC], am[KC], al[KC];
#pragma unroll
    for (int ch = 0; ch < KC; ++ch) split::split8(f[ch], ah[ch], am[ch], al[ch]);
    load_f(f, c0 + 32 < last ? c0 + 32 : c0);
    // (the small partial products of all ranks before the large ones, so that most of the chain's
    //  roundings are small)
#pragma unroll
    for (int ch = 0; ch < KC; ++ch)
#pragma unroll
      for (int q = 0; q < PX; ++q) {
        acc[q] = split::mfma16(al[ch], bh[ch][q], acc[q]);
        acc[q] = split::mfma16(am[ch], bm[ch][q], acc[q]);
        acc[q] = split::mfma16(ah[ch], bl[ch][q], acc[q]);
        acc[q] = split::mfma16(am[ch], bh[ch][q], acc[q]);
        acc[q] = split::mfma16(ah[ch], bm[ch][q], acc[q]);
      }
#pragma unroll
    for (int ch = 0; ch < KC; ++ch)
#pragma unroll
      for (int q = 0; q < PX; ++q) acc[q] = split::mfma16(ah[ch], bh[ch][q], acc[q]);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int c = c0 + 8 * (v >> 2) + 4 * hi + (v & 3);
      if (c >= C) continue;
      if constexpr (VEC) {
        OV o;
#pragma unroll
        for (int q = 0; q < PX; ++q) o[q] = Out::down(acc[q][v]);
        const size_t at = oat[0] + (size_t)c * HW;
        if (!live[0]) continue;
        if constexpr (STORE == kStoreThrough) {         // (below kStreamBytes: 32-bit offsets)
          typedef unsigned words __attribute__((ext_vector_type(sizeof(OV) / 4)));
          const words w = __builtin_bit_cast(words, o);
          if constexpr (sizeof(OV) == 16)
            __builtin_amdgcn_raw_buffer_store_b128(w, drs, (unsigned)at * sizeof(raw), 0, buffer_policy(STORE));
          else
            __builtin_amdgcn_raw_buffer_store_b64(w, drs, (unsigned)at * sizeof(raw), 0, buffer_policy(STORE));
        } else if constexpr (STORE == kStoreStreamed) {
          __builtin_nontemporal_store(o, reinterpret_cast<OV*>(dst + at));
        } else {
          *reinterpret_cast<OV*>(dst + at) = o;
        }
      } else {
#pragma unroll
        for (int q = 0; q < PX; ++q)
          if (live[q]) dst[oat[q] + (size_t)c * HW] = Out::down(acc[q][v]);
      }
    }
  }
}

template <class Out>
hipError_t launch(ExpandArgs a, const ReduceArgs& sums, hipStream_t st) {
  // four pixels a lane while the parts of its ranks leave room for four accumulators
  const int px = a.R <= 32 ? 4 : 2;
  const long blocks = (a.pixels + 32 * px - 1) / (32 * px);
  const int all = (a.C + 31) / 32;
  // channel slices until there are about eight waves per compute unit
  a.cblocks = all;
  while (a.cblocks > 1 && blocks * ((all + a.cblocks - 1) / a.cblocks) < 8l * num_compute_units())
    a.cblocks = (a.cblocks + 1) / 2;
  a.slices = (all + a.cblocks - 1) / a.cblocks;
  a.items = blocks * a.slices;
  const unsigned grid = (unsigned)((a.items + kThreads / 64 - 1) / (kThreads / 64));
  const bool vec = a.HW % px == 0 && reinterpret_cast<uintptr_t>(a.Z) % (4 * px) == 0 &&
                   reinterpret_cast<uintptr_t>(a.dst) % (sizeof(typename Out::raw) * px) == 0;
  const size_t plane = a.HW * sizeof(typename Out::raw);
  // (two-pixel pieces of 16-bit elements are a dword: plain)
  const int store = vec && px * sizeof(typename Out::raw) >= 8
                        ? store_policy(a.dst, plane, plane * (a.pixels / a.HW) * a.C, kStreamBytes) : kStorePlain;
#define CP4_EXPAND(KC_, PX_)                                                             \
  {                                                                                      \
    constexpr bool wide = PX_ * sizeof(typename Out::raw) >= 8;                          \
    auto k = !vec ? rank_expand_kernel<Out, KC_, PX_, false, kStorePlain>                \
             : store == kStoreStreamed ? rank_expand_kernel<Out, KC_, PX_, true, wide ? kStoreStreamed : kStorePlain> \
             : store == kStoreThrough ? rank_expand_kernel<Out, KC_, PX_, true, wide ? kStoreThrough : kStorePlain>   \
                                      : rank_expand_kernel<Out, KC_, PX_, true, kStorePlain>;              \
    k<<<a.rblocks + grid, kThreads, 0, st>>>(a, sums);                                                   \
  }
  if (a.R <= 16) CP4_EXPAND(1, 4)
  else if (a.R <= 32) CP4_EXPAND(2, 4)
  else if (a.R <= 48) CP4_EXPAND(3, 2)
  else CP4_EXPAND(4, 2)
#undef CP4_EXPAND
  return hipGetLastError();
}

}  // namespace

hipError_t rank_expand_reduce_launch(const float* F, const float* Z, void* dst, int dtype, int N, int C,
                                     int HW, int R, const ReduceArgs& sums, hipStream_t st) {
  if (R > 64) return hipErrorInvalidValue;         // (four chunks of ranks)
  ExpandArgs a{};
  a.F = F; a.Z = Z; a.dst = dst;
  a.C = C; a.R = R; a.HW = HW;
  a.pixels = (long)N * HW;
  a.rblocks = (reduce_blocks(sums) + 7) / 8 * 8;
  if (dtype == CP4_DTYPE_BF16) return launch<ToBF16>(a, sums, st);
  if (dtype == CP4_DTYPE_F16) return launch<ToF16>(a, sums, st);
  return launch<ToF32>(a, sums, st);
}

}  // namespace cp4
