// Backward of a layer's epilogue y = act(conv + bias): the output gradient behind the
// activation, dya = dy where y > 0 (ReLU), and the bias gradient dbias[t] = sum dya over
// images and pixels, in one pass over dy and y; and the element-type conversions of the
// layer's 16-bit activations where a pass runs in fp32.
//
// Bound by HBM: y and dy are read once and dya is written once, 16 bytes a lane (the rate of
// a copy: N32 T256 56x56 fp32, 308 MB, 52 us, N16 T64 224x224, 617 MB, 119 us; a comparison,
// a product and a sum one after the other took 136 and 460 us).  A channel's pixels of all
// images are cut into segments, one workgroup each: about eight workgroups per compute unit
// on large layers, at least four loads a lane on small ones.  Each segment leaves one
// partial bias sum, added in index order by a second small launch (none where a channel is
// one segment), so the result does not depend on scheduling.
#include <algorithm>

#include "cp4_internal.h"

namespace cp4 {
namespace {

constexpr int kThreads = 256;
constexpr int kBatch = 4;          // 16-byte pieces of dy (and of y) a lane has in flight

// Element types in memory and their value as fp32.
struct F32 {
  using raw = float;
  static __device__ __forceinline__ float up(raw v) { return v; }
  static __device__ __forceinline__ raw down(float v) { return v; }
};
struct BF16 {
  using raw = unsigned short;
  static __device__ __forceinline__ float up(raw v) { return __uint_as_float((unsigned)v << 16); }
  static __device__ __forceinline__ raw down(float v) {
    return __builtin_bit_cast(raw, static_cast<__bf16>(v));       // round to nearest even
  }
};
struct F16 {
  using raw = unsigned short;
  static __device__ __forceinline__ float up(raw v) {
    return (float)__builtin_bit_cast(_Float16, v);
  }
  static __device__ __forceinline__ raw down(float v) {
    return __builtin_bit_cast(raw, static_cast<_Float16>(v));     // round to nearest even
  }
};

// dy behind a ReLU: the product with the comparison's 0 or 1, so that an infinite or NaN
// gradient at a clipped output stays visible (NaN) to whoever watches the gradients for it.
__device__ __forceinline__ float masked(float d, float y) { return d * (y > 0.f ? 1.f : 0.f); }

// V elements at any element-aligned address (planes of an odd number of pixels start
// anywhere): one 16-byte access, which the memory pipeline takes at such addresses too.
template <class T, int V>
struct Piece {
  typedef typename T::raw vec __attribute__((ext_vector_type(V), aligned(sizeof(typename T::raw))));
  vec v;
};

struct ActGradArgs {
  const void *y, *dy;
  void* out;            // null: bias sums only
  float* part;          // [T][S]; null: no bias gradient
  int N, T, S;
  unsigned HW, U;       // pixels of a plane, pieces per plane (the last may be short)
  unsigned dn, dj;      // kThreads = dn * U + dj
};

template <class In, class Out, bool MASK>
__global__ __launch_bounds__(kThreads) void act_grad_kernel(ActGradArgs a) {
  constexpr int V = 16 / sizeof(typename In::raw);
  using InV = typename Piece<In, V>::vec;
  using OutV = typename Piece<Out, V>::vec;
  const int t = blockIdx.y, s = blockIdx.x;
  const typename In::raw* y = static_cast<const typename In::raw*>(a.y);
  const typename In::raw* dy = static_cast<const typename In::raw*>(a.dy);
  typename Out::raw* out = static_cast<typename Out::raw*>(a.out);
  const unsigned long long units = (unsigned long long)a.N * a.U;
  const unsigned long long u0 = units * s / a.S, u1 = units * (s + 1) / a.S;
  unsigned long long u = u0 + threadIdx.x;
  unsigned n = (unsigned)(u / a.U), j = (unsigned)(u - (unsigned long long)n * a.U);
  float sum = 0.f;
  while (u < u1) {
    InV vy[kBatch], vd[kBatch];
    size_t at[kBatch];
    unsigned left[kBatch];          // elements of the piece that exist (0: past the segment)
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      const bool in = u < u1;
      at[b] = in ? ((size_t)n * a.T + t) * a.HW + (size_t)j * V : 0;
      left[b] = in ? min((unsigned)V, a.HW - j * V) : 0u;
      if (left[b] == V) {
        vd[b] = *reinterpret_cast<const InV*>(dy + at[b]);
        if (MASK) vy[b] = *reinterpret_cast<const InV*>(y + at[b]);
      }
      u += kThreads;
      n += a.dn;
      j += a.dj;
      if (j >= a.U) {
        j -= a.U;
        ++n;
      }
    }
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      if (left[b] == V) {
        OutV o;
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const float d = In::up(vd[b][e]);
          const float m = MASK ? masked(d, In::up(vy[b][e])) : d;
          sum += m;
          o[e] = Out::down(m);
        }
        if (out) *reinterpret_cast<OutV*>(out + at[b]) = o;
      } else {
        for (unsigned e = 0; e < left[b]; ++e) {       // a plane's last, short piece
          const float d = In::up(dy[at[b] + e]);
          const float m = MASK ? masked(d, In::up(y[at[b] + e])) : d;
          sum += m;
          if (out) out[at[b] + e] = Out::down(m);
        }
      }
    }
  }
  if (!a.part) return;
  __shared__ float waves[kThreads / 64];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
  if ((threadIdx.x & 63) == 0) waves[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0)
    a.part[(size_t)t * a.S + s] = ((waves[0] + waves[1]) + waves[2]) + waves[3];
}

// dbias[t] = the S partial sums of channel t; a wave per channel.
__global__ __launch_bounds__(kThreads) void bias_sum_kernel(const float* __restrict__ part,
                                                            float* __restrict__ dbias, int T,
                                                            int S) {
  const int t = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T) return;
  float sum = 0.f;
  for (int s = lane; s < S; s += 64) sum += part[(size_t)t * S + s];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
  if (lane == 0) dbias[t] = sum;
}

template <class In, class Out>
__global__ __launch_bounds__(kThreads) void convert_kernel(const typename In::raw* __restrict__ src,
                                                           typename Out::raw* __restrict__ dst,
                                                           size_t n) {
  constexpr int V = 8;
  using InV = typename Piece<In, V>::vec;
  using OutV = typename Piece<Out, V>::vec;
  const size_t step = (size_t)gridDim.x * kThreads, pieces = n / V;
  const size_t first = (size_t)blockIdx.x * kThreads + threadIdx.x;
  for (size_t i = first; i < pieces; i += step) {
    const InV v = *reinterpret_cast<const InV*>(src + i * V);
    OutV o;
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] = Out::down(In::up(v[e]));
    *reinterpret_cast<OutV*>(dst + i * V) = o;
  }
  for (size_t i = pieces * V + first; i < n; i += step) dst[i] = Out::down(In::up(src[i]));
}

template <class In, class Out>
hipError_t launch_mask(const ActGradArgs& a, hipStream_t st) {
  const dim3 grid(a.S, a.T);
  if (a.y) act_grad_kernel<In, Out, true><<<grid, kThreads, 0, st>>>(a);
  else act_grad_kernel<In, Out, false><<<grid, kThreads, 0, st>>>(a);
  return hipGetLastError();
}

int vector_elems(int dtype) { return dtype == CP4_DTYPE_F32 ? 4 : 8; }

}  // namespace

int act_grad_segments(int N, int T, size_t HW, int dtype) {
  const size_t V = vector_elems(dtype), units = (size_t)N * ((HW + V - 1) / V);
  // a channel of up to two batches a lane stays one segment: no second launch
  if (units <= 2 * kBatch * kThreads) return 1;
  const size_t most = std::max<size_t>(1, (size_t)8 * num_compute_units() / T);
  return (int)std::min(most, units / (kBatch * kThreads));
}

hipError_t act_grad_launch(const void* y, const void* dy, void* out, int dtype, bool out_f32,
                           float* dbias, float* part, int N, int T, size_t HW, hipStream_t st) {
  const int V = vector_elems(dtype);
  ActGradArgs a{};
  a.y = y; a.dy = dy; a.out = out;
  a.N = N; a.T = T; a.S = act_grad_segments(N, T, HW, dtype);
  a.HW = (unsigned)HW;
  a.U = (unsigned)((HW + V - 1) / V);
  a.dn = kThreads / a.U;
  a.dj = kThreads % a.U;
  a.part = dbias ? (a.S == 1 ? dbias : part) : nullptr;
  hipError_t e;
  if (dtype == CP4_DTYPE_F32) e = launch_mask<F32, F32>(a, st);
  else if (dtype == CP4_DTYPE_BF16) e = out_f32 ? launch_mask<BF16, F32>(a, st) : launch_mask<BF16, BF16>(a, st);
  else e = out_f32 ? launch_mask<F16, F32>(a, st) : launch_mask<F16, F16>(a, st);
  if (e != hipSuccess || !dbias || a.S == 1) return e;
  bias_sum_kernel<<<(T + 3) / 4, kThreads, 0, st>>>(part, dbias, T, a.S);
  return hipGetLastError();
}

hipError_t convert_launch(const void* src, int src_dtype, void* dst, int dst_dtype, size_t n,
                          hipStream_t st) {
  if (n == 0) return hipSuccess;
  const size_t blocks = (n / 8 + kThreads) / kThreads;
  const unsigned grid = (unsigned)std::min<size_t>(blocks, (size_t)16 * num_compute_units());
  const auto* s16 = static_cast<const unsigned short*>(src);
  auto* d16 = static_cast<unsigned short*>(dst);
  const auto* s32 = static_cast<const float*>(src);
  auto* d32 = static_cast<float*>(dst);
  if (src_dtype == CP4_DTYPE_BF16 && dst_dtype == CP4_DTYPE_F32)
    convert_kernel<BF16, F32><<<grid, kThreads, 0, st>>>(s16, d32, n);
  else if (src_dtype == CP4_DTYPE_F16 && dst_dtype == CP4_DTYPE_F32)
    convert_kernel<F16, F32><<<grid, kThreads, 0, st>>>(s16, d32, n);
  else if (src_dtype == CP4_DTYPE_F32 && dst_dtype == CP4_DTYPE_BF16)
    convert_kernel<F32, BF16><<<grid, kThreads, 0, st>>>(s32, d16, n);
  else if (src_dtype == CP4_DTYPE_F32 && dst_dtype == CP4_DTYPE_F16)
    convert_kernel<F32, F16><<<grid, kThreads, 0, st>>>(s32, d16, n);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace cp4
