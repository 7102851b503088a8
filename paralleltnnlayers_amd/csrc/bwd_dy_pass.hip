// One pass over the output gradient of a layer behind a ReLU for everything in its backward that
// reads it: with dya = dy where y > 0 and Cc = the filtered rank planes of x,
//   G3[n,r,p] = sum_t FK[t,r] dya[n,t,p]     dFK[t,r] = sum_{n,p} dya[n,t,p] Cc[n,r,p]
//   dbias[t]  = sum_{n,p} dya[n,t,p]
// so dya never goes to memory.  (As passes of their own: the mask and the bias gradient read dy and y and
// write dya, the contraction and the gradient GEMM read it once each - five times the plane
// where this kernel moves two.)
//
// Bound by reading dy and y.  A workgroup takes chunks of 64 pixels of one image and all T
// channels (up to 256), a wave per 32 channels; eight waves a compute unit where the channel
// count allows (5 at 160 channels, 6 at 96 and 192, 7 at 224), each with a whole chunk's dy and y
// (64 registers) in flight while it works on the chunk before.  Rows move as 16 bytes a lane, 256
// contiguous bytes a channel.  A wave's 32 x 64 tile of dya lies in LDS, its own: read by rows
// (channel x 8 pixels) it is the A operand of the dFK product, read by columns (pixel x 8
// channels) the B operand of the contraction; exact fp32 products from three bf16 parts.  The
// contraction's partial sums over a wave's channels go over its tile, which nothing reads any
// more, and are added over the waves in order; Cc's fragments are split once a workgroup.  Two
// barriers a chunk.  dFK and the bias sums stay in registers over a workgroup's contiguous
// range of chunks: one partial set per workgroup, added in order by the caller's reduction.
// 248 registers with four waves and more; with two or three (64 and 96 channels), where a thread
// also holds two pieces of Cc, 256 and six of them in scratch memory.
// N32 T256 56x56 R32 (206 MB) in a training step, by kernel traces: 63 us, 3.3 TB/s of rows in 256-byte
// pieces; 66.9 with plain stores of G3, 69.9 with the factor's loads in branches as well.  With y's
// signs from the forward pass (BITS; 3 MB instead of y's 103) 50.7 us.
#include <algorithm>
#include <cstdint>

#include "cp4_internal.h"
#include "split_bf16.h"
#include "store_policy.h"

namespace cp4 {
namespace {

using split::f32x16;
using split::u32x4;

constexpr int kPix = 64;                 // pixels of a chunk
constexpr int kRow = kPix + 4;           // LDS row stride: 16-byte rows, four banks apart
constexpr int kTile = 32 * kRow;         // floats of a wave's tile
constexpr int kMaxWaves = 8;           // 256 channels
constexpr int kFrag = 4 * 3 * 2 * 32;    // 16-byte fragments of a chunk of Cc: [step][part][half][rank]

struct DyPassArgs {
  const float *dy, *y, *FK, *Cc;
  const unsigned short* bits;            // FwdArgs::save_mask of the forward; null: y
  float *G3, *partK, *partB;             // partB null: no bias gradient
  int T, R, HW, cpi, chunks;             // chunks per image and in all
  int lines;                             // G3's planes are whole cache lines
};

// KZ: (rank, octet) pairs of Cc a thread loads and splits (256 of them a chunk).
// BITS: y's signs from the forward pass, 16 channels of a pixel in 16 bits, instead of y.
template <int KZ, bool BITS>
__global__ __launch_bounds__(512, 2) void dy_pass_kernel(DyPassArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int lane = threadIdx.x & 63, l32 = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int T = a.T, R = a.R, HW = a.HW, c0 = 32 * wave;
  float* tile = lds + wave * kTile;
  u32x4* Zf = reinterpret_cast<u32x4*>(lds + waves * kTile);
  // workgroups of a die (blockIdx & 7): consecutive ranges
  const unsigned die = blockIdx.x & 7, per = gridDim.x >> 3, rest = gridDim.x & 7;
  const unsigned wg = die * per + (die < rest ? die : rest) + (blockIdx.x >> 3);
  const int i0 = (int)((long)a.chunks * wg / gridDim.x), i1 = (int)((long)a.chunks * (wg + 1) / gridDim.x);

  // This wave's rows of FK, split: the contraction's A operand (zero past the last rank).  Every
  // other wave takes them with the sign reversed and its partial sums are subtracted: the matrix
  // cores' sums come out low by a few hundredths of a unit in the last place whatever their sign, which
  // a sum over all pixels into the nearly cancelling factor gradients brings to the front
  // (N32 C256 T256 56x56 R32: G3's mean error 1.9e-8 of its deviation, 4e-11 with the signs reversed;
  // dFC 4.2e-6 of its norm off, 2.9e-7 with them).  With 3, 5 or 7 waves one wave's share of the drift is
  // left: dFC at N53 C128 T96 56x56 R32 1.0e-6, at N27 T224 4.0e-7.
  const float sign = wave & 1 ? -1.f : 1.f;
  float fk[2][8];
#pragma unroll
  for (int ch = 0; ch < 2; ++ch)
#pragma unroll
    for (int e = 0; e < 8; ++e)      // (clamped, not branched: sixteen branches waited for a load each)
      fk[ch][e] = a.FK[(size_t)(c0 + 16 * ch + 8 * hi + e) * R + (l32 < R ? l32 : 0)];

  // ---- loads: row 4 j + lane / 16 of the wave's channels, four pixels a lane ----
  const int lrow = lane >> 4, lcol = 4 * (lane & 15);
  float4 dv[8], yv[BITS ? 1 : 8], zv[KZ][2];
  uint2 bits[2];                     // BITS: the lane's four pixels, channels 4 j + lrow with even and with odd j
  // (clamped, not branched; values outside are dropped where they are used.  Cc's first: its
  // fragments are made before the rows are waited for)
  auto load_z = [&](int i) {
    const int n = i / a.cpi;
    const int p0 = (i - n * a.cpi) * kPix;
#pragma unroll
    for (int k = 0; k < KZ; ++k) {
      const int it = (threadIdx.x + k * blockDim.x) & 255, zr = it >> 3, pz = p0 + 8 * (it & 7);
      const float* z = a.Cc + ((size_t)n * R + (zr < R ? zr : 0)) * HW;
      zv[k][0] = *reinterpret_cast<const float4*>(z + (pz < HW ? pz : 0));
      zv[k][1] = *reinterpret_cast<const float4*>(z + (pz + 4 < HW ? pz + 4 : 0));
    }
  };
  auto row_at = [&](int i) {
    const int n = i / a.cpi;
    const int p = (i - n * a.cpi) * kPix + lcol;
    return ((size_t)n * T + c0 + lrow) * HW + (p < HW ? p : 0);
  };
  auto load_row = [&](size_t at, int j) {
    dv[j] = *reinterpret_cast<const float4*>(a.dy + at + (size_t)(4 * j) * HW);
    if constexpr (!BITS) yv[j] = *reinterpret_cast<const float4*>(a.y + at + (size_t)(4 * j) * HW);
  };
  auto load_bits = [&](int i) {
    const int n = i / a.cpi;
    const int p = (i - n * a.cpi) * kPix + lcol;
    const unsigned short* m = a.bits + ((size_t)n * (T >> 5) + wave) * 2 * HW + (p < HW ? p : 0);
    bits[0] = *reinterpret_cast<const uint2*>(m);
    bits[1] = *reinterpret_cast<const uint2*>(m + HW);
  };
  auto deposit_z = [&](int i) {
#pragma unroll
    for (int k = 0; k < KZ; ++k) {
      const int it = threadIdx.x + k * blockDim.x, zr = (it >> 3) & 31, zo = it & 7;
      const int pz = (i % a.cpi) * kPix + 8 * zo;
      const bool in0 = zr < R && pz < HW, in1 = zr < R && pz + 4 < HW;
      const float v[8] = {in0 ? zv[k][0].x : 0.f, in0 ? zv[k][0].y : 0.f, in0 ? zv[k][0].z : 0.f,
                          in0 ? zv[k][0].w : 0.f, in1 ? zv[k][1].x : 0.f, in1 ? zv[k][1].y : 0.f,
                          in1 ? zv[k][1].z : 0.f, in1 ? zv[k][1].w : 0.f};
      const unsigned flip = (i - i0) & 1 ? 0x80000000u : 0u;      // the chunk's sign, see accK
      float sv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) sv[e] = __uint_as_float(__float_as_uint(v[e]) ^ flip);
      if (it < 256) {
        u32x4 h, m, l;
        split::split8(sv, h, m, l);
        u32x4* dst = Zf + ((zo >> 1) * 6 + (zo & 1)) * 32 + zr;
        dst[0] = h;
        dst[64] = m;
        dst[128] = l;
      }
    }
  };
  // dFK, with the opposite sign after every other chunk (those chunks' Cc has it reversed), for
  // the same reason as above: a workgroup's chunks are one chain of sums.  (dFK of N32 C256 T256 56x56
  // R32: 4.3e-7 of its norm off without, 3.2e-7 with; N128 C128 T64: 6.8e-7, 3.4e-7.  No time: 57
  // shapes within 0.3 % of each other on the mean.)
  f32x16 accK = (f32x16)(0.f);
  float bs[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) bs[j] = 0.f;
  {                                  // (every workgroup has a chunk)
    load_z(i0);
    const size_t at = row_at(i0);
    if constexpr (BITS) load_bits(i0);
#pragma unroll
    for (int j = 0; j < 8; ++j) load_row(at, j);
  }
  u32x4 fh[2], fm[2], fl[2];
#pragma unroll
  for (int ch = 0; ch < 2; ++ch) {
#pragma unroll
    for (int e = 0; e < 8; ++e) fk[ch][e] = l32 < R ? sign * fk[ch][e] : 0.f;
    split::split8(fk[ch], fh[ch], fm[ch], fl[ch]);
  }
  deposit_z(i0);
  __syncthreads();
  for (int i = i0; i < i1; ++i) {
    const int n = i / a.cpi;
    const int p0 = (i - n * a.cpi) * kPix;
    // ---- the held rows behind the activation, into the tile ----
    // (the next chunk's row is requested as one goes to the tile; past the last, that one again)
    const bool in = p0 + lcol < HW;
    const int inext = i + 1 < i1 ? i + 1 : i;
    const size_t next = row_at(inext);
    load_z(inext);
    [[maybe_unused]] const uint2 held[2] = {bits[0], bits[1]};
    if constexpr (BITS) load_bits(inext);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float4 m = dv[j];
      // (a product, as dy * (y > 0): a non-finite dy at a clipped output stays visible)
      if constexpr (BITS) {
        // channel 4 j + lrow: bit 4 (j / 2) + lrow of its half's 16
        const unsigned sh = 4 * (j >> 1) + lrow;
        m.x *= (float)((held[j & 1].x >> sh) & 1u);
        m.y *= (float)((held[j & 1].x >> (sh + 16)) & 1u);
        m.z *= (float)((held[j & 1].y >> sh) & 1u);
        m.w *= (float)((held[j & 1].y >> (sh + 16)) & 1u);
      } else {
        m.x *= yv[j].x > 0.f ? 1.f : 0.f;
        m.y *= yv[j].y > 0.f ? 1.f : 0.f;
        m.z *= yv[j].z > 0.f ? 1.f : 0.f;
        m.w *= yv[j].w > 0.f ? 1.f : 0.f;
      }
      m.x = in ? m.x : 0.f;
      m.y = in ? m.y : 0.f;
      m.z = in ? m.z : 0.f;
      m.w = in ? m.w : 0.f;
      bs[j] += (m.x + m.y) + (m.z + m.w);
      *reinterpret_cast<float4*>(tile + (4 * j + lrow) * kRow + lcol) = m;
      load_row(next, j);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // ---- dFK: rows of the tile against Cc ----
    accK = -accK;
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const float* ap = tile + l32 * kRow + 16 * st + 8 * hi;
      const float4 a0 = *reinterpret_cast<const float4*>(ap);
      const float4 a1 = *reinterpret_cast<const float4*>(ap + 4);
      const float v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
      u32x4 ah, am, al;
      split::split8(v, ah, am, al);
      const u32x4* zp = Zf + (st * 6 + hi) * 32 + l32;
      accK = split::mfma_split(ah, am, al, zp[0], zp[64], zp[128], accK);
    }
    // ---- G3: FK against columns of the tile ----
    f32x16 accG[2];
#pragma unroll
    for (int pb = 0; pb < 2; ++pb) {
      // (the small partial products of both channel chunks before the large ones, so that most
      //  of the chain's roundings are small)
      f32x16 g = (f32x16)(0.f);
      u32x4 bh[2];
#pragma unroll
      for (int ch = 0; ch < 2; ++ch) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = tile[(16 * ch + 8 * hi + e) * kRow + 32 * pb + l32];
        u32x4 bm, bl;
        split::split8(v, bh[ch], bm, bl);
        g = split::mfma16(fl[ch], bh[ch], g);
        g = split::mfma16(fm[ch], bm, g);
        g = split::mfma16(fh[ch], bl, g);
        g = split::mfma16(fm[ch], bh[ch], g);
        g = split::mfma16(fh[ch], bm, g);
      }
      g = split::mfma16(fh[0], bh[0], g);
      accG[pb] = split::mfma16(fh[1], bh[1], g);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int pb = 0; pb < 2; ++pb)
#pragma unroll
      for (int v = 0; v < 16; ++v) tile[(16 * pb + v) * 64 + lane] = accG[pb][v];
    __syncthreads();              // partial sums complete; Cc's fragments read by every wave
    for (int k = wave; k < 32; k += waves) {
      // (all of an entry's reads together: one after the other they were 6 us of the kernel)
      float t[kMaxWaves], s = 0.f;
#pragma unroll
      for (int w = 0; w < kMaxWaves; ++w) t[w] = lds[(w < waves ? w : 0) * kTile + k * 64 + lane];
#pragma unroll
      for (int w = 0; w < kMaxWaves; ++w)
        if (w < waves) s = w & 1 ? s - t[w] : s + t[w];
      const int v = k & 15, r = 8 * (v >> 2) + 4 * hi + (v & 3);
      const int p = p0 + 32 * (k >> 4) + l32;
      if (r < R && p < HW) {
        float* g = a.G3 + ((size_t)n * R + r) * HW + p;
        if (a.lines) store_through(g, s);
        else *g = s;
      }
    }
    deposit_z(inext);
    __syncthreads();              // tiles free, the next chunk's fragments complete
  }
  // ---- one partial set per workgroup ----
  if ((i1 - i0 - 1) & 1) accK = -accK;
  float* pk = a.partK + ((size_t)wg * T + c0) * R;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int d = 8 * (v >> 2) + 4 * hi + (v & 3);
    if (l32 < R) pk[(size_t)d * R + l32] = accK[v];
  }
  if (a.partB) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float s = bs[j];
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) s += __shfl_down(s, off, 16);
      if ((lane & 15) == 0) a.partB[(size_t)wg * T + c0 + 4 * j + lrow] = s;
    }
  }
}

int grid_of(int N, int T, int HW) {
  const long chunks = (long)N * ((HW + kPix - 1) / kPix);
  const long wgs = (long)num_compute_units() * std::max(1, 8 / (T / 32));
  return (int)std::min(chunks, wgs);
}

}  // namespace

// 64 to 256 output channels in whole blocks of 32, ranks up to 32, rows that move as 16 bytes, and
// gain over the passes on their own: it saves the masked dy's way to memory and back, and pays for a
// second pass over the rank planes (Cc before the others), a launch, FK and a partial set per
// workgroup, and workgroups that sit out the last round of chunks.  The line, in us, fits
// 450 layers (T 64-256, R 1-32, filters 1-7, C 16-512, 17x17 to 240x240) timed both ways from two
// chunks a workgroup on; the choice is 0.2 % off the better one on the mean, 6.5 % at worst,
// the pass everywhere 1.5 and 19 % (N21 C64 T96 56x56 R16, two chunks a workgroup: 78 us, 70 apart;
// N63, six: 139, 155).
bool bwd_dy_pass_supported(int N, int T, int R, int HW) {
  if (T % 32 != 0 || T < 64 || T > 256 || R < 1 || R > 32 || HW % 4 != 0) return false;
  const long chunks = (long)N * ((HW + kPix - 1) / kPix);
  const long wgs = (long)num_compute_units() * std::max(1, 8 / (T / 32));
  if (chunks < 2 * wgs) return false;
  const double pixels = 1e-6 * N * HW;
  const double idle = 1e-6 * ((chunks + wgs - 1) / wgs * wgs - chunks) * kPix;
  return T * (1.7 * pixels - 0.75 * idle) - 2.1 * R * pixels > 11.6;
}
int bwd_dy_pass_sets(int N, int T, int HW) { return grid_of(N, T, HW); }

hipError_t bwd_dy_pass_launch(const float* dy, const float* y, const unsigned short* bits,
                              const float* FK, const float* Cc, float* G3, float* partK, float* partB,
                              int N, int T, int R, int HW, hipStream_t st) {
  if (!y) return hipErrorInvalidValue;
  DyPassArgs a{};
  a.dy = dy; a.y = y; a.bits = bits; a.FK = FK; a.Cc = Cc; a.G3 = G3; a.partK = partK; a.partB = partB;
  a.T = T; a.R = R; a.HW = HW;
  a.lines = store_policy(G3, HW * sizeof(float), (size_t)N * R * HW * sizeof(float), ~(size_t)0) == kStoreThrough;
  a.cpi = (HW + kPix - 1) / kPix;
  a.chunks = N * a.cpi;
  const int waves = T / 32;
  const size_t lds = (size_t)waves * kTile * sizeof(float) + kFrag * 16;
  auto k = bits ? (waves >= 4 ? dy_pass_kernel<1, true> : dy_pass_kernel<2, true>)
                : (waves >= 4 ? dy_pass_kernel<1, false> : dy_pass_kernel<2, false>);
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  k<<<grid_of(N, T, HW), 64 * waves, lds, st>>>(a);
  return hipGetLastError();
}

}  // namespace cp4
