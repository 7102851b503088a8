// Dense filter gradient with few input channels and up to 64 output channels, as in a network's
// first layer: dK[k][(c, i, j)] = sum over pixels of dy[k][p] x[c][p + (i, j)], exact fp32 products from
// three bf16 parts on v_mfma_f32_16x16x32_bf16 (the sums of bwd_filter_dense_tiles.hip, which
// stages both operands in LDS).
//
// Here dy, the large operand, goes from memory to the matrix cores through registers alone: a lane of
// the A operand holds one output channel and eight consecutive pixels, which are 32 contiguous bytes of
// dy, and a wave that takes all blocks of output channels and all columns of its 32 pixels reads
// every value once.  x, a few channels, lies in LDS with its halo, split, in two buffers.
//
// A persistent workgroup of eight waves walks over tiles of 8 x 32 pixels, a wave per row; per tile a wave
// puts the B fragments of its row together (five dwords a part, shifted where a column starts on an odd
// cell), then block by block of output channels masks, splits and multiplies the held dy and requests
// the same block of the next tile; x of the next tile is split into the other buffer; one barrier.
// The loop has no branch of its own in all this: behind the last tile its x is staged once more, into the
// buffer that nobody reads, and whether dy's sums are wanted is a build (SUMS).  Where a branch stood, code that
// reads a product or overwrites its addend could land right behind it, and the compiler leaves no wait for
// the matrix cores on such an edge; tests/test_matrix_waits_cpu.py walks the listing for it.
// A tile's products are added up apart and go to the accumulators in one correctly rounded
// addition, with x's sign reversed every other tile: the matrix cores' sums come out low by a little
// whatever their sign.
//
// Bound by reading dy: N16 C3 K64 224x224 (205 MB and 6 MB of signs) 49 us, 4.3 TB/s; with both operands
// through LDS 74 (24 M vector instructions, 96 for four values staged, where 12 M are spent here on
// everything).  The factor gradients of 96 layers of C 1-16, T 1-64, filters 1-5, 14x16 to 512x512
// 1.14 times as fast on the mean, none slower by more than the runs differ.
//
// MASK: dy counts everywhere (0) or where y > 0 - y itself (1) or its signs from the forward pass (2).  Its
// sums per channel may leave as the bias gradient's partial sets (SUMS; always there in the masked builds).
#include "dense_tiles.h"
#include "split_bf16.h"

namespace cp4 {
namespace {

using split::u32x2;
using split::u32x4;
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kTH = kWaves, kTW = 32;
constexpr int kSlots = 2;                    // groups of four cells of x a thread stages per tile
constexpr int kMaxBlocks = 15;               // 16 x 16 blocks of dK a wave holds (16: 23 registers in scratch)

struct DirectPlan {
  int tilesX, tilesY, ntiles;
  int XR, plane;                             // cells of a channel's rows; cells of a plane of parts
  unsigned chmagic;                          // ceil(2^32 / groups of four cells a channel)
  int stage;                                 // bytes of both buffers
};

__device__ __forceinline__ f32x4 mfma16x16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(split::bf16x8, a),
                                                 __builtin_bit_cast(split::bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 load16(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// FS: filter; RB: blocks of 16 output channels; CB: blocks of 16 columns (c, i, j).
template <int FS, int RB, int CB, int MASK, bool SUMS>
__global__ __launch_bounds__(kThreads, 2) void dense_direct_kernel(BwdFilterArgs a, DirectPlan pl,
                                                                   float* partial) {
  constexpr int PH = kTH + FS - 1, LEAD = FS > 1 ? 4 : 0, XS = kTW + 2 * LEAD;
  constexpr int PB = (RB + 1) / 2;                   // 16-byte pieces of signs: two blocks share one
  constexpr unsigned kOut = 0x80000000u;             // an offset past any image: the load returns zero
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, part = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.H, W = a.W, HW = H * W, T = a.T, C = a.C, NC = C * FS * FS;
  const int bits_image = ((T + 31) >> 5) * 2 * HW;   // 16-bit words of signs an image

  // this lane's column of every block: its first cell in a plane, for the wave's row
  int boff[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    int n = 16 * cb + l16;
    n = n < NC ? n : NC - 1;                         // (past the last: sums that are not kept)
    const int c = n / (FS * FS), tap = n - c * (FS * FS), i = tap / FS, j = tap - i * FS;
    boff[cb] = c * pl.XR + (wave + i) * XS + j + LEAD - a.pad + 8 * part;
  }
  // the cells of x this thread stages
  int xc[kSlots], xr[kSlots], xcol[kSlots];
  const int groups = C * PH * (XS / 4);
#pragma unroll
  for (int q = 0; q < kSlots; ++q) {
    const int g = tid + kThreads * q;
    const int c = C == 1 ? 0 : (int)__umulhi((unsigned)g, pl.chmagic), r = g - c * (PH * (XS / 4));
    xc[q] = g < groups ? c : -1;
    xr[q] = r / (XS / 4);
    xcol[q] = 4 * (r - xr[q] * (XS / 4));
  }

  f32x4 acc[RB][CB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
  [[maybe_unused]] float bs[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) bs[rb] = 0.f;

  struct Tile {
    int n, h0, w0;
  };
  const int per_image = pl.tilesX * pl.tilesY;
  auto tile_at = [&](int t) {
    const int n = t / per_image, rem = t - n * per_image, ty = rem / pl.tilesX;
    return Tile{__builtin_amdgcn_readfirstlane(n), __builtin_amdgcn_readfirstlane(kTH * ty),
                __builtin_amdgcn_readfirstlane(kTW * (rem - ty * pl.tilesX))};
  };

  // ---- dy: block rb of the wave's row of a tile; zeros past the image and past the last channel ----
  f32x4 dv[RB][2];
  [[maybe_unused]] f32x4 yv[MASK == 1 ? RB : 1][2];
  [[maybe_unused]] u32x4 bits[MASK == 2 ? PB : 1];
  const unsigned lofs = (unsigned)(l16 * HW + 8 * part) * 4u;
  [[maybe_unused]] const unsigned bofs = (unsigned)(((l16 >> 2) & 1) * HW + 8 * part) * 2u;
  auto load_block = [&](const Tile& tl, bool some, int rb) {
    const bool row = some && tl.h0 + wave < H;       // (the same for all lanes)
    const size_t img = (size_t)tl.n * T * HW;
    const __amdgpu_buffer_rsrc_t drs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.dy + img), 0, T * HW * 4, 0x00020000);
    const int at = row ? (tl.h0 + wave) * W + tl.w0 : 0;
    const unsigned soff = (unsigned)(16 * rb * HW + at) * 4u;
    const unsigned v0 = row && tl.w0 + 8 * part < W ? lofs : kOut;
    const unsigned v1 = row && tl.w0 + 8 * part + 4 < W ? lofs + 16u : kOut;
    dv[rb][0] = load16(drs, v0, soff);
    dv[rb][1] = load16(drs, v1, soff);
    if constexpr (MASK == 1) {
      const __amdgpu_buffer_rsrc_t yrs = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float*>(a.act_y + img), 0, T * HW * 4, 0x00020000);
      yv[rb][0] = load16(yrs, v0, soff);
      yv[rb][1] = load16(yrs, v1, soff);
    }
    if constexpr (MASK == 2) {
      // (past the row's end dy is zero, whatever the signs; past the image's last sign the descriptor's range is
      // checked dword by dword, so that the half of a load that lies before it arrives)
      if ((rb & 1) == 0) {
        const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<unsigned short*>(a.act_bits + (size_t)tl.n * bits_image), 0, bits_image * 2, 0x00020000);
        bits[rb >> 1] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(brs, row ? bofs : kOut, (unsigned)(rb * HW + at) * 2u, 0));
      }
    }
  };
  // ---- x: the tile and its halo, zeros outside the image ----
  f32x4 xv[kSlots];
  auto load_x = [&](const Tile& tl) {
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.x + (size_t)tl.n * C * HW), 0, C * HW * 4, 0x00020000);
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
      const int h = tl.h0 - a.pad + xr[q], w = tl.w0 - LEAD + xcol[q];
      const bool in = xc[q] >= 0 && (unsigned)h < (unsigned)H && (unsigned)w < (unsigned)W;
      xv[q] = load16(xrs, in ? (unsigned)(xc[q] * HW + h * W + w) * 4u : kOut, 0);
    }
  };
  auto deposit_x = [&](int buf, float sign) {
#pragma unroll
    for (int q = 0; q < kSlots; ++q)
      if (xc[q] >= 0) {
        const float v[4] = {sign * xv[q][0], sign * xv[q][1], sign * xv[q][2], sign * xv[q][3]};
        u32x2 h, m, l;
        split::split4(v, h, m, l);
        unsigned char* dst = lds + 2 * (size_t)(buf * 3 * pl.plane + xc[q] * pl.XR + xr[q] * XS + xcol[q]);
        *reinterpret_cast<u32x2*>(dst) = h;
        *reinterpret_cast<u32x2*>(dst + 2 * pl.plane) = m;
        *reinterpret_cast<u32x2*>(dst + 4 * pl.plane) = l;
      }
  };

  const TileRange tr = tiles_of_workgroup(pl.ntiles);
  if (tr.first < tr.end) {
    const Tile tl = tile_at(tr.first);
    load_x(tl);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) load_block(tl, true, rb);
    deposit_x(0, 1.f);
  }
  __syncthreads();
  float sign = 1.f;                                  // of the current tile's x
  int buf = 0;
  for (int t = tr.first; t < tr.end; t += tr.step) {
    const bool more = t + tr.step < tr.end;
    const Tile nxt = tile_at(more ? t + tr.step : t);
    load_x(nxt);
    // ---- B: cells off ... off + 7 of each plane, the dwords from off / 2 shifted by its parity ----
    u32x4 bh[CB], bm[CB], bl[CB];
    const unsigned* xp = reinterpret_cast<const unsigned*>(lds) + (buf * 3 * pl.plane >> 1);
    const int pw = pl.plane >> 1;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      const unsigned* p = xp + (boff[cb] >> 1);
      const unsigned shift = (unsigned)(boff[cb] & 1) * 16u;
      unsigned d[3][5];
#pragma unroll
      for (int i = 0; i < 5; ++i) {
        d[0][i] = p[i];
        d[1][i] = p[pw + i];
        d[2][i] = p[2 * pw + i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bh[cb][i] = __builtin_amdgcn_alignbit(d[0][i + 1], d[0][i], shift);
        bm[cb][i] = __builtin_amdgcn_alignbit(d[1][i + 1], d[1][i], shift);
        bl[cb][i] = __builtin_amdgcn_alignbit(d[2][i + 1], d[2][i], shift);
      }
    }
    // ---- A, block by block of output channels ----
    [[maybe_unused]] u32x4 held[MASK == 2 ? PB : 1];
    if constexpr (MASK == 2)
#pragma unroll
      for (int i = 0; i < PB; ++i) held[i] = bits[i];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = dv[rb][e >> 2][e & 3];
      // (a product, as dy * (y > 0): a non-finite dy at a clipped output stays visible)
      if constexpr (MASK == 1) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= yv[rb][e >> 2][e & 3] > 0.f ? 1.f : 0.f;
      }
      if constexpr (MASK == 2) {
        // channel 16 rb + l16: bit 8 (rb & 1) + 4 (l16 / 8) + l16 % 4 of its pixel's 16
        const unsigned at = 8 * (rb & 1) + 4 * (l16 >> 3) + (l16 & 3);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          v[e] *= (float)__builtin_amdgcn_ubfe(held[rb >> 1][e >> 1], at + 16 * (e & 1), 1);
      }
      if constexpr (SUMS) bs[rb] += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
      // (the blocks' loads stay apart: moved about, a step of N16 C3 K64 224x224 took 117 us instead of 111; beside
      // many accumulators arithmetic may move, or 40 registers go to scratch)
      __builtin_amdgcn_sched_barrier(RB * CB > 9 ? 15 : 0);
      u32x4 ah, am, al;
      split::split8(v, ah, am, al);
      load_block(nxt, more, rb);
      f32x4 p[CB];
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) p[cb] = mfma16x16(al, bh[cb], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) p[cb] = mfma16x16(am, bm[cb], p[cb]);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) p[cb] = mfma16x16(ah, bl[cb], p[cb]);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) p[cb] = mfma16x16(am, bh[cb], p[cb]);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) p[cb] = mfma16x16(ah, bm[cb], p[cb]);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) p[cb] = mfma16x16(ah, bh[cb], p[cb]);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int v4 = 0; v4 < 4; ++v4) acc[rb][cb][v4] = __builtin_fmaf(sign, p[cb][v4], acc[rb][cb][v4]);
    }
    sign = -sign;
    buf ^= 1;
    deposit_x(buf, sign);
    __syncthreads();
  }

  // ---- the waves' sums, in order through LDS: one partial set per workgroup ----
  float* red = reinterpret_cast<float*>(lds);
  if (SUMS && a.dbias) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float s = bs[rb];
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      if (part == 0) red[(wave * RB + rb) * 16 + l16] = s;
    }
    __syncthreads();
    if (tid < T) {
      float s[kWaves];
#pragma unroll
      for (int w = 0; w < kWaves; ++w) s[w] = red[w * RB * 16 + tid];
      a.bias_part[(size_t)blockIdx.x * T + tid] =
          ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    }
    __syncthreads();
  }
  float* out = partial + (size_t)blockIdx.x * T * NC;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    // accumulator element v: row 4 * (lane / 16) + v, column lane % 16 of its block
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[((wave * CB + cb) * 16 + 4 * part + v) * 16 + l16] = acc[rb][cb][v];
    __syncthreads();
    for (int e = tid; e < CB * 256; e += kThreads) {
      const int n = 16 * (e >> 8) + (e & 15), k = 16 * rb + ((e >> 4) & 15);
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) s += red[w * CB * 256 + e];
      if (k < T && n < NC) out[(size_t)k * NC + n] = s;
    }
    __syncthreads();
  }
}

bool make_direct_plan(const cp4_shape& s, DirectPlan* pl) {
  const int FS = (int)s.Y, C = (int)s.C, T = (int)s.T, PH = kTH + FS - 1, XS = kTW + (FS > 1 ? 8 : 0);
  const int NC = C * FS * FS, RB = (T + 15) / 16, CB = (NC + 15) / 16;
  if (s.W % 4 != 0 || RB > 4 || CB > 5 || RB * CB > kMaxBlocks) return false;
  const int groups = PH * (XS / 4);
  if (C * groups > kSlots * kThreads) return false;
  // (buffer offsets of an image's channels and of blocks past the last)
  if ((size_t)64 * s.H * s.W * sizeof(float) >= (1ull << 30)) return false;
  pl->tilesX = ((int)s.W + kTW - 1) / kTW;
  pl->tilesY = ((int)s.H + kTH - 1) / kTH;
  const long tiles = (long)s.N * pl->tilesX * pl->tilesY;
  if (tiles >= (1l << 30)) return false;
  pl->ntiles = (int)tiles;
  // channels two banks apart modulo four: a block's columns span two channels, whose reads then meet
  // no bank twice
  pl->XR = PH * XS + 4;
  pl->plane = (C * pl->XR + 16) / 8 * 8;             // (a column's reads end up to two cells past the last)
  pl->chmagic = (unsigned)((0x100000000ull + (unsigned)groups - 1) / (unsigned)groups);
  pl->stage = 2 * 6 * pl->plane;
  return true;
}

template <int FS, int RB, int CB>
hipError_t launch_blocks(const BwdFilterArgs& a, const DirectPlan& pl, float* partial, int sets, hipStream_t st) {
  if constexpr (RB * CB > kMaxBlocks) {
    return hipErrorInvalidValue;                     // (make_direct_plan refuses them)
  } else {
    const int bytes = kWaves * CB * 256 * 4;
    const size_t lds = pl.stage > bytes ? pl.stage : bytes;
    auto k = a.act_bits ? dense_direct_kernel<FS, RB, CB, 2, true>
             : a.act_y  ? dense_direct_kernel<FS, RB, CB, 1, true>
             : a.dbias  ? dense_direct_kernel<FS, RB, CB, 0, true> : dense_direct_kernel<FS, RB, CB, 0, false>;
    if (lds > 64 * 1024) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
    }
    k<<<sets, kThreads, lds, st>>>(a, pl, partial);
    return hipGetLastError();
  }
}
template <int FS, int CB>
hipError_t launch_cb(const BwdFilterArgs& a, const DirectPlan& pl, float* partial, int sets, hipStream_t st) {
  switch ((a.T + 15) / 16) {
    case 1: return launch_blocks<FS, 1, CB>(a, pl, partial, sets, st);
    case 2: return launch_blocks<FS, 2, CB>(a, pl, partial, sets, st);
    case 3: return launch_blocks<FS, 3, CB>(a, pl, partial, sets, st);
    default: return launch_blocks<FS, 4, CB>(a, pl, partial, sets, st);
  }
}

}  // namespace

int dense_direct_sets(const cp4_shape& s, bool aligned16) {
  DirectPlan pl;
  if (!aligned16 || s.Y != s.X || !(s.Y == 1 || s.Y == 3 || s.Y == 5) || s.pad > s.Y - 1 || s.N == 0 ||
      !fits_int_indexing((int)s.N, (int)s.H, (int)s.W) || !make_direct_plan(s, &pl))
    return 0;
  const int cus = num_compute_units();
  return pl.ntiles < cus ? pl.ntiles : cus;
}

hipError_t dense_direct_launch(const BwdFilterArgs& a, float* partial, int sets, hipStream_t st) {
  cp4_shape s{};
  s.N = a.N; s.C = a.C; s.T = a.T; s.H = a.H; s.W = a.W; s.pad = a.pad; s.Y = a.Y; s.X = a.X; s.Rank = a.R;
  DirectPlan pl;
  if (!make_direct_plan(s, &pl)) return hipErrorInvalidValue;
  const int CB = (a.C * a.Y * a.X + 15) / 16;
  if (a.Y == 1) return launch_cb<1, 1>(a, pl, partial, sets, st);
  if (a.Y == 5) {
    switch (CB) {
      case 2: return launch_cb<5, 2>(a, pl, partial, sets, st);
      case 4: return launch_cb<5, 4>(a, pl, partial, sets, st);
      default: return launch_cb<5, 5>(a, pl, partial, sets, st);
    }
  }
  switch (CB) {
    case 1: return launch_cb<3, 1>(a, pl, partial, sets, st);
    case 2: return launch_cb<3, 2>(a, pl, partial, sets, st);
    case 3: return launch_cb<3, 3>(a, pl, partial, sets, st);
    case 4: return launch_cb<3, 4>(a, pl, partial, sets, st);
    default: return launch_cb<3, 5>(a, pl, partial, sets, st);
  }
}

}  // namespace cp4
