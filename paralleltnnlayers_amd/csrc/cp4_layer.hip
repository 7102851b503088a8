// C ABI of a whole layer, y = act(conv + bias): which passes a call needs, on which element
// type each runs, and where their intermediates lie in the caller's workspace.
#include <algorithm>
#include <array>
#include <map>
#include <mutex>

#include "cp4_internal.h"
#include "plan_memo.h"

namespace {

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Where the parts of a backward call lie in its workspace (byte offsets; a part that the
// call does not need has no bytes) and which passes run on 16-bit activations as they are.
struct BackwardPlan {
  bool dx16, filter16;       // dx / the factor gradients on the 16-bit activations (16-bit layers only)
  bool act16, act32;         // dy behind the activation is written in the layer's type / as fp32
  bool may_mask;             // the factor gradients may take the mask and the bias gradient along
  size_t act16_at, act32_at; // ... here
  size_t x32_at, dx32_at;    // widened x, fp32 dx before it is rounded
  size_t bias_at, pass_at;   // partial bias sums, the passes' own workspace
  size_t pass_bytes, total;
  size_t g1_bytes;           // of the passes' workspace, at its end: the call runs without them too
};

size_t elements(const cp4_shape& s, unsigned channels) {
  return (size_t)s.N * channels * s.H * s.W;
}
size_t out_elements(const cp4_shape& s, const cp4_geometry* g) {
  return (size_t)s.N * s.T * (g ? (size_t)g->out_h * g->out_w : (size_t)s.H * s.W);
}

BackwardPlan make_backward_plan(const cp4_shape& s, const cp4_geometry* g, int dtype, int act,
                                int wanted) {
  BackwardPlan p{};
  const bool half = dtype != CP4_DTYPE_F32;
  const bool dx = wanted & CP4_WANT_DX, filter = wanted & CP4_WANT_FACTORS;
  const size_t ny = out_elements(s, g), nx = elements(s, s.C);
  p.dx16 = half && dx && cp4_bf16_supported(&s, 1);
  p.filter16 = half && filter && cp4_bf16_backward_filter_supported(&s);
  // (the 16-bit factor gradients bring dx along on the reference's own geometry)
  p.dx16 = p.dx16 || (dx && p.filter16 && s.Y == s.X && 2 * s.pad + 1 == s.Y);
  const bool dx32 = half && dx && !p.dx16, filter32 = half && filter && !p.filter16;
  // (fp32 layers: the "16" part is dy in the layer's own type)
  p.act16 = act != CP4_ACT_NONE && (half ? p.dx16 || p.filter16 : dx || filter);
  p.act32 = dx32 || filter32;
  size_t at = 0;
  auto take = [&](bool needed, size_t bytes) {
    const size_t here = at;
    if (needed) at += align256(bytes);
    return here;
  };
  p.act16_at = take(p.act16, ny * (half ? 2 : 4));
  p.act32_at = take(p.act32, ny * 4);
  p.x32_at = take(filter32, nx * 4);
  p.dx32_at = take(dx32, nx * 4);
  const int seg = cp4::act_grad_segments((int)s.N, (int)s.T, ny / ((size_t)s.N * s.T), dtype);
  p.may_mask = !g && !half && filter && (act != CP4_ACT_NONE || (wanted & CP4_WANT_BIAS));
  size_t parts = p.may_mask && !dx ? std::max(seg, cp4::num_compute_units()) : seg > 1 ? seg : 0;
  if (filter && !filter32) parts = std::max(parts, cp4::layer_bias_sets(s, g));
  p.bias_at = take((wanted & CP4_WANT_BIAS) && parts, s.T * parts * 4);
  p.pass_at = at;
  if (g) p.pass_bytes = dx || filter ? cp4_conv2d_backward_ex_workspace_bytes(&s, g) : 0;
  else p.pass_bytes = filter ? cp4_conv2d_backward_filter_workspace_bytes(&s) : 0;
  p.total = at + align256(p.pass_bytes);
  // (room for G1 where the three-launch variant runs, which then brings dx along)
  if (!g && !half && dx && filter && cp4::layer_filter_forms_g1(s)) {
    p.pass_bytes = align256(p.pass_bytes);
    p.g1_bytes = align256((size_t)s.N * s.Rank * s.H * s.W * 4);
    p.total += p.g1_bytes;
  }
  return p;
}

using PlanKey = std::array<unsigned, 20>;
PlanKey plan_key(const cp4_shape& s, const cp4_geometry* g, int dtype, int act, int wanted) {
  const cp4_geometry none{0, 0, 0, 0, 0, 0};
  const cp4_geometry& gg = g ? *g : none;
  return {s.N, s.H, s.W, s.pad, s.T, s.C, s.Y, s.X, s.Rank, gg.stride_h, gg.stride_w,
          gg.pad_top, gg.pad_left, gg.out_h, gg.out_w, (unsigned)dtype, (unsigned)act,
          (unsigned)wanted, (unsigned)cp4::num_compute_units(), cp4::tuned_choices()};
}
template <class Plan, class Make>
Plan remembered(std::mutex& mu, std::map<PlanKey, Plan>& plans, const PlanKey& key, Make make) {
  static thread_local cp4::PlanMemo<PlanKey, Plan> memo;
  return memo.get(key, [&] {
    std::lock_guard<std::mutex> lk(mu);
    auto it = plans.find(key);
    if (it != plans.end()) return it->second;
    if (plans.size() > 4096) plans.clear();
    return plans[key] = make();
  });
}

// The plan of a call, remembered: planning asks the backward-filter kernels for theirs,
// several microseconds of host time that every step of a small layer would wait for.  (It
// depends on the device by its compute units, and on which variants were tuned.)
BackwardPlan backward_plan(const cp4_shape& s, const cp4_geometry* g, int dtype, int act,
                           int wanted) {
  static std::mutex mu;
  static std::map<PlanKey, BackwardPlan> plans;
  return remembered(mu, plans, plan_key(s, g, dtype, act, wanted),
                    [&] { return make_backward_plan(s, g, dtype, act, wanted); });
}

// Bytes of y's signs that a forward call leaves for its backward call; 0: none.
size_t make_keep_plan(const cp4_shape& s, const cp4_geometry* g, int dtype, int act, int wanted) {
  const bool filter = wanted & CP4_WANT_FACTORS, dx = wanted & CP4_WANT_DX;
  if (g || dtype != CP4_DTYPE_F32 || act != CP4_ACT_RELU || !filter || s.N == 0) return 0;
  // (operands on 16-byte boundaries; a call whose are not may take another route and leave them)
  const int variant = cp4::layer_filter_masks(s, nullptr, nullptr, nullptr, nullptr,
                                              reinterpret_cast<const float*>(256), dx);
  // (a first layer's step waits for the host up to some 64 MB of y, and memory for the signs is 4 us more
  // of that: N2 and N4 C3 K64 224x224 R16, 26 and 51 MB, 62 and 61 us without, 68 and 66 with; N8 and N16
  // 100 and 147 without, 75 and 130 with.  That layer alone was timed, on either side of the line.)
  // (nor where the tile kernel runs instead of the direct one: on rows off the multiples of four it would read the
  // signs one by one, N16 C3 K64 225x225 R16 241 us without, 248 with, and on others they gain nothing beyond
  // what the forward pays, N20 C3 K64 5x5 148x148 115.5 and 116.5, 224x224 184 and 179)
  if (!variant || (variant == 3 && (elements(s, s.T) < (size_t)16 << 20 ||
                                    !cp4::bwd_filter_dense_tiles_reads_signs(s, true))))
    return 0;
  return cp4::layer_forward_keeps(s) ? align256((size_t)s.N * ((s.T + 31) / 32) * s.H * s.W * 4) : 0;
}
// (remembered as the backward plan is; what a call takes up is decided by its operands)
size_t keep_plan(const cp4_shape& s, const cp4_geometry* g, int dtype, int act, int wanted) {
  static std::mutex mu;
  static std::map<PlanKey, size_t> plans;
  return remembered(mu, plans, plan_key(s, g, dtype, act, wanted),
                    [&] { return make_keep_plan(s, g, dtype, act, wanted); });
}

thread_local int g_route = 0;      // of this thread's last cp4_layer_backward
thread_local int g_mask_inside = 0, g_dx_beside = 0;

cp4_status check_layer(const cp4_shape* s, const cp4_geometry* g, int dtype, int act) {
  cp4_status rc = g ? cp4::check_layer_geometry(s, g) : cp4::check_layer_shape(s);
  if (rc != CP4_OK) return rc;
  if (act != CP4_ACT_NONE && act != CP4_ACT_RELU)
    return cp4::fail_with(CP4_ERR_UNSUPPORTED, "activation must be CP4_ACT_NONE or CP4_ACT_RELU");
  if (dtype != CP4_DTYPE_F32 && dtype != CP4_DTYPE_BF16 && dtype != CP4_DTYPE_F16)
    return cp4::fail_with(CP4_ERR_UNSUPPORTED, "dtype must be a cp4_dtype");
  if (g && dtype != CP4_DTYPE_F32)
    return cp4::fail_with(CP4_ERR_UNSUPPORTED, "a layer with a geometry takes fp32 activations");
  return CP4_OK;
}

#define CP4_TRY(call)                     \
  do {                                    \
    const cp4_status rc_ = (call);        \
    if (rc_ != CP4_OK) return rc_;        \
  } while (0)
#define CP4_LAUNCH(call)                                      \
  do {                                                        \
    const hipError_t e_ = (call);                             \
    if (e_ != hipSuccess) return cp4::fail_hip(e_, #call);    \
  } while (0)

}  // namespace

extern "C" {

size_t cp4_layer_forward_workspace_bytes(const cp4_shape* shape, const cp4_geometry* g, int dtype) {
  if (check_layer(shape, g, dtype, CP4_ACT_NONE) != CP4_OK || shape->N == 0) return 0;
  if (dtype == CP4_DTYPE_F32 || cp4_bf16_supported(shape, 0)) return 0;
  return align256(elements(*shape, shape->C) * 4) + align256(elements(*shape, shape->T) * 4);
}

cp4_status cp4_layer_forward(const cp4_shape* shape, const cp4_geometry* g, int dtype,
                             const void* x, const float* FK, const float* FC, const float* FH,
                             const float* FW, const float* bias, int activation, void* y,
                             void* workspace, size_t workspace_bytes, cp4_stream stream) {
  CP4_TRY(check_layer(shape, g, dtype, activation));
  if (dtype == CP4_DTYPE_F32) {
    const float* xf = static_cast<const float*>(x);
    float* yf = static_cast<float*>(y);
    return g ? cp4_conv2d_forward_ex(shape, g, xf, FK, FC, FH, FW, bias, activation, yf, stream)
             : cp4_conv2d_forward_bias_act(shape, xf, FK, FC, FH, FW, bias, activation, yf, stream);
  }
  if (shape->N == 0) return CP4_OK;
  if (cp4_bf16_supported(shape, 0))
    return dtype == CP4_DTYPE_BF16
               ? cp4_conv2d_forward_bf16(shape, x, FK, FC, FH, FW, bias, activation, y, stream)
               : cp4_conv2d_forward_f16(shape, x, FK, FC, FH, FW, bias, activation, y, stream);
  if (!x || !y) return cp4::fail_with(CP4_ERR_NULL_POINTER, "x or y is NULL");
  if (!workspace || workspace_bytes < cp4_layer_forward_workspace_bytes(shape, g, dtype))
    return cp4::fail_with(CP4_ERR_WORKSPACE, "workspace smaller than cp4_layer_forward_workspace_bytes");
  const size_t nx = elements(*shape, shape->C), ny = elements(*shape, shape->T);
  float* x32 = static_cast<float*>(workspace);
  float* y32 = reinterpret_cast<float*>(static_cast<unsigned char*>(workspace) + align256(nx * 4));
  hipStream_t st = static_cast<hipStream_t>(stream);
  CP4_LAUNCH(cp4::convert_launch(x, dtype, x32, CP4_DTYPE_F32, nx, st));
  CP4_TRY(cp4_conv2d_forward_bias_act(shape, x32, FK, FC, FH, FW, bias, activation, y32, stream));
  CP4_LAUNCH(cp4::convert_launch(y32, CP4_DTYPE_F32, y, dtype, ny, st));
  return CP4_OK;
}

size_t cp4_layer_kept_bytes(const cp4_shape* shape, const cp4_geometry* g, int dtype, int activation,
                            int wanted) {
  if (check_layer(shape, g, dtype, activation) != CP4_OK || shape->N == 0) return 0;
  return keep_plan(*shape, g, dtype, activation, wanted);
}

cp4_status cp4_layer_forward_keeping(const cp4_shape* shape, const cp4_geometry* g, int dtype,
                                     const void* x, const float* FK, const float* FC,
                                     const float* FH, const float* FW, const float* bias,
                                     int activation, int wanted, void* y, void* kept,
                                     size_t kept_bytes, int* parts, void* workspace,
                                     size_t workspace_bytes, cp4_stream stream) {
  if (!parts) return cp4::fail_with(CP4_ERR_NULL_POINTER, "parts is NULL");
  *parts = 0;
  CP4_TRY(check_layer(shape, g, dtype, activation));
  if (kept && shape->N && !(reinterpret_cast<uintptr_t>(kept) & 255)) {
    const size_t room = keep_plan(*shape, g, dtype, activation, wanted);
    if (room && kept_bytes >= room)
      return cp4::layer_forward_keeping(shape, static_cast<const float*>(x), FK, FC, FH, FW, bias,
                                        activation, static_cast<float*>(y),
                                        static_cast<unsigned short*>(kept), parts, stream);
  }
  return cp4_layer_forward(shape, g, dtype, x, FK, FC, FH, FW, bias, activation, y, workspace,
                           workspace_bytes, stream);
}

size_t cp4_layer_backward_workspace_bytes(const cp4_shape* shape, const cp4_geometry* g, int dtype,
                                          int activation, int wanted) {
  if (check_layer(shape, g, dtype, activation) != CP4_OK || shape->N == 0) return 0;
  return backward_plan(*shape, g, dtype, activation, wanted).total;
}

cp4_status cp4_layer_backward(const cp4_shape* shape, const cp4_geometry* g, int dtype,
                              const void* x, const void* y, const void* dy, const float* FK,
                              const float* FC, const float* FH, const float* FW, int activation,
                              void* dx, float* dFK, float* dFC, float* dFH, float* dFW,
                              float* dbias, void* workspace, size_t workspace_bytes,
                              cp4_stream stream) {
  return cp4_layer_backward_kept(shape, g, dtype, x, y, dy, FK, FC, FH, FW, activation, dx, dFK, dFC,
                                 dFH, dFW, dbias, nullptr, 0, 0, workspace, workspace_bytes, stream);
}

cp4_status cp4_layer_backward_kept(const cp4_shape* shape, const cp4_geometry* g, int dtype,
                                   const void* x, const void* y, const void* dy, const float* FK,
                                   const float* FC, const float* FH, const float* FW, int activation,
                                   void* dx, float* dFK, float* dFC, float* dFH, float* dFW,
                                   float* dbias, const void* kept, size_t kept_bytes, int parts_kept,
                                   void* workspace, size_t workspace_bytes, cp4_stream stream) {
  g_route = g_mask_inside = g_dx_beside = 0;
  CP4_TRY(check_layer(shape, g, dtype, activation));
  const cp4_shape& s = *shape;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool filter = dFK || dFC || dFH || dFW;
  if (filter && (!dFK || !dFC || !dFH || !dFW))
    return cp4::fail_with(CP4_ERR_NULL_POINTER, "all four factor gradients or none");
  if (s.N == 0) {            // empty batch: the gradients of the parameters are zero
    if (filter)
      CP4_TRY(cp4_conv2d_backward_filter(shape, nullptr, nullptr, FK, FC, FH, FW, dFK, dFC, dFH,
                                         dFW, nullptr, 0, stream));
    if (dbias) CP4_LAUNCH(cp4::zero_f32_launch(dbias, s.T, st));
    return CP4_OK;
  }
  if (!dy || (filter && !x) || (activation != CP4_ACT_NONE && !y))
    return cp4::fail_with(CP4_ERR_NULL_POINTER, "dy, x (factor gradients) or y (activation) is NULL");
  const int wanted =
      (dx ? CP4_WANT_DX : 0) | (filter ? CP4_WANT_FACTORS : 0) | (dbias ? CP4_WANT_BIAS : 0);
  const BackwardPlan p = backward_plan(s, g, dtype, activation, wanted);
  const size_t least = p.total - p.g1_bytes;
  if (least && (!workspace || workspace_bytes < least ||
                (reinterpret_cast<uintptr_t>(workspace) & 255)))
    return cp4::fail_with(CP4_ERR_WORKSPACE, "workspace smaller than "
                          "cp4_layer_backward_workspace_bytes or not on a 256-byte boundary");
  const size_t pass_bytes = p.pass_bytes + (workspace_bytes >= p.total ? p.g1_bytes : 0);
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  const size_t plane = out_elements(s, g) / ((size_t)s.N * s.T);
  const int N = (int)s.N, T = (int)s.T;
  const bool half = dtype != CP4_DTYPE_F32;
  const void* ym = activation == CP4_ACT_NONE ? nullptr : y;
  // 1. dy behind the activation, with the bias gradient
  const void* dya = dy;                                     // in the layer's type
  const float* dy32 = reinterpret_cast<const float*>(ws + p.act32_at);
  float* parts = reinterpret_cast<float*>(ws + p.bias_at);
  if (p.may_mask) {
    // a route that masks dy as it reads it: dy behind the activation never goes to memory
    const float *xf = static_cast<const float*>(x), *yf = static_cast<const float*>(ym),
                *dyf = static_cast<const float*>(dy);
    float* mask_ws = p.act16 ? reinterpret_cast<float*>(ws + p.act16_at) : nullptr;
    const int variant = cp4::layer_filter_masks(s, xf, yf, dyf, ws + p.pass_at, mask_ws, dx != nullptr);
    if (variant) {
      g_dx_beside = variant != 3 && dx;
      g_route = variant == 3 ? CP4_ROUTE_MASKED_TILES : CP4_ROUTE_DY_PASS | (dx ? CP4_ROUTE_DX_FROM_G1 : 0);
      const unsigned short* bits = nullptr;
      const uintptr_t at = reinterpret_cast<uintptr_t>(xf) | reinterpret_cast<uintptr_t>(yf) |
                           reinterpret_cast<uintptr_t>(dyf);
      if (kept && parts_kept == CP4_KEEP_MASK && !(reinterpret_cast<uintptr_t>(kept) & 255) &&
          (variant != 3 || cp4::bwd_filter_dense_tiles_reads_signs(s, (at & 15) == 0))) {
        const size_t room = keep_plan(s, g, dtype, activation, wanted);
        if (room && kept_bytes >= room) {
          bits = static_cast<const unsigned short*>(kept);
          g_route |= CP4_ROUTE_KEPT_MASK;
        }
      }
      return cp4::layer_backward_filter_masked(variant, shape, xf, yf, dyf, FK, FC, FH, FW, dFK, dFC,
                                               dFH, dFW, static_cast<float*>(dx), dbias, parts, mask_ws,
                                               bits, ws + p.pass_at, pass_bytes, stream);
    }
  }
  // or one whose contraction masks dy as it reads it and leaves it in memory for the others
  const cp4::LayerMask mask{ym, ws + p.act16_at, dbias, parts};
  int inside = 0;
  if (filter && !p.act32 && (!half || p.filter16) && (ym || dbias))
    inside = cp4::layer_filter_takes_mask(s, g, dtype, x, dy, ws + p.pass_at);
  if (inside && ym) dya = mask.masked;
  g_mask_inside = inside != 0;
  if (p.act16 && !inside) {
    CP4_LAUNCH(cp4::act_grad_launch(ym, dy, ws + p.act16_at, dtype, false, dbias, parts, N, T, plane, st));
    dya = ws + p.act16_at;
  }
  if (p.act32)
    CP4_LAUNCH(cp4::act_grad_launch(ym, dy, ws + p.act32_at, dtype, true, p.act16 ? nullptr : dbias,
                                    parts, N, T, plane, st));
  if (!p.act16 && !p.act32 && dbias && !inside)
    CP4_LAUNCH(cp4::act_grad_launch(ym, dy, nullptr, dtype, false, dbias, parts, N, T, plane, st));
  // 2. the factor gradients, and the input gradient with them where their pass has G1 at hand:
  // dx = FC G1 reads R planes an image, the pass of its own contracts the T channels of dy again
  // (N32 C256 56x56 R32: 26 against 56 us)
  void* pass_ws = ws + p.pass_at;
  bool dx_done = !dx;
  if (filter && (!half || p.filter16)) {
    CP4_TRY(cp4::layer_backward_filter(shape, g, dtype, x, inside ? dy : dya, FK, FC, FH, FW, dFK, dFC,
                                       dFH, dFW, pass_ws, pass_bytes, dx, &dx_done,
                                       inside && !half && !g ? inside : -1, inside ? &mask : nullptr,
                                       stream));
    if (dx && dx_done) {
      g_dx_beside = 1;
      if (cp4::layer_dx_variant() != 2) g_route |= CP4_ROUTE_DX_FROM_G1;
    }
    dx_done = dx_done || !dx;
  } else if (filter) {
    float* x32 = reinterpret_cast<float*>(ws + p.x32_at);
    CP4_LAUNCH(cp4::convert_launch(x, dtype, x32, CP4_DTYPE_F32, elements(s, s.C), st));
    CP4_TRY(cp4_conv2d_backward_filter(shape, x32, dy32, FK, FC, FH, FW, dFK, dFC, dFH, dFW, pass_ws,
                                       pass_bytes, stream));
  }
  if (dx_done) return CP4_OK;
  // 3. the input gradient on its own
  if (g)
    return cp4_conv2d_backward_data_ex(shape, g, static_cast<const float*>(dya), FK, FC, FH, FW,
                                       static_cast<float*>(dx), pass_ws, pass_bytes, stream);
  if (!half)
    return cp4_conv2d_backward_data(shape, static_cast<const float*>(dya), FK, FC, FH, FW,
                                    static_cast<float*>(dx), stream);
  if (p.dx16)
    return (dtype == CP4_DTYPE_BF16 ? cp4_conv2d_backward_data_bf16 : cp4_conv2d_backward_data_f16)(
        shape, dya, FK, FC, FH, FW, dx, stream);
  float* dx32 = reinterpret_cast<float*>(ws + p.dx32_at);
  CP4_TRY(cp4_conv2d_backward_data(shape, dy32, FK, FC, FH, FW, dx32, stream));
  CP4_LAUNCH(cp4::convert_launch(dx32, CP4_DTYPE_F32, dx, dtype, elements(s, s.C), st));
  return CP4_OK;
}

int cp4_layer_last_backward_route(void) { return g_route; }
int cp4_layer_last_backward_mask_inside(void) { return g_mask_inside; }
int cp4_layer_last_backward_dx_beside(void) { return g_dx_beside; }

}  // extern "C"
