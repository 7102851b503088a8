// Internal interface between the C ABI (cp4_capi.hip) and the kernel
// translation units.  Every launcher validates nothing: the C ABI has already
// checked pointers and shape, and each launcher's own `*_supported` predicate
// says whether its kernel's assumptions hold for a shape.
#ifndef CP4_INTERNAL_H
#define CP4_INTERNAL_H

#include <hip/hip_runtime.h>

#include "cp4/capi.h"

namespace cp4 {

// Operands of one forward-shaped launch.  Backward-data is the same kernel
// with x<-dy, Cin<-T, Cout<-C, Fin<-FK, Fout<-FC and flipped taps
// (Cuda_kernels/cp4Conv2dBackwardData.cu:79-87,98-108).
struct FwdKernelArgs {
  const float* x;     // [N, Cin, H, W]
  const float* Fin;   // [Cin, R]
  const float* Fout;  // [Cout, R]
  const float* FH;    // [Y, R]
  const float* FW;    // [X, R]
  float* y;           // [N, Cout, H, W]
  int N, Cin, Cout, H, W, pad, Y, X, R;
  int flip;           // 1: tap index t reads factor row (taps-1-t)
  // Output epilogue y = act(conv + bias[k]); only kernels that say so apply it
  // (the caller runs bias_act_launch after the others).
  const float* bias;  // [Cout] or null
  int act;            // 0: none, 1: max(., 0)
  // Rank and channel passes (rank-pass build of the producer / consumer kernel only): the
  // factor pointers may address a column block of wider matrices - ldf is their row
  // stride in floats (0: R) -, x a slice of Cin channels out of wider images - ldx is
  // the distance between images in elements (0: Cin * H * W) - and accumulate != 0 adds
  // to y instead of overwriting it.
  int ldf;
  size_t ldx;
  int accumulate;
  // 2-D-tap build of the producer / consumer kernel only: depthwise filter
  // [Y, X, R] used instead of the outer product FH x FW (FH, FW unused then).
  const float* taps2d;
  // Producer / consumer kernel: the device's fault record, four ints (may be null).
  int* fault;
  // Layer geometry beyond the reference's (stride 1, `pad` zeros before the image,
  // an H x W output): output pixel (ho, wo) reads x at (sh*ho + i - pt, sw*wo + j - pl),
  // the output plane is Ho x Wo.  sh == 0: the reference's geometry, the other
  // fields unused.  Only kernels that say so take sh != 0.
  int sh, sw, pt, pl, Ho, Wo;
  // Strided build of the producer / consumer kernel only: the adjoint of a strided
  // layer (its backward-data pass).  The H x W input plane is then the strided
  // layer's output gradient and the Ho x Wo output plane its input gradient:
  // output pixel (h, w) sums tap (i, j) times input pixel ((h + pt - i) / sh,
  // (w + pl - j) / sw) wherever both divisions are exact and land inside the plane
  // (flip unused).
  int transposed;
  // Strided build only, set by its own entry points: a filter of ty x tx taps that runs as
  // the square window of Y = X taps around it (even and rectangular filters); 0: Y, X.
  int ty, tx;
  // For a training step's backward pass (the saving build of the producer / consumer kernel, the
  // few-channel kernel; null: not wanted): one bit an output, y > 0, as
  // [N][blocks of 32 output channels][2][H * W] of 16 bits - half h, bit 4 a + b is channel 8 a + 4 h + b of
  // the block.
  unsigned short* save_mask;
  // Recomposed-filter kernel only: the dense filter [Cout, Cin, Y, X] itself, taps in
  // the order the pass reads them; the four factors are unused then.
  const float* dense;
};
// ... with what the launchers alone read (a launch costs by the bytes of its arguments, too: 2.6 us of
// host time with 60 of them, 3.0 with 360).
struct FwdArgs : FwdKernelArgs {
  // Not 0: the launch that follows reads y back (a later pass, the bias / activation kernel); y
  // leaves the caches only from so many bytes on.
  size_t reread;
  // Producer / consumer kernel: a tuned strip height (tile height in the tiled
  // build), log2 of the tile width (tiled build) and role split (1: off) that
  // replace the planner's choice; 0 leaves it to the planner.
  int tune_th, tune_lgwt, tune_split2;
  // Producer / consumer kernel: polls before a wait between waves gives up (0: the default).
  int spin_limit;
};

// The geometry of a launch with the defaults filled in.
struct Geometry {
  int sh, sw, pt, pl, Ho, Wo;
};
inline Geometry geometry_of(const FwdArgs& a) {
  if (a.sh == 0) return Geometry{1, 1, a.pad, a.pad, a.H, a.W};
  return Geometry{a.sh, a.sw, a.pt, a.pl, a.Ho, a.Wo};
}

// The C ABI's argument checks and its error record (cp4_last_error_message), for entry points
// in other files.
cp4_status check_layer_shape(const cp4_shape*);
cp4_status check_layer_geometry(const cp4_shape*, const cp4_geometry*);
cp4_status fail_with(cp4_status, const char* what);
cp4_status fail_hip(hipError_t, const char* where);

// A layer's mask and bias gradient inside the passes of its factor gradients: dy counts where
// y > 0 and is written so, in its own type, to `masked` as the contraction reads it (y null: dy as
// it is); dbias (may be null) is summed as the gradient GEMM reads that, in partial sets in
// bias_part.
struct LayerMask {
  const void* y;
  void* masked;
  float *dbias, *bias_part;
};

// The forward pass of a layer, leaving y's signs (FwdArgs::save_mask) in `mask` (null: not wanted) where
// the kernel that runs can; *parts says whether (CP4_KEEP_MASK) or not (0).
cp4_status layer_forward_keeping(const cp4_shape*, const float* x, const float* FK, const float* FC,
                                 const float* FH, const float* FW, const float* bias, int activation,
                                 float* y, unsigned short* mask, int* parts, cp4_stream);
// Whether the kernel of a layer's forward pass can leave them (aligned operands).
bool layer_forward_keeps(const cp4_shape&);

// The backward-filter entry points with the input gradient beside the factors' where the
// variant that runs has it at hand (`dx` may be null; *dx_done says whether it was written).
// dtype: a cp4_dtype, the type of x, dy and dx; `geometry` as in the _ex entry points.  `mask`
// (may be null): with the variant that layer_filter_takes_mask gave for these operands; `variant`
// is -1 without it.
cp4_status layer_backward_filter(const cp4_shape*, const cp4_geometry*, int dtype, const void* x,
                                 const void* dy, const float* FK, const float* FC, const float* FH,
                                 const float* FW, float* dFK, float* dFC, float* dFH, float* dFW,
                                 void* workspace, size_t workspace_bytes, void* dx, bool* dx_done,
                                 int variant, const LayerMask* mask, cp4_stream);
// Whether such a call of a layer with aligned operands forms G1 for dx (the three-launch variant): it does
// where its workspace has N * R * H * W floats more.
bool layer_filter_forms_g1(const cp4_shape&);
// Counts the changes of the tuned choices.
unsigned tuned_choices();
// The fp32 variant in which this thread's last such call wrote dx; 0: another pass, or none did.
int layer_dx_variant();
// The backward-filter variant (strided and 16-bit layers: any number above 0) that such a call
// runs with the mask and the bias gradient in it; 0: none does.
int layer_filter_takes_mask(const cp4_shape&, const cp4_geometry*, int dtype, const void* x,
                            const void* dy, const void* workspace);
// Most partial sets of T floats that any of those variants leaves of the bias gradient.
size_t layer_bias_sets(const cp4_shape&, const cp4_geometry*);
cp4_status layer_backward_filter_masked(int variant, const cp4_shape*, const float* x, const float* act_y,
                                        const float* dy, const float* FK, const float* FC,
                                        const float* FH, const float* FW, float* dFK, float* dFC,
                                        float* dFH, float* dFW, float* dx, float* dbias,
                                        float* bias_part, float* mask_ws, const unsigned short* bits, void* workspace,
                                        size_t workspace_bytes, cp4_stream);

// The backward-filter variant that an fp32 layer's factor gradients (and, want_dx, its input
// gradient) run with the mask and the bias gradient in it, with operands of these addresses; 0:
// none does.  mask_ws null: no room for the matrix-core variant's partial sets.
int layer_filter_masks(const cp4_shape&, const float* x, const float* y, const float* dy,
                       const void* workspace, const float* mask_ws, bool want_dx);

// Compute units of the current device (256 when no device can be asked).
int num_compute_units();


// The matrix-core kernels index pixels, strips and work items with 32-bit
// integers: planes up to 2^24 pixels and batch x plane products that keep every
// such count below 2^31.  Larger problems run on the general kernels, whose
// indices are 64-bit throughout.
inline bool fits_int_indexing(int N, int H, int W) {
  const size_t HW = (size_t)H * W;
  return HW <= (1u << 24) && (size_t)N * HW < (1ull << 35) && (size_t)N * H < (1ull << 30);
}

bool fwd_general_supported(const FwdArgs&);
hipError_t fwd_general_launch(const FwdArgs&, hipStream_t);
// Recomposed-filter direct convolution for very few channels on both sides.
bool fwd_dense_small_supported(const FwdArgs&);
hipError_t fwd_dense_small_launch(const FwdArgs&, hipStream_t);
// Its plan for a shape: 16 x 64 tiles in all and LDS bytes per workgroup (false: no plan).
bool fwd_dense_small_plan_info(const FwdArgs&, long* tiles, size_t* lds_bytes);
bool fwd_mfma_supported(const FwdArgs&);
hipError_t fwd_mfma_launch(const FwdArgs&, hipStream_t);
bool fwd_split_supported(const FwdArgs&);
hipError_t fwd_split_launch(const FwdArgs&, hipStream_t);
// Few short phases in small workgroups, for small problems (ranks up to 32).
bool fwd_light_supported(const FwdArgs&);
hipError_t fwd_light_launch(const FwdArgs&, hipStream_t);
// Persistent small workgroups over 2-D tiles, taps and output contraction in registers:
// few channels (up to 64 in), up to 16 ranks, planes of any width.
bool fwd_few_supported(const FwdArgs&);
hipError_t fwd_few_launch(const FwdArgs&, hipStream_t);
bool fwd_few_plan(const FwdArgs&, int* rows, int* cols, int* workgroups);
bool fwd_pipe_supported(const FwdArgs&);
hipError_t fwd_pipe_launch(const FwdArgs&, hipStream_t);
// Rows per strip and workgroups of the whole-row strip plan (false: no plan).
bool fwd_pipe_strip_plan(const FwdArgs&, int* rows, int* workgroups);
// Producer / consumer kernel with a 64-rank plane: ranks 33 - 64 in one pass (1x1 and 3x3
// filters, up to 256 input channels); honours FwdArgs::ldf, ldx and accumulate.
bool fwd_pipe64_supported(const FwdArgs&);
hipError_t fwd_pipe64_launch(const FwdArgs&, hipStream_t);
bool fwd_pipe64_plan(const FwdArgs&, int* rows, int* workgroups);
// The same kernel compiled with the bias / activation epilogue in its stores.
bool fwd_pipe_epi_supported(const FwdArgs&);
hipError_t fwd_pipe_epi_launch(const FwdArgs&, hipStream_t);
// ... and with FwdArgs::save_mask: the same y, bit for bit, and its signs.
bool fwd_pipe_save_supported(const FwdArgs&);
hipError_t fwd_pipe_save_launch(const FwdArgs&, hipStream_t);
// The same kernel with bfloat16 x and y in memory (FwdArgs::x / y point at
// 16-bit elements; factors and bias stay fp32), epilogue included.
bool fwd_pipe_io16_supported(const FwdArgs&);
hipError_t fwd_pipe_io16_launch(const FwdArgs&, hipStream_t);
// The same with IEEE half-precision x and y in memory.
bool fwd_pipe_iof16_supported(const FwdArgs&);
hipError_t fwd_pipe_iof16_launch(const FwdArgs&, hipStream_t);
// The few-channel and the recomposed-filter kernel likewise (the latter for filters up to 7 x 7).
bool fwd_few_io16_supported(const FwdArgs&);
hipError_t fwd_few_io16_launch(const FwdArgs&, hipStream_t);
bool fwd_few_iof16_supported(const FwdArgs&);
hipError_t fwd_few_iof16_launch(const FwdArgs&, hipStream_t);
bool fwd_dense_small_io16_supported(const FwdArgs&);
hipError_t fwd_dense_small_io16_launch(const FwdArgs&, hipStream_t);
bool fwd_dense_small_iof16_supported(const FwdArgs&);
hipError_t fwd_dense_small_iof16_launch(const FwdArgs&, hipStream_t);
// The same kernel honouring FwdArgs::ldf and FwdArgs::accumulate (rank passes).
bool fwd_pipe_rankpass_supported(const FwdArgs&);
hipError_t fwd_pipe_rankpass_launch(const FwdArgs&, hipStream_t);
// The same kernel on tiles of TH rows x Wt columns (wide planes).
bool fwd_pipe_tiled_supported(const FwdArgs&);
hipError_t fwd_pipe_tiled_launch(const FwdArgs&, hipStream_t);
bool fwd_pipe_tiled_epi_supported(const FwdArgs&);          // ... with the bias / activation epilogue
hipError_t fwd_pipe_tiled_epi_launch(const FwdArgs&, hipStream_t);
// The same kernel for a stride or an output plane of its own (FwdArgs::sh ...
// all filled in by the caller).
bool fwd_pipe_strided_supported(const FwdArgs&);
hipError_t fwd_pipe_strided_launch(const FwdArgs&, hipStream_t);
// The same kernel with a depthwise Y x X filter (FwdArgs::taps2d) in its tap step.
bool fwd_pipe_taps2d_supported(const FwdArgs&);
hipError_t fwd_pipe_taps2d_launch(const FwdArgs&, hipStream_t);
// In-place y[n,k,:] = act(y[n,k,:] + bias[k]) for variants without the epilogue.
hipError_t bias_act_launch(float* y, const float* bias, int act, size_t N, size_t K, size_t HW,
                           hipStream_t);

// Backward of the epilogue: out = dy where y > 0 (y null: dy itself; out null: not wanted, in
// `dtype` or widened to fp32) and dbias[t] = its sum over images and pixels (null: not wanted;
// `part`: T * act_grad_segments floats of scratch).  dtype: a cp4_dtype.
int act_grad_segments(int N, int T, size_t HW, int dtype);
hipError_t act_grad_launch(const void* y, const void* dy, void* out, int dtype, bool out_f32,
                           float* dbias, float* part, int N, int T, size_t HW, hipStream_t);
// Element-wise conversion between fp32 and a 16-bit type (cp4_dtype), round to nearest even.
hipError_t convert_launch(const void* src, int src_dtype, void* dst, int dst_dtype, size_t n,
                          hipStream_t);

// Backward-filter (factor gradients).
struct BwdFilterArgs {
  const float *x, *dy, *FK, *FC, *FH, *FW;
  float *dFK, *dFC, *dFH, *dFW;
  void* workspace;
  int N, C, T, H, W, pad, Y, X, R;
  // Matrix-core variant only, 3-factor CP op: a depthwise filter [Y, X, R] in place
  // of FH x FW and its gradient (FH, FW, dFH, dFW unused then).
  const float* taps2d;
  float* dtaps2d;
  // Matrix-core and three-launch variants: not null, the input gradient too, dx = FC G1 (in the type of
  // x; the forward's adjoint only where 2 * pad = Y - 1 = X - 1 or with a geometry).
  void* dx;
  // Three-launch variant: room for G1, [N, R, H, W], which it forms for dx only.
  float* g1_ws;
  // Where the variant's _masks function says so: dy counts where act_y > 0 (null: everywhere) and
  // dbias[t], its sum over images and pixels, comes along; all null: neither.  Scratch:
  // bias_part, T floats per compute unit (dense gradient) or partial set (_bias_sets), mask_ws, N * T * H * W
  // elements (matrix cores: dy behind the activation or, in the masked launch, partial sets).
  const float* act_y;
  float *dbias, *bias_part, *mask_ws;
  // y's signs from the layer's forward pass (FwdArgs::save_mask; null: it left none), which the direct filter
  // gradient and the masked launch read instead of act_y.
  const unsigned short* act_bits;
};
// general (VALU, any shape) and matrix-core variants
size_t bwd_filter_workspace_bytes(const cp4_shape&);
hipError_t bwd_filter_launch(const BwdFilterArgs&, hipStream_t);
bool bwd_filter_mfma_supported(const cp4_shape&);
size_t bwd_filter_mfma_workspace_bytes(const cp4_shape&);
bool bwd_filter_mfma_taps2d_supported(const cp4_shape&);   // with BwdFilterArgs::taps2d
hipError_t bwd_filter_mfma_launch(const BwdFilterArgs&, hipStream_t);
// That launch and the strided one take BwdFilterArgs::act_y and dbias (operands and workspace on
// 16-byte boundaries or not), and the partial sets of the bias gradient they leave.
bool bwd_filter_mfma_masks(const cp4_shape&, bool aligned16);
bool bwd_filter_mfma_strided_masks(const cp4_shape&, const Geometry&, bool aligned16);
bool bwd_filter_mfma_mask_pays(const cp4_shape& dy_planes, bool smaller_than_x);
int bwd_filter_mfma_bias_sets(const cp4_shape&);
// The same with the layer's activation mask and bias gradient in it (BwdFilterArgs::act_y,
// dbias, mask_ws); operands on 16-byte boundaries.
bool bwd_filter_mfma_dy_pass_masks(const cp4_shape&);
hipError_t bwd_filter_mfma_masked_launch(const BwdFilterArgs&, hipStream_t);
// One pass over dy behind a ReLU (y, its output; bits, where the forward left them: FwdArgs::save_mask):
// G3, `sets` partial sets [set][T][R] of dFK and [set][T] of dbias.
bool bwd_dy_pass_supported(int N, int T, int R, int HW);
int bwd_dy_pass_sets(int N, int T, int HW);
hipError_t bwd_dy_pass_launch(const float* dy, const float* y, const unsigned short* bits,
                              const float* FK, const float* Cc, float* G3, float* partK, float* partB,
                              int N, int T, int R, int HW, hipStream_t);
// Matrix-core variant with the tap step inside the gradient GEMMs (three launches;
// square odd filters up to 5 with 2 * pad == Y - 1, channel counts multiples of 16,
// H * W a multiple of 4, x / dy / workspace 16-byte aligned).
bool bwd_filter_fused_supported(const cp4_shape&);
// Where the three-launch variant is the faster one (small and medium problems, whose
// time is launches and first-load latencies rather than bandwidth).
bool bwd_filter_fused_preferred(const cp4_shape&);
size_t bwd_filter_fused_workspace_bytes(const cp4_shape&);
bool bwd_filter_fused_mask_pays(const cp4_shape&);
int bwd_filter_fused_bias_sets(const cp4_shape&);      // takes BwdFilterArgs::act_y and dbias throughout
hipError_t bwd_filter_fused_launch(const BwdFilterArgs&, hipStream_t);
// Few channels on both sides (square filters of 1, 3, 5 taps; T * C up to 256 with plain
// multiply-adds, or up to 64 output channels and 16384 entries of the dense gradient on the
// matrix cores): the dense filter gradient over tiles of pixels, then the chain rule onto the
// factors (three launches, no [N, R, H, W] intermediates).
bool bwd_filter_dense_tiles_supported(const cp4_shape&);
bool bwd_filter_dense_tiles_preferred(const cp4_shape&);
size_t bwd_filter_dense_tiles_workspace_bytes(const cp4_shape&);
hipError_t bwd_filter_dense_tiles_launch(const BwdFilterArgs&, hipStream_t);
// The route takes the layer's activation mask and bias gradient with it (BwdFilterArgs::act_y).
bool bwd_filter_dense_tiles_masks(const cp4_shape&);
// Whether it reads y's signs (BwdFilterArgs::act_bits) where they are at hand; aligned16: x, dy and act_y on
// 16-byte boundaries.
bool bwd_filter_dense_tiles_reads_signs(const cp4_shape&, bool aligned16);
// 0: the plain multiply-add tile kernel, 1: the matrix-core one, wherever both can run the
// shape; anything else: the route's own choice.
void bwd_filter_dense_tiles_force_kernel(int which);
// A layer with a stride and zeros of its own before the image (BwdFilterArgs::H, W: the
// input plane; pad unused; dy on the geometry's Ho x Wo grid).
bool bwd_filter_mfma_strided_supported(const cp4_shape&, const Geometry&);
size_t bwd_filter_mfma_strided_workspace_bytes(const cp4_shape&, const Geometry&);
hipError_t bwd_filter_mfma_strided_launch(const BwdFilterArgs&, const Geometry&, hipStream_t);
// The same with bfloat16 x and dy in memory (BwdFilterArgs::x / dy point at 16-bit
// elements); split-bf16 kernels only: C and T multiples of 16.
bool bwd_filter_mfma_io16_supported(const cp4_shape&);
size_t bwd_filter_mfma_io16_workspace_bytes(const cp4_shape&);
hipError_t bwd_filter_mfma_io16_launch(const BwdFilterArgs&, hipStream_t);
// The same with IEEE half-precision x and dy in memory.
bool bwd_filter_mfma_iof16_supported(const cp4_shape&);
size_t bwd_filter_mfma_iof16_workspace_bytes(const cp4_shape&);
hipError_t bwd_filter_mfma_iof16_launch(const BwdFilterArgs&, hipStream_t);
hipError_t bwd_filter_full_launch(const cp4_shape&, const float* x,
                                  const float* dy, float* dK, int accumulate,
                                  hipStream_t);

// Utilities.
hipError_t recompose_launch(const cp4_shape&, const float* FK, const float* FC,
                            const float* FH, const float* FW, float* K,
                            hipStream_t);
hipError_t count_exceeding_launch(const float* A, const float* B, size_t n,
                                  float tol, unsigned long long* d_count,
                                  hipStream_t);
hipError_t random_uniform_launch(float* dst, size_t n, unsigned long long seed,
                                 hipStream_t);
// 3-factor CP sibling op: its factors as a CP4 of rank Y*Rank (s.Rank is the CP
// rank), and the fold of the CP4 factor gradients back onto the three factors.
hipError_t cp3_expand_launch(const cp4_shape& s, const float* K0, const float* K1,
                             const float* K2, float* FK, float* FC, float* FH, float* FW,
                             hipStream_t);
hipError_t cp3_fold_launch(const cp4_shape& s, const float* dFK, const float* dFC,
                           const float* dFW, float* dK0, float* dK1, float* dK2, hipStream_t);
// dst[row*ld_dst + c] = src[row*ld_src + c], c < cols (column blocks of factor matrices)
hipError_t copy_columns_launch(const float* src, int ld_src, float* dst, int ld_dst, int rows,
                               int cols, hipStream_t);
// dst[plane][ot + sh*u][ol + sw*v] = src[plane][u][v] on `planes` planes of h x w
// set into canvases of Hc x Wc; every other canvas cell is written as zero.
hipError_t embed_launch(const float* src, float* dst, size_t planes, int h, int w, int Hc, int Wc,
                        int ot, int ol, int sh, int sw, hipStream_t);
// Reshaped-CP sibling op: its dense filter (transposed != 0: the input-gradient
// pass's filter [C][T][Y][X], taps reversed) and the fold of a dense filter
// gradient [T][C][Y][X] back onto K0 [S0,T0,R], K1 [S1,T1,R], KC [Y,X,R].
hipError_t rcp_recompose_launch(const float* K0, const float* K1, const float* KC, float* out,
                                int S0, int S1, int T0, int T1, int Y, int X, int R,
                                int transposed, hipStream_t);
hipError_t rcp_fold_launch(const float* dK, const float* K0, const float* K1, const float* KC,
                           float* dK0, float* dK1, float* dKC, int S0, int S1, int T0, int T1,
                           int Y, int X, int R, hipStream_t);
// dst [cols, rows] = transpose of src [rows, cols]
hipError_t transpose_f32_launch(const float* src, float* dst, int rows, int cols, hipStream_t);
hipError_t copy_f32_launch(float* dst, const float* src, size_t n, hipStream_t);
hipError_t add_f32_launch(float* dst, const float* src, size_t n, hipStream_t);   // dst += src
// dst [groups][rows_padded][row_elems] = src [groups][rows][row_elems] with zero rows appended: up to
// four such jobs in one launch (a plain copy: one group of one row).
struct PadJob {
  const float* src;
  float* dst;
  size_t groups, rows, rows_padded, row_elems;
};
constexpr int kMaxPadJobs = 4;
hipError_t pad_rows_launch(const PadJob* jobs, int n, hipStream_t st);
// Fill kernel rather than a memset node, so that callers may capture the
// empty-batch paths into a graph like every other launch.
hipError_t zero_f32_launch(float* dst, size_t n, hipStream_t);

}  // namespace cp4
#endif
