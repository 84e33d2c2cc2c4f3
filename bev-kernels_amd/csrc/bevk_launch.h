// Internal launcher interface between the C ABI (binding.cpp) and the kernel
// translation units. Arguments are already validated by the caller; each launcher
// only enqueues work and returns the HIP status of the launch.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bevk_common.h"

namespace bevk {

// Compute units of the current device (cached per device; 0 when the query fails).
int device_cus();

struct MsdaArgs {
  const void *value;
  const int64_t *spatial_shapes;
  const int64_t *level_start_index;
  const void *sampling_loc;
  const void *attn_weight;
  void *output;
  int batch, spatial_size, num_heads, channels, num_levels, num_query, num_point;
};

hipError_t launch_msda_forward(int dtype, const MsdaArgs &a, bool force_generic,
                               hipStream_t stream);

// MSDA backward: f holds the forward inputs (f.output unused).
struct MsdaBwdArgs {
  MsdaArgs f;
  const void *grad_output;
  int64_t go_stride[4];  // grad_output strides over (batch, query, head, channel), elements
  void *grad_value, *grad_loc, *grad_attn;
  void *workspace;       // fp32 accumulator for 16-bit dtypes, then the sorted path's buffers
  int64_t workspace_bytes;
  bool fresh = false;    // fp32 / fp64 grad_value is written, not added to
};

// Bytes of fp32 accumulator the 16-bit backward needs at least (0 for f32 / f64).
int64_t msda_backward_workspace_min(int dtype, int64_t value_elems);
// Bytes that also hold the buffers of the sorted grad_value path (D = 32; 64 with many
// samples), which runs when the workspace is at least this large.
int64_t msda_backward_workspace_bytes(int dtype, int64_t batch, int64_t spatial_size,
                                      int64_t num_heads, int64_t channels, int64_t num_levels,
                                      int64_t num_query, int64_t num_point);
// force_generic: the per-unit atomic kernel for every level (no coarse split, no grid
// owner pass, no D = 32 kernel).
hipError_t launch_msda_backward(int dtype, const MsdaBwdArgs &a, bool force_generic,
                                hipStream_t stream);

struct DcnGeom {
  int batch, channels, height, width, height_col, width_col;
  int kernel_h, kernel_w, pad_h, pad_w, stride_h, stride_w, dil_h, dil_w;
  int deformable_group;
  int gate = 0;  // NHWC column-to-image: whole samples with h <= -1, w <= -1, h >= H or w >= W
                 // contribute nothing (the NCHW layer's rule)
  int grad_ld = 0; // NHWC column-to-image: row length of grad_offset and grad_mask (0: 2T and T)
};

// NCHW modulated im2col; `tiled` picks the geometry-reuse kernel (im2col_opt).
hipError_t launch_im2col_nchw(int dtype, const DcnGeom &g, const void *data_im,
                              const void *data_offset, const void *data_mask,
                              void *data_col, bool tiled, hipStream_t stream);

// NHWC gather (offsets [M][dg][2T], mask [M][dg][T]). fused_y (dg == 1): data_offset is the raw [.., 3T] offset-conv output.
hipError_t launch_im2col_nhwc(int dtype, const DcnGeom &g, const void *data_im,
                              const void *data_offset, bool fused_y, const void *data_mask,
                              void *data_col, hipStream_t stream);

// Fused NHWC implicit-GEMM forward (dg == 1). w_packed: layout of launch_dcn_pack_weight.
// geo (DcnGeo): kGeoMask / kGeoY read data_offset (and data_mask) in the input dtype;
// kGeoYF32 reads an fp32 y [M][3T] as data_offset and adds y_bias [3T] (fp32, may be
// null); kGeoRegular ignores data_offset / data_mask and writes fp32 `out`, with an fp32
// `bias`. relu: max(out, 0) in the epilogue (not for kGeoRegular).
hipError_t launch_dcn_fused_nhwc(int dtype, const DcnGeom &g, int channels_out,
                                 const void *data_im, const void *data_offset, int geo,
                                 const void *data_mask, const void *w_packed,
                                 const void *bias, void *out, hipStream_t stream,
                                 const float *y_bias = nullptr, bool relu = false);

// fp16 / bf16 implicit GEMM with the weight in MFMA-fragment blocks (<= 9 taps).
bool dcn_fused_h_supported(const DcnGeom &g);
hipError_t launch_dcn_fused_h(int dtype, const DcnGeom &g, int channels_out, const void *x,
                              const void *off, int geo, const void *msk,
                              const void *w_packed, const void *bias, void *out,
                              hipStream_t stream, const float *y_bias = nullptr,
                              bool relu = false, float *part = nullptr);
// Bytes of the scratch `part` (16-byte aligned) with which this shape runs K in parts (geo
// kGeoMask / kGeoYF32, 16-byte aligned output); 0 where it runs whole.
int64_t dcn_fused_h_parts_bytes(int dtype, const DcnGeom &g, int channels_out);
// K parts of that shape (1: whole) and the 16-row blocks of a workgroup (0: whole).
int dcn_fused_h_parts(int dtype, const DcnGeom &g, int channels_out, int *row_blocks);

// One-launch DCNv2 forward with the offset conv inside (fp16 / bf16 on the persistent
// kernel): y = conv(x, w_off) + b_off (fp32, kept in LDS and written to y_out), offsets
// y[:, :2T], mask sigmoid(y[:, 2T:]), then the deformable implicit GEMM (+ bias, relu).
// Returns false (and launches nothing) when the shape does not take the persistent
// kernel; the caller then runs the offset conv and launch_dcn_fused_nhwc (kGeoYF32).
bool dcn_mega_supported(int dtype, const DcnGeom &g, int channels_out, const void *out);
hipError_t launch_dcn_mega(int dtype, const DcnGeom &g, int channels_out, const void *x,
                           const void *w_off_packed, const float *b_off,
                           const void *w_packed, const void *bias, bool relu, float *y_out,
                           void *out, hipStream_t stream);

// Elements of the packed weight: fp32 Cout * K; half types ceil(Cout/32) * ceil(K/16) * 512.
int64_t dcn_packed_weight_elems(int dtype, int cout, int K);
// Weight [Cout][C][kh*kw] (module layout; [Cout][kh*kw][C] with src_tc) -> packed: fp32
// [Cout][kh*kw][C]; fp16 / bf16 MFMA-fragment blocks (block (n/32, k/16), lane
// (n%32) + 32*((k%16)/8), 8 consecutive k), k = t*C + c, zero outside [0, Cout) x [0, K).
hipError_t launch_dcn_pack_weight(int dtype, const void *weight, int cout, int C, int T,
                                  void *packed, hipStream_t stream, bool src_tc = false);

// 16-bit layer preparation: weight [cout][C][T] and w_off [n3][C][T] packed, b_off [n3] (b_dtype, or
// null; n3 <= 64) as fp32.
hipError_t launch_dcn_prep16(int dtype, const void *weight, int cout, const void *w_off, int n3, int C,
                             int T, const void *b_off, int b_dtype, void *packed, void *packed_off,
                             float *b_out, hipStream_t stream);

// fp32 products on the bf16 matrix cores (three bf16 pieces per operand, dcn_f32.hip).
// Split weight of n columns and k reduction elements (with its flags), from the module weight
// [Cout][C][T]: n = Cout, k = t*C + c (C % 32 == 0), or transposed n = t*C + c, k = Cout
// (C % 16 == 0, Cout % 32 == 0); T <= 9, 16-byte aligned buffers.
int64_t f32_split_weight_bytes(int64_t n, int64_t k);
hipError_t launch_f32_split_weight(const float *weight, int cout, int C, int T, bool transposed,
                                   void *packed, hipStream_t stream);
// out[m, n] = sum_k A[m, k] W[n, k] (+ bias): A the deformable columns of geometry g (dg == 1,
// <= 9 taps, geo kGeoMask / kGeoY / kGeoYF32; M and K must match it), or with g == nullptr the
// matrix x [M][K]. K % 32 == 0, x under 2 GiB, 16-byte aligned x.
hipError_t launch_f32_split(const DcnGeom *g, int channels_out, int M, int K, const void *x,
                            const void *off, int geo, const void *msk, const void *w_split,
                            const float *bias, float *out, hipStream_t stream, bool relu);

// The whole NCHW fp32 layer (groups == 1, any deformable_group): x [B, C, H, W], off [B, dg*2T, Ho,
// Wo], msk [B, dg*T, Ho, Wo], weight [Cout, C, kh, kw] -> out [B, Cout, Ho, Wo]. C % 32 == 0, at
// most 9 taps; with deformable groups a 16-byte aligned output and columns under 2 GiB.
int64_t dcn_layer_f32_workspace_bytes(const DcnGeom &g, int channels_out);
hipError_t launch_dcn_layer_f32(const DcnGeom &g, int cout, const float *x, const float *off,
                                const float *msk, const float *weight, const float *bias,
                                void *workspace, float *out, hipStream_t stream);

// Input gradient of a plain convolution with n3 <= 32 outputs: out [B*H*W][C] (out_dtype) =
// addend (fp32, or null) + the transposed convolution of y32 [B*Ho*Wo][32] (columns past n3 zero)
// with w_off [n3][C][T], split by launch_f32_split_offset_weight into
// f32_split_weight_bytes(C, 32 T) bytes.
hipError_t launch_f32_split_offset_weight(const float *w_off, int n3, int C, int T, void *packed,
                                          hipStream_t stream);
hipError_t launch_f32_tconv(const DcnGeom &g, const float *y32, const void *w_split,
                            const float *addend, int out_dtype, void *out, hipStream_t stream);

// Weight gradient [Cout][C][T] (out_dtype) = sum over the M pixels of dout [M][Cout] times cols
// [M][T*C] (both dtype). Cout and C multiples of 16 bytes' worth of elements, T <= 25; the
// workspace holds weight_grad_workspace_bytes.
int64_t weight_grad_workspace_bytes(int dtype, int64_t M, int C, int T, int cout);
hipError_t launch_weight_grad(int dtype, const void *cols, const void *dout, int64_t M, int C, int T,
                              int cout, void *workspace, int out_dtype, void *grad_w,
                              hipStream_t stream);

// The offset conv's weight gradient [n3][C][T] (out_dtype) from its input x [B, H, W, C] and fp32
// output gradient y32 [M][32] (n3 <= 32 columns used; C % 4 == 0).
int64_t offset_weight_grad_workspace_bytes(const DcnGeom &g, int n3);
hipError_t launch_offset_weight_grad(int x_dtype, const DcnGeom &g, int n3, const void *x,
                                     const float *y32, void *workspace, int out_dtype, void *grad_w,
                                     hipStream_t stream);

// out[c] (out_dtype) = fp32 sum over the rows of src [rows][ld], c < n; ld a multiple of 16 bytes'
// worth of elements, src 16-byte aligned.
int64_t column_sums_workspace_bytes(int n);
hipError_t launch_column_sums(int dtype, const void *src, int64_t rows, int ld, int n, void *workspace,
                              int out_dtype, void *out, hipStream_t stream);

// dst[b][c][r] = src[b][r][c] for 2- or 4-byte elements (NCHW <-> NHWC).
hipError_t launch_transpose(int elem_bytes, const void *src, void *dst, int batch, int rows,
                            int cols, hipStream_t stream);

// NHWC gather whose offsets / pre-sigmoid mask come from an fp32 y [M][3T] plus an fp32
// bias [3T] (the fused front end: y is the offset conv without its bias).
hipError_t launch_im2col_nhwc_yf32(int dtype, const DcnGeom &g, const void *data_im,
                                   const float *y, const float *y_bias, void *data_col,
                                   hipStream_t stream);

// NCHW column-to-image backward (any dg), gradients in the input dtype: grad_im accumulated
// with atomics (caller zeroes it; skipped when null), grad_offset / grad_mask written
// (skipped when grad_offset is null).
hipError_t launch_col2im_nchw(int dtype, const DcnGeom &g, const void *col, const void *im,
                              const void *off, const void *msk, void *grad_im,
                              void *grad_offset, void *grad_mask, hipStream_t stream);

// NHWC column-to-image backward (offsets [M][dg][2T], mask [M][dg][T]): grad_im [B,H,W,C] fp32 accumulated with atomics
// (caller zeroes it; skipped when null), grad_offset [M][dg][2T] and grad_mask [M][dg][T] fp32
// written (skipped when grad_offset is null). fused_y (dg == 1): offsets / pre-sigmoid mask
// from y [M][3T] and grad_mask is the gradient of the pre-sigmoid value.
hipError_t launch_col2im_nhwc(int dtype, const DcnGeom &g, const void *dcol, const void *im,
                              const void *off, bool fused_y, const void *msk, float *grad_im,
                              float *grad_offset, float *grad_mask, hipStream_t stream);

}  // namespace bevk
