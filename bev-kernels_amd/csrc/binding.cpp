// C ABI of libbevk.so: argument validation, error reporting and dispatch onto the
// kernel launchers. The entry points keep the argument order of the reference's
// pybind11 functions (naotic/bev-kernels csrc/binding.cpp:142-191 and
// csrc_musa/msda/binding_musa.mu:545-557) with tensors lowered to device pointers.
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <mutex>
#include <string>

#include "../../include/bev_kernels.h"
#include "bevk_launch.h"

namespace {

thread_local std::string g_last_error;

int fail(int code, const char *fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

int ok() { return BEVK_OK; }

int hip_status(hipError_t e, const char *what) {
  if (e == hipSuccess) return ok();
  return fail(BEVK_ERR_HIP, "%s: HIP error %d (%s)", what, (int)e, hipGetErrorString(e));
}

const char *dtype_name(int dtype) {
  switch (dtype) {
    case BEVK_F32: return "Float";
    case BEVK_F16: return "Half";
    case BEVK_BF16: return "BFloat16";
    case BEVK_F64: return "Double";
    default: return "unknown";
  }
}

bool valid_dtype(int dtype) { return dtype >= BEVK_F32 && dtype <= BEVK_F64; }

int dtype_size(int dtype) {
  switch (dtype) {
    case BEVK_F32: return 4;
    case BEVK_F16: case BEVK_BF16: return 2;
    default: return 8;
  }
}

// The kernels address one image (or, for the fused kernel, the whole input) through a
// 32-bit buffer range with an out-of-range sentinel just past its end.
constexpr long long kMaxBufferBytes = (1LL << 31) - 256;

// Shared geometry checks of the DCN entry points; the output size must follow the
// convolution formula (modulated_deform_conv.py:364-365).
int check_geom(const char *fn, const bevk::DcnGeom &g) {
  if (g.batch < 0 || g.channels < 0 || g.height < 0 || g.width < 0)
    return fail(BEVK_ERR_INVALID, "%s: negative input size", fn);
  if (g.kernel_h <= 0 || g.kernel_w <= 0 || g.stride_h <= 0 || g.stride_w <= 0 ||
      g.dil_h <= 0 || g.dil_w <= 0 || g.pad_h < 0 || g.pad_w < 0)
    return fail(BEVK_ERR_INVALID,
                "%s: kernel, stride and dilation must be positive and padding non-negative", fn);
  if (g.deformable_group <= 0)
    return fail(BEVK_ERR_INVALID, "%s: deformable_group must be positive", fn);
  if (g.channels % g.deformable_group != 0)
    return fail(BEVK_ERR_INVALID, "%s: channels (%d) must be divisible by deformable_group (%d)",
                fn, g.channels, g.deformable_group);
  const int ho = (g.height + 2 * g.pad_h - (g.dil_h * (g.kernel_h - 1) + 1)) / g.stride_h + 1;
  const int wo = (g.width + 2 * g.pad_w - (g.dil_w * (g.kernel_w - 1) + 1)) / g.stride_w + 1;
  if (g.height_col != ho || g.width_col != wo)
    return fail(BEVK_ERR_INVALID,
                "%s: output size (%d, %d) does not match the convolution geometry (%d, %d)", fn,
                g.height_col, g.width_col, ho, wo);
  if (ho <= 0 || wo <= 0)
    return fail(BEVK_ERR_INVALID, "%s: empty output (%d x %d)", fn, ho, wo);
  return ok();
}

bevk::DcnGeom make_geom(int batch_size, int channels, int height_im, int width_im,
                        int height_col, int width_col, int kernel_h, int kernel_w, int pad_h,
                        int pad_w, int stride_h, int stride_w, int dilation_h, int dilation_w,
                        int deformable_group) {
  bevk::DcnGeom g;
  g.batch = batch_size; g.channels = channels; g.height = height_im; g.width = width_im;
  g.height_col = height_col; g.width_col = width_col;
  g.kernel_h = kernel_h; g.kernel_w = kernel_w; g.pad_h = pad_h; g.pad_w = pad_w;
  g.stride_h = stride_h; g.stride_w = stride_w; g.dil_h = dilation_h; g.dil_w = dilation_w;
  g.deformable_group = deformable_group;
  return g;
}

int im2col_nchw_common(const char *fn, bool tiled, int dtype, const void *data_im,
                       const void *data_offset, const void *data_mask, const bevk::DcnGeom &g,
                       void *data_col, void *stream) {
  g_last_error.clear();
  if (!valid_dtype(dtype)) return fail(BEVK_ERR_INVALID, "%s: unknown dtype code %d", fn, dtype);
  if (int rc = check_geom(fn, g)) return rc;
  const long long cols = (long long)g.channels * g.kernel_h * g.kernel_w * g.batch *
                         g.height_col * g.width_col;
  if (cols == 0) return ok();
  if ((long long)g.channels * g.height * g.width * dtype_size(dtype) > kMaxBufferBytes)
    return fail(BEVK_ERR_INVALID, "%s: one input image exceeds 2 GiB", fn);
  if (!data_im || !data_offset || !data_mask || !data_col)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_im2col_nchw(dtype, g, data_im, data_offset, data_mask,
                                             data_col, tiled, (hipStream_t)stream),
                    fn);
}

}  // namespace

extern "C" {

const char *bevk_last_error(void) { return g_last_error.c_str(); }

const char *bevk_version(void) { return "bevk 0.1.0 gfx950"; }

int bevk_modulated_deformable_im2col(int dtype, const void *data_im, const void *data_offset,
                                     const void *data_mask, int batch_size, int channels,
                                     int height_im, int width_im, int height_col, int width_col,
                                     int kernel_h, int kernel_w, int pad_h, int pad_w,
                                     int stride_h, int stride_w, int dilation_h, int dilation_w,
                                     int deformable_group, void *data_col, void *stream) {
  return im2col_nchw_common(
      "modulated_deformable_im2col", false, dtype, data_im, data_offset, data_mask,
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w,
                deformable_group),
      data_col, stream);
}

int bevk_modulated_deformable_im2col_opt(
    int dtype, const void *data_im, const void *data_offset, const void *data_mask,
    int batch_size, int channels, int height_im, int width_im, int height_col, int width_col,
    int kernel_h, int kernel_w, int pad_h, int pad_w, int stride_h, int stride_w,
    int dilation_h, int dilation_w, int deformable_group, void *data_col, void *stream) {
  return im2col_nchw_common(
      "modulated_deformable_im2col_opt", true, dtype, data_im, data_offset, data_mask,
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w,
                deformable_group),
      data_col, stream);
}

int bevk_modulated_deformable_im2col_nhwc(
    int dtype, const void *data_im, const void *data_offset, int offset_last_dim,
    const void *data_mask, int batch_size, int channels, int height_im, int width_im,
    int height_col, int width_col, int kernel_h, int kernel_w, int pad_h, int pad_w,
    int stride_h, int stride_w, int dilation_h, int dilation_w, int deformable_group,
    void *data_col, void *stream) {
  const char *fn = "modulated_deformable_im2col_nhwc";
  g_last_error.clear();
  // dcn_fused_nhwc_cuda.cu:34-35
  if (deformable_group != 1)
    return fail(BEVK_ERR_INVALID, "NHWC fused path supports deformable_group == 1 only");
  if (!valid_dtype(dtype)) return fail(BEVK_ERR_INVALID, "%s: unknown dtype code %d", fn, dtype);
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w, 1);
  if (int rc = check_geom(fn, g)) return rc;
  const int taps = kernel_h * kernel_w;
  if (offset_last_dim != 2 * taps && offset_last_dim != 3 * taps)
    return fail(BEVK_ERR_INVALID, "%s: offset last dim must be 2T (%d) or 3T (%d), got %d", fn,
                2 * taps, 3 * taps, offset_last_dim);
  const bool fused_y = offset_last_dim == 3 * taps;  // dcn_fused_nhwc_cuda.cu:54
  const long long m = (long long)batch_size * height_col * width_col;
  // dcn_fused_nhwc_cuda.cu:37-40
  if (m * taps * channels >= 2147483647LL)
    return fail(BEVK_ERR_INVALID, "NHWC gather: Col element count exceeds int32 range");
  if (m * taps * channels == 0) return ok();
  if ((long long)height_im * width_im * channels * dtype_size(dtype) > kMaxBufferBytes)
    return fail(BEVK_ERR_INVALID, "%s: one input image exceeds 2 GiB", fn);
  if (!data_im || !data_offset || (!fused_y && !data_mask) || !data_col)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_im2col_nhwc(dtype, g, data_im, data_offset, fused_y, data_mask,
                                             data_col, (hipStream_t)stream),
                    fn);
}

int bevk_modulated_deformable_col2im_nchw(
    int dtype, const void *data_col, const void *data_im, const void *data_offset,
    const void *data_mask, int batch_size, int channels, int height_im, int width_im,
    int height_col, int width_col, int kernel_h, int kernel_w, int pad_h, int pad_w,
    int stride_h, int stride_w, int dilation_h, int dilation_w, int deformable_group,
    void *grad_im, void *grad_offset, void *grad_mask, void *stream) {
  const char *fn = "modulated_deformable_col2im";
  g_last_error.clear();
  if (!valid_dtype(dtype)) return fail(BEVK_ERR_INVALID, "%s: unknown dtype code %d", fn, dtype);
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w,
                deformable_group);
  if (int rc = check_geom(fn, g)) return rc;
  const long long n = (long long)batch_size * deformable_group * kernel_h * kernel_w *
                      height_col * width_col;
  if (n == 0 || channels == 0) return ok();
  if ((grad_offset == nullptr) != (grad_mask == nullptr))
    return fail(BEVK_ERR_INVALID, "%s: grad_offset and grad_mask go together", fn);
  if (!data_col || !data_offset || !data_mask || (!grad_im && !grad_offset) ||
      (grad_offset && !data_im))
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  // 16-bit grad_im takes packed pair atomics: its first element must start a pair
  if (grad_im && dtype_size(dtype) == 2 && reinterpret_cast<uintptr_t>(grad_im) % 4 != 0)
    return fail(BEVK_ERR_INVALID, "%s: 16-bit grad_im must be 4-byte aligned", fn);
  return hip_status(bevk::launch_col2im_nchw(dtype, g, data_col, data_im, data_offset, data_mask,
                                             grad_im, grad_offset, grad_mask,
                                             (hipStream_t)stream),
                    fn);
}

int bevk_modulated_deformable_col2im_nhwc(
    int dtype, const void *dcol, const void *data_im, const void *data_offset,
    int offset_last_dim, const void *data_mask, int batch_size, int channels, int height_im,
    int width_im, int height_col, int width_col, int kernel_h, int kernel_w, int pad_h, int pad_w,
    int stride_h, int stride_w, int dilation_h, int dilation_w, int deformable_group,
    float *grad_im, float *grad_offset, float *grad_mask, void *stream) {
  const char *fn = "modulated_deformable_col2im_nhwc";
  g_last_error.clear();
  if (deformable_group != 1)
    return fail(BEVK_ERR_INVALID, "NHWC fused path supports deformable_group == 1 only");
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(dtype));
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w, 1);
  if (int rc = check_geom(fn, g)) return rc;
  const int taps = kernel_h * kernel_w;
  if (offset_last_dim != 2 * taps && offset_last_dim != 3 * taps)
    return fail(BEVK_ERR_INVALID, "%s: offset last dim must be 2T (%d) or 3T (%d), got %d", fn,
                2 * taps, 3 * taps, offset_last_dim);
  const bool fused_y = offset_last_dim == 3 * taps;
  const long long m = (long long)batch_size * height_col * width_col;
  if (m * taps * channels >= 2147483647LL)
    return fail(BEVK_ERR_INVALID, "NHWC col2im: Col element count exceeds int32 range");
  if (m * taps == 0) return ok();
  if ((grad_offset == nullptr) != (grad_mask == nullptr))
    return fail(BEVK_ERR_INVALID, "%s: grad_offset and grad_mask go together", fn);
  if (!dcol || !data_offset || (!fused_y && !data_mask) || (!grad_im && !grad_offset) ||
      (grad_offset && !data_im))
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_col2im_nhwc(dtype, g, dcol, data_im, data_offset, fused_y,
                                             data_mask, grad_im, grad_offset, grad_mask,
                                             (hipStream_t)stream),
                    fn);
}

int bevk_dcn_layer_im2col_nhwc(int dtype, const void *data_im, const void *data_offset,
                               const void *data_mask, int batch_size, int channels, int height_im,
                               int width_im, int height_col, int width_col, int kernel_h,
                               int kernel_w, int pad_h, int pad_w, int stride_h, int stride_w,
                               int dilation_h, int dilation_w, int deformable_group,
                               void *data_col, void *stream) {
  const char *fn = "dcn_layer_im2col_nhwc";
  g_last_error.clear();
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(dtype));
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w,
                deformable_group);
  if (int rc = check_geom(fn, g)) return rc;
  const long long taps = (long long)kernel_h * kernel_w;
  const long long m = (long long)batch_size * height_col * width_col;
  if (m * taps * channels >= 2147483647LL || m * taps * deformable_group >= 2147483647LL)
    return fail(BEVK_ERR_INVALID, "NHWC gather: Col element count exceeds int32 range");
  if (m * taps * channels == 0) return ok();
  if ((long long)channels * height_im * width_im * dtype_size(dtype) > kMaxBufferBytes)
    return fail(BEVK_ERR_INVALID, "%s: one input image exceeds 2 GiB", fn);
  if (!data_im || !data_offset || !data_mask || !data_col)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_im2col_nhwc(dtype, g, data_im, data_offset, false, data_mask,
                                             data_col, (hipStream_t)stream),
                    fn);
}

int bevk_dcn_layer_col2im_nhwc(
    int dtype, const void *dcol, const void *data_im, const void *data_offset,
    const void *data_mask, int batch_size, int channels, int height_im, int width_im,
    int height_col, int width_col, int kernel_h, int kernel_w, int pad_h, int pad_w, int stride_h,
    int stride_w, int dilation_h, int dilation_w, int deformable_group, float *grad_im,
    float *grad_offset, float *grad_mask, void *stream) {
  const char *fn = "dcn_layer_col2im_nhwc";
  g_last_error.clear();
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(dtype));
  bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w,
                deformable_group);
  if (int rc = check_geom(fn, g)) return rc;
  g.gate = 1;
  const long long taps = (long long)kernel_h * kernel_w;
  const long long m = (long long)batch_size * height_col * width_col;
  if (m * taps * channels >= 2147483647LL || m * taps * deformable_group >= 2147483647LL)
    return fail(BEVK_ERR_INVALID, "NHWC col2im: Col element count exceeds int32 range");
  if (m * taps == 0) return ok();
  if (!dcol || !data_im || !data_offset || !data_mask || !grad_im || !grad_offset || !grad_mask)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_col2im_nhwc(dtype, g, dcol, data_im, data_offset, false,
                                             data_mask, grad_im, grad_offset, grad_mask,
                                             (hipStream_t)stream),
                    fn);
}

// Static scratch of the allocation-free front end
// (bevk_modulated_deformable_fused_im2col_nhwc_noalloc): the packed offset-conv weight and
// the fp32 offset-conv output y [M][3T] of one call. Every GPU the library runs on holds
// its own copy until the process ends; calls that overlap on one GPU share it and race.
static constexpr size_t kNoAllocScratchBytes = size_t(16) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

// The device address of `scratch` on the current device, looked up once per device (the
// host-side name is not a device address: kernels and copies take this pointer).
static constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mutex;
static void *g_scratch_ptr[kMaxScratchDevices];

static int device_scratch(const char *fn, void **out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxScratchDevices)
    return fail(BEVK_ERR_HIP, "%s: no usable current HIP device", fn);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr)
      return fail(BEVK_ERR_HIP, "%s: hipGetSymbolAddress(scratch) failed: %s", fn,
                  hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

// Workspace of the fused front end: packed offset-conv weight, then y [M][3T] fp32.
static long long fused_im2col_ws_parts(int dtype, long long m, int taps, int channels,
                                       long long *y_offset) {
  const long long packed = bevk::dcn_packed_weight_elems(dtype, 3 * taps, taps * channels) *
                           dtype_size(dtype);
  *y_offset = (packed + 255) / 256 * 256;
  return *y_offset + m * 3 * taps * (long long)sizeof(float);
}

int64_t bevk_dcn_fused_im2col_nhwc_workspace_bytes(int dtype, int batch_size, int channels,
                                                   int height_col, int width_col, int kernel_h,
                                                   int kernel_w) {
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16) return -1;
  if (batch_size < 0 || channels < 0 || height_col < 0 || width_col < 0 || kernel_h <= 0 ||
      kernel_w <= 0)
    return -1;
  long long y_offset = 0;
  return fused_im2col_ws_parts(dtype, (long long)batch_size * height_col * width_col,
                               kernel_h * kernel_w, channels, &y_offset);
}

// The fused front end (offset conv + sigmoid + gather into the columns) with its scratch
// in the caller's `workspace`, or (static_scratch) in the library's static scratch, whose
// capacity is then workspace_bytes: a larger need is an error.
static int fused_im2col_run(
    const char *fn, bool static_scratch, int dtype, const void *data_im, const void *w_off, const float *b_off,
    int batch_size, int channels, int height_im, int width_im, int height_col, int width_col,
    int kernel_h, int kernel_w, int pad_h, int pad_w, int stride_h, int stride_w,
    int dilation_h, int dilation_w, int deformable_group, void *workspace,
    int64_t workspace_bytes, void *data_col, void *stream) {
  g_last_error.clear();
  // dcn_fused_nhwc_cuda.cu:99-100
  if (deformable_group != 1)
    return fail(BEVK_ERR_INVALID, "NHWC fused path supports deformable_group == 1 only");
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(dtype));
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w, 1);
  if (int rc = check_geom(fn, g)) return rc;
  const int taps = kernel_h * kernel_w;
  if (dtype != BEVK_F32 && taps > 9)
    return fail(BEVK_ERR_UNSUPPORTED,
                "%s: kernels of more than 9 taps are fp32-only (use the split path)", fn);
  const long long m = (long long)batch_size * height_col * width_col;
  // dcn_fused_nhwc_cuda.cu:101-103
  if (m * taps * channels >= 2147483647LL)
    return fail(BEVK_ERR_INVALID, "NHWC fused: Col element count exceeds int32 range");
  if (m * taps * channels == 0) return ok();
  const int vec = 16 / dtype_size(dtype);
  if (channels % vec != 0)
    return fail(BEVK_ERR_UNSUPPORTED,
                "%s: channels (%d) must be a positive multiple of %d for '%s'", fn, channels,
                vec, dtype_name(dtype));
  if ((long long)batch_size * height_im * width_im * channels * dtype_size(dtype) >
          kMaxBufferBytes ||
      m >= (1LL << 30))
    return fail(BEVK_ERR_INVALID, "%s: problem too large for 32-bit buffer offsets", fn);
  long long y_offset = 0;
  const long long need = fused_im2col_ws_parts(dtype, m, taps, channels, &y_offset);
  if (workspace_bytes < need)
    return static_scratch
               ? fail(BEVK_ERR_INVALID,
                      "%s: this shape needs %lld bytes of scratch; the library's static "
                      "scratch holds %lld (use the workspace entry point)",
                      fn, need, (long long)workspace_bytes)
               : fail(BEVK_ERR_INVALID, "%s: workspace of %lld bytes, %lld needed", fn,
                      (long long)workspace_bytes, need);
  if (!data_im || !w_off || !b_off || !data_col || (!static_scratch && !workspace))
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  if (static_scratch) {
    if (int rc = device_scratch(fn, &workspace)) return rc;
  }
  const hipStream_t st = (hipStream_t)stream;
  void *packed = workspace;
  float *y = reinterpret_cast<float *>(static_cast<char *>(workspace) + y_offset);
  // 1. offset-conv weight [3T][T][C] -> the fused kernel's layout. The fp32 layout
  //    [3T][T * C] is w_off as given: no pass. (Half types: reading w_off unpacked, 32 rows
  //    of 32 bytes per load, measured 3 us slower at res4 than packing it first.)
  const void *w_conv = w_off;
  if (dtype != BEVK_F32) {
    if (int rc = hip_status(bevk::launch_dcn_pack_weight(dtype, w_off, 3 * taps, channels,
                                                         taps, packed, st, /*src_tc=*/true),
                            fn))
      return rc;
    w_conv = packed;
  }
  // 2. y = offset conv without bias, fp32 accumulation, fp32 output (matrix cores)
  if (int rc = hip_status(bevk::launch_dcn_fused_nhwc(dtype, g, 3 * taps, data_im, nullptr,
                                                      bevk::kGeoRegular, nullptr, w_conv,
                                                      nullptr, y, st),
                          fn))
    return rc;
  // 3. sigmoid, bias and the deformable gather into the columns
  return hip_status(bevk::launch_im2col_nhwc_yf32(dtype, g, data_im, y, b_off, data_col, st),
                    fn);
}

int bevk_modulated_deformable_fused_im2col_nhwc(
    int dtype, const void *data_im, const void *w_off, const float *b_off, int batch_size,
    int channels, int height_im, int width_im, int height_col, int width_col, int kernel_h,
    int kernel_w, int pad_h, int pad_w, int stride_h, int stride_w, int dilation_h,
    int dilation_w, int deformable_group, void *workspace, int64_t workspace_bytes,
    void *data_col, void *stream) {
  return fused_im2col_run("modulated_deformable_fused_im2col_nhwc", false, dtype, data_im,
                          w_off, b_off, batch_size, channels, height_im, width_im, height_col,
                          width_col, kernel_h, kernel_w, pad_h, pad_w, stride_h, stride_w,
                          dilation_h, dilation_w, deformable_group, workspace,
                          workspace_bytes, data_col, stream);
}

int bevk_modulated_deformable_fused_im2col_nhwc_noalloc(
    int dtype, const void *data_im, const void *w_off, const float *b_off, int batch_size,
    int channels, int height_im, int width_im, int height_col, int width_col, int kernel_h,
    int kernel_w, int pad_h, int pad_w, int stride_h, int stride_w, int dilation_h,
    int dilation_w, int deformable_group, void *data_col, void *stream) {
  return fused_im2col_run("modulated_deformable_fused_im2col_nhwc_noalloc", true, dtype, data_im,
                          w_off, b_off, batch_size, channels, height_im, width_im, height_col,
                          width_col, kernel_h, kernel_w, pad_h, pad_w, stride_h, stride_w,
                          dilation_h, dilation_w, deformable_group, nullptr,
                          (int64_t)kNoAllocScratchBytes, data_col, stream);
}

int64_t bevk_dcn_packed_weight_bytes(int dtype, int channels_out, int kernel_h, int kernel_w,
                                      int channels) {
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16) return -1;
  if (channels_out < 0 || kernel_h <= 0 || kernel_w <= 0 || channels < 0) return -1;
  return bevk::dcn_packed_weight_elems(dtype, channels_out, kernel_h * kernel_w * channels) *
         dtype_size(dtype);
}

int bevk_dcn_pack_weight(int dtype, const void *weight, int channels_out, int kernel_h,
                         int kernel_w, int channels, void *packed, void *stream) {
  const char *fn = "dcn_pack_weight";
  g_last_error.clear();
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(dtype));
  if (channels_out < 0 || kernel_h <= 0 || kernel_w <= 0 || channels < 0)
    return fail(BEVK_ERR_INVALID, "%s: invalid weight shape", fn);
  const long long bytes = bevk::dcn_packed_weight_elems(dtype, channels_out,
                                                        kernel_h * kernel_w * channels) *
                          dtype_size(dtype);
  if (bytes == 0) return ok();
  if (bytes > kMaxBufferBytes)
    return fail(BEVK_ERR_INVALID, "%s: weight too large for 32-bit buffer offsets", fn);
  if (!weight || !packed) return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_dcn_pack_weight(dtype, weight, channels_out, channels,
                                                 kernel_h * kernel_w, packed,
                                                 (hipStream_t)stream),
                    fn);
}

int bevk_transpose(int dtype, const void *src, void *dst, int batch, int rows, int cols,
                   void *stream) {
  const char *fn = "transpose";
  g_last_error.clear();
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(dtype));
  if (batch < 0 || rows < 0 || cols < 0)
    return fail(BEVK_ERR_INVALID, "%s: negative size", fn);
  if (batch == 0 || rows == 0 || cols == 0) return ok();
  if (batch > 65535 || (rows + 63) / 64 > 65535 || (cols + 63) / 64 > (1 << 30))
    return fail(BEVK_ERR_INVALID, "%s: shape exceeds the launch grid", fn);
  if (!src || !dst) return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_transpose(dtype_size(dtype), src, dst, batch, rows, cols,
                                           (hipStream_t)stream),
                    fn);
}

int bevk_dcn_fused_fwd_nhwc(int dtype, const void *data_im, const void *data_offset,
                            int offset_last_dim, const void *data_mask, const void *weight_packed,
                            const void *bias, int batch_size, int channels, int height_im,
                            int width_im, int height_col, int width_col, int channels_out,
                            int kernel_h, int kernel_w, int pad_h, int pad_w, int stride_h,
                            int stride_w, int dilation_h, int dilation_w, void *out,
                            void *stream) {
  const char *fn = "dcn_fused_fwd_nhwc";
  g_last_error.clear();
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(dtype));
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w, 1);
  if (int rc = check_geom(fn, g)) return rc;
  if (channels_out < 0) return fail(BEVK_ERR_INVALID, "%s: negative channels_out", fn);
  const int taps = kernel_h * kernel_w;
  if (offset_last_dim != 2 * taps && offset_last_dim != 3 * taps)
    return fail(BEVK_ERR_INVALID, "%s: offset last dim must be 2T (%d) or 3T (%d), got %d", fn,
                2 * taps, 3 * taps, offset_last_dim);
  const bool fused_y = offset_last_dim == 3 * taps;
  const long long m = (long long)batch_size * height_col * width_col;
  if (m * channels_out == 0) return ok();
  const int vec = 16 / dtype_size(dtype);
  if (channels <= 0 || channels % vec != 0)
    return fail(BEVK_ERR_UNSUPPORTED,
                "%s: channels (%d) must be a positive multiple of %d for '%s'", fn, channels,
                vec, dtype_name(dtype));
  if ((long long)batch_size * height_im * width_im * channels * dtype_size(dtype) >
          kMaxBufferBytes ||
      (long long)taps * channels * channels_out * dtype_size(dtype) > kMaxBufferBytes ||
      m >= (1LL << 30))
    return fail(BEVK_ERR_INVALID, "%s: problem too large for 32-bit buffer offsets", fn);
  if (bevk::dcn_packed_weight_elems(dtype, channels_out, taps * channels) * dtype_size(dtype) >
      kMaxBufferBytes)
    return fail(BEVK_ERR_INVALID, "%s: weight too large for 32-bit buffer offsets", fn);
  if (!data_im || !data_offset || (!fused_y && !data_mask) || !weight_packed || !out)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_dcn_fused_nhwc(dtype, g, channels_out, data_im, data_offset,
                                                fused_y ? bevk::kGeoY : bevk::kGeoMask,
                                                data_mask, weight_packed, bias, out,
                                                (hipStream_t)stream),
                    fn);
}

int64_t bevk_f32_split_weight_bytes(int n, int k) {
  return n < 0 || k < 0 ? -1 : bevk::f32_split_weight_bytes(n, k);
}

int bevk_dcn_split_weight(const void *weight, int channels_out, int kernel_h, int kernel_w,
                          int channels, int transposed, void *split, void *stream) {
  const char *fn = "dcn_split_weight";
  g_last_error.clear();
  if (channels_out <= 0 || kernel_h <= 0 || kernel_w <= 0 || channels <= 0)
    return fail(BEVK_ERR_INVALID, "%s: invalid weight shape", fn);
  const int taps = kernel_h * kernel_w;
  if (taps > 9 || channels % (transposed ? 16 : 32) != 0 || (transposed && channels_out % 32 != 0))
    return fail(BEVK_ERR_UNSUPPORTED,
                "%s: at most 9 taps, and channels in whole blocks of the split layout", fn);
  const long long n = transposed ? (long long)channels * taps : channels_out;
  const long long k = transposed ? channels_out : (long long)channels * taps;
  if (bevk::f32_split_weight_bytes(n, k) > kMaxBufferBytes)
    return fail(BEVK_ERR_INVALID, "%s: weight too large for 32-bit buffer offsets", fn);
  if (!weight || !split) return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_f32_split_weight(static_cast<const float *>(weight), channels_out,
                                                  channels, taps, transposed != 0, split,
                                                  (hipStream_t)stream),
                    fn);
}

int bevk_gemm_f32(const void *a, const void *weight_split, int m, int k, int n, void *out,
                  void *stream) {
  const char *fn = "gemm_f32";
  g_last_error.clear();
  if (m < 0 || n < 0 || k <= 0 || k % 32 != 0)
    return fail(BEVK_ERR_INVALID, "%s: sizes must not be negative and k a multiple of 32", fn);
  if (m == 0 || n == 0) return ok();
  if ((long long)m * k * 4 > kMaxBufferBytes ||
      bevk::f32_split_weight_bytes(n, k) > kMaxBufferBytes || m >= (1 << 30))
    return fail(BEVK_ERR_INVALID, "%s: problem too large for 32-bit buffer offsets", fn);
  if (!a || !weight_split || !out) return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_f32_split(nullptr, n, m, k, a, nullptr, bevk::kGeoMask, nullptr,
                                           weight_split, nullptr, static_cast<float *>(out),
                                           (hipStream_t)stream, false),
                    fn);
}

static int weight_grad_check(const char *fn, int dtype, long long m, int channels, int taps,
                             int channels_out) {
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(dtype));
  const int vec = 16 / dtype_size(dtype);
  if (m <= 0 || m >= (1LL << 30) || channels <= 0 || channels_out <= 0 || channels % vec != 0 ||
      channels_out % vec != 0 || taps <= 0 || taps > 25)
    return fail(BEVK_ERR_UNSUPPORTED,
                "%s: channels must be positive multiples of %d for '%s', at most 25 taps", fn, vec,
                dtype_name(dtype));
  if ((long long)channels * taps * dtype_size(dtype) * 64 > (1 << 28) ||
      (long long)channels_out * dtype_size(dtype) * 64 > (1 << 28))
    return fail(BEVK_ERR_INVALID, "%s: rows too long for 32-bit buffer offsets", fn);
  return 0;
}

int64_t bevk_dcn_weight_grad_workspace_bytes(int dtype, int64_t m, int channels, int taps,
                                             int channels_out) {
  if (weight_grad_check("dcn_weight_grad", dtype, m, channels, taps, channels_out)) return -1;
  return bevk::weight_grad_workspace_bytes(dtype, m, channels, taps, channels_out);
}

int bevk_dcn_weight_grad(int dtype, const void *cols, const void *dout, int64_t m, int channels,
                         int taps, int channels_out, void *workspace, int64_t workspace_bytes,
                         int out_dtype, void *grad_weight, void *stream) {
  const char *fn = "dcn_weight_grad";
  g_last_error.clear();
  if (int rc = weight_grad_check(fn, dtype, m, channels, taps, channels_out)) return rc;
  if (out_dtype != BEVK_F32 && out_dtype != BEVK_F16 && out_dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(out_dtype));
  if (workspace_bytes < bevk::weight_grad_workspace_bytes(dtype, m, channels, taps, channels_out))
    return fail(BEVK_ERR_INVALID, "%s: workspace too small", fn);
  if (!cols || !dout || !workspace || !grad_weight)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_weight_grad(dtype, cols, dout, m, channels, taps, channels_out,
                                             workspace, out_dtype, grad_weight,
                                             (hipStream_t)stream),
                    fn);
}

// The NHWC split layer's backward steps: checks shared by the two entry points below.
static int layer_backward_check(const char *fn, int dtype, const bevk::DcnGeom &g) {
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(dtype));
  if (int rc = check_geom(fn, g)) return rc;
  const long long taps = (long long)g.kernel_h * g.kernel_w;
  const long long m = (long long)g.batch * g.height_col * g.width_col;
  if (taps > 9 || g.channels <= 0 || g.channels % 8 != 0)
    return fail(BEVK_ERR_UNSUPPORTED, "%s: at most 9 taps and channels a multiple of 8", fn);
  if (m * taps * g.channels >= 2147483647LL || m * 32 * 4 > kMaxBufferBytes ||
      (long long)g.batch * g.height * g.width * g.channels * 4 > kMaxBufferBytes)
    return fail(BEVK_ERR_INVALID, "%s: problem too large for 32-bit buffer offsets", fn);
  return 0;
}

int bevk_dcn_split_col2im_nhwc(int dtype, const void *dcol, const void *data_im, const void *y,
                               int batch_size, int channels, int height_im, int width_im,
                               int height_col, int width_col, int kernel_h, int kernel_w, int pad_h,
                               int pad_w, int stride_h, int stride_w, int dilation_h,
                               int dilation_w, float *grad_im, float *grad_y, void *stream) {
  const char *fn = "dcn_split_col2im_nhwc";
  g_last_error.clear();
  bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w, 1);
  if (int rc = layer_backward_check(fn, dtype, g)) return rc;
  if ((long long)batch_size * height_col * width_col == 0) return ok();
  if (!dcol || !data_im || !y || !grad_im || !grad_y)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  g.grad_ld = 32;
  return hip_status(bevk::launch_col2im_nhwc(dtype, g, dcol, data_im, y, true, nullptr, grad_im,
                                             grad_y, grad_y + 2 * kernel_h * kernel_w,
                                             (hipStream_t)stream),
                    fn);
}

// Workspace of the offset conv's backward: the split weight, then the larger of the weight
// gradient's parts and the column sums' (run one after the other).
static long long offset_backward_split_bytes(const bevk::DcnGeom &g) {
  return (bevk::f32_split_weight_bytes(g.channels, 32LL * g.kernel_h * g.kernel_w) + 255) / 256 * 256;
}
static long long offset_backward_ws(const bevk::DcnGeom &g) {
  const int n3 = 3 * g.kernel_h * g.kernel_w;
  const long long a = bevk::offset_weight_grad_workspace_bytes(g, n3);
  const long long b = bevk::column_sums_workspace_bytes(n3);
  return offset_backward_split_bytes(g) + (a > b ? a : b);
}

int64_t bevk_dcn_offset_conv_backward_workspace_bytes(int batch_size, int channels, int height_col,
                                                      int width_col, int kernel_h, int kernel_w) {
  bevk::DcnGeom g{};
  g.batch = batch_size; g.channels = channels; g.height_col = height_col; g.width_col = width_col;
  g.kernel_h = kernel_h; g.kernel_w = kernel_w;
  if (batch_size <= 0 || channels <= 0 || height_col <= 0 || width_col <= 0 || kernel_h <= 0 ||
      kernel_w <= 0 || kernel_h * kernel_w > 9)
    return -1;
  return offset_backward_ws(g);
}

int bevk_dcn_offset_conv_backward(int dtype, const void *data_im, const float *w_off,
                                  const float *grad_y, const float *addend, int batch_size,
                                  int channels, int height_im, int width_im, int height_col,
                                  int width_col, int kernel_h, int kernel_w, int pad_h, int pad_w,
                                  int stride_h, int stride_w, int dilation_h, int dilation_w,
                                  void *workspace, int64_t workspace_bytes, void *grad_im,
                                  int weight_dtype, void *grad_w, void *grad_b, void *stream) {
  const char *fn = "dcn_offset_conv_backward";
  g_last_error.clear();
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w, 1);
  if (int rc = layer_backward_check(fn, dtype, g)) return rc;
  if (weight_dtype != BEVK_F32 && weight_dtype != BEVK_F16 && weight_dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn,
                dtype_name(weight_dtype));
  const long long m = (long long)batch_size * height_col * width_col;
  if (m == 0) return fail(BEVK_ERR_INVALID, "%s: empty batch", fn);
  if (!data_im || !w_off || !grad_y || !workspace || !grad_im || !grad_w || !grad_b)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  if (workspace_bytes < offset_backward_ws(g))
    return fail(BEVK_ERR_INVALID, "%s: workspace too small", fn);
  const hipStream_t st = (hipStream_t)stream;
  const int taps = kernel_h * kernel_w, n3 = 3 * taps;
  void *parts = static_cast<char *>(workspace) + offset_backward_split_bytes(g);
  hipError_t e = bevk::launch_f32_split_offset_weight(w_off, n3, channels, taps, workspace, st);
  if (e == hipSuccess) e = bevk::launch_f32_tconv(g, grad_y, workspace, addend, dtype, grad_im, st);
  if (e == hipSuccess)
    e = bevk::launch_offset_weight_grad(dtype, g, n3, data_im, grad_y, parts, weight_dtype, grad_w, st);
  if (e == hipSuccess)
    e = bevk::launch_column_sums(BEVK_F32, grad_y, m, 32, n3, parts, weight_dtype, grad_b, st);
  return hip_status(e, fn);
}

int64_t bevk_column_sums_workspace_bytes(int n) { return n < 0 ? -1 : bevk::column_sums_workspace_bytes(n); }

int bevk_column_sums(int dtype, const void *src, int64_t rows, int n, void *workspace,
                     int64_t workspace_bytes, int out_dtype, void *out, void *stream) {
  const char *fn = "column_sums";
  g_last_error.clear();
  if (dtype < BEVK_F32 || dtype > BEVK_BF16 || out_dtype < BEVK_F32 || out_dtype > BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "%s: fp32, fp16 and bf16 only", fn);
  if (rows <= 0 || n <= 0 || n % (16 / dtype_size(dtype)) != 0 ||
      reinterpret_cast<uintptr_t>(src) % 16 != 0)
    return fail(BEVK_ERR_INVALID, "%s: rows must be 16-byte vectors of a 16-byte aligned matrix", fn);
  if (workspace_bytes < bevk::column_sums_workspace_bytes(n))
    return fail(BEVK_ERR_INVALID, "%s: workspace too small", fn);
  if (!src || !workspace || !out) return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_column_sums(dtype, src, rows, n, n, workspace, out_dtype, out,
                                             (hipStream_t)stream),
                    fn);
}

// Shared checks of the offset-conv entry points (dg == 1, fused-kernel dtypes, channel
// vectors, 32-bit buffer offsets). Returns 0 or the failure code.
static int check_offset_conv(const char *fn, int dtype, const bevk::DcnGeom &g) {
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16)
    return fail(BEVK_ERR_UNSUPPORTED, "\"%s\" not implemented for '%s'", fn, dtype_name(dtype));
  if (int rc = check_geom(fn, g)) return rc;
  const int taps = g.kernel_h * g.kernel_w;
  if (dtype != BEVK_F32 && taps > 9)
    return fail(BEVK_ERR_UNSUPPORTED,
                "%s: kernels of more than 9 taps are fp32-only for the offset conv", fn);
  const int vec = 16 / dtype_size(dtype);
  if (g.channels <= 0 || g.channels % vec != 0)
    return fail(BEVK_ERR_UNSUPPORTED,
                "%s: channels (%d) must be a positive multiple of %d for '%s'", fn, g.channels,
                vec, dtype_name(dtype));
  const long long m = (long long)g.batch * g.height_col * g.width_col;
  if ((long long)g.batch * g.height * g.width * g.channels * dtype_size(dtype) >
          kMaxBufferBytes ||
      m >= (1LL << 30))
    return fail(BEVK_ERR_INVALID, "%s: problem too large for 32-bit buffer offsets", fn);
  return 0;
}

int bevk_dcn_offset_conv_nhwc(int dtype, const void *data_im, const void *w_off_packed,
                              const float *b_off, int batch_size, int channels, int height_im,
                              int width_im, int height_col, int width_col, int kernel_h,
                              int kernel_w, int pad_h, int pad_w, int stride_h, int stride_w,
                              int dilation_h, int dilation_w, float *y, void *stream) {
  const char *fn = "dcn_offset_conv_nhwc";
  g_last_error.clear();
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w, 1);
  if (int rc = check_offset_conv(fn, dtype, g)) return rc;
  const int taps = kernel_h * kernel_w;
  if ((long long)batch_size * height_col * width_col == 0) return ok();
  if (!data_im || !w_off_packed || !y) return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  return hip_status(bevk::launch_dcn_fused_nhwc(dtype, g, 3 * taps, data_im, nullptr,
                                                bevk::kGeoRegular, nullptr, w_off_packed, b_off,
                                                y, (hipStream_t)stream),
                    fn);
}

int bevk_dcn_mega_fwd_nhwc(int dtype, const void *data_im, const void *w_off_packed,
                           const float *b_off, const void *weight_packed, const void *bias,
                           int batch_size, int channels, int height_im, int width_im,
                           int height_col, int width_col, int channels_out, int kernel_h,
                           int kernel_w, int pad_h, int pad_w, int stride_h, int stride_w,
                           int dilation_h, int dilation_w, int act_relu, float *y, void *out,
                           void *stream) {
  const char *fn = "dcn_mega_fwd_nhwc";
  g_last_error.clear();
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w, 1);
  if (int rc = check_offset_conv(fn, dtype, g)) return rc;
  if (channels_out < 0) return fail(BEVK_ERR_INVALID, "%s: negative channels_out", fn);
  const int taps = kernel_h * kernel_w;
  const long long m = (long long)batch_size * height_col * width_col;
  if (m == 0) return ok();
  if ((long long)taps * channels * channels_out * dtype_size(dtype) > kMaxBufferBytes ||
      bevk::dcn_packed_weight_elems(dtype, channels_out, taps * channels) * dtype_size(dtype) >
          kMaxBufferBytes)
    return fail(BEVK_ERR_INVALID, "%s: weight too large for 32-bit buffer offsets", fn);
  if (!data_im || !w_off_packed || !y || (channels_out > 0 && (!weight_packed || !out)))
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  const hipStream_t st = (hipStream_t)stream;
  if (channels_out > 0 && bevk::dcn_mega_supported(dtype, g, channels_out, out))
    return hip_status(bevk::launch_dcn_mega(dtype, g, channels_out, data_im, w_off_packed, b_off,
                                            weight_packed, bias, act_relu != 0, y, out, st),
                      fn);
  // Other shapes: the offset conv (with its bias) into y, then the fused kernel reading y.
  if (int rc = hip_status(bevk::launch_dcn_fused_nhwc(dtype, g, 3 * taps, data_im, nullptr,
                                                      bevk::kGeoRegular, nullptr, w_off_packed,
                                                      b_off, y, st),
                          fn))
    return rc;
  if (channels_out == 0) return ok();
  return hip_status(bevk::launch_dcn_fused_nhwc(dtype, g, channels_out, data_im, y,
                                                bevk::kGeoYF32, nullptr, weight_packed, bias,
                                                out, st, nullptr, act_relu != 0),
                    fn);
}

// ---------------------------------------------------------------------------------------
// Whole layers from the module's own weights: packing, offset conv, deformable product and layout
// changes behind one call and one caller-owned workspace.
// ---------------------------------------------------------------------------------------

static long long up256(long long b) { return (b + 255) / 256 * 256; }

// fp32 shapes of the split product (dcn_f32.hip).
static bool split_takes(const bevk::DcnGeom &g, int channels_out) {
  const long long taps = (long long)g.kernel_h * g.kernel_w;
  return taps <= 9 && g.channels > 0 && g.channels % 32 == 0 &&
         (long long)g.batch * g.height * g.width * g.channels * 4 <= kMaxBufferBytes &&
         bevk::f32_split_weight_bytes(channels_out, taps * g.channels) <= kMaxBufferBytes &&
         (long long)g.batch * g.height_col * g.width_col < (1LL << 30);
}

static bevk::DcnGeom ws_geom(int batch_size, int channels, int height_im, int width_im, int height_col,
                             int width_col, int kernel_h, int kernel_w, int dg) {
  return make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h, kernel_w,
                   0, 0, 1, 1, 1, 1, dg);
}

static bool ws_sizes_ok(const bevk::DcnGeom &g, int channels_out) {
  return g.batch > 0 && g.channels > 0 && g.height > 0 && g.width > 0 && g.height_col > 0 &&
         g.width_col > 0 && g.kernel_h > 0 && g.kernel_w > 0 && channels_out > 0 &&
         g.deformable_group > 0 && g.channels % g.deformable_group == 0;
}

int64_t bevk_dcn_layer_nchw_f32_workspace_bytes(int batch_size, int channels, int height_im,
                                                int width_im, int height_col, int width_col,
                                                int channels_out, int kernel_h, int kernel_w,
                                                int deformable_group) {
  const bevk::DcnGeom g = ws_geom(batch_size, channels, height_im, width_im, height_col, width_col,
                                  kernel_h, kernel_w, deformable_group);
  if (!ws_sizes_ok(g, channels_out) || !split_takes(g, channels_out) || batch_size > 65535) return -1;
  const long long k = (long long)kernel_h * kernel_w * channels;
  if (deformable_group > 1 &&
      ((long long)batch_size * height_col * width_col * k * 4 > kMaxBufferBytes ||
       channels / deformable_group % 4 != 0))
    return -1;
  return bevk::dcn_layer_f32_workspace_bytes(g, channels_out);
}

int bevk_dcn_layer_nchw_f32(const float *data_im, const float *data_offset, const float *data_mask,
                            const float *weight, const float *bias, int batch_size, int channels,
                            int height_im, int width_im, int height_col, int width_col,
                            int channels_out, int kernel_h, int kernel_w, int pad_h, int pad_w,
                            int stride_h, int stride_w, int dilation_h, int dilation_w,
                            int deformable_group, void *workspace, int64_t workspace_bytes,
                            float *out, void *stream) {
  const char *fn = "dcn_layer_nchw_f32";
  g_last_error.clear();
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w,
                deformable_group);
  if (int rc = check_geom(fn, g)) return rc;
  const int64_t need = bevk_dcn_layer_nchw_f32_workspace_bytes(
      batch_size, channels, height_im, width_im, height_col, width_col, channels_out, kernel_h,
      kernel_w, deformable_group);
  if (need < 0) return fail(BEVK_ERR_UNSUPPORTED, "%s: shape not taken", fn);
  if (workspace_bytes < need) return fail(BEVK_ERR_INVALID, "%s: workspace too small", fn);
  if (!data_im || !data_offset || !data_mask || !weight || !workspace || !out)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  if (deformable_group > 1 && reinterpret_cast<uintptr_t>(out) % 16 != 0)
    return fail(BEVK_ERR_INVALID, "%s: out must be 16-byte aligned", fn);
  return hip_status(bevk::launch_dcn_layer_f32(g, channels_out, data_im, data_offset, data_mask, weight,
                                               bias, workspace, out, (hipStream_t)stream),
                    fn);
}

// Workspace of the NHWC layers: the main weight's packed or split form, and with the offset conv
// its packed weight and fp32 bias; then the K parts' sums.
struct NhwcWs {
  long long w_off, b_off, part, total;
  bool split;
  long long parts;
};
static bool nhwc_ws(int dtype, const bevk::DcnGeom &g, int cout, bool layer, NhwcWs *out) {
  if (dtype != BEVK_F32 && dtype != BEVK_F16 && dtype != BEVK_BF16) return false;
  if (!ws_sizes_ok(g, cout) || g.channels % (16 / dtype_size(dtype)) != 0) return false;
  const int T = g.kernel_h * g.kernel_w, K = T * g.channels, es = dtype_size(dtype);
  if ((long long)g.batch * g.height * g.width * g.channels * es > kMaxBufferBytes ||
      (long long)g.batch * g.height_col * g.width_col >= (1LL << 30) ||
      (long long)K * (cout + 32) * es > kMaxBufferBytes)
    return false;
  if (layer && dtype != BEVK_F32 && T > 9) return false;
  if (layer && 3 * T > 64) return false;
  NhwcWs w;
  w.split = dtype == BEVK_F32 && split_takes(g, cout);
  w.parts = dtype == BEVK_F32 ? 0 : bevk::dcn_fused_h_parts_bytes(dtype, g, cout);
  long long at = up256(w.split ? bevk::f32_split_weight_bytes(cout, K)
                               : bevk::dcn_packed_weight_elems(dtype, cout, K) * es);
  w.w_off = at;
  if (layer) at += up256(bevk::dcn_packed_weight_elems(dtype, 3 * T, K) * es);
  w.b_off = at;
  if (layer) at += 256;
  w.part = at;
  w.total = at + w.parts;
  *out = w;
  return true;
}

int64_t bevk_dcn_nhwc_workspace_bytes(int dtype, int with_offset_conv, int batch_size, int channels,
                                      int height_im, int width_im, int height_col, int width_col,
                                      int channels_out, int kernel_h, int kernel_w) {
  NhwcWs w;
  const bevk::DcnGeom g = ws_geom(batch_size, channels, height_im, width_im, height_col, width_col,
                                  kernel_h, kernel_w, 1);
  return nhwc_ws(dtype, g, channels_out, with_offset_conv != 0, &w) ? w.total : -1;
}

int bevk_dcn_nhwc_parts(int dtype, int batch_size, int channels, int height_im, int width_im,
                        int height_col, int width_col, int channels_out, int kernel_h, int kernel_w,
                        int *row_blocks) {
  NhwcWs w;
  const bevk::DcnGeom g = ws_geom(batch_size, channels, height_im, width_im, height_col, width_col,
                                  kernel_h, kernel_w, 1);
  int rows = 0;
  const int parts = nhwc_ws(dtype, g, channels_out, false, &w) && dtype != BEVK_F32
                        ? bevk::dcn_fused_h_parts(dtype, g, channels_out, &rows)
                        : 1;
  if (row_blocks) *row_blocks = rows;
  return parts;
}

// The deformable product from a packed / split weight in the workspace; y_f32: offsets are the
// fp32 y.
static hipError_t nhwc_product(int dtype, const bevk::DcnGeom &g, int cout, const NhwcWs &w, char *ws,
                               const void *x, const void *off, int geo, const void *mask,
                               const void *bias, bool relu, void *out, hipStream_t st) {
  if (w.split)
    return bevk::launch_f32_split(&g, cout, g.batch * g.height_col * g.width_col,
                                  g.kernel_h * g.kernel_w * g.channels, x, off, geo, mask, ws,
                                  static_cast<const float *>(bias), static_cast<float *>(out), st, relu);
  if (w.parts > 0 && (geo == bevk::kGeoMask || geo == bevk::kGeoYF32) &&
      reinterpret_cast<uintptr_t>(out) % 16 == 0)
    return bevk::launch_dcn_fused_h(dtype, g, cout, x, off, geo, mask, ws, bias, out, st, nullptr, relu,
                                    reinterpret_cast<float *>(ws + w.part));
  return bevk::launch_dcn_fused_nhwc(dtype, g, cout, x, off, geo, mask, ws, bias, out, st, nullptr, relu);
}

int bevk_dcn_conv_nhwc(int dtype, const void *data_im, const void *data_offset, int offset_last_dim,
                       const void *data_mask, const void *weight, const void *bias, int batch_size,
                       int channels, int height_im, int width_im, int height_col, int width_col,
                       int channels_out, int kernel_h, int kernel_w, int pad_h, int pad_w,
                       int stride_h, int stride_w, int dilation_h, int dilation_w, void *workspace,
                       int64_t workspace_bytes, void *out, void *stream) {
  const char *fn = "dcn_conv_nhwc";
  g_last_error.clear();
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w, 1);
  if (int rc = check_geom(fn, g)) return rc;
  const int taps = kernel_h * kernel_w;
  if (offset_last_dim != 2 * taps && offset_last_dim != 3 * taps)
    return fail(BEVK_ERR_INVALID, "%s: offset last dim must be 2T (%d) or 3T (%d), got %d", fn,
                2 * taps, 3 * taps, offset_last_dim);
  const bool y = offset_last_dim == 3 * taps;
  NhwcWs w;
  if (!nhwc_ws(dtype, g, channels_out, false, &w))
    return fail(BEVK_ERR_UNSUPPORTED, "%s: shape not taken", fn);
  if (workspace_bytes < w.total) return fail(BEVK_ERR_INVALID, "%s: workspace too small", fn);
  if (!data_im || !data_offset || (!y && !data_mask) || !weight || !workspace || !out)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  const hipStream_t st = (hipStream_t)stream;
  char *ws = static_cast<char *>(workspace);
  hipError_t e = w.split ? bevk::launch_f32_split_weight(static_cast<const float *>(weight), channels_out,
                                                         channels, taps, false, ws, st)
                         : bevk::launch_dcn_pack_weight(dtype, weight, channels_out, channels, taps, ws, st);
  if (e == hipSuccess)
    e = nhwc_product(dtype, g, channels_out, w, ws, data_im, data_offset,
                     y ? bevk::kGeoY : bevk::kGeoMask, data_mask, bias, false, out, st);
  return hip_status(e, fn);
}

int bevk_dcn_layer_nhwc(int dtype, const void *data_im, const void *w_off, const void *b_off,
                        int b_off_dtype, const void *weight, const void *bias, int batch_size,
                        int channels, int height_im, int width_im, int height_col, int width_col,
                        int channels_out, int kernel_h, int kernel_w, int pad_h, int pad_w,
                        int stride_h, int stride_w, int dilation_h, int dilation_w, int act_relu,
                        void *workspace, int64_t workspace_bytes, float *y, void *out, void *stream) {
  const char *fn = "dcn_layer_nhwc";
  g_last_error.clear();
  const bevk::DcnGeom g =
      make_geom(batch_size, channels, height_im, width_im, height_col, width_col, kernel_h,
                kernel_w, pad_h, pad_w, stride_h, stride_w, dilation_h, dilation_w, 1);
  if (int rc = check_geom(fn, g)) return rc;
  NhwcWs w;
  if (!nhwc_ws(dtype, g, channels_out, true, &w))
    return fail(BEVK_ERR_UNSUPPORTED, "%s: shape not taken", fn);
  if (workspace_bytes < w.total) return fail(BEVK_ERR_INVALID, "%s: workspace too small", fn);
  if (b_off != nullptr && (b_off_dtype < BEVK_F32 || b_off_dtype > BEVK_BF16 ||
                           (dtype == BEVK_F32 && b_off_dtype != BEVK_F32)))
    return fail(BEVK_ERR_UNSUPPORTED, "%s: b_off must be float32 or a 16-bit layer's type", fn);
  if (!data_im || !w_off || !weight || !workspace || !y || !out)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  const hipStream_t st = (hipStream_t)stream;
  const int taps = kernel_h * kernel_w, n3 = 3 * taps;
  char *ws = static_cast<char *>(workspace);
  void *packed_off = ws + w.w_off;
  const float *bo = static_cast<const float *>(b_off);
  hipError_t e;
  if (dtype == BEVK_F32) {
    e = bevk::launch_dcn_pack_weight(dtype, w_off, n3, channels, taps, packed_off, st);
    if (e == hipSuccess)
      e = w.split ? bevk::launch_f32_split_weight(static_cast<const float *>(weight), channels_out,
                                                  channels, taps, false, ws, st)
                  : bevk::launch_dcn_pack_weight(dtype, weight, channels_out, channels, taps, ws, st);
  } else {
    float *b32 = reinterpret_cast<float *>(ws + w.b_off);
    e = bevk::launch_dcn_prep16(dtype, weight, channels_out, w_off, n3, channels, taps, b_off,
                                b_off_dtype, ws, packed_off, b32, st);
    if (b_off != nullptr) bo = b32;
  }
  if (e != hipSuccess) return hip_status(e, fn);
  if (w.parts == 0 && bevk::dcn_mega_supported(dtype, g, channels_out, out))
    return hip_status(bevk::launch_dcn_mega(dtype, g, channels_out, data_im, packed_off, bo, ws, bias,
                                            act_relu != 0, y, out, st),
                      fn);
  e = bevk::launch_dcn_fused_nhwc(dtype, g, n3, data_im, nullptr, bevk::kGeoRegular, nullptr, packed_off,
                                  bo, y, st);
  if (e == hipSuccess)
    e = nhwc_product(dtype, g, channels_out, w, ws, data_im, y, bevk::kGeoYF32, nullptr, bias,
                     act_relu != 0, out, st);
  return hip_status(e, fn);
}

int bevk_msda_forward(int dtype, const void *value, const int64_t *spatial_shapes,
                      const int64_t *level_start_index, const void *sampling_loc,
                      const void *attn_weight, int batch, int spatial_size, int num_heads,
                      int channels, int num_levels, int num_query, int num_point,
                      int im2col_step, int force_generic, void *output, void *stream) {
  const char *fn = "msda_forward";
  g_last_error.clear();
  if (!valid_dtype(dtype)) return fail(BEVK_ERR_INVALID, "%s: unknown dtype code %d", fn, dtype);
  if (batch < 0 || spatial_size < 0 || num_heads < 0 || channels < 0 || num_levels < 0 ||
      num_query < 0 || num_point < 0)
    return fail(BEVK_ERR_INVALID, "%s: negative size", fn);
  if (im2col_step <= 0) return fail(BEVK_ERR_INVALID, "%s: im2col_step must be positive", fn);
  // binding_musa.mu:308-309
  const int step = batch < im2col_step ? batch : im2col_step;
  if (step > 0 && batch % step != 0)
    return fail(BEVK_ERR_INVALID, "batch must divide im2col_step");
  const long long n = (long long)batch * num_query * num_heads * channels;
  if (n == 0) return ok();
  if (!value || !spatial_shapes || !level_start_index || !sampling_loc || !attn_weight ||
      !output)
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  bevk::MsdaArgs a;
  a.value = value; a.spatial_shapes = spatial_shapes; a.level_start_index = level_start_index;
  a.sampling_loc = sampling_loc; a.attn_weight = attn_weight; a.output = output;
  a.batch = batch; a.spatial_size = spatial_size; a.num_heads = num_heads;
  a.channels = channels; a.num_levels = num_levels; a.num_query = num_query;
  a.num_point = num_point;
  return hip_status(
      bevk::launch_msda_forward(dtype, a, force_generic != 0, (hipStream_t)stream), fn);
}

int64_t bevk_msda_backward_workspace_bytes(int dtype, int batch, int spatial_size,
                                           int num_heads, int channels, int num_levels,
                                           int num_query, int num_point) {
  if (!valid_dtype(dtype) || batch < 0 || spatial_size < 0 || num_heads < 0 || channels < 0 ||
      num_levels < 0 || num_query < 0 || num_point < 0)
    return -1;
  return bevk::msda_backward_workspace_bytes(dtype, batch, spatial_size, num_heads, channels,
                                             num_levels, num_query, num_point);
}

static int msda_backward_run(const char *fn, bool fresh, int dtype, const void *value, const int64_t *spatial_shapes,
                             const int64_t *level_start_index, const void *sampling_loc,
                             const void *attn_weight, const void *grad_output, int64_t go_stride_b,
                             int64_t go_stride_q, int64_t go_stride_h, int64_t go_stride_c,
                             int batch, int spatial_size, int num_heads, int channels,
                             int num_levels, int num_query, int num_point, int im2col_step,
                             int force_generic_col2im, void *grad_value, void *grad_sampling_loc,
                             void *grad_attn_weight, void *workspace, int64_t workspace_bytes,
                             void *stream) {
  g_last_error.clear();
  if (!valid_dtype(dtype)) return fail(BEVK_ERR_INVALID, "%s: unknown dtype code %d", fn, dtype);
  if (batch < 0 || spatial_size < 0 || num_heads < 0 || channels < 0 || num_levels < 0 ||
      num_query < 0 || num_point < 0)
    return fail(BEVK_ERR_INVALID, "%s: negative size", fn);
  if (im2col_step <= 0) return fail(BEVK_ERR_INVALID, "%s: im2col_step must be positive", fn);
  // binding_musa.mu:438-439
  const int step = batch < im2col_step ? batch : im2col_step;
  if (step > 0 && batch % step != 0)
    return fail(BEVK_ERR_INVALID, "batch must divide im2col_step");
  const int64_t value_elems = (int64_t)batch * spatial_size * num_heads * channels;
  const int64_t need = bevk::msda_backward_workspace_min(dtype, value_elems);
  if (workspace_bytes < need)
    return fail(BEVK_ERR_INVALID, "%s: workspace of %lld bytes, %lld needed", fn,
                (long long)workspace_bytes, (long long)need);
  const long long units = (long long)batch * num_query * num_heads;
  // 16-bit grad_value is fully written (narrowed from the cleared accumulator) even when
  // there are no queries; with no values there is nothing to write at all
  if (value_elems == 0 || (units == 0 && need == 0 && !fresh)) return ok();
  if (channels == 0) return ok();
  if (!value || !spatial_shapes || !level_start_index || !grad_value ||
      (units > 0 && (!sampling_loc || !attn_weight || !grad_output || !grad_sampling_loc ||
                     !grad_attn_weight)) ||
      (need > 0 && !workspace))
    return fail(BEVK_ERR_INVALID, "%s: null tensor pointer", fn);
  if (units * 64 >= (1LL << 42))
    return fail(BEVK_ERR_INVALID, "%s: problem too large", fn);
  bevk::MsdaBwdArgs a;
  a.f.value = value; a.f.spatial_shapes = spatial_shapes;
  a.f.level_start_index = level_start_index; a.f.sampling_loc = sampling_loc;
  a.f.attn_weight = attn_weight; a.f.output = nullptr;
  a.f.batch = batch; a.f.spatial_size = spatial_size; a.f.num_heads = num_heads;
  a.f.channels = channels; a.f.num_levels = num_levels; a.f.num_query = num_query;
  a.f.num_point = num_point;
  a.grad_output = grad_output;
  a.go_stride[0] = go_stride_b; a.go_stride[1] = go_stride_q;
  a.go_stride[2] = go_stride_h; a.go_stride[3] = go_stride_c;
  a.grad_value = grad_value; a.grad_loc = grad_sampling_loc; a.grad_attn = grad_attn_weight;
  a.workspace = workspace;
  a.workspace_bytes = workspace_bytes;
  a.fresh = fresh;
  return hip_status(
      bevk::launch_msda_backward(dtype, a, force_generic_col2im != 0, (hipStream_t)stream), fn);
}

int bevk_msda_backward(int dtype, const void *value, const int64_t *spatial_shapes,
                       const int64_t *level_start_index, const void *sampling_loc,
                       const void *attn_weight, const void *grad_output, int64_t go_stride_b,
                       int64_t go_stride_q, int64_t go_stride_h, int64_t go_stride_c,
                       int batch, int spatial_size, int num_heads, int channels,
                       int num_levels, int num_query, int num_point, int im2col_step,
                       int force_generic_col2im, void *grad_value, void *grad_sampling_loc,
                       void *grad_attn_weight, void *workspace, int64_t workspace_bytes,
                       void *stream) {
  return msda_backward_run("msda_backward", false, dtype, value, spatial_shapes, level_start_index, sampling_loc, attn_weight, grad_output,
                           go_stride_b, go_stride_q, go_stride_h, go_stride_c, batch, spatial_size,
                           num_heads, channels, num_levels, num_query, num_point, im2col_step,
                           force_generic_col2im, grad_value, grad_sampling_loc, grad_attn_weight,
                           workspace, workspace_bytes, stream);
}

int bevk_msda_gradients(int dtype, const void *value, const int64_t *spatial_shapes,
                        const int64_t *level_start_index, const void *sampling_loc,
                        const void *attn_weight, const void *grad_output, int64_t go_stride_b,
                        int64_t go_stride_q, int64_t go_stride_h, int64_t go_stride_c,
                        int batch, int spatial_size, int num_heads, int channels,
                        int num_levels, int num_query, int num_point, int im2col_step,
                        int force_generic_col2im, void *grad_value, void *grad_sampling_loc,
                        void *grad_attn_weight, void *workspace, int64_t workspace_bytes,
                        void *stream) {
  return msda_backward_run("msda_gradients", true, dtype, value, spatial_shapes, level_start_index, sampling_loc, attn_weight, grad_output,
                           go_stride_b, go_stride_q, go_stride_h, go_stride_c, batch, spatial_size,
                           num_heads, channels, num_levels, num_query, num_point, im2col_step,
                           force_generic_col2im, grad_value, grad_sampling_loc, grad_attn_weight,
                           workspace, workspace_bytes, stream);
}

}  // extern "C"
