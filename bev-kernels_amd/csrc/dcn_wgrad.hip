// DCNv2 weight gradient on gfx950: grad_w[n][c][t] = sum_m dO[m][n] * cols[m][t*C + c], the
// contraction over the output pixels m of the columns' gradient step.
//
// A workgroup (4 waves) computes a TN x 128 tile (output channels x columns) over one part of
// the pixels, wave tiles TN/2 x 64 of v_mfma_f32_16x16x32. Both operands have their pixels in
// rows, the MFMA wants 8 consecutive pixels of one channel per lane: a thread loads 16 bytes
// of 8 consecutive rows and pairs neighbouring rows' elements with v_perm on the way into LDS
// (one instruction per two elements), so no transposed copy exists anywhere and every global
// load is a run of 512 or 256 bytes. LDS holds the fragments in the order they are read.
//   16-bit types: products exact, fp32 sums; 64 pixels per step.
//   fp32: three exact bf16 pieces per element and six products, the small ones summed apart
//         (dcn_f32.hip has the arithmetic and its errors); 32 pixels per step. A tile that
//         meets NaN or Inf is computed again in plain fp32.
// The parts' fp32 sums [parts][n][k] go to a workspace and weight_grad_reduce adds them in part
// order (the same result every run), permutes (t, c) to (c, t) and rounds once.
//
// Measured: 34,800 pixels x 2,304 columns x 256 channels (41 GFLOP) bf16 72 us (library fp32
// product of converted operands 648 us and the conversions 80), fp32 302 us (648), the same work
// at 8,700 x 4,608 x 512 bf16 80, fp32 281 us (357): the matrix cores in fp32 (six products, 205
// us at the rate of a large library product), loads and LDS in 16 bits. Errors against 64 bits
// 3e-7 (library fp32 1.8e-6).
// Why this tile: 128 x 128 leaves room for two workgroups per CU (LDS 32 / 48 KB), so one
// multiplies while the other loads and cuts; the pixels are split into enough parts for that
// many workgroups, which costs 4 bytes per output element and part.
#include "bevk_common.h"
#include "bevk_launch.h"

#include <algorithm>
#include <type_traits>

namespace bevk {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kTK = 128;  // columns per tile

struct WParams {
  const void *dout, *cols;
  float *part;
  int M, N, K;        // pixels, output channels, columns (T * C)
  int rows, parts;    // pixels per part (a multiple of the step), parts
  int ntn, ntk, per_xcd;
};

template <typename T> struct Kind {
  static constexpr int kPlanes = 1, kVec = 8, kStep = 64;
};
template <> struct Kind<float> {
  static constexpr int kPlanes = 3, kVec = 4, kStep = 32;
};

template <typename T> __device__ __forceinline__ floatx4 mfma(int4v a, int4v b, floatx4 c) {
  if constexpr (std::is_same_v<T, f16>)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a),
                                                  __builtin_bit_cast(half8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float high_part(float v) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & 0xffff0000u);
}
// High halves of two words (first in the low half), or low halves.
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}
__device__ __forceinline__ uint32_t pack_lo(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x05040100u);
}

// LDS byte address of (column, pixel octet) in one operand plane: 16-column blocks, 4 octets
// of 256 bytes each per 32 pixels; the column is rotated by its block, so the 16 lanes of a
// store (columns 4 or 8 apart over several blocks) touch every bank once.
template <int COLS>
__device__ __forceinline__ int frag_at(int col, int oct) {
  const int blk = col >> 4;
  return (oct >> 2) * (COLS * 64) + blk * 1024 + (oct & 3) * 256 + (((col & 15) + blk) & 15) * 16;
}

template <typename T, int TN>
__global__ void __launch_bounds__(kThreads, 2) weight_grad_kernel(const WParams p) {
  using KD = Kind<T>;
  constexpr int P = KD::kPlanes, V = KD::kVec, ST = KD::kStep;
  constexpr int kA = TN * ST * 2, kB = kTK * ST * 2;  // bytes of one plane of each operand
  constexpr int RA = TN / 32, RB = 4;                 // 16-blocks per wave: dO, columns
  __shared__ __attribute__((aligned(16))) char lds[P * (kA + kB)];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD x takes a contiguous range of (part, tile): the tiles of a part share its rows in L2.
  const int L = (int)(blockIdx.x & 7) * p.per_xcd + (int)(blockIdx.x >> 3);
  const int ntiles = p.ntn * p.ntk;
  if (L >= ntiles * p.parts) return;  // uniform
  const int part = L / ntiles, tile = L - part * ntiles;
  const int n0 = (tile % p.ntn) * TN, k0 = (tile / p.ntn) * kTK;
  const int m0 = part * p.rows, rows = min(p.rows, p.M - m0);
  // Rows past the part end are out of range and read zeros. Columns past N or K read the next
  // row and only reach outputs that are not stored.
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(static_cast<const T *>(p.dout) + (int64_t)m0 * p.N,
                                              (uint32_t)rows * (uint32_t)p.N * sizeof(T));
  const __amdgpu_buffer_rsrc_t rb = make_rsrc(static_cast<const T *>(p.cols) + (int64_t)m0 * p.K,
                                              (uint32_t)rows * (uint32_t)p.K * sizeof(T));
  // Load unit of the thread: V columns of 8 consecutive pixels. The first half of the threads
  // (waves 0, 1) loads columns' rows, the second dO's.
  constexpr int kUnits = kTK / V * (ST / 8);  // 128
  static_assert(kUnits == kThreads / 2, "one unit per thread");
  const bool is_a = wave >= 2;
  const int u = tid & (kUnits - 1);
  const int cw = is_a ? TN / V : kTK / V;  // units across the columns
  const bool live = !is_a || u < TN / V * (ST / 8);
  const int uc = (u % cw) * V, uo = live ? u / cw : 0;
  const uint32_t ld = (uint32_t)(is_a ? p.N : p.K) * sizeof(T);
  const uint32_t voff = (uint32_t)(uo * 8) * ld + (uint32_t)((is_a ? n0 : k0) + uc) * sizeof(T);
  uint4v v[8];
  auto load = [&](int s) __attribute__((always_inline)) {
    const uint32_t so = (uint32_t)(s * ST) * ld;
#pragma unroll
    for (int r = 0; r < 8; ++r)
      v[r] = __builtin_bit_cast(uint4v, is_a ? __builtin_amdgcn_raw_buffer_load_b128(ra, voff + so + r * ld, 0, 0)
                                             : __builtin_amdgcn_raw_buffer_load_b128(rb, voff + so + r * ld, 0, 0));
  };
  float nf = 0.f;  // NaN once a non-finite value was cut
  auto store = [&]() __attribute__((always_inline)) {
    if (!live) return;
    char *base = lds + (is_a ? 0 : P * kA);
    const int plane = is_a ? kA : kB;
    if constexpr (P == 1) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        int4v o;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[j] = (int)(e & 1 ? pack_hi(v[2 * j][e >> 1], v[2 * j + 1][e >> 1])
                             : pack_lo(v[2 * j][e >> 1], v[2 * j + 1][e >> 1]));
        *reinterpret_cast<int4v *>(base + (is_a ? frag_at<TN>(uc + e, uo) : frag_at<kTK>(uc + e, uo))) = o;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int4v h, m, l;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t x[2], y[2], z[2];
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            x[q] = v[2 * j + q][e];
            const float f = __builtin_bit_cast(float, x[q]);
            const float r = f - high_part(f);
            y[q] = __builtin_bit_cast(uint32_t, r);
            const float t = r - high_part(r);
            z[q] = __builtin_bit_cast(uint32_t, t);
            nf += t;
          }
          h[j] = (int)pack_hi(x[0], x[1]);
          m[j] = (int)pack_hi(y[0], y[1]);
          l[j] = (int)pack_hi(z[0], z[1]);
        }
        char *d = base + (is_a ? frag_at<TN>(uc + e, uo) : frag_at<kTK>(uc + e, uo));
        *reinterpret_cast<int4v *>(d) = h;
        *reinterpret_cast<int4v *>(d + plane) = m;
        *reinterpret_cast<int4v *>(d + 2 * plane) = l;
      }
    }
  };

  floatx4 acc[RA][RB];
#pragma unroll
  for (int i = 0; i < RA; ++i)
#pragma unroll
    for (int j = 0; j < RB; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int wa = (wave & 1) * RA, wb = (wave >> 1) * RB;  // the wave's first blocks
  auto frag = [&](const char *base, int blk, int plane) __attribute__((always_inline)) {
    return *reinterpret_cast<const int4v *>(base + plane + blk * 1024 + (lane >> 4) * 256 +
                                            (((lane & 15) + blk) & 15) * 16);
  };
  const int nsteps = (rows + ST - 1) / ST;
  load(0);
  for (int s = 0; s < nsteps; ++s) {
    store();
    __syncthreads();
    load(s + 1);  // past the part end: out of range, zeros, not used
#pragma unroll
    for (int sub = 0; sub < ST / 32; ++sub) {
      const char *la = lds + sub * TN * 64, *lb = lds + P * kA + sub * kTK * 64;
      int4v a[RA][P];
#pragma unroll
      for (int i = 0; i < RA; ++i)
#pragma unroll
        for (int q = 0; q < P; ++q) a[i][q] = frag(la, wa + i, q * kA);
#pragma unroll
      for (int j = 0; j < RB; ++j) {
        int4v b[P];
#pragma unroll
        for (int q = 0; q < P; ++q) b[q] = frag(lb, wb + j, q * kB);
        if constexpr (P == 1) {
#pragma unroll
          for (int i = 0; i < RA; ++i) acc[i][j] = mfma<T>(a[i][0], b[0], acc[i][j]);
        } else {
          constexpr int kTa[5] = {2, 0, 1, 1, 0}, kTb[5] = {0, 2, 1, 0, 1};
          floatx4 lo[RA];
#pragma unroll
          for (int q = 0; q < 5; ++q)
#pragma unroll
            for (int i = 0; i < RA; ++i)
              lo[i] = mfma<T>(a[i][kTa[q]], b[kTb[q]], q == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : lo[i]);
#pragma unroll
          for (int i = 0; i < RA; ++i) acc[i][j] = mfma<T>(a[i][0], b[0], acc[i][j]);
#pragma unroll
          for (int i = 0; i < RA; ++i) acc[i][j] += lo[i];
        }
      }
    }
    __syncthreads();
  }

  // Lane: column k = 16 j + (lane & 15), channels n = 16 i + 4 (lane >> 4) + e.
  float *out = p.part + (int64_t)part * p.N * p.K;
  if constexpr (P == 3) {
    if (__syncthreads_or(!(nf == nf))) {
      // plain fp32: column tid % 128, every second channel
      const float *dp = static_cast<const float *>(p.dout) + (int64_t)m0 * p.N;
      const float *cp = static_cast<const float *>(p.cols) + (int64_t)m0 * p.K;
      const int k = k0 + (tid & (kTK - 1));
      if (k >= p.K) return;
      for (int n = n0 + (tid >> 7); n < min(n0 + TN, p.N); n += 2) {
        float sum = 0.f;
        for (int m = 0; m < rows; ++m)
          sum = __builtin_fmaf(dp[(int64_t)m * p.N + n], cp[(int64_t)m * p.K + k], sum);
        out[(int64_t)n * p.K + k] = sum;
      }
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < RA; ++i)
#pragma unroll
    for (int j = 0; j < RB; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = n0 + (wa + i) * 16 + 4 * (lane >> 4) + e, k = k0 + (wb + j) * 16 + (lane & 15);
        if (n < p.N && k < p.K) out[(int64_t)n * p.K + k] = acc[i][j][e];
      }
}

// grad_w[n][c][t] = sum over parts of part[.][n][t*C + c], in part order. A workgroup takes up
// to 64 channels c of one n and all taps: runs of 64 floats per tap in, one run out.
template <typename O>
__global__ void __launch_bounds__(kThreads) weight_grad_reduce(const float *__restrict__ part,
                                                               O *__restrict__ gw, int N, int C,
                                                               int T, int parts) {
  extern __shared__ float s[];  // [T][65]
  const int n = (int)blockIdx.x, c0 = (int)blockIdx.y * 64, cn = min(64, C - c0);
  const int64_t K = (int64_t)T * C, NK = (int64_t)N * K;
  for (int i = threadIdx.x; i < T * 64; i += kThreads) {
    const int t = i >> 6, c = i & 63;
    if (c >= cn) continue;
    const float *src = part + (int64_t)n * K + (int64_t)t * C + c0 + c;
    float sum = 0.f;
#pragma unroll 4
    for (int q = 0; q < parts; ++q) sum += src[q * NK];
    s[t * 65 + c] = sum;
  }
  __syncthreads();
  O *dst = gw + ((int64_t)n * C + c0) * T;
  for (int i = threadIdx.x; i < cn * T; i += kThreads) {
    const int c = i / T, t = i - c * T;
    dst[i] = static_cast<O>(s[t * 65 + c]);
  }
}

// Parts of the pixels: the count with the least (workgroups of the fullest CU) x (steps of a
// part) x (time a step takes with a full CU: fp32 1.8 / 1.0 us for 128 / 64 output channels,
// 16-bit types 0.7 / 0.45; alone on a CU 1.4 times that) plus the parts' sums written and read
// at 4 TB/s. Whole steps, and rows that a 31-bit buffer range holds.
struct Plan {
  int tn, parts, rows;
};
Plan plan(int dtype, int64_t M, int64_t N, int64_t K) {
  const int es = dtype == 0 ? 4 : 2, st = dtype == 0 ? 32 : 64;
  Plan pl;
  pl.tn = N > 64 ? 128 : 64;
  const double step_us = dtype == 0 ? (N > 64 ? 1.83 : 1.0) : (N > 64 ? 0.7 : 0.45);
  const int64_t tiles = ((N + pl.tn - 1) / pl.tn) * ((K + kTK - 1) / kTK);
  const int64_t steps = (M + st - 1) / st, cus = std::max(1, device_cus());
  const int64_t cap = (((int64_t)1 << 31) - 4096) / (std::max(N, K) * es * st);
  int64_t best = 0;
  double best_t = 0;
  for (int64_t parts = 1; parts <= std::min<int64_t>(steps, 64) || best == 0; ++parts) {
    const int64_t per = (steps + parts - 1) / parts;
    if (per > cap) continue;
    const int64_t depth = (tiles * parts + cus - 1) / cus;
    const double t = (double)depth * (per + 2) * step_us * (depth == 1 ? 1.4 : 1.0) +
                     (double)(parts * N * K) * 8e-6 / 4.0;
    if (best == 0 || t < best_t) {
      best_t = t;
      best = per;
    }
  }
  pl.rows = (int)(best * st);
  pl.parts = (int)((steps + best - 1) / best);
  return pl;
}

template <typename T>
void launch_tn(const WParams &p, int tn, hipStream_t stream) {
  if (tn == 128)
    hipLaunchKernelGGL((weight_grad_kernel<T, 128>), dim3(8 * p.per_xcd), dim3(kThreads), 0, stream, p);
  else
    hipLaunchKernelGGL((weight_grad_kernel<T, 64>), dim3(8 * p.per_xcd), dim3(kThreads), 0, stream, p);
}

}  // namespace

int64_t weight_grad_workspace_bytes(int dtype, int64_t M, int C, int T, int cout) {
  const int64_t K = (int64_t)C * T;
  return plan(dtype, M, cout, K).parts * (int64_t)cout * K * 4;
}

hipError_t launch_weight_grad(int dtype, const void *cols, const void *dout, int64_t M, int C, int T,
                              int cout, void *workspace, int out_dtype, void *grad_w,
                              hipStream_t stream) {
  const int K = C * T;
  const Plan pl = plan(dtype, M, cout, K);
  WParams p;
  p.dout = dout; p.cols = cols; p.part = static_cast<float *>(workspace);
  p.M = (int)M; p.N = cout; p.K = K;
  p.rows = pl.rows; p.parts = pl.parts;
  p.ntn = (cout + pl.tn - 1) / pl.tn;
  p.ntk = (K + kTK - 1) / kTK;
  const int64_t wgs = (int64_t)p.ntn * p.ntk * p.parts;
  if (wgs > (1 << 28)) return hipErrorInvalidValue;
  p.per_xcd = (int)((wgs + 7) / 8);
  switch (dtype) {
    case 0: launch_tn<float>(p, pl.tn, stream); break;
    case 1: launch_tn<f16>(p, pl.tn, stream); break;
    case 2: launch_tn<bf16>(p, pl.tn, stream); break;
    default: return hipErrorInvalidValue;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const dim3 grid((unsigned)cout, (unsigned)((C + 63) / 64));
  const size_t lds = (size_t)T * 65 * sizeof(float);
  switch (out_dtype) {
    case 0: hipLaunchKernelGGL((weight_grad_reduce<float>), grid, dim3(kThreads), lds, stream, p.part,
                               static_cast<float *>(grad_w), cout, C, T, pl.parts); break;
    case 1: hipLaunchKernelGGL((weight_grad_reduce<f16>), grid, dim3(kThreads), lds, stream, p.part,
                               static_cast<f16 *>(grad_w), cout, C, T, pl.parts); break;
    case 2: hipLaunchKernelGGL((weight_grad_reduce<bf16>), grid, dim3(kThreads), lds, stream, p.part,
                               static_cast<bf16 *>(grad_w), cout, C, T, pl.parts); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace bevk
