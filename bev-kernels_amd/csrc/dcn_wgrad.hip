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
//   fp32: three bf16 pieces per element (cut2) and six products, the small ones summed apart
//         (dcn_f32.hip has the arithmetic and its errors); 32 pixels per step. A tile that
//         meets NaN or Inf is computed again in plain fp32.
// The parts' fp32 sums [parts][n][k] go to a workspace and weight_grad_reduce adds them in part
// order (the same result every run), permutes (t, c) to (c, t) and rounds once.
//
// Measured: 34,800 pixels x 2,304 columns x 256 channels (41 GFLOP) bf16 72 us (library fp32
// product of converted operands 648 us and the conversions 80), fp32 302 us (648), the same work
// at 8,700 x 4,608 x 512 bf16 80, fp32 281 us (357): the matrix cores in fp32 (six products, 205
// us at the rate of a large library product), loads and LDS in 16 bits. Errors against 64 bits at 2,304 / 8,700 / 34,800
// pixels 1.3e-7 / 1.8e-7 / 3.5e-7 (library fp32 0.9e-6 / 1.7e-6 / 1.8e-6).
// The offset conv's weight gradient (CONV) runs the same tiles with plain-convolution columns
// read from the input itself (16-bit inputs are exact in one or two of the pieces, so fewer
// products) and the 3T <= 32 columns of its fp32 output gradient.
//
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
  const void *dout, *cols;  // CONV: cols is the input [B, H, W, C]
  float *part;
  int M, N, K;        // pixels, output channels, columns (T * C)
  int rows, parts;    // pixels per part (a multiple of the step), parts
  int ntn, ntk, per_xcd;
  int ldn;                  // row length of dout
  int C, H, W, Ho, Wo, kw, ph, pw, sh, sw, dh, dw;  // CONV
  uint32_t x_bytes;
};

// bf16 pieces that hold a value of T exactly.
template <typename T> constexpr int pieces() { return std::is_same_v<T, float> ? 3 : std::is_same_v<T, f16> ? 2 : 1; }

// Planes of the two operands, elements of a load and pixels of a step: 16-bit operands go to
// the matrix cores as they are, fp32 dO is cut and X (the columns' type) with it.
template <typename T, typename X> struct Kind {
  static constexpr int PA = 1, PB = 1, V = 8, kStep = 64;
  using M = T;
};
template <typename X> struct Kind<float, X> {
  static constexpr int PA = 3, PB = pieces<X>(), V = 4, kStep = 32;
  using M = bf16;
};

template <typename T> __device__ __forceinline__ floatx4 mfma(int4v a, int4v b, floatx4 c) {
  if constexpr (std::is_same_v<T, f16>)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a),
                                                  __builtin_bit_cast(half8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
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

template <typename T, typename X, int TN, bool CONV>
__global__ void __launch_bounds__(kThreads, 2) weight_grad_kernel(const WParams p) {
  using KD = Kind<T, X>;
  using MT = typename KD::M;
  constexpr int PA = KD::PA, PB = KD::PB, V = KD::V, ST = KD::kStep;
  constexpr int kA = TN * ST * 2, kB = kTK * ST * 2;  // bytes of one plane of each operand
  constexpr int RA = TN / 32, RB = 4;                 // 16-blocks per wave: dO, columns
  __shared__ __attribute__((aligned(16))) char lds[PA * kA + PB * kB];
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
  // row (CONV: the last tap's) and only reach outputs that are not stored.
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(static_cast<const T *>(p.dout) + (int64_t)m0 * p.ldn,
                                              (uint32_t)rows * (uint32_t)p.ldn * sizeof(T));
  const __amdgpu_buffer_rsrc_t rb =
      CONV ? make_rsrc(p.cols, p.x_bytes)
           : make_rsrc(static_cast<const X *>(p.cols) + (int64_t)m0 * p.K,
                       (uint32_t)rows * (uint32_t)p.K * sizeof(X));
  // Load unit of the thread: V columns of 8 consecutive pixels. The first half of the threads
  // (waves 0, 1) loads columns, the second dO.
  constexpr int kUnits = kTK / V * (ST / 8);  // 128
  static_assert(kUnits == kThreads / 2, "one unit per thread");
  const bool is_a = wave >= 2;
  const int u = tid & (kUnits - 1);
  const int cw = is_a ? TN / V : kTK / V;  // units across the columns
  const bool live = !is_a || u < TN / V * (ST / 8);
  const int uc = (u % cw) * V, uo = live ? u / cw : 0;
  const uint32_t ld = is_a ? (uint32_t)p.ldn * sizeof(T) : (uint32_t)p.K * sizeof(X);
  const uint32_t voff = (uint32_t)(uo * 8) * ld +
                        (is_a ? (uint32_t)(n0 + uc) * sizeof(T) : (uint32_t)(k0 + uc) * sizeof(X));
  // CONV: the unit's tap and channel, and the output pixel (cb, ch, cw_) of its next first row.
  const int kc = min(k0 + uc, p.K - V);
  const int tap = CONV ? kc / p.C : 0;
  const int dy = CONV ? (tap / p.kw) * p.dh - p.ph : 0, dx = CONV ? (tap % p.kw) * p.dw - p.pw : 0;
  const uint32_t cc = CONV ? (uint32_t)(kc - tap * p.C) : 0u;
  int cm = m0 + uo * 8, cb = 0, ch = 0, cx = 0;
  if (CONV) {
    cb = cm / (p.Ho * p.Wo);
    const int r = cm - cb * p.Ho * p.Wo;
    ch = r / p.Wo;
    cx = r - ch * p.Wo;
  }
  auto carry = [&]() __attribute__((always_inline)) {
    while (cx >= p.Wo) {
      cx -= p.Wo;
      if (++ch == p.Ho) { ch = 0; ++cb; }
    }
  };
  uint4v v[8];
  auto load = [&](int s) __attribute__((always_inline)) {
    if (is_a || !CONV) {
      const uint32_t so = (uint32_t)(s * ST) * ld;
#pragma unroll
      for (int r = 0; r < 8; ++r)
        v[r] = __builtin_bit_cast(uint4v, is_a ? __builtin_amdgcn_raw_buffer_load_b128(ra, voff + so + r * ld, 0, 0)
                                               : __builtin_amdgcn_raw_buffer_load_b128(rb, voff + so + r * ld, 0, 0));
    } else {
      const int h0 = ch, x0 = cx, b0 = cb;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int ih = ch * p.sh + dy, iw = cx * p.sw + dx;
        const bool ok = cm + r < m0 + rows && ih >= 0 && ih < p.H && iw >= 0 && iw < p.W;
        const uint32_t at = ok ? ((uint32_t)((cb * p.H + ih) * p.W + iw) * (uint32_t)p.C + cc) * sizeof(X)
                               : p.x_bytes;
        if constexpr (sizeof(X) == 4) {
          v[r] = __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(rb, at, 0, 0));
        } else {
          typedef uint32_t u2 __attribute__((ext_vector_type(2)));
          const u2 w = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(rb, at, 0, 0));
          v[r] = uint4v{w[0], w[1], 0u, 0u};
        }
        ++cx;
        carry();
      }
      cm += ST;
      ch = h0; cx = x0 + ST; cb = b0;
      carry();
    }
  };
  float nf = 0.f;  // NaN once a non-finite value was cut
  // Element e of v[r] as fp32 bits (cut operands).
  auto elem = [&](int r, int e, auto tag) __attribute__((always_inline)) {
    using E = decltype(tag);
    if constexpr (std::is_same_v<E, float>) {
      return v[r][e];
    } else if constexpr (std::is_same_v<E, bf16>) {
      return e & 1 ? v[r][e >> 1] & 0xffff0000u : v[r][e >> 1] << 16;
    } else {
      const unsigned short hw = (unsigned short)(e & 1 ? v[r][e >> 1] >> 16 : v[r][e >> 1]);
      return __builtin_bit_cast(uint32_t, (float)__builtin_bit_cast(f16, hw));
    }
  };
  auto store_cut = [&](char *base, int plane, auto cols_tag, auto tag) __attribute__((always_inline)) {
    constexpr int COLS = decltype(cols_tag)::value, NP = pieces<decltype(tag)>();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int4v o[3];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x = __builtin_bit_cast(float, elem(2 * j, e, tag));
        const float y = __builtin_bit_cast(float, elem(2 * j + 1, e, tag));
        if constexpr (NP == 1) {
          o[0][j] = (int)pack_hi(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y));
          nf += (x - x) + (y - y);
        } else {
          const Cut2 c = cut2(x, y);
          o[0][j] = c.h;
          o[1][j] = c.m;
          o[2][j] = c.l;
          nf += c.nf;
        }
      }
      char *d = base + frag_at<COLS>(uc + e, uo);
#pragma unroll
      for (int q = 0; q < NP; ++q) *reinterpret_cast<int4v *>(d + q * plane) = o[q];
    }
  };
  auto store_raw = [&](char *base, auto cols_tag) __attribute__((always_inline)) {
    constexpr int COLS = decltype(cols_tag)::value;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      int4v o;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        o[j] = (int)(e & 1 ? pack_hi(v[2 * j][e >> 1], v[2 * j + 1][e >> 1])
                           : pack_lo(v[2 * j][e >> 1], v[2 * j + 1][e >> 1]));
      *reinterpret_cast<int4v *>(base + frag_at<COLS>(uc + e, uo)) = o;
    }
  };
  auto store = [&]() __attribute__((always_inline)) {
    using CA = std::integral_constant<int, TN>;
    using CB = std::integral_constant<int, kTK>;
    if (!live) return;
    if (is_a) {
      if constexpr (PA == 1) store_raw(lds, CA{});
      else store_cut(lds, kA, CA{}, float{});
    } else {
      if constexpr (PA == 1) store_raw(lds + PA * kA, CB{});
      else store_cut(lds + PA * kA, kB, CB{}, X{});
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
      const char *la = lds + sub * TN * 64, *lb = lds + PA * kA + sub * kTK * 64;
      int4v a[RA][PA];
#pragma unroll
      for (int i = 0; i < RA; ++i)
#pragma unroll
        for (int q = 0; q < PA; ++q) a[i][q] = frag(la, wa + i, q * kA);
#pragma unroll
      for (int j = 0; j < RB; ++j) {
        int4v b[PB];
#pragma unroll
        for (int q = 0; q < PB; ++q) b[q] = frag(lb, wb + j, q * kB);
        if constexpr (PA == 1) {
#pragma unroll
          for (int i = 0; i < RA; ++i) acc[i][j] = mfma<MT>(a[i][0], b[0], acc[i][j]);
        } else {
          // small products (piece qa of dO, qb of the columns, qa + qb <= 2), then the large one
          floatx4 lo[RA];
#pragma unroll
          for (int i = 0; i < RA; ++i) lo[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int sum = 2; sum >= 1; --sum)
#pragma unroll
            for (int qa = sum; qa >= 0; --qa)
              if (sum - qa < PB)
#pragma unroll
                for (int i = 0; i < RA; ++i) lo[i] = mfma<MT>(a[i][qa], b[sum - qa < PB ? sum - qa : 0], lo[i]);
#pragma unroll
          for (int i = 0; i < RA; ++i) acc[i][j] = mfma<MT>(a[i][0], b[0], acc[i][j]);
#pragma unroll
          for (int i = 0; i < RA; ++i) acc[i][j] += lo[i];
        }
      }
    }
    __syncthreads();
  }

  // Lane: column k = 16 j + (lane & 15), channels n = 16 i + 4 (lane >> 4) + e.
  float *out = p.part + (int64_t)part * p.N * p.K;
  if constexpr (PA == 3) {
    if (__syncthreads_or(!(nf == nf))) {
      // plain fp32: column tid % 128, every second channel
      const float *dp = static_cast<const float *>(p.dout) + (int64_t)m0 * p.ldn;
      const X *cp = static_cast<const X *>(p.cols);
      const int k = k0 + (tid & (kTK - 1));
      if (k >= p.K) return;
      const int t = CONV ? k / p.C : 0, c = CONV ? k - t * p.C : 0;
      for (int n = n0 + (tid >> 7); n < min(n0 + TN, p.N); n += 2) {
        float sum = 0.f;
        for (int m = 0; m < rows; ++m) {
          float x = 0.f;
          if constexpr (CONV) {
            const int mm = m0 + m, b = mm / (p.Ho * p.Wo), r = mm - b * p.Ho * p.Wo;
            const int ih = (r / p.Wo) * p.sh - p.ph + (t / p.kw) * p.dh;
            const int iw = (r % p.Wo) * p.sw - p.pw + (t % p.kw) * p.dw;
            if (ih >= 0 && ih < p.H && iw >= 0 && iw < p.W)
              x = (float)cp[((int64_t)(b * p.H + ih) * p.W + iw) * p.C + c];
          } else {
            x = (float)cp[(int64_t)(m0 + m) * p.K + k];
          }
          sum = __builtin_fmaf(dp[(int64_t)m * p.ldn + n], x, sum);
        }
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
Plan plan(int dtype, int64_t M, int64_t N, int64_t K, bool conv = false) {
  const int es = dtype == 0 ? 4 : 2, st = dtype == 0 ? 32 : 64;
  Plan pl;
  pl.tn = conv ? 32 : N > 64 ? 128 : 64;
  const double step_us = conv ? 0.7 : dtype == 0 ? (N > 64 ? 1.83 : 1.0) : (N > 64 ? 0.7 : 0.45);
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
  const dim3 g(8 * p.per_xcd), b(kThreads);
  if (tn == 128) hipLaunchKernelGGL((weight_grad_kernel<T, T, 128, false>), g, b, 0, stream, p);
  else hipLaunchKernelGGL((weight_grad_kernel<T, T, 64, false>), g, b, 0, stream, p);
}

hipError_t launch_reduce(const WParams &p, int C, int T, int out_dtype, void *grad_w,
                         hipStream_t stream) {
  const dim3 grid((unsigned)p.N, (unsigned)((C + 63) / 64)), b(kThreads);
  const size_t lds = (size_t)T * 65 * sizeof(float);
  switch (out_dtype) {
    case 0: hipLaunchKernelGGL((weight_grad_reduce<float>), grid, b, lds, stream, p.part,
                               static_cast<float *>(grad_w), p.N, C, T, p.parts); break;
    case 1: hipLaunchKernelGGL((weight_grad_reduce<f16>), grid, b, lds, stream, p.part,
                               static_cast<f16 *>(grad_w), p.N, C, T, p.parts); break;
    case 2: hipLaunchKernelGGL((weight_grad_reduce<bf16>), grid, b, lds, stream, p.part,
                               static_cast<bf16 *>(grad_w), p.N, C, T, p.parts); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Column sums of a [rows][ld] matrix: a workgroup sums its share of the rows for 8 or 4
// columns per lane, row by row over its waves, into part[workgroup][n]; column_sums_total adds
// the workgroups in order and rounds once.
constexpr int kSumBlocks = 256;
template <typename T>
__global__ void __launch_bounds__(kThreads) column_sums_kernel(const T *__restrict__ src, int64_t rows,
                                                               int ld, int n, float *__restrict__ part) {
  constexpr int V = 16 / sizeof(T);
  __shared__ float s[kThreads][V + 1];
  const int vecs = ld / V;  // 16-byte vectors per row
  const int per = min(vecs, kThreads), lanes = kThreads / per;  // rows side by side
  const int64_t r0 = rows * blockIdx.x / gridDim.x, r1 = rows * (blockIdx.x + 1) / gridDim.x;
  for (int v0 = 0; v0 < vecs; v0 += per) {
    const int col = v0 + threadIdx.x % per, row = threadIdx.x / per;
    float a[V];
#pragma unroll
    for (int e = 0; e < V; ++e) a[e] = 0.f;
    if (row < lanes && col < vecs) {
#pragma unroll 4
      for (int64_t r = r0 + row; r < r1; r += lanes) {
        const Vec<T, V> x = load_vec<T, V>(src + r * ld + col * V);
#pragma unroll
        for (int e = 0; e < V; ++e) a[e] += (float)x.v[e];
      }
    }
#pragma unroll
    for (int e = 0; e < V; ++e) s[threadIdx.x][e] = a[e];
    __syncthreads();
    if ((int)threadIdx.x < per && col < vecs) {
      for (int l = 1; l < lanes; ++l)
#pragma unroll
        for (int e = 0; e < V; ++e) a[e] += s[threadIdx.x + l * per][e];
#pragma unroll
      for (int e = 0; e < V; ++e)
        if (col * V + e < n) part[(int64_t)blockIdx.x * n + col * V + e] = a[e];
    }
    __syncthreads();
  }
}
template <typename O>
__global__ void __launch_bounds__(64) column_sums_total(const float *__restrict__ part, int blocks, int n,
                                                        O *__restrict__ out) {
  const int c = (int)blockIdx.x, l = threadIdx.x;
  float a = 0.f;
  for (int b = l; b < blocks; b += 64) a += part[(int64_t)b * n + c];
  for (int d = 32; d >= 1; d >>= 1) a += __shfl_down(a, d, 64);
  if (l == 0) out[c] = static_cast<O>(a);
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
  WParams p{};
  p.dout = dout; p.cols = cols; p.part = static_cast<float *>(workspace);
  p.M = (int)M; p.N = cout; p.K = K; p.ldn = cout;
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
  return launch_reduce(p, C, T, out_dtype, grad_w, stream);
}

int64_t offset_weight_grad_workspace_bytes(const DcnGeom &g, int n3) {
  const int64_t K = (int64_t)g.channels * g.kernel_h * g.kernel_w;
  const int64_t M = (int64_t)g.batch * g.height_col * g.width_col;
  return plan(0, M, 32, K, true).parts * (int64_t)n3 * K * 4;
}

hipError_t launch_offset_weight_grad(int x_dtype, const DcnGeom &g, int n3, const void *x,
                                     const float *y32, void *workspace, int out_dtype, void *grad_w,
                                     hipStream_t stream) {
  const int T = g.kernel_h * g.kernel_w, K = g.channels * T;
  const int64_t M = (int64_t)g.batch * g.height_col * g.width_col;
  const Plan pl = plan(0, M, 32, K, true);
  WParams p{};
  p.dout = y32; p.cols = x; p.part = static_cast<float *>(workspace);
  p.M = (int)M; p.N = n3; p.K = K; p.ldn = 32;
  p.rows = pl.rows; p.parts = pl.parts;
  p.ntn = 1;
  p.ntk = (K + kTK - 1) / kTK;
  p.per_xcd = (int)(((int64_t)p.ntk * p.parts + 7) / 8);
  p.C = g.channels; p.H = g.height; p.W = g.width; p.Ho = g.height_col; p.Wo = g.width_col;
  p.kw = g.kernel_w; p.ph = g.pad_h; p.pw = g.pad_w; p.sh = g.stride_h; p.sw = g.stride_w;
  p.dh = g.dil_h; p.dw = g.dil_w;
  p.x_bytes = (uint32_t)((int64_t)g.batch * g.height * g.width * g.channels * (x_dtype == 0 ? 4 : 2));
  const dim3 grid(8 * p.per_xcd), b(kThreads);
  switch (x_dtype) {
    case 0: hipLaunchKernelGGL((weight_grad_kernel<float, float, 32, true>), grid, b, 0, stream, p); break;
    case 1: hipLaunchKernelGGL((weight_grad_kernel<float, f16, 32, true>), grid, b, 0, stream, p); break;
    case 2: hipLaunchKernelGGL((weight_grad_kernel<float, bf16, 32, true>), grid, b, 0, stream, p); break;
    default: return hipErrorInvalidValue;
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_reduce(p, g.channels, T, out_dtype, grad_w, stream);
}

int64_t column_sums_workspace_bytes(int n) { return (int64_t)kSumBlocks * n * 4; }

hipError_t launch_column_sums(int dtype, const void *src, int64_t rows, int ld, int n, void *workspace,
                              int out_dtype, void *out, hipStream_t stream) {
  float *part = static_cast<float *>(workspace);
  const int blocks = (int)std::max<int64_t>(1, std::min<int64_t>(kSumBlocks, rows / 16));
  switch (dtype) {
    case 0: hipLaunchKernelGGL((column_sums_kernel<float>), dim3(blocks), dim3(kThreads), 0, stream,
                               static_cast<const float *>(src), rows, ld, n, part); break;
    case 1: hipLaunchKernelGGL((column_sums_kernel<f16>), dim3(blocks), dim3(kThreads), 0, stream,
                               static_cast<const f16 *>(src), rows, ld, n, part); break;
    case 2: hipLaunchKernelGGL((column_sums_kernel<bf16>), dim3(blocks), dim3(kThreads), 0, stream,
                               static_cast<const bf16 *>(src), rows, ld, n, part); break;
    default: return hipErrorInvalidValue;
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  switch (out_dtype) {
    case 0: hipLaunchKernelGGL((column_sums_total<float>), dim3(n), dim3(64), 0, stream, part, blocks, n,
                               static_cast<float *>(out)); break;
    case 1: hipLaunchKernelGGL((column_sums_total<f16>), dim3(n), dim3(64), 0, stream, part, blocks, n,
                               static_cast<f16 *>(out)); break;
    case 2: hipLaunchKernelGGL((column_sums_total<bf16>), dim3(n), dim3(64), 0, stream, part, blocks, n,
                               static_cast<bf16 *>(out)); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace bevk
