// fp32 implicit GEMM on the bf16 matrix cores (gfx950): the fp32 DCNv2 forward and the plain
// fp32 products of its backward.
//
//   out[m, n] = sum_k A[m, k] * W[n, k] (+ bias[n])
//
// with A either the deformable columns of an NHWC input, built on the fly (m = (b, oh, ow),
// k = t*C + c), or the rows of a matrix. Every fp32 operand is cut into three bf16 pieces
// (cut2 in bevk_common.h: exact from 2^-110 up), x = h + m + l, and a product is taken as
//   h*h' + (h*m' + m*h') + (m*m' + h*l' + l*h'),
// six v_mfma_f32_16x16x32_bf16 with fp32 accumulation. What is left out (m*l' + l*m' + l*l')
// is below 2^-23 of the product and of either sign, and the large sum is rounded twice
// per 32 terms instead of once per two terms as with v_mfma_f32_32x32x2_f32, so the sums come
// out closer to the exact ones: 2-norm errors against 64 bits at 64 / 512 / 2,304 / 4,608 terms
// 0.5e-7 / 1.5e-7 / 3.3e-7 / 4.7e-7, where a library fp32 product has 1.4e-7 / 4.1e-7 / 8.6e-7
// / 12e-7 and this layer's fp32 matrix kernel had 5.9e-7 at 2,304 (all six products in one
// accumulator: 7.3e-7). Operands below 2^-110 lose low bits (all nonzero operands of one side at
// 2^-115: 1.1e-6, at 2^-120: 3.5e-5; the library product 2.8e-7).
//
// Bound: the matrix cores. Six cameras at 256 channels of 58 x 100 to 256 (41 GFLOP): 500 us
// on the fp32 matrix cores (82 TFLOP/s of 157), 205-220 us here (1.1-1.2 PFLOP/s of bf16
// products, where a large bf16 library product reaches 1.2 on the same card); with the module's
// preparation launch 225-232 us a call. Left out in turn in an earlier form of 253 us a call: four of
// the six products 100, the gathers 64, the weight loads 12, the blend and cut 10.
// Pairs of row blocks with four independent MFMA chains, or two chains for the small products,
// measured the same or slower: their dependent chain is not what limits.
//
// Non-finite operands do not survive the cut (inf - inf, 0 * inf), nor do those that round to
// Inf as a bf16 (from 3.396e38 up): a workgroup that meets one (in its columns, or flagged when the
// weight was split) computes its tile again in plain fp32 (slow_tile), which has the reference's
// NaN / Inf behaviour.
#include "bevk_common.h"
#include "bevk_launch.h"

#include <hip/amd_detail/amd_hip_unsafe_atomics.h>

#include <algorithm>

namespace bevk {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef int int2v __attribute__((ext_vector_type(2)));

constexpr int kMaxTaps = 9;
constexpr int kThreads = 512;   // 8 waves
constexpr int kBK = 32;         // K step: 128 bytes of an fp32 row
constexpr int kRows = -1;       // GEO: A is a matrix, not deformable columns
constexpr int kTConv = -2;      // GEO: transposed plain convolution of y [B, Ho, Wo, 32]: output
                                // rows are input pixels, 32 terms per tap
constexpr bool deform(int geo) { return geo >= 0; }
constexpr int kBlkBytes = 3072; // split weight block: 16 columns x 32 k, three planes

struct TapGeo {
  float w[4];
  uint32_t o[4];
};

struct Params {
  const void *x, *off, *msk;  // kRows: x is the matrix [M][K]
  const float *yb;
  const void *w;              // split weight, then its flags
  const uint32_t *flags;
  const float *bias;
  const float *addend;        // kTConv: added to the sum before the rounding
  void *out;
  int out_kind;               // 0 fp32, 1 fp16, 2 bf16 (16 bits: kTConv only)
  int plane;                  // > 0: out is [B, Cout, plane] with m = (b, position), fp32
  int relu;
  int C, H, W, Ho, Wo, Cout, kw, ph, pw, sh, sw, dh, dw, M, taps;
  int nb_total, kb_total;     // 16-column blocks, 32-k blocks
  int rb_total, mch, nt, kparts, ksteps;  // 16-row blocks, row chunks, column tiles, K parts
  int per_xcd;
  uint32_t x_bytes, w_bytes;
};

__device__ __forceinline__ floatx4 mfma(int4v a, int4v b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Tap geometry of output row m, tap t: corner byte offsets (out of range when the corner is
// outside the image) and mask-folded bilinear weights; the sample is zero unless -1 < h < H
// and -1 < w < W (modulated_deform_conv.py:256-258, fused_tl.py:146-174).
template <int GEO>
__device__ __forceinline__ TapGeo tap_geo(const Params &p, int m, int t) {
  TapGeo G;
  G.w[0] = G.w[1] = G.w[2] = G.w[3] = 0.f;
  G.o[0] = G.o[1] = G.o[2] = G.o[3] = p.x_bytes;
  const int HoWo = p.Ho * p.Wo;
  const int b = m / HoWo, r = m - b * HoWo, oh = r / p.Wo, ow = r - oh * p.Wo;
  const int ki = t / p.kw, kj = t - ki * p.kw;
  float dy, dx, mk;
  tap_offsets<float, GEO>(p.off, p.msk, p.yb, m, t, p.taps, dy, dx, mk);
  const float h = (float)(oh * p.sh - p.ph + ki * p.dh) + dy;
  const float w = (float)(ow * p.sw - p.pw + kj * p.dw) + dx;
  if (h > -1.f && w > -1.f && h < (float)p.H && w < (float)p.W) {
    const float fh = floorf(h), fw = floorf(w);
    const int hl = (int)fh, wl = (int)fw;
    const float lh = h - fh, lw = w - fw, hh = 1.f - lh, hw = 1.f - lw;
    const uint32_t rowb = (uint32_t)p.C * 4u;
    const uint32_t base = (uint32_t)(b * p.H * p.W + hl * p.W + wl) * rowb;
    const bool y0 = hl >= 0, y1 = hl + 1 <= p.H - 1, x0 = wl >= 0, x1 = wl + 1 <= p.W - 1;
    if (y0 && x0) { G.w[0] = hh * hw * mk; G.o[0] = base; }
    if (y0 && x1) { G.w[1] = hh * lw * mk; G.o[1] = base + rowb; }
    if (y1 && x0) { G.w[2] = lh * hw * mk; G.o[2] = base + (uint32_t)p.W * rowb; }
    if (y1 && x1) { G.w[3] = lh * lw * mk; G.o[3] = base + (uint32_t)(p.W + 1) * rowb; }
  }
  return G;
}

// kTConv: the output pixel of y whose tap t reads input pixel m, or out of range.
__device__ __forceinline__ uint32_t tconv_offset(const Params &p, int m, int t) {
  const int HW = p.H * p.W;
  const int b = m / HW, r = m - b * HW, ih = r / p.W, iw = r - ih * p.W;
  const int ki = t / p.kw, kj = t - ki * p.kw;
  const int nh = ih + p.ph - ki * p.dh, nw = iw + p.pw - kj * p.dw;
  const int oh = nh / p.sh, ow = nw / p.sw;
  const bool ok = nh >= 0 && nw >= 0 && oh * p.sh == nh && ow * p.sw == nw && oh < p.Ho && ow < p.Wo;
  return ok ? (uint32_t)((b * p.Ho + oh) * p.Wo + ow) * (kBK * 4u) : p.x_bytes;
}

// One output value: bias, addend, ReLU and the rounding of 16-bit outputs.
__device__ __forceinline__ void emit(const Params &p, int m, int n, float v, float bias) {
  int64_t at = (int64_t)m * p.Cout + n;
  if (p.plane > 0) {
    const int b = m / p.plane;
    at = ((int64_t)b * p.Cout + n) * p.plane + (m - b * p.plane);
  }
  v += bias;
  if (p.addend != nullptr) v = p.addend[at] + v;
  if (p.relu) v = v < 0.f ? 0.f : v;  // NaN stays NaN, as torch.relu
  if (p.kparts > 1) unsafeAtomicAdd(static_cast<float *>(p.out) + at, v);
  else if (p.out_kind == 0) static_cast<float *>(p.out)[at] = v;
  else if (p.out_kind == 1) static_cast<f16 *>(p.out)[at] = static_cast<f16>(v);
  else static_cast<bf16 *>(p.out)[at] = static_cast<bf16>(v);
}

// LDS address (bytes) of the A tile's 16-byte fragment piece (row, chunk of 8 k) inside one
// plane: rows in 16-row blocks of 1 KB, stored in the order the MFMA fragments are read, so a
// fragment read is 1 KB of consecutive addresses. The row is rotated by 4 per chunk: the
// gather's 8-byte stores (4 rows x 8 half chunks per 32 lanes) then touch every bank once.
__device__ __forceinline__ int a_off(int row, int chunk) {
  return (row >> 4) * 1024 + chunk * 256 + (((row & 15) + 4 * chunk) & 15) * 16;
}

template <int NRB, int GEO>
struct Shape {
  static constexpr int kRowsN = NRB * 16;
  static constexpr int kPlane = NRB * 1024;              // bytes of one A plane
  static constexpr int kSlots = kRowsN * (kBK / 4);      // (row, 4 channels) slots per step
  static constexpr int kNS = (kSlots + kThreads - 1) / kThreads;
  static constexpr int kFullWaves = (kSlots - (kNS - 1) * kThreads) / kWave;
  static constexpr int kNQ = deform(GEO) ? 4 : 1;       // loads per slot
};

// The K loop of one wave. Per step: the MFMAs of A buffer `buf`; meanwhile the next step's
// corners (in registers since the last step) are blended, cut and stored into the other
// buffer, and the loads of the step after are issued (as dcn_fused_h.hip's symmetric kernel:
// about one step of gathers in flight per wave, weight fragments two steps ahead).
template <int NRB, int WN, int GEO, int NS>
__device__ __forceinline__ float k_loop(const Params &p, const TapGeo *geo, char *ring, int n0,
                                        int m0, int k0, int nk, floatx4 (&acc)[NRB * WN / 8][2]) {
  using S = Shape<NRB, GEO>;
  constexpr int R = NRB * WN / 8;   // row blocks of the wave
  constexpr int NP = NS * 4;        // blend pieces per step (slot x element)
  constexpr int NA = NS > 0 ? NS : 1;
  constexpr int NQ = S::kNQ;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, wm = wave / WN;
  const int kv = tid & 7;
  const int spt = GEO == kRows ? p.kb_total : GEO == kTConv ? 1 : p.C / kBK;  // K steps per tap
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(p.x, p.x_bytes);
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(p.w, p.w_bytes);

  uint32_t bo[2];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    const int nb = (n0 >> 4) + wn * 2 + cb;
    bo[cb] = nb < p.nb_total ? (uint32_t)nb * (uint32_t)p.kb_total * kBlkBytes + (uint32_t)lane * 16u
                             : p.w_bytes;
  }
  auto issue_b = [&](int ks, int4v (&br)[2][3]) __attribute__((always_inline)) {
    const uint32_t so = (uint32_t)min(ks, p.kb_total - 1) * kBlkBytes;
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
      for (int q = 0; q < 3; ++q)
        br[cb][q] = __builtin_amdgcn_raw_buffer_load_b128(wr, bo[cb] + q * 1024, so, 0);
  };

  auto slot_row = [&](int i) __attribute__((always_inline)) { return (tid >> 3) + i * (kThreads / 8); };
  floatx4 ra[NA][NQ];
  int it = k0 / spt, ics = k0 - it * spt;  // tap and step in the tap of the next loads
  int bt = it, bcs = ics;                  // the same for the next blend
  // Corner offsets (for the next loads) and weights (for the next blend) of one slot, read
  // from the table a slot ahead of their use.
  uint32_t go[NQ];
  floatx4 w4;
  auto load_go = [&](int i) __attribute__((always_inline)) {
    if constexpr (GEO == kRows) {
      const int m = m0 + slot_row(i);
      go[0] = m < p.M ? ((uint32_t)m * (uint32_t)p.kb_total * kBK + (uint32_t)kv * 4u) * 4u : p.x_bytes;
    } else {
      const int4v o = *reinterpret_cast<const int4v *>(geo[slot_row(i) * p.taps + min(it, p.taps - 1)].o);
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        go[q] = (uint32_t)o[q] == p.x_bytes ? p.x_bytes : (uint32_t)o[q] + (uint32_t)kv * 16u;
    }
  };
  auto load_w = [&](int i) __attribute__((always_inline)) {
    if constexpr (deform(GEO))
      w4 = *reinterpret_cast<const floatx4 *>(geo[slot_row(i) * p.taps + bt].w);
  };
  auto issue_slot = [&](int i) __attribute__((always_inline)) {
    // past the last K step: a step read before, not used
    const uint32_t so = (uint32_t)(GEO == kRows ? min(ics, spt - 1) : ics) * (kBK * 4u);
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      ra[i][q] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(xr, go[q], so, 0));
  };
  auto next_issue = [&]() __attribute__((always_inline)) {
    if (++ics == spt && GEO != kRows) {
      ics = 0;
      ++it;
    }
  };
  auto next_blend = [&]() __attribute__((always_inline)) {
    if (++bcs == spt) {
      bcs = 0;
      bt = min(bt + 1, p.taps - 1);
    }
  };
  float nf = 0.f;  // NaN once a non-finite value was cut
  float pv = 0.f;  // the even element of a pair
  Cut2 pc[2];
  auto blend_one = [&](int i, int e) __attribute__((always_inline)) {
    float v;
    if constexpr (!deform(GEO)) {
      v = ra[i][0][e];
    } else {
      v = w4[0] * ra[i][0][e];
      v = __builtin_fmaf(w4[1], ra[i][1][e], v);
      v = __builtin_fmaf(w4[2], ra[i][2][e], v);
      v = __builtin_fmaf(w4[3], ra[i][3][e], v);
    }
    if (e % 2 == 0) {
      pv = v;
    } else {
      pc[e / 2] = cut2(pv, v);
      nf += pc[e / 2].nf;
    }
  };
  auto store_slot = [&](int i, char *buf) __attribute__((always_inline)) {
    char *d = buf + a_off(slot_row(i), kv >> 1) + (kv & 1) * 8;
    *reinterpret_cast<int2v *>(d) = int2v{pc[0].h, pc[1].h};
    *reinterpret_cast<int2v *>(d + S::kPlane) = int2v{pc[0].m, pc[1].m};
    *reinterpret_cast<int2v *>(d + 2 * S::kPlane) = int2v{pc[0].l, pc[1].l};
  };

  const int fa = a_off(lane & 15, lane >> 4) + wm * R * 1024;  // the wave's first fragment
  auto step = [&](int ks, int4v (&br)[2][3]) __attribute__((always_inline)) {
    const char *tile = ring + (ks & 1) * 3 * S::kPlane;
    char *next = ring + ((ks + 1) & 1) * 3 * S::kPlane;
    int4v af[2][3];
    auto read_frag = [&](int rb) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < 3; ++q)
        af[rb & 1][q] = *reinterpret_cast<const int4v *>(tile + q * S::kPlane + rb * 1024 + fa);
    };
    read_frag(0);
    next_issue();
    if constexpr (NS > 0) {
      load_w(0);
      load_go(0);
    }
#pragma unroll
    for (int rb = 0; rb < R; ++rb) {
      if (rb + 1 < R) read_frag(rb + 1);
      const int4v(&a)[3] = af[rb & 1];
      // The five small products are summed by themselves and added once, so the large sum is
      // rounded twice per K step instead of six times.
      floatx4 lo[2];
      constexpr int kTa[5] = {2, 0, 1, 1, 0}, kTb[5] = {0, 2, 1, 0, 1};
#pragma unroll
      for (int q = 0; q < 5; ++q)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
          lo[cb] = mfma(a[kTa[q]], br[cb][kTb[q]],
                                q == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : lo[cb]);
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) acc[rb][cb] = mfma(a[0], br[cb][0], acc[rb][cb]);
#pragma unroll
      for (int pp = 0; pp < NP; ++pp) {
        if (pp * R / (NA * 4) != rb) continue;
        blend_one(pp / 4, pp % 4);
        if (pp % 4 == 3) {
          store_slot(pp / 4, next);
          issue_slot(pp / 4);
          if (pp / 4 + 1 < NS) {
            load_w(pp / 4 + 1);
            load_go(pp / 4 + 1);
          }
        }
      }
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) acc[rb][cb] += lo[cb];
      __builtin_amdgcn_sched_barrier(0);
    }
    next_blend();
    issue_b(k0 + ks + 2, br);
    __syncthreads();
  };

  int4v b0[2][3], b1[2][3];
  issue_b(k0, b0);
  issue_b(k0 + 1, b1);
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    load_go(i);
    issue_slot(i);
  }
  next_issue();
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    load_w(i);
    load_go(i);
#pragma unroll
    for (int e = 0; e < 4; ++e) blend_one(i, e);
    store_slot(i, ring);
    issue_slot(i);
  }
  next_blend();
  __syncthreads();
  int ks = 0;
  for (; ks + 2 <= nk; ks += 2) {
    step(ks, b0);
    step(ks + 1, b1);
  }
  if (ks < nk) step(ks, b0);
  return nf;
}

// The tile in plain fp32, one output column per thread and 16 rows at a time: only for tiles
// that meet a non-finite operand.
template <int NRB, int WN, int GEO>
__device__ __forceinline__ void slow_tile(const Params &p, const TapGeo *geo, float *At, int n0, int m0,
                                       int rows, int k0, int nk, bool add_bias) {
  constexpr int BN = WN * 32, RT = 16 * BN / kThreads, S4 = deform(GEO) ? 4 : 1;
  const int tid = threadIdx.x, n = n0 + tid % BN, r0 = (tid / BN) * RT;
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(p.x, p.x_bytes);
  const int spt = GEO == kRows ? p.kb_total : GEO == kTConv ? 1 : p.C / kBK;
  const unsigned short *w = static_cast<const unsigned short *>(p.w);
  for (int rb = 0; rb * 16 < rows; ++rb) {
    float s[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) s[r] = 0.f;
    for (int ks = k0; ks < k0 + nk; ++ks) {
      __syncthreads();
      {
        const int row = tid >> 5, c = tid & 31;
        float v = 0.f;
        if constexpr (GEO == kRows) {
          const int m = m0 + rb * 16 + row;
          if (m < p.M) v = buffer_load_one<float>(xr, ((uint32_t)m * (uint32_t)p.kb_total + ks) * (kBK * 4u) + c * 4u);
        } else {
          const int t = ks / spt;
          const TapGeo G = geo[(rb * 16 + row) * p.taps + t];
          const uint32_t cb = (uint32_t)((ks - t * spt) * kBK + c) * 4u;
          for (int q = 0; q < S4; ++q) {
            const float xv = G.o[q] == p.x_bytes ? 0.f : buffer_load_one<float>(xr, G.o[q] + cb);
            v = !deform(GEO) ? xv : q == 0 ? G.w[0] * xv : __builtin_fmaf(G.w[q], xv, v);
          }
        }
        At[row * kBK + c] = v;
      }
      __syncthreads();
      if (n < p.Cout) {
        const unsigned short *blk = w + ((int64_t)(n >> 4) * p.kb_total + ks) * (kBlkBytes / 2);
        for (int kk = 0; kk < kBK; ++kk) {
          const int e = ((n & 15) + 16 * (kk >> 3)) * 8 + (kk & 7);
          float wv = 0.f;
          for (int q = 2; q >= 0; --q)
            wv += __builtin_bit_cast(float, (uint32_t)blk[q * 512 + e] << 16);
#pragma unroll
          for (int r = 0; r < RT; ++r) s[r] = __builtin_fmaf(At[(r0 + r) * kBK + kk], wv, s[r]);
        }
      }
    }
    const float bv = (add_bias && p.bias != nullptr && n < p.Cout) ? p.bias[n] : 0.f;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int m = m0 + rb * 16 + r0 + r;
      if (m < p.M && rb * 16 + r0 + r < rows && n < p.Cout) emit(p, m, n, s[r], bv);
    }
  }
}

// One workgroup: up to NRB 16-row blocks x 32 WN columns, the whole K or one of two parts.
template <int NRB, int WN, int GEO>
__global__ void __launch_bounds__(kThreads) f32_gemm_kernel(const Params p) {
  using S = Shape<NRB, GEO>;
  constexpr int R = NRB * WN / 8;
  __shared__ __attribute__((aligned(16))) char ring[2 * 3 * S::kPlane];
  __shared__ __attribute__((aligned(16))) TapGeo geo[GEO == kRows ? 1 : S::kRowsN * kMaxTaps];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroup b runs on XCD b % 8 and each XCD takes a contiguous range of (column tile,
  // K part, row chunk), rows fastest: its L2 keeps the weight of few column tiles and the
  // image rows of neighbouring chunks.
  const int L = (int)(blockIdx.x & 7) * p.per_xcd + (int)(blockIdx.x >> 3);
  if (L >= p.mch * p.nt * p.kparts) return;  // uniform
  const int mc = L % p.mch, nk_id = L / p.mch;
  const int kz = nk_id % p.kparts, n0 = (nk_id / p.kparts) * (WN * 32);
  const int rb0 = (int)((int64_t)p.rb_total * mc / p.mch);
  const int nrb = (int)((int64_t)p.rb_total * (mc + 1) / p.mch) - rb0;  // at most NRB
  const int m0 = rb0 * 16, rows = nrb * 16;
  const int k0 = kz * p.ksteps, nk = min(p.ksteps, p.kb_total - k0);

  bool bad = false;  // a non-finite weight in this tile's columns and K part
  for (int nb = n0 >> 4; nb < min((n0 >> 4) + 2 * WN, p.nb_total); ++nb)
    for (int kb = tid; kb < nk; kb += kThreads) bad |= p.flags[(int64_t)nb * p.kb_total + k0 + kb] != 0;
  if constexpr (GEO != kRows) {
    for (int g = tid; g < S::kRowsN * p.taps; g += kThreads) {
      const int row = g / p.taps, t = g - row * p.taps, m = m0 + row;
      if (row < rows && m < p.M) {
        if constexpr (GEO == kTConv) geo[g].o[0] = tconv_offset(p, m, t);
        else geo[g] = tap_geo<GEO>(p, m, t);
      } else {
        TapGeo G;
        G.w[0] = G.w[1] = G.w[2] = G.w[3] = 0.f;
        G.o[0] = G.o[1] = G.o[2] = G.o[3] = p.x_bytes;
        geo[g] = G;
      }
    }
    __syncthreads();
  }
  floatx4 acc[R][2];
#pragma unroll
  for (int i = 0; i < R; ++i) acc[i][0] = acc[i][1] = floatx4{0.f, 0.f, 0.f, 0.f};
  float nf = 0.f;
  if (wave < S::kFullWaves)
    nf = k_loop<NRB, WN, GEO, S::kNS>(p, geo, ring, n0, m0, k0, nk, acc);
  else if constexpr (S::kFullWaves < 8)
    nf = k_loop<NRB, WN, GEO, S::kNS - 1>(p, geo, ring, n0, m0, k0, nk, acc);
  bad |= !(nf == nf);
  if (__syncthreads_or(bad)) {
    slow_tile<NRB, WN, GEO>(p, geo, reinterpret_cast<float *>(ring), n0, m0, rows, k0, nk, kz == 0);
    return;
  }
  const int wn = wave % WN, wm = wave / WN;
  if (p.plane > 0 && (p.plane & 1) == 0) {
    // NCHW: a lane's four rows are consecutive positions of its channel's plane
    float *outf = static_cast<float *>(p.out);
    const bool quad = (p.plane & 3) == 0;
#pragma unroll
    for (int rb = 0; rb < R; ++rb) {
      const int row = (wm * R + rb) * 16 + 4 * (lane >> 4);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const int m = m0 + row + 2 * hf;
        if (row >= rows || m >= p.M || (quad && hf)) continue;
        const int b = m / p.plane;
        const int64_t at = (int64_t)b * p.Cout * p.plane + (m - b * p.plane);
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
          const int n = n0 + wn * 32 + cb * 16 + (lane & 15);
          if (n >= p.Cout) continue;
          const float bv = p.bias != nullptr ? p.bias[n] : 0.f;
          const floatx4 v = acc[rb][cb] + floatx4{bv, bv, bv, bv};
          typedef float floatx2 __attribute__((ext_vector_type(2)));
          float *d = outf + at + (int64_t)n * p.plane;
          if (quad) *reinterpret_cast<floatx4 *>(d) = v;
          else *reinterpret_cast<floatx2 *>(d) = hf ? floatx2{v[2], v[3]} : floatx2{v[0], v[1]};
        }
      }
    }
    return;
  }
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    const int n = n0 + wn * 32 + cb * 16 + (lane & 15);
    const float bv = (kz == 0 && p.bias != nullptr && n < p.Cout) ? p.bias[n] : 0.f;
#pragma unroll
    for (int rb = 0; rb < R; ++rb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = (wm * R + rb) * 16 + 4 * (lane >> 4) + e, m = m0 + row;
        if (row < rows && m < p.M && n < p.Cout) emit(p, m, n, acc[rb][cb][e], bv);
      }
  }
}

// Small problems: a workgroup takes one 16-row block x 64 columns and its eight waves take every
// eighth K step each, without barriers: a lane builds its MFMA A fragment (one row, 8 channels)
// straight from the corners, the next step's loads are in flight while a step multiplies, and the
// waves' sums meet in LDS at the end. The tiled kernel needs about 1.4 us per K step when few
// workgroups are on the chip (each step waits for its loads and a barrier); here eight steps wait
// together. A whole layer of 64 channels of 32 x 32 to 64: 23.5 -> 16 us.
constexpr int kSmallCols = 64;
template <int GEO>
__global__ void __launch_bounds__(kThreads) f32_small_kernel(const Params p) {
  constexpr int NQ = deform(GEO) ? 4 : 1, NB = kSmallCols / 16, kPitch = kSmallCols + 1;
  __shared__ __attribute__((aligned(16))) TapGeo geo[deform(GEO) ? 16 * kMaxTaps : 1];
  __shared__ float red[8][16 * kPitch];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int L = (int)(blockIdx.x & 7) * p.per_xcd + (int)(blockIdx.x >> 3);
  if (L >= p.mch * p.nt) return;  // uniform
  const int m0 = L % p.mch * 16, n0 = L / p.mch * kSmallCols;
  const int spt = GEO == kRows ? p.kb_total : p.C / kBK;
  bool bad = false;
  for (int i = tid; i < NB * p.kb_total; i += kThreads) {
    const int nb = (n0 >> 4) + i / p.kb_total;
    bad |= nb < p.nb_total && p.flags[(int64_t)nb * p.kb_total + i % p.kb_total] != 0;
  }
  if constexpr (deform(GEO)) {
    for (int g = tid; g < 16 * p.taps; g += kThreads) {
      const int row = g / p.taps, t = g - row * p.taps, m = m0 + row;
      TapGeo G;
      G.w[0] = G.w[1] = G.w[2] = G.w[3] = 0.f;
      G.o[0] = G.o[1] = G.o[2] = G.o[3] = p.x_bytes;
      if (m < p.M) G = tap_geo<GEO>(p, m, t);
      geo[g] = G;
    }
    __syncthreads();
  }
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(p.x, p.x_bytes);
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(p.w, p.w_bytes);
  const int row = lane & 15, oct = lane >> 4;
  uint32_t bo[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int nb = (n0 >> 4) + j;
    bo[j] = nb < p.nb_total ? (uint32_t)nb * (uint32_t)p.kb_total * kBlkBytes + (uint32_t)lane * 16u
                            : p.w_bytes;
  }
  struct Step {
    floatx4 a[NQ][2], w;
    int4v b[NB][3];
  };
  auto load = [&](int ks, Step &st) __attribute__((always_inline)) {
    uint32_t o[NQ];
    if constexpr (GEO == kRows) {
      const int m = m0 + row;
      o[0] = m < p.M ? ((uint32_t)m * (uint32_t)p.kb_total + (uint32_t)ks) * (kBK * 4u) + (uint32_t)oct * 32u
                     : p.x_bytes;
    } else {
      const int t = ks / spt;
      const TapGeo &G = geo[row * p.taps + t];
      const uint32_t cb = (uint32_t)(ks - t * spt) * (kBK * 4u) + (uint32_t)oct * 32u;
      st.w = *reinterpret_cast<const floatx4 *>(G.w);
#pragma unroll
      for (int q = 0; q < NQ; ++q) o[q] = G.o[q] == p.x_bytes ? p.x_bytes : G.o[q] + cb;
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
        st.a[q][hf] = __builtin_bit_cast(
            floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                         xr, o[q] == p.x_bytes ? p.x_bytes : o[q] + hf * 16u, 0, 0));
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int q = 0; q < 3; ++q)
        st.b[j][q] = __builtin_amdgcn_raw_buffer_load_b128(wr, bo[j] + q * 1024, (uint32_t)ks * kBlkBytes, 0);
  };
  floatx4 hi[NB], lo[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) hi[j] = lo[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  float nf = 0.f;
  auto multiply = [&](const Step &st) __attribute__((always_inline)) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = st.a[0][e >> 2][e & 3];
      if constexpr (deform(GEO)) {
        v[e] *= st.w[0];
#pragma unroll
        for (int q = 1; q < NQ; ++q) v[e] = __builtin_fmaf(st.w[q], st.a[q][e >> 2][e & 3], v[e]);
      }
    }
    int4v a[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const Cut2 c = cut2(v[2 * e], v[2 * e + 1]);
      a[0][e] = c.h; a[1][e] = c.m; a[2][e] = c.l;
      nf += c.nf;
    }
    constexpr int kTa[5] = {2, 0, 1, 1, 0}, kTb[5] = {0, 2, 1, 0, 1};
#pragma unroll
    for (int q = 0; q < 5; ++q)
#pragma unroll
      for (int j = 0; j < NB; ++j) lo[j] = mfma(a[kTa[q]], st.b[j][kTb[q]], lo[j]);
#pragma unroll
    for (int j = 0; j < NB; ++j) hi[j] = mfma(a[0], st.b[j][0], hi[j]);
  };
  const int kb = p.kb_total;
  if (wave < kb) {
    Step s0, s1;
    load(wave, s0);
    for (int ks = wave;;) {  // a step past the end repeats the last one, not used
      load(min(ks + 8, kb - 1), s1);
      multiply(s0);
      if ((ks += 8) >= kb) break;
      load(min(ks + 8, kb - 1), s0);
      multiply(s1);
      if ((ks += 8) >= kb) break;
    }
  }
  bad |= !(nf == nf);
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      red[wave][(4 * (lane >> 4) + e) * kPitch + 16 * j + (lane & 15)] = hi[j][e] + lo[j][e];
  const bool slow = __syncthreads_or(bad);
  // Two outputs per thread: consecutive rows of a column (NCHW: a channel's positions), or
  // consecutive columns of a row.
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int i = 2 * tid + u;
    const int r = p.plane > 0 ? i & 15 : i / kSmallCols, c = p.plane > 0 ? i >> 4 : i % kSmallCols;
    const int m = m0 + r, n = n0 + c;
    if (m >= p.M || n >= p.Cout) continue;
    float v = 0.f;
    if (!slow) {
#pragma unroll
      for (int w = 0; w < 8; ++w) v += red[w][r * kPitch + c];
    } else {  // plain fp32
      for (int k = 0; k < kb * kBK; ++k) {
        const int ks = k / kBK, kk = k % kBK;
        float x = 0.f;
        if constexpr (GEO == kRows) {
          x = static_cast<const float *>(p.x)[(int64_t)m * kb * kBK + k];
        } else {
          const int t = ks / spt;
          const TapGeo &G = geo[r * p.taps + t];
          for (int q = 0; q < 4; ++q) {
            const float xv = G.o[q] == p.x_bytes
                                 ? 0.f
                                 : buffer_load_one<float>(xr, G.o[q] + (uint32_t)(k - t * spt * kBK) * 4u);
            x = q == 0 ? G.w[0] * xv : __builtin_fmaf(G.w[q], xv, x);
          }
        }
        const unsigned short *blk = static_cast<const unsigned short *>(p.w) +
                                    ((int64_t)(n >> 4) * kb + ks) * (kBlkBytes / 2);
        const int e = ((n & 15) + 16 * (kk >> 3)) * 8 + (kk & 7);
        float wv = 0.f;
        for (int q = 2; q >= 0; --q) wv += __builtin_bit_cast(float, (uint32_t)blk[q * 512 + e] << 16);
        v = __builtin_fmaf(x, wv, v);
      }
    }
    emit(p, m, n, v, p.bias != nullptr ? p.bias[n] : 0.f);
  }
}

// The three pieces of a lane's 8 values of a split block. A pair with a value that is not finite
// or rounds to Inf is cut off instead (the pieces of a finite value still add up to it; Inf and NaN
// are kept whole in the first piece), for slow_tile. Returns whether there was one.
__device__ __forceinline__ bool store_split(char *d, const float (&v)[8]) {
  int4v h, m, l;
  bool bad = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    Cut2 c = cut2(v[2 * e], v[2 * e + 1]);
    if (!(c.nf == c.nf)) {
      bad = true;
      uint32_t p[2][3];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        float x = v[2 * e + q];
        if (!(x == x)) x = __builtin_nanf("");
        const bool fin = __builtin_fabsf(x) <= 3.402823466e38f;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          p[q][i] = i == 0 || fin ? __builtin_bit_cast(uint32_t, x) & 0xffff0000u : 0u;
          x -= __builtin_bit_cast(float, p[q][i]);
        }
      }
      c.h = (int)(p[0][0] >> 16 | p[1][0]);
      c.m = (int)(p[0][1] >> 16 | p[1][1]);
      c.l = (int)(p[0][2] >> 16 | p[1][2]);
    }
    h[e] = c.h; m[e] = c.m; l[e] = c.l;
  }
  *reinterpret_cast<int4v *>(d) = h;
  *reinterpret_cast<int4v *>(d + 1024) = m;
  *reinterpret_cast<int4v *>(d + 2048) = l;
  return bad;
}

// ---------------------------------------------------------------------------------------
// Split weight: blocks [N / 16][K / 32] of 3 KB, planes h, m, l of 64 lanes x 8 bf16 in the
// MFMA fragment order (lane l: column l % 16, k = 8 (l / 16) .. + 8), then one flag word per
// block (a non-finite value in it). From the module weight w [Cout][C][T]:
//   TRANS false: n = Cout, k = t*C + c (the forward);
//   TRANS true:  n = t*C + c, k = Cout (columns' gradient dO @ W).
// A workgroup stages a 16 x 32 (n x c, or c x Cout) group of all taps through LDS, where each
// source row's span is contiguous.
// ---------------------------------------------------------------------------------------
constexpr int kSplitLds = 16 * (32 * kMaxTaps + 1);  // floats; 32 x (16 * 9 + 1) is fewer + 16
template <bool TRANS>
__device__ __forceinline__ void split_weight_block(const float *__restrict__ w, char *packed,
                                                   uint32_t *__restrict__ flags, int cout, int C, int T,
                                                   int kb_total, int bx, int by, float *s) {
  constexpr int RO = TRANS ? 32 : 16, CO = TRANS ? 16 : 32;  // source rows (Cout), channels
  static_assert(RO * (CO * kMaxTaps + 1) <= kSplitLds + 16, "LDS of a block");
  const int r0 = bx * RO, c0 = by * CO;
  const int span = CO * T, pitch = span + 1;
  const int vspan = span / 4;  // CO is a multiple of 16
  const bool aligned = (reinterpret_cast<uintptr_t>(w) & 15) == 0;
  for (int i = threadIdx.x; i < RO * vspan; i += 256) {
    const int r = i / vspan, v = (i - r * vspan) * 4;
    const float *src = w + ((int64_t)(r0 + r) * C + c0) * T + v;
    floatx4 x = {0.f, 0.f, 0.f, 0.f};
    if (r0 + r < cout) {
      if (aligned) x = *reinterpret_cast<const floatx4 *>(src);
      else x = floatx4{src[0], src[1], src[2], src[3]};
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s[r * pitch + v + e] = x[e];
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  for (int t = threadIdx.x >> 6; t < T; t += 4) {  // a wave takes whole blocks (one per tap)
    const int64_t blk = TRANS ? (int64_t)((t * C + c0) >> 4) * kb_total + bx
                              : (int64_t)bx * kb_total + ((t * C + c0) >> 5);
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int n = lane & 15, k = (lane >> 4) * 8 + e;
      v[e] = TRANS ? s[k * pitch + n * T + t] : s[n * pitch + k * T + t];
    }
    const bool bad = store_split(packed + blk * kBlkBytes + lane * 16, v);
    const bool any = __any(bad);
    if (lane == 0) flags[blk] = any ? 1u : 0u;
  }
}
template <bool TRANS>
__global__ void __launch_bounds__(256) split_weight_kernel(const float *__restrict__ w, char *packed,
                                                           uint32_t *__restrict__ flags, int cout,
                                                           int C, int T, int kb_total) {
  __shared__ float s[kSplitLds + 16];
  split_weight_block<TRANS>(w, packed, flags, cout, C, T, kb_total, (int)blockIdx.x, (int)blockIdx.y, s);
}

// Everything the NCHW layer's forward needs before its product, in one launch (five short ones
// cost more than a small layer itself: a call with 64 channels of 32 x 32 took 70 us with seven
// launches and takes 28 with three): the input,
// offsets and mask as NHWC copies (64 x 64 tiles through LDS), the split weight, and the cleared
// output where K runs in two parts. Workgroups are dealt to the jobs in that order.
struct PrepJob {
  const float *src;
  float *dst;
  int rows, cols, tr, tc, first;  // [batch][rows][cols] -> [batch][cols][rows], tiles, first block
};
struct PrepParams {
  PrepJob t[3];
  const float *w;
  char *packed;
  uint32_t *flags;
  int cout, C, T, kb_total, nbo, first_w, first_clear, nblocks;
  float *clear;
  int64_t clear4;
};
__global__ void __launch_bounds__(256) f32_prep_kernel(const PrepParams p) {
  __shared__ float s[kSplitLds + 16];
  const int blk = (int)blockIdx.x;
  if (blk >= p.first_clear) {
    const int64_t step = (int64_t)(p.nblocks - p.first_clear) * 256;
    for (int64_t i = (int64_t)(blk - p.first_clear) * 256 + threadIdx.x; i < p.clear4; i += step)
      reinterpret_cast<floatx4 *>(p.clear)[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    return;
  }
  if (blk >= p.first_w) {
    const int i = blk - p.first_w;
    split_weight_block<false>(p.w, p.packed, p.flags, p.cout, p.C, p.T, p.kb_total, i % p.nbo, i / p.nbo, s);
    return;
  }
  const PrepJob &j = blk >= p.t[2].first ? p.t[2] : blk >= p.t[1].first ? p.t[1] : p.t[0];
  const int R = j.rows, C = j.cols;
  int i = blk - j.first;
  const int tc = i % j.tc;
  i /= j.tc;
  const int r0 = (i % j.tr) * 64, c0 = tc * 64;
  const float *src = j.src + (int64_t)(i / j.tr) * R * C;
  float *dst = j.dst + (int64_t)(i / j.tr) * R * C;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const bool vin = (C & 3) == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0;
  const bool vout = (R & 3) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = r0 + ty + 16 * q, c = c0 + 4 * tx;
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    if (vin && r < R && c < C) {
      v = *reinterpret_cast<const floatx4 *>(src + (int64_t)r * C + c);
    } else if (r < R) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < C) v[e] = src[(int64_t)r * C + c + e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s[(ty + 16 * q) * 65 + 4 * tx + e] = v[e];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int c = c0 + ty + 16 * q, r = r0 + 4 * tx;
    floatx4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = s[(4 * tx + e) * 65 + ty + 16 * q];
    if (c >= C) continue;
    if (vout && r < R) {
      *reinterpret_cast<floatx4 *>(dst + (int64_t)c * R + r) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (r + e < R) dst[(int64_t)c * R + r + e] = v[e];
    }
  }
}

// Split offset-conv weight for kTConv: columns n = c, terms k = 32 t + j from w_off [n3][C][T]
// (j < n3 <= 32, zero past it). One wave per block (n / 16, t).
__global__ void __launch_bounds__(256) split_offset_weight_kernel(const float *__restrict__ w,
                                                                  char *packed,
                                                                  uint32_t *__restrict__ flags,
                                                                  int n3, int C, int T, int blocks) {
  const int blk = (int)blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (blk >= blocks) return;
  const int nb = blk / T, t = blk - nb * T, c = nb * 16 + (lane & 15);
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int j = (lane >> 4) * 8 + e;
    v[e] = j < n3 && c < C ? w[((int64_t)j * C + c) * T + t] : 0.f;
  }
  const bool bad = store_split(packed + (int64_t)blk * kBlkBytes + lane * 16, v);
  const bool any = __any(bad);
  if (lane == 0) flags[blk] = any ? 1u : 0u;
}

__global__ void __launch_bounds__(256) clear_f32x4(float *__restrict__ p, int64_t n4) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256)
    reinterpret_cast<float4 *>(p)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Tile height, tile width and K parts. A K step of a workgroup moves NRB * 8 KB of corner
// lines (a quarter of that from a matrix) and 48 KB of weight per 256 columns through the CU's
// vector memory path, about 38 cycles per KB, under NRB * BN * 1.5 cycles of matrix-core work
// per SIMD; the plan with the least (rounds over the CUs) x (steps) x (the larger of the two)
// runs. Tiles of up to 3 row blocks of a matrix leave room for two workgroups on a CU, whose
// steps overlap (8,700 x 512 x 4,608: 220 us with 3 row blocks, 254 with 8; 34,800 x 256 x
// 2,304: 281 and 297). Two K parts add into a cleared output (two addends: the same result in
// any order). Swept over 8 layers and 6 products from 9 to 300 us, the choice was the fastest
// or within 7% of it, one layer 10% off.
// The small kernel: a set of eight K steps moves 160 KB (112 from a matrix) through a CU's vector
// memory path, 2.3 us (1.7), a launch and the final sums take 3 us. Measured against the tiled
// kernel, whole layers: 256 channels of 15 x 25 to 256 33 / 41 us, 512 to 512 62 / 66, 128 of
// 30 x 40 23 / 29; 64 of 58 x 100 26 / 25, 96 to 160 of 4 x 20 x 30 32 / 30: the rule picks the
// faster of each.
struct Plan {
  int nrb, kparts, mch, bn;  // nrb 0: the small kernel
};
Plan plan(const Params &p, int bn_max, bool rows_mode, bool can_split, bool nchw, bool small) {
  const int cus = std::max(1, device_cus());
  Plan best{0, 1, 0, bn_max};
  double best_t = 0;
  for (int bn = bn_max; bn >= 64; bn /= 2)
    for (int kparts = 1; kparts <= (can_split ? 2 : 1); ++kparts)
      for (int nrb = 9; nrb >= 2; --nrb) {
        if ((bn == 128 && nrb % 2) || (bn == 64 && nrb % 4)) continue;
        const int64_t mch = (p.rb_total + nrb - 1) / nrb;
        const int64_t wgs = mch * ((p.Cout + bn - 1) / bn) * kparts;
        const int64_t rounds = (wgs + cus - 1) / cus;
        const int steps = (p.kb_total + kparts - 1) / kparts;
        const double kb = (rows_mode ? 2.0 : 8.0) * nrb + 48.0 * bn / 256, mm = 1.5 * nrb * bn;
        const bool two = rows_mode && nrb <= 3 && wgs > cus;
        double t = two ? steps * std::max(20.0 * kb, mm) + 1200.0
                       : steps * (std::max(38.0 * kb, mm) + 250.0) + 6000.0;
        t *= (double)rounds;
        if (kparts == 2) t += 8000.0 + (double)p.M * p.Cout * 8.0 / 1600.0;  // clear and add
        if (kparts == 2 && nchw) t += 8000.0 + (double)p.M * p.Cout * 8.0 / 1600.0;  // layout change
        if (best.nrb == 0 || t < best_t) {
          best_t = t;
          best = Plan{nrb, kparts, (int)mch, bn};
        }
      }
  const int64_t wgs = (int64_t)p.rb_total * ((p.Cout + kSmallCols - 1) / kSmallCols);
  const double t = (double)((wgs + cus - 1) / cus) *
                   ((p.kb_total + 7) / 8 * (rows_mode ? 4000.0 : 5600.0) + 7000.0);
  if (t < best_t && small) best = Plan{0, 1, p.rb_total, kSmallCols};
  return best;
}

template <int NRB, int WN, int GEO>
void launch_one(const Params &p, hipStream_t stream) {
  hipLaunchKernelGGL((f32_gemm_kernel<NRB, WN, GEO>), dim3(8 * p.per_xcd), dim3(kThreads), 0, stream, p);
}

// Fills in the tiling; returns the tile height and width. nchw: the caller changes the layout of
// a two-part output afterwards.
template <int GEO>
Plan make_plan(Params &p, bool nchw) {
  p.rb_total = (p.M + 15) / 16;
  const bool can_split = deform(GEO) && !p.relu && p.kb_total >= 16 && (int64_t)p.M * p.Cout % 4 == 0 &&
                         reinterpret_cast<uintptr_t>(p.out) % 16 == 0;
  const Plan pl = plan(p, p.Cout > 128 ? 256 : (p.Cout > 64 ? 128 : 64), !deform(GEO), can_split, nchw,
                       GEO != kTConv);
  p.nt = (p.Cout + pl.bn - 1) / pl.bn;
  p.mch = pl.mch;
  p.kparts = pl.kparts;
  p.ksteps = (p.kb_total + pl.kparts - 1) / pl.kparts;
  return pl;
}

template <int GEO>
hipError_t launch_geo(Params p, const Plan &pl, bool cleared, hipStream_t stream) {
  const int bn = pl.bn;
  const int64_t n_out = (int64_t)p.M * p.Cout;
  const int64_t wgs = (int64_t)p.mch * p.nt * p.kparts;
  if (wgs > (1 << 28)) return hipErrorInvalidValue;
  p.per_xcd = (int)((wgs + 7) / 8);
  if constexpr (GEO != kTConv) {
    if (pl.nrb == 0) {
      hipLaunchKernelGGL((f32_small_kernel<GEO>), dim3(8 * p.per_xcd), dim3(kThreads), 0, stream, p);
      return hipGetLastError();
    }
  }
  if (p.kparts == 2 && !cleared) {
    const int64_t n4 = n_out / 4;
    hipLaunchKernelGGL(clear_f32x4, dim3((unsigned)std::min<int64_t>((n4 + 255) / 256, 4096)),
                       dim3(256), 0, stream, static_cast<float *>(p.out), n4);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (bn == 256) {
    switch (pl.nrb) {
      case 2: launch_one<2, 8, GEO>(p, stream); break;
      case 3: launch_one<3, 8, GEO>(p, stream); break;
      case 4: launch_one<4, 8, GEO>(p, stream); break;
      case 5: launch_one<5, 8, GEO>(p, stream); break;
      case 6: launch_one<6, 8, GEO>(p, stream); break;
      case 7: launch_one<7, 8, GEO>(p, stream); break;
      case 8: launch_one<8, 8, GEO>(p, stream); break;
      default: launch_one<9, 8, GEO>(p, stream); break;
    }
  } else if (bn == 128) {
    switch (pl.nrb) {
      case 2: launch_one<2, 4, GEO>(p, stream); break;
      case 4: launch_one<4, 4, GEO>(p, stream); break;
      case 6: launch_one<6, 4, GEO>(p, stream); break;
      default: launch_one<8, 4, GEO>(p, stream); break;
    }
  } else {
    if (pl.nrb == 4) launch_one<4, 2, GEO>(p, stream);
    else launch_one<8, 2, GEO>(p, stream);
  }
  return hipGetLastError();
}

}  // namespace

int64_t f32_split_weight_bytes(int64_t n, int64_t k) {
  return ((n + 15) / 16) * ((k + 31) / 32) * (kBlkBytes + 4);
}

hipError_t launch_f32_split_weight(const float *w, int cout, int C, int T, bool transposed,
                                   void *packed, hipStream_t stream) {
  const int n = transposed ? C * T : cout, k = transposed ? cout : C * T;
  const int kb = (k + 31) / 32;
  char *d = static_cast<char *>(packed);
  uint32_t *flags = reinterpret_cast<uint32_t *>(d + (int64_t)((n + 15) / 16) * kb * kBlkBytes);
  if (transposed)
    hipLaunchKernelGGL((split_weight_kernel<true>), dim3((cout + 31) / 32, C / 16), dim3(256), 0,
                       stream, w, d, flags, cout, C, T, kb);
  else
    hipLaunchKernelGGL((split_weight_kernel<false>), dim3((cout + 15) / 16, C / 32), dim3(256), 0,
                       stream, w, d, flags, cout, C, T, kb);
  return hipGetLastError();
}

namespace {
Params make_params(const DcnGeom *g, int channels_out, int M, int K, const void *x, const void *off,
                   const void *msk, const void *w_split, const float *bias, float *out, bool relu) {
  Params p{};
  p.x = x; p.off = off; p.msk = msk; p.w = w_split; p.bias = bias; p.out = out;
  p.relu = relu ? 1 : 0;
  p.Cout = channels_out;
  p.nb_total = (channels_out + 15) / 16;
  p.M = M;
  p.kb_total = K / kBK;
  p.taps = 1;
  if (g != nullptr) {
    p.C = g->channels; p.H = g->height; p.W = g->width; p.Ho = g->height_col; p.Wo = g->width_col;
    p.kw = g->kernel_w; p.ph = g->pad_h; p.pw = g->pad_w; p.sh = g->stride_h; p.sw = g->stride_w;
    p.dh = g->dil_h; p.dw = g->dil_w;
    p.taps = g->kernel_h * g->kernel_w;
    p.x_bytes = (uint32_t)((int64_t)g->batch * g->height * g->width * g->channels * 4);
  } else {
    p.x_bytes = (uint32_t)((int64_t)M * K * 4);
  }
  p.w_bytes = (uint32_t)((int64_t)p.nb_total * p.kb_total * kBlkBytes);
  p.flags = reinterpret_cast<const uint32_t *>(static_cast<const char *>(w_split) + p.w_bytes);
  return p;
}
}  // namespace

hipError_t launch_f32_split(const DcnGeom *g, int channels_out, int M, int K, const void *x,
                            const void *off, int geo, const void *msk, const void *w_split,
                            const float *bias, float *out, hipStream_t stream, bool relu) {
  Params p = make_params(g, channels_out, M, K, x, off, msk, w_split, bias, out, relu);
  if (g == nullptr) {
    const Plan pl = make_plan<kRows>(p, false);
    return launch_geo<kRows>(p, pl, false, stream);
  }
  const Plan pl = make_plan<kGeoMask>(p, false);
  if (geo == kGeoMask) return launch_geo<kGeoMask>(p, pl, false, stream);
  return launch_geo<kGeoYF32>(p, pl, false, stream);  // fp32 y: kGeoY and kGeoYF32 (no bias) are the same
}

// Workspace of the NCHW layer's forward, 256-byte pieces: NHWC input, offsets and mask, split
// weight, then columns (deformable groups) or the NHWC output (room for a two-part product).
namespace {
struct LayerWs {
  int64_t off, msk, w, last, total;
};
LayerWs layer_ws(const DcnGeom &g, int cout) {
  auto up = [](int64_t b) { return (b + 255) / 256 * 256; };
  const int64_t T = g.kernel_h * g.kernel_w, M = (int64_t)g.batch * g.height_col * g.width_col;
  LayerWs l;
  l.off = up((int64_t)g.batch * g.height * g.width * g.channels * 4);
  l.msk = l.off + up(M * g.deformable_group * 2 * T * 4);
  l.w = l.msk + up(M * g.deformable_group * T * 4);
  l.last = l.w + up(f32_split_weight_bytes(cout, T * g.channels));
  l.total = l.last + up(g.deformable_group > 1 ? M * T * g.channels * 4 : M * cout * 4);
  return l;
}
}  // namespace

int64_t dcn_layer_f32_workspace_bytes(const DcnGeom &g, int channels_out) {
  return layer_ws(g, channels_out).total;
}

hipError_t launch_dcn_layer_f32(const DcnGeom &g, int cout, const float *x, const float *off,
                                const float *msk, const float *weight, const float *bias,
                                void *workspace, float *out, hipStream_t stream) {
  const int T = g.kernel_h * g.kernel_w, dg = g.deformable_group, HoWo = g.height_col * g.width_col;
  const int M = g.batch * HoWo, K = T * g.channels;
  const LayerWs l = layer_ws(g, cout);
  char *ws = static_cast<char *>(workspace);
  float *xn = reinterpret_cast<float *>(ws), *on = reinterpret_cast<float *>(ws + l.off);
  float *mn = reinterpret_cast<float *>(ws + l.msk), *last = reinterpret_cast<float *>(ws + l.last);
  Params p = make_params(dg > 1 ? nullptr : &g, cout, M, K, dg > 1 ? last : xn, on, mn, ws + l.w, bias,
                         out, false);
  p.plane = HoWo;
  // 16-byte stores of four positions need an aligned output
  const bool nchw = reinterpret_cast<uintptr_t>(out) % 16 == 0;
  if (!nchw) p.plane = 0;
  Plan pl = dg > 1 ? make_plan<kRows>(p, true) : make_plan<kGeoMask>(p, true);
  const bool two = p.kparts == 2 || !nchw;  // NHWC output first
  if (two && dg > 1) return hipErrorInvalidValue;  // checked by the caller: out is aligned
  if (two) {
    p.plane = 0;
    p.out = last;
  }
  PrepParams q{};
  int blocks = 0;
  const float *src[3] = {x, off, msk};
  float *dst[3] = {xn, on, mn};
  const int rows[3] = {g.channels, dg * 2 * T, dg * T};
  const int cols[3] = {g.height * g.width, HoWo, HoWo};
  for (int i = 0; i < 3; ++i) {
    PrepJob &j = q.t[i];
    j.src = src[i]; j.dst = dst[i]; j.rows = rows[i]; j.cols = cols[i];
    j.tr = (rows[i] + 63) / 64;
    j.tc = (cols[i] + 63) / 64;
    j.first = blocks;
    const int64_t n = (int64_t)g.batch * j.tr * j.tc;
    if (blocks + n > (1 << 30)) return hipErrorInvalidValue;
    blocks += (int)n;
  }
  q.w = weight;
  q.packed = ws + l.w;
  q.flags = const_cast<uint32_t *>(p.flags);
  q.cout = cout; q.C = g.channels; q.T = T; q.kb_total = p.kb_total;
  q.nbo = p.nb_total;
  q.first_w = blocks;
  blocks += q.nbo * (g.channels / 32);
  q.first_clear = blocks;
  if (p.kparts == 2) {
    q.clear = last;
    q.clear4 = (int64_t)M * cout / 4;
    blocks += (int)std::min<int64_t>((q.clear4 + 1023) / 1024, 2048);
  }
  q.nblocks = blocks;
  hipLaunchKernelGGL(f32_prep_kernel, dim3(blocks), dim3(256), 0, stream, q);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (dg > 1) {
    e = launch_im2col_nhwc(0, g, xn, on, false, mn, last, stream);
    return e != hipSuccess ? e : launch_geo<kRows>(p, pl, false, stream);
  }
  e = launch_geo<kGeoMask>(p, pl, true, stream);
  if (e != hipSuccess || !two) return e;
  return launch_transpose(4, last, out, g.batch, HoWo, cout, stream);
}

hipError_t launch_f32_tconv(const DcnGeom &g, const float *y32, const void *w_split,
                            const float *addend, int out_dtype, void *out, hipStream_t stream) {
  Params p{};
  p.x = y32; p.w = w_split; p.addend = addend; p.out = out; p.out_kind = out_dtype;
  p.Cout = g.channels;
  p.nb_total = (g.channels + 15) / 16;
  p.M = g.batch * g.height * g.width;
  p.taps = g.kernel_h * g.kernel_w;
  p.kb_total = p.taps;
  p.H = g.height; p.W = g.width; p.Ho = g.height_col; p.Wo = g.width_col;
  p.kw = g.kernel_w; p.ph = g.pad_h; p.pw = g.pad_w; p.sh = g.stride_h; p.sw = g.stride_w;
  p.dh = g.dil_h; p.dw = g.dil_w;
  p.x_bytes = (uint32_t)((int64_t)g.batch * g.height_col * g.width_col * kBK * 4);
  p.w_bytes = (uint32_t)((int64_t)p.nb_total * p.kb_total * kBlkBytes);
  p.flags = reinterpret_cast<const uint32_t *>(static_cast<const char *>(w_split) + p.w_bytes);
  const Plan pl = make_plan<kTConv>(p, false);
  return launch_geo<kTConv>(p, pl, false, stream);
}

hipError_t launch_f32_split_offset_weight(const float *w_off, int n3, int C, int T, void *packed,
                                          hipStream_t stream) {
  char *d = static_cast<char *>(packed);
  uint32_t *flags = reinterpret_cast<uint32_t *>(d + (int64_t)((C + 15) / 16) * T * kBlkBytes);
  const int blocks = ((C + 15) / 16) * T;
  hipLaunchKernelGGL(split_offset_weight_kernel, dim3((blocks + 3) / 4), dim3(256), 0, stream, w_off,
                     d, flags, n3, C, T, blocks);
  return hipGetLastError();
}

}  // namespace bevk
