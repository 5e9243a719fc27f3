// The strict NF24 packed-weight GEMM on the fp16 matrix cores: out = bias +
// X * decode(W) for calls of more than 32 rows.
//
// fp32 MFMA peaks at 157 TFLOP/s on this part, fp16 MFMA at sixteen times
// that, so each fp32 operand is carried as two fp16 values and each product
// as three fp16 products with fp32 accumulation:
//   x * s = xh + 2^-11 xl,  p / 256 = wh + wl,
//   acc = sum xh*wh + xh*wl + xl*(2^-11 wh),
//   out = bias + acc * (256 / s) * scale[n]
// with p = (int32)code01 * 256 + q2 the integer payload (the reference's
// decode, scripts/gemm_nf24_i16_avx512.c:26-33, is fp32(p) * scale[n]) and s
// a power of two per row of x.
//   * w: p / 256 lies within +-2^15 and hi = fp16(p / 256) leaves a residual
//     of at most 12 bits, so wh + wl is p / 256 to within one unit of 2^-23
//     for every code the format can hold, and exactly for |p| < 2^22 (the
//     packer's payloads stay below 2^17).  scale[n] is applied once, to the
//     sum.
//   * x: the pair holds x * s to within one unit of fp32's last place from
//     2^-13 on, and to 2^-36 below: xl is kept 2^11 times larger, so that it
//     does not run out of fp16's range with xh, and meets a copy of wh taken
//     down by as much (exact: wh is a multiple of 2^-8).
//   * the dropped xl*wl is below 2^-22 of the product (2^-24 rms).
// Products of fp16 values are exact in fp32, and the matrix core rounds its
// accumulator twice per 16 k and term instead of once per k, so the error
// against 64 bits is below the fp32 MFMA kernel's (N(0, 1) x, K = 1024:
// 3.6e-7 against 5.7e-7 relative).
//
// Row scale.  s brings the largest of the row's first 32 values (of all of
// them, when those are zero) to [2^3, 2^4): 2^12 of headroom, and as much
// below for values that matter beside weights which are zero for the large
// ones.  The pairs of a row do not serve where |x * s| reaches fp16's infinity
// (the workgroup sees that in its accumulators), or where the largest of four
// neighbouring values is less than 2^-17 and not zero (seen while staging):
// their pairs would hold less than 2^-19 of it.  Such rows are found by a scan,
// get a scale from the whole row (largest value to [2^14, 2^15)) and the
// workgroup runs its K loop once more; rows whose values spread too far for
// that as well, or are not all finite, are then summed as fp32 products.  All
// of this depends on the row alone, so a row's result does not depend on the
// rows it shares a tile with.  What the pairs lose is at most 2^-36 / s of a
// value, 2^-39 of the row's largest, beside values that large in its group of
// four.
//
// A call pays for such rows with the second pass: 4096 x 1024 x 3072 with one
// value of 1e6 80 -> 180 us (fp32 tiles: 196), a feature 3000 times the others
// 213, 1e5 times 262; 600 times, in the first pass, 90 (with a headroom of 2^9
// and without the shift of xl: 197); all of x times 1e10 (a scan, kSmallScale) 141.
//
// Tiling: BM x BN workgroup tile, WM x WN waves, a wave owns MB x NB blocks
// of 32 x 32 (the accumulator layout the epilogues of nf24_gemm_common.h
// take).  K advances 32 per step; x (split on the way in) and the decoded W
// are staged in LDS as fp16 rows of 64 bytes, four 16-byte chunks of 8 k,
// swizzled as in nf24_gemm_bf16.hip: chunk c of row r sits at position
// c ^ ((r >> 2) & 3) and W tile column r in LDS row w_row(r), which keeps
// the 128-bit fragment reads and the staging stores off each other's banks.
// LDS is double-buffered with one barrier per step.  A step's MFMAs run in
// groups of 3 * kNB, and each group carries a share of the next step's staging
// between them: a unit is split or decoded and stored from registers that were
// loaded a step earlier, and the step after that is loaded into them, so no
// wave waits for memory inside a step.  (Staged after the MFMAs instead, from
// loads of the same step: 4096 x 1024 x 3072 84 us, 12294 x 4096 x 1024 350,
// fused QKV over 8194 rows 261, 600 x 1024 x 1024 34.)  The check of each four
// values and the shifted copy of wh cost 2 to 3 % of the larger calls.
//
// Measured against the fp32 MFMA tiles: 4096 x 1024 x 3072 197 -> 79 us (326
// TFLOP/s), 12294 x 4096 x 1024 gated 817 -> 319 us (323), fused QKV over 8194
// rows 496 -> 243 us, 600 x 1024 x 1024 47 -> 27 us.  What bounds it: the fp16
// matrix cores at the clock they hold; three products at 326 TFLOP/s are 0.98
// PFLOP/s, a plain 8192^3 fp16 library product on the same card 1.11.  Grids of
// one round or less are bound by a tile's chain of K steps instead (27 us at
// K = 1024 for the smallest).

#include "nf24_gemm_common.h"

#include <type_traits>

namespace tsplat {
namespace nf24 {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));

template <int BM_, int BN_, int WM_, int WN_, int WK_ = 4>
struct F16Cfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_;
  static constexpr int WK = WK_;  // k rows of a W staging unit (4 columns wide)
  static constexpr int BK = 32;
  static constexpr int kThreads = WM * WN * 64;
  // waves per SIMD the register budget must allow: the workgroup's own, two
  // workgroups per CU for the four-wave shapes
  static constexpr int kMinWaves = WM * WN == 4 ? 2 : WM * WN / 4;
  static constexpr int kTM = BM / WM, kTN = BN / WN;
  static constexpr int kMB = kTM / 32, kNB = kTN / 32;
  static constexpr int kXUnits = BM * BK / 4;           // (row, 4 k)
  static constexpr int kWUnits = (BN / 4) * (BK / WK);  // (4 columns, WK k)
  static constexpr int kXIter = (kXUnits + kThreads - 1) / kThreads;
  static constexpr int kWIter = (kWUnits + kThreads - 1) / kThreads;
  static_assert(WK == 2 || WK == 4, "W units are 2 or 4 k rows deep");
  static_assert(kXUnits % 64 == 0 && kWUnits % 64 == 0, "a partial iteration must cover whole waves");
  static_assert(kTM % 32 == 0 && kTN % 32 == 0, "wave tile must be 32-aligned");
  static_assert(kThreads >= BM, "a thread for every row");
  // unit j of this thread exists (uniform over a wave)
  template <int kUnits, int kIter>
  __device__ static constexpr bool unit(int tid, int j) {
    return kUnits % kThreads == 0 || j + 1 < kIter || tid + j * kThreads < kUnits;
  }
};

__device__ __forceinline__ int chunk_offset(int r, int c) { return r * 32 + ((c ^ ((r >> 2) & 3)) << 3); }
__device__ __forceinline__ int w_row(int r) { return r ^ (((r >> 4) & 1) | ((r >> 5) & 2)); }
__device__ __forceinline__ half8 lds_frag(const _Float16* src) { return *reinterpret_cast<const half8*>(src); }
__device__ __forceinline__ floatx16 mfma_f16(const half8& a, const half8& b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// (hi, lo) fp16 pairs of a and b: hi = fp16(v), lo = fp16(v - hi), the
// difference exact in fp32.
__device__ __forceinline__ void split2(float a, float b, unsigned& hi, unsigned& lo) {
  const half2v h = __builtin_convertvector(floatx2{a, b}, half2v);
  hi = __builtin_bit_cast(unsigned, h);
  lo = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a - (float)h[0], b - (float)h[1]}, half2v));
}
// The same of x[i] * s for a power of two s, given v = x * s, with lo kLoShift
// times larger.  (Each step an instruction: x * s - hi and its shift are mixed
// fp32 / fp16 FMAs.)
constexpr int kLoShift = 2048;
__device__ __forceinline__ void split2_shifted(const floatx4& x, const floatx4& v, float s, int i, unsigned& hi,
                                               unsigned& lo) {
  const half2v h = __builtin_convertvector(floatx2{v[i], v[i + 1]}, half2v);
  hi = __builtin_bit_cast(unsigned, h);
  const half2v l = {(_Float16)fmaf(fmaf(x[i], s, -(float)h[0]), (float)kLoShift, 0.0f),
                    (_Float16)fmaf(fmaf(x[i + 1], s, -(float)h[1]), (float)kLoShift, 0.0f)};
  lo = __builtin_bit_cast(unsigned, l);
}

// p / 256 of column e of a staged unit row (two int16 codes per word, four
// int8 codes per word, these with their sign bits flipped): the bytes side by
// side are (p + 128) * 256 as an int32, of at most 24 significant bits, so
// the conversion and the difference are exact in fp32.
constexpr uint32_t kFlipQ2 = 0x80808080u;
__device__ __forceinline__ float w_payload(const uint32_t (&c)[2], uint32_t q_flipped, int e) {
  const uint32_t sel = ((e & 1) ? 0x0706000cu : 0x0504000cu) | ((uint32_t)e << 8);
  return fmaf((float)(int32_t)__builtin_amdgcn_perm(c[e >> 1], q_flipped, sel), 0x1p-16f, -0.5f);
}

template <int NW>
__device__ __forceinline__ void store_pairs(_Float16* dst, const unsigned (&w)[NW]) {
  if constexpr (NW == 2) *reinterpret_cast<uintx2*>(dst) = uintx2{w[0], w[1]};
  else *reinterpret_cast<unsigned*>(dst) = w[0];
}

// A row's pairs serve where |x * s| stays below kRowTop (fp16's infinity) and
// the largest of each four values (a staging unit) that are not all zero
// reaches kUnitMin.
constexpr float kRowTop = 65520.0f;
constexpr uint32_t kUnitMin = (127u - 17u) << 23;  // bits of 2^-17
// Scales that may take a normal value to zero (a unit of those looks like zeros
// while it is staged): rows under one are looked at again, and their pairs serve
// where that befalls no value.  (A check of x instead of x * s while staging: 600 x
// 1024 x 1024 28.7 against 26.5 us.)
constexpr float kSmallScale = 0x1p-23f;

// The power of two that brings a magnitude (as bits) to [2^kTop, 2^(kTop + 1)),
// with a normal reciprocal.
constexpr int kFirstTop = 3;   // the largest of the row's first 32 values
constexpr int kWholeTop = 14;  // the largest of the row
template <int kTop>
__device__ __forceinline__ float row_scale(uint32_t mx_bits) {
  const int field = 254 + kTop - (int)(mx_bits >> 23);  // exponent field of 2^(kTop - e)
  return mx_bits == 0 ? 1.0f : __uint_as_float((uint32_t)min(max(field, 1), 253) << 23);
}

// Largest of x over eight lanes (lane ^ 1, ^ 2, then the row's halves
// mirrored).
__device__ __forceinline__ uint32_t max8(uint32_t x) {
  x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xb1, 0xf, 0xf, true));
  x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4e, 0xf, 0xf, true));
  return max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xf, 0xf, true));
}
__device__ __forceinline__ float max_abs(const floatx4& v) {
  return fmaxf(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fabsf(v[2])), fabsf(v[3]));
}

// bias + x * decode(W) in fp32 products for a block of 32 rows, the lane's row
// `row` (in range), and the wave's columns from col0: sums in the accumulator
// layout, straight from memory (rare: no tile is shared).
template <class C>
__device__ __forceinline__ void fp32_rows(const GemmArgs& a, int row, int col0, int g, int l32,
                                          floatx16 (&sum)[C::kNB]) {
  // kTurn k a turn for each half (half g on k0 + kTurn * g ..): a turn's loads
  // are in flight together, and no more of them than the registers beside the
  // tile's accumulators hold
  constexpr int kTurn = C::kMinWaves <= 2 ? 8 : 4;
  float sc[C::kNB];
#pragma unroll
  for (int nb = 0; nb < C::kNB; ++nb) {
    const int col = min(col0 + nb * 32 + l32, a.n_count - 1);
    sc[nb] = a.scale[a.n_start + col];
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[nb][r] = a.bias[a.n_start + col];
  }
#pragma unroll 1
  for (int k0 = kTurn * g; k0 - kTurn * g < a.K; k0 += 2 * kTurn) {
    const float* x = a.x + (int64_t)row * a.stride_x;
    float xv[kTurn];
    int c[kTurn][C::kNB], q[kTurn][C::kNB];
#pragma unroll
    for (int i = 0; i < kTurn; ++i) {
      const int k = min(k0 + i, a.K - 1);
      xv[i] = x[k];
      const int64_t w = (int64_t)k * a.N + a.n_start;
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb) {
        const int64_t o = w + min(col0 + nb * 32 + l32, a.n_count - 1);
        c[i][nb] = a.code01[o];
        q[i][nb] = a.q2[o];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kTurn; ++i) {
      const bool in = k0 + i < a.K;
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb)
        sum[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(
            in ? xv[i] : 0.0f, in ? (float)(c[i][nb] * 256 + q[i][nb]) * sc[nb] : 0.0f, sum[nb], 0, 0, 0);
    }
  }
}

// kVec: x rows 16-byte aligned with K % 4 == 0; N, n_start, n_count
// multiples of 4 with code01 8-byte and q2 4-byte aligned, loaded through
// buffer resources (rows past M and columns past n_count carry kBufOob, code
// rows past K lie past the end of the planes: all read 0).
template <class C, bool kVec, int kEpi>
__global__ __launch_bounds__(C::kThreads) __attribute__((amdgpu_waves_per_eu(C::kMinWaves)))
void nf24_gemm_f16_kernel(GemmArgs a) {
  __shared__ __attribute__((aligned(16))) _Float16 xs[2][2][C::BM * C::BK];  // [buffer][hi, lo]
  __shared__ __attribute__((aligned(16))) _Float16 ws[2][2][C::BN * C::BK];
  __shared__ __attribute__((aligned(16))) float row_sc[C::BM];  // s of each row
  __shared__ uint8_t row_flag[C::BM];  // the row's pairs do not serve
  __shared__ int second;               // the scales are those of the second pass

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / C::WN, wn = wave % C::WN;
  const int g = lane >> 5;
  const int l32 = lane & 31;

  const int tiles_n = (a.n_count + C::BN - 1) / C::BN;
  const int tile = xcd_tile_index(blockIdx.x, gridDim.x);
  const int m0 = (tile / tiles_n) * C::BM;
  const int c0 = (tile % tiles_n) * C::BN;
  const int rows = min(C::BM, a.M - m0);

  auto x_unit = [&](int j) { return C::template unit<C::kXUnits, C::kXIter>(tid, j); };
  auto w_unit = [&](int j) { return C::template unit<C::kWUnits, C::kWIter>(tid, j); };

  // W units: columns w_col .. w_col+3 of the tile, k rows w_k .. w_k+WK-1.
  int w_col[C::kWIter], w_k[C::kWIter];
  bool w_ok[C::kWIter][4];
#pragma unroll
  for (int j = 0; j < C::kWIter; ++j) {
    const int u = tid + j * C::kThreads;
    w_col[j] = 4 * (u % (C::BN / 4));
    w_k[j] = C::WK * (u / (C::BN / 4));
#pragma unroll
    for (int e = 0; e < 4; ++e) w_ok[j][e] = w_unit(j) && c0 + w_col[j] + e < a.n_count;
  }

  floatx4 xr[C::kXIter];
  uint32_t cr[C::kWIter][C::WK][2];    // k row i: int16 codes of columns 0,1 | 2,3
  uint32_t qr[C::kWIter][C::WK];       // k row i: int8 codes of columns 0..3

  // code element offset past both planes: itself and doubled (mod 2^32) it is
  // at least kBufOob, whatever in-range step is added
  constexpr uint32_t kWOob = 0xc0000000u;
  __amdgpu_buffer_rsrc_t rx, rc, rq;
  uint32_t x_off[C::kXIter], w_off[C::kWIter];
  if constexpr (kVec) {
    rx = buffer_rsrc(a.x + (int64_t)m0 * a.stride_x, ((int64_t)(rows - 1) * a.stride_x + a.K) * 4);
#pragma unroll
    for (int j = 0; j < C::kXIter; ++j) {
      const int idx = tid + j * C::kThreads;
      const int row = idx / (C::BK / 4);
      x_off[j] = row < rows ? (uint32_t)(row * a.stride_x + 4 * (idx % (C::BK / 4))) * 4u : kBufOob;
    }
    rc = buffer_rsrc(a.code01, (int64_t)a.K * a.N * 2);
    rq = buffer_rsrc(a.q2, (int64_t)a.K * a.N);
#pragma unroll
    for (int j = 0; j < C::kWIter; ++j) {
      const uint32_t e = (uint32_t)(w_k[j] * a.N + a.n_start + c0 + w_col[j]);
      w_off[j] = w_ok[j][0] ? e : kWOob;
    }
  }

  // x unit j (4 consecutive k of its row) of the step at k0.
  auto load_x = [&](int j, int k0) {
    const int idx = tid + j * C::kThreads;
    const int kc = idx % (C::BK / 4);
    floatx4 v = {0, 0, 0, 0};
    if constexpr (kVec) {
      // K % 4 == 0: a unit lies wholly inside or past the row's K floats
      const uint32_t off = (k0 + 4 * kc < a.K) ? x_off[j] + 4u * (uint32_t)k0 : kBufOob;
      const auto u = __builtin_amdgcn_raw_buffer_load_b128(rx, (int)off, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = __uint_as_float(u[e]);
    } else {
      const int row = idx / (C::BK / 4);
      const float* src = a.x + (int64_t)(m0 + row) * a.stride_x + k0 + 4 * kc;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (row < rows && k0 + 4 * kc + e < a.K) ? src[e] : 0.0f;
    }
    return v;
  };
  // W unit j (WK code rows of 4 columns) of the step at k0.
  auto load_w = [&](int j, int k0) {
#pragma unroll
    for (int i = 0; i < C::WK; ++i) {
      if constexpr (kVec) {
        const uint32_t e = w_off[j] + (uint32_t)(k0 + i) * (uint32_t)a.N;
        const auto c = __builtin_amdgcn_raw_buffer_load_b64(rc, (int)(2u * e), 0, 0);
        cr[j][i][0] = c[0];
        cr[j][i][1] = c[1];
        qr[j][i] = __builtin_amdgcn_raw_buffer_load_b32(rq, (int)e, 0, 0);
      } else {
        const int gk = k0 + w_k[j] + i;
        const int64_t off = (int64_t)gk * a.N + a.n_start + c0 + w_col[j];
        uint32_t c[4], q = 0u;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool ok = w_ok[j][e] && gk < a.K;
          c[e] = ok ? (uint16_t)a.code01[off + e] : 0u;
          q |= (ok ? (uint32_t)(uint8_t)a.q2[off + e] : 0u) << (8 * e);
        }
        cr[j][i][0] = c[0] | (c[1] << 16);
        cr[j][i][1] = c[2] | (c[3] << 16);
        qr[j][i] = q;
      }
    }
  };
  auto load_tile = [&](int k0) {
#pragma unroll
    for (int j = 0; j < C::kXIter; ++j)
      if (x_unit(j)) xr[j] = load_x(j, k0);
#pragma unroll
    for (int j = 0; j < C::kWIter; ++j)
      if (w_unit(j)) load_w(j, k0);
  };

  // A step's staging in kStages parts: x unit j, then column e of W unit j.
  // A part places its values in LDS buffer buf and, its registers free, loads
  // the step at k_next into them.
  // LDS positions: x units of a thread are a multiple of 16 rows apart, and
  // the four columns of a W unit (w_col a multiple of 4) are rows whose two
  // low bits alone differ.
  static_assert(C::kThreads / (C::BK / 4) % 16 == 0, "x units keep the swizzle");
  // 4-k unit kc of a row: chunk kc/2, half kc%2
  const int x_dst = chunk_offset(tid / (C::BK / 4), (tid % (C::BK / 4)) >> 1) + 4 * (tid & 1);
  int w_dst[C::kWIter];
#pragma unroll
  for (int j = 0; j < C::kWIter; ++j) w_dst[j] = chunk_offset(w_row(w_col[j]), w_k[j] >> 3) + (w_k[j] & 7);
  constexpr int kStages = C::kXIter + 4 * C::kWIter;
  float rsc[C::kXIter];  // scale of x unit j's row
  // bits of the smallest of its units' maxima so far, less one (so that a
  // maximum of zero is the largest of all)
  uint32_t low = 0xffffffffu;
  auto stage = [&](int part, int buf, int k_next) {
    if (part < C::kXIter) {
      const int j = part;
      if (!x_unit(j)) return;
      const floatx4 v = xr[j] * rsc[j];
      low = min(low, __float_as_uint(max_abs(v)) - 1u);
      unsigned hi[2], lo[2];
      split2_shifted(xr[j], v, rsc[j], 0, hi[0], lo[0]);
      split2_shifted(xr[j], v, rsc[j], 2, hi[1], lo[1]);
      const int off = x_dst + j * (C::kThreads / (C::BK / 4)) * 32;
      store_pairs(&xs[buf][0][off], hi);
      store_pairs(&xs[buf][1][off], lo);
      xr[j] = load_x(j, k_next);
    } else {
      const int j = (part - C::kXIter) / 4, e = (part - C::kXIter) % 4;
      if (!w_unit(j)) return;
      unsigned hi[C::WK / 2], lo[C::WK / 2];
#pragma unroll
      for (int i = 0; i < C::WK / 2; ++i) {
        const float p0 = w_payload(cr[j][2 * i], qr[j][2 * i] ^ kFlipQ2, e);
        const float p1 = w_payload(cr[j][2 * i + 1], qr[j][2 * i + 1] ^ kFlipQ2, e);
        split2(p0, p1, hi[i], lo[i]);
      }
      const int off = w_dst[j] ^ (e * 32);
      store_pairs(&ws[buf][0][off], hi);
      store_pairs(&ws[buf][1][off], lo);
      if (e == 3) load_w(j, k_next);
    }
  };

  // Largest magnitude (as bits) of the row of x unit idx, over the row's eight
  // lanes (plain loads: this is rare).
  auto row_max = [&](int idx) {
    const int row = min(idx / (C::BK / 4), rows - 1);
    const float* src = a.x + (int64_t)(m0 + row) * a.stride_x;
    uint32_t mx = 0;
#pragma unroll 1
    for (int k = 4 * (idx % (C::BK / 4)); k < a.K; k += 4 * C::BK)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        mx = max(mx, __float_as_uint(src[min(k + i / 4 * C::BK + i % 4, a.K - 1)]) & 0x7fffffffu);
    return max8(mx);
  };
  auto set_scale = [&](int idx, float scale) {
    if (idx < C::kXUnits && idx % (C::BK / 4) == 0) row_sc[idx / (C::BK / 4)] = scale;
  };
  // row_flag: the rows whose pairs under the present scales do not serve.
  auto find_rows = [&](int first) {
#pragma unroll 1
    for (int idx = first; idx < C::kXUnits; idx += C::kThreads) {
      const int row = idx / (C::BK / 4), kc = idx % (C::BK / 4);
      const float* src = a.x + (int64_t)(m0 + min(row, rows - 1)) * a.stride_x;
      const float s = row_sc[row];
      bool bad = false;
#pragma unroll 1
      for (int k = 4 * kc; k < a.K; k += 4 * C::BK) {
        float v[4][4];  // four units' loads in flight
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[u][e] = src[min(k + u * C::BK + e, a.K - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          uint32_t mx = 0;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float w = k + u * C::BK + e < a.K ? fabsf(v[u][e] * s) : 0.0f;
            bad |= !(w < kRowTop) || (s < kSmallScale && w == 0.0f && v[u][e] != 0.0f);
            mx = max(mx, __float_as_uint(w));
          }
          bad |= mx - 1u < kUnitMin - 1u;
        }
      }
      const uint32_t any = max8(bad ? 1u : 0u);
      if (kc == 0) row_flag[row] = row < rows && any != 0;
    }
  };

  // vector ALU instructions between two MFMAs of a step: the staging's share
  constexpr int kStageAlu = 5;
  floatx16 acc[C::kMB][C::kNB];
  const int nk = (a.K + C::BK - 1) / C::BK;
  // Fragment positions: a step of 32 rows or columns moves neither the
  // swizzle nor (kTN = 32 * kNB, kNB <= 2) what w_row adds, 16 k flip bit 1 of
  // the chunk.
  static_assert(C::kNB <= 2, "w_row over the wave's columns");
  const int a_src = chunk_offset(wm * C::kTM + l32, g);
  const int b_src = chunk_offset(w_row(wn * C::kTN + l32), g);

  load_tile(0);
#pragma unroll
  for (int j = 0; j < C::kXIter; ++j) {
    uint32_t mx = 0;
    if (x_unit(j)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = max(mx, __float_as_uint(xr[j][e]) & 0x7fffffffu);
    }
    mx = max8(mx);
    // rows whose first 32 values are zero: the rest of the row decides
    const int idx = tid + j * C::kThreads;
    const bool zero = mx == 0 && x_unit(j) && idx / (C::BK / 4) < rows;
    if (__builtin_amdgcn_ballot_w64(zero) != 0) {
      const uint32_t rest = row_max(idx);
      if (mx == 0) mx = rest;
    }
    set_scale(idx, row_scale<kFirstTop>(mx));
  }
  // `second` lives in LDS, where the compiler does not know it: one K loop in
  // the code for both passes, the second being the exception.
  if (tid == 0) second = 0;
  __syncthreads();
  // One K step on LDS buffer P: 2 * kMB groups of MFMAs (16 k, one row block),
  // each with the fragment reads of the next group and, in all but the last
  // step, a share of the next step's staging between its MFMAs.
  auto step = [&](auto staged, int P, int k_next) {
    constexpr int kGroups = 2 * C::kMB;
    half8 ah[2], al[2], bh[2][C::kNB], bl[2][C::kNB], bs[C::kNB];
    auto read_a = [&](int grp) {
      const int off = (a_src ^ (grp / C::kMB * 16)) + grp % C::kMB * 32 * 32;
      ah[grp & 1] = lds_frag(&xs[P][0][off]);
      al[grp & 1] = lds_frag(&xs[P][1][off]);
    };
    auto read_b = [&](int s) {
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb) {
        const int off = (b_src ^ (s * 16)) + nb * 32 * 32;
        bh[s][nb] = lds_frag(&ws[P][0][off]);
        bl[s][nb] = lds_frag(&ws[P][1][off]);
      }
    };
    // two waves a SIMD have the registers to read a group ahead; the shapes
    // of three and more have another wave to run while they wait
    constexpr bool kAhead = C::kMinWaves <= 2;
    if (kAhead) {
      read_b(0);
      read_a(0);
    }
#pragma unroll
    for (int grp = 0; grp < kGroups; ++grp) {
      const int s = grp / C::kMB, mb = grp % C::kMB;
      if (!kAhead) {
        if (mb == 0) read_b(s);
        read_a(grp);
      } else if (grp + 1 < kGroups) {
        if (mb + 1 == C::kMB) read_b(s + 1);
        read_a(grp + 1);
      }
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb) acc[mb][nb] = mfma_f16(ah[grp & 1], bh[s][nb], acc[mb][nb]);
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb) acc[mb][nb] = mfma_f16(ah[grp & 1], bl[s][nb], acc[mb][nb]);
      if (mb == 0) {
#pragma unroll
        for (int nb = 0; nb < C::kNB; ++nb) bs[nb] = bh[s][nb] * (_Float16)(1.0f / kLoShift);
      }
      auto share = [&](int first, int end, int mfmas) {
        if constexpr (decltype(staged)::value) {
#pragma unroll
          for (int u = first; u < end; ++u) stage(u, P ^ 1, k_next);
          // an MFMA, then what fits beside it (mask 8: MFMA, 2: vector ALU)
#pragma unroll
          for (int i = 0; i < mfmas; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, kStageAlu, 0);
          }
        }
      };
      const int first = grp * kStages / kGroups, end = (grp + 1) * kStages / kGroups;
      if (mb == 0) {
        // (apart, or the products that wait for bs are chained behind it)
        share(first, end, 2 * C::kNB);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb) acc[mb][nb] = mfma_f16(al[grp & 1], bs[nb], acc[mb][nb]);
      if (mb != 0) share(first, end, 3 * C::kNB);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  bool rest = false;  // some rows' pairs serve under neither scale
  for (;;) {
    int tid_x = tid;  // (addresses that are not kept over the K loop)
    asm volatile("" : "+v"(tid_x));
#pragma unroll
    for (int j = 0; j < C::kXIter; ++j) rsc[j] = row_sc[x_unit(j) ? (tid_x + j * C::kThreads) / (C::BK / 4) : 0];
#pragma unroll
    for (int u = 0; u < kStages; ++u) stage(u, 0, min(1, nk - 1) * C::BK);
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < C::kMB; ++mb)
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0.0f;
    for (int kt = 0; kt + 1 < nk; ++kt) {
      // (the last staged step loads its own tile again, unused)
      step(std::true_type{}, kt & 1, min(kt + 2, nk - 1) * C::BK);
      __syncthreads();
    }
    step(std::false_type{}, (nk - 1) & 1, 0);
    // 0 * acc is NaN for an accumulator that is not finite
    float chk = 0.0f;
#pragma unroll
    for (int mb = 0; mb < C::kMB; ++mb)
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) chk = fmaf(acc[mb][nb][r], 0.0f, chk);
    asm volatile("" : "+v"(tid_x));
    const bool bad = chk != 0.0f || low < kUnitMin - 1u || row_sc[min(tid_x, C::BM - 1)] < kSmallScale;
    if (!__builtin_amdgcn_readfirstlane(__syncthreads_or(bad))) break;
    rest = __builtin_amdgcn_readfirstlane(second) != 0;
    find_rows(tid_x);
    __syncthreads();
    const bool any = __builtin_amdgcn_readfirstlane(__syncthreads_or(row_flag[min(tid_x, C::BM - 1)])) != 0;
    rest = rest && any;
    if (rest || !any) break;
    // Those rows' scales from the whole row, and once more (the other rows' sums
    // come out as they were).
    if (tid == 0) second = 1;
#pragma unroll 1
    for (int idx = tid_x; idx < C::kXUnits; idx += C::kThreads) {
      const bool flagged = row_flag[idx / (C::BK / 4)] != 0;
      if (__builtin_amdgcn_ballot_w64(flagged) == 0) continue;
      const uint32_t mx = row_max(idx);
      if (flagged) set_scale(idx, row_scale<kWholeTop>(mx));
    }
    low = 0xffffffffu;
    int k_first = 0;  // (a step of its own, for the addresses)
    asm volatile("" : "+s"(k_first));
    load_tile(k_first);
  }

  // The wave's coordinates again, from a copy of the thread index that the
  // compiler cannot relate to the one above, so that the epilogue's addresses
  // are not held (or spilled) over the K loop.
  int tid_e = tid;
  asm volatile("" : "+v"(tid_e));
  const int wave_e = __builtin_amdgcn_readfirstlane(tid_e >> 6);
  const int row_e = (wave_e / C::WN) * C::kTM, col_e = (wave_e % C::WN) * C::kTN;
  const int g_e = (tid_e >> 5) & 1, l_e = tid_e & 31;

  // out before the epilogue, a row block at a time (all the row scales at once
  // would spill): bias + acc * (256 / s) * scale, the powers of two applied to
  // acc together, before scale's fraction in [1, 2): nothing on the way to the
  // result is larger than it, or rounded before it.
  float bv[C::kNB], frac[C::kNB];
  int expo[C::kNB];
#pragma unroll
  for (int nb = 0; nb < C::kNB; ++nb) {
    const int col = c0 + col_e + nb * 32 + l_e;
    const float sc = col < a.n_count ? a.scale[a.n_start + col] : 0.0f;
    bv[nb] = col < a.n_count ? a.bias[a.n_start + col] : 0.0f;
    frac[nb] = 2.0f * __builtin_amdgcn_frexp_mantf(sc);
    expo[nb] = __builtin_amdgcn_frexp_expf(sc) + (8 - 1 + 127);
  }
#pragma unroll
  for (int mb = 0; mb < C::kMB; ++mb) {
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const floatx4 rs = *reinterpret_cast<const floatx4*>(&row_sc[row_e + mb * 32 + 8 * r4 + 4 * g_e]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int nb = 0; nb < C::kNB; ++nb) {
          const float t = __builtin_amdgcn_ldexpf(acc[mb][nb][4 * r4 + e], expo[nb] - (int)(__float_as_uint(rs[e]) >> 23));
          acc[mb][nb][4 * r4 + e] = fmaf(t, frac[nb], bv[nb]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  if (rest) {
    // The sums of the rows left over, as fp32 products.
#pragma unroll 1
    for (int mb = 0; mb < C::kMB; ++mb) {
      const int row_b = row_e + mb * 32;
      if (__builtin_amdgcn_ballot_w64(row_flag[row_b + l_e] != 0) == 0) continue;
      floatx16 sum[C::kNB];
      fp32_rows<C>(a, m0 + min(row_b + l_e, rows - 1), c0 + col_e, g_e, l_e, sum);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const bool take = row_flag[row_b + 8 * (r / 4) + 4 * g_e + r % 4] != 0;
#pragma unroll
        for (int m = 0; m < C::kMB; ++m)
#pragma unroll
          for (int nb = 0; nb < C::kNB; ++nb)
            acc[m][nb][r] = take && m == mb ? sum[nb][r] : acc[m][nb][r];
      }
    }
  }

  asm volatile("" : "+v"(tid_e));
  const int wave_s = __builtin_amdgcn_readfirstlane(tid_e >> 6);
  const int row_s = m0 + (wave_s / C::WN) * C::kTM, col_s = c0 + (wave_s % C::WN) * C::kTN;
  if constexpr (kEpi == kEpiQkv) {
    qkv_epilogue<C>(a, acc, row_s, col_s, (tid_e >> 5) & 1, tid_e & 31);
  } else {
    store_result<C::kMB, C::kNB, kEpi>(a, acc, row_s, col_s, (tid_e >> 5) & 1, tid_e & 31);
  }
}

using F16Large = F16Cfg<256, 256, 2, 4>;     // 8 waves of 128 x 64
using F16Wide = F16Cfg<256, 192, 4, 3, 2>;   // 12 waves of 64 x 64
using F16Tall = F16Cfg<192, 256, 3, 4, 2>;   // 12 waves of 64 x 64
using F16Half = F16Cfg<256, 128, 8, 2, 2>;   // 16 waves of 32 x 64
using F16Narrow = F16Cfg<128, 64, 4, 1, 2>;  // 4 waves of 32 x 64, two workgroups per CU

template <class C, bool kVec>
int launch_cfg(const GemmArgs& a, int epi, hipStream_t stream) {
  const int64_t tiles = (int64_t)((a.M + C::BM - 1) / C::BM) * ((a.n_count + C::BN - 1) / C::BN);
  if (tiles <= 0 || tiles > 0x7fffffff) return kErrDims;
  const dim3 grid((unsigned)tiles), block(C::kThreads);
  switch (epi) {
    case kEpiStore:
      hipLaunchKernelGGL((nf24_gemm_f16_kernel<C, kVec, kEpiStore>), grid, block, 0, stream, a);
      break;
    case kEpiQkv:
      if constexpr (C::kTN == 64 && C::kNB == 2)
        hipLaunchKernelGGL((nf24_gemm_f16_kernel<C, kVec, kEpiQkv>), grid, block, 0, stream, a);
      else
        return kErrDims;
      break;
    case kEpilogueGelu:
      hipLaunchKernelGGL((nf24_gemm_f16_kernel<C, kVec, kEpilogueGelu>), grid, block, 0, stream, a);
      break;
    case kEpilogueGated:
      hipLaunchKernelGGL((nf24_gemm_f16_kernel<C, kVec, kEpilogueGated>), grid, block, 0, stream, a);
      break;
    case kEpilogueAdd:
      hipLaunchKernelGGL((nf24_gemm_f16_kernel<C, kVec, kEpilogueAdd>), grid, block, 0, stream, a);
      break;
    default:
      return kErrDims;
  }
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

// The tile shapes the launch model chooses from: a round of the chip
// (CUs x wgs_per_cu workgroups) costs `round` us at K = 1024, measured on
// grids of one to twelve full rounds; the model is rounds x cost, a partial
// round as much as a whole one (a nearly empty one takes 70, 56, 56, 42 and 31
// us: its K steps follow one another at any load).
struct F16Choice {
  int bm, bn, wgs_per_cu, round;
};
constexpr F16Choice kChoices[] = {
    {256, 256, 1, 94}, {256, 192, 1, 82}, {192, 256, 1, 75}, {256, 128, 1, 57}, {128, 64, 2, 38}};
constexpr int kNumChoices = sizeof(kChoices) / sizeof(kChoices[0]);

int64_t model_time(int i, int M, int n_count) {
  const F16Choice& c = kChoices[i];
  const int64_t tiles = (int64_t)((M + c.bm - 1) / c.bm) * ((n_count + c.bn - 1) / c.bn);
  const int64_t slots = (int64_t)compute_units() * c.wgs_per_cu;
  return (tiles + slots - 1) / slots * c.round;
}

// Index into kChoices with the smallest modelled time (a tie keeps the
// earlier entry).
int pick(int M, int n_count) {
  int best = 0;
  for (int i = 1; i < kNumChoices; ++i)
    if (model_time(i, M, n_count) < model_time(best, M, n_count)) best = i;
  return best;
}

}  // namespace

bool gemm_f16_vector(const GemmParams& p) {
  return (reinterpret_cast<uintptr_t>(p.x) % 16 == 0) && (p.stride_x % 4 == 0) && (p.K % 4 == 0) &&
         (p.N % 4 == 0) && (p.n_start % 4 == 0) && (p.n_count % 4 == 0) &&
         (reinterpret_cast<uintptr_t>(p.code01) % 8 == 0) && (reinterpret_cast<uintptr_t>(p.q2) % 4 == 0) &&
         vec_buffers_fit(p, F16Large::BM, F16Large::BK);
}

// Calls that the vector loads do not take read element by element, and that is
// then the cost.  The fp32 tiles serve those
//   * whose weight they load in pairs of columns (N % 4 == 2): 33 to 255 rows of
//     1024 x 1002 47 us against 58 to 64 here, 12294 x 1024 x 254 85 against
//     115, 4096 x 4096 x 254 185 against 270;
//   * of 256 rows and columns or more, where both read element by element (9000
//     x 1030 x 998 302 against 348).
// The fp16 products serve the other small ones (33 to 255 rows of 1030 x 1024
// 84 to 94 us there, 58 here; 4096 x 1024 x 5 91 and 60): the weight decides
// first, so that an unaligned column range of a small call holds the bits of
// the whole call.
bool gemm_f16_takes(const GemmParams& p) {
  if (gemm_f16_vector(p)) return true;
  GemmParams whole = p;
  whole.n_start = 0;
  whole.n_count = p.N;
  if (!gemm_f16_vector(whole) && pair_loads_fit(whole, F16Large::BM, F16Large::BK)) return false;
  return p.M < 256 || p.n_count < 256;
}

int launch_gemm_f16(const GemmParams& p, int epi, const QkvArgs& e, const GemmEpilogueParams& ep, int row0,
                    hipStream_t stream) {
  GemmArgs a{p.x, p.code01, p.q2, p.scale, p.bias, p.out,
             p.M, p.K, p.N, p.n_start, p.n_count, p.stride_x, p.stride_out, e,
             ep.gate, ep.gate_stride, ep.rows_per_batch, row0, 0, 0};
  if (!gemm_f16_vector(p)) return launch_cfg<F16Narrow, false>(a, epi, stream);
  // At most 32 rows past the last multiple of 256 run on the few-row kernels
  // when they would add a round of tiles (their workspace is the only thing
  // that can fail, so they go first).  Without the workspace (a capture that
  // would need it to grow) they stay in the tiles, except where the fp32 tiles
  // split them off too: those calls fail, as they do in every mode.
  const int rem = p.M % 256;
  if (rem != 0 && rem <= 32 &&
      model_time(pick(p.M, p.n_count), p.M, p.n_count) >
          model_time(pick(p.M - rem, p.n_count), p.M - rem, p.n_count)) {
    GemmParams t = p;
    t.x = p.x + (int64_t)(p.M - rem) * p.stride_x;
    if (p.out != nullptr) t.out = p.out + (int64_t)(p.M - rem) * p.stride_out;
    t.M = rem;
    const int st = launch_strict_tail(t, epi, e, ep, row0 + p.M - rem, stream);
    if (st == kOk) a.M = p.M - rem;
    else if (st != kErrWorkspace || fp32_tail_rows(p.M, p.n_count) != 0) return st;
  }
  switch (pick(a.M, p.n_count)) {
    case 0: return launch_cfg<F16Large, true>(a, epi, stream);
    case 1: return launch_cfg<F16Wide, true>(a, epi, stream);
    case 2: return launch_cfg<F16Tall, true>(a, epi, stream);
    case 3: return launch_cfg<F16Half, true>(a, epi, stream);
    default: return launch_cfg<F16Narrow, true>(a, epi, stream);
  }
}

}  // namespace nf24
}  // namespace tsplat
