// The strict NF24 packed-weight GEMM on the fp16 matrix cores: out = bias +
// X * decode(W) for calls of more than 32 rows.
//
// fp32 MFMA peaks at 157 TFLOP/s on this part, fp16 MFMA at sixteen times
// that, so each fp32 operand is carried as two fp16 values and each product
// as three fp16 products with fp32 accumulation:
//   x * s = xh + xl,  p / 256 = wh + wl,  acc = sum xh*wh + xh*wl + xl*wh,
//   out = bias + acc * (256 / s) * scale[n]
// with p = (int32)code01 * 256 + q2 the integer payload (the reference's
// decode, scripts/gemm_nf24_i16_avx512.c:26-33, is fp32(p) * scale[n]) and s
// a power of two per row of x.
//   * w: p / 256 lies within +-2^15 and hi = fp16(p / 256) leaves a residual
//     of at most 12 bits, so wh + wl is p / 256 to within one unit of 2^-23
//     for every code the format can hold, and exactly for |p| < 2^22 (the
//     packer's payloads stay below 2^17).  scale[n] is applied once, to the
//     sum.
//   * x: xh + xl holds x * s to within one unit of fp32's last place as long
//     as |x| is above 2^-24 of the row's scale; below that the error is at
//     most 2^-25 / s, i.e. 2^-31 of the largest value the scale was set from.
//   * the dropped xl*wl is below 2^-22 of the product (2^-24 rms).
// Products of fp16 values are exact in fp32, and the matrix core rounds its
// accumulator twice per 16 k and term instead of once per k, so the error
// against 64 bits is below the fp32 MFMA kernel's (N(0, 1) x, K = 1024:
// 3.6e-7 against 5.7e-7 relative).
//
// Row scale.  s brings the largest of the row's first 32 values (all of
// them, when those are zero) to [2^6, 2^7): 2^9 of headroom below fp16's
// largest value.  It depends on that row alone, so a row's result does not
// depend on the rows it shares a tile with.  A larger value further along the
// row makes xh infinite and with it the row's sums; the workgroup sees that
// in its accumulators, sets the scale of those rows from a scan of the whole
// row and runs the K loop once more, with xh held to +-65504: an infinity or
// NaN of x itself is then one in xl, which meets wh alone, and the sums are
// what fp32 products would give, an infinity of the products' sign, or NaN
// where wh is zero or the signs disagree.
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
// fused QKV over 8194 rows 261, 600 x 1024 x 1024 34.)
//
// Measured against the fp32 MFMA tiles: 4096 x 1024 x 3072 197 -> 78 us (330
// TFLOP/s), 12294 x 4096 x 1024 788 -> 284 us (363), 12294 x 1024 x 4096 765 ->
// 299 us, fused QKV over 8194 rows 496 -> 233 us, 600 x 1024 x 1024 47 -> 32
// us.  What bounds it: the fp16 matrix cores at the clock they hold; three
// products at 363 TFLOP/s are 1.09 PFLOP/s, a plain 8192^3 fp16 library product
// on the same card 1.11.  Grids of one round or less are bound by a tile's
// chain of K steps instead (31 us at K = 1024 for the smallest).

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
__device__ __forceinline__ void split2(float a, float b, float hi_a, float hi_b, unsigned& hi, unsigned& lo) {
  const half2v h = __builtin_convertvector(floatx2{hi_a, hi_b}, half2v);
  hi = __builtin_bit_cast(unsigned, h);
  lo = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a - (float)h[0], b - (float)h[1]}, half2v));
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

// Row scale from the bits of the row's largest magnitude: the power of two
// that brings it to [2^6, 2^7), with a normal reciprocal.
__device__ __forceinline__ float row_scale(uint32_t mx_bits) {
  const int field = 260 - (int)(mx_bits >> 23);  // exponent field of 2^(6 - e)
  return mx_bits == 0 ? 1.0f : __uint_as_float((uint32_t)min(max(field, 1), 253) << 23);
}

// Largest of x over eight lanes (a swizzle has no lane addresses to hold, and
// so none that the QKV epilogue would share and keep over the K loop).
__device__ __forceinline__ uint32_t max8(uint32_t x) {
  x = max(x, (uint32_t)__builtin_amdgcn_ds_swizzle((int)x, (1 << 10) | 0x1f));  // lane ^ 1
  x = max(x, (uint32_t)__builtin_amdgcn_ds_swizzle((int)x, (2 << 10) | 0x1f));
  return max(x, (uint32_t)__builtin_amdgcn_ds_swizzle((int)x, (4 << 10) | 0x1f));
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
  __shared__ uint8_t row_flag[C::BM];  // the first pass left the row without finite sums
  __shared__ int second;

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
  // the step at k_next into them.  limit: bound of xh, infinite in the first
  // pass.
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
  auto stage = [&](int part, int buf, float limit, int k_next) {
    if (part < C::kXIter) {
      const int j = part;
      if (!x_unit(j)) return;
      const floatx4 v = xr[j] * rsc[j];
      float m[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) m[e] = __builtin_amdgcn_fmed3f(v[e], -limit, limit);
      unsigned hi[2], lo[2];
      split2(v[0], v[1], m[0], m[1], hi[0], lo[0]);
      split2(v[2], v[3], m[2], m[3], hi[1], lo[1]);
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
        split2(p0, p1, p0, p1, hi[i], lo[i]);
      }
      const int off = w_dst[j] ^ (e * 32);
      store_pairs(&ws[buf][0][off], hi);
      store_pairs(&ws[buf][1][off], lo);
      if (e == 3) load_w(j, k_next);
    }
  };

  // Largest magnitude (as bits) among the values from k0 on of the row of x
  // unit idx, over the row's eight lanes (plain loads: this is rare).
  auto row_max = [&](int idx, int k0) {
    const int row = min(idx / (C::BK / 4), rows - 1);
    const float* src = a.x + (int64_t)(m0 + row) * a.stride_x + 4 * (idx % (C::BK / 4));
    uint32_t mx = 0;
#pragma unroll 1
    for (int k = k0; k < a.K; k += C::BK)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (k + 4 * (idx % (C::BK / 4)) + e < a.K) mx = max(mx, __float_as_uint(src[k + e]) & 0x7fffffffu);
    mx = max8(mx);
    return mx;
  };
  auto set_scale = [&](int idx, uint32_t mx) {
    if (idx < C::kXUnits && idx % (C::BK / 4) == 0) row_sc[idx / (C::BK / 4)] = row_scale(mx);
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
      const uint32_t rest = row_max(idx, C::BK);
      if (mx == 0) mx = rest;
    }
    set_scale(idx, mx);
  }
  // `second` lives in LDS, where the compiler does not know it: one K loop in
  // the code for both passes, the second being the exception.
  if (tid == 0) second = 0;
  __syncthreads();
  // One K step on LDS buffer P: 2 * kMB groups of MFMAs (16 k, one row block),
  // each with the fragment reads of the next group and, in all but the last
  // step, a share of the next step's staging between its MFMAs.
  auto step = [&](auto staged, int P, float limit, int k_next) {
    constexpr int kGroups = 2 * C::kMB;
    half8 ah[2], al[2], bh[2][C::kNB], bl[2][C::kNB];
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
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb) acc[mb][nb] = mfma_f16(al[grp & 1], bh[s][nb], acc[mb][nb]);
      if constexpr (decltype(staged)::value) {
#pragma unroll
        for (int u = grp * kStages / kGroups; u < (grp + 1) * kStages / kGroups; ++u)
          stage(u, P ^ 1, limit, k_next);
        // an MFMA, then what fits beside it (mask 8: MFMA, 2: vector ALU)
#pragma unroll
        for (int i = 0; i < 3 * C::kNB; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, kStageAlu, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (;;) {
    const float limit = __builtin_amdgcn_readfirstlane(second) != 0 ? 65504.0f : INFINITY;
#pragma unroll
    for (int j = 0; j < C::kXIter; ++j) rsc[j] = row_sc[x_unit(j) ? (tid + j * C::kThreads) / (C::BK / 4) : 0];
#pragma unroll
    for (int u = 0; u < kStages; ++u) stage(u, 0, limit, min(1, nk - 1) * C::BK);
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < C::kMB; ++mb)
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0.0f;
    for (int kt = 0; kt + 1 < nk; ++kt) {
      // (the last staged step loads its own tile again, unused)
      step(std::true_type{}, kt & 1, limit, min(kt + 2, nk - 1) * C::BK);
      __syncthreads();
    }
    step(std::false_type{}, (nk - 1) & 1, limit, 0);
    __syncthreads();
    // 0 * acc is NaN for an accumulator that is not finite
    float chk = 0.0f;
#pragma unroll
    for (int mb = 0; mb < C::kMB; ++mb)
#pragma unroll
      for (int nb = 0; nb < C::kNB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) chk = fmaf(acc[mb][nb][r], 0.0f, chk);
    if (!__builtin_amdgcn_readfirstlane(__syncthreads_or(chk != 0.0f))) break;
    if (__builtin_amdgcn_readfirstlane(second) != 0) break;
    // Scales of the rows with such sums from the whole row, and once more.
    for (int i = tid; i < C::BM; i += C::kThreads) row_flag[i] = 0;
    __syncthreads();
    if (tid == 0) second = 1;
#pragma unroll
    for (int mb = 0; mb < C::kMB; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        bool bad = false;
#pragma unroll
        for (int nb = 0; nb < C::kNB; ++nb) bad |= !(fabsf(acc[mb][nb][r]) < INFINITY);
        if (bad) row_flag[wm * C::kTM + mb * 32 + 8 * (r / 4) + 4 * g + r % 4] = 1;
      }
    __syncthreads();
#pragma unroll 1
    for (int idx = tid; idx < C::kXUnits; idx += C::kThreads) {
      const bool flagged = row_flag[idx / (C::BK / 4)] != 0;
      if (__builtin_amdgcn_ballot_w64(flagged) == 0) continue;
      const uint32_t mx = row_max(idx, 0);
      if (flagged) set_scale(idx, mx);
    }
    load_tile(0);
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

  if constexpr (kEpi == kEpiQkv) {
    qkv_epilogue<C>(a, acc, m0 + row_e, c0 + col_e, g_e, l_e);
  } else {
    store_result<C::kMB, C::kNB, kEpi>(a, acc, m0 + row_e, c0 + col_e, g_e, l_e);
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

// Operands the vector loads do not take (unaligned, odd strides or sizes)
// make the element-wise loads the cost, where the fp32 tiles are the faster
// (9000 x 998 x 1030 302 against 348 us, 4096 x 1002 x 3070 304 against 353),
// so from 256 rows and columns on those calls stay with nf24_gemm.hip.  Below,
// where either is a few tiles, the fp16 products serve every call, so that an
// unaligned column range of a small call holds the bits of the whole call.
bool gemm_f16_takes(const GemmParams& p) { return p.M < 256 || p.n_count < 256 || gemm_f16_vector(p); }

int launch_gemm_f16(const GemmParams& p, int epi, const QkvArgs& e, const GemmEpilogueParams& ep, int row0,
                    hipStream_t stream) {
  GemmArgs a{p.x, p.code01, p.q2, p.scale, p.bias, p.out,
             p.M, p.K, p.N, p.n_start, p.n_count, p.stride_x, p.stride_out, e,
             ep.gate, ep.gate_stride, ep.rows_per_batch, row0, 0, 0};
  if (!gemm_f16_vector(p)) return launch_cfg<F16Narrow, false>(a, epi, stream);
  // At most 32 rows past the last multiple of 256 run on the few-row kernels
  // when they would add a round of tiles (their workspace is the only thing
  // that can fail, so they go first).
  const int rem = p.M % 256;
  if (rem != 0 && rem <= 32 &&
      model_time(pick(p.M, p.n_count), p.M, p.n_count) >
          model_time(pick(p.M - rem, p.n_count), p.M - rem, p.n_count)) {
    GemmParams t = p;
    t.x = p.x + (int64_t)(p.M - rem) * p.stride_x;
    if (p.out != nullptr) t.out = p.out + (int64_t)(p.M - rem) * p.stride_out;
    t.M = rem;
    const int st = launch_strict_tail(t, epi, e, ep, row0 + p.M - rem, stream);
    if (st != kOk) return st;
    a.M = p.M - rem;
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
