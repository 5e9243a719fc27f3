// The strict exact SDPA on the fp16 matrix cores.
//
// Same operation and softmax as sdpa.hip -- out[q] = sum_j softmax_j(q.k_j
// * 0.125 + bias[j]) v_j over all keys, online (max, sum) merge, no Lq x Lk
// matrix.  fp32 MFMA peaks at 157 TFLOP/s, fp16 MFMA at sixteen times that,
// so every operand of the two products is carried as two fp16 values under a
// power-of-two scale and each product as three fp16 products with fp32
// accumulation:
//   q sq = qh + ql,  k sk = kh + kl,  S = (qh.kh + ql.kh + qh.kl) / (sq sk)
//   2^11 p = ph + pl, v sv = vh + vl, O = (ph vh + pl vh + ph vl) / (2^11 sv)
// A pair holds its value to one unit of fp32's last place down to 2^-2, and to
// 2^-25 below that; the dropped low x low product is below 2^-22 of the product
// (2^-24 rms).  sq is the query row's own, sk and sv are the key tile's: they
// bring its largest magnitude to [2^14, 2^15) (v's to [2^11, 2^15)).  Products of
// fp16 values are exact in fp32 and the matrix core rounds its accumulator twice
// per 16 products, so the error against 64 bits is below the fp32 MFMA kernel's
// (16 heads, L = 16384: 1.5e-6 against 2.3e-6 relative; L = 8194 with log(8194)
// on one key 2.2e-7, as there).
//
// What the pairs do not serve.  Values far below their tile's largest lose
// precision, and that matters where the large ones do not count: keys that a
// bias removes, dims that q leaves out.  So every four neighbouring values of v
// that are not all zero have to reach 2^-5 of the scale (2^-16 of the tile's
// largest value at worst; they are then held to 2^-20), and where values of q or
// k spread over more than 2^18 |q| |k| has to stay below 2^14, so that what a
// score loses (64 dims of 2^-39 |q| |k|) stays below 2^-20.  A workgroup that
// meets a tile which fails this, an infinity in q or k, or tiles of v more than
// 2^64 apart, runs its queries and keys as fp32 products (sdpa_fp32.h) instead:
// what another key or dim holds costs a result nothing that it would not cost
// there.  (8194 keys with a bias, 50 of them masked and holding 1e30: 2166 us; the
// fp32 tiles 2150.)
//
// Softmax in log2 units with a lazy reference: p = exp2(x - m + 4) for a
// reference m that follows the running maximum only when that has moved by
// more than 4, so p stays below 2^8 and most 32-key blocks rescale nothing;
// the sums and the outputs share the factor, which 2^7 more bring up to the
// pairs' range.  Without a bias the exponent is one FMA of the accumulator; with
// one as well, and a block that moves the reference computes its scores again.
//
// Mapping, fragments and LDS image as in sdpa_bf16.hip: a wave owns 32
// queries and computes S^T = K Q^T with v_mfma_f32_32x32x16_f16, each lane
// holding 16 keys of one query per 32-key block; P^T is the B operand of O^T
// += V^T P^T straight from the accumulator, V^T rows stored with bits 2 and 3
// of the key index swapped; rows of 72 fp16 in LDS.
//
// Wide launches first stage every 64-key tile of every (b, h) once
// (sdpa_f16_presplit_kernel) and the main kernel copies the planes into LDS;
// otherwise each workgroup splits the tiles it reads.  Both place the same
// values, so they give the same bits.
//
// Measured (16 heads) against the fp32 MFMA kernel: L = 16384 7.89 -> 2.79 ms
// (394 TFLOP/s), 8194 with a key bias 2.15 -> 0.82 ms, 4096 x 2048 282 -> 157 us,
// 2 x 4096 x 4096 1022 -> 424 us, 577 52 -> 37 us, 2 x 1025 x 513 87 -> 50 us (a
// scale per head instead, from a look at all of its keys: 2.80 ms, 0.82 ms, 159,
// 429, 42 and 56 us).  What bounds it: the fp16 matrix
// cores at the clock they hold, 1.2 PFLOP/s at L = 16384 where a plain 8192^3
// fp16 library product reaches 1.11 (waves of 64 queries, which read half the
// LDS fragments per product, 3.05 against 2.97 ms; wave priorities no change).
// The 128-query tiles are split along the keys where CUs would idle
// (plan_key_ranges): 300 x 9000 654 -> 88 us.

#include "sdpa_fp32.h"

namespace tsplat {
namespace sdpa {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx16 mfma_f16(const half8& a, const half8& b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

constexpr int kWaitVmcnt0 = 0x0f70;  // s_waitcnt operand: vector-memory count 0 only
// log2 of p at the reference, and how far the maximum may pass it: large
// enough for the fp16 pairs of p and for few moves, small enough that the
// exponent's last place (it grows with |x - m + 4|) stays finer than the
// score's own.
constexpr float kPBase = 4.0f;
constexpr float kSlack = 4.0f;
// The reference before any key: no key's own, which ends the search for it (a
// bias may make a finite score of any size).
constexpr float kStart = -INFINITY;
// Largest |q| |k| (of a wave's queries, of a key tile) whose scores the pairs
// serve: any, short of the scales' own range, where neither operand's values
// spread over more than its pairs hold; elsewhere as long as 64 dims of 2^-39
// |q| |k| stay below 2^-20 of a log2 unit.
constexpr float kPairTop = 0x1p96f;
constexpr int kEvRange = 1024;  // beyond any ev
// How far apart the tiles' scales of v may be: outputs below 2^44 in the unit
// of one tile stay in range in that of another.
constexpr int kEvSpread = 64;
constexpr float kWideTop = 0x1p14f;
// |q| |k| from which 64 dims may score 2^20 log2 units (2^19.5 here).
constexpr float kFarScores = 0x1p16f;
// p is taken up by 2^kPShift before it is split: below 2^15, and held to 2^-25,
// 2^-36 of a weight at the reference (many small weights add up: 16384 of them,
// each 2^-30 of one key's, were lost to the pairs, not to their sum).  After the
// exponential, so that its argument stays small.
constexpr int kPShift = 7;

// Position of tile key k in a V^T row: bits 2 and 3 swapped.
__device__ __forceinline__ int vt_pos(int k) { return (k & ~12) | ((k & 4) << 1) | ((k & 8) >> 1); }

// (hi, lo) of a and b: hi = fp16(v), lo = fp16(v - hi), the difference exact
// in fp32.
__device__ __forceinline__ void split2(float a, float b, unsigned& hi, unsigned& lo) {
  const half2v h = __builtin_convertvector(floatx2{a, b}, half2v);
  hi = __builtin_bit_cast(unsigned, h);
  lo = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a - (float)h[0], b - (float)h[1]}, half2v));
}

__device__ __forceinline__ void split4(const floatx4& v, half4v& hi, half4v& lo) {
  unsigned h[2], l[2];
  split2(v[0], v[1], h[0], l[0]);
  split2(v[2], v[3], h[1], l[1]);
  hi = __builtin_bit_cast(half4v, uintx2{h[0], h[1]});
  lo = __builtin_bit_cast(half4v, uintx2{l[0], l[1]});
}

// Elements 8c..8c+7 of an accumulator block, split.
__device__ __forceinline__ void split8(const floatx16& s, int c, half8& hi, half8& lo) {
  unsigned h[4], l[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) split2(s[8 * c + 2 * e], s[8 * c + 2 * e + 1], h[e], l[e]);
  hi = __builtin_bit_cast(half8, uintx4{h[0], h[1], h[2], h[3]});
  lo = __builtin_bit_cast(half8, uintx4{l[0], l[1], l[2], l[3]});
}

// Exponent of the power of two that brings a magnitude (as bits) to [2^14,
// 2^15), of a normal number and with a normal reciprocal; 0 for zero, infinity
// and NaN.
__device__ __forceinline__ int scale_exp(uint32_t mx_bits) {
  const int e = 14 + 127 - (int)(mx_bits >> 23);
  return mx_bits == 0 || mx_bits >= 0x7f800000u ? 0 : min(e, 126);
}
__device__ __forceinline__ float pow2(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// Bits of |x|, 0 for an infinity or NaN.
__device__ __forceinline__ uint32_t finite_bits(float x) {
  const uint32_t u = __float_as_uint(x) & 0x7fffffffu;
  return u < 0x7f800000u ? u : 0u;
}

// Largest magnitude of four values (an infinity's is infinite, a NaN's none).
__device__ __forceinline__ uint32_t max4(const floatx4& v) {
  return __float_as_uint(fmaxf(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fabsf(v[2])), fabsf(v[3])));
}

// Magnitudes of one K/V tile (as bits): the largest of k and of v, and (negated,
// so that all four are maxima and 0 stands for none) the smallest among the
// largest of each staging unit of four that is not all zero.
struct TileMax {
  uint32_t kmax, vmax, klow, vlow;
};
__device__ __forceinline__ void merge(TileMax& m, const TileMax& o) {
  m.kmax = max(m.kmax, o.kmax);
  m.vmax = max(m.vmax, o.vmax);
  m.klow = max(m.klow, o.klow);
  m.vlow = max(m.vlow, o.vlow);
}
template <int kLoads>
__device__ __forceinline__ TileMax unit_max(const floatx4 (&kr)[kLoads], const floatx4 (&vr)[kLoads]) {
  TileMax m = {0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const uint32_t k = max4(kr[j]), v = max4(vr[j]);
    merge(m, TileMax{k, v, 0u - k, 0u - v});
  }
  return m;
}
template <int kCtrl>
__device__ __forceinline__ TileMax dpp(const TileMax& m) {
  return TileMax{(uint32_t)__builtin_amdgcn_mov_dpp((int)m.kmax, kCtrl, 0xf, 0xf, true),
                 (uint32_t)__builtin_amdgcn_mov_dpp((int)m.vmax, kCtrl, 0xf, 0xf, true),
                 (uint32_t)__builtin_amdgcn_mov_dpp((int)m.klow, kCtrl, 0xf, 0xf, true),
                 (uint32_t)__builtin_amdgcn_mov_dpp((int)m.vlow, kCtrl, 0xf, 0xf, true)};
}
// Over the 16 lanes of a row: lane ^ 1, lane ^ 2, halves mirrored, row mirrored.
__device__ __forceinline__ void row_max(TileMax& m) {
  merge(m, dpp<0xb1>(m));
  merge(m, dpp<0x4e>(m));
  merge(m, dpp<0x141>(m));
  merge(m, dpp<0x140>(m));
}

// The maxima over the workgroup, uniform, with a barrier in between; red is
// written again no sooner than another barrier later.
template <int kWaves>
__device__ __forceinline__ TileMax reduce_max(TileMax m, uintx4 (&red)[kWaves * 4]) {
  const int tid = threadIdx.x;
  row_max(m);
  if (tid % 16 == 0) red[tid / 16] = uintx4{m.kmax, m.vmax, m.klow, m.vlow};
  __syncthreads();
  const uintx4 u = red[tid % (kWaves * 4)];
  m = TileMax{u[0], u[1], u[2], u[3]};
  row_max(m);
  if constexpr (kWaves > 4) {
    static_assert(kWaves == 16, "one row, or a wave, of partial maxima");
#pragma unroll
    for (int d = 16; d < 64; d <<= 1)
      merge(m, TileMax{(uint32_t)__shfl_xor((int)m.kmax, d), (uint32_t)__shfl_xor((int)m.vmax, d),
                       (uint32_t)__shfl_xor((int)m.klow, d), (uint32_t)__shfl_xor((int)m.vlow, d)});
  }
  return TileMax{(uint32_t)__builtin_amdgcn_readfirstlane(m.kmax), (uint32_t)__builtin_amdgcn_readfirstlane(m.vmax),
                 (uint32_t)__builtin_amdgcn_readfirstlane(m.klow), (uint32_t)__builtin_amdgcn_readfirstlane(m.vlow)};
}

// A tile's scales, uniform over the workgroup: k * 2^ek and v * 2^ev bring the
// largest finite magnitude to [2^14, 2^15) and, ev a multiple of 4 (so that tiles
// of like values share it and the outputs keep their unit), to [2^11, 2^15).
struct TileInfo {
  int ek, ev;
  uint32_t flags;
  float kmax;
};
constexpr uint32_t kKWide = 1;  // some unit of k is below 2^-4 of its scale
constexpr uint32_t kVZero = 2;  // v has no finite value but zero
constexpr uint32_t kVInf = 4;   // an infinity in v: zero in the planes
constexpr uint32_t kFp32 = 8;   // the pairs do not serve: an infinity in k, or a unit
                                // of v below 2^-5 of its scale, or v of 2^100 and more
template <int kWaves, int kLoads>
__device__ __forceinline__ TileInfo tile_info(const floatx4 (&kr)[kLoads], const floatx4 (&vr)[kLoads],
                                              uintx4 (&red)[kWaves * 4]) {
  TileMax m = reduce_max<kWaves>(unit_max(kr, vr), red);
  TileInfo t;
  t.flags = 0;
  if (m.vmax >= 0x7f800000u) {  // (uniform, rare) the same of v's finite values
    t.flags = kVInf;
    TileMax f = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      uint32_t v = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) v = max(v, finite_bits(vr[j][e]));
      merge(f, TileMax{0, v, 0, 0u - v});
    }
    __syncthreads();
    f = reduce_max<kWaves>(f, red);
    m.vmax = f.vmax;
    m.vlow = f.vlow;
  }
  t.ek = scale_exp(m.kmax);
  t.ev = scale_exp(m.vmax) & ~3;
  t.kmax = __uint_as_float(m.kmax);
  if (m.vmax == 0) t.flags |= kVZero;
  if (m.klow != 0 && __uint_as_float(0u - m.klow) * pow2(t.ek) < 0x1p-4f) t.flags |= kKWide;
  if (m.kmax >= 0x7f800000u || __uint_as_float(m.vmax) >= 0x1p100f ||
      (m.vlow != 0 && __uint_as_float(0u - m.vlow) * pow2(t.ev) < 0x1p-5f))
    t.flags |= kFp32;
  return t;
}
// Whether the pairs serve a tile for queries of at most qmax, whose own spread
// allows |q| |k| up to q_top.
__device__ __forceinline__ bool pairs_serve(uint32_t flags, float kmax, float qmax, float q_top) {
  return (flags & kFp32) == 0 && qmax * kmax <= ((flags & kKWide) != 0 ? fminf(q_top, kWideTop) : q_top);
}

template <int kLayout>
__device__ __forceinline__ int64_t head_stride(const SdpaArgs& a) {
  return kLayout == 1 ? (int64_t)kD * a.Lkp : (int64_t)a.Lk * kD;
}

// LDS image of one K/V tile: fp16 planes of kPlaneElems elements, 0 = K hi,
// 1 = V^T hi, 2 = K lo, 3 = V^T lo; rows (one key, one dim) of 72.
constexpr int kTileKeys = 64;
constexpr int kRowElems = kTileKeys + 8;
constexpr int kPlaneElems = kTileKeys * kRowElems;
constexpr int kPlanes = 4;
static_assert(kTileKeys == kD, "K rows and V^T rows share one stride");

// Fetches thread tid's kLoads float4 units of K and V for the tile at key0.
template <int kLayout, int kThreads, int kLoads>
__device__ __forceinline__ void fetch_kv(const SdpaArgs& a, const float* kbase, const float* vbase, int tid,
                                         int key0, floatx4 (&kr)[kLoads], floatx4 (&vr)[kLoads]) {
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int idx = tid + j * kThreads;
    if constexpr (kLayout == 0) {
      fetch_units_kv<kTileKeys>(a, kbase, vbase, idx, key0, kr[j], vr[j]);
    } else {
      kr[j] = fetch_unit<true, kTileKeys>(a, kbase, idx, key0);
      vr[j] = fetch_unit<true, kTileKeys>(a, vbase, idx, key0);
    }
  }
}

// Scales and splits the fetched units and places them in the planes: K as
// key rows, V transposed to dim rows with its keys at vt_pos.
template <int kLayout, int kThreads, int kLoads>
__device__ __forceinline__ void place_kv(int tid, const TileInfo& t, const floatx4 (&kr)[kLoads],
                                         const floatx4 (&vr)[kLoads], _Float16* planes) {
  _Float16* khi = planes;
  _Float16* vhi = planes + kPlaneElems;
  _Float16* klo = planes + 2 * kPlaneElems;
  _Float16* vlo = planes + 3 * kPlaneElems;
  const float sk = pow2(t.ek), sv = pow2(t.ev);
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int idx = tid + j * kThreads;
    half4v kh, kl, vh, vl;
    split4(kr[j] * sk, kh, kl);
    floatx4 v = vr[j] * sv;
    if (t.flags & kVInf) {  // (uniform)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fabsf(v[e]) < INFINITY ? v[e] : 0.0f;
    }
    split4(v, vh, vl);
    const int row = idx / (kD / 4), c = idx % (kD / 4);
    if constexpr (kLayout == 0) {
      // key row, dims 4c..4c+3
      *reinterpret_cast<half4v*>(&khi[row * kRowElems + 4 * c]) = kh;
      *reinterpret_cast<half4v*>(&klo[row * kRowElems + 4 * c]) = kl;
      const int p = vt_pos(row);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        vhi[(4 * c + e) * kRowElems + p] = vh[e];
        vlo[(4 * c + e) * kRowElems + p] = vl[e];
      }
    } else {
      // dim row, keys 4c..4c+3 (contiguous in V^T: vt_pos keeps bits 0-1)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        khi[(4 * c + e) * kRowElems + row] = kh[e];
        klo[(4 * c + e) * kRowElems + row] = kl[e];
      }
      *reinterpret_cast<half4v*>(&vhi[row * kRowElems + vt_pos(4 * c)]) = vh;
      *reinterpret_cast<half4v*>(&vlo[row * kRowElems + vt_pos(4 * c)]) = vl;
    }
  }
}

// Global image of the staged tiles: per (b*H + h, tile of 64 keys), the LDS
// planes without their row padding, the tile's TileInfo, then with a key bias
// its 64 bias values in log2 units (zero past Lk).
constexpr int kPlaneBytes = kPlanes * kTileKeys * kTileKeys * 2;
constexpr int kInfoBytes = 16;
template <bool kBias>
constexpr int kImageTileBytes = kPlaneBytes + kInfoBytes + (kBias ? kTileKeys * 4 : 0);
constexpr int kPreThreads = 256;

template <int kLayout, bool kBias>
__global__ __launch_bounds__(kPreThreads) void sdpa_f16_presplit_kernel(SdpaArgs a, uintx4* out, int ntiles) {
  constexpr int kLoads = kTileKeys * kD / 4 / kPreThreads;
  constexpr int kUnits = kPlanes * kTileKeys * kTileKeys / 8;  // 16-byte units of the planes
  __shared__ __attribute__((aligned(16))) _Float16 lds[kPlanes * kPlaneElems];
  __shared__ uintx4 red[kPreThreads / 16];
  const int tid = threadIdx.x;
  const int bh = blockIdx.x / ntiles, tile = blockIdx.x % ntiles;
  const int64_t head = head_stride<kLayout>(a);
  floatx4 kr[kLoads], vr[kLoads];
  fetch_kv<kLayout, kPreThreads, kLoads>(a, a.k + bh * head, a.v + bh * head, tid, tile * kTileKeys, kr, vr);
  const TileInfo info = tile_info<kPreThreads / 64>(kr, vr, red);
  place_kv<kLayout, kPreThreads, kLoads>(tid, info, kr, vr, lds);
  __syncthreads();
  uintx4* dst = out + (int64_t)blockIdx.x * (kImageTileBytes<kBias> / 16);
#pragma unroll
  for (int j = 0; j < kUnits / kPreThreads; ++j) {
    const int u = tid + j * kPreThreads;
    const int p = u / (kUnits / kPlanes), r = (u / 8) % kTileKeys, ch = u % 8;
    dst[u] = *reinterpret_cast<const uintx4*>(&lds[p * kPlaneElems + r * kRowElems + 8 * ch]);
  }
  if (tid == 0)
    dst[kUnits] = uintx4{(unsigned)info.ek, (unsigned)info.ev, info.flags, __float_as_uint(info.kmax)};
  if (kBias && tid < kTileKeys) {
    const int key = tile * kTileKeys + tid;
    const float* brow = a.bias + (int64_t)(bh % a.H) * a.bias_head_stride;
    reinterpret_cast<float*>(dst + kUnits + 1)[tid] = key < a.Lk ? brow[key] * kLog2e : 0.0f;
  }
}

// kLayout: 0 = k and v [B, H, Lk, 64]; 1 = both key-contiguous [B, H, 64,
// Lkp].  kWaves waves of 32 queries share each tile of 64 keys, taken in two
// 32-key blocks.  kPre: the tiles come from the presplit image `pre`.
//
// A workgroup that meets a tile the pairs do not serve (pairs_serve, or values
// of v too far apart for one unit of the outputs) drops what it has and runs
// its queries and keys as fp32 products instead (sdpa_fp32.h); with the image it
// looks first.  An infinity in v changes only its own dims: their outputs, and
// no others, come from such a pass at the end.
template <int kLayout, bool kBias, int kWaves, bool kPre>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(kWaves == 4 ? 2 : 4)))
void sdpa_f16_kernel(SdpaArgs a, const uintx4* pre) {
  constexpr int kThreads = kWaves * 64;
  constexpr int kBQ = kWaves * 32;
  constexpr int kUnits = kTileKeys * kD / 4;  // float4 of K (and of V) per tile
  constexpr int kLoads = kPre ? 1 : kUnits / kThreads;
  constexpr int kPUnits = kPlanes * kTileKeys * kD / 8;  // 16-byte units of a tile's image planes
  constexpr int kPLoads = kPre ? kPUnits / kThreads : 1;
  static_assert(kPre ? kPLoads * kThreads == kPUnits : kLoads * kThreads == kUnits, "tile split");
  static_assert(kThreads >= kTileKeys, "bias row load");
  __shared__ union {
    __attribute__((aligned(16))) _Float16 planes[2][kPlanes * kPlaneElems];
    Fp32Lds<kLayout, kTileKeys> fp32;
  } lds;
  __shared__ __attribute__((aligned(16))) float bbuf[2][kTileKeys];
  __shared__ uintx4 red[kWaves * 4];
  auto& kvl = lds.planes;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;
  const int l32 = lane & 31;

  const TileWork w = tile_work(a);
  int bh, qb;
  tile_coords(a, w.tile, kBQ, bh, qb);
  // A wave whose 32 queries all lie past Lq only helps stage K/V.
  const bool wave_live = qb * kBQ + wave * 32 < a.Lq;
  const int h = bh % a.H;
  const int qrow = qb * kBQ + wave * 32 + l32;
  const bool q_ok = qrow < a.Lq;

  const float* kbase = a.k + bh * head_stride<kLayout>(a);
  const float* vbase = a.v + bh * head_stride<kLayout>(a);
  const float* brow = kBias ? a.bias + (int64_t)h * a.bias_head_stride : nullptr;
  constexpr int kTileBytes = kImageTileBytes<kBias>;
  const char* pbase = kPre ? reinterpret_cast<const char*>(pre) +
                                 (int64_t)bh * ((a.Lk + kTileKeys - 1) / kTileKeys) * kTileBytes
                           : nullptr;

  // Q slices in registers: dims 16c + 8g + i of the query under its own scale.
  half8 qh[4], ql[4];
  int eq;  // exponent of the query's scale
  // The pairs serve a tile's scores where qmax, the workgroup's largest |q|, times
  // the tile's largest |k| is at most q_top.
  float qmax, q_top;
  {
    const float* qp = a.q + ((int64_t)bh * a.Lq + (q_ok ? qrow : 0)) * kD + 8 * g;
    floatx4 x[8];
    uint32_t mx = 0, low = 0;
    bool inf = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = q_ok ? *reinterpret_cast<const floatx4*>(qp + 16 * (i / 2) + 4 * (i % 2)) : floatx4{0, 0, 0, 0};
      uint32_t m = max4(x[i]);
      inf |= m >= 0x7f800000u;
      low = max(low, 0u - m);
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = max(mx, finite_bits(x[i][e]));
    }
    mx = __float_as_uint(pair_max(__uint_as_float(mx)));
    eq = scale_exp(mx);
    // (4 neighbouring dims of a query below 2^-4 of its scale)
    const bool wide = low != 0 && __uint_as_float(0u - low) * pow2(eq) < 0x1p-4f;
    TileMax m = {mx, 0, wide ? 1u : 0u, inf ? 1u : 0u};
    m = reduce_max<kWaves>(m, red);
    qmax = __uint_as_float(m.kmax);
    q_top = m.vlow != 0 ? -1.0f : m.klow != 0 ? kWideTop : kPairTop;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      half4v hi[2], lo[2];
      split4(x[2 * c] * pow2(eq), hi[0], lo[0]);
      split4(x[2 * c + 1] * pow2(eq), hi[1], lo[1]);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        qh[c][e] = hi[e / 4][e % 4];
        ql[c][e] = lo[e / 4][e % 4];
      }
    }
  }

  floatx4 kr[kLoads], vr[kLoads];
  uintx4 pr[kPLoads];
  float br = 0.0f;
  // load(key0, buf): kPre fetches this thread's 16-byte units of the tile's
  // image planes, and the last wave copies the bias row straight into LDS
  // buffer buf; otherwise the fp32 units and the bias value.  store(buf)
  // places them in LDS buffer buf, before the barrier that publishes it.
  // (tid_s: the units' addresses are formed where they are used, not held over
  // the tile)
  auto load = [&](int key0, int buf) {
    int tid_s = tid;
    if constexpr (kWaves == 16 && !kPre) asm volatile("" : "+v"(tid_s));
    if constexpr (kPre) {
      const char* src = pbase + (int64_t)(key0 / kTileKeys) * kTileBytes;
#pragma unroll
      for (int j = 0; j < kPLoads; ++j) pr[j] = reinterpret_cast<const uintx4*>(src)[tid + j * kThreads];
      if (kBias && __builtin_amdgcn_readfirstlane(wave) == kWaves - 1)
        __builtin_amdgcn_global_load_lds(src + kPUnits * 16 + kInfoBytes + lane * 4,
                                         (__attribute__((address_space(3))) void*)(&bbuf[buf][0]), 4, 0, 0);
    } else {
      fetch_kv<kLayout, kThreads, kLoads>(a, kbase, vbase, tid_s, key0, kr, vr);
      if (kBias && tid < kTileKeys) {
        const int key = key0 + tid;
        br = key < a.Lk ? brow[key] * kLog2e : 0.0f;
      }
    }
  };
  TileInfo info;  // of the tile placed last
  auto store = [&](int key0, int buf) {
    int tid_s = tid;
    if constexpr (kWaves == 16 && !kPre) asm volatile("" : "+v"(tid_s));
    if constexpr (kPre) {
#pragma unroll
      for (int j = 0; j < kPLoads; ++j) {
        const int u = tid + j * kThreads;
        const int p = u / (kPUnits / kPlanes), r = (u / 8) % kTileKeys, ch = u % 8;
        *reinterpret_cast<uintx4*>(&kvl[buf][p * kPlaneElems + r * kRowElems + 8 * ch]) = pr[j];
      }
      if constexpr (kBias) __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
      const auto* ip = reinterpret_cast<const __attribute__((address_space(4))) unsigned*>(
          reinterpret_cast<uintptr_t>(pbase + (int64_t)(key0 / kTileKeys) * kTileBytes + kPlaneBytes));
      info = TileInfo{(int)ip[0], (int)ip[1], ip[2], __uint_as_float(ip[3])};
    } else {
      info = tile_info<kWaves>(kr, vr, red);
      place_kv<kLayout, kThreads, kLoads>(tid_s, info, kr, vr, kvl[buf]);
      if (kBias && tid < kTileKeys) bbuf[buf][tid_s] = br;
    }
  };

  floatx16 o[2];
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.0f;
  float m_run = kStart;  // the reference
  // some query's reference, or with a bias a score before it, may be beyond 2^20
  // (uniform over the wave): exponents are then differences of rounded scores, 0
  // at the maximum
  bool huge = false;
  float l_run = 0.0f;
  int ev = 0;  // the outputs' unit: 2^-ev

  // (all uniform over the workgroup)
  const int ntiles = (w.k_end - w.k_begin + kTileKeys - 1) / kTileKeys;
  int served = 1, v_inf = 0;
  int ev_min = kEvRange, ev_max = -kEvRange;
  if constexpr (kPre) {
    bool bad = false, inf = false;
    uint32_t hi = 0, lo = 0;
    for (int i = tid; i < ntiles; i += kThreads) {
      const uintx4 u = *reinterpret_cast<const uintx4*>(pbase + (int64_t)(w.k_begin / kTileKeys + i) * kTileBytes +
                                                        kPlaneBytes);
      bad |= !pairs_serve(u[2], __uint_as_float(u[3]), qmax, q_top);
      inf |= (u[2] & kVInf) != 0;
      if ((u[2] & kVZero) == 0) {
        hi = max(hi, (uint32_t)(kEvRange + (int)u[1]));
        lo = max(lo, (uint32_t)(kEvRange - (int)u[1]));
      }
    }
    const TileMax m = reduce_max<kWaves>(TileMax{bad, inf, hi, lo}, red);
    served = m.kmax == 0 && (int)(m.klow + m.vlow) <= 2 * kEvRange + kEvSpread ? 1 : 0;
    v_inf = (int)m.vmax;
  }
  // Whether the tile placed last is one to go on with.
  auto take = [&] {
    v_inf |= (int)(info.flags & kVInf);
    if ((info.flags & kVZero) == 0) {
      ev_min = min(ev_min, info.ev);
      ev_max = max(ev_max, info.ev);
    }
    served = pairs_serve(info.flags, info.kmax, qmax, q_top) && ev_max - ev_min <= kEvSpread ? 1 : 0;
    return served != 0;
  };

  if (served != 0) {
    load(w.k_begin, 0);
    store(w.k_begin, 0);
    if (!kPre) (void)take();
    __syncthreads();
  }

  for (int t = 0; served != 0 && t < ntiles; ++t) {
    const int buf = t & 1;
    const int key0 = w.k_begin + t * kTileKeys;
    if (t + 1 < ntiles) load(key0 + kTileKeys, buf ^ 1);
    const _Float16* kh_ = kvl[buf];
    const _Float16* vh_ = kvl[buf] + kPlaneElems;
    const _Float16* kl_ = kvl[buf] + 2 * kPlaneElems;
    const _Float16* vl_ = kvl[buf] + 3 * kPlaneElems;
    const bool tail = key0 + kTileKeys > a.Lk;

    if (wave_live) {
      // log2 units per unit of the score accumulator, kept positive and finite,
      // so that a masked score stays -inf
      const float c1 =
          __builtin_amdgcn_fmed3f(__builtin_amdgcn_ldexpf(0.125f * kLog2e, -eq - info.ek), 0x1p-126f, 0x1p127f);
      if (kBias) huge |= qmax * info.kmax > kFarScores;
      if (info.ev != ev && (info.flags & kVZero) == 0) {
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[db][r] = __builtin_amdgcn_ldexpf(o[db][r], info.ev - ev);
        ev = info.ev;
      }
      // The 16-wave kernels have 128 registers: with a bias, or tiles split
      // here, the blocks and their phases are kept apart (one block in flight,
      // no instruction moved between scores, softmax and P V), or they spill.
      constexpr bool kTight = kWaves == 16 && (kBias || !kPre);
      constexpr int kBlockUnroll = kTight ? 1 : 2;
#pragma unroll kBlockUnroll
      for (int kb = 0; kb < kTileKeys / 32; ++kb) {
        floatx16 s;
        float m_ref;
        // Once, and with a bias again when the reference has to move: the
        // exponents x - m + 4 are then one FMA each (rounded at their own size,
        // not at x's), taken under the reference so far (0 before any key).
        for (;;) {
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int off = (kb * 32 + l32) * kRowElems + 16 * c + 8 * g;
            const half8 kf = *reinterpret_cast<const half8*>(kh_ + off);
            const half8 kfl = *reinterpret_cast<const half8*>(kl_ + off);
            s = mfma_f16(kf, qh[c], s);
            s = mfma_f16(kf, ql[c], s);
            s = mfma_f16(kfl, qh[c], s);
          }
          if constexpr (kTight) __builtin_amdgcn_sched_barrier(0);
          const bool fresh = m_run == kStart;
          m_ref = kBias && fresh ? 0.0f : m_run;
          if constexpr (kBias) {
            const float sub = huge ? 0.0f : m_ref - kPBase;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
              const floatx4 bb = *reinterpret_cast<const floatx4*>(&bbuf[buf][kb * 32 + 8 * r4 + 4 * g]);
#pragma unroll
              for (int e = 0; e < 4; ++e) s[4 * r4 + e] = fmaf(s[4 * r4 + e], c1, bb[e] - sub);
            }
          }
          if (tail) {
            const int valid = a.Lk - key0 - 4 * g;
#pragma unroll
            for (int r = 0; r < 16; ++r)
              if (kb * 32 + 8 * (r / 4) + (r % 4) >= valid) s[r] = -INFINITY;
          }
          float mx = -INFINITY;
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
          mx = pair_max(mx);
          if constexpr (!kBias) {
            mx *= c1;
          } else if (huge) {
            // (the maximum from the scores as they are: the next reference has
            // to be exact also where this one is a mask of many digits)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = (s[r] - m_ref) + kPBase;
          } else {
            mx = (mx - kPBase) + m_ref;
          }
          const bool move = fresh ? mx > -INFINITY : mx > m_run + kSlack;
          if (__builtin_amdgcn_ballot_w64(move) == 0) break;
          const float m_new = move ? mx : m_run;
          const float alpha = move ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
          l_run *= alpha;
#pragma unroll
          for (int db = 0; db < 2; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
          m_run = m_new;
          huge |= __builtin_amdgcn_ballot_w64(m_run != kStart && fabsf(m_run) > 0x1p20f) != 0;
          if constexpr (!kBias) {
            m_ref = m_run;
            break;
          }
        }
        float ce = kBias ? 1.0f : c1, re = kBias ? 0.0f : m_ref - kPBase;
        if (!kBias && huge) {
#pragma clang fp contract(off)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] = (s[r] * c1 - m_ref) + kPBase;
          ce = 1.0f;
          re = 0.0f;
        }
        float ls = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          s[r] = __builtin_amdgcn_exp2f(kBias ? s[r] : fmaf(s[r], ce, -re)) * (float)(1 << kPShift);
          ls += s[r];
        }
        l_run += ls;

        if constexpr (kTight) __builtin_amdgcn_sched_barrier(0);
        // O^T[d][query] += V^T P^T, two 16-key slices per 32-key block.
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          half8 ph, pl;
          split8(s, c, ph, pl);
#pragma unroll
          for (int db = 0; db < 2; ++db) {
            const int off = (db * 32 + l32) * kRowElems + kb * 32 + 16 * c + 8 * g;
            const half8 vf = *reinterpret_cast<const half8*>(vh_ + off);
            const half8 vfl = *reinterpret_cast<const half8*>(vl_ + off);
            o[db] = mfma_f16(vf, ph, o[db]);
            o[db] = mfma_f16(vf, pl, o[db]);
            o[db] = mfma_f16(vfl, ph, o[db]);
          }
        }
      }
    }  // wave_live

    if (t + 1 < ntiles) {
      store(key0 + kTileKeys, buf ^ 1);
      if (!kPre && !take()) break;
    }
    __syncthreads();
  }

  // (nothing of the query tile's coordinates is kept over the key tiles)
  SdpaArgs e = a;
  int tid_e = tid;
  asm volatile("" : "+s"(e.Lq), "+s"(e.H), "+v"(tid_e));
  tid_e &= kThreads - 1;  // (its range)
  if (served != 0) {
    // the outputs of weights exp2(x - m_run), as the fp32 tiles' partial rows
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[db][r] = __builtin_amdgcn_ldexpf(o[db][r], -(int)kPBase - kPShift - ev);
    // (without a key, the fp32 tiles' reference, which is no larger than a key's)
    store_rows<kBQ>(e, o, fmaxf(m_run, -FLT_MAX), l_run * 0x1p-11f, tid_e);
    if (v_inf == 0) return;
  }
  __syncthreads();
  sdpa_fp32_tile<kLayout, kBias, kWaves, kTileKeys, true>(e, lds.fp32.k, lds.fp32.v, bbuf, tid_e, served != 0);
}

template <int kLayout, bool kBias, int kWaves, bool kPre>
int launch_shape(const SdpaParams& p, hipStream_t stream, const TilePlan& pl, const uintx4* pre) {
  return launch_plan(make_args(p), p, pl, kWaves * 32, stream, [&](dim3 grid, const SdpaArgs& a) {
    hipLaunchKernelGGL((sdpa_f16_kernel<kLayout, kBias, kWaves, kPre>), grid, dim3(kWaves * 64), 0, stream, a,
                       pre);
  });
}

// Largest presplit image the library allocates for one call (512 bytes per
// key and head, as much as the fp32 K and V).
constexpr size_t kPreMaxImageBytes = size_t(2) << 30;

// Keys from which tiles of 128 queries may be split along the keys (the plan's
// model was fitted there).
constexpr int kRangeMinKeys = 1024;

// Query tiles of 512 per head from which the presplit pass is used: the pass
// against every workgroup splitting the tiles it reads, 8 tiles 424 against 487
// us (2 x 16 heads, 4096 x 4096) and 116 against 122 (4096 x 1024), 4 tiles 212
// against 222, key-contiguous k/v 239 against 274 (4 x 16 heads, 2048 x 2048); 2
// tiles 131 against 130, one 86 against 73.
constexpr int kPreMinQueryTiles = 4;

template <int kLayout, bool kBias>
int launch_sized(SdpaParams p, hipStream_t stream) {
  const int cus = compute_units();
  const int64_t heads = (int64_t)p.B * p.H, qtiles = (p.Lq + 511) / 512;
  const bool wide = heads * qtiles >= cus;
  const int64_t ntiles = (p.Lk + kTileKeys - 1) / kTileKeys;
  TilePlan pl;
  if (!plan_tiles(p.B, p.H, p.Lq, p.Lk, wide ? 512 : 128, kTileKeys, kD, wide ? cus : 0, pl)) return kErrDims;
  // Few queries leave CUs of the 128-query tiles idle: those are split along
  // the keys, where there is room for the ranges' rows.  Elsewhere (a small
  // caller scratch, no memory, or a capture that would need the workspace to
  // grow) they run whole, with the sums in one order instead of the ranges'.
  const TilePlan whole = pl;
  if (!wide && p.Lk >= kRangeMinKeys) {
    plan_key_ranges(p.B, p.H, p.Lq, p.Lk, 128, kTileKeys, kD, cus, pl);
    if (p.scratch != nullptr && pl.scratch_bytes > p.scratch_bytes) pl = whole;
  }
  const size_t part_bytes = (pl.scratch_bytes + 255) / 256 * 256;
  const size_t image_bytes = (size_t)heads * ntiles * kImageTileBytes<kBias>;
  bool image = wide && p.scratch == nullptr && qtiles >= kPreMinQueryTiles &&
               image_bytes <= kPreMaxImageBytes && heads * ntiles <= 0x7fffffff;
  uintx4* img = nullptr;
  if (p.scratch == nullptr && (image || (!wide && pl.pieces > 0))) {
    // One buffer: partials, image.  Without it the workgroups split k and v
    // themselves, with the same result.
    void* ws = stream_workspace(stream, part_bytes + (image ? image_bytes : 0), kSlotSdpaPartial);
    if (ws == nullptr) {
      image = false;
      if (!wide) pl = whole;
    } else {
      p.scratch = static_cast<float*>(ws);
      p.scratch_bytes = pl.scratch_bytes;
      img = reinterpret_cast<uintx4*>(static_cast<char*>(ws) + part_bytes);
    }
  }
  if (image) {
    hipLaunchKernelGGL((sdpa_f16_presplit_kernel<kLayout, kBias>), dim3((unsigned)(heads * ntiles)),
                       dim3(kPreThreads), 0, stream, make_args(p), img, (int)ntiles);
    if (hipGetLastError() != hipSuccess) return kErrLaunch;
    return launch_shape<kLayout, kBias, 16, true>(p, stream, pl, img);
  }
  if (wide) return launch_shape<kLayout, kBias, 16, false>(p, stream, pl, nullptr);
  return launch_shape<kLayout, kBias, 4, false>(p, stream, pl, nullptr);
}

}  // namespace
}  // namespace sdpa

int launch_sdpa_f16(const SdpaParams& p, hipStream_t stream) {
  using namespace sdpa;
  const bool bias = p.bias != nullptr;
  if (p.kv_packed) return bias ? launch_sized<1, true>(p, stream) : launch_sized<1, false>(p, stream);
  return bias ? launch_sized<0, true>(p, stream) : launch_sized<0, false>(p, stream);
}

}  // namespace tsplat
