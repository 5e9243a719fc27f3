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
// A pair holds its value to one unit of fp32's last place down to 2^-24 of
// the scale and to 2^-25 of the scale below that; the dropped low x low
// product is below 2^-22 of the product (2^-24 rms).  sq is the query row's
// own, sk and sv are the (b, h)'s: they bring the largest finite magnitude to
// [2^14, 2^15), so what a score or an output loses to the scale is below
// 2^-37 of |q| |k|max or |v|max.  Products of fp16 values are exact in fp32
// and the matrix core rounds its accumulator twice per 16 products, so the
// error against 64 bits is below the fp32 MFMA kernel's (16 heads, L = 16384:
// 1.5e-6 against 2.3e-6 relative; L = 8194 with log(8194) on one key 2.2e-7,
// as there).
//
// Softmax in log2 units with a lazy reference: p = exp2(x - m + 4) for a
// reference m that follows the running maximum only when that has moved by
// more than 4, so p stays below 2^8 and most 32-key blocks rescale nothing;
// the sums and the outputs share the factor, which 2^7 more bring up to the
// pairs' range.  Without a bias the exponent is
// one FMA of the accumulator; with one as well, and a block that moves the
// reference computes its scores again.
//
// An infinity or NaN of k or v does not enter the scales and sits in the low
// part alone (the high part is held to +-65504), where it meets qh or ph: the
// score or output it makes is the one fp32 products would give.
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
// Measured (16 heads) against the fp32 MFMA kernel: L = 16384 7.88 -> 2.75 ms
// (400 TFLOP/s), 12294 4.57 -> 1.62 ms, 8194 with a key bias 2.14 -> 0.81 ms,
// 4096 x 2048 280 -> 143 us, 577 52 -> 39 us.  What bounds it: the fp16 matrix
// cores at the clock they hold, 1.2 PFLOP/s at L = 16384 where a plain 8192^3
// fp16 library product reaches 1.11 (waves of 64 queries, which read half the
// LDS fragments per product, 3.05 against 2.97 ms; wave priorities no change).
// The 128-query tiles are split along the keys where CUs would idle
// (plan_key_ranges): 300 x 9000 420 -> 102 us.

#include "sdpa_common.h"

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
constexpr float kStart = -3.0e38f;   // the reference before any key
// p is taken up by 2^kPShift before it is split: below 2^15, and held to 2^-25,
// 2^-36 of a weight at the reference (many small weights add up: 16384 of them,
// each 2^-30 of one key's, were lost to the pairs, not to their sum).  After the
// exponential, so that its argument stays small.
constexpr int kPShift = 7;

// Position of tile key k in a V^T row: bits 2 and 3 swapped.
__device__ __forceinline__ int vt_pos(int k) { return (k & ~12) | ((k & 4) << 1) | ((k & 8) >> 1); }

// (hi, lo) of a and b: hi = fp16(v), lo = fp16(v - hi), the difference exact
// in fp32.  kClamp: hi within fp16's finite range.
template <bool kClamp>
__device__ __forceinline__ void split2(float a, float b, unsigned& hi, unsigned& lo) {
  const float ca = kClamp ? __builtin_amdgcn_fmed3f(a, -65504.0f, 65504.0f) : a;
  const float cb = kClamp ? __builtin_amdgcn_fmed3f(b, -65504.0f, 65504.0f) : b;
  const half2v h = __builtin_convertvector(floatx2{ca, cb}, half2v);
  hi = __builtin_bit_cast(unsigned, h);
  lo = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a - (float)h[0], b - (float)h[1]}, half2v));
}

template <bool kClamp>
__device__ __forceinline__ void split4(const floatx4& v, half4v& hi, half4v& lo) {
  unsigned h[2], l[2];
  split2<kClamp>(v[0], v[1], h[0], l[0]);
  split2<kClamp>(v[2], v[3], h[1], l[1]);
  hi = __builtin_bit_cast(half4v, uintx2{h[0], h[1]});
  lo = __builtin_bit_cast(half4v, uintx2{l[0], l[1]});
}

// Elements 8c..8c+7 of an accumulator block, split.
__device__ __forceinline__ void split8(const floatx16& s, int c, half8& hi, half8& lo) {
  unsigned h[4], l[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) split2<false>(s[8 * c + 2 * e], s[8 * c + 2 * e + 1], h[e], l[e]);
  hi = __builtin_bit_cast(half8, uintx4{h[0], h[1], h[2], h[3]});
  lo = __builtin_bit_cast(half8, uintx4{l[0], l[1], l[2], l[3]});
}

// Power of two that brings a magnitude (as bits) to [2^14, 2^15), with a
// normal reciprocal; 1 for zero.
__device__ __forceinline__ float scale_for(uint32_t mx_bits) {
  const int field = 268 - (int)(mx_bits >> 23);
  return mx_bits == 0 ? 1.0f : __uint_as_float((uint32_t)min(max(field, 1), 253) << 23);
}
__device__ __forceinline__ float inverse_pow2(float s) {
  return __uint_as_float((254u << 23) - __float_as_uint(s));
}

// Bits of |x|, 0 for an infinity or NaN.
__device__ __forceinline__ uint32_t finite_bits(float x) {
  const uint32_t u = __float_as_uint(x) & 0x7fffffffu;
  return u < 0x7f800000u ? u : 0u;
}

// Largest finite magnitudes of k and v (as bits) over units first, first +
// step, ... below `end` of one (b, h); a unit is 4 consecutive floats.
template <int kLayout>
__device__ __forceinline__ void kv_max(const SdpaArgs& a, const float* kbase, const float* vbase, int64_t first,
                                       int64_t end, int step, uint32_t& km, uint32_t& vm) {
  for (int64_t u = first; u < end; u += step) {
    const floatx4 kx = *reinterpret_cast<const floatx4*>(kbase + 4 * u);
    const floatx4 vx = *reinterpret_cast<const floatx4*>(vbase + 4 * u);
    // key-contiguous rows: keys past Lk are not part of the operand
    const int key = kLayout == 1 ? (int)(u % (a.Lkp / 4)) * 4 : 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = kLayout == 0 || key + e < a.Lk;
      km = max(km, in ? finite_bits(kx[e]) : 0u);
      vm = max(vm, in ? finite_bits(vx[e]) : 0u);
    }
  }
}
template <int kLayout>
__device__ __forceinline__ int64_t kv_units(const SdpaArgs& a) {
  return kLayout == 1 ? (int64_t)kD * a.Lkp / 4 : (int64_t)a.Lk * kD / 4;
}
template <int kLayout>
__device__ __forceinline__ int64_t head_stride(const SdpaArgs& a) {
  return kLayout == 1 ? (int64_t)kD * a.Lkp : (int64_t)a.Lk * kD;
}

__device__ __forceinline__ uint32_t wave_max(uint32_t x) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) x = max(x, (uint32_t)__shfl_xor((int)x, d));
  return x;
}

// Magnitudes of k and v over one of the kMaxParts parts of a (b, h)'s keys:
// maxes[bh][part] = (k, v).
constexpr int kMaxParts = 16;
constexpr int kMaxThreads = 256;
template <int kLayout>
__global__ __launch_bounds__(kMaxThreads) void sdpa_f16_max_kernel(SdpaArgs a, uint2* maxes) {
  __shared__ uint32_t red[2][kMaxThreads / 64];
  const int bh = blockIdx.x / kMaxParts, part = blockIdx.x % kMaxParts;
  const int64_t units = kv_units<kLayout>(a), per = (units + kMaxParts - 1) / kMaxParts;
  uint32_t km = 0, vm = 0;
  kv_max<kLayout>(a, a.k + bh * head_stride<kLayout>(a), a.v + bh * head_stride<kLayout>(a),
                  part * per + threadIdx.x, min(units, (part + 1) * per), kMaxThreads, km, vm);
  km = wave_max(km);
  vm = wave_max(vm);
  if (threadIdx.x % 64 == 0) {
    red[0][threadIdx.x / 64] = km;
    red[1][threadIdx.x / 64] = vm;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < kMaxThreads / 64; ++i) {
      km = max(km, red[0][i]);
      vm = max(vm, red[1][i]);
    }
    maxes[blockIdx.x] = uint2{km, vm};
  }
}

// sk and sv of a (b, h) from its parts.
__device__ __forceinline__ void head_scales(const uint2* maxes, int bh, float& sk, float& sv) {
  const uint2 m = maxes[(int64_t)bh * kMaxParts + threadIdx.x % kMaxParts];
  sk = scale_for(wave_max(m.x));
  sv = scale_for(wave_max(m.y));
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
__device__ __forceinline__ void place_kv(int tid, float sk, float sv, const floatx4 (&kr)[kLoads],
                                         const floatx4 (&vr)[kLoads], _Float16* planes) {
  _Float16* khi = planes;
  _Float16* vhi = planes + kPlaneElems;
  _Float16* klo = planes + 2 * kPlaneElems;
  _Float16* vlo = planes + 3 * kPlaneElems;
#pragma unroll
  for (int j = 0; j < kLoads; ++j) {
    const int idx = tid + j * kThreads;
    half4v kh, kl, vh, vl;
    split4<true>(kr[j] * sk, kh, kl);
    split4<true>(vr[j] * sv, vh, vl);
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
// planes without their row padding, then with a key bias the tile's 64 bias
// values in log2 units (zero past Lk).
template <bool kBias>
constexpr int kImageTileBytes = kPlanes * kTileKeys * kTileKeys * 2 + (kBias ? kTileKeys * 4 : 0);
constexpr int kPreThreads = 256;

template <int kLayout, bool kBias>
__global__ __launch_bounds__(kPreThreads) void sdpa_f16_presplit_kernel(SdpaArgs a, const uint2* maxes, uintx4* out,
                                                                        int ntiles) {
  constexpr int kLoads = kTileKeys * kD / 4 / kPreThreads;
  constexpr int kUnits = kPlanes * kTileKeys * kTileKeys / 8;  // 16-byte units of the planes
  __shared__ __attribute__((aligned(16))) _Float16 lds[kPlanes * kPlaneElems];
  const int tid = threadIdx.x;
  const int bh = blockIdx.x / ntiles, tile = blockIdx.x % ntiles;
  const int64_t head = head_stride<kLayout>(a);
  floatx4 kr[kLoads], vr[kLoads];
  fetch_kv<kLayout, kPreThreads, kLoads>(a, a.k + bh * head, a.v + bh * head, tid, tile * kTileKeys, kr, vr);
  float sk, sv;
  head_scales(maxes, bh, sk, sv);
  place_kv<kLayout, kPreThreads, kLoads>(tid, sk, sv, kr, vr, lds);
  __syncthreads();
  uintx4* dst = out + (int64_t)blockIdx.x * (kImageTileBytes<kBias> / 16);
#pragma unroll
  for (int j = 0; j < kUnits / kPreThreads; ++j) {
    const int u = tid + j * kPreThreads;
    const int p = u / (kUnits / kPlanes), r = (u / 8) % kTileKeys, ch = u % 8;
    dst[u] = *reinterpret_cast<const uintx4*>(&lds[p * kPlaneElems + r * kRowElems + 8 * ch]);
  }
  if (kBias && tid < kTileKeys) {
    const int key = tile * kTileKeys + tid;
    const float* brow = a.bias + (int64_t)(bh % a.H) * a.bias_head_stride;
    reinterpret_cast<float*>(dst + kUnits)[tid] = key < a.Lk ? brow[key] * kLog2e : 0.0f;
  }
}

// kLayout: 0 = k and v [B, H, Lk, 64]; 1 = both key-contiguous [B, H, 64,
// Lkp].  kWaves waves of 32 queries share each tile of 64 keys, taken in two
// 32-key blocks.  kPre: the tiles come from the presplit image `pre` (kLayout
// is then unused).  maxes: sdpa_f16_max_kernel's result, or null, and the
// workgroup looks through its (b, h)'s k and v itself.
template <int kLayout, bool kBias, int kWaves, bool kPre>
__global__ __launch_bounds__(kWaves * 64) void sdpa_f16_kernel(SdpaArgs a, const uint2* maxes, const uintx4* pre) {
  constexpr int kThreads = kWaves * 64;
  constexpr int kBQ = kWaves * 32;
  constexpr int kUnits = kTileKeys * kD / 4;  // float4 of K (and of V) per tile
  constexpr int kLoads = kPre ? 1 : kUnits / kThreads;
  constexpr int kPUnits = kPlanes * kTileKeys * kD / 8;  // 16-byte units of a tile's image planes
  constexpr int kPLoads = kPre ? kPUnits / kThreads : 1;
  static_assert(kPre ? kPLoads * kThreads == kPUnits : kLoads * kThreads == kUnits, "tile split");
  static_assert(kThreads >= kTileKeys, "bias row load");
  __shared__ __attribute__((aligned(16))) _Float16 kvl[2][kPlanes * kPlaneElems];
  __shared__ __attribute__((aligned(16))) float bbuf[2][kTileKeys];

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

  const float* kbase = a.k + (int64_t)bh * head_stride<kLayout>(a);
  const float* vbase = a.v + (int64_t)bh * head_stride<kLayout>(a);
  const float* brow = kBias ? a.bias + (int64_t)h * a.bias_head_stride : nullptr;
  constexpr int kTileBytes = kImageTileBytes<kBias>;
  const char* pbase = kPre ? reinterpret_cast<const char*>(pre) +
                                 (int64_t)bh * ((a.Lk + kTileKeys - 1) / kTileKeys) * kTileBytes
                           : nullptr;

  float sk, sv;
  if (kPre || maxes != nullptr) {
    head_scales(maxes, bh, sk, sv);
  } else {
    uint32_t km = 0, vm = 0;
    kv_max<kLayout>(a, kbase, vbase, tid, kv_units<kLayout>(a), kThreads, km, vm);
    km = wave_max(km);
    vm = wave_max(vm);
    uint32_t* red = reinterpret_cast<uint32_t*>(&kvl[0][0]);
    if (lane == 0) {
      red[2 * wave] = km;
      red[2 * wave + 1] = vm;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kWaves; ++i) {
      km = max(km, red[2 * i]);
      vm = max(vm, red[2 * i + 1]);
    }
    __syncthreads();
    sk = scale_for(km);
    sv = scale_for(vm);
  }
  sk = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(sk)));
  sv = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(sv)));

  // Q slices in registers: dims 16c + 8g + i of the query under its own scale.
  half8 qh[4], ql[4];
  float c1;  // log2 units per unit of the score accumulator
  {
    const float* qp = a.q + ((int64_t)bh * a.Lq + (q_ok ? qrow : 0)) * kD + 8 * g;
    floatx4 x[8];
    uint32_t mx = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = q_ok ? *reinterpret_cast<const floatx4*>(qp + 16 * (i / 2) + 4 * (i % 2)) : floatx4{0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 4; ++e) mx = max(mx, finite_bits(x[i][e]));
    }
    mx = __float_as_uint(pair_max(__uint_as_float(mx)));
    const float sq = scale_for(mx);
    // kept positive and finite, so that a masked score stays -inf
    c1 = __builtin_amdgcn_fmed3f(0.125f * kLog2e * inverse_pow2(sq) * inverse_pow2(sk), 0x1p-126f, 0x1p127f);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      half4v hi[2], lo[2];
      split4<false>(x[2 * c] * sq, hi[0], lo[0]);
      split4<false>(x[2 * c + 1] * sq, hi[1], lo[1]);
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
        __builtin_amdgcn_global_load_lds(src + kPUnits * 16 + lane * 4,
                                         (__attribute__((address_space(3))) void*)(&bbuf[buf][0]), 4, 0, 0);
    } else {
      fetch_kv<kLayout, kThreads, kLoads>(a, kbase, vbase, tid_s, key0, kr, vr);
      if (kBias && tid < kTileKeys) {
        const int key = key0 + tid;
        br = key < a.Lk ? brow[key] * kLog2e : 0.0f;
      }
    }
  };
  auto store = [&](int buf) {
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
    } else {
      place_kv<kLayout, kThreads, kLoads>(tid_s, sk, sv, kr, vr, kvl[buf]);
      if (kBias && tid < kTileKeys) bbuf[buf][tid] = br;
    }
  };

  floatx16 o[2];
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.0f;
  float m_run = kStart;  // the reference
  // some query's reference is beyond 2^20 (uniform over the wave): exponents
  // are then differences of rounded scores, 0 at the maximum
  bool huge = false;
  float l_run = 0.0f;

  const int ntiles = (w.k_end - w.k_begin + kTileKeys - 1) / kTileKeys;
  load(w.k_begin, 0);
  store(0);
  __syncthreads();

  for (int t = 0; t < ntiles; ++t) {
    const int buf = t & 1;
    const int key0 = w.k_begin + t * kTileKeys;
    if (t + 1 < ntiles) load(key0 + kTileKeys, buf ^ 1);
    const _Float16* kh_ = kvl[buf];
    const _Float16* vh_ = kvl[buf] + kPlaneElems;
    const _Float16* kl_ = kvl[buf] + 2 * kPlaneElems;
    const _Float16* vl_ = kvl[buf] + 3 * kPlaneElems;
    const bool tail = key0 + kTileKeys > a.Lk;

    if (wave_live) {
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
            if (huge) {
#pragma unroll
              for (int r = 0; r < 16; ++r) s[r] = (s[r] - m_ref) + kPBase;
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
          mx = kBias ? (mx - kPBase) + m_ref : mx * c1;
          const bool move = fresh ? mx > -INFINITY : mx > m_run + kSlack;
          if (__builtin_amdgcn_ballot_w64(move) == 0) break;
          const float m_new = move ? mx : m_run;
          const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
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

    if (t + 1 < ntiles) store(buf ^ 1);
    __syncthreads();
  }

  // sums and outputs of weights of at most 1 (kPBase + kSlack + kPShift = 15),
  // which overflow no sooner than the result
  const float unscale = inverse_pow2(sv);
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = o[db][r] * 0x1p-15f * unscale;
  store_rows<kBQ>(a, o, m_run, l_run * 0x1p-15f);
}

template <int kLayout, bool kBias, int kWaves, bool kPre>
int launch_shape(const SdpaParams& p, hipStream_t stream, const TilePlan& pl, const uint2* maxes, const uintx4* pre) {
  return launch_plan(make_args(p), p, pl, kWaves * 32, stream, [&](dim3 grid, const SdpaArgs& a) {
    hipLaunchKernelGGL((sdpa_f16_kernel<kLayout, kBias, kWaves, kPre>), grid, dim3(kWaves * 64), 0, stream, a,
                       maxes, pre);
  });
}

// Largest presplit image the library allocates for one call (512 bytes per
// key and head, as much as the fp32 K and V).
constexpr size_t kPreMaxImageBytes = size_t(2) << 30;

// Keys from which the magnitudes of a (b, h)'s k and v are worth a launch of
// their own; below, every workgroup looks through them.
constexpr int kMaxLaunchKeys = 1024;

// Query tiles of 512 per head from which the presplit pass is used (the
// break-even of sdpa_bf16.hip's pass, which moves the same bytes).
template <int kLayout>
constexpr int kPreMinQueryTiles = kLayout == 1 ? 6 : 12;

template <int kLayout, bool kBias>
int launch_sized(SdpaParams p, hipStream_t stream) {
  const int cus = compute_units();
  const int64_t heads = (int64_t)p.B * p.H, qtiles = (p.Lq + 511) / 512;
  const bool wide = heads * qtiles >= cus;
  const int64_t ntiles = (p.Lk + kTileKeys - 1) / kTileKeys;
  TilePlan pl;
  if (!plan_tiles(p.B, p.H, p.Lq, p.Lk, wide ? 512 : 128, kTileKeys, kD, wide ? cus : 0, pl)) return kErrDims;
  const size_t max_bytes = (size_t)heads * kMaxParts * sizeof(uint2);
  // Few queries leave CUs of the 128-query tiles idle: those are split along
  // the keys, where there is room for the ranges' rows.  (Below kMaxLaunchKeys
  // every workgroup looks through all of k and v first, whatever its range.)
  const TilePlan whole = pl;
  if (!wide && p.Lk >= kMaxLaunchKeys) {
    plan_key_ranges(p.B, p.H, p.Lq, p.Lk, 128, kTileKeys, kD, cus, pl);
    if (p.scratch != nullptr && pl.scratch_bytes + 256 + max_bytes > p.scratch_bytes) pl = whole;
  }
  const size_t part_bytes = (pl.scratch_bytes + 255) / 256 * 256;
  const size_t image_bytes = (size_t)heads * ntiles * kImageTileBytes<kBias>;
  bool image = wide && p.scratch == nullptr && qtiles >= kPreMinQueryTiles<kLayout> &&
               image_bytes <= kPreMaxImageBytes && heads * ntiles <= 0x7fffffff;
  uint2* maxes = nullptr;
  if (p.scratch != nullptr) {
    // behind the key-split partials, where the caller's scratch has room
    if (p.Lk >= kMaxLaunchKeys && part_bytes + max_bytes <= p.scratch_bytes)
      maxes = reinterpret_cast<uint2*>(reinterpret_cast<char*>(p.scratch) + part_bytes);
  } else if (image || p.Lk >= kMaxLaunchKeys) {
    // One buffer: partials, magnitudes, image.  Without it (allocation
    // failure, or a capture that would need it to grow) the workgroups look
    // through and split k and v themselves, with the same result.
    void* ws = image ? stream_workspace(stream, part_bytes + max_bytes + image_bytes, kSlotSdpaPartial) : nullptr;
    if (ws == nullptr) {
      image = false;
      if (p.Lk >= kMaxLaunchKeys) ws = stream_workspace(stream, part_bytes + max_bytes, kSlotSdpaPartial);
    }
    if (ws == nullptr && !wide) pl = whole;
    if (ws != nullptr) {
      p.scratch = static_cast<float*>(ws);
      p.scratch_bytes = pl.scratch_bytes;
      maxes = reinterpret_cast<uint2*>(static_cast<char*>(ws) + part_bytes);
    }
  }
  const SdpaArgs a = make_args(p);
  if (maxes != nullptr) {
    hipLaunchKernelGGL(sdpa_f16_max_kernel<kLayout>, dim3((unsigned)(heads * kMaxParts)), dim3(kMaxThreads), 0, stream,
                       a, maxes);
    if (hipGetLastError() != hipSuccess) return kErrLaunch;
  }
  if (image) {
    auto* img = reinterpret_cast<uintx4*>(reinterpret_cast<char*>(maxes) + max_bytes);
    hipLaunchKernelGGL((sdpa_f16_presplit_kernel<kLayout, kBias>), dim3((unsigned)(heads * ntiles)),
                       dim3(kPreThreads), 0, stream, a, maxes, img, (int)ntiles);
    if (hipGetLastError() != hipSuccess) return kErrLaunch;
    return launch_shape<0, kBias, 16, true>(p, stream, pl, maxes, img);
  }
  if (wide) return launch_shape<kLayout, kBias, 16, false>(p, stream, pl, maxes, nullptr);
  return launch_shape<kLayout, kBias, 4, false>(p, stream, pl, maxes, nullptr);
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
