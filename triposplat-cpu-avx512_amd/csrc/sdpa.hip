// Exact online-softmax SDPA for gfx950 (head dim 64) on fp32 MFMA.  Serves the
// strict calls of fewer than kF16MinKeys keys; the others run on the fp16
// matrix cores (sdpa_f16.hip, 1.2-2.8x faster), whose workgroups take the same
// tile for keys that fp16 pairs do not hold.
//
// Reference semantics: scripts/native_sdpa_avx512_exact_q8t512.c:137-332 and
// the packed/BLHD variant scripts/native_sdpa_avx512_exact_q8t512_packed.c:3-158:
// out[q] = sum_j softmax_j(q.k_j * 0.125 + bias[j]) v_j, exact, with a
// running (max, sum) merged tile by tile; no Lq x Lk matrix, no pruning.
//
// The tile itself: sdpa_fp32.h.

#include "sdpa_fp32.h"

namespace tsplat {
namespace sdpa {
namespace {

template <int kLayout, bool kBias, int kWaves, int kBKV, bool kSplit>
__global__ __launch_bounds__(kWaves * 64) void sdpa_kernel(SdpaArgs a) {
  __shared__ __attribute__((aligned(16))) typename Fp32Lds<kLayout, kBKV>::K k;
  __shared__ __attribute__((aligned(16))) typename Fp32Lds<kLayout, kBKV>::V v;
  __shared__ __attribute__((aligned(16))) typename Fp32Lds<kLayout, kBKV>::Bias bias;
  sdpa_fp32_tile<kLayout, kBias, kWaves, kBKV, kSplit>(a, k, v, bias, threadIdx.x);
}

template <int kLayout, bool kBias, int kWaves, int kBKV, bool kSplit>
int launch_shape(const SdpaParams& p, hipStream_t stream) {
  return launch_tiles(make_args(p), p, kWaves * 32, kBKV, 0, stream, [&](dim3 grid, const SdpaArgs& a) {
    hipLaunchKernelGGL((sdpa_kernel<kLayout, kBias, kWaves, kBKV, kSplit>), grid, dim3(kWaves * 64), 0,
                       stream, a);
  });
}

// Grids too small to give every CU one 512-query workgroup use 4 waves.  A key
// bias runs the per-32-key-block softmax (kSplit).  (One key tile: nothing to
// split along the keys.)
template <int kLayout, bool kBias>
int launch_sized(const SdpaParams& p, hipStream_t stream) {
  const int64_t wide_tiles = (int64_t)p.B * p.H * ((p.Lq + 511) / 512);
  if (wide_tiles < compute_units()) return launch_shape<kLayout, kBias, 4, 64, false>(p, stream);
  return launch_shape<kLayout, kBias, 16, 64, kBias>(p, stream);
}

// Fewest keys for the fp16-product kernel (sdpa_f16.hip): one of its key
// tiles.  16 heads of 12294 queries over 65 keys take it 89 us, the kernel
// here 109; below a tile both are bound by the launch and the queries' loads,
// and a single key's value comes back exactly here.
constexpr int kF16MinKeys = 64;

}  // namespace

}  // namespace sdpa

// Shapes measured on MI355X at B=1, H=16, L=16384 (fp32 TFLOP/s): 16 waves x
// 64-key tiles 140 (unpacked) / 135 (packed) without a bias, the same tile
// split per 32-key block 134.7 with a key bias (unsplit 124: it spills), 16 x
// 128 split 130-134, 8 x 64 135-137, 4 x 64 121-123.  Storing the operand
// that arrives key-major for V (or dim-major for K) transposed in LDS, so all
// fragments are 128-bit reads, costs 2-4 %: the wider fragments push the
// 16-wave kernels into spills.
int launch_sdpa(const SdpaParams& p, hipStream_t stream) {
  using namespace sdpa;
  if (p.precision != kPrecisionFp32) return launch_sdpa_bf16(p, stream);
  if (p.Lk >= kF16MinKeys) return launch_sdpa_f16(p, stream);
  const bool bias = p.bias != nullptr;
  if (p.kv_packed) return bias ? launch_sized<1, true>(p, stream) : launch_sized<1, false>(p, stream);
  return bias ? launch_sized<0, true>(p, stream) : launch_sized<0, false>(p, stream);
}

}  // namespace tsplat
