// bf16-weight linear support for gfx950 (the products themselves: skinny_linear.hip and
// fused_linear.hip for few rows, big_bf16.hip for more, or for large weights; a model's
// forwards go by their rows, the per-op calls by tiles, K and weights, bf16_linear_into):
// y = bf16(x) @ W^T with fp32 accumulation, rounded to bf16 like the reference's
// bf16 matmul output (backends/mlx_ops.py:122-125).
//
// Device weight layout (produced once at upload from row-major W[N][K]):
//   wb[((nt*KC + kc)*64 + l)*8 + e] = W[32*nt + (l&31)][16*kc + 8*(l>>5) + e],  KC = K/16
// one n-tile x 16-k chunk is a contiguous 1 KiB (one 16-byte load per lane).
// The activation is ACT_BF16 (natural order).
#include "common.h"
#include "launch.h"

extern "C" __global__ void bf16_repack_kernel(const uint16_t* __restrict__ w,
                                              uint16_t* __restrict__ wb, int N, int K) {
  const int KC = K >> 4;
  const int64_t total = (int64_t)N * K / 8;  // 16-byte chunks
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t l = i & 63;
    const int64_t tk = i >> 6;  // nt*KC + kc
    const int64_t nt = tk / KC, kc = tk % KC;
    const int64_t n = 32 * nt + (l & 31);
    const int64_t k = 16 * kc + 8 * (l >> 5);
    *(u32x4*)(wb + i * 8) = *(const u32x4*)(w + n * K + k);
  }
}

namespace drt {

void bf16_repack(const uint16_t* w, int N, int K, uint16_t* wb, hipStream_t s) {
  require(N % 32 == 0 && K % 16 == 0, "bf16 linear needs N % 32 == 0 and K % 16 == 0");
  const int64_t work = (int64_t)N * K / 8;
  const int blocks = (int)std::min<int64_t>((work + 255) / 256, 65536);
  hipLaunchKernelGGL(bf16_repack_kernel, dim3(blocks), dim3(256), 0, s, w, wb, N, K);
  DRT_HIP(hipGetLastError());
}

}  // namespace drt

// ---- small fp32 <-> bf16 helpers used by the per-op entry points ----
// eight values per thread; the last n % 8 one by one
extern "C" __global__ __launch_bounds__(256) void to_bf16_kernel(const float* __restrict__ x,
                                                                 uint16_t* __restrict__ o,
                                                                 int64_t n) {
  const int64_t i = (blockIdx.x * (int64_t)256 + threadIdx.x) * 8;
  if (i + 8 <= n) {
    const f32x4 a = *(const f32x4_e*)(x + i), b = *(const f32x4_e*)(x + i + 4);
    uint16_t h[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h[e] = float_to_bf16_bits(a[e]);
      h[4 + e] = float_to_bf16_bits(b[e]);
    }
    *(u32x4_e*)(o + i) = __builtin_bit_cast(u32x4, h);
  } else {
    for (int64_t j = i; j < n; ++j) o[j] = float_to_bf16_bits(x[j]);
  }
}

namespace drt {

void to_bf16(const float* x, uint16_t* o, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(to_bf16_kernel, dim3((unsigned)((n + 2047) / 2048)), dim3(256), 0, s, x, o, n);
  DRT_HIP(hipGetLastError());
}

}  // namespace drt
