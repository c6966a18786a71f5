// The decoder's passes between its matrix products (gfx950), 16-bit storage, fp32
// arithmetic: residual add with the RMSNorm that reads it, and the gated MLP's
// SiLU(gate) * up.
//
// Both are bound by HBM (prefill) or by the launch (decode): as tensor code each
// was two kernels and the second read back what the first had just written.
// MI355X, 2 x 512 prompt tokens, bf16: SiLU and product over 1024 x 14336 22.4 + 18.1
// -> 19.4 us (4.5 TB/s), add and norm over 1024 x 4096 5.8 + 8.9 -> 8.7 us (3.9
// TB/s); that prefill call 1392 -> 1345 us over two layers; a decode step of 128
// candidates through 32 layers 7.11 -> 6.62 ms.
// Roundings are the tensor code's: the sum to the storage type before the norm
// reads it, SiLU to the storage type before the product.

#include <math.h>

#include "common.h"

namespace be {

typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

template <typename T>
__device__ __forceinline__ void load8(const T* p, float (&v)[8]) {
  const u16x8 u = *reinterpret_cast<const u16x8*>(p);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint16_t b = u[e];
    v[e] = to_f32(__builtin_bit_cast(T, b));
  }
}
template <typename T>
__device__ __forceinline__ void store8(T* p, const float (&v)[8]) {
  u16x8 u;
#pragma unroll
  for (int e = 0; e < 8; ++e) u[e] = __builtin_bit_cast(uint16_t, from_f32<T>(v[e]));
  *reinterpret_cast<u16x8*>(p) = u;
}

constexpr int kNormChunks = 4;   // 8-element chunks a thread holds: rows of up to 8192 (longer ones keep the tensor code)

// One workgroup per row: x + delta (to sum, rounded), then sum * rsqrt(mean(sum^2)
// + eps) * w (to out).  The row stays in registers between the two.
template <typename T>
__global__ __launch_bounds__(256) void add_rms_norm_kernel(const T* x, const T* delta, const T* w, T* sum, T* out, int n,
                                                          float eps) {
  __shared__ float part[4];
  const int64_t base = (int64_t)blockIdx.x * n;
  const int nc = n / 8;
  float v[kNormChunks][8], d[8], s = 0.f;
#pragma unroll
  for (int u = 0; u < kNormChunks; ++u) {
    const int c = u * 256 + threadIdx.x;
    if (c >= nc) continue;
    load8(x + base + c * 8, v[u]);
    load8(delta + base + c * 8, d);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[u][e] = to_f32(from_f32<T>(v[u][e] + d[e]));
      s = fmaf(v[u][e], v[u][e], s);
    }
    store8(sum + base + c * 8, v[u]);
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  const float r = rsqrtf((part[0] + part[1] + part[2] + part[3]) / (float)n + eps);
#pragma unroll
  for (int u = 0; u < kNormChunks; ++u) {
    const int c = u * 256 + threadIdx.x;
    if (c >= nc) continue;
    load8(w + c * 8, d);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[u][e] = v[u][e] * r * d[e];
    store8(out + base + c * 8, v[u]);
  }
}

// One thread per 8 columns: rows of [gate | up], each n wide.
template <typename T>
__global__ __launch_bounds__(256) void silu_mul_kernel(const T* gu, T* out, int n) {
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c * 8 >= n) return;
  const T* gp = gu + (int64_t)blockIdx.x * 2 * n + c * 8;
  float g[8], u[8];
  load8(gp, g);
  load8(gp + n, u);
#pragma unroll
  for (int e = 0; e < 8; ++e) g[e] = to_f32(from_f32<T>(g[e] / (1.f + expf(-g[e])))) * u[e];
  store8(out + (int64_t)blockIdx.x * n + c * 8, g);
}

}  // namespace be

extern "C" int be_add_rms_norm(const void* x, const void* delta, const void* weight, void* sum, void* out, int dtype,
                               int rows, int n, float eps, void* stream) {
  BE_REQUIRE(rows >= 0, "rows must be >= 0");
  if (rows == 0) return BE_OK;
  BE_REQUIRE(x && delta && weight && sum && out, "null pointer");
  BE_REQUIRE(dtype == BE_F16 || dtype == BE_BF16, "add_rms_norm supports fp16 / bf16 storage");
  BE_REQUIRE(n > 0 && n % 8 == 0 && n <= be::kNormChunks * 256 * 8, "row length %d: a multiple of 8 up to %d", n,
             be::kNormChunks * 256 * 8);
  BE_REQUIRE((((uintptr_t)x | (uintptr_t)delta | (uintptr_t)weight | (uintptr_t)sum | (uintptr_t)out) & 15) == 0,
             "operands must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == BE_BF16)
    be::add_rms_norm_kernel<be::bf16_t><<<rows, 256, 0, st>>>((const be::bf16_t*)x, (const be::bf16_t*)delta,
                                                             (const be::bf16_t*)weight, (be::bf16_t*)sum,
                                                             (be::bf16_t*)out, n, eps);
  else
    be::add_rms_norm_kernel<be::f16_t><<<rows, 256, 0, st>>>((const be::f16_t*)x, (const be::f16_t*)delta,
                                                            (const be::f16_t*)weight, (be::f16_t*)sum, (be::f16_t*)out,
                                                            n, eps);
  BE_HIP_CHECK(hipGetLastError());
  return BE_OK;
}

extern "C" int be_silu_mul(const void* gate_up, void* out, int dtype, int rows, int n, void* stream) {
  BE_REQUIRE(rows >= 0, "rows must be >= 0");
  if (rows == 0) return BE_OK;
  BE_REQUIRE(gate_up && out, "null pointer");
  BE_REQUIRE(dtype == BE_F16 || dtype == BE_BF16, "silu_mul supports fp16 / bf16 storage");
  BE_REQUIRE(n > 0 && n % 8 == 0 && n <= (1 << 24), "row length %d: a multiple of 8", n);
  BE_REQUIRE((((uintptr_t)gate_up | (uintptr_t)out) & 15) == 0, "operands must be 16-byte aligned");
  const dim3 blocks((unsigned)rows, (unsigned)((n / 8 + 255) / 256));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == BE_BF16)
    be::silu_mul_kernel<be::bf16_t><<<blocks, 256, 0, st>>>((const be::bf16_t*)gate_up, (be::bf16_t*)out, n);
  else
    be::silu_mul_kernel<be::f16_t><<<blocks, 256, 0, st>>>((const be::f16_t*)gate_up, (be::f16_t*)out, n);
  BE_HIP_CHECK(hipGetLastError());
  return BE_OK;
}
