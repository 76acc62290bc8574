// Exhaustive checks of device arithmetic that the preparation kernels rest on, for
// tests/test_gpu_device_checks.py: each entry point launches kernels that walk a
// whole range of inputs and count the disagreements in `result` (device memory,
// uint64: disagreements, missed non-finite results, the least input of either, inputs
// whose results were compared).
#include <stdint.h>

#include "prep16_device.h"

namespace convrot {
namespace {

constexpr unsigned kGrid = 4096, kBlock = 256;

__device__ void report(unsigned long long* result, int which, unsigned long long input) {
  atomicAdd(&result[which], 1ull);
  atomicMin(&result[2], input);
}

// rcp_newton against the float64 quotient rounded to float32 (53 >= 2 * 24 + 2
// bits: rounding twice changes nothing), every float32 in [1, 2^126).
__global__ __launch_bounds__(kBlock) void reciprocal_kernel(unsigned long long* result) {
  const uint32_t first = 0x3f800000u, last = 0x7e800000u;  // 1, 2^126
  unsigned long long compared = 0;
  for (uint32_t bits = first + blockIdx.x * kBlock + threadIdx.x; bits < last; bits += kGrid * kBlock) {
    ++compared;
    const float d = __uint_as_float(bits);
    if (__float_as_uint(rcp_newton(d)) != __float_as_uint((float)(1.0 / (double)d))) report(result, 0, bits);
  }
  atomicAdd(&result[3], compared);
}

// A 16-bit value with an exponent within +-32 (bf16) or +-16 (float16) of a's.
template <int DT>
__device__ uint32_t beside(uint32_t a, uint32_t h) {
  constexpr int kShift = DT == kBF16 ? 7 : 10, kTop = DT == kBF16 ? 254 : 30, kSpan = DT == kBF16 ? 64 : 32;
  int e = (int)((a >> kShift) & (DT == kBF16 ? 255u : 31u)) + (int)((h >> 20) % (unsigned)kSpan) - kSpan / 2;
  e = e < 0 ? 0 : e > kTop ? kTop : e;
  return (h & 0x8000u) | ((uint32_t)e << kShift) | (h & ((1u << kShift) - 1));
}

template <int DT>
__device__ bool finite16(uint32_t v) {
  const uint32_t inf = DT == kBF16 ? 0x7f80u : 0x7c00u;
  return (v & 0x7fffu) < inf;
}

// The packed butterfly (EXACT = false) against the float32 one on every pair of
// 16-bit values, the pair in two of the four places and zeros or values of like
// magnitude in the others.  Zeros may differ in sign.  Where the float32
// butterfly gives a non-finite result the packed one must give one too (its
// caller then repeats the row in float32), whatever the other results are.
template <int DT, bool REGS>
__global__ __launch_bounds__(kBlock) void butterfly_kernel(unsigned long long* result, int p0, int p1, int zeros) {
  const Matrices m = matrices(threadIdx.x & 63);
  const uint32_t thread = blockIdx.x * kBlock + threadIdx.x;
  unsigned long long compared = 0;
  for (uint32_t k = 0; k < (1u << 12); ++k) {
    const uint32_t pair = thread | (k << 20);
    uint32_t v[8];  // two butterflies' a, b, c, d
    uint32_t h = pair * 0x9e3779b9u + 0x7f4a7c15u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      h ^= h >> 15;
      h *= 0x2c1b3c6du;
      h ^= h >> 12;
      v[i] = zeros ? 0u : beside<DT>(pair & 0xffffu, h);
    }
    const uint32_t a = pair & 0xffffu, b = pair >> 16;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = i == p0 ? a : i == p1 ? b : v[i];
#pragma unroll
    for (int i = 4; i < 8; ++i) v[i] = i - 4 == p0 ? b : i - 4 == p1 ? a : v[i];
    uint32_t x[4], y[4];
    if constexpr (REGS) {  // the two side by side, across four registers
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = y[i] = v[i] | (v[4 + i] << 16);
      pk_stage_regs<DT, false>(m, x[0], x[1], x[2], x[3]);
      pk_stage_regs<DT, true>(m, y[0], y[1], y[2], y[3]);
    } else {  // each in a run of two registers
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = y[i] = v[2 * i] | (v[2 * i + 1] << 16);
      pk_stage_run<DT, false>(m, x[0], x[1]);
      pk_stage_run<DT, false>(m, x[2], x[3]);
      pk_stage_run<DT, true>(m, y[0], y[1]);
      pk_stage_run<DT, true>(m, y[2], y[3]);
    }
    bool same = true, packed_finite = true, exact_finite = true;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t g = (x[i >> 1] >> (16 * (i & 1))) & 0xffffu, w = (y[i >> 1] >> (16 * (i & 1))) & 0xffffu;
      same &= g == w || ((g | w) & 0x7fffu) == 0;
      packed_finite &= finite16<DT>(g);
      exact_finite &= finite16<DT>(w);
    }
    compared += exact_finite;
    if (exact_finite && !same) report(result, 0, pair);
    if (!exact_finite && packed_finite) report(result, 1, pair);
  }
  atomicAdd(&result[3], compared);
}

template <int DT, bool REGS>
hipError_t butterflies(unsigned long long* result, hipStream_t stream) {
  for (int p0 = 0; p0 < 3; ++p0)
    for (int p1 = p0 + 1; p1 < 4; ++p1)
      for (int zeros = 0; zeros < 2; ++zeros) {
        hipLaunchKernelGGL((butterfly_kernel<DT, REGS>), dim3(kGrid), dim3(kBlock), 0, stream, result, p0, p1, zeros);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
      }
  return hipSuccess;
}

}  // namespace
}  // namespace convrot

extern "C" int check_reciprocal(unsigned long long* result, void* stream) {
  hipLaunchKernelGGL(convrot::reciprocal_kernel, dim3(convrot::kGrid), dim3(convrot::kBlock), 0, (hipStream_t)stream,
                     result);
  return (int)hipGetLastError();
}

// bf16: 1, else float16; regs: pk_stage_regs, else pk_stage_run.
extern "C" int check_butterflies(int bf16, int regs, unsigned long long* result, void* stream) {
  using namespace convrot;
  const hipStream_t s = (hipStream_t)stream;
  return (int)(bf16 ? (regs ? butterflies<kBF16, true>(result, s) : butterflies<kBF16, false>(result, s))
                    : (regs ? butterflies<kF16, true>(result, s) : butterflies<kF16, false>(result, s)));
}
