// Device pieces of the ConvRot preparation shared by the preparation kernel
// (prep.hip) and the few-row linear (linear_rows.hip): the butterfly with its
// per-op rounding, the lane <-> feature layout of a wave's 1024-feature block
// and its LDS exchanges, row loads, the row scale, the code of a ratio and the
// GELU producer's tanh GELU.
// The layout is described in prep.hip.
#pragma once

#include "convrot_device.h"

namespace convrot {

constexpr int kRegionFloats = 1280;  // per wave: 1024 features + 1/4 padding

// One radix-4 butterfly with a dtype rounding after every add (core.py:89-91):
//   a+b+c-d, a+b-c+d, a-b+c+d, -a+b+c+d, each evaluated left to right.
// rnd(-a+b) == -rnd(a-b) exactly, so the fourth output reuses a-b.
template <int DT>
__device__ __forceinline__ void radix4(float& a, float& b, float& c, float& d) {
  const float t1 = rnd<DT>(a + b);
  const float t2 = rnd<DT>(a - b);
  const float u0 = rnd<DT>(t1 + c);
  const float u1 = rnd<DT>(t1 - c);
  const float u2 = rnd<DT>(t2 + c);
  const float u3 = rnd<DT>(c - t2);
  a = rnd<DT>(u0 - d);
  b = rnd<DT>(u1 + d);
  c = rnd<DT>(u2 + d);
  d = rnd<DT>(u3 + d);
}

// Stage along d0 (register slots 4r .. 4r+3).
template <int DT>
__device__ __forceinline__ void stage_lo(float (&v)[16]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) radix4<DT>(v[4 * r], v[4 * r + 1], v[4 * r + 2], v[4 * r + 3]);
}

// Stage along the digit held in register-slot bits 2-3.
template <int DT>
__device__ __forceinline__ void stage_hi(float (&v)[16]) {
#pragma unroll
  for (int d0 = 0; d0 < 4; ++d0) radix4<DT>(v[d0], v[4 + d0], v[8 + d0], v[12 + d0]);
}

// Index inside the group of register run `run` (slots 4*run .. 4*run+3,
// digit d0 = 0..3) for a lane at position p of its group during phase PH.
// Phase 1: (d1, d0) in registers, the lane owns features 16p .. 16p+15.
// Phase PH >= 2: (d_PH, d0) in registers, the remaining digits
// d1..d_{S-1} (skipping d_PH) come from p, lowest first.
template <int S, int PH>
__device__ __forceinline__ int run_index(int p, int run) {
  if constexpr (PH == 1) {
    return 16 * p + 4 * run;
  } else {
    int i = 0, pp = p, w = 4;
#pragma unroll
    for (int t = 1; t < S; ++t, w *= 4) {
      int digit;
      if (t == PH) {
        digit = run;
      } else {
        digit = pp & 3;
        pp >>= 2;
      }
      i += digit * w;
    }
    return i;
  }
}

// Padded LDS offset (floats): 4 floats of padding after every 16 features,
// which keeps the phase-1 writes and the phase-2 reads bank-conflict free.
__device__ __forceinline__ int lds_off(int i) { return i + 4 * (i >> 4); }

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Move the lane's 16 values from the phase PH-1 layout to the phase PH layout
// through the wave's LDS region and run stage PH.
template <int DT, int S, int PH>
__device__ __forceinline__ void exchange_and_stage(float (&v)[16], float* region, int p) {
#pragma unroll
  for (int run = 0; run < 4; ++run) {
    const int i = run_index<S, PH - 1>(p, run);
    *(float4*)(region + lds_off(i)) = make_float4(v[4 * run], v[4 * run + 1], v[4 * run + 2], v[4 * run + 3]);
  }
  wave_lds_fence();
#pragma unroll
  for (int run = 0; run < 4; ++run) {
    const int i = run_index<S, PH>(p, run);
    const float4 t = *(const float4*)(region + lds_off(i));
    v[4 * run] = t.x;
    v[4 * run + 1] = t.y;
    v[4 * run + 2] = t.z;
    v[4 * run + 3] = t.w;
  }
  wave_lds_fence();
  stage_hi<DT>(v);
}

template <int DT, int S>
__device__ __forceinline__ void rotate16(float (&v)[16], float* region, int p) {
  if constexpr (S >= 1) stage_lo<DT>(v);
  if constexpr (S >= 2) stage_hi<DT>(v);
  if constexpr (S >= 3) exchange_and_stage<DT, S, 2>(v, region, p);
  if constexpr (S >= 4) exchange_and_stage<DT, S, 3>(v, region, p);
  if constexpr (S >= 5) exchange_and_stage<DT, S, 4>(v, region, p);
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// 16 consecutive elements at byte `off` of the row's buffer (16-byte loads);
// offsets at or beyond the row's end read as zero (buffer range check).
template <int DT>
__device__ __forceinline__ void load16(__amdgpu_buffer_rsrc_t row, uint32_t off, float (&v)[16]) {
  if constexpr (DT == kF32) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(row, (int)(off + 16 * q), 0, 0);
      // __uint_as_float, not __builtin_bit_cast: this compiler bit_casts a
      // vector-element operand from element 0's storage
      v[4 * q] = __uint_as_float(t.x);
      v[4 * q + 1] = __uint_as_float(t.y);
      v[4 * q + 2] = __uint_as_float(t.z);
      v[4 * q + 3] = __uint_as_float(t.w);
    }
  } else {
    const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(row, (int)off, 0, 0);
    const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(row, (int)(off + 16), 0, 0);
    const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if constexpr (DT == kBF16) {
        v[2 * q] = bf16_lo(w[q]);
        v[2 * q + 1] = bf16_hi(w[q]);
      } else {
        typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
        const f16x2 h = __builtin_bit_cast(f16x2, w[q]);
        v[2 * q] = (float)h[0];
        v[2 * q + 1] = (float)h[1];
      }
    }
  }
}

// max(m, |a|, |b|) in one v_max3_f32 with |.| source modifiers (m >= 0).  As
// C++ the compiler inserts canonicalizing moves and separate abs masks.
__device__ __forceinline__ float absmax3(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(a), "v"(b), "v"(m));
  return r;
}

// Maximum over the wave of a non-negative float (bit patterns of non-negative
// floats order like unsigned integers): DPP quad swaps and row mirrors leave
// every lane of a 16-lane row with the row maximum, then four readlanes.
__device__ __forceinline__ float wave_max_nonneg(float x) {
  uint32_t v = __builtin_bit_cast(uint32_t, x);
  v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
  v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
  v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, true));  // row_half_mirror
  v = max(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xF, 0xF, true));  // row_mirror
  const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
  const uint32_t r1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
  const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 32);
  const uint32_t r3 = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
  return __builtin_bit_cast(float, max(max(r0, r1), max(r2, r3)));
}

// Signed code in [-7, 7] of a ratio: clamp, then round half to even by adding
// 1.5 * 2^23 (the float add rounds to the nearest integer, ties to even, and
// leaves the integer in the low mantissa bits in two's complement).
__device__ __forceinline__ uint32_t code_bits(float ratio) {
  const float c = __builtin_amdgcn_fmed3f(ratio, -7.0f, 7.0f);
  return __builtin_bit_cast(uint32_t, c + 12582912.0f);
}

// Four codes (low bytes of code_bits) gathered into one int8x4 word.
__device__ __forceinline__ uint32_t gather_bytes(uint32_t b0, uint32_t b1, uint32_t b2, uint32_t b3) {
  const uint32_t lo = __builtin_amdgcn_perm(b1, b0, 0x0c0c0400u);
  const uint32_t hi = __builtin_amdgcn_perm(b3, b2, 0x04000c0cu);
  return lo | hi;
}

// Row scale (core.py:154-156) of the row's absmax, and for bf16 the factor
// that turns an unnormalized rotated value into its ratio.
template <int DT>
struct RowScale {
  float scale, inv;
};

template <int DT>
__device__ __forceinline__ RowScale<DT> row_scale(float amax, float norm) {
  if constexpr (DT == kBF16) amax *= norm;  // x / sqrt(G) is exact in bf16
  float floor_v;
  if constexpr (DT == kBF16) floor_v = __builtin_bit_cast(float, 0x2edc0000u);  // bf16(1e-10)
  else if constexpr (DT == kF16) floor_v = 0.0f;                                // f16(1e-10) underflows
  else floor_v = 1e-10f;
  RowScale<DT> r;
  r.scale = rnd<DT>(fmaxf(amax, floor_v) / 7.0f);
  r.inv = DT == kBF16 ? (1.0f / r.scale) * norm : 0.0f;
  return r;
}

// Ratio of a rotated value (bf16: unnormalized, else normalized) to the row scale.
template <int DT>
__device__ __forceinline__ float code_ratio(float v, const RowScale<DT>& s) {
  if constexpr (DT == kBF16) return round_bf16(v * s.inv);
  else return s.scale > 0.0f ? rnd<DT>(v / s.scale) : 0.0f;  // 0/0 on an all-zero f16 row
}

// 1 / d, correctly rounded, for d in [1, 2^126): one Newton step from v_rcp_f32.
// The step alone would leave a start value one ulp below at the all-ones
// significand wrong; the hardware's is not.  Every float32 of the range is
// compared with the float64 quotient in tests/test_gpu_device_checks.py.
__device__ __forceinline__ float rcp_newton(float d) {
  const float y = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(__builtin_fmaf(-d, y, 1.0f), y, y);
}

// tanh GELU of the fused GELU producer, float32, in this fixed sequence (the
// same IEEE operations, in the same order, as the CPU oracle's gelu_tanh32):
//   x3 = (x * x) * x;  u = kBeta * fma(kKappa, x3, x)
//   q = 2 / (exp(2|u|) + 1)  (0 where 2|u| > 88 or u is NaN)
//   1 + tanh(u) = u >= 0 ? 2 - q : q  (no cancellation on either side)
//   y = (0.5 * x) * (1 + tanh(u))
// with exp(z) = 2^n e^r, n = rint(z log2 e), r = z - n ln2 by two fmas
// (Cody-Waite), e^r by its degree-7 Taylor polynomial (Horner, fma).
//
// Cheaper forms of the same values:
//  * rint by adding and subtracting 1.5 * 2^23 (|z log2 e| < 2^7), which leaves
//    n in the low bits of the sum: 2^n p is an integer add to p's exponent
//    (p in [0.7, 1.42], n <= 127: no overflow, no denormal);
//  * 2 / s as the reciprocal of s / 2 (exact halving), by rcp_newton.
// 35 VALU operations with a conversion and a division in them became 29.
__device__ __forceinline__ float gelu_tanh32(float x) {
  const float x3 = (x * x) * x;
  const float u = 0x1.988454p-1f * __builtin_fmaf(0x1.6e4e26p-5f, x3, x);
  const float z = fabsf(u) + fabsf(u);
  const float t = z * 0x1.715476p+0f + 12582912.0f;
  const float n = t - 12582912.0f;
  float r = __builtin_fmaf(-n, 0x1.62e4p-1f, z);
  r = __builtin_fmaf(-n, 0x1.7f7d1cp-20f, r);
  float p = 0x1.a01a02p-13f;
  p = __builtin_fmaf(p, r, 0x1.6c16c2p-10f);
  p = __builtin_fmaf(p, r, 0x1.111112p-7f);
  p = __builtin_fmaf(p, r, 0x1.555556p-5f);
  p = __builtin_fmaf(p, r, 0x1.555556p-3f);
  p = __builtin_fmaf(p, r, 0x1p-1f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  const float e = __uint_as_float(__float_as_uint(p) + (__float_as_uint(t) << 23));
  const float d = 0.5f * (e + 1.0f);
  const float q = z <= 88.0f ? rcp_newton(d) : 0.0f;
  const float onept = u >= 0.0f ? 2.0f - q : q;
  return (0.5f * x) * onept;
}

}  // namespace convrot
