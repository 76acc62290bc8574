// Arithmetic of the preparation of 16-bit activations, two values to a register
// (prep.hip's prep16_kernel, which says why): packing and the radix-4 butterflies.
#pragma once

#include "prep_device.h"

namespace convrot {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// A lane's rows of the constant matrices (row lane % 4 of each 4 x 4), applied
// to B = (x0, x1, y0, y1):
//   sum   x0 + y0, x1 + y1, x0 - y0, x1 - y1
//   id    x0, x1, y0, y1
//   minus -y0, -y1, y0, y1       plus  y0, y1, y0, y1
// and on a run (a, b, c, d) of digit 0:
//   t     t1 = a + b, t2 = a - b (0, 0)       last  -d, d, d, d
//   u     on (t1, t2, c, d): u0 = t1 + c, u1 = t1 - c, u2 = t2 + c, u3 = c - t2
// id with the +-d of minus, plus or last as the accumulator adds a stage's last
// term to all four sums at once.
struct Matrices {
  uint2 sum, id, minus, plus, t, last, u;
};

__device__ __forceinline__ Matrices matrices(int lane) {
  const uint32_t P0 = 0x3f80u, N0 = 0xbf80u, P1 = P0 << 16, N1 = N0 << 16;  // +-1 in the low / high half
  const int i = lane & 3;
  const auto row = [i](uint32_t a, uint32_t b, uint32_t c, uint32_t d) { return i == 0 ? a : i == 1 ? b : i == 2 ? c : d; };
  Matrices m;
  m.sum = make_uint2(row(P0, P1, P0, P1), row(P0, P1, N0, N1));
  m.id = make_uint2(row(P0, P1, 0u, 0u), row(0u, 0u, P0, P1));
  m.minus = make_uint2(0u, row(N0, N1, P0, P1));
  m.plus = make_uint2(0u, row(P0, P1, P0, P1));
  m.t = make_uint2(row(P0 | P1, P0 | N1, 0u, 0u), 0u);
  m.last = make_uint2(0u, row(N1, P1, P1, P1));
  m.u = make_uint2(row(P0, P0, P1, N1), row(P0, N0, P0, P0));
  return m;
}

__device__ __forceinline__ f32x4 mfma4(uint2 a, uint32_t x, uint32_t y, f32x4 c = (f32x4){0.f, 0.f, 0.f, 0.f}) {
  const uint2 b = make_uint2(x, y);
  return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
}

__device__ __forceinline__ f16x2 as_f16(uint32_t w) { return __builtin_bit_cast(f16x2, w); }
__device__ __forceinline__ uint32_t as_u32(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }

template <int DT>
__device__ __forceinline__ float pk_lo(uint32_t w) {
  if constexpr (DT == kBF16) return bf16_lo(w);
  else return (float)as_f16(w).x;
}
template <int DT>
__device__ __forceinline__ float pk_hi(uint32_t w) {
  if constexpr (DT == kBF16) return bf16_hi(w);
  else return (float)as_f16(w).y;
}
template <int DT>
__device__ __forceinline__ uint32_t pk_make(float lo, float hi) {
  if constexpr (DT == kBF16) return pack_bf16x2(lo, hi);
  else return pack_f16x2(lo, hi);
}

// One radix-4 along digit 0 on a packed run (a, b), (c, d); in radix4's order.
// EXACT: by radix4 itself, for values that may not be finite.
template <int DT, bool EXACT>
__device__ __forceinline__ void pk_stage_run(const Matrices& m, uint32_t& x, uint32_t& y) {
  if constexpr (EXACT) {
    float a = pk_lo<DT>(x), b = pk_hi<DT>(x), c = pk_lo<DT>(y), d = pk_hi<DT>(y);
    asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));  // float32 adds (a v_fma_mix negates a NaN)
    radix4<DT>(a, b, c, d);
    x = pk_make<DT>(a, b);
    y = pk_make<DT>(c, d);
  } else if constexpr (DT == kBF16) {
    const f32x4 d = mfma4(m.last, x, y), t = mfma4(m.t, x, y);
    const f32x4 u = mfma4(m.u, pack_bf16x2(t[0], t[1]), y);
    const f32x4 o = mfma4(m.id, pack_bf16x2(u[0], u[1]), pack_bf16x2(u[2], u[3]), d);
    x = pack_bf16x2(o[0], o[1]);
    y = pack_bf16x2(o[2], o[3]);
  } else {
    const f16x2 ab = as_f16(x), cd = as_f16(y);
    const f16x2 t = ab.xx + (f16x2){ab.y, -ab.y};
    const f16x2 u01 = t.xx + (f16x2){cd.x, -cd.x}, u23 = (f16x2){t.y, -t.y} + cd.xx;
    x = as_u32(u01 + (f16x2){-cd.y, cd.y});
    y = as_u32(u23 + cd.yy);
  }
}

// Two radix-4s side by side, the digit across four registers.
template <int DT, bool EXACT>
__device__ __forceinline__ void pk_stage_regs(const Matrices& m, uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) {
  if constexpr (EXACT) {
    float l[4] = {pk_lo<DT>(a), pk_lo<DT>(b), pk_lo<DT>(c), pk_lo<DT>(d)};
    float h[4] = {pk_hi<DT>(a), pk_hi<DT>(b), pk_hi<DT>(c), pk_hi<DT>(d)};
    asm volatile("" : "+v"(l[0]), "+v"(l[1]), "+v"(l[2]), "+v"(l[3]), "+v"(h[0]), "+v"(h[1]), "+v"(h[2]), "+v"(h[3]));
    radix4<DT>(l[0], l[1], l[2], l[3]);
    radix4<DT>(h[0], h[1], h[2], h[3]);
    a = pk_make<DT>(l[0], h[0]);
    b = pk_make<DT>(l[1], h[1]);
    c = pk_make<DT>(l[2], h[2]);
    d = pk_make<DT>(l[3], h[3]);
  } else if constexpr (DT == kBF16) {
    const f32x4 t = mfma4(m.sum, a, b), dm = mfma4(m.minus, c, d), dp = mfma4(m.plus, c, d);
    const f32x4 u01 = mfma4(m.sum, pack_bf16x2(t[0], t[1]), c), u23 = mfma4(m.sum, c, pack_bf16x2(t[2], t[3]));
    const f32x4 o01 = mfma4(m.id, pack_bf16x2(u01[0], u01[1]), pack_bf16x2(u01[2], u01[3]), dm);
    const f32x4 o23 = mfma4(m.id, pack_bf16x2(u23[0], u23[1]), pack_bf16x2(u23[2], u23[3]), dp);
    a = pack_bf16x2(o01[0], o01[1]);
    b = pack_bf16x2(o01[2], o01[3]);
    c = pack_bf16x2(o23[0], o23[1]);
    d = pack_bf16x2(o23[2], o23[3]);
  } else {
    const f16x2 va = as_f16(a), vb = as_f16(b), vc = as_f16(c), vd = as_f16(d);
    const f16x2 t1 = va + vb, t2 = va - vb;
    a = as_u32((t1 + vc) - vd);
    b = as_u32((t1 - vc) + vd);
    c = as_u32((t2 + vc) + vd);
    d = as_u32((vc - t2) + vd);
  }
}

}  // namespace convrot
