// Fused ConvRot activation preparation for gfx950: normalized regular-Hadamard
// rotation + rowwise absmax + symmetric A4 quantization + packing, one pass.
//
// Replaces the reference's two-pass Metal kernels (one threadgroup per row,
// a barrier per butterfly stage, the row read and rotated twice:
// /root/reference/src/convrot_mlx/core.py:205-304 packed, :307-327 int8,
// :330-370 rotate-only) and reproduces the eager contract bit for bit
// (regular_hadamard core.py:64-94, quantize_signed_int4_rowwise :149-158).
//
// Data layout and work split
//  * One workgroup per row, W waves per row, NI iterations per wave.  In one
//    iteration a wave owns 1024 consecutive features: lane l holds the 16
//    consecutive features [16l, 16l+16) in registers (two 16-byte loads).
//  * A feature index inside a group of G = 4^S is written in base 4 as
//    (d_{S-1} ... d1 d0).  Stage s of the butterfly runs along digit d_s
//    (stride 4^s).  Phase 1 keeps (d1, d0) in registers and runs stages 0
//    and 1 without any data movement; every later stage s keeps (d_s, d0) in
//    registers and is reached through one LDS exchange (four 16-byte writes,
//    four 16-byte reads per lane, wave-private region, no workgroup barrier).
//  * The rotated row stays in registers (NI*16 floats per lane) until the
//    row absmax is known -- one HBM read of x instead of the reference's two.
//  * bf16 rounding after every add costs one v_cvt_pk_bf16_f32 (see
//    round_bf16); the division by scale is a multiply by a correctly rounded
//    reciprocal, which is exact for bf16 operands (r/scale can never lie
//    within 2^-16.8 of a bf16 rounding midpoint, so an error below 2^-23
//    cannot change the rounded ratio).  f16/f32 inputs use a true division.
#include <stdlib.h>

#include "convrot_device.h"
#include "convrot_launch.h"
#include "prep16_device.h"

namespace convrot {
namespace {

constexpr int kMaxWaves = 16;
constexpr int kMaxBlocks = 64;  // 1024-feature blocks of the longest row (65536 features)

// Four codes packed as four nibbles, low nibble = lowest feature (core.py:101-105).
__device__ __forceinline__ uint32_t gather_nibbles(uint32_t b0, uint32_t b1, uint32_t b2, uint32_t b3) {
  const uint32_t bytes = gather_bytes(b0, b1, b2, b3) & 0x0f0f0f0fu;
  const uint32_t pairs = bytes | (bytes >> 4);  // byte0 = n0|n1<<4, byte2 = n2|n3<<4
  return __builtin_amdgcn_perm(0u, pairs, 0x0c0c0200u);
}

// FP6 operand codes.  A code v is stored as the e2m3 encoding of v/8: for
// |v| <= 7 that is the subnormal with mantissa |v| (sign bit 5, exponent bits
// 4..3 zero), so the field is the sign-magnitude form of v; the GEMM's MFMA
// scales both operands by 2^3 and sums the exact products v*w.  Zero codes
// are +0.
//
// Four A4 codes as FP6 fields, packed as a 24-bit field (code j at bits
// 6j..6j+5).  m0..m3 are code_bits of the ratios' magnitudes (low byte |q| in
// 0..7) and r0..r3 the ratios, whose signs pick the negative codes.
__device__ __forceinline__ uint32_t fp6_piece(uint32_t m0, uint32_t m1, uint32_t m2, uint32_t m3, float r0, float r1,
                                              float r2, float r3) {
  const uint32_t mag = gather_bytes(m0, m1, m2, m3);
  const uint32_t pos = mag;                                                    // 0 .. 7
  const uint32_t neg = __builtin_amdgcn_perm(0x27262524u, 0x23222100u, mag);  // 0, -1 .. -7
  // selector 9 / 11: the sign bit of the second / first operand, over the byte
  const uint32_t sm = __builtin_amdgcn_perm(__float_as_uint(r1), __float_as_uint(r0), 0x0c0c0b09u) |
                      __builtin_amdgcn_perm(__float_as_uint(r3), __float_as_uint(r2), 0x0b090c0cu);
  const uint32_t codes = (neg & sm) | (pos & ~sm);
  const uint32_t y = (codes & 0x003f003fu) | ((codes >> 2) & 0x0fc00fc0u);  // 12-bit pairs at bits 0, 16
  return (y & 0xfffu) | ((y >> 4) & 0xfff000u);
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x32 __attribute__((ext_vector_type(32)));
typedef int i32x6 __attribute__((ext_vector_type(6)));

// A pair of bf16 ratios with the sign cleared on each negative one of
// magnitude at most 0.5 (bits 0x3f00), i.e. on each ratio whose code
// rint(ratio) is 0: bit 15 of h + 0x40ff (per half, mod 2^16) is set for
// exactly those negative halves (and for positive halves above 0.5, whose
// sign bit is already clear).
__device__ __forceinline__ uint32_t zero_code_sign_fix(uint32_t h) {
  const u16x2 s = __builtin_bit_cast(u16x2, h) + (u16x2){0x40ff, 0x40ff};
  return h & ~(__builtin_bit_cast(uint32_t, s) & 0x80008000u);
}

// FP6 fields of 16 bf16 ratios (8 packed pairs, lowest feature first), whose
// magnitudes are at most 7.04 (as every bf16 ratio is, the scale being
// bf16(absmax / 7)): v_cvt_scalef32_pk32_fp6_bf16 divides by the scale 8 and
// rounds to the e2m3 grid of eighths with ties to even, so field i is
// rint(ratio_i) / 8 -- the code with its sign -- and fields 0..15 fill the
// first 96 bits (the other 16 inputs are zero).
__device__ __forceinline__ void fp6_fields16(const uint32_t (&hp)[8], uint32_t& d0, uint32_t& d1, uint32_t& d2) {
  const u32x16 in = {hp[0], hp[1], hp[2], hp[3], hp[4], hp[5], hp[6], hp[7], 0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
  const i32x6 f = __builtin_amdgcn_cvt_scalef32_pk32_fp6_bf16(__builtin_bit_cast(bf16x32, in), 8.0f);
  d0 = (uint32_t)f[0];
  d1 = (uint32_t)f[1];
  d2 = (uint32_t)f[2];
}

// Sum of a float64 over the wave (butterfly: every lane ends with the total,
// added in the same order in every lane).
__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
  return v;
}

// Producers: what the preparation reads as its input rows.
enum Producer : int {
  kProPlain = CONVROT_PRODUCER_PLAIN,        // x
  kProModulate = CONVROT_PRODUCER_MODULATE,  // (1 + scale) * layer_norm(x) + shift
  kProGelu = CONVROT_PRODUCER_GELU,          // [head | gelu_tanh(x)], each with its own row stride
};

// Arguments of the producers beyond x (unused fields are ignored).
struct ProducerArgs {
  const void* shift;  // kProModulate: [vectors, K] shift and scale rows
  const void* scale;
  int rows_per_vector;
  float eps;
  const void* head;     // kProGelu: [rows, head_features] at head_stride elements per row
  int head_features;    //   (0: no head), a multiple of 16
  int64_t head_stride;
  int64_t x_stride;     // kProGelu: elements per row of x (x has K - head_features features)
};

// PRO = kProModulate: the fused modulated producer.  Each row is first replaced by
//   y = rb(rb(rb(1 + scale) * rb((x - mean) * rstd)) + shift)
// (LayerNorm without affine parameters, then the adaLN modulation with a
// dtype rounding after every op), with the shift / scale row
// v = row / rows_per_vector.  Then the ConvRot preparation runs on y as it
// would on x.  The moments are float64 sums in a fixed order that does not
// depend on the launch plan: lane l of 1024-feature block b adds features
// 16l .. 16l+15 in order, the 64 lanes are combined by the xor butterfly of
// wave_sum_f64, and the block sums are added in block order.
//
// PRO = kProGelu: the fused GELU producer.  Feature f of a row is head[f] for
// f < head_features and rb(gelu_tanh32(x[f - head_features])) after that;
// padding past K reads zeros, and gelu(0) = 0.
template <int DT, int S, int NI, int MODE, int PRO>
__global__ __launch_bounds__(1024) void prep_kernel(const void* __restrict__ x, void* __restrict__ out,
                                                     float* __restrict__ scales, int K, ProducerArgs pa) {
  constexpr bool PRE = PRO == kProModulate;
  extern __shared__ float lds[];
  __shared__ float wave_max[kMaxWaves];
  __shared__ double block_moments[PRE ? kMaxBlocks : 1][2];

  constexpr int G = (S == 0) ? 1 : (1 << (2 * S));
  constexpr int LG = (S >= 3) ? (G / 16) : 1;        // lanes per group
  constexpr int GS = (S >= 3) ? G : 16;               // features per lane group
  constexpr bool kImplicitNorm = (DT == kBF16);      // x/sqrt(G) is exact in bf16
  constexpr float kNorm = (S == 0) ? 1.0f : 1.0f / (float)(1 << S);

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int nwaves = blockDim.x >> 6;
  int64_t row = blockIdx.x;
  if constexpr (MODE == CONVROT_PREP_FP6 || MODE == CONVROT_PREP_INT8_BLOCKED) {
    // Workgroups go round-robin to the 8 XCDs.  The 16 rows of a block
    // share its cache lines, so each XCD takes runs of consecutive rows (a
    // multiple of 16 each) and its L2 merges the rows' pieces of a line.
    const int64_t run = ((int64_t)gridDim.x / (8 * 16)) * 16;
    if (row < 8 * run) row = (row & 7) * run + (row >> 3);
  }
  const int chunks = K >> 4;
  constexpr int kEsize = DT == kF32 ? 4 : 2;
  const __amdgpu_buffer_rsrc_t xrow = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const char*)x + row * (PRO == kProGelu ? pa.x_stride : (int64_t)K) * kEsize), (short)0,
      (PRO == kProGelu ? K - pa.head_features : K) * kEsize, 0x00020000);
  const __amdgpu_buffer_rsrc_t hrow = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(PRO == kProGelu && pa.head_features ? (const char*)pa.head + row * pa.head_stride * kEsize
                                                  : (const char*)x),
      (short)0, PRO == kProGelu ? pa.head_features * kEsize : 0, 0x00020000);
  float* region = lds + wave * kRegionFloats + (lane / LG) * (G + G / 4);
  const int p = lane % LG;

  float keep[NI][16];
  float amax = 0.0f;

  if constexpr (PRE) {
    const int real_blocks = (chunks + 63) >> 6;
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int block = wave * NI + it;
      load16<DT>(xrow, (uint32_t)(block * 64 + lane) * (16u * kEsize), keep[it]);  // past the row end: zeros
      double b1 = 0.0, b2 = 0.0;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const double d = (double)keep[it][j];
        b1 += d;
        b2 += d * d;
      }
      b1 = wave_sum_f64(b1);
      b2 = wave_sum_f64(b2);
      if (lane == 0 && block < real_blocks) {
        block_moments[block][0] = b1;
        block_moments[block][1] = b2;
      }
    }
    __syncthreads();
    double s1 = 0.0, s2 = 0.0;
    for (int b = 0; b < real_blocks; ++b) {
      s1 += block_moments[b][0];
      s2 += block_moments[b][1];
    }
    const double m64 = s1 / (double)K;
    double var = s2 / (double)K - m64 * m64;
    var = var > 0.0 ? var : 0.0;
    const float mean = (float)m64;
    const float rstd = (float)(1.0 / sqrt(var + (double)pa.eps));
    const int64_t vrow = row / pa.rows_per_vector;
    const __amdgpu_buffer_rsrc_t shrow = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const char*)pa.shift + vrow * K * kEsize), (short)0, K * kEsize, 0x00020000);
    const __amdgpu_buffer_rsrc_t scrow = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const char*)pa.scale + vrow * K * kEsize), (short)0, K * kEsize, 0x00020000);
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int chunk = (wave * NI + it) * 64 + lane;
      if (chunk >= chunks) continue;  // padding stays zero (whole groups lie past K)
      float sh[16], sc[16];
      load16<DT>(shrow, (uint32_t)chunk * (16u * kEsize), sh);
      load16<DT>(scrow, (uint32_t)chunk * (16u * kEsize), sc);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        // The float32 product is rounded before the dtype rounding, as in the
        // eager graph: left to itself the compiler folds multiply-and-narrow
        // into one v_fma_mix (a single rounding of the exact product to f16),
        // which differs where the float32 product lands on an f16 midpoint.
        float prod = (keep[it][j] - mean) * rstd;
        asm volatile("" : "+v"(prod));
        const float ln = rnd<DT>(prod);
        keep[it][j] = rnd<DT>(rnd<DT>(rnd<DT>(1.0f + sc[j]) * ln) + sh[j]);
      }
    }
  }

  // FP6 output: every iteration's loads go out before the first rotation, so
  // the wave's whole share of the row is in flight at once (5 % faster at
  // 4608 x 15360, 1 % at K = 3072; the INT8 output ran 3-15 % slower so)
  constexpr bool kPrefetch = PRO == kProPlain && MODE == CONVROT_PREP_FP6;
  if constexpr (kPrefetch) {
#pragma unroll
    for (int it = 0; it < NI; ++it)
      load16<DT>(xrow, (uint32_t)((wave * NI + it) * 64 + lane) * (16u * kEsize), keep[it]);  // past the end: zeros
  }
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int block = wave * NI + it;
    const int chunk = block * 64 + lane;
    float (&v)[16] = keep[it];
    if constexpr (PRO == kProPlain && !kPrefetch) {
      load16<DT>(xrow, (uint32_t)chunk * (16u * kEsize), v);  // chunks past the row end read zeros
    } else if constexpr (PRO == kProGelu) {
      const int f0 = chunk * 16;  // head_features % 16 == 0: a chunk lies in one segment
      if (f0 < pa.head_features) {
        load16<DT>(hrow, (uint32_t)f0 * kEsize, v);
      } else {
        load16<DT>(xrow, (uint32_t)(f0 - pa.head_features) * kEsize, v);  // past the end: zeros
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          // the float32 result is rounded on its own, as the oracle does (no
          // multiply-and-narrow folding into one v_fma_mix for f16)
          float g = gelu_tanh32(v[j]);
          asm volatile("" : "+v"(g));
          v[j] = rnd<DT>(g);
        }
      }
    }
    rotate16<DT, S>(v, region, p);
    if constexpr (!kImplicitNorm && S > 0 && MODE != CONVROT_PREP_ROTATE) {
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = rnd<DT>(v[j] * kNorm);
    }
    if constexpr (MODE != CONVROT_PREP_ROTATE) {
#pragma unroll
      for (int j = 0; j < 16; j += 2) amax = absmax3(amax, v[j], v[j + 1]);
    }
  }

  // ---- row scale (core.py:154-156)
  RowScale<DT> rs{};
  if constexpr (MODE != CONVROT_PREP_ROTATE) {
    amax = wave_max_nonneg(amax);
    if (nwaves > 1) {
      if (lane == 0) wave_max[wave] = amax;
      __syncthreads();
      amax = wave_max[0];
      for (int w = 1; w < nwaves; ++w) amax = fmaxf(amax, wave_max[w]);
    }
    rs = row_scale<DT>(amax, kNorm);
    if (wave == 0 && lane == 0) scales[row] = rs.scale;
  }

  // ---- quantize + store, phase-final layout
  constexpr int PHF = (S >= 3) ? (S - 1) : 1;
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int block = wave * NI + it;
    const int chunk = block * 64 + lane;
    if (chunk >= chunks) continue;
    const int64_t gbase = row * K + (int64_t)block * 1024 + (lane / LG) * GS;
    const float (&v)[16] = keep[it];
    uint32_t q[16];
    float rt[16];
    constexpr bool kFp6Cvt = MODE == CONVROT_PREP_FP6 && DT == kBF16;  // FP6 by the conversion instruction
    if constexpr (MODE != CONVROT_PREP_ROTATE && !kFp6Cvt) {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float ratio = code_ratio<DT>(v[j], rs);
        // FP6 keeps |q| and the ratio's sign (rint is symmetric: |rint(c)| = rint(|c|))
        q[j] = code_bits(MODE == CONVROT_PREP_FP6 ? fabsf(ratio) : ratio);
        rt[j] = ratio;
      }
    }
    if constexpr (MODE == CONVROT_PREP_FP6) {
      // 16 consecutive features (a group's half stream, 12 bytes) are 4 runs
      // of 4: the lane's own 4 runs for groups up to 16, else run r of the 4
      // lanes of a quad (lane k holding features 4k .. 4k+3 of it), which
      // lane r of the quad gathers through the wave's LDS region.
      uint32_t d0, d1, d2;
      int fh;  // first feature (in the row) of the half this lane writes
      const int qb = lane & ~3, k = lane & 3;
      uint32_t* xr = (uint32_t*)(lds + wave * kRegionFloats);
      if constexpr (kFp6Cvt) {
        // bf16 ratios, two to a register (run r in hp[2r], hp[2r+1]), then one
        // conversion instruction for the lane's 16 features
        uint32_t hp[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) hp[i] = zero_code_sign_fix(pack_bf16x2(v[2 * i] * rs.inv, v[2 * i + 1] * rs.inv));
        if constexpr (S >= 3) {
          wave_lds_fence();
#pragma unroll
          for (int run = 0; run < 4; ++run)
            *(uint2*)(xr + (qb + run) * 8 + 2 * k) = make_uint2(hp[2 * run], hp[2 * run + 1]);
          wave_lds_fence();
          const uint4 g0 = *(const uint4*)(xr + (qb + k) * 8), g1 = *(const uint4*)(xr + (qb + k) * 8 + 4);
          hp[0] = g0.x, hp[1] = g0.y, hp[2] = g0.z, hp[3] = g0.w;
          hp[4] = g1.x, hp[5] = g1.y, hp[6] = g1.z, hp[7] = g1.w;
        }
        fp6_fields16(hp, d0, d1, d2);
      } else {
        // each run's four codes as a 24-bit field
        uint32_t pc[4];
#pragma unroll
        for (int run = 0; run < 4; ++run)
          pc[run] = fp6_piece(q[4 * run], q[4 * run + 1], q[4 * run + 2], q[4 * run + 3], rt[4 * run],
                              rt[4 * run + 1], rt[4 * run + 2], rt[4 * run + 3]);
        if constexpr (S >= 3) {
          wave_lds_fence();
#pragma unroll
          for (int run = 0; run < 4; ++run) xr[(qb + run) * 4 + k] = pc[run];
          wave_lds_fence();
          const uint4 g = *(const uint4*)(xr + (qb + k) * 4);
          pc[0] = g.x, pc[1] = g.y, pc[2] = g.z, pc[3] = g.w;
        }
        d0 = pc[0] | (pc[1] << 24);
        d1 = (pc[1] >> 8) | (pc[2] << 16);
        d2 = (pc[2] >> 16) | (pc[3] << 8);
      }
      if constexpr (S >= 3) fh = block * 1024 + (lane / LG) * GS + run_index<S, PHF>(p & ~3, k);
      else fh = block * 1024 + lane * 16;
      const int64_t mblocks = ((int64_t)gridDim.x + 15) >> 4;
      uint8_t* blk = (uint8_t*)out + ((int64_t)(fh >> 7) * mblocks + (row >> 4)) * 1536;
      const int L = ((fh >> 5) & 3) * 16 + (int)(row & 15);
      // The two halves of a 32-feature group share slot L: 12 bytes of the
      // first, then the second's first dword (its other 8 bytes go to the
      // block's tail).  They sit in lanes kPair apart (bit 4 of fh is lane bit
      // 2 for groups of 256 and 1024, lane bit 0 otherwise), so the first lane
      // writes the whole 16-byte slot: two stores a pair instead of three.
      // Both lanes of a pair are past the row end or neither (K % 128 == 0).
      constexpr int kPair = (S == 4 || S == 5) ? 4 : 1;
      const uint32_t d0_second = (uint32_t)__shfl_down((int)d0, kPair);
      if ((fh & 16) == 0) {
        *(uint4*)(blk + 16 * L) = make_uint4(d0, d1, d2, d0_second);
      } else {
        *(uint2*)(blk + 1024 + 8 * L) = make_uint2(d1, d2);
      }
      continue;
    }
#pragma unroll
    for (int run = 0; run < 4; ++run) {
      const int64_t f = gbase + run_index<(S >= 3 ? S : 3), PHF>(p, run);
      const float* vr = &v[4 * run];
      if constexpr (MODE == CONVROT_PREP_INT8_BLOCKED) {
        // the blocks the mid-size W4A4 GEMM's MFMA reads: 16 rows x 128 features, 1 KB for each 16-feature half
        const int fr = (int)(f - row * K);
        const int64_t mblocks = ((int64_t)gridDim.x + 15) >> 4;
        uint8_t* blk = (uint8_t*)out + ((int64_t)(fr >> 7) * mblocks + (row >> 4)) * 2048;
        *(uint32_t*)(blk + (fr & 16) * 64 + (((fr >> 5) & 3) * 16 + (int)(row & 15)) * 16 + (fr & 15)) =
            gather_bytes(q[4 * run], q[4 * run + 1], q[4 * run + 2], q[4 * run + 3]);
      } else if constexpr (MODE == CONVROT_PREP_INT8) {
        ((uint32_t*)out)[f >> 2] = gather_bytes(q[4 * run], q[4 * run + 1], q[4 * run + 2], q[4 * run + 3]);
      } else if constexpr (MODE == CONVROT_PREP_PACKED) {
        ((uint16_t*)out)[f >> 2] =
            (uint16_t)gather_nibbles(q[4 * run], q[4 * run + 1], q[4 * run + 2], q[4 * run + 3]);
      } else {
        // core.py:94 -- y / sqrt(G), rounded to the dtype
        store_out4<DT>(out, f, rnd<DT>(vr[0] * kNorm), rnd<DT>(vr[1] * kNorm), rnd<DT>(vr[2] * kNorm),
                       rnd<DT>(vr[3] * kNorm));
      }
    }
  }
}

// ---- 16-bit activations, two to a register
//
// The butterfly's cost is its rounding: with one value a register every add is
// a v_add_f32 and a conversion that rounds a single value (20 operations a
// radix-4, 5 a value and stage; MI355X issues a conversion every 1.9 ns a
// SIMD, an add every 1.3).  Here the values stay packed in x's type:
//  * float16: v_pk_add_f16, whose sum is the float32 sum rounded (24 >= 2 * 11
//    + 2 bits: rounding twice changes nothing), 1.25 operations a value and stage;
//  * bfloat16, which has no packed add: v_mfma_f32_4x4x4_16b_bf16 as one.  Its B
//    operand is the lane's own four values (two registers) and its A operand a
//    constant 4 x 4 matrix of 0, 1 and -1, so a lane's four results are sums and
//    differences of its values, which one conversion packs two at a time.  Every
//    such sum of two finite bf16 values, rounded to bf16, is the float32 sum
//    rounded, whatever the other two values are (their products are zeros): where
//    the exponents are within 16 the sum is exact in 24 bits, beyond that both round
//    to the larger.  tests/test_gpu_device_checks.py runs the butterflies on all
//    2^32 pairs, denormals among them, in each place of the four.
//    1.25 conversions a value and stage are left to the vector unit; the matrix
//    unit's 0.9 instructions run beside them.
// An infinity or NaN would reach the lane's other sums as 0 * inf, so a wave
// that ends with one (or with an overflow) rotates its share again in float32;
// only signs of zeros differ, which no code keeps (so ROTATE outputs of bf16
// stay with the kernel above); float16 rows take the same way (only the sign of
// a NaN may differ from prep_kernel's there).
//
// FP6 output, prep_kernel -> this kernel (back-to-back launches over cold
// buffers, us): bf16 G = 256 4608 x 3072 16.6 -> 13.8, 4608 x 15360 59.5 -> 51.7
// (3.8 TB/s), 8800 x 16384 112 -> 101-104, GELU 8800 x 16384 215 -> 172; float16
// 10017 x 2688 31.3 -> 23.5, 8800 x 16384 150 -> 103; packed output bf16
// 12288 x 3072 35.1 -> 26.5.  What is left above the bytes (8800 x 16384: 397 MB,
// 78 us at a copy's 5.1 TB/s) is the vector work, still 60 % of that time, where
// it does not overlap the loads, and the FP6 slots' 16-byte stores.
// Registers for 5, 6 and 8 waves a SIMD at 4, 3 and 1 iterations: left alone the
// compiler takes 4 waves' worth (4608 x 3072: 15.2 us).

// A run of four packed features in the wave's LDS: its two dwords lie in two
// planes of kPlane dwords, one dword of padding after every four runs
// (conflict-free but for phase 3's two-way).  In planes a lane reads the same
// dword of two runs with one ds_read2_b32, into the register pair that the
// stage's MFMA takes; whole runs (8 bytes) would leave the pairs to v_movs.
constexpr int kPlane = 324;  // past a ds_read2's offsets and no multiple of 64: the planes are not paired
constexpr int kPkRegion = 2 * kPlane;  // dwords of a wave's LDS (the FP6 output's transpose takes 512)
__device__ __forceinline__ int pk_off(int i) { return (i >> 2) + (i >> 4); }

template <int DT, int S, int PH, bool EXACT>
__device__ __forceinline__ void pk_exchange_and_stage(const Matrices& m, uint32_t (&h)[8], uint32_t* region, int p) {
#pragma unroll
  for (int run = 0; run < 4; ++run) {
    uint32_t* at = region + pk_off(run_index<S, PH - 1>(p, run));
    at[0] = h[2 * run];
    at[kPlane] = h[2 * run + 1];
  }
  wave_lds_fence();
#pragma unroll
  for (int run = 0; run < 4; ++run) {
    const uint32_t* at = region + pk_off(run_index<S, PH>(p, run));
    h[2 * run] = at[0];
    h[2 * run + 1] = at[kPlane];
  }
  wave_lds_fence();
#pragma unroll
  for (int i = 0; i < 2; ++i) pk_stage_regs<DT, EXACT>(m, h[i], h[2 + i], h[4 + i], h[6 + i]);
}

// rotate16 on packed values (h[2 * run], h[2 * run + 1]: a run's four features).
template <int DT, int S, bool EXACT = false>
__device__ __forceinline__ void pk_rotate16(const Matrices& m, uint32_t (&h)[8], uint32_t* region, int p) {
#pragma unroll
  for (int r = 0; r < 4; ++r) pk_stage_run<DT, EXACT>(m, h[2 * r], h[2 * r + 1]);
  if constexpr (S >= 2) {
#pragma unroll
    for (int i = 0; i < 2; ++i) pk_stage_regs<DT, EXACT>(m, h[i], h[2 + i], h[4 + i], h[6 + i]);
  }
  if constexpr (S >= 3) pk_exchange_and_stage<DT, S, 2, EXACT>(m, h, region, p);
  if constexpr (S >= 4) pk_exchange_and_stage<DT, S, 3, EXACT>(m, h, region, p);
  if constexpr (S >= 5) pk_exchange_and_stage<DT, S, 4, EXACT>(m, h, region, p);
}

// 16 consecutive 16-bit elements at byte `off` of a row (past its end: zeros).
__device__ __forceinline__ void pk_load16(__amdgpu_buffer_rsrc_t row, uint32_t off, uint32_t (&h)[8]) {
  const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(row, (int)off, 0, 0);
  const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(row, (int)(off + 16), 0, 0);
  h[0] = a.x, h[1] = a.y, h[2] = a.z, h[3] = a.w, h[4] = b.x, h[5] = b.y, h[6] = b.z, h[7] = b.w;
}

// Largest magnitude of 16 packed values, folded into the halves of `m` as bit
// patterns (they order like the magnitudes, infinity and NaN on top).
__device__ __forceinline__ uint32_t pk_absmax(uint32_t m, const uint32_t (&h)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const u16x2 v = __builtin_bit_cast(u16x2, h[i] & 0x7fff7fffu);
    m = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, m), v));
  }
  return m;
}

// The float16 ratio of a finite value to a finite scale from inv = 1 / scale
// (0 for a zero scale): one correction step, whose float32 quotient rounds to
// the float16 the true division's rounds to (checked over every pair of
// significands, tests/test_prep16.py).
__device__ __forceinline__ float f16_quotient(float v, float scale, float inv) {
  const float q = v * inv;
  return __builtin_fmaf(__builtin_fmaf(-q, scale, v), inv, q);
}

// Two packed ratios clamped to [-7, 7] (a float16 scale may be a denormal far
// below absmax / 7), with +0 for the codes that are zero.
__device__ __forceinline__ uint32_t f16_clamp_sign_fix(uint32_t w) {
  const f16x2 seven = {(_Float16)7.0f, (_Float16)7.0f};
  const uint32_t h = as_u32(__builtin_elementwise_max(__builtin_elementwise_min(as_f16(w), seven), -seven));
  const u16x2 s = __builtin_bit_cast(u16x2, h) + (u16x2){0x47ff, 0x47ff};  // bit 15: negative, at most 0.5
  return h & ~(__builtin_bit_cast(uint32_t, s) & 0x80008000u);
}

typedef _Float16 f16x32 __attribute__((ext_vector_type(32)));

template <int DT>
__device__ __forceinline__ void pk_fp6_fields16(const uint32_t (&hp)[8], uint32_t& d0, uint32_t& d1, uint32_t& d2) {
  if constexpr (DT == kBF16) {
    fp6_fields16(hp, d0, d1, d2);
  } else {
    const u32x16 in = {hp[0], hp[1], hp[2], hp[3], hp[4], hp[5], hp[6], hp[7], 0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
    const i32x6 f = __builtin_amdgcn_cvt_scalef32_pk32_fp6_f16(__builtin_bit_cast(f16x32, in), 8.0f);
    d0 = (uint32_t)f[0];
    d1 = (uint32_t)f[1];
    d2 = (uint32_t)f[2];
  }
}

// prep_kernel for 16-bit x with S >= 1 (bf16: not ROTATE), the same work split
// and the same bits.
template <int DT, int S, int NI, int MODE, int PRO>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(PRO == kProModulate ? 4 : NI == 4 || S == 5 ? 5 : NI == 3 ? 6 : 8)))
void prep16_kernel(const void* __restrict__ x, void* __restrict__ out,
                                                       float* __restrict__ scales, int K, ProducerArgs pa) {
  static_assert(S >= 1 && (DT == kF16 || (DT == kBF16 && MODE != CONVROT_PREP_ROTATE)), "see above");
  constexpr bool PRE = PRO == kProModulate;
  extern __shared__ uint32_t lds16[];
  uint32_t* const lds = lds16;
  __shared__ float wave_max[kMaxWaves];
  __shared__ double block_moments[PRE ? kMaxBlocks : 1][2];

  constexpr int G = 1 << (2 * S);
  constexpr int LG = (S >= 3) ? (G / 16) : 1, GS = (S >= 3) ? G : 16;  // lanes of a group, features of a lane group
  constexpr int PHF = (S >= 3) ? (S - 1) : 1;
  constexpr float kNorm = 1.0f / (float)(1 << S);

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int nwaves = blockDim.x >> 6;
  int64_t row = blockIdx.x;
  if constexpr (MODE == CONVROT_PREP_FP6 || MODE == CONVROT_PREP_INT8_BLOCKED) {  // as prep_kernel
    const int64_t run = ((int64_t)gridDim.x / (8 * 16)) * 16;
    if (row < 8 * run) row = (row & 7) * run + (row >> 3);
  }
  const int chunks = K >> 4;
  const __amdgpu_buffer_rsrc_t xrow = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const char*)x + row * (PRO == kProGelu ? pa.x_stride : (int64_t)K) * 2), (short)0,
      (PRO == kProGelu ? K - pa.head_features : K) * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t hrow = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(PRO == kProGelu && pa.head_features ? (const char*)pa.head + row * pa.head_stride * 2
                                                  : (const char*)x),
      (short)0, PRO == kProGelu ? pa.head_features * 2 : 0, 0x00020000);
  uint32_t* wave_lds = lds + wave * kPkRegion;
  uint32_t* region = wave_lds + (lane / LG) * pk_off(G);
  const int p = lane % LG;
  const Matrices mat = matrices(lane);

  uint32_t h[NI][8];
  // ---- producer: x's 16 values of an iteration, past the row end zeros
  float mean = 0.0f, rstd = 0.0f;
  const int64_t vrow = PRE ? row / pa.rows_per_vector : 0;
  auto load = [&](int it, uint32_t (&v)[8]) {
    const int f0 = ((wave * NI + it) * 64 + lane) * 16;
    if (PRO == kProGelu && f0 < pa.head_features) {  // head_features % 16 == 0: a chunk lies in one segment
      pk_load16(hrow, (uint32_t)f0 * 2u, v);
    } else {
      pk_load16(xrow, (uint32_t)(f0 - (PRO == kProGelu ? pa.head_features : 0)) * 2u, v);
    }
  };
  auto produce = [&](int it, uint32_t (&v)[8]) {
    const int chunk = (wave * NI + it) * 64 + lane;
    if constexpr (PRO == kProGelu) {
      if (chunk * 16 >= pa.head_features) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          // the float32 result is rounded on its own, as the oracle does (no
          // multiply-and-narrow folding into one v_fma_mix for f16)
          float lo = gelu_tanh32(pk_lo<DT>(v[i])), hi = gelu_tanh32(pk_hi<DT>(v[i]));
          asm volatile("" : "+v"(lo), "+v"(hi));
          v[i] = pk_make<DT>(lo, hi);
        }
      }
    } else if constexpr (PRE) {
      if (chunk < chunks) {  // padding stays zero (whole groups lie past K)
        const __amdgpu_buffer_rsrc_t shrow = __builtin_amdgcn_make_buffer_rsrc(
            (void*)((const char*)pa.shift + vrow * K * 2), (short)0, K * 2, 0x00020000);
        const __amdgpu_buffer_rsrc_t scrow = __builtin_amdgcn_make_buffer_rsrc(
            (void*)((const char*)pa.scale + vrow * K * 2), (short)0, K * 2, 0x00020000);
        uint32_t sh[8], sc[8];
        pk_load16(shrow, (uint32_t)chunk * 32u, sh);
        pk_load16(scrow, (uint32_t)chunk * 32u, sc);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float plo = (pk_lo<DT>(v[i]) - mean) * rstd, phi = (pk_hi<DT>(v[i]) - mean) * rstd;
          asm volatile("" : "+v"(plo), "+v"(phi));  // rounded before the dtype rounding, as in prep_kernel
          const float lo = rnd<DT>(rnd<DT>(1.0f + pk_lo<DT>(sc[i])) * rnd<DT>(plo)) + pk_lo<DT>(sh[i]);
          const float hi = rnd<DT>(rnd<DT>(1.0f + pk_hi<DT>(sc[i])) * rnd<DT>(phi)) + pk_hi<DT>(sh[i]);
          v[i] = pk_make<DT>(lo, hi);
        }
      }
    }
  };

  // every iteration's loads go out first: the wave's share of the row in flight at once
#pragma unroll
  for (int it = 0; it < NI; ++it) load(it, h[it]);
  if constexpr (PRE) {
    const int real_blocks = (chunks + 63) >> 6;
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int block = wave * NI + it;
      __builtin_amdgcn_sched_barrier(0);
      double b1 = 0.0, b2 = 0.0;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const double d = (double)(j & 1 ? pk_hi<DT>(h[it][j >> 1]) : pk_lo<DT>(h[it][j >> 1]));
        b1 += d;
        b2 = __builtin_fma(d, d, b2);  // the square is exact
      }
      b1 = wave_sum_f64(b1);
      b2 = wave_sum_f64(b2);
      if (lane == 0 && block < real_blocks) {
        block_moments[block][0] = b1;
        block_moments[block][1] = b2;
      }
    }
    __syncthreads();
    double s1 = 0.0, s2 = 0.0;
    for (int b = 0; b < real_blocks; ++b) {
      s1 += block_moments[b][0];
      s2 += block_moments[b][1];
    }
    const double m64 = s1 / (double)K;
    double var = s2 / (double)K - m64 * m64;
    var = var > 0.0 ? var : 0.0;
    mean = (float)m64;
    rstd = (float)(1.0 / sqrt(var + (double)pa.eps));
  }

  uint32_t pmax = 0;
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    if constexpr (PRO != kProPlain) __builtin_amdgcn_sched_barrier(0);  // one iteration's operands in registers at a time
    produce(it, h[it]);
    pk_rotate16<DT, S>(mat, h[it], region, p);
    if constexpr (DT == kF16 && MODE != CONVROT_PREP_ROTATE) {
      const f16x2 norm = {(_Float16)kNorm, (_Float16)kNorm};
#pragma unroll
      for (int i = 0; i < 8; ++i) h[it][i] = as_u32(as_f16(h[it][i]) * norm);
    }
    pmax = pk_absmax(pmax, h[it]);
  }

  // ---- row scale (core.py:154-156)
  RowScale<DT> rs{};
  constexpr uint32_t kInf = DT == kBF16 ? 0x7f80u : 0x7c00u;
  const uint32_t top = __float_as_uint(wave_max_nonneg(__uint_as_float(max(pmax & 0xffffu, pmax >> 16))));
  bool bad = top >= kInf;  // this wave holds an infinity or NaN (wave-uniform)
  float amax = DT == kBF16 ? bf16_lo(top) : (float)as_f16(top).x;
  if (bad) {  // once more by the float32 butterfly, as prep_kernel does (absmax3 passes over NaN)
    float exact = 0.0f;
#pragma unroll 1
    for (int it = 0; it < NI; ++it) {
      uint32_t w[8];
      load(it, w);
      produce(it, w);
      pk_rotate16<DT, S, true>(mat, w, region, p);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if constexpr (DT == kF16 && MODE != CONVROT_PREP_ROTATE)
          w[i] = pk_make<DT>(pk_lo<DT>(w[i]) * kNorm, pk_hi<DT>(w[i]) * kNorm);
        exact = absmax3(exact, pk_lo<DT>(w[i]), pk_hi<DT>(w[i]));
      }
#pragma unroll
      for (int k = 0; k < NI; ++k)
#pragma unroll
        for (int i = 0; i < 8; ++i) h[k][i] = k == it ? w[i] : h[k][i];
    }
    amax = wave_max_nonneg(exact);
  }
  if constexpr (MODE != CONVROT_PREP_ROTATE) {
    if (nwaves > 1) {
      if (lane == 0) wave_max[wave] = amax;
      __syncthreads();
      amax = wave_max[0];
      for (int w = 1; w < nwaves; ++w) amax = fmaxf(amax, wave_max[w]);
    }
    rs = row_scale<DT>(amax, kNorm);
    if (wave == 0 && lane == 0) scales[row] = rs.scale;
    bad |= !(rs.scale < __builtin_inff());
  }
  const float finv = DT == kF16 && rs.scale > 0.0f ? 1.0f / rs.scale : 0.0f;

  // ---- quantize + store, phase-final layout
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int block = wave * NI + it;
    const int chunk = block * 64 + lane;
    if (chunk >= chunks) continue;
    const uint32_t (&v)[8] = h[it];
    float ratio[16];  // unrounded where they are packed next (FP6)
    if constexpr (MODE != CONVROT_PREP_ROTATE) {
      if (DT == kF16 && bad) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          ratio[2 * i] = code_ratio<DT>(pk_lo<DT>(v[i]), rs), ratio[2 * i + 1] = code_ratio<DT>(pk_hi<DT>(v[i]), rs);
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float r = i & 1 ? pk_hi<DT>(v[i >> 1]) : pk_lo<DT>(v[i >> 1]);
          ratio[i] = DT == kBF16 ? r * rs.inv : f16_quotient(r, rs.scale, finv);
          if constexpr (MODE != CONVROT_PREP_FP6) ratio[i] = rnd<DT>(ratio[i]);
        }
      }
    }
    const int64_t mblocks = ((int64_t)gridDim.x + 15) >> 4;
    if constexpr (MODE == CONVROT_PREP_FP6) {
      // 16 consecutive features (a group's half stream, 12 bytes) are 4 runs
      // of 4: the lane's own 4 runs for groups up to 16, else run r of the 4
      // lanes of a quad (lane k holding features 4k .. 4k+3 of it), which
      // lane r of the quad gathers through the wave's LDS region.
      uint32_t d0, d1, d2;
      const int qb = lane & ~3, k = lane & 3;
      uint32_t* xr = wave_lds;
      uint32_t hp[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        hp[i] = pk_make<DT>(ratio[2 * i], ratio[2 * i + 1]);
        if constexpr (DT == kBF16) hp[i] = zero_code_sign_fix(hp[i]);
        else hp[i] = bad ? hp[i] : f16_clamp_sign_fix(hp[i]);
      }
      if constexpr (S >= 3) {
        wave_lds_fence();
#pragma unroll
        for (int run = 0; run < 4; ++run)
          *(uint2*)(xr + (qb + run) * 8 + 2 * k) = make_uint2(hp[2 * run], hp[2 * run + 1]);
        wave_lds_fence();
        const uint4 g0 = *(const uint4*)(xr + (qb + k) * 8), g1 = *(const uint4*)(xr + (qb + k) * 8 + 4);
        hp[0] = g0.x, hp[1] = g0.y, hp[2] = g0.z, hp[3] = g0.w;
        hp[4] = g1.x, hp[5] = g1.y, hp[6] = g1.z, hp[7] = g1.w;
      }
      if (DT == kF16 && bad) {  // NaN ratios: the codes of prep_kernel's float16
        uint32_t pc[4];
#pragma unroll
        for (int run = 0; run < 4; ++run) {
          float r[4];
          r[0] = pk_lo<DT>(hp[2 * run]), r[1] = pk_hi<DT>(hp[2 * run]);
          r[2] = pk_lo<DT>(hp[2 * run + 1]), r[3] = pk_hi<DT>(hp[2 * run + 1]);
          pc[run] = fp6_piece(code_bits(fabsf(r[0])), code_bits(fabsf(r[1])), code_bits(fabsf(r[2])),
                              code_bits(fabsf(r[3])), r[0], r[1], r[2], r[3]);
        }
        d0 = pc[0] | (pc[1] << 24);
        d1 = (pc[1] >> 8) | (pc[2] << 16);
        d2 = (pc[2] >> 16) | (pc[3] << 8);
      } else {
        pk_fp6_fields16<DT>(hp, d0, d1, d2);
      }
      int fh;  // first feature (in the row) of the half this lane writes
      if constexpr (S >= 3) fh = block * 1024 + (lane / LG) * GS + run_index<S, PHF>(p & ~3, k);
      else fh = block * 1024 + lane * 16;
      uint8_t* blk = (uint8_t*)out + ((int64_t)(fh >> 7) * mblocks + (row >> 4)) * 1536;
      const int L = ((fh >> 5) & 3) * 16 + (int)(row & 15);
      // The two halves of a 32-feature group share slot L: 12 bytes of the
      // first, then the second's first dword (its other 8 bytes go to the
      // block's tail).  They sit in lanes kPair apart (bit 4 of fh is lane bit
      // 2 for groups of 256 and 1024, lane bit 0 otherwise), so the first lane
      // writes the whole 16-byte slot: two stores a pair instead of three.
      // Both lanes of a pair are past the row end or neither (K % 128 == 0).
      constexpr int kPair = (S == 4 || S == 5) ? 4 : 1;
      const uint32_t d0_second = (uint32_t)__shfl_down((int)d0, kPair);
      if ((fh & 16) == 0) {
        *(uint4*)(blk + 16 * L) = make_uint4(d0, d1, d2, d0_second);
      } else {
        *(uint2*)(blk + 1024 + 8 * L) = make_uint2(d1, d2);
      }
    } else {
#pragma unroll
      for (int run = 0; run < 4; ++run) {
        const int fr = block * 1024 + (lane / LG) * GS + run_index<(S >= 3 ? S : 3), PHF>(p, run);
        const int64_t f = row * K + fr;
        if constexpr (MODE == CONVROT_PREP_ROTATE) {
          // core.py:94 -- y / sqrt(G), rounded to the dtype
          const f16x2 norm = {(_Float16)kNorm, (_Float16)kNorm};
          *(uint2*)((uint16_t*)out + f) =
              make_uint2(as_u32(as_f16(v[2 * run]) * norm), as_u32(as_f16(v[2 * run + 1]) * norm));
        } else {
          const uint32_t q0 = code_bits(ratio[4 * run]), q1 = code_bits(ratio[4 * run + 1]),
                         q2 = code_bits(ratio[4 * run + 2]), q3 = code_bits(ratio[4 * run + 3]);
          if constexpr (MODE == CONVROT_PREP_INT8_BLOCKED) {
            uint8_t* blk = (uint8_t*)out + ((int64_t)(fr >> 7) * mblocks + (row >> 4)) * 2048;
            *(uint32_t*)(blk + (fr & 16) * 64 + (((fr >> 5) & 3) * 16 + (int)(row & 15)) * 16 + (fr & 15)) =
                gather_bytes(q0, q1, q2, q3);
          } else if constexpr (MODE == CONVROT_PREP_INT8) {
            ((uint32_t*)out)[f >> 2] = gather_bytes(q0, q1, q2, q3);
          } else {
            ((uint16_t*)out)[f >> 2] = (uint16_t)gather_nibbles(q0, q1, q2, q3);
          }
        }
      }
    }
  }
}

// Which rows prep16_kernel prepares; rounding and codes are the same on both.
// prep_kernel stays the faster one (us, prep16_kernel against it) for
//  * bf16 rows of four blocks a wave behind the modulated producer, which spill
//    (8800 x 16384: 193 against 174);
//  * plain bf16 rows of groups up to 64 with FP6 output up to 16384 features, where
//    the butterfly is short and the FP6 stores are the bound: finishing rows sooner,
//    prep16_kernel has more 16-row blocks open at once and writes their lines back
//    in more pieces (8800 x 16384, G = 64: 118-123 MB against 108, 104 against
//    96; 4877 x 29568, many more waves a row: 110 against 149).  G = 64 wins up to
//    12288 features and on few rows (1536 x 16384: 22.2 against 30.8); G = 16 only
//    on very short rows or few 1024-feature blocks in all (8800 x 8192 57 against 55,
//    2000 x 12288 22.5 against 19.7, but 7020 x 1152 9.4 against 10.2, 381 x 12288
//    7.0 against 7.2);
//  * other plain bf16 rows of groups of 4, there (packed 1061 x 14336 13.5 against
//    12.4; int8 682 x 28032 17.2 against 18.0);
//  * float16 ROTATE on one iteration: plain at G = 64 beyond 10240 features and
//    12288 blocks in all (2000 x 12288 22.3 against 21.2; 2048 x 10240 19.7 against
//    20.1, 710 x 14336 11.4 against 12.2), modulated at G up to 16 (5879 x 7168,
//    G = 16: 43.5 against 40.3).
enum Packed : int { kNoRows, kCode64Rows, kCode16Rows, kRotateRows, kAllRows };
constexpr int64_t kFewRows = 2048, kFewBlocks = 12288;
constexpr Packed prep_packed(int dtype, int log4g, int ni, int mode, int producer) {
  if (log4g < 1 || dtype == kF32) return kNoRows;
  if (dtype == kBF16) {
    if (mode == CONVROT_PREP_ROTATE || (producer == kProModulate && ni == 4)) return kNoRows;
    if (producer == kProPlain && (log4g == 1 || (mode == CONVROT_PREP_FP6 && log4g <= 3)))
      return log4g == 3 ? kCode64Rows : kCode16Rows;
  } else if (mode == CONVROT_PREP_ROTATE && ni == 1) {
    if (producer == kProPlain && log4g == 3) return kRotateRows;
    if (producer == kProModulate && log4g <= 2) return kNoRows;
  }
  return kAllRows;
}
constexpr bool prep_packed_rows(Packed p, int64_t rows, int64_t K) {
  switch (p) {
    case kCode64Rows: return K <= 12288 || K > 16384 || rows <= kFewRows;
    case kCode16Rows: return K < 2048 || K > 16384 || rows * ((K + 1023) / 1024) < kFewBlocks;
    case kRotateRows: return K <= 10240 || rows * ((K + 1023) / 1024) < kFewBlocks;
    default: return p == kAllRows;
  }
}

// The producer of a launch and its arguments.
struct Modulation {
  int producer;  // kProPlain, kProModulate or kProGelu
  ProducerArgs args;
};

template <int DT, int S, int NI, int MODE, int PRO>
void launch_prep_pro(const void* x, void* out, float* scales, int64_t rows, int K, int waves, const ProducerArgs& args,
                     hipStream_t stream) {
  constexpr Packed kPacked = prep_packed(DT, S, NI, MODE, PRO);
  const auto launch = [&](void (*kernel)(const void*, void*, float*, int, ProducerArgs), int region) {
    const size_t lds_bytes = S >= 3 ? (size_t)waves * (size_t)region * 4 : 0;
    hipLaunchKernelGGL(kernel, dim3((unsigned)rows), dim3(64 * waves), lds_bytes, stream, x, out, scales, K, args);
  };
  if constexpr (kPacked != kNoRows) {
    if (prep_packed_rows(kPacked, rows, K)) return launch(prep16_kernel<DT, S, NI, MODE, PRO>, kPkRegion);
  }
  if constexpr (kPacked != kAllRows) launch(prep_kernel<DT, S, NI, MODE, PRO>, kRegionFloats);
}

template <int DT, int S, int NI, int MODE>
hipError_t launch_prep_t(const void* x, void* out, float* scales, int64_t rows, int K, int waves,
                         const Modulation& mod, hipStream_t stream) {
  if constexpr (S == 0) {  // no rotation: the plain producer only
    launch_prep_pro<DT, S, NI, MODE, kProPlain>(x, out, scales, rows, K, waves, mod.args, stream);
  } else {
    if (mod.producer == kProModulate)
      launch_prep_pro<DT, S, NI, MODE, kProModulate>(x, out, scales, rows, K, waves, mod.args, stream);
    else if (mod.producer == kProGelu)
      launch_prep_pro<DT, S, NI, MODE, kProGelu>(x, out, scales, rows, K, waves, mod.args, stream);
    else
      launch_prep_pro<DT, S, NI, MODE, kProPlain>(x, out, scales, rows, K, waves, mod.args, stream);
  }
  return hipGetLastError();
}

template <int DT, int S, int NI>
hipError_t launch_prep_mode(int mode, const void* x, void* out, float* scales, int64_t rows, int K,
                            int waves, const Modulation& mod, hipStream_t stream) {
  switch (mode) {
    case CONVROT_PREP_PACKED:
      return launch_prep_t<DT, S, NI, CONVROT_PREP_PACKED>(x, out, scales, rows, K, waves, mod, stream);
    case CONVROT_PREP_FP6:
      return launch_prep_t<DT, S, NI, CONVROT_PREP_FP6>(x, out, scales, rows, K, waves, mod, stream);
    case CONVROT_PREP_INT8_BLOCKED:
      return launch_prep_t<DT, S, NI, CONVROT_PREP_INT8_BLOCKED>(x, out, scales, rows, K, waves, mod, stream);
    case CONVROT_PREP_INT8:
      return launch_prep_t<DT, S, NI, CONVROT_PREP_INT8>(x, out, scales, rows, K, waves, mod, stream);
    default: return launch_prep_t<DT, S, NI, CONVROT_PREP_ROTATE>(x, out, scales, rows, K, waves, mod, stream);
  }
}

template <int DT, int S>
hipError_t launch_prep_ni(int ni, int mode, const void* x, void* out, float* scales, int64_t rows, int K,
                          int waves, const Modulation& mod, hipStream_t stream) {
  switch (ni) {
    case 1: return launch_prep_mode<DT, S, 1>(mode, x, out, scales, rows, K, waves, mod, stream);
    case 3: return launch_prep_mode<DT, S, 3>(mode, x, out, scales, rows, K, waves, mod, stream);
    default: return launch_prep_mode<DT, S, 4>(mode, x, out, scales, rows, K, waves, mod, stream);
  }
}

template <int DT>
hipError_t launch_prep_s(int s, int ni, int mode, const void* x, void* out, float* scales, int64_t rows,
                         int K, int waves, const Modulation& mod, hipStream_t stream) {
  switch (s) {
    case 0: return launch_prep_ni<DT, 0>(ni, mode, x, out, scales, rows, K, waves, mod, stream);
    case 1: return launch_prep_ni<DT, 1>(ni, mode, x, out, scales, rows, K, waves, mod, stream);
    case 2: return launch_prep_ni<DT, 2>(ni, mode, x, out, scales, rows, K, waves, mod, stream);
    case 3: return launch_prep_ni<DT, 3>(ni, mode, x, out, scales, rows, K, waves, mod, stream);
    case 4: return launch_prep_ni<DT, 4>(ni, mode, x, out, scales, rows, K, waves, mod, stream);
    default: return launch_prep_ni<DT, 5>(ni, mode, x, out, scales, rows, K, waves, mod, stream);
  }
}

}  // namespace

// Pick (iterations per wave, waves per row) so that 1024*NI*W covers K with
// the fewest idle 1024-feature blocks; NI in {3, 4, 1}, W <= 16.  Few rows
// (M <= 2048) take one iteration per wave and more waves per row instead, so
// that enough waves are in flight to cover the load latency.  The packed kernel
// differs (us):
//  * few rows take one iteration only up to 12288 blocks in all (bf16 1536 x 15360,
//    one -> four: 21.4 -> 18.7, modulated 39.1 -> 34.2, though that runs on
//    prep_kernel, and not on two waves: 1667 x 8192 21.5 -> 25.3).  Plain rotated
//    outputs (float16 2000 x 12288, G = 64: 22.5 -> 24.9), the GELU producer and plain
//    groups up to 16 of at most 12 blocks (bf16 1536 x 12288, G = 16: 12.5 -> 13.6)
//    gain nothing;
//  * plain FP6 rows of groups up to 64 (bf16: 64, up to 12288 features) take one
//    iteration where four would be taken, with fewer rows and so fewer 16-row blocks
//    open: bf16 G = 64 8800 x 8192 58.3 -> 51.4, float16 G = 16 8800 x 16384 124 -> 93.5;
//  * else 13 to 16 blocks are four waves of four, as 15 and 16 are on any kernel
//    (bf16 G = 256 FP6 4608 x 13312, thirteen of one -> four of four: 58.0 -> 47.8).
static bool prep_plan(int64_t rows, int64_t K, int dtype, int log4g, int mode, int producer, int* ni_out, int* waves_out) {
  const int64_t blocks = (K + 1023) / 1024;
  {  // tuning override: force the iterations per wave
    const int ni = tuning(kTunePrepNi);
    if (ni == 1 || ni == 3 || ni == 4) {
      const int64_t w = (blocks + ni - 1) / ni;
      if (w <= kMaxWaves) {
        *ni_out = ni;
        *waves_out = (int)w;
        return true;
      }
    }
  }
  const Packed packed = prep_packed(dtype, log4g, 3, mode, producer);
  const bool coded = packed != kNoRows && packed != kCode16Rows && producer != kProGelu &&
                     !(producer == kProPlain && mode == CONVROT_PREP_ROTATE);
  const bool deep = coded && rows * blocks > kFewBlocks && (log4g > 2 || producer != kProPlain || blocks > 12) &&
                    (dtype != kBF16 || producer != kProModulate || blocks > 8);
  const bool spread = producer == kProPlain && mode == CONVROT_PREP_FP6 &&
                      (packed == kCode64Rows ? K <= 12288 : packed == kAllRows && log4g <= 2);
  if (blocks <= kMaxWaves && rows <= kFewRows && !deep) {
    *ni_out = 1;
    *waves_out = (int)blocks;
    return true;
  }
  if (coded && blocks > 12 && blocks <= 16) {
    *ni_out = spread ? 1 : 4;
    *waves_out = spread ? (int)blocks : 4;
    return true;
  }
  int best_ni = 0, best_w = 0;
  int64_t best_idle = -1;
  const int cand[3] = {3, 4, 1};
  for (int c = 0; c < 3; ++c) {
    const int ni = cand[c];
    const int64_t w = (blocks + ni - 1) / ni;
    if (w > kMaxWaves) continue;
    const int64_t idle = w * ni - blocks;
    if (best_idle < 0 || idle < best_idle) {
      best_idle = idle;
      best_ni = ni;
      best_w = (int)w;
    }
  }
  // Three iterations on more than four waves lose to four iterations on at
  // most four waves with one idle block: at 4608 rows, 15 blocks run 7 % faster
  // as 4 waves x 4 than as 5 waves x 3 (12 blocks stay 4 x 3).
  if (best_ni == 3 && best_w > 4) {
    const int64_t w4 = (blocks + 3) / 4;
    if (w4 <= 4 && w4 * 4 - blocks <= best_idle + 1) {
      best_ni = 4;
      best_w = (int)w4;
      best_idle = w4 * 4 - blocks;
    }
  }
  if (best_idle < 0) return false;
  if (spread && best_ni == 4 && blocks <= kMaxWaves) best_ni = 1, best_w = (int)blocks;
  *ni_out = best_ni;
  *waves_out = best_w;
  return true;
}

bool prep_route(int64_t rows, int64_t K, int dtype, int log4g, int mode, int producer, int* iterations, int* waves,
                bool* packed) {
  if (!prep_plan(rows, K, dtype, log4g, mode, producer, iterations, waves)) return false;
  *packed = prep_packed_rows(prep_packed(dtype, log4g, *iterations, mode, producer), rows, K);
  return true;
}

namespace {

hipError_t launch_prep_any(const void* x, int dtype, int64_t rows, int64_t K, int log4g, int mode, void* out,
                           float* scales, const Modulation& mod, hipStream_t stream) {
  int ni = 0, waves = 0;
  if (!prep_plan(rows, K, dtype, log4g, mode, mod.producer, &ni, &waves)) return hipErrorInvalidValue;
  if (rows == 0) return hipSuccess;
  switch (dtype) {
    case kF32: return launch_prep_s<kF32>(log4g, ni, mode, x, out, scales, rows, (int)K, waves, mod, stream);
    case kF16: return launch_prep_s<kF16>(log4g, ni, mode, x, out, scales, rows, (int)K, waves, mod, stream);
    default: return launch_prep_s<kBF16>(log4g, ni, mode, x, out, scales, rows, (int)K, waves, mod, stream);
  }
}

}  // namespace

hipError_t launch_prep(const void* x, int dtype, int64_t rows, int64_t K, int log4g, int mode, void* out,
                       float* scales, hipStream_t stream) {
  Modulation mod{};
  mod.producer = kProPlain;
  return launch_prep_any(x, dtype, rows, K, log4g, mode, out, scales, mod, stream);
}

hipError_t launch_prep_modulated(const void* x, int dtype, int64_t rows, int64_t K, int log4g, int mode,
                                 const void* shift, const void* scale, int64_t rows_per_vector, float eps,
                                 void* out, float* scales, hipStream_t stream) {
  Modulation mod{};
  mod.producer = kProModulate;
  mod.args.shift = shift;
  mod.args.scale = scale;
  mod.args.rows_per_vector = (int)rows_per_vector;
  mod.args.eps = eps;
  return launch_prep_any(x, dtype, rows, K, log4g, mode, out, scales, mod, stream);
}

hipError_t launch_prep_gelu(const void* head, int64_t head_features, int64_t head_stride, const void* x,
                            int64_t x_features, int64_t x_stride, int dtype, int64_t rows, int log4g, int mode,
                            void* out, float* scales, hipStream_t stream) {
  Modulation mod{};
  mod.producer = kProGelu;
  mod.args.head = head;
  mod.args.head_features = (int)head_features;
  mod.args.head_stride = head_stride;
  mod.args.x_stride = x_stride;
  return launch_prep_any(x, dtype, rows, head_features + x_features, log4g, mode, out, scales, mod, stream);
}

}  // namespace convrot
