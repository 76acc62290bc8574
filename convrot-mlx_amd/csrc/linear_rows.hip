// ConvRot linear for a few token rows in one launch on gfx950: the activation
// preparation (rotation, and for W4A4 the absmax and A4 codes) inside the
// weight-streaming GEMM, from x to the output.
//
// Serves ConvRotLinear where a call is launches and latency (a modulation row
// of a diffusion transformer, a decoder's single row): the reference runs the
// preparation and the matmul as two kernels (/root/reference/src/convrot_mlx/
// core.py:1270-1313), and so do this library's larger sizes.  The weights are
// all that has to come from HBM; a workgroup starts their loads, then rotates
// the rows itself while they are in flight.  Every workgroup repeats the
// preparation (a row of 3072 features is three wave-blocks on eight waves),
// which costs less than the second launch and the trip of the codes through
// memory as long as the rows are few.
//
// The arithmetic is the two kernels': the preparation's bits (prep_device.h),
// exact integer dots, and ((f(dot) * xs) * ws) + bias; for W4A16 the rotated
// row in x's type, float32 sums of 16x codes, (dots * ws) + bias.
//
// Work split: TG * KS waves; wave (tg, ks) takes weight tile TG * g + tg (16
// output features) of the workgroup's groups g, g + gridDim.x, ... and the
// k-blocks [ks * KPW, (ks + 1) * KPW), then every KS * KPW; the KS partial sums
// of a tile meet in LDS.  One workgroup fills a CU, so that a CU prepares the
// rows once; the next group's weights are loaded before the current group's
// MFMAs and the epilogues go round the waves, so that it always has weights in
// flight.
#include <algorithm>
#include <type_traits>

#include "convrot_device.h"
#include "convrot_launch.h"
#include "prep_device.h"

namespace convrot {
namespace {

constexpr int kMaxRows = 16;   // token rows: one MFMA column each
constexpr int kRowPad = 16;    // bytes of padding after an LDS row

typedef unsigned int u32x4r __attribute__((ext_vector_type(4)));

// Four rotated values of x's type, at element f of an LDS row.
template <int DT>
__device__ __forceinline__ void lds_store4(uint8_t* row, int f, const float* v) {
  if constexpr (DT == kF32) *(float4*)(row + 4 * f) = make_float4(v[0], v[1], v[2], v[3]);
  else if constexpr (DT == kBF16) *(uint2*)(row + 2 * f) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  else *(uint2*)(row + 2 * f) = make_uint2(pack_f16x2(v[0], v[1]), pack_f16x2(v[2], v[3]));
}

// LDS of a launch (dynamic), in order: the rotated rows (x's type, kRowPad
// after each, padded to whole 128-feature blocks), for A4 the code rows, then
// the waves' exchange buffers and, once the rows are rotated, the two buffers
// of their partial sums.
struct RowsLds {
  int rot_stride, code_stride;  // bytes of a row
  int codes, work;              // byte offsets
  int bytes;
};

inline RowsLds rows_lds(int64_t M, int64_t kblocks, int esize, bool a4, int waves) {
  RowsLds l;
  l.rot_stride = (int)(kblocks * 128 * esize + kRowPad);
  l.code_stride = (int)(kblocks * 128 + kRowPad);
  l.codes = (int)M * l.rot_stride;
  l.work = l.codes + (a4 ? (int)M * l.code_stride : 0);
  l.bytes = l.work + std::max(waves * kRegionFloats * 4, 2 * waves * 1024);
  return l;
}

template <int DT, int S, bool A4, int TG, int KS, int KPW>
__global__ __launch_bounds__(TG* KS * 64) __attribute__((amdgpu_waves_per_eu(4)))
void linear_rows_kernel(const void* __restrict__ x, const uint8_t* __restrict__ wq,
                        const float* __restrict__ wscales, const float* __restrict__ bias, void* __restrict__ out,
                        int M, int N, int K, int nblocks, int kblocks, int groups, RowsLds lay, GatedResidual gr) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  using Acc = typename std::conditional<A4, i32x4, f32x4>::type;
  __shared__ uint32_t row_max[kMaxRows];
  __shared__ float row_xs[kMaxRows];
  constexpr int kThreads = TG * KS * 64;
  constexpr int kEsize = DT == kF32 ? 4 : 2;
  constexpr int G = 1 << (2 * S), LG = G / 16;  // features and lanes of a group
  constexpr float kNorm = 1.0f / (float)(1 << S);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tg = wave / KS, ks = wave % KS;
  const int q = lane >> 4, r = lane & 15;

  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      (void*)wq, (short)0, (int)((int64_t)kblocks * nblocks * 1024), 0x00020000);
  // k-blocks at or past kblocks read zeros (past the buffer); a tile past the
  // last one reads the next k-block's first (its outputs are not stored)
  auto load_w = [&](int g, int kb0, uint4 (&w)[KPW]) {
#pragma unroll
    for (int i = 0; i < KPW; ++i) {
      const uint32_t off = (uint32_t)(kb0 + i) * (uint32_t)nblocks + (uint32_t)(g * TG + tg);
      const u32x4r v = __builtin_amdgcn_raw_buffer_load_b128(
          rw, (int)((kb0 + i < kblocks ? off * 1024u + (uint32_t)lane * 16u : 0x80000000u)), 0, 0);
      w[i] = make_uint4(v.x, v.y, v.z, v.w);
    }
  };
  // the epilogue wave's weight scales and bias, 4 features a lane
  float ws[4], bs[4];
  auto load_epi = [&](int g) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = min((g * TG + tg) * 16 + 4 * q + j, N - 1);
      ws[j] = wscales[n];
      bs[j] = bias ? bias[n] : 0.0f;
    }
  };

  int g = blockIdx.x, kb0 = ks * KPW, turn = 0;
  uint4 w[KPW];
  load_w(g, kb0, w);
  if (ks == 0) load_epi(g);

  // ---- preparation: rotated rows in LDS, then their codes
  if (A4 && threadIdx.x < kMaxRows) row_max[threadIdx.x] = 0;
  if constexpr (!A4) {  // zeros past K: the weights there are zero, the product must be too
    for (int i = K + (int)threadIdx.x; i < kblocks * 128; i += kThreads)
      for (int m = 0; m < M; ++m) *(uint16_t*)(smem + m * lay.rot_stride + 2 * i) = 0;
  }
  if constexpr (A4) __syncthreads();
  const int chunks = K >> 4, blocks = (chunks + 63) >> 6;
  float* region = (float*)(smem + lay.work) + wave * kRegionFloats + (lane / LG) * (G + G / 4);
  const int p = lane % LG;
  for (int u = wave; u < M * blocks; u += TG * KS) {
    const int m = u / blocks, block = u - m * blocks, chunk = block * 64 + lane;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const char*)x + (int64_t)m * K * kEsize), (short)0, K * kEsize, 0x00020000);
    float v[16];
    load16<DT>(xr, (uint32_t)chunk * (16u * kEsize), v);  // past the row end: zeros
    rotate16<DT, S>(v, region, p);
    if constexpr (!A4 || DT != kBF16) {  // bf16 codes take the factor in the scale
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = rnd<DT>(v[j] * kNorm);
    }
    if constexpr (A4) {
      float amax = 0.0f;
#pragma unroll
      for (int j = 0; j < 16; j += 2) amax = absmax3(amax, v[j], v[j + 1]);
      amax = wave_max_nonneg(amax);
      if (lane == 0) atomicMax(&row_max[m], __float_as_uint(amax));  // non-negative: ordered as integers
    }
    if (chunk < chunks) {
      uint8_t* row = smem + m * lay.rot_stride;
      const int f0 = block * 1024 + (lane / LG) * G;
#pragma unroll
      for (int run = 0; run < 4; ++run) lds_store4<DT>(row, f0 + run_index<S, S - 1>(p, run), &v[4 * run]);
    }
  }
  __syncthreads();
  if constexpr (A4) {
    for (int m = 0; m < M; ++m) {
      const RowScale<DT> sc = row_scale<DT>(__uint_as_float(row_max[m]), kNorm);
      if (threadIdx.x == 0) row_xs[m] = sc.scale;
      const uint8_t* row = smem + m * lay.rot_stride;
      uint32_t* codes = (uint32_t*)(smem + lay.codes + m * lay.code_stride);
      for (int i = threadIdx.x; i < K / 4; i += kThreads) {
        float v[4];
        load_elem4<DT>(row, 4 * i, v);
        codes[i] = gather_bytes(code_bits(code_ratio<DT>(v[0], sc)), code_bits(code_ratio<DT>(v[1], sc)),
                                code_bits(code_ratio<DT>(v[2], sc)), code_bits(code_ratio<DT>(v[3], sc)));
      }
    }
    __syncthreads();
  }

  // ---- weight stream
  const int mrow = r < M ? r : M - 1;  // columns past M repeat the last row and are not stored
  const uint8_t* arow = smem + (A4 ? lay.codes + mrow * lay.code_stride : mrow * lay.rot_stride);
  Acc acc = {};
  for (;;) {
    int g2 = g, kn = kb0 + KS * KPW;
    // uniform over the workgroup: the batch of the last k-block, whatever the wave's share of it
    const bool last = kn - ks * KPW >= kblocks;
    if (last) g2 = g + (int)gridDim.x, kn = ks * KPW;
    const bool more = g2 < groups;
    uint4 wn[KPW];
    if (more) load_w(g2, kn, wn);
#pragma unroll
    for (int i = 0; i < KPW; ++i) {
      if (kb0 + i >= kblocks) break;  // wave-uniform
      const uint32_t wd[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
#pragma unroll
      for (int c = 0; c < (A4 ? 2 : 4); ++c) {
        const i32x4 a = *(const i32x4*)(arow + (kb0 + i) * (A4 ? 128 : 256) + (A4 ? 32 : 64) * q + 16 * c);
        if constexpr (A4) {
          uint32_t l0, h0, l1, h1;
          nibbles_x16(wd[2 * c], l0, h0);
          nibbles_x16(wd[2 * c + 1], l1, h1);
          acc = __builtin_amdgcn_mfma_i32_16x16x64_i8((i32x4){(int)l0, (int)h0, (int)l1, (int)h1}, a, acc, 0, 0, 0);
        } else {
          acc = mfma16<DT>(expand8<DT>(wd[c]), a, acc);
        }
      }
    }
    if (last) {
      // partial sums through one of two buffers: a wave reaches the barrier of
      // the group after next only when this group's epilogue is done
      Acc(*buf)[64] = (Acc(*)[64])(smem + lay.work) + (turn & 1) * TG * KS;
      buf[wave][lane] = acc;
      acc = Acc{};
      __syncthreads();
      if (ks == turn % KS && r < M) {
        Acc s = buf[tg * KS][lane];
#pragma unroll
        for (int w2 = 1; w2 < KS; ++w2) s += buf[tg * KS + w2][lane];
        const int n = (g * TG + tg) * 16 + 4 * q;
        if (n < N) {
          const float xs = A4 ? row_xs[r] : 1.0f;
          float o[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if constexpr (A4) o[j] = (((float)(s[j] >> 4) * xs) * ws[j]) + bs[j];
            else o[j] = s[j] * (ws[j] * 0.0625f) + bs[j];  // codes were scaled by 16
          }
          const bool vec_ok = (N & 3) == 0;
          if (gr.residual) gate_residual4<DT>(gr, r, n, N, vec_ok, o);
          const int64_t idx = (int64_t)r * N + n;
          if (vec_ok) {
            store_out4<DT>(out, idx, o[0], o[1], o[2], o[3]);
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (n + j < N) store_out<DT>(out, idx + j, o[j]);
          }
        }
      }
      ++turn;
      if (more && ks == turn % KS) load_epi(g2);
    }
    if (!more) break;
    g = g2, kb0 = kn;
#pragma unroll
    for (int i = 0; i < KPW; ++i) w[i] = wn[i];
  }
}

template <int DT, int S, bool A4, int TG, int KS, int KPW>
hipError_t launch_rows_t(const void* x, const uint8_t* wq, const float* ws, const float* bias, int64_t M, int64_t N,
                         int64_t K, void* out, const GatedResidual& gr, hipStream_t stream) {
  const int nblocks = (int)((N + 15) / 16), kblocks = (int)((K + 127) / 128);
  const int groups = (nblocks + TG - 1) / TG;
  const RowsLds lay = rows_lds(M, kblocks, DT == kF32 ? 4 : 2, A4, TG * KS);
  hipLaunchKernelGGL((linear_rows_kernel<DT, S, A4, TG, KS, KPW>), dim3((unsigned)std::min(groups, device_cus())),
                     dim3(64 * TG * KS), (size_t)lay.bytes, stream, x, wq, ws, bias, out, (int)M, (int)N, (int)K,
                     nblocks, kblocks, groups, lay, gr);
  return hipGetLastError();
}

// Tiles a workgroup and waves a tile (TG, KS, KPW).  The choice is the least of
//   rounds of workgroups over the CUs x (k-blocks a CU loads in a round + 24),
// the loaded blocks counted whole batches of KS * KPW, and 24 for what a round
// costs besides: as many tiles a workgroup as make one round (a CU prepares the
// rows once), but no batch that is mostly past K.  At M = 1 it is within 1.6 % of
// the best of the five at each of 27 shapes timed but one (5 %).  Measured at M = 1,
// bf16, the preparation and GEMM launches against this one (HIP-graph replays
// over > 256 MB of weights, us):
//   K -> N         W4A4             W4A16            tiles, (TG, KS, KPW)
//   3072 -> 3072    6.31 ->  5.01    6.66 ->  5.22     192  (1, 8, 3)
//   3072 -> 6144    7.22 ->  5.66    7.52 ->  6.32     384  (2, 8, 3)
//   3072 -> 9216    8.18 ->  6.50    9.47 ->  7.61     576  (3, 5, 5)
//   3072 -> 12288   9.82 ->  7.62   10.23 ->  8.53     768  (3, 5, 5)
//   3072 -> 18432  12.91 ->  9.32   12.94 -> 10.62    1152  (5, 3, 8)
//   3072 -> 21504  14.06 -> 10.91   14.36 -> 12.67    1344  (3, 5, 5), two rounds
//   6144 -> 16384  14.07 -> 12.99   15.57 -> 15.26    1024  (2, 8, 3), two rounds
//   12288 -> 3072  10.83 ->  9.48   12.40 -> 10.79     192  (1, 16, 3)
//   16384 -> 9216  25.73 -> 19.42   31.64 -> 25.19     576  (3, 5, 5)
// The next choice loses 3-15 % in each row.  What is left above the weights'
// 2.8 us (9216: 14.2 MB) is the launch, the row's load and the rotation and
// quantization before the first MFMA (~2.5 us).
struct RowsSplit {
  int cfg, tg, ks, kpw;
};
constexpr RowsSplit kRowsSplits[] = {{5, 5, 3, 8}, {3, 3, 5, 5}, {2, 2, 8, 3}, {1, 1, 8, 3}, {16, 1, 16, 3}};

int rows_split(int64_t N, int64_t K, bool a4) {
  if (const int v = tuning(kTuneRowsCfg); v >= 0) return v;
  const int64_t nblocks = (N + 15) / 16, kblocks = (K + 127) / 128, cus = device_cus();
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (const RowsSplit& c : kRowsSplits) {
    const int64_t groups = (nblocks + c.tg - 1) / c.tg;
    if (c.cfg == 1 && groups > cus) continue;  // two tiles a workgroup load as much in fewer rounds
    const int64_t rounds = (groups + cus - 1) / cus;
    const int64_t batches = (kblocks + c.ks * c.kpw - 1) / (c.ks * c.kpw);
    const int64_t cost = rounds * (batches * c.tg * c.ks * c.kpw + 24);
    // ties: one tile a workgroup, sixteen waves on a long K (8192 -> 2048: 7.03 against 7.14); W4A16 of 769
    // to 1024 tiles, two rounds of two tiles on sixteen waves instead of one of five on fifteen, to expand the
    // weights (3072 -> 14336, M = 1 9.66 against 9.89, M = 3 10.5 against 11.1; 2304 -> 14336 9.66 against 9.48)
    const bool wide = c.cfg == 2 && best == 5 && !a4 && K >= 2560 && nblocks <= 4 * cus;
    const bool tie = cost == best_cost && ((c.cfg == 16 && K > 6144) || wide);
    if (cost < best_cost || tie) best = c.cfg, best_cost = cost;
  }
  return best;
}

template <int DT, int S, bool A4>
hipError_t launch_rows_nb(const void* x, const uint8_t* wq, const float* ws, const float* bias, int64_t M, int64_t N,
                          int64_t K, void* out, const GatedResidual& gr, hipStream_t stream) {
  switch (rows_split(N, K, A4)) {
    case 16: return launch_rows_t<DT, S, A4, 1, 16, 3>(x, wq, ws, bias, M, N, K, out, gr, stream);
    case 1: return launch_rows_t<DT, S, A4, 1, 8, 3>(x, wq, ws, bias, M, N, K, out, gr, stream);
    case 2: return launch_rows_t<DT, S, A4, 2, 8, 3>(x, wq, ws, bias, M, N, K, out, gr, stream);
    case 5: return launch_rows_t<DT, S, A4, 5, 3, 8>(x, wq, ws, bias, M, N, K, out, gr, stream);
    default: return launch_rows_t<DT, S, A4, 3, 5, 5>(x, wq, ws, bias, M, N, K, out, gr, stream);
  }
}

template <int DT, bool A4>
hipError_t launch_rows_s(int s, const void* x, const uint8_t* wq, const float* ws, const float* bias, int64_t M,
                         int64_t N, int64_t K, void* out, const GatedResidual& gr, hipStream_t stream) {
  return s == 3 ? launch_rows_nb<DT, 3, A4>(x, wq, ws, bias, M, N, K, out, gr, stream)
                : launch_rows_nb<DT, 4, A4>(x, wq, ws, bias, M, N, K, out, gr, stream);
}

}  // namespace

// 32 KB of rows: one row of any length this library's models have, and LDS
// left for the exchanges.  How many rows are still worth it is the caller's
// choice (ConvRotLinear's rule is beside LINEAR_ROWS_MAX in core.py).
bool linear_rows_eligible(int64_t M, int64_t K, int dtype, int log4g, bool a4) {
  const int64_t esize = dtype == kF32 ? 4 : 2;
  return M >= 1 && M <= kMaxRows && (log4g == 3 || log4g == 4) && (a4 || dtype != kF32) && K % 32 == 0 &&
         M * K * esize <= 32768;
}

hipError_t launch_linear_rows(const void* x, int dtype, int log4g, bool a4, const uint8_t* qweight,
                              const float* wscales, const float* bias, int64_t M, int64_t N, int64_t K, void* out,
                              const GatedResidual& gr, hipStream_t stream) {
  if (M == 0 || N == 0) return hipSuccess;
  if (!linear_rows_eligible(M, K, dtype, log4g, a4)) return hipErrorInvalidValue;
  if (a4) {
    switch (dtype) {
      case kF32: return launch_rows_s<kF32, true>(log4g, x, qweight, wscales, bias, M, N, K, out, gr, stream);
      case kF16: return launch_rows_s<kF16, true>(log4g, x, qweight, wscales, bias, M, N, K, out, gr, stream);
      default: return launch_rows_s<kBF16, true>(log4g, x, qweight, wscales, bias, M, N, K, out, gr, stream);
    }
  }
  return dtype == kF16 ? launch_rows_s<kF16, false>(log4g, x, qweight, wscales, bias, M, N, K, out, gr, stream)
                       : launch_rows_s<kBF16, false>(log4g, x, qweight, wscales, bias, M, N, K, out, gr, stream);
}

}  // namespace convrot
