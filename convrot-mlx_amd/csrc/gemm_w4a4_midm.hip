// W4A4 GEMM for tens to a few hundred token rows on gfx950: blocked int8 A4
// codes x packed signed int4 weights on 16x16x64 i8 MFMA, exact int32 sums,
// the tiled kernels' epilogue ((f(dot) * xs) * ws) + bias.
//
// Serves ConvRotLinear between the few-row kernel and the FP6 tiles (the
// reference's mpp_w4a4_int8_matmul, /root/reference/src/convrot_mlx/
// core.py:1088-1120, on the same codes).  A 128 x 128 tile there makes N / 128
// workgroups of one row tile, each walking K alone: 77 x 3072 -> 3072 ran 24
// workgroups on 256 CUs.  Here a workgroup takes 16 * NB output features of
// all its rows and its eight waves split K, so that the weights stream through
// every CU at once and each byte of them once; the price is that every
// workgroup reads the codes, from L2.  CONVROT_PREP_INT8_BLOCKED therefore
// lays them out as the MFMA reads them: a wave's load is 1 KB in a row (row-major
// codes would give each lane its own cache access, 4 lanes to 64 bytes).
#include "convrot_device.h"
#include "convrot_launch.h"

namespace convrot {
namespace {

constexpr int kWaves = 8;

typedef unsigned int u32x4m __attribute__((ext_vector_type(4)));

template <int FM, int NB>
struct Operands {
  i32x4 a[FM][2];
  uint4 w[NB];
};

// A workgroup owns NB weight tiles (16 features) and FM token tiles (16 rows);
// wave w multiplies k-blocks w, w + 8, ...  Blocks past the last row tile or
// weight tile read the next k-block's, or zeros past the end: rows and columns
// that are not stored.  K past its end within a k-block: the weights are zero.
template <int ODT, int FM, int NB>
__global__ __launch_bounds__(kWaves * 64) void w4a4_midm_kernel(
    const uint8_t* __restrict__ act, const float* __restrict__ xscales, const uint8_t* __restrict__ wq,
    const float* __restrict__ wscales, const float* __restrict__ bias, void* __restrict__ out, int M, int N,
    int mblocks, int nblocks, int kblocks, GatedResidual gr) {
  constexpr int NF = NB * FM, PER = (NF + kWaves - 1) / kWaves;  // fragments, and a wave's share of the epilogue
  __shared__ __attribute__((aligned(16))) i32x4 red[kWaves][NF][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nb0 = blockIdx.x * NB, mb0 = blockIdx.y * FM;
  const int q = lane >> 4, r = lane & 15;

  // the epilogue's scales and bias, before the weights: their round trip is over when the sums are
  float xs[PER], ws[PER][4], bs[PER][4];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int f = wave + i * kWaves, t = f / FM, fm = f % FM;
    xs[i] = xscales[min((mb0 + fm) * 16 + r, M - 1)];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = min((nb0 + t) * 16 + 4 * q + j, N - 1);
      ws[i][j] = wscales[n];
      bs[i][j] = bias ? bias[n] : 0.0f;
    }
  }

  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      (void*)act, (short)0, (int)((uint32_t)kblocks * (uint32_t)mblocks * 2048u), 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      (void*)wq, (short)0, (int)((uint32_t)kblocks * (uint32_t)nblocks * 1024u), 0x00020000);
  auto load = [&](int kb, Operands<FM, NB>& o) {
    const uint32_t ao = ((uint32_t)kb * (uint32_t)mblocks + (uint32_t)mb0) * 2048u + (uint32_t)lane * 16u;
    const uint32_t wo = ((uint32_t)kb * (uint32_t)nblocks + (uint32_t)nb0) * 1024u + (uint32_t)lane * 16u;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const u32x4m v = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)(wo + 1024u * t), 0, 0);
      o.w[t] = make_uint4(v.x, v.y, v.z, v.w);
    }
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const u32x4m v = __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(ao + 2048u * fm + 1024u * ks), 0, 0);
        o.a[fm][ks] = (i32x4){(int)v.x, (int)v.y, (int)v.z, (int)v.w};
      }
  };
  i32x4 acc[NB][FM];
#pragma unroll
  for (int t = 0; t < NB; ++t)
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) acc[t][fm] = (i32x4){0, 0, 0, 0};
  auto multiply = [&](const Operands<FM, NB>& o) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        uint32_t l0, h0, l1, h1;
        nibbles_x16(ks ? o.w[t].z : o.w[t].x, l0, h0);
        nibbles_x16(ks ? o.w[t].w : o.w[t].y, l1, h1);
        const i32x4 b = (i32x4){(int)l0, (int)h0, (int)l1, (int)h1};
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
          acc[t][fm] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b, o.a[fm][ks], acc[t][fm], 0, 0, 0);
      }
  };

  // one k-block ahead
  int kb = wave;
  if (kb < kblocks) {
    Operands<FM, NB> o0, o1;
    load(kb, o0);
    for (;;) {
      const bool m1 = kb + kWaves < kblocks;
      if (m1) load(kb + kWaves, o1);
      multiply(o0);
      if (!m1) break;
      const bool m0 = kb + 2 * kWaves < kblocks;
      if (m0) load(kb + 2 * kWaves, o0);
      multiply(o1);
      if (!m0) break;
      kb += 2 * kWaves;
    }
  }

#pragma unroll
  for (int t = 0; t < NB; ++t)
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) red[wave][t * FM + fm][lane] = acc[t][fm];
  __syncthreads();
  const bool vec_ok = (N & 3) == 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int f = wave + i * kWaves, t = f / FM, fm = f % FM;
    if (f >= NF) continue;
    const int m = (mb0 + fm) * 16 + r, n = (nb0 + t) * 16 + 4 * q;
    if (m >= M || n >= N) continue;
    i32x4 s = red[0][f][lane];
#pragma unroll
    for (int w2 = 1; w2 < kWaves; ++w2) s += red[w2][f][lane];
    float o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (((float)(s[j] >> 4) * xs[i]) * ws[i][j]) + bs[i][j];
    if (gr.residual) gate_residual4<ODT>(gr, m, n, N, vec_ok, o);
    const int64_t idx = (int64_t)m * N + n;
    if (vec_ok) {
      store_out4<ODT>(out, idx, o[0], o[1], o[2], o[3]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < N) store_out<ODT>(out, idx + j, o[j]);
    }
  }
}

template <int ODT, int FM, int NB>
hipError_t launch_midm_t(const uint8_t* act, const float* xs, const uint8_t* wq, const float* ws, const float* bias,
                         int64_t M, int64_t N, int64_t K, void* out, const GatedResidual& gr, hipStream_t stream) {
  const int mblocks = (int)((M + 15) / 16), nblocks = (int)((N + 15) / 16), kblocks = (int)((K + 127) / 128);
  hipLaunchKernelGGL((w4a4_midm_kernel<ODT, FM, NB>),
                     dim3((unsigned)((nblocks + NB - 1) / NB), (unsigned)((mblocks + FM - 1) / FM)),
                     dim3(kWaves * 64), 0, stream, act, xs, wq, ws, bias, out, (int)M, (int)N, mblocks, nblocks,
                     kblocks, gr);
  return hipGetLastError();
}

template <int ODT>
hipError_t launch_midm_odt(const uint8_t* act, const float* xs, const uint8_t* wq, const float* ws,
                           const float* bias, int64_t M, int64_t N, int64_t K, void* out, const GatedResidual& gr,
                           hipStream_t stream) {
  int fm = 0, nb = 0;
  midm_plan(M, N, K, &fm, &nb);
#define CONVROT_MIDM(FM_, NB_) \
  if (fm == FM_ && nb == NB_) return launch_midm_t<ODT, FM_, NB_>(act, xs, wq, ws, bias, M, N, K, out, gr, stream);
  CONVROT_MIDM(2, 1) CONVROT_MIDM(2, 2) CONVROT_MIDM(2, 3) CONVROT_MIDM(2, 4) CONVROT_MIDM(3, 1)
  CONVROT_MIDM(3, 2) CONVROT_MIDM(3, 3) CONVROT_MIDM(4, 3) CONVROT_MIDM(5, 2)
#undef CONVROT_MIDM
  return hipErrorInvalidValue;
}

// Row and weight tiles of a workgroup: the least modelled time over
//   rounds x (fixed + batches x (0.211 + 0.079 FM + 0.053 FM NB)) us,
// batches = ceil(k-blocks / 8 waves), fitted to HIP-graph timings of 54 products
// (M = 6 .. 255; 1472 -> 7936, 2048 -> 2048, 3072 -> 3072 and 9216, 8192 -> 8192,
// 12288 -> 3072): its choice is 0.5 % over the best split on average, 5 % at
// worst.  Workgroups of few registers share a CU: each of the `per_cu` costs 0.7
// of the first, and hides the others' fixed time (reduction and epilogue).
struct MidmSplit {
  int fm, nb, per_cu;
  double fixed;
};
constexpr MidmSplit kMidmSplits[] = {{2, 1, 3, 0.3}, {2, 2, 2, 0.3}, {2, 3, 1, 1.2}, {2, 4, 1, 1.2}, {3, 1, 2, 0.3},
                                     {3, 2, 1, 1.2}, {3, 3, 1, 1.2}, {4, 3, 1, 1.2}, {5, 2, 1, 1.2}};

double midm_cost(const MidmSplit& s, int64_t M, int64_t N, int64_t K, int64_t cus) {
  const int64_t kblocks = (K + 127) / 128;
  const int64_t wgs = ((M + 15) / 16 + s.fm - 1) / s.fm * (((N + 15) / 16 + s.nb - 1) / s.nb);
  const int64_t full = wgs / (cus * s.per_cu), rest = wgs - full * cus * s.per_cu;
  const double shared = 1.0 + 0.7 * (s.per_cu - 1);
  const double last = rest ? 1.0 + 0.7 * (double)((rest + cus - 1) / cus - 1) : 0.0;
  const double block = 0.211 + 0.079 * s.fm + 0.053 * s.fm * s.nb;
  return ((double)full * shared + last) * (s.fixed + (double)((kblocks + kWaves - 1) / kWaves) * block);
}

// The best split and its cost.  `cus` comes from one device query: this runs on
// every call of a layer.
const MidmSplit& midm_best(int64_t M, int64_t N, int64_t K, int64_t cus, double* cost) {
  const MidmSplit* best = &kMidmSplits[0];
  *cost = midm_cost(*best, M, N, K, cus);
  for (const MidmSplit& s : kMidmSplits)
    if (const double c = midm_cost(s, M, N, K, cus); c < *cost) best = &s, *cost = c;
  return *best;
}

}  // namespace

// Whether the blocked codes are the faster form for a W4A4 product (INT8
// operands).  From 16 rows they win against the few-row kernel, which reads the
// weights once for every 16 rows (preparation and GEMM, HIP-graph replays, us:
// M = 32, 3072 -> 9216 13.8 -> 8.8, 12288 -> 3072 15.1 -> 13.4; M = 16
// 3072 -> 3072 7.5 -> 7.2), below that only where there are many weight tiles
// (M = 6, 3072 -> 9216 9.1 -> 8.3, but 12288 -> 3072 10.9 -> 12.1, M = 12,
// 16384 -> 4096 16.3 -> 17.2) and not too many (M = 5: 1024 -> 8448 6.4 -> 6.6,
// 3072 -> 9216 8.8 -> 8.0, 16384 -> 12288 28.0 -> 27.1, 16384 -> 16384 30.7 -> 32.0).
// Against the 128-row tiles, one of which walks K in ~0.47 us a k-block whatever
// M, they win until their rounds add up: M = 77, 3072 -> 3072 19.9 -> 8.5,
// 9216 19.9 -> 12.3, 12288 -> 3072 57.3 -> 17.8; M = 255, 3072 -> 3072
// 20.4 -> 11.3, 12288 -> 3072 51.4 -> 26.4; but 3072 -> 18432 M = 64
// 21.0 -> 16.9, M = 77 21.1 -> 24.4.  The model is 20 % low on many rounds, 40 %
// where a wave has one or two k-blocks (1024 -> 18432, M = 77: 11.5 -> 12.0 if
// taken) and 60 % on K past 12288 (16384 -> 16384, M = 77 56.8 -> 60.6, 16384 ->
// 8448, M = 129 59.9 -> 62.0; but 12288 -> 12288, M = 129 56.9 -> 47.4).
bool midm_preferred(int64_t M, int64_t N, int64_t K) {
  const int64_t nblocks = (N + 15) / 16, kblocks = (K + 127) / 128;
  if (M > 255 || M < 5 || N <= 0 || K <= 0) return false;
  if (tuning(kTuneMidmCfg) >= 0) return true;
  for (const TuneKey k : {kTuneGemmTile, kTuneGemmSk, kTuneGemmNoDma, kTuneGemmSmallmMax, kTuneW4a4SmallmCfg})
    if (tuning(k) >= 0) return false;  // a kernel of row-major codes is asked for
  if (M < 16) return nblocks > 512 && N * K < (1ll << 28);
  if (M <= 32 || (M <= 64 && N * K <= kSmallMWideElems)) return true;
  const int64_t cus = device_cus();
  const double tiles = (double)(((M + 127) / 128) * ((N + 127) / 128)) / (double)cus;
  const double tiled = 3.5 + 0.45 * (double)kblocks * (tiles > 1.0 ? tiles : 1.0);
  double cost = 0.0;
  midm_best(M, N, K, cus, &cost);
  const double low = kblocks < 16 ? 1.4 : kblocks > 96 ? 1.6 : 1.2;  // how far the model may be below
  return low * cost < tiled;
}

void midm_plan(int64_t M, int64_t N, int64_t K, int* fm, int* nb) {
  const int forced = tuning(kTuneMidmCfg);
  for (const MidmSplit& s : kMidmSplits)
    if (forced == 10 * s.fm + s.nb) {
      *fm = s.fm, *nb = s.nb;
      return;
    }
  double cost = 0.0;
  const MidmSplit& s = midm_best(M, N, K, device_cus(), &cost);
  *fm = s.fm, *nb = s.nb;
}

bool midm_split_known(int cfg) {
  for (const MidmSplit& s : kMidmSplits)
    if (cfg == 10 * s.fm + s.nb) return true;
  return false;
}

hipError_t launch_w4a4_midm(const uint8_t* act, const float* xscales, const uint8_t* qweight, const float* wscales,
                            const float* bias, int64_t M, int64_t N, int64_t K, void* out, int out_dtype,
                            hipStream_t stream, const GatedResidual& gr) {
  if (M == 0 || N == 0) return hipSuccess;
  switch (out_dtype) {
    case kF32: return launch_midm_odt<kF32>(act, xscales, qweight, wscales, bias, M, N, K, out, gr, stream);
    case kF16: return launch_midm_odt<kF16>(act, xscales, qweight, wscales, bias, M, N, K, out, gr, stream);
    default: return launch_midm_odt<kBF16>(act, xscales, qweight, wscales, bias, M, N, K, out, gr, stream);
  }
}

}  // namespace convrot
