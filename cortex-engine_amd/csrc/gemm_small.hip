// bf16 linears with few rows for gfx950 (one to a few samples: latency, not throughput):
//
//   y[m, n] = epi( sum_k a[m, k] w[n, k] ),  a = bf16 rows, or LayerNorm of fp32 rows rounded to bf16
//   epi: * w_scale[n] (+ bias[n]) (-> erf-GELU) (+ fp32 residual) -> bf16 | fp32
//
// What bounds it: with 256 rows a 128 x 128 tiling puts 8 to 32 workgroups on 256 CUs, each walking K
// step by step behind a barrier, and the K split that fills the chip needs a second launch for its sums;
// every launch pays its latency, not its work.  Here a workgroup owns a 32 x 32 tile (128 to 512 of them)
// and its 8 or 16 wavefronts split K: a wavefront's operands go from L2 straight into registers in MFMA order
// (16 bytes a lane), up to 4 steps of 32 K in flight at once, with no
// barrier before the one that exchanges the partial tiles through LDS.  All of K = 512 is one memory
// round trip.  The weight comes in fragment order (cortex_frag_weight): a 16-row, 32-K fragment is 1 KiB in
// one piece.  From plain rows it is 64 bytes of 16 rows, which a CU took in at 21 bytes a cycle whatever the number of
// wavefronts or the MFMA shape (256 x 512 x 2048: 9.4 us, 4.3 this way); the MLP's hidden rows are written and read
// in that order too.  (int8 rows, for weights that stay int8 in memory, are widened
// before their MFMAs: the same values in the same order, the same results.)  The price is operand traffic (every
// tile reads 32 rows of each operand, 32 MB of L2 reads at 256 x 2048 x 512), so larger row counts keep the larger
// tiles (the rule: small_linear_ok in ops.py).
//
// With LayerNorm (K up to 1024) the wavefront holds its K part of the 32 fp32 rows in registers: two
// exchanges of partial sums give mean and variance (two passes over registers), and no row kernel runs
// before.
#include <hip/hip_runtime.h>

#include "common.h"
#include "gemm.h"

namespace cortex {

namespace {

constexpr int SM_T = 32;
constexpr int SM_LD = 36;  // floats per row of a partial tile in LDS
constexpr int SM_MAXC = 4;  // 32-K steps in flight per wavefront

struct SmallArgs {
  int M, N, K;
  const void* x;
  int64_t ld_x;
  const float* gamma;
  const float* beta;
  float eps;
  int x_frag, out_frag;    // x / out in fragment order, M rounded up to 16 rows
  const void* w;           // bf16 in fragment order, or int8 rows
  int64_t ld_w;            // (int8)
  const float* w_scale;
  const float* bias;
  int act;
  const float* res;
  int64_t ld_res;
  int res_rows;
  void* out;
  int64_t ld_out;
  int mt;                  // row tiles
};

__device__ __forceinline__ float act_of(float v, int act, bool bf16_out) {
  if (act != ACT_GELU) return v;
  return bf16_out ? gelu_erf_bf16out(v) : gelu_erf(v);
}

// STEPS: the K part of a wavefront in 32-K steps, C of them in flight at a time.
// A weight fragment as loaded: bf16, or 8 int8 values widened right before their MFMAs.
template <class TW>
struct WFrag {
  bf16x8 v;
  __device__ __forceinline__ bf16x8 get() const { return v; }
};
template <>
struct WFrag<int8_t> {
  uint2 v;
  __device__ __forceinline__ bf16x8 get() const { return widen_i8x8(v); }
};

template <int NW, int STEPS, bool LN, class TOUT, class TW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 4))) void gemm_small_kernel(SmallArgs g) {
  constexpr int C = STEPS < SM_MAXC ? STEPS : SM_MAXC;
  static_assert((!LN || STEPS <= SM_MAXC), "steps");
  __shared__ __attribute__((aligned(16))) float part[NW][SM_T][SM_LD];
  __shared__ float red[2][NW][SM_T];
  const int tid = threadIdx.x, lane = tid & 63, wid = wave_uniform(tid >> 6);
  const int r = lane & 15, c8 = (lane >> 4) * 8;
  // neighbouring workgroups share the weight rows: each XCD takes a contiguous range of column tiles
  const int id = xcd_affine(blockIdx.x, gridDim.x);
  const int m0 = (id % g.mt) * SM_T, n0 = (id / g.mt) * SM_T;
  const int k0 = wid * STEPS * 32 + c8;
  const int kb = g.K >> 5, mb = (g.M - 1) >> 4, nb = (g.N - 1) >> 4;  // 32-K blocks, last 16-row blocks
  int64_t m[2];
  const TW* wp[2];
  constexpr int WS = sizeof(TW) == 1 ? 32 : 512;  // elements between 32-K steps
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    m[t] = min(m0 + 16 * t + r, g.M - 1);
    wp[t] = reinterpret_cast<const TW*>(g.w) +
            (sizeof(TW) == 1 ? min(n0 + 16 * t + r, g.N - 1) * g.ld_w + k0
                             : ((int64_t)min((n0 >> 4) + t, nb) * kb + wid * STEPS) * 512 + lane * 8);
  }
  typedef decltype(WFrag<TW>::v) wraw;

  f32x4 acc[2][2] = {};  // [row tile][column tile]
  auto multiply = [&](const bf16x8 (&a)[2], const WFrag<TW> (&wr)[2]) {
    const bf16x8 w[2] = {wr[0].get(), wr[1].get()};
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], a[i], acc[i][j], 0, 0, 0);
  };
  if constexpr (LN) {
    float v[2][STEPS][8];
    WFrag<TW> wf[STEPS][2];
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const float* xp = reinterpret_cast<const float*>(g.x) + m[t] * g.ld_x + k0 + s * 32;
        *reinterpret_cast<float4*>(v[t][s]) = *reinterpret_cast<const float4*>(xp);
        *reinterpret_cast<float4*>(v[t][s] + 4) = *reinterpret_cast<const float4*>(xp + 4);
      }
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) wf[s][t].v = *reinterpret_cast<const wraw*>(wp[t] + s * WS);
    __builtin_amdgcn_sched_barrier(0);  // every load goes out before the first wait
    float mean[2] = {0.0f, 0.0f}, rstd[2];
    const float inv_k = 1.0f / (float)g.K;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {  // the mean, then the squared deviations from it
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float u = 0.0f;
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float d = v[t][s][j] - mean[t];
            u += pass == 0 ? v[t][s][j] : d * d;
          }
        u += __shfl_xor(u, 16, 64);
        u += __shfl_xor(u, 32, 64);
        if (lane < 16) red[pass][wid][16 * t + lane] = u;
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float u = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; w += 2) u += red[pass][w][16 * t + r] + red[pass][w + 1][16 * t + r];
        if (pass == 0)
          mean[t] = u * inv_k;
        else
          rstd[t] = 1.0f / sqrtf(u * inv_k + g.eps);
      }
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      bf16x8 af[2];
#pragma unroll
      for (int j = 0; j < 8; j += 4) {
        const float4 gm = *reinterpret_cast<const float4*>(g.gamma + k0 + s * 32 + j);
        const float4 bt = *reinterpret_cast<const float4*>(g.beta + k0 + s * 32 + j);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          af[t][j] = (bf16)((v[t][s][j] - mean[t]) * rstd[t] * gm.x + bt.x);
          af[t][j + 1] = (bf16)((v[t][s][j + 1] - mean[t]) * rstd[t] * gm.y + bt.y);
          af[t][j + 2] = (bf16)((v[t][s][j + 2] - mean[t]) * rstd[t] * gm.z + bt.z);
          af[t][j + 3] = (bf16)((v[t][s][j + 3] - mean[t]) * rstd[t] * gm.w + bt.w);
        }
      }
      multiply(af, wf[s]);
    }
  } else {
    const bf16* xp[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
      xp[t] = reinterpret_cast<const bf16*>(g.x) +
              (g.x_frag ? ((int64_t)min((m0 >> 4) + t, mb) * kb + wid * STEPS) * 512 + lane * 8 : m[t] * g.ld_x + k0);
    const int xs = g.x_frag ? 512 : 32;  // elements between 32-K steps
    bf16x8 af[C][2];
    WFrag<TW> wf[C][2];
#pragma unroll
    for (int s = 0; s < C; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        af[s][t] = *reinterpret_cast<const bf16x8*>(xp[t] + s * xs);
        wf[s][t].v = *reinterpret_cast<const wraw*>(wp[t] + s * WS);
      }
    __builtin_amdgcn_sched_barrier(0);  // every load goes out before the first wait
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      multiply(af[s % C], wf[s % C]);
      if (s + C < STEPS) {  // the slot's next step: C - 1 steps are in flight behind it
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          af[s % C][t] = *reinterpret_cast<const bf16x8*>(xp[t] + (s + C) * xs);
          wf[s % C][t].v = *reinterpret_cast<const wraw*>(wp[t] + (s + C) * WS);
        }
      }
    }
  }

  // partial tiles: lane holds rows 16 i + r, columns 16 j + 4 (lane / 16) .. +3
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) *reinterpret_cast<f32x4*>(&part[wid][16 * i + r][16 * j + (lane >> 4) * 4]) = acc[i][j];
  // OPT outputs per thread; their epilogue operands load while the exchange runs
  constexpr int OPT = SM_T * SM_T / (64 * NW), TPR = SM_T / OPT;
  const int mr = tid / TPR, nc = tid % TPR * OPT;
  const int mo = m0 + mr, no = n0 + nc;
  float sc[OPT], bi[OPT] = {}, rv[OPT] = {};
#pragma unroll
  for (int e = 0; e < OPT; ++e) sc[e] = 1.0f;
  if (mo < g.M) {
#pragma unroll
    for (int e = 0; e < OPT; ++e) {
      if (no + e >= g.N) continue;
      if (g.w_scale) sc[e] = g.w_scale[no + e];
      if (g.bias) bi[e] = g.bias[no + e];
      if (g.res) rv[e] = g.res[(int64_t)(g.res_rows > 0 ? mo % g.res_rows : mo) * g.ld_res + no + e];
    }
  }
  __syncthreads();
  if (mo >= g.M) return;
  float s[OPT] = {};
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int e = 0; e < OPT; ++e) s[e] += part[w][mr][nc + e];
  // (fragment order: columns 8 q .. 8 q + 7 of a row are 16 bytes, in block (row / 16, column / 32))
  TOUT* o = reinterpret_cast<TOUT*>(g.out) +
            (g.out_frag ? ((int64_t)(mo >> 4) * (g.N >> 5) + (no >> 5)) * 512 + (((no >> 3) & 3) * 16 + (mo & 15)) * 8 + (no & 7)
                        : (int64_t)mo * g.ld_out + no);
#pragma unroll
  for (int e = 0; e < OPT; ++e) {
    float v = s[e] * sc[e];
    if (g.bias) v += bi[e];
    v = act_of(v, g.act, sizeof(TOUT) == 2);
    if (g.res) v += rv[e];
    s[e] = v;
  }
  if constexpr (OPT == 2) {
    if (no + 1 < g.N && (g.ld_out & 1) == 0 && ((uintptr_t)g.out & (2 * sizeof(TOUT) - 1)) == 0) {
      typedef TOUT pair_t __attribute__((ext_vector_type(2)));
      *reinterpret_cast<pair_t*>(o) = (pair_t){from_f32<TOUT>(s[0]), from_f32<TOUT>(s[1])};
      return;
    }
  }
#pragma unroll
  for (int e = 0; e < OPT; ++e)
    if (no + e < g.N) o[e] = from_f32<TOUT>(s[e]);
}

template <int NW, int STEPS, bool LN>
int launch_small(const SmallArgs& g, int out_dtype, int64_t tiles, hipStream_t stream) {
  const dim3 grid((unsigned)tiles), block(64 * NW);
  const bool f32 = out_dtype == DT_F32, i8 = g.ld_w > 0;
  if (f32 && i8)
    hipLaunchKernelGGL((gemm_small_kernel<NW, STEPS, LN, float, int8_t>), grid, block, 0, stream, g);
  else if (f32)
    hipLaunchKernelGGL((gemm_small_kernel<NW, STEPS, LN, float, bf16>), grid, block, 0, stream, g);
  else if (i8)
    hipLaunchKernelGGL((gemm_small_kernel<NW, STEPS, LN, bf16, int8_t>), grid, block, 0, stream, g);
  else
    hipLaunchKernelGGL((gemm_small_kernel<NW, STEPS, LN, bf16, bf16>), grid, block, 0, stream, g);
  CORTEX_CHECK_LAUNCH("gemm_small_kernel");
  return OK;
}

}  // namespace

}  // namespace cortex

using namespace cortex;

extern "C" int cortex_linear_small(int64_t M, int64_t N, int64_t K, int x_dtype, const void* x, int64_t ld_x,
                                   const float* gamma, const float* beta, float eps, int w_dtype, const void* w,
                                   int64_t ld_w, const float* w_scale, const float* bias, int act, const float* residual,
                                   int64_t ld_res, int64_t res_rows, int out_dtype, void* out, int64_t ld_out,
                                   hipStream_t stream) {
  CORTEX_CHECK_ARG(M >= 0 && N >= 0 && K >= 0, "cortex_linear_small: negative shape");
  if (M == 0 || N == 0) return OK;
  const bool ln = gamma != nullptr;
  CORTEX_CHECK_ARG(x && w && out, "cortex_linear_small: null x, w or out");
  CORTEX_CHECK_ARG(K == 256 || K == 512 || K == 768 || K == 1024 || (!ln && (K == 2048 || K == 3072)),
                   "cortex_linear_small: K must be 256, 512, 768 or 1024 (2048 or 3072 without LayerNorm)");
  CORTEX_CHECK_ARG(N % 16 == 0, "cortex_linear_small: N must be a multiple of 16");
  CORTEX_CHECK_ARG(w_dtype == DT_BF16_FRAG || (w_dtype == DT_I8 && ld_w >= K),
                   "cortex_linear_small: the weight must be bf16 in fragment order (7) or int8 rows (3)");
  CORTEX_CHECK_ARG(ln ? (x_dtype == DT_F32 && beta != nullptr)
                      : ((x_dtype == DT_BF16 || x_dtype == DT_BF16_FRAG) && beta == nullptr),
                   "cortex_linear_small: bf16 rows (also in fragment order), or fp32 rows with gamma and beta");
  CORTEX_CHECK_ARG(act == ACT_NONE || act == ACT_GELU, "cortex_linear_small: unknown activation %d", act);
  CORTEX_CHECK_ARG(out_dtype == DT_F32 || out_dtype == DT_BF16 || out_dtype == DT_BF16_FRAG,
                   "cortex_linear_small: out must be fp32 or bf16 (also in fragment order)");
  CORTEX_CHECK_ARG(out_dtype != DT_BF16_FRAG || N % 32 == 0,
                   "cortex_linear_small: rows in fragment order need N a multiple of 32");
  CORTEX_CHECK_ARG((x_dtype == DT_BF16_FRAG || ld_x >= K) && (out_dtype == DT_BF16_FRAG || ld_out >= N) &&
                       (!residual || ld_res >= N),
                   "cortex_linear_small: a row stride is smaller than its row");
  auto a16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  CORTEX_CHECK_ARG(a16(x) && (x_dtype == DT_BF16_FRAG || ld_x % (ln ? 4 : 8) == 0) &&
                       (w_dtype == DT_I8 ? ((uintptr_t)w & 7) == 0 && ld_w % 8 == 0 : a16(w)) && a16(gamma) &&
                       a16(beta) && (out_dtype != DT_BF16_FRAG || a16(out)),
                   "cortex_linear_small: operands must be 16-byte aligned rows");
  CORTEX_CHECK_ARG(M <= (1 << 20) && N <= (1 << 20) && res_rows <= (1 << 20), "cortex_linear_small: shape too large");
  SmallArgs g = {};
  g.M = (int)M;
  g.N = (int)N;
  g.K = (int)K;
  g.x = x;
  g.ld_x = ld_x;
  g.x_frag = x_dtype == DT_BF16_FRAG;
  g.out_frag = out_dtype == DT_BF16_FRAG;
  g.gamma = gamma;
  g.beta = beta;
  g.eps = eps;
  g.w = w;
  g.ld_w = w_dtype == DT_I8 ? ld_w : 0;
  g.w_scale = w_scale;
  g.bias = bias;
  g.act = act;
  g.res = residual;
  g.ld_res = ld_res;
  g.res_rows = (int)res_rows;
  g.out = out;
  g.ld_out = ld_out;
  g.mt = (int)cdiv(M, SM_T);
  const int64_t tiles = g.mt * cdiv(N, SM_T);
  CORTEX_CHECK_ARG(tiles <= 0x7fffffffLL, "cortex_linear_small: shape too large");
  switch (K) {  // 8 wavefronts, 16 where each would still have four steps and more to walk
    case 256:
      return ln ? launch_small<8, 1, true>(g, out_dtype, tiles, stream) : launch_small<8, 1, false>(g, out_dtype, tiles, stream);
    case 512:
      return ln ? launch_small<8, 2, true>(g, out_dtype, tiles, stream) : launch_small<8, 2, false>(g, out_dtype, tiles, stream);
    case 768:
      return ln ? launch_small<8, 3, true>(g, out_dtype, tiles, stream) : launch_small<8, 3, false>(g, out_dtype, tiles, stream);
    case 1024:
      return ln ? launch_small<16, 2, true>(g, out_dtype, tiles, stream) : launch_small<16, 2, false>(g, out_dtype, tiles, stream);
    case 2048: return launch_small<16, 4, false>(g, out_dtype, tiles, stream);
    default: return launch_small<16, 6, false>(g, out_dtype, tiles, stream);
  }
}
