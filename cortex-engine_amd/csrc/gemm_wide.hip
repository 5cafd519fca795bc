// Residual bf16 GEMM on 256 x 256 tiles for gfx950 (MLP-down with many rows):
//
//   y[m, n] = (sum_k a[m, k] w[n, k]) * w_scale[n] (+ bias[n]) + residual[m, n],  a (M, K), w (N, K) bf16 rows, fp32 out
//
// What bounds it: memory (65536 x 512 x 2048: 537 MB, 104 us at the 5.1 TB/s of a copy), the matrix cores
// (throttled by power to 1.83 PFLOP/s on random data: 75 us) and, close behind, the LDS: a K step of 64 writes 64 KiB into it and reads what the wavefronts need of it.  Eight wavefronts of
// 128 x 64 read 192 KiB per step of 2048 MFMA cycles, 125 bytes a cycle with the writes, all that the LDS
// gives; four of 128 x 128 read 128 KiB, 94.  One wavefront per SIMD then has to keep its matrix core busy by
// itself: v_mfma_f32_32x32x16_bf16 is issued at the full rate by one wavefront (16x16x32 only every 27 of its
// 16 cycles), the fragments of the next 16 of K are read between the MFMAs of this one, and so is the refill
// of the ring (two stages of 64 K).
//
// Persistent: a workgroup per CU walks its tiles in XCD order; after a tile's last step the next tile's two
// stages are issued, and land while the epilogue runs.  The epilogue takes 32 rows x 64 columns of a wavefront
// at a time through LDS of its own, so that residual and output rows move in whole 256-byte pieces and a lane's
// scale and bias columns stay the same.
//
// Against 256 x 128 tiles of eight wavefronts (repeated alone, on several GPUs): 32768 x 512 x 2048 87.6 -> 76 .. 79 us,
// 65536 x 512 x 2048 178.7 -> 160 .. 170, 36864 x 768 x 3072 225 -> 194 .. 198.  (With a bf16 output and the GELU in place of the residual, K = 512, it is the
// slower form, 205 against 216 us at 65536 x 2048 x 512: one wavefront per SIMD has nothing to overlap the
// epilogue's arithmetic with.)
#include <hip/hip_runtime.h>

#include "common.h"
#include "gemm.h"

namespace cortex {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int GW_T = 256, GW_BK = 64;
constexpr int GW_OP = GW_T * 128;           // bytes of one operand's stage (256 rows of 64 bf16)
constexpr int GW_STAGE = 2 * GW_OP;
constexpr int GW_RING = 2 * GW_STAGE;       // 128 KiB
constexpr int GW_LD = 64;                   // floats per row of the epilogue's 32 x 64 patch
constexpr int GW_PATCH = 32 * GW_LD * 4;    // 8 KiB per wavefront, 16-byte chunk c of row r at c ^ (r % 16)
constexpr int GW_LDS = GW_RING + 4 * GW_PATCH;
static_assert(GW_LDS <= 160 * 1024, "LDS");

struct WideArgs {
  int M, N, K;
  const unsigned char* x;
  uint32_t ld_x;  // bytes
  const unsigned char* w;
  uint32_t ld_w;
  const float* w_scale;
  const float* bias;
  const float* res;
  int64_t ld_res;
  int res_rows;
  void* out;
  int64_t ld_out;
  int nt, tiles;
};

__global__ __launch_bounds__(256, 1) void gemm_wide_kernel(WideArgs g) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[GW_LDS];
  const int tid = threadIdx.x, lane = tid & 63, wid = wave_uniform(tid >> 6);
  const int wm = wid >> 1, wn = wid & 1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  const int nk = g.K / GW_BK;

  // Transfers: block i of this wavefront holds rows (wid * 8 + i) * 8 + lane / 8; the 16-byte chunk c of row r lies
  // at c ^ ((r >> 1) & 7), so the 16 rows that one pass of a fragment read touches cover all bank groups.
  const int tr = wid * 64 + (lane >> 3), tc = lane & 7;
  uint32_t a_off[8], w_off[8];
  auto tile_offsets = [&](int t) __attribute__((always_inline)) {
    const int m0 = t / g.nt * GW_T, n0 = t % g.nt * GW_T;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = tr + 8 * i;
      const uint32_t c = (uint32_t)((tc ^ ((r >> 1) & 7)) * 16);
      a_off[i] = (uint32_t)min(m0 + r, g.M - 1) * g.ld_x + c;
      w_off[i] = (uint32_t)(n0 + r) * g.ld_w + c;
    }
  };
  auto issue = [&](int i, int kt, int s) __attribute__((always_inline)) {  // transfer i (0 .. 15) of stage kt
    const uint32_t to = lds0 + s * GW_STAGE + (i < 8 ? 0 : GW_OP) + (wid * 8 + (i & 7)) * 1024;
    lds_dma_m0<16>((i < 8 ? g.x : g.w) + kt * 128, i < 8 ? a_off[i & 7] : w_off[i & 7], to);
  };

  // fragment addresses inside an operand's stage: row (lane % 32) of a 32-row tile, chunk 2 q + lane / 32
  int f_off[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = lane & 31;
    f_off[q] = r * 128 + (((2 * q + (lane >> 5)) ^ ((r >> 1) & 7)) << 4);
  }
  struct Frags {
    bf16x8 a[4], w[4];
  };
  auto read = [&](int i, int s, int q, Frags& f) __attribute__((always_inline)) {  // fragment i (0 .. 7) of quarter q
    const unsigned char* p = smem + s * GW_STAGE + f_off[q];
    if (i < 4)
      f.a[i] = *reinterpret_cast<const bf16x8*>(p + (wm * 128 + 32 * i) * 128);
    else
      f.w[i - 4] = *reinterpret_cast<const bf16x8*>(p + GW_OP + (wn * 128 + 32 * (i - 4)) * 128);
  };

  f32x16 acc[4][4];  // [row tile][column tile]
  int t = xcd_affine(blockIdx.x, g.tiles);
  int next = blockIdx.x;
  tile_offsets(t);
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < 16; ++i) issue(i, s, s);

  for (;;) {
    // scale and bias of this lane's columns: 4 of each 64-column patch
    constexpr int NC = 4, LPR = 64 / NC;  // columns per lane, lanes per row
    const int m0 = t / g.nt * GW_T, n0 = t % g.nt * GW_T;
    const int pc = n0 + wn * 128 + lane % LPR * NC;
    float sc[2][NC], bi[2][NC];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int e = 0; e < NC; ++e) {
        sc[p][e] = g.w_scale ? g.w_scale[pc + 64 * p + e] : 1.0f;
        bi[p][e] = g.bias ? g.bias[pc + 64 * p + e] : 0.0f;
      }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    wait_vm<0>();
    __builtin_amdgcn_s_barrier();  // stages 0 and 1 of this tile are in LDS
    Frags f[2];
#pragma unroll
    for (int i = 0; i < 8; ++i) read(i, 0, 0, f[0]);
    for (int kt = 0; kt < nk; ++kt) {
      const int s = kt & 1;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        // Quarter 3 starts with every wavefront done reading this stage (its last fragments are in
        // registers) and the next stage landed.  The freed slot's 16 transfers go out in quarter 3
        // and in quarter 0 of the next stage, three quarters before they are waited for.
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): quarter q's fragments
        if (q == 3) {
          wait_vm<0>();
          __builtin_amdgcn_s_barrier();
        }
        const bool more = q == 3 ? kt + 2 < nk : q == 0 && kt >= 1 && kt + 1 < nk;
        const bool nxt = q < 3 || kt + 1 < nk;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          __builtin_amdgcn_sched_barrier(0);
          if (nxt) {
            read(2 * u, q < 3 ? s : s ^ 1, (q + 1) & 3, f[(q + 1) & 1]);
            read(2 * u + 1, q < 3 ? s : s ^ 1, (q + 1) & 3, f[(q + 1) & 1]);
          }
          if (more) {
            // (quarter 3: the first half of stage kt + 2 into this slot; quarter 0: the second half of stage
            // kt + 1, whose slot the stage before this one freed)
            issue((q == 3 ? 0 : 8) + 2 * u, q == 3 ? kt + 2 : kt + 1, q == 3 ? s : s ^ 1);
            issue((q == 3 ? 0 : 8) + 2 * u + 1, q == 3 ? kt + 2 : kt + 1, q == 3 ? s : s ^ 1);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[u][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[q & 1].w[j], f[q & 1].a[u], acc[u][j], 0, 0, 0);
        }
      }
    }

    // the next tile's first stages (every wavefront has its last fragments: the barrier of quarter 3)
    next += gridDim.x;
    const bool again = next < g.tiles;
    const int tn = again ? xcd_affine(next, g.tiles) : 0;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int e = 0; e < NC; ++e) asm volatile("" ::"v"(sc[p][e]), "v"(bi[p][e]));  // loaded before the transfers
    if (again) {
      tile_offsets(tn);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 16; ++i) issue(i, s, s);
    }

    float* patch = reinterpret_cast<float*>(smem + GW_RING + wid * GW_PATCH);
    constexpr int RPI = 64 / LPR;  // rows per pass of the wavefront
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int mp = m0 + wm * 128 + 32 * i;
        float4 rv[32 / RPI];
#pragma unroll
        for (int x = 0; x < 32 / RPI; ++x) {
          const int m = min(mp + x * RPI + lane / LPR, g.M - 1);
          rv[x] = *reinterpret_cast<const float4*>(
              g.res + (int64_t)(g.res_rows > 0 ? m % g.res_rows : m) * g.ld_res + pc + 64 * p);
        }
        // lane: row lane % 32, columns 32 j + 8 b + 4 (lane / 32) .. +3 of the patch
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const f32x16& v = acc[i][2 * p + j];
            *reinterpret_cast<f32x4*>(patch + (lane & 31) * GW_LD + ((8 * j + 2 * b + (lane >> 5)) ^ (lane & 15)) * 4) =
                (f32x4){v[4 * b], v[4 * b + 1], v[4 * b + 2], v[4 * b + 3]};
          }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the patch is this wavefront's own)
#pragma unroll
        for (int x = 0; x < 32 / RPI; ++x) {
          const int r = x * RPI + lane / LPR, m = mp + r;
          float v[NC];
#pragma unroll
          for (int e = 0; e < NC; e += 4)
            *reinterpret_cast<f32x4*>(v + e) = *reinterpret_cast<const f32x4*>(
                patch + r * GW_LD + ((lane % LPR * (NC / 4) + e / 4) ^ (r & 15)) * 4);
#pragma unroll
          for (int e = 0; e < NC; ++e) v[e] = v[e] * sc[p][e] + bi[p][e];
          if (m < g.M)
            *reinterpret_cast<float4*>(reinterpret_cast<float*>(g.out) + (int64_t)m * g.ld_out + pc + 64 * p) =
                make_float4(v[0] + rv[x].x, v[1] + rv[x].y, v[2] + rv[x].z, v[3] + rv[x].w);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next patch overwrites it
      }
    if (!again) break;
    t = tn;
  }
}

}  // namespace

// Returns 1 when it launched, 0 when the request is outside its form, negative on error.
int try_gemm_wide(const GemmArgs& g, hipStream_t stream) {
  if (g.N % GW_T != 0 || g.K % GW_BK != 0 || g.K > (1 << 20) || g.M > 0x7fffffff - GW_T) return 0;
  // long K (at 1024 the two forms are equal, 57 us at 65500 x 256) and rounds of tiles that fill the CUs: a last round
  // of an eighth costs what it would full (24576 x 768 x 3072, 288 tiles: 163 us in the other form, 180 here)
  const int64_t tiles = cdiv(g.M, GW_T) * (g.N / GW_T);
  const int64_t ncu = cu_count();
  if (g.K < 2048 || tiles > 0x3fffffff || tiles < ncu || tiles * 4 < cdiv(tiles, ncu) * ncu * 3) return 0;
  if (g.M * g.ld_x * 2 > 0xffffffffll || g.N * g.ld_w * 2 > 0xffffffffll) return 0;
  WideArgs a = {};
  a.M = (int)g.M;
  a.N = (int)g.N;
  a.K = (int)g.K;
  a.x = reinterpret_cast<const unsigned char*>(g.x);
  a.ld_x = (uint32_t)(g.ld_x * 2);
  a.w = reinterpret_cast<const unsigned char*>(g.w);
  a.ld_w = (uint32_t)(g.ld_w * 2);
  a.w_scale = g.w_scale;
  a.bias = reinterpret_cast<const float*>(g.bias);
  a.res = reinterpret_cast<const float*>(g.res);
  a.ld_res = g.ld_res;
  a.res_rows = g.res_rows > 0 && g.res_rows < g.M ? (int)g.res_rows : 0;
  a.out = g.out;
  a.ld_out = g.ld_out;
  a.nt = (int)(g.N / GW_T);
  a.tiles = (int)tiles;
  hipLaunchKernelGGL(gemm_wide_kernel, dim3((unsigned)ncu), dim3(256), 0, stream, a);
  CORTEX_CHECK_LAUNCH("gemm_wide_kernel");
  return 1;
}

}  // namespace cortex
