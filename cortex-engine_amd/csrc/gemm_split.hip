// fp32 norm + linear on the bf16 matrix cores for gfx950:  y = epi( norm(x) . W^T ), fp32 in and out.
//
// An fp32 value is the exact sum of three bf16 values (split_parts.h).  A product of two fp32 operands is then
// the sum of nine bf16 products, every one exact in fp32; the three of order 2^-24 and below (a2 w3, a3 w2,
// a3 w3, unbiased: the parts' signs are independent) are left out, less than the rounding of one
// fp32 addition.  An int8 weight is a bf16 value by itself: three products, none left out.  All sums
// are fp32, in the MFMA accumulators: per 32 of K 6 accumulations of 16 products with an int8 weight and
// 12 with an fp32 one, against 8 of 4 on the fp32 MFMA, but only the leading product's are large, so the
// error against 64 bits is not larger (2-norm, N(0, 1) rows, fp32 MFMA -> here: K 512 4.0e-7 -> 2.1e-7
// with an int8 weight, 3.4e-7 with an fp32 one; K 2048 8.1e-7 -> 4.2e-7 and 7.0e-7).
//
// At the bottom of the range it is larger: an operand value below 2^-110 is off by up to 2^-134, half of
// bf16's smallest step (its parts are not flushed, but end there), where the fp32 MFMA kept its 24 bits.
// N(0, 1) rows scaled by 2^-110: 1.7e-7, as unscaled; by 2^-114 5.8e-7, 2^-118 8.8e-6, 2^-126 2.2e-3 (the
// fp32 MFMA 2.8e-7 throughout).  Beside values near 1 that is far below their rounding.
//
// What bounds it.  v_mfma_f32_16x16x4_f32 gives 157 TFLOP/s, v_mfma_f32_16x16x32_bf16 2.5 PFLOP/s:
// six products of the latter are 2.6 times, three 5.3 times the former's rate.  The operand refill
// of a 128 x 128 tile is 48 KiB (24 + 8 with an int8 weight) per 96 (48) MFMAs of a wavefront, half
// of a bf16 GEMM's per MFMA, since every fragment read from LDS is used up to six times.  The matrix
// cores, throttled by power, give 1.83 PFLOP/s on random data (a loop of MFMAs on registers); at 8192 x
// 512 x 2048 this kernel runs at 1.2 PFLOP/s of bf16 products with an fp32 weight, with int8 and a residual at 0.83.
//
// Two launches.  split_prep_kernel applies the norm (statistics computed on the spot) and writes
// the parts of the rows and of the weight as planes in MFMA fragment order: per 32 rows and 16 of
// K one 1 KiB block a plane, lane l's 8 values (row l % 32, K 8 (l / 32) ..) at 16 l.  So the GEMM's
// direct-to-LDS transfers and its fragment reads are linear, without a swizzle or a bank conflict,
// and no column tile repeats the norm or the split.  Rows go in chunks that the caller's workspace
// holds; the weight's planes are written with the first chunk.
#include <hip/hip_runtime.h>

#include "common.h"
#include "gemm.h"
#include "split_parts.h"

namespace cortex {

namespace {

constexpr int SP_BLK = 1024;  // bytes of one plane's 32 x 16 block
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct SplitArgs {
  int64_t M, N, K, KB;       // rows of this chunk, columns, depth, 32-K blocks
  const float* x;            // first row of the chunk
  int64_t ld_x;
  int norm;
  const void* gamma;
  const void* beta;
  int gamma_dtype;
  float eps;
  int x_vec, g_vec;          // 16-byte aligned rows of x; fp32 16-byte aligned gamma and beta
  const void* w;
  int w_dtype, w_layout, w_vec;
  int64_t ld_w;
  unsigned char* a_planes;   // [32-row block][32-K block][16-K half][3][1 KiB]
  unsigned char* w_planes;   // [32-column block][32-K block][16-K half][1 | 3][1 KiB]
  int64_t rb, nb;            // 32-row blocks, 32-column blocks
  int64_t w_blocks;          // prep workgroups for the weight (0: its planes are there already)
  const float* w_scale;
  const float* bias;
  int act;
  const float* res;
  int64_t ld_res, res_rows, m_base;  // m_base: row of the whole call that this chunk starts at
  float* out;
  int64_t ld_out;
  int mt, nt;                // output tiles
};

__device__ __forceinline__ float load_param(const void* p, int dtype, int64_t i) {
  if (dtype == DT_BF16) return (float)reinterpret_cast<const bf16*>(p)[i];
  if (dtype == DT_F16) return (float)reinterpret_cast<const f16*>(p)[i];
  return reinterpret_cast<const float*>(p)[i];
}

// the parts of a lane's 16 values of one 32-K block: two 16-K blocks of three planes each
__device__ __forceinline__ void put_planes(unsigned char* dst, const float (&v)[16], int lane) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const Parts s = split8<true>(v + h * 8);
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8*>(dst + (h * 3 + q) * SP_BLK + lane * 16) = s.p[q];
  }
}

// Lane l of every wavefront works on row l % 32, K 8 (l / 32) and 16 + 8 (l / 32) of a 32-K block.  Bound
// by memory: 4 bytes read and 6 written per element of x, in whole 128-byte segments and 1 KiB
// blocks.  A workgroup takes 32 rows of the weight, or of x without a norm, and SP_KC 32-K blocks of
// them (every load in flight before the first use), and with a norm 32 whole rows, held in
// registers up to K = 1024 (a longer row is read again for each pass).
constexpr int SP_PW = 8;    // wavefronts of a prep workgroup
constexpr int SP_KC = 16;   // 32-K blocks of a workgroup: two per wavefront
constexpr int SP_KEEP = 4;  // 32-K blocks per wavefront held in registers

__device__ __forceinline__ void load_f32x8(const float* p, float (&v)[8]) {
  const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

// the lane's values of 32-K block kb of one row (element stride step): k .. k + 7 and k + 16 .. k + 23 with
// k = 32 kb + c8, zero past the row's end.  fast (uniform): an aligned block inside the matrix; the
// branch on it stays scalar, so that no load waits for another path's write to its registers.
__device__ __forceinline__ void load_row16(const float* row, int64_t step, int kb, int c8, int K, bool ok, bool fast,
                                           float (&v)[16]) {
  if (fast) {
    const float* p = row + kb * 32 + c8;
    load_f32x8(p, *reinterpret_cast<float(*)[8]>(v));
    load_f32x8(p + 16, *reinterpret_cast<float(*)[8]>(v + 8));
  } else {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int k = kb * 32 + (j >> 3) * 16 + c8 + (j & 7);
      v[j] = ok && k < K ? row[k * step] : 0.0f;
    }
  }
}
__device__ __forceinline__ int k_of(int kb, int c8, int j) { return kb * 32 + (j >> 3) * 16 + c8 + (j & 7); }

__global__ __launch_bounds__(64 * SP_PW) void split_prep_kernel(SplitArgs g) {
  __shared__ float red[2][SP_PW][32];
  const int tid = threadIdx.x, lane = tid & 63, wid = wave_uniform(tid >> 6);
  const int r = lane & 31, c8 = (lane >> 5) * 8;
  const int K = (int)g.K, KB = (int)g.KB, kc = (KB + SP_KC - 1) / SP_KC;
  const bool weight = (int64_t)blockIdx.x < g.w_blocks;
  if (weight || g.norm == NORM_NONE) {
    const int64_t id = weight ? blockIdx.x : blockIdx.x - g.w_blocks;
    const int64_t blk = id / kc, n = blk * 32 + r;
    const int kb0 = (int)(id % kc) * SP_KC + wid;
    const int64_t rows = weight ? g.N : g.M;
    const bool ok = n < rows, whole = blk * 32 + 32 <= rows;
    const int64_t row = ok ? n : 0;
    constexpr int NB = SP_KC / SP_PW;
    if (weight && g.w_dtype == DT_I8) {
      const int8_t* p = reinterpret_cast<const int8_t*>(g.w) + row * g.ld_w;
      uint2 raw[NB][2];
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int kb = kb0 + SP_PW * i, k = kb * 32 + h * 16 + c8;
          if (g.w_vec && whole && kb * 32 + 32 <= K) {
            raw[i][h] = *reinterpret_cast<const uint2*>(p + k);
          } else {
            int8_t q[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = ok && k + j < K ? p[k + j] : (int8_t)0;
            raw[i][h] = __builtin_bit_cast(uint2, q);
          }
        }
#pragma unroll
      for (int i = 0; i < NB; ++i)
        if (kb0 + SP_PW * i < KB)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            *reinterpret_cast<bf16x8*>(g.w_planes + ((blk * KB + kb0 + SP_PW * i) * 2 + h) * SP_BLK + lane * 16) =
                widen_i8x8(raw[i][h]);
      return;
    }
    const bool kn = weight && g.w_layout == 1;
    const float* p = weight ? reinterpret_cast<const float*>(g.w) + (kn ? row : row * g.ld_w) : g.x + row * g.ld_x;
    const int64_t step = kn ? g.ld_w : 1;
    const bool vec = weight ? g.w_vec && !kn : g.x_vec;
    float v[NB][16];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int kb = kb0 + SP_PW * i;
      load_row16(p, step, kb, c8, K, ok, vec && whole && kb * 32 + 32 <= K, v[i]);
    }
    unsigned char* dst = weight ? g.w_planes : g.a_planes;
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (kb0 + SP_PW * i < KB) put_planes(dst + (blk * KB + kb0 + SP_PW * i) * 6 * SP_BLK, v[i], lane);
    return;
  }

  const int64_t rb = (int64_t)blockIdx.x - g.w_blocks, m = rb * 32 + r;
  const bool ok = m < g.M, fast = g.x_vec && rb * 32 + 32 <= g.M;
  const float* row = g.x + (ok ? m : 0) * g.ld_x;
  unsigned char* dst = g.a_planes + rb * KB * 6 * SP_BLK;
  auto load = [&](int kb, float (&v)[16]) { load_row16(row, 1, kb, c8, K, ok, fast && kb * 32 + 32 <= K, v); };
  float keep[SP_KEEP][16];
#pragma unroll
  for (int i = 0; i < SP_KEEP; ++i)
    if (wid + SP_PW * i < KB) load(wid + SP_PW * i, keep[i]);
  auto row_sum = [&](int slot, auto&& term) {  // sum over the row of term(value), in every lane of the row
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < SP_KEEP; ++i) {
      const int kb = wid + SP_PW * i;
      if (kb < KB) {
#pragma unroll
        for (int j = 0; j < 16; ++j) s += k_of(kb, c8, j) < K ? term(keep[i][j]) : 0.0f;
      }
    }
    for (int kb = wid + SP_PW * SP_KEEP; kb < KB; kb += SP_PW) {
      float v[16];
      load(kb, v);
#pragma unroll
      for (int j = 0; j < 16; ++j) s += k_of(kb, c8, j) < K ? term(v[j]) : 0.0f;
    }
    s += __shfl_xor(s, 32, 64);
    if (lane < 32) red[slot][wid][lane] = s;
    __syncthreads();
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < SP_PW; w += 2) t += red[slot][w][r] + red[slot][w + 1][r];
    return t;
  };
  const float inv_k = 1.0f / (float)K;
  float mean = 0.0f, st;
  if (g.norm == NORM_LAYER) {
    mean = row_sum(0, [](float v) { return v; }) * inv_k;
    const float var = row_sum(1, [mean](float v) { return (v - mean) * (v - mean); }) * inv_k;
    st = 1.0f / sqrtf(var + g.eps);
  } else {
    st = sqrtf(row_sum(0, [](float v) { return v * v; }) * inv_k + g.eps);
  }
  auto put = [&](int kb, const float (&x)[16]) {
    float gm[16], bt[16], v[16];
    if (g.g_vec && kb * 32 + 32 <= K) {
      load_row16(reinterpret_cast<const float*>(g.gamma), 1, kb, c8, K, true, true, gm);
      if (g.beta) load_row16(reinterpret_cast<const float*>(g.beta), 1, kb, c8, K, true, true, bt);
    } else {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int k = k_of(kb, c8, j);
        gm[j] = k < K ? load_param(g.gamma, g.gamma_dtype, k) : 0.0f;
        bt[j] = g.beta && k < K ? load_param(g.beta, g.gamma_dtype, k) : 0.0f;
      }
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      if (g.norm == NORM_LAYER)
        v[j] = (x[j] - mean) * st * gm[j] + (g.beta ? bt[j] : 0.0f);
      else
        v[j] = (x[j] / st) * gm[j];
      if (!ok || k_of(kb, c8, j) >= K) v[j] = 0.0f;
    }
    put_planes(dst + (int64_t)kb * 6 * SP_BLK, v, lane);
  };
#pragma unroll
  for (int i = 0; i < SP_KEEP; ++i)
    if (wid + SP_PW * i < KB) put(wid + SP_PW * i, keep[i]);
  for (int kb = wid + SP_PW * SP_KEEP; kb < KB; kb += SP_PW) {
    float v[16];
    load(kb, v);
    put(kb, v);
  }
}

template <int BM_, int BN_, int WP_, int STAGES_, int MINW_>
struct SplitTile {
  static constexpr int BM = BM_, BN = BN_, WP = WP_, S = STAGES_, MINW = MINW_;
  static constexpr int TM = BM / 64, TN = BN / 64;  // 32 x 32 tiles of a wavefront (2 x 2 wavefronts)
  static constexpr int A_STAGE = BM / 32 * 6 * SP_BLK, W_STAGE = BN / 32 * 2 * WP * SP_BLK, STAGE = A_STAGE + W_STAGE;
  static constexpr int AB = A_STAGE / SP_BLK / 4, WB = W_STAGE / SP_BLK / 4, PER = AB + WB;  // a wavefront's transfers a step
  static constexpr int LDS = S * STAGE;
  static_assert(A_STAGE / SP_BLK % 4 == 0 && W_STAGE / SP_BLK % 4 == 0, "transfer split");
  static_assert(PER * (S - 1) < 64 && S >= 2, "vmcnt range");
};

// The GEMM on the planes.  v_mfma_f32_32x32x16_bf16: one wavefront per SIMD issues it every 32
// cycles, the full rate (16x16x32, half the work each, every 27 instead of 16).  A ring of S stages
// of 32 K; the fragments of step kt + 1 are read into a second register set while step kt is
// multiplied, and a step's slot is free as soon as its fragments are in registers: its refill has
// S - 1 steps to land.
template <class TL>
__global__ __launch_bounds__(256, TL::MINW) void gemm_split_kernel(SplitArgs g) {
  constexpr int TM = TL::TM, TN = TL::TN, WP = TL::WP, S = TL::S;
  constexpr int NA = TM * TN == 1 ? 2 : 1;  // a lone tile: one accumulator per 16-K half, no serial chain
  __shared__ __attribute__((aligned(1024))) unsigned char smem[TL::LDS];
  const int lane = threadIdx.x & 63, wid = wave_uniform((int)(threadIdx.x >> 6));
  const int id = xcd_affine(blockIdx.x, gridDim.x);
  const int tm = id / g.nt, tn = id % g.nt;
  const int wm = wid >> 1, wn = wid & 1;
  const int64_t KB = g.KB;
  const int nk = (int)KB;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  const uint32_t lane16 = lane * 16;

  // source of each of this wavefront's transfers at K block 0 (row blocks clamped to the last one)
  const unsigned char* a_src[TL::AB];
  const unsigned char* w_src[TL::WB];
#pragma unroll
  for (int i = 0; i < TL::AB; ++i) {
    const int q = wid * TL::AB + i;
    const int64_t rb = min((int64_t)tm * (TL::BM / 32) + q / 6, g.rb - 1);
    a_src[i] = g.a_planes + (rb * KB * 6 + q % 6) * SP_BLK;
  }
#pragma unroll
  for (int i = 0; i < TL::WB; ++i) {
    const int q = wid * TL::WB + i;
    const int64_t nb = min((int64_t)tn * (TL::BN / 32) + q / (2 * WP), g.nb - 1);
    w_src[i] = g.w_planes + (nb * KB * 2 * WP + q % (2 * WP)) * SP_BLK;
  }
  // transfer i of step kt into slot s
  auto issue_one = [&](int i, int kt, int s) __attribute__((always_inline)) {
    if (i < TL::AB)
      lds_dma_m0<16>(a_src[i] + (int64_t)kt * 6 * SP_BLK, lane16, lds0 + s * TL::STAGE + (wid * TL::AB + i) * SP_BLK);
    else
      lds_dma_m0<16>(w_src[i - TL::AB] + (int64_t)kt * 2 * WP * SP_BLK, lane16,
                     lds0 + s * TL::STAGE + TL::A_STAGE + (wid * TL::WB + i - TL::AB) * SP_BLK);
  };
  auto issue = [&](int kt, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TL::PER; ++i) issue_one(i, kt, s);
  };

  f32x16 acc[NA][TM][TN] = {};
  // fragments of one step, those of the first 16-K half first: f[h][0 .. 3 TM) the rows' (tile i, part q at 3 i + q),
  // then the weight's (tile j, part q at WP j + q)
  constexpr int FA = 3 * TM, FH = FA + WP * TN, FR = 2 * FH;
  struct Frags {
    bf16x8 f[FR];
  };
  const unsigned char* ap = smem + wm * TM * 6 * SP_BLK + lane16;
  const unsigned char* wp = smem + TL::A_STAGE + wn * TN * 2 * WP * SP_BLK + lane16;
  auto read_one = [&](int i, int s, Frags& f) __attribute__((always_inline)) {
    const int h = i / FH, k = i % FH;
    f.f[i] = *reinterpret_cast<const bf16x8*>(
        k < FA ? ap + s * TL::STAGE + (k / 3 * 6 + h * 3 + k % 3) * SP_BLK
               : wp + s * TL::STAGE + ((k - FA) / WP * 2 * WP + h * WP + (k - FA) % WP) * SP_BLK);
  };
  auto product = [&](const Frags& f, int h, int qa, int qw) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[h % NA][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            f.f[h * FH + 3 * i + qa], f.f[h * FH + FA + WP * j + qw], acc[h % NA][i][j], 0, 0, 0);
  };
  // One step: the products (the small ones first) in 2 x 3 or 2 x 6 groups of MFMAs, with the next step's
  // fragment reads and the refill of the freed slot spread between the groups: issued in one go they
  // would fill the LDS queue and keep the matrix core waiting (measured at 8192 x 512 x 2048: 108 us
  // in one go).
  constexpr int NP = WP == 3 ? 6 : 3, G = 2 * NP;
  constexpr int QA[6] = {2, WP == 3 ? 0 : 1, WP == 3 ? 1 : 0, 1, 0, 0}, QW[6] = {0, WP == 3 ? 2 : 0, WP == 3 ? 1 : 0, 0, 1, 0};
  constexpr int GR = G > 2 ? G - 2 : G;  // groups that carry reads: the last two cover their latency
  auto step = [&](int kt, int s, int s1, bool more, bool next, const Frags& cur, Frags& nxt)
                  __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): step kt's fragments are in registers
    if (kt + S <= nk)
      wait_vm<TL::PER*(S - 2)>();        // own transfers of step kt + 1 (later ones in flight)
    else
      wait_vm<0>();
    __builtin_amdgcn_s_barrier();        // every wavefront's: step kt + 1 visible, step kt's slot free
#pragma unroll
    for (int u = 0; u < G; ++u) {
      __builtin_amdgcn_sched_barrier(0);
      if (next && u < GR) {
#pragma unroll
        for (int i = FR * u / GR; i < FR * (u + 1) / GR; ++i) read_one(i, s1, nxt);
      }
      if (more) {
#pragma unroll
        for (int i = TL::PER * u / G; i < TL::PER * (u + 1) / G; ++i) issue_one(i, kt + S, s);
      }
      __builtin_amdgcn_sched_barrier(0);
      product(cur, u % 2, QA[u / 2], QW[u / 2]);
    }
  };

#pragma unroll
  for (int p = 0; p < S; ++p)
    if (p < nk) issue(p, p);
  if (nk >= S)
    wait_vm<TL::PER*(S - 1)>();
  else
    wait_vm<0>();
  __builtin_amdgcn_s_barrier();
  Frags f0, f1;
#pragma unroll
  for (int i = 0; i < FR; ++i) read_one(i, 0, f0);
  int kt = 0, sl = 0;
  auto after = [](int s) __attribute__((always_inline)) { return s + 1 == S ? 0 : s + 1; };
  for (; kt + 1 + S < nk; kt += 2) {
    const int s1 = after(sl), s2 = after(s1);
    step(kt, sl, s1, true, true, f0, f1);
    step(kt + 1, s1, s2, true, true, f1, f0);
    sl = s2;
  }
  for (; kt < nk; kt += 2) {
    const int s1 = after(sl), s2 = after(s1);
    step(kt, sl, s1, kt + S < nk, kt + 1 < nk, f0, f1);
    if (kt + 1 < nk) step(kt + 1, s1, s2, kt + 1 + S < nk, kt + 2 < nk, f1, f0);
    sl = s2;
  }

  // A lane holds one output column of each tile, so a wavefront's store writes two whole 128-byte
  // lines (four columns a lane, 16-byte stores into 32 rows at once: 12.8 us instead of the stores
  // at 8192 x 512).
  const int64_t res_rows = g.res_rows;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t n = (int64_t)tn * TL::BN + (wn * TN + j) * 32 + (lane & 31);
    if (n >= g.N) continue;
    const float sc = g.w_scale ? g.w_scale[n] : 1.0f, bi = g.bias ? g.bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int64_t m0 = (int64_t)tm * TL::BM + (wm * TM + i) * 32 + (lane >> 5) * 4;
      float rv[16];
      if (g.res) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int64_t m = min(m0 + (e >> 2) * 8 + (e & 3), g.M - 1);
          rv[e] = g.res[(res_rows > 0 ? (g.m_base + m) % res_rows : m) * g.ld_res + n];
        }
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t m = m0 + (e >> 2) * 8 + (e & 3);
        float v = acc[0][i][j][e];
        if constexpr (NA == 2) v += acc[1][i][j][e];
        v *= sc;
        if (g.bias) v += bi;
        if (g.act == ACT_GELU) v = gelu_erf(v);
        if (g.res) v += rv[e];
        if (m < g.M) g.out[m * g.ld_out + n] = v;
      }
    }
  }
}

template <class TL>
int launch_split(SplitArgs g, hipStream_t stream) {
  g.mt = (int)cdiv(g.M, TL::BM);
  g.nt = (int)cdiv(g.N, TL::BN);
  hipLaunchKernelGGL((gemm_split_kernel<TL>), dim3((unsigned)((int64_t)g.mt * g.nt)), dim3(256), 0, stream, g);
  CORTEX_CHECK_LAUNCH("gemm_split_kernel");
  return OK;
}

constexpr int64_t SP_A_MAX = 256ll << 20;  // planes of the rows, at most, in the workspace asked for (128 have to fit)
constexpr int64_t SP_W_MAX = 256ll << 20;  // planes of the weight; a larger one is not taken

int64_t w_plane_bytes(int64_t N, int64_t K, int w_dtype) {
  return cdiv(N, 32) * cdiv(K, 32) * 2 * SP_BLK * (w_dtype == DT_I8 ? 1 : 3);
}
// rows of one chunk are a multiple of 128 (the tallest tile)
int64_t chunk_bytes(int64_t K) { return 4 * cdiv(K, 32) * 6 * SP_BLK; }

}  // namespace

}  // namespace cortex

using namespace cortex;

extern "C" {

int64_t cortex_norm_linear_split_workspace_bytes(int64_t M, int64_t N, int64_t K, int w_dtype) {
  if (M < 1 || N < 1 || K < 1 || (w_dtype != DT_I8 && w_dtype != DT_F32)) return 0;
  if (N > (1ll << 31) || K > (1ll << 24) || w_plane_bytes(N, K, w_dtype) > SP_W_MAX) return 0;
  const int64_t per = chunk_bytes(K);
  if (per > SP_A_MAX) return 0;
  int64_t chunks = cdiv(M, 128);
  if (chunks * per > SP_A_MAX) chunks = SP_A_MAX / per;
  return w_plane_bytes(N, K, w_dtype) + chunks * per;
}

int cortex_norm_linear_split(int64_t M, int64_t N, int64_t K, const float* x, int64_t ld_x, int norm, const void* gamma,
                             const void* beta, int gamma_dtype, float eps, int w_dtype, int w_layout, const void* w,
                             int64_t ld_w, const float* w_scale, const float* bias, int act, const float* residual,
                             int64_t ld_res, int64_t res_rows, float* out, int64_t ld_out, void* workspace,
                             int64_t workspace_bytes, hipStream_t stream) {
  CORTEX_CHECK_ARG(M >= 0 && N >= 0 && K >= 0, "cortex_norm_linear_split: negative shape");
  if (M == 0 || N == 0) return OK;
  CORTEX_CHECK_ARG(K > 0, "cortex_norm_linear_split: K must be positive");
  CORTEX_CHECK_ARG(x && w && out && workspace, "cortex_norm_linear_split: null x, w, out or workspace");
  CORTEX_CHECK_ARG(ld_x >= K && ld_out >= N, "cortex_norm_linear_split: ld_x < K or ld_out < N");
  CORTEX_CHECK_ARG(w_dtype == DT_I8 || w_dtype == DT_F32, "cortex_norm_linear_split: the weight must be int8 or fp32");
  CORTEX_CHECK_ARG(w_layout == 0 || (w_layout == 1 && w_dtype == DT_F32),
                   "cortex_norm_linear_split: int8 weights must be (N, K)");
  CORTEX_CHECK_ARG(w_layout == 0 ? ld_w >= K : ld_w >= N, "cortex_norm_linear_split: ld_w too small for the layout");
  CORTEX_CHECK_ARG(norm == NORM_NONE || norm == NORM_LAYER || norm == NORM_RMS,
                   "cortex_norm_linear_split: unknown norm %d", norm);
  CORTEX_CHECK_ARG(norm == NORM_NONE || gamma, "cortex_norm_linear_split: norm needs gamma");
  CORTEX_CHECK_ARG(gamma_dtype == DT_F32 || gamma_dtype == DT_BF16 || gamma_dtype == DT_F16,
                   "cortex_norm_linear_split: unsupported gamma dtype %d", gamma_dtype);
  CORTEX_CHECK_ARG(act == ACT_NONE || act == ACT_GELU, "cortex_norm_linear_split: unknown activation %d", act);
  CORTEX_CHECK_ARG(residual == nullptr || ld_res >= N, "cortex_norm_linear_split: ld_res < N");
  CORTEX_CHECK_ARG(N <= (1ll << 31) && K <= (1ll << 24), "cortex_norm_linear_split: N or K too large");
  CORTEX_CHECK_ARG(((uintptr_t)workspace & 15) == 0, "cortex_norm_linear_split: workspace must be 16-byte aligned");
  const int64_t wb = w_plane_bytes(N, K, w_dtype), per = chunk_bytes(K);
  int64_t chunks = (workspace_bytes - wb) / per;
  if (workspace_bytes < wb || chunks < 1) {
    set_error("cortex_norm_linear_split: workspace of %lld bytes, at least %lld needed", (long long)workspace_bytes,
              (long long)(wb + per));
    return E_WORKSPACE;
  }
  if (chunks > (1 << 20)) chunks = 1 << 20;
  auto a16 = [](const void* p, int64_t ld) { return ((uintptr_t)p & 15) == 0 && ld % 4 == 0; };
  SplitArgs g = {};
  g.N = N;
  g.K = K;
  g.KB = cdiv(K, 32);
  g.ld_x = ld_x;
  g.norm = norm;
  g.gamma = gamma;
  g.beta = norm == NORM_LAYER ? beta : nullptr;
  g.gamma_dtype = gamma_dtype;
  g.eps = eps;
  g.x_vec = a16(x, ld_x) ? 1 : 0;
  g.g_vec = gamma_dtype == DT_F32 && a16(gamma, 0) && a16(beta, 0) ? 1 : 0;
  g.w = w;
  g.w_dtype = w_dtype;
  g.w_layout = w_layout;
  g.w_vec = w_dtype == DT_I8 ? (((uintptr_t)w & 7) == 0 && ld_w % 8 == 0) : a16(w, ld_w);
  g.ld_w = ld_w;
  g.w_planes = reinterpret_cast<unsigned char*>(workspace);
  g.a_planes = g.w_planes + wb;
  g.nb = cdiv(N, 32);
  const int64_t kc = cdiv(g.KB, SP_KC);  // prep workgroups per 32 rows without a norm
  g.w_scale = w_scale;
  g.bias = bias;
  g.act = act;
  g.ld_res = ld_res;
  g.res_rows = res_rows;
  g.ld_out = ld_out;
  for (int64_t m = 0; m < M; m += chunks * 128) {
    g.M = M - m < chunks * 128 ? M - m : chunks * 128;
    g.x = x + m * ld_x;
    g.rb = cdiv(g.M, 32);
    g.w_blocks = m == 0 ? g.nb * kc : 0;
    g.m_base = m;
    g.res = residual ? (res_rows > 0 ? residual : residual + m * ld_res) : nullptr;
    g.out = out + m * ld_out;
    const int64_t prep = g.w_blocks + g.rb * (norm == NORM_NONE ? kc : 1);
    hipLaunchKernelGGL(split_prep_kernel, dim3((unsigned)prep), dim3(64 * SP_PW), 0, stream, g);
    CORTEX_CHECK_LAUNCH("split_prep_kernel");
    const int64_t tiles = cdiv(g.M, 128) * cdiv(N, 128);
    CORTEX_CHECK_ARG(cdiv(g.M, 64) * cdiv(N, 64) <= 0x7fffffffLL, "cortex_norm_linear_split: N too large for the grid");
    // Tile by shape (whole calls, us; 128 x 128 / 64 x 64).  64 x 64 tiles fill more of the chip while 128 x 128 ones
    // are at most one per CU, and just above, where those start a second round; from there on 128 x 128 ones,
    // which refill half as much per MFMA.  Their epilogue reads 64 residual values a lane with nothing beside
    // it, so with a residual the line lies higher.
    //   int8 (128 x 128 with two stages, two workgroups a CU).  At 256, 288, 320 and 384 tiles: 8192 .. 12288 x 512 x
    //   512 31.0 / 28.2, 36.5 / 32.8, 38.5 / 34.2, 42.8 / 42.6, with a residual 44.5 / 31.0, 46.3 / 37.1, 46.9 / 37.8, 47.4 / 41.0 and
    //   53.3 / 51.8 at 512; x 512 x 2048 86.1 / 90.7, 110 / 104, 114 / 114, 130 / 137, with a residual 101 / 87, 115 / 101, 120 /
    //   108, 134 / 132 and 175 / 214 at 512.
    //   fp32 (144 KiB, one workgroup a CU).  K = 512 43.7 / 41.8, 60.7 / 46.3 (280), 61.7 / 48.0, 66.2 / 56.6, with a residual
    //   54.0 / 41.3, 79.1 / 46.1, 81.4 / 47.3, 86.8 / 53.3; K = 2048 122 / 129, 183 / 148 (280), 191 / 159, 206 / 191, with a residual
    //   129 / 124, 202 / 143, 207 / 152, 224 / 189 and 260 / 272 at 512; without one, from 7/8 of the CUs on 2048 x 2048 x
    //   512 40.8 / 50.1, 16384 x 256 x 256 34.0 / 33.5, 4096 x 1024 x 2048 109 / 118.  64 x 64 take a fourth stage while one
    //   workgroup a CU is all there is (256 x 512 x 2048: 31 against 33; 1024 x 1536 x 512 with two a CU: 31 against 28).
    // The fp32 MFMA kernel before, whole call with the norm: 8192 x 2048 x 512 273 us -> 69 (int8), 314 ->
    // 125 (fp32, (K, N)); 256 x 512 x 2048 without 178 -> 22 and 232 -> 31; 64 x 256 x 256 62 -> 10.
    const int64_t ncu = cu_count(), line = residual ? ncu * 3 / 2 : ncu * 5 / 4;
    int rc;
    if (w_dtype == DT_I8)
      rc = tiles > line ? launch_split<SplitTile<128, 128, 1, 2, 2>>(g, stream)
                        : launch_split<SplitTile<64, 64, 1, 4, 2>>(g, stream);
    else if (tiles > line || (!residual && tiles > ncu * 7 / 8 && tiles <= ncu))
      rc = launch_split<SplitTile<128, 128, 3, 3, 1>>(g, stream);
    else
      rc = cdiv(g.M, 64) * cdiv(N, 64) > ncu ? launch_split<SplitTile<64, 64, 3, 3, 2>>(g, stream)
                                             : launch_split<SplitTile<64, 64, 3, 4, 1>>(g, stream);
    if (rc != OK) return rc;
  }
  return OK;
}

}  // extern "C"
