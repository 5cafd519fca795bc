// fp32 attention on the bf16 matrix cores for gfx950 (head dim 64): every fp32 operand -- queries, keys,
// values and the probabilities -- as the exact sum of three bf16 parts (split_parts.h), six products of order up
// to 2^-16 each (exact, summed in fp32), as gemm_split.hip does for the linears; the softmax in fp32, its
// probabilities by the hardware's exp2 (0 below 2^-126, where the largest of a row is at least 1).
//
// What bounds it.  On the fp32 MFMA (157 TFLOP/s) a 32 x 64 block of scores and its P V cost 8192 cycles
// of a SIMD; six bf16 products cost 3072 (v_mfma_f32_32x32x16_bf16).  Beside them a wavefront spends about
// 1500 cycles of VALU on the softmax and the parts of P and 900 on its share of splitting the K and V
// tile, which other wavefronts of the SIMD cover.
//
// Workgroup: 4 wavefronts of 32 queries each (WK 1), or, where that leaves CUs without a workgroup, 2 x 32
// queries with the keys of a tile split between two wavefronts (WK 2) that merge their sums at the end.
// Keys come in tiles of 64: fp32 rows global -> registers one tile ahead, split there and written to
// LDS as planes in MFMA fragment order (48 KiB: two workgroups share a CU), so every fragment is one
// linear 16-byte read per lane.
//   S^T = K Q^T   a lane holds 16 keys (8 (r / 4) + 4 (lane / 32) + r % 4) of one query (lane % 32) per 32
//                 keys, so the softmax is lane-local apart from one exchange with lane ^ 32;
//   O^T += V^T P^T  with the keys of a 16-key step in the order the lane holds them: V's planes are
//                 written in that order, so P goes from the score registers straight into the MFMA.
// The tiles to visit are listed in LDS first: those with a key that the length and the key mask allow and,
// with a tile mask (block_e a multiple of 64), that one of the workgroup's query tiles allows.
#include <hip/hip_runtime.h>

#include "attention.h"
#include "common.h"
#include "split_parts.h"

namespace cortex {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int AS_KT = 64;         // keys per tile
constexpr int AS_TILES = 512;     // tiles of the list (32768 keys)
constexpr int AS_BLK = 1024;      // one plane's block of 32 x 16 operand values
constexpr int AS_V0 = 24 * AS_BLK;  // V planes behind the K planes
constexpr float AS_RESCALE = 8.0f;  // log2 units by which a tile must raise the reference max to move it

__device__ __forceinline__ void put_parts(unsigned char* dst, const Parts& s) {
#pragma unroll
  for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8*>(dst + q * AS_BLK) = s.p[q];
}
__device__ __forceinline__ Parts get_parts(const unsigned char* src) {
  Parts s;
#pragma unroll
  for (int q = 0; q < 3; ++q) s.p[q] = *reinterpret_cast<const bf16x8*>(src + q * AS_BLK);
  return s;
}
// this wavefront's LDS accesses done, then every wavefront's
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// products a_i b_j in the order of their size, small ones first
constexpr int AS_PA[6] = {2, 0, 1, 1, 0, 0}, AS_PB[6] = {0, 2, 1, 0, 1, 0};

template <int WK>
__global__ __launch_bounds__(256, 2) void attention_split_kernel(AttnArgs a) {
  constexpr int WQ = 4 / WK, QB = 32 * WQ;
  constexpr int KH = 2 / WK;  // 32-key halves of a tile per wavefront
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * AS_V0];
  __shared__ uint64_t kmask[AS_TILES];
  __shared__ uint16_t klist[AS_TILES];
  const int tid = threadIdx.x, lane = tid & 63, wid = wave_uniform(tid >> 6);
  const int fr = lane & 31, h = lane >> 5;
  const int wq = wid % WQ, wk = wid / WQ;

  // the query blocks of one (sample, head) on one XCD (shared K and V in its L2)
  const int nqb = gridDim.x, id = xcd_affine(blockIdx.x + nqb * blockIdx.y, nqb * gridDim.y);
  const int64_t bh = id / nqb, q0 = (int64_t)(id % nqb) * QB;
  const int64_t b = bh / a.H, hd = bh - b * a.H;
  int64_t len = a.Lk;
  const float* Kb = reinterpret_cast<const float*>(a.k) + hd * a.k_sh;
  const float* Vb = reinterpret_cast<const float*>(a.v) + hd * a.v_sh;
  if (a.kv_off) {
    // offsets come from the caller: clamp them to the Lk key rows of the view
    const int64_t r0 = min(max(a.kv_off[b], (int64_t)0), a.Lk);
    len = min(max(a.kv_off[b + 1], r0), a.Lk) - r0;
    Kb += r0 * a.k_sl;
    Vb += r0 * a.v_sl;
  } else {
    Kb += b * a.k_sb;
    Vb += b * a.v_sb;
  }
  if (a.kv_len) len = min(len, a.kv_len[b]);
  if (len < 0) len = 0;
  len = wave_uniform(len);

  const int64_t qr = q0 + wq * 32 + fr, q = min(qr, a.Lq - 1);  // this lane's query
  const uint8_t* bm = a.block_mask ? a.block_mask + b * a.bm_sb : nullptr;
  const int64_t kpt = bm ? a.block_e / AS_KT : 1, qi = bm ? q / a.block_l : 0;

  // ---- the tiles to visit
  int n = 0;
  {
    const int nt = (int)cdiv(len, AS_KT);
    const uint8_t* km = a.key_mask ? a.key_mask + b * a.km_sb : nullptr;
    for (int t = wid; t < nt; t += 4) {
      const int64_t j = (int64_t)t * AS_KT + lane;
      const uint64_t bits = __ballot(j < len && (!km || km[min(j, len - 1)] != 0));
      if (lane == 0) kmask[t] = bits;
    }
    __syncthreads();
    const int64_t qa = bm ? q0 / a.block_l : 0, qb = bm ? min(min(q0 + QB, a.Lq) - 1, a.Lq - 1) / a.block_l : 0;
    for (int t0 = 0; t0 < nt; t0 += 64) {
      const int t = min(t0 + lane, nt - 1);
      bool any = t0 + lane < nt && kmask[t] != 0;
      if (any && bm) {
        const int64_t kj = t / kpt;
        any = false;
        for (int64_t i = qa; i <= qb && !any; ++i) any = i < a.n_qt && kj < a.n_kt && bm[i * a.n_kt + kj] != 0;
      }
      const uint64_t w = __ballot(any);
      if (any && wid == 0) klist[n + __popcll(w & ((1ull << lane) - 1))] = (uint16_t)(t0 + lane);
      n += __popcll(w);
    }
    __syncthreads();
  }

  Parts qf[4];  // B operand of S^T: query fr, head dims 16 ks + 8 h ..
  {
    const float* Qp = reinterpret_cast<const float*>(a.q) + b * a.q_sb + hd * a.q_sh + q * a.q_sl;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      float v[8];
      *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(Qp + ks * 16 + h * 8);
      *reinterpret_cast<float4*>(v + 4) = *reinterpret_cast<const float4*>(Qp + ks * 16 + h * 8 + 4);
      qf[ks] = split8<true>(v);
    }
  }

  // ---- a tile's share of this wavefront: two 32-key x 16-dim units of K, two 8-key x 64-dim units of V
  float kr[2][8], vr[2][8];
  uint8_t bm_ok = 1;
  auto load_tile = [&](int t) __attribute__((always_inline)) {
    if (bm) {
      const int64_t kj = t / kpt;
      bm_ok = qi < a.n_qt && kj < a.n_kt ? bm[qi * a.n_kt + kj] : 0;
    }
    const int64_t k0 = (int64_t)t * AS_KT;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int ku = wid * 2 + u;
      const float* kp = Kb + min(k0 + (ku >> 2) * 32 + fr, len - 1) * a.k_sl + (ku & 3) * 16 + h * 8;
      *reinterpret_cast<float4*>(kr[u]) = *reinterpret_cast<const float4*>(kp);
      *reinterpret_cast<float4*>(kr[u] + 4) = *reinterpret_cast<const float4*>(kp + 4);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int64_t key = min(k0 + (ku >> 1) * 16 + (j >> 2) * 8 + (ku & 1) * 4 + (j & 3), len - 1);
        vr[u][j] = Vb[key * a.v_sl + lane];
      }
    }
  };
  auto stage_tile = [&](int t) __attribute__((always_inline)) {
    const int64_t rem = len - (int64_t)t * AS_KT;
    if (rem < AS_KT) {  // rows past the end count as 0: their probability 0 times the last row's infinity is NaN
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int ku = wid * 2 + u;
          if ((ku >> 1) * 16 + (j >> 2) * 8 + (ku & 1) * 4 + (j & 3) >= rem) vr[u][j] = 0.0f;
        }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int ku = wid * 2 + u;
      put_parts(smem + ku * 3 * AS_BLK + lane * 16, split8<true>(kr[u]));
      put_parts(smem + AS_V0 + ((lane >> 5) * 4 + (ku >> 1)) * 3 * AS_BLK + ((ku & 1) * 32 + fr) * 16,
                split8<true>(vr[u]));
    }
  };

  float m_run = -INFINITY, l_run = 0.0f;
  f32x16 o[2] = {};
  const float sl = a.scale_log2;

  if (n > 0) load_tile(wave_uniform((int)klist[0]));
  for (int i = 0; i < n; ++i) {
    const int t = wave_uniform((int)klist[i]);
    const uint64_t bits = (uint64_t)wave_uniform((int64_t)kmask[t]);
    stage_tile(t);
    const bool ok_q = bm_ok != 0;
    lds_barrier();
    if (i + 1 < n) load_tile(wave_uniform((int)klist[i + 1]));
    if (!bm || __any(ok_q)) {
      f32x16 s[KH];
#pragma unroll
      for (int x = 0; x < KH; ++x) {
        const int kh = WK == 1 ? x : wk;
        f32x16 acc[2] = {};  // (two chains)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const Parts kf = get_parts(smem + (kh * 4 + ks) * 3 * AS_BLK + lane * 16);
#pragma unroll
          for (int p = 0; p < 6; ++p)
            acc[p & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf.p[AS_PA[p]], qf[ks].p[AS_PB[p]], acc[p & 1], 0, 0, 0);
        }
        s[x] = acc[0] + acc[1];
      }
      const bool masked = bits != ~0ull || bm;
      float mx = -INFINITY;
#pragma unroll
      for (int x = 0; x < KH; ++x) {
        const int kh = WK == 1 ? x : wk;
        const uint32_t word = (ok_q ? (uint32_t)(bits >> (32 * kh)) : 0u) >> (4 * h);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float v = s[x][r] * sl;
          if (masked) v = (word >> (8 * (r >> 2) + (r & 3))) & 1 ? v : -INFINITY;
          s[x][r] = v;
          mx = fmaxf(mx, v);
        }
      }
      // the reference max moves only when a score exceeds it by AS_RESCALE (wave-uniform, rare)
      if (__any(mx > m_run + AS_RESCALE)) {
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run, mx);
        const float alpha = m_new == -INFINITY ? 1.0f : exp2f(m_run - m_new);  // m_run = -inf -> 0
        m_run = m_new;
        l_run *= alpha;
        o[0] *= alpha;
        o[1] *= alpha;
      }
      const float ref = m_run == -INFINITY ? 0.0f : m_run;  // (no key allowed so far: exp2(-inf) = 0)
#pragma unroll
      for (int x = 0; x < KH; ++x) {
        const int kh = WK == 1 ? x : wk;
#pragma unroll
        for (int gl = 0; gl < 2; ++gl) {
          float p[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            p[j] = __builtin_amdgcn_exp2f(s[x][8 * gl + j] - ref);
            l_run += p[j];
          }
          const Parts pf = split8<false>(p);
#pragma unroll
          for (int d = 0; d < 2; ++d) {
            const Parts vf = get_parts(smem + AS_V0 + (d * 4 + kh * 2 + gl) * 3 * AS_BLK + lane * 16);
#pragma unroll
            for (int e = 0; e < 6; ++e)
              o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.p[AS_PA[e]], pf.p[AS_PB[e]], o[d], 0, 0, 0);
          }
        }
      }
    }
    lds_barrier();  // every wavefront is done with the tile
  }

  l_run += __shfl_xor(l_run, 32, 64);
  // ---- rows out through LDS: 256-byte rows, four per store
  constexpr int LDO = 68;  // floats per row (the pad keeps a column's rows on different banks)
  float* rows = reinterpret_cast<float*>(smem) + wq * 32 * LDO;
  if constexpr (WK == 2) {
    float* part = reinterpret_cast<float*>(smem) + WQ * 32 * LDO;  // the second wavefront's sums: [34][64] each
    float* mine = part + wq * 34 * 64 + lane;
    if (wk == 1) {
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(d * 16 + r) * 64] = o[d][r];
      mine[32 * 64] = m_run;
      mine[33 * 64] = l_run;
    }
    lds_barrier();
    if (wk == 0) {
      const float m2 = mine[32 * 64], l2 = mine[33 * 64], m = fmaxf(m_run, m2);
      const float f1 = m_run == -INFINITY ? 0.0f : exp2f(m_run - m), f2 = m2 == -INFINITY ? 0.0f : exp2f(m2 - m);
      l_run = l_run * f1 + l2 * f2;
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] = o[d][r] * f1 + mine[(d * 16 + r) * 64] * f2;
    }
  }
  if (wk == 0) {
    const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int r = 0; r < 16; r += 4) {
        const f32x4 v = {o[d][r] * inv, o[d][r + 1] * inv, o[d][r + 2] * inv, o[d][r + 3] * inv};
        *reinterpret_cast<f32x4*>(rows + fr * LDO + d * 32 + 2 * r + 4 * h) = v;
      }
  }
  lds_barrier();
  const int per = 32 / WK;  // rows of its query group that a wavefront stores
#pragma unroll
  for (int i = 0; i < per; i += 4) {
    const int r = wk * per + i + (lane >> 4);
    const int64_t qo = q0 + wq * 32 + r;
    if (qo < a.Lq)
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + b * a.o_sb + hd * a.o_sh + qo * a.o_sl +
                                (lane & 15) * 4) = *reinterpret_cast<const f32x4*>(rows + r * LDO + (lane & 15) * 4);
  }
}

}  // namespace

int try_attention_split(const AttnArgs& a, int dtype, hipStream_t stream) {
  if (dtype != DT_F32 || a.Dh != 64 || !a.vec || a.Lk > (int64_t)AS_TILES * AS_KT) return 0;
  if (a.block_mask && a.block_e % AS_KT != 0) return 0;
  if (((uintptr_t)a.out & 15) || a.o_sb % 4 || a.o_sh % 4 || a.o_sl % 4) return 0;
  const int64_t nbh = a.B * a.H, nq = cdiv(a.Lq, 128);
  if (nbh > 65535 || cdiv(a.Lq, 64) * nbh > 0x7fffffffLL) return 0;
  // 128 queries a workgroup (K and V split once per 128 queries) once that gives every CU one
  if (nq * nbh >= cu_count()) {
    hipLaunchKernelGGL((attention_split_kernel<1>), dim3((unsigned)nq, (unsigned)nbh), dim3(256), 0, stream, a);
  } else {
    hipLaunchKernelGGL((attention_split_kernel<2>), dim3((unsigned)cdiv(a.Lq, 64), (unsigned)nbh), dim3(256), 0, stream,
                       a);
  }
  CORTEX_CHECK_LAUNCH("attention_split_kernel");
  return 1;
}

}  // namespace cortex
