// 2-simplicial attention backward for fp32 operands of small molecules (at
// most 32 tokens, head_dim <= 32 and a multiple of 4) on gfx950 (CDNA4),
// deterministic (no atomics).
//
// The pair formulation of simplicial_pair_bwd.hip (the gradient of
// simplicial_attention.py:206-344; triton_simplicial_attention.py:332-782) in
// fp32 throughout: five products of n^3 D multiply-adds on fp32 MFMA 16x16x4
// where the ownership kernel (simplicial_bwd.hip) takes eleven.
//   S, dP  C[query 4 g + r][pair (j, k0 + r16)] = sum_d q / go [query][d] W / Z [pair][d]
//   dS = P (dP - go . out), P = exp(S - lse)
//   G^T, H^T [d][pair] += q^T / go^T [d][query] dS / P [query][pair]: accumulator r (query 4 g + r) is the B
//          operand of K step r as it is
//   dq^T [d][query] += W^T [d][pair] dS^T [pair][query]: dS turned through a per-wave LDS scratch
//   dk1_j = sum_k G_jk (.) k2_k, dk2_k = sum_j G_jk (.) k1_j (dv1, dv2 from H)
// One workgroup of W = 4 or 8 waves per (molecule, head); a wave takes j = wave, wave + W, ... with both key tiles of a
// molecule inside, so dk1_j / dv1_j are finished by one reduction over the lanes that hold the keys, and dq, dk2,
// dv2 partials of the waves are added in wave order at the end.  MFMA-bound: 80 MFMA of 32 cycles per (j, 16
// keys) at two query tiles, with the rest (about 150 VALU and LDS instructions) beside them.
#include <algorithm>

#include "mf_common.h"

namespace mf {
namespace spf32b {

constexpr int MN = 32;        // tokens at most
constexpr int DP = 32;        // head_dim at most
constexpr int KS = DP + 4;    // row stride (floats)
constexpr int NC = DP / 4;    // K steps of S, and a lane's contiguous d
constexpr int ND = DP / 16;
constexpr int SS = 16 + 4;    // row stride of the dS scratch

struct Params {
  const float* q;
  const float* k1;
  const float* v1;
  const float* k2;
  const float* v2;
  const float* go;
  const float* out;
  const float* lse;
  const uint8_t* qv;
  const uint8_t* pkv;
  const uint8_t* pv;
  float* dq;
  float* dk1;
  float* dv1;
  float* dk2;
  float* dv2;
  const void* u;   // factorized bias, element type bias_dtype (BIAS); gradients NULL = not wanted
  const void* v;
  const void* w;
  const void* gate;
  float* du;
  float* dvb;
  float* dw;
  float* dgate;
  int bias_dtype;
  int H, N, D;
};

// LDS of W waves (floats)
template <int W>
struct Lds {
  float op[W > 6 ? W : 6][MN * KS];     // q, go, k1, v1, k2, v2 (compacted, zero past the counts); later the partials
  float scr[W][2][16 * SS];             // dS of a query tile, [pair][query]
  float lse2[MN], dlt[MN];
  uint32_t bits[MN];                    // valid keys of each j
  int kidx[MN], qidx[MN];
};
template <int W>
struct LdsBias {
  float ut[MN * KS], vt[MN * KS], w[MN * KS];  // u^T [j][i], v^T [k][i], w [j][k]
  float gate[MN];
  float dg[W][MN];
};

__device__ __forceinline__ float load_any(const void* p, size_t idx, int dtype) {
  if (dtype == MF_DTYPE_F32) return static_cast<const float*>(p)[idx];
  if (dtype == MF_DTYPE_BF16) return static_cast<float>(static_cast<const __bf16*>(p)[idx]);
  return static_cast<float>(static_cast<const _Float16*>(p)[idx]);
}

__device__ __forceinline__ mf_f32x4 mma(float a, float b, mf_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// DPP lane moves within rows of 16: quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_ror 4 and 8.
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __uint_as_float(uint32_t(__builtin_amdgcn_update_dpp(0, int(__float_as_uint(x)), CTRL, 0xf, 0xf, false)));
}
constexpr int kXor1 = 0xb1, kXor2 = 0x4e, kRor4 = 0x124, kRor8 = 0x128;

// Sums over each 16-lane row of four values: lane r16 returns the sum of v[r16 & 3].
__device__ __forceinline__ float row16_sum4(const float v0, const float v1, const float v2, const float v3, int r16) {
  const bool o1 = (r16 & 1) != 0, o2 = (r16 & 2) != 0;
  const float a = (o1 ? v1 : v0) + dpp<kXor1>(o1 ? v0 : v1);
  const float b = (o1 ? v3 : v2) + dpp<kXor1>(o1 ? v2 : v3);
  float x = (o2 ? b : a) + dpp<kXor2>(o2 ? a : b);
  x += dpp<kRor4>(x);
  return x + dpp<kRor8>(x);
}

__device__ __forceinline__ float sum_groups(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float y = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(y), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Rows 0 .. n - 1 of the waves' partials (row stride KS, wave stride MN KS) added in wave order into the rows
// of `dst` that idx names.
template <int W>
__device__ __forceinline__ void write_rows(const float* part, float* dst, const int* idx, int n, int D, size_t rbase) {
  for (int u = threadIdx.x; u < n * (D / 4); u += W * 64) {
    const int i = u / (D / 4), c = 4 * (u % (D / 4));
    float4 s = *reinterpret_cast<const float4*>(part + i * KS + c);
#pragma unroll
    for (int w = 1; w < W; ++w) {
      const float4 x = *reinterpret_cast<const float4*>(part + w * MN * KS + i * KS + c);
      s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
    }
    *reinterpret_cast<float4*>(dst + (rbase + idx[i]) * D + c) = s;
  }
}

// NT query tiles, NK key tiles.
template <int NT, int NK, bool BIAS, int W>
__device__ __forceinline__ void body(const Params& p, Lds<W>& L, LdsBias<W>* X, int nk, int nq, size_t rbase) {
  constexpr int kThreads = W * 64;
  const int lane = lane_id(), wave = wave_id();
  const int g = lane >> 4, r16 = lane & 15;
  const int N = p.N, D = p.D;
  const float *Q = L.op[0], *GO = L.op[1], *K1 = L.op[2], *V1 = L.op[3], *K2 = L.op[4], *V2 = L.op[5];
  float* scr = &L.scr[wave][0][0];
  // A operands of S and dP: query 16 t + r16 at d = NC g + c (BIAS: read where they are used, the bias sums take
  // their registers)
  float qf[BIAS ? 1 : NT][NC], gf[BIAS ? 1 : NT][NC];
  auto rows_of = [&](int t, int c, float4& x, float4& y) {
    x = *reinterpret_cast<const float4*>(Q + (16 * t + r16) * KS + NC * g + c);
    y = *reinterpret_cast<const float4*>(GO + (16 * t + r16) * KS + NC * g + c);
  };
  if constexpr (!BIAS) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int c = 0; c < NC; c += 4) {
        float4 x, y;
        rows_of(t, c, x, y);
        qf[t][c] = x.x; qf[t][c + 1] = x.y; qf[t][c + 2] = x.z; qf[t][c + 3] = x.w;
        gf[t][c] = y.x; gf[t][c + 1] = y.y; gf[t][c + 2] = y.z; gf[t][c + 3] = y.w;
      }
  }
  mf_f32x4 dqa[NT][ND];            // d = 16 dt + 4 g + r, query 16 t + r16
  float dk2a[NK][ND][4], dv2a[NK][ND][4];  // d = 16 dt + 4 g + r, key 16 kt + r16
  float dva[NK][NT][4], accg[NT][4];       // BIAS: query 16 t + 4 g + r, key 16 kt + r16
#pragma unroll
  for (int t = 0; t < NT; ++t) {
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) dqa[t][dt] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) accg[t][r] = 0.0f;
  }
#pragma unroll
  for (int kt = 0; kt < NK; ++kt) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) dk2a[kt][dt][r] = dv2a[kt][dt][r] = 0.0f;
#pragma unroll
      for (int t = 0; t < NT; ++t) dva[kt][t][r] = 0.0f;
    }
  }

  for (int j = wave; j < nk; j += W) {
    const uint32_t bits = L.bits[j];
    float k1a[NC], v1a[NC];  // d = NC g + c
#pragma unroll
    for (int c = 0; c < NC; c += 4) {
      const float4 x = *reinterpret_cast<const float4*>(K1 + j * KS + NC * g + c);
      const float4 y = *reinterpret_cast<const float4*>(V1 + j * KS + NC * g + c);
      k1a[c] = x.x; k1a[c + 1] = x.y; k1a[c + 2] = x.z; k1a[c + 3] = x.w;
      v1a[c] = y.x; v1a[c + 1] = y.y; v1a[c + 2] = y.z; v1a[c + 3] = y.w;
    }
    float x1[ND][4], y1[ND][4], dus[NT][4];
    mf_f32x4 dqt[NT][ND];  // this j's pairs, summed on their own
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) {
#pragma unroll
      for (int r = 0; r < 4; ++r) x1[dt][r] = y1[dt][r] = 0.0f;
#pragma unroll
      for (int t = 0; t < NT; ++t) dqt[t][dt] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) dus[t][r] = 0.0f;
#pragma unroll
    for (int kt = 0; kt < NK; ++kt) {
      const int k0 = 16 * kt;
      const bool ok = (bits >> (k0 + r16)) & 1u;
      // B operands: W, Z of pair (j, k0 + r16) at d = NC g + c
      // (two sums of half of d each, S in the forward's own order, so that P = exp(S - lse) is its P)
      mf_f32x4 sh[2][NT], dph[2][NT], s[NT], dp[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) sh[0][t] = sh[1][t] = dph[0][t] = dph[1][t] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; c += 4) {
        constexpr int kHalf = NC / 2;
        static_assert(kHalf % 4 == 0, "whole steps");
        mf_f32x4(&sc)[NT] = sh[c / kHalf];
        mf_f32x4(&dc)[NT] = dph[c / kHalf];
        const float4 x = *reinterpret_cast<const float4*>(K2 + (k0 + r16) * KS + NC * g + c);
        const float4 y = *reinterpret_cast<const float4*>(V2 + (k0 + r16) * KS + NC * g + c);
        const float wv[4] = {x.x * k1a[c], x.y * k1a[c + 1], x.z * k1a[c + 2], x.w * k1a[c + 3]};
        const float zv[4] = {y.x * v1a[c], y.y * v1a[c + 1], y.z * v1a[c + 2], y.w * v1a[c + 3]};
        if constexpr (BIAS) {
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            float4 q4, g4;
            rows_of(t, c, q4, g4);
            sc[t] = mma(q4.x, wv[0], sc[t]); dc[t] = mma(g4.x, zv[0], dc[t]);
            sc[t] = mma(q4.y, wv[1], sc[t]); dc[t] = mma(g4.y, zv[1], dc[t]);
            sc[t] = mma(q4.z, wv[2], sc[t]); dc[t] = mma(g4.z, zv[2], dc[t]);
            sc[t] = mma(q4.w, wv[3], sc[t]); dc[t] = mma(g4.w, zv[3], dc[t]);
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              sc[t] = mma(qf[t][c + e], wv[e], sc[t]);
              dc[t] = mma(gf[t][c + e], zv[e], dc[t]);
            }
        }
      }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[t][r] = sh[0][t][r] + sh[1][t][r];
          dp[t][r] = dph[0][t][r] + dph[1][t][r];
        }
      float dwj = 0.0f;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const float4 l4 = *reinterpret_cast<const float4*>(L.lse2 + 16 * t + 4 * g);
        const float4 d4 = *reinterpret_cast<const float4*>(L.dlt + 16 * t + 4 * g);
        const float l2[4] = {l4.x, l4.y, l4.z, l4.w}, dl[4] = {d4.x, d4.y, d4.z, d4.w};
        float base[4] = {0.f, 0.f, 0.f, 0.f}, gt[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (BIAS) {
          const float4 g4 = *reinterpret_cast<const float4*>(X->gate + 16 * t + 4 * g);
          const float4 u4 = *reinterpret_cast<const float4*>(X->ut + j * KS + 16 * t + 4 * g);
          const float4 v4 = *reinterpret_cast<const float4*>(X->vt + (k0 + r16) * KS + 16 * t + 4 * g);
          const float wjk = X->w[j * KS + k0 + r16];
          gt[0] = g4.x; gt[1] = g4.y; gt[2] = g4.z; gt[3] = g4.w;
          // (0 at a dropped pair: dS is 0 there, but the terms may be -inf or NaN)
          base[0] = ok ? (u4.x + v4.x) + wjk : 0.0f; base[1] = ok ? (u4.y + v4.y) + wjk : 0.0f;
          base[2] = ok ? (u4.z + v4.z) + wjk : 0.0f; base[3] = ok ? (u4.w + v4.w) + wjk : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float s2 = s[t][r];
          if constexpr (BIAS) s2 = fmaf(gt[r], base[r], s2);
          s2 = fmaf(s2, kLog2e, -l2[r]);
          const float pr = ok ? fast_exp2(s2) : 0.0f;
          s[t][r] = pr;
          dp[t][r] = pr * (dp[t][r] - dl[r]);
          if constexpr (BIAS) {
            accg[t][r] = fmaf(dp[t][r], base[r], accg[t][r]);
            dwj = fmaf(gt[r], dp[t][r], dwj);
            dva[kt][t][r] += dp[t][r];
            dus[t][r] += dp[t][r];
          }
        }
        // dS [pair r16][query 4 g + r]
        *reinterpret_cast<float4*>(scr + t * 16 * SS + r16 * SS + 4 * g) =
            float4{dp[t][0], dp[t][1], dp[t][2], dp[t][3]};
      }
      if constexpr (BIAS) {
        if (p.dw != nullptr) {
          const float x = sum_groups(dwj);
          if (g == 0 && k0 + r16 < nk) p.dw[(rbase + L.kidx[j]) * N + L.kidx[k0 + r16]] = x;
        }
      }
      // G^T, H^T [d = 16 dt + 4 g + r][key k0 + r16], and the sums they enter
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) {
        mf_f32x4 gg = mf_f32x4{0.f, 0.f, 0.f, 0.f}, hh = gg;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int o = (16 * t + 4 * g + r) * KS + 16 * dt + r16;
            gg = mma(Q[o], dp[t][r], gg);
            hh = mma(GO[o], s[t][r], hh);
          }
        const float4 k2 = *reinterpret_cast<const float4*>(K2 + (k0 + r16) * KS + 16 * dt + 4 * g);
        const float4 v2 = *reinterpret_cast<const float4*>(V2 + (k0 + r16) * KS + 16 * dt + 4 * g);
        const float4 k1 = *reinterpret_cast<const float4*>(K1 + j * KS + 16 * dt + 4 * g);
        const float4 v1 = *reinterpret_cast<const float4*>(V1 + j * KS + 16 * dt + 4 * g);
        const float k2r[4] = {k2.x, k2.y, k2.z, k2.w}, v2r[4] = {v2.x, v2.y, v2.z, v2.w};
        const float k1r[4] = {k1.x, k1.y, k1.z, k1.w}, v1r[4] = {v1.x, v1.y, v1.z, v1.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          x1[dt][r] = fmaf(k2r[r], gg[r], x1[dt][r]);
          y1[dt][r] = fmaf(v2r[r], hh[r], y1[dt][r]);
          dk2a[kt][dt][r] = fmaf(k1r[r], gg[r], dk2a[kt][dt][r]);
          dv2a[kt][dt][r] = fmaf(v1r[r], hh[r], dv2a[kt][dt][r]);
        }
      }
      // dq^T: A = W^T of pairs (j, k0 + 4 g + r) at d = 16 dt + r16, B = dS of those pairs and query 16 t + r16
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float b[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) b[t] = scr[t * 16 * SS + (4 * g + r) * SS + r16];
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) {
          const float a = K1[j * KS + 16 * dt + r16] * K2[(k0 + 4 * g + r) * KS + 16 * dt + r16];
#pragma unroll
          for (int t = 0; t < NT; ++t) dqt[t][dt] = mma(a, b[t], dqt[t][dt]);
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) dqa[t][dt][r] += dqt[t][dt][r];
    // dk1_j, dv1_j at d = 16 dt + 4 g + (r16 & 3), in lanes r16 >> 2 == dt; du_ij likewise with t
    float xs = 0.0f, ys = 0.0f, us = 0.0f;
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) {
      const float a = row16_sum4(x1[dt][0], x1[dt][1], x1[dt][2], x1[dt][3], r16);
      const float b = row16_sum4(y1[dt][0], y1[dt][1], y1[dt][2], y1[dt][3], r16);
      xs = (r16 >> 2) == dt ? a : xs;
      ys = (r16 >> 2) == dt ? b : ys;
    }
    const int d = 16 * (r16 >> 2) + 4 * g + (r16 & 3);
    if (d < D) {
      const size_t o = (rbase + L.kidx[j]) * D + d;
      p.dk1[o] = xs;
      p.dv1[o] = ys;
    }
    if constexpr (BIAS) {
      if (p.du != nullptr) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const float a = row16_sum4(dus[t][0], dus[t][1], dus[t][2], dus[t][3], r16);
          us = (r16 >> 2) == t ? a : us;
        }
        const int i = 16 * (r16 >> 2) + 4 * g + (r16 & 3);  // the query index: the same lanes as d
        if (r16 < 4 * NT && i < nq) p.du[(rbase + L.qidx[i]) * N + L.kidx[j]] = X->gate[i] * us;
      }
    }
  }

  // ---- the waves' partials ----
  float* part = &L.op[0][0];  // [W][MN][KS] over the operands
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
      *reinterpret_cast<float4*>(part + wave * MN * KS + (16 * t + r16) * KS + 16 * dt + 4 * g) =
          float4{dqa[t][dt][0], dqa[t][dt][1], dqa[t][dt][2], dqa[t][dt][3]};
  __syncthreads();
  write_rows<W>(part, p.dq, L.qidx, nq, D, rbase);
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    __syncthreads();
#pragma unroll
    for (int kt = 0; kt < NK; ++kt)
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) {
        const float* a = which ? dv2a[kt][dt] : dk2a[kt][dt];
        *reinterpret_cast<float4*>(part + wave * MN * KS + (16 * kt + r16) * KS + 16 * dt + 4 * g) =
            float4{a[0], a[1], a[2], a[3]};
      }
    __syncthreads();
    write_rows<W>(part, which ? p.dv2 : p.dk2, L.kidx, nk, D, rbase);
  }
  if constexpr (BIAS) {
    __syncthreads();
    // dv_bias partials [key][query], dgate partials
#pragma unroll
    for (int kt = 0; kt < NK; ++kt)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        *reinterpret_cast<float4*>(part + wave * MN * KS + (16 * kt + r16) * KS + 16 * t + 4 * g) =
            float4{dva[kt][t][0], dva[kt][t][1], dva[kt][t][2], dva[kt][t][3]};
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float x = row16_sum4(accg[t][0], accg[t][1], accg[t][2], accg[t][3], r16);
      if (r16 < 4) X->dg[wave][16 * t + 4 * g + r16] = x;
    }
    __syncthreads();
    if (p.dvb != nullptr) {
      for (int u = threadIdx.x; u < nq * nk; u += kThreads) {
        const int i = u / nk, k = u % nk, o = k * KS + i;
        float s = part[o];
#pragma unroll
        for (int w = 1; w < W; ++w) s += part[w * MN * KS + o];
        p.dvb[(rbase + L.qidx[i]) * N + L.kidx[k]] = X->gate[i] * s;
      }
    }
    if (p.dgate != nullptr && int(threadIdx.x) < nq) {
      const int i = threadIdx.x;
      float s = X->dg[0][i];
#pragma unroll
      for (int w = 1; w < W; ++w) s += X->dg[w][i];
      p.dgate[rbase + L.qidx[i]] = s;
    }
  }
}

// Zeros at the padded entries of the gradients (mk, mq: valid keys and queries), so that the caller needs no fill:
// five launches, nine with a bias (forward and backward of 128 molecules of up to 29 atoms, 8 heads of 32: 138 -> 122
// us).  Called after the
// operand loads have arrived: a load that waits behind stores waits for them too.
template <bool BIAS, int W>
__device__ __forceinline__ void zero_padding(const Params& p, unsigned long long mk, unsigned long long mq, size_t rbase) {
  const int N = p.N, D = p.D;
  const int row = threadIdx.x / (DP / 4), c = 4 * (threadIdx.x % (DP / 4));
  if (row < N && c < D) {
    const size_t o = (rbase + row) * D + c;
    if (!((mq >> row) & 1u)) *reinterpret_cast<float4*>(p.dq + o) = float4{0.f, 0.f, 0.f, 0.f};
    if (!((mk >> row) & 1u)) {
      *reinterpret_cast<float4*>(p.dk2 + o) = float4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<float4*>(p.dv2 + o) = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e) p.dk1[o + e] = p.dv1[o + e] = 0.0f;  // (these two may be unaligned)
    }
  }
  if constexpr (BIAS) {
    for (int u = threadIdx.x; u < N * N; u += W * 64) {
      const int a = u / N, e = u % N;
      const size_t o = rbase * N + u;
      const bool k = (mk >> e) & 1u, q = k && ((mq >> a) & 1u), j = k && ((mk >> a) & 1u);
      if (p.du != nullptr && !q) p.du[o] = 0.0f;
      if (p.dvb != nullptr && !q) p.dvb[o] = 0.0f;
      if (p.dw != nullptr && !j) p.dw[o] = 0.0f;
    }
    if (p.dgate != nullptr && int(threadIdx.x) < N && !((mq >> threadIdx.x) & 1u)) p.dgate[rbase + threadIdx.x] = 0.0f;
  }
}

template <bool BIAS, int W>
__global__ void __launch_bounds__(W * 64, 2) pair_f32_bwd_kernel(Params p) {
  constexpr int kThreads = W * 64;
  extern __shared__ __attribute__((aligned(16))) unsigned char dyn[];
  Lds<W>& L = *reinterpret_cast<Lds<W>*>(dyn);
  LdsBias<W>* X = reinterpret_cast<LdsBias<W>*>(dyn + sizeof(Lds<W>));
  static_assert(sizeof(Lds<W>) % 16 == 0, "16-byte rows");
  const int N = p.N, D = p.D;
  const int tid = threadIdx.x, lane = lane_id();
  const int bh = blockIdx.x, b = bh / p.H;
  const size_t rbase = size_t(bh) * N;
  const bool vk = lane < N && p.pkv[size_t(b) * N + min(lane, N - 1)] != 0;
  const bool vq = lane < N && p.qv[size_t(b) * N + min(lane, N - 1)] != 0;
  const unsigned long long mk = __ballot(vk), mq = __ballot(vq);
  const int nk = __popcll(mk), nq = __popcll(mq);
  if (nk == 0 || nq == 0) {  // no pair or no query: every gradient is zero
    zero_padding<BIAS, W>(p, 0ull, 0ull, rbase);
    return;
  }
  const unsigned long long below = (1ull << lane) - 1ull;
  if (vk) L.kidx[__popcll(mk & below)] = lane;  // (every wave writes the same lists)
  if (vq) L.qidx[__popcll(mq & below)] = lane;
  __syncthreads();
  // ---- stage the six operands (row u / 8, 16-byte piece u % 8: one row per eight threads, the first 256) and
  // go . out ----
  static_assert(kThreads >= MN * (DP / 4) && MN * (DP / 4) % 64 == 0, "one pass of whole waves");
  if (tid < MN * (DP / 4)) {
    const int row = tid / (DP / 4), c = 4 * (tid % (DP / 4)), cc = min(c, D - 4);
    const size_t oq = (rbase + L.qidx[min(row, nq - 1)]) * D + cc, ok = (rbase + L.kidx[min(row, nk - 1)]) * D + cc;
    float4 x[6], o;
    x[0] = *reinterpret_cast<const float4*>(p.q + oq);
    x[1] = *reinterpret_cast<const float4*>(p.go + oq);
    x[2] = *reinterpret_cast<const float4*>(p.k1 + ok);
    x[3] = *reinterpret_cast<const float4*>(p.v1 + ok);
    x[4] = *reinterpret_cast<const float4*>(p.k2 + ok);
    x[5] = *reinterpret_cast<const float4*>(p.v2 + ok);
    o = *reinterpret_cast<const float4*>(p.out + oq);
    const float l = p.lse[rbase + L.qidx[min(row, nq - 1)]] * kLog2e;
    const float4 z{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 6; ++t) {
      if (row >= (t < 2 ? nq : nk) || c >= D) x[t] = z;
      *reinterpret_cast<float4*>(&L.op[t][row * KS + c]) = x[t];
    }
    float s = x[1].x * o.x;
    s = fmaf(x[1].y, o.y, s); s = fmaf(x[1].z, o.z, s); s = fmaf(x[1].w, o.w, s);
    s += dpp<kXor1>(s);
    s += dpp<kXor2>(s);
    s += dpp<0x141>(s);  // row_half_mirror: the other quad of the eight lanes
    if (c == 0) {
      L.dlt[row] = row < nq ? s : 0.0f;
      L.lse2[row] = row < nq ? l : INFINITY;
    }
    // valid keys of j (one row per eight threads: four keys each, joined over the lanes)
    uint32_t bits = 0u;
    const int j = row;
    if (j < nk) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = c + e;
        const bool on = k < nk && (p.pv == nullptr || p.pv[(size_t(b) * N + L.kidx[j]) * N + L.kidx[min(k, nk - 1)]] != 0);
        bits |= on ? 1u << k : 0u;
      }
    }
    bits |= __float_as_uint(dpp<kXor1>(__uint_as_float(bits)));
    bits |= __float_as_uint(dpp<kXor2>(__uint_as_float(bits)));
    bits |= __float_as_uint(dpp<0x141>(__uint_as_float(bits)));
    if (c == 0) L.bits[j] = bits;
  }
  if constexpr (BIAS) {
    for (int u = tid; u < MN * MN; u += kThreads) {
      const int a = u / MN, e = u % MN;
      const size_t qk = (rbase + L.qidx[min(a, nq - 1)]) * N + L.kidx[min(e, nk - 1)];
      X->ut[e * KS + a] = load_any(p.u, qk, p.bias_dtype);
      X->vt[e * KS + a] = load_any(p.v, qk, p.bias_dtype);
      X->w[a * KS + e] = load_any(p.w, (rbase + L.kidx[min(a, nk - 1)]) * N + L.kidx[min(e, nk - 1)], p.bias_dtype);
    }
    // (1 on the padding rows: there lse = inf makes P = 0 whatever finite or -inf terms it multiplies)
    if (tid < MN) X->gate[tid] = tid < nq ? load_any(p.gate, rbase + L.qidx[tid], p.bias_dtype) : 1.0f;
  }
  __syncthreads();
  zero_padding<BIAS, W>(p, mk, mq, rbase);
  if (nq > 16) {
    if (nk > 16) body<2, 2, BIAS, W>(p, L, X, nk, nq, rbase);
    else body<2, 1, BIAS, W>(p, L, X, nk, nq, rbase);
  } else {
    if (nk > 16) body<1, 2, BIAS, W>(p, L, X, nk, nq, rbase);
    else body<1, 1, BIAS, W>(p, L, X, nk, nq, rbase);
  }
}

template <bool BIAS, int W>
int launch(const Params& p, int bh, hipStream_t stream) {
  constexpr size_t lds = sizeof(Lds<W>) + (BIAS ? sizeof(LdsBias<W>) : 0);
  const int st = ensure_dynamic_lds(reinterpret_cast<const void*>(pair_f32_bwd_kernel<BIAS, W>), int(lds));
  if (st != MF_OK) return st;
  hipLaunchKernelGGL((pair_f32_bwd_kernel<BIAS, W>), dim3(unsigned(bh)), dim3(W * 64), lds, stream, p);
  MF_HIP_CHECK(hipGetLastError());
  return MF_OK;
}

// Four waves a (molecule, head), two of its workgroups to a CU; eight where every workgroup has a CU to itself.
template <bool BIAS>
int launch_for(const Params& p, int bh, int num_cus, hipStream_t stream) {
  return bh <= num_cus ? launch<BIAS, 8>(p, bh, stream) : launch<BIAS, 4>(p, bh, stream);
}

}  // namespace spf32b

// fp32 operands and grad_out of at most 32 tokens and head_dim <= 32, whole and aligned 16-byte rows, with or
// without a factorized bias.  (All rows of a molecule and both key tiles' sums stay in LDS and registers; larger
// calls and the rank terms take the ownership kernel.)
bool simplicial_pair_f32_bwd_serves(const mf_simplicial_bwd_args* a) {
  if (a->dtype != MF_DTYPE_F32 || a->grad_dtype != MF_DTYPE_F32 || a->grads_dtype != MF_DTYPE_F32) return false;
  if (a->tokens > spf32b::MN || a->head_dim > spf32b::DP || a->head_dim % 4 != 0) return false;
  if (a->angle_left != nullptr || a->message_left != nullptr) return false;
  if (!a->dq || !a->dk1 || !a->dv1 || !a->dk2 || !a->dv2) return false;
  if (int64_t(a->batch) * a->heads > 0x7fffffff) return false;
  for (const void* ptr : {a->q, a->k1, a->v1, a->k2, a->v2, a->grad_out, (const void*)a->out, (const void*)a->dq,
                          (const void*)a->dk2, (const void*)a->dv2})
    if (reinterpret_cast<uintptr_t>(ptr) % 16 != 0) return false;
  return true;
}

int simplicial_pair_f32_bwd_launch(const mf_simplicial_bwd_args* a, int num_cus, hipStream_t stream) {
  using namespace spf32b;
  Params p{};
  p.q = static_cast<const float*>(a->q);
  p.k1 = static_cast<const float*>(a->k1);
  p.v1 = static_cast<const float*>(a->v1);
  p.k2 = static_cast<const float*>(a->k2);
  p.v2 = static_cast<const float*>(a->v2);
  p.go = static_cast<const float*>(a->grad_out);
  p.out = a->out;
  p.lse = a->lse;
  p.qv = a->query_valid; p.pkv = a->pair_key_valid; p.pv = a->pair_valid;
  p.dq = static_cast<float*>(a->dq);
  p.dk1 = static_cast<float*>(a->dk1);
  p.dv1 = static_cast<float*>(a->dv1);
  p.dk2 = static_cast<float*>(a->dk2);
  p.dv2 = static_cast<float*>(a->dv2);
  p.u = a->bias_u; p.v = a->bias_v; p.w = a->bias_w; p.gate = a->bias_gate;
  p.du = static_cast<float*>(a->du);
  p.dvb = static_cast<float*>(a->dv_bias);
  p.dw = static_cast<float*>(a->dw);
  p.dgate = static_cast<float*>(a->dgate);
  p.bias_dtype = a->bias_dtype;
  p.H = a->heads; p.N = a->tokens; p.D = a->head_dim;
  const int bh = a->batch * a->heads;
  return a->bias_u != nullptr ? launch_for<true>(p, bh, num_cus, stream) : launch_for<false>(p, bh, num_cus, stream);
}

}  // namespace mf
