// 2-simplicial attention forward for fp32 operands of small molecules (at most
// 64 tokens, head_dim <= 64 and a multiple of 4) on gfx950 (CDNA4).
//
// Formulation (simplicial_attention.py:206-344): the valid pairs p = (j, k) are
// the keys of plain attention, with key W_p = k1_j (.) k2_k and value Z_p =
// v1_j (.) v2_k, so a tile of 16 pairs serves 16 queries at a time; the general
// kernel (simplicial_fwd.hip) gives every query its own nk x nk slab of 16 x 16
// tiles.  Everything is fp32: fp32 MFMA 16x16x4, fp32 softmax and sums.
//
//   S^T[pair][query] = sum_d W[pair][d] q[query][d]   pairs (j, k0 + 0..15), A = W formed in
//       registers; the K index of step c of lane group g is d = (DP / 4) g + c, so a lane's d are
//       contiguous in LDS
//   O^T[d][query]   += sum_pair Z[pair][d] P[pair][query]      accumulator r of S^T (pair 4 g + r) is the
//       B operand of K step r as it is; A = Z formed in registers
//   S += gate_i (u_ij + v_ik + w_jk) in fp32 with a factorized bias
//
// One workgroup of W waves per (molecule, head, 16 QT queries): four waves and two query tiles, or eight and one in
// small calls.  The waves split the j rows; each keeps an
// offset per query that follows its running maximum (moved only when a logit exceeds it by more than
// kRescaleSlack, for the query's four lane groups together, so P <= 2^8), and the partial (O, max, sum)
// meet in LDS at the end.  MFMA-bound: an iteration (one j, 16 keys, 32 queries, head_dim 32) is 32 MFMA of 32
// cycles against about 80 VALU instructions.  128 QM9-like molecules of 9-29 atoms, 8 heads, head_dim 32: 42 us at a
// cold clock (134 us on the general kernel; 7.7 us of fp32 MFMA for the valid work, 13 with the tiles' padding, the
// rest is the start of a workgroup -- masks, rows, barriers -- and the uneven molecules of one round).
#include <algorithm>

#include "mf_common.h"

namespace mf {
namespace spf32 {

constexpr int kMaxN = 64;               // tokens
constexpr float kRescaleSlack = 8.0f;   // log2 units
constexpr int kSmallGrid = 1;           // workgroups of one query tile per CU up to which they are taken

struct Params {
  const float* q;
  const float* k1;
  const float* v1;
  const float* k2;
  const float* v2;
  const uint8_t* qv;
  const uint8_t* pkv;
  const uint8_t* pv;
  float* out;
  float* out_f32;
  float* lse;
  const void* u;     // factorized bias, element type bias_dtype (BIAS)
  const void* v;
  const void* w;
  const void* gate;
  int bias_dtype;
  int H, N, D, NP;   // NP: N rounded up to 16
};

// LDS (floats): the four key / value operands [NP][KS], then (BIAS) u^T [NP j][16 QT i + 4], v [16 QT i][NP + 4],
// w [NP j][NP + 4]; the waves' partial outputs [W][16 QT][DP + 4] reuse the operands' place.
template <int DP, bool BIAS, int QT, int W>
struct Lay {
  static constexpr int KS = DP + 4;
  static constexpr int UI = 16 * QT + 4;
  __host__ __device__ static int operands(int NP) {
    const int rows = 4 * NP * KS, parts = W * 16 * QT * KS;
    return rows > parts ? rows : parts;
  }
  __host__ __device__ static int floats(int NP) {
    return operands(NP) + (BIAS ? NP * UI + (16 * QT + NP) * (NP + 4) : 0);
  }
};

__device__ __forceinline__ float load_any(const void* p, size_t idx, int dtype) {
  if (dtype == MF_DTYPE_F32) return static_cast<const float*>(p)[idx];
  if (dtype == MF_DTYPE_BF16) return static_cast<float>(static_cast<const __bf16*>(p)[idx]);
  return static_cast<float>(static_cast<const _Float16*>(p)[idx]);
}

// Maximum / sum over the four 16-lane groups, in every lane (gfx950 lane swaps).
__device__ __forceinline__ float max_groups(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float y = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(y), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_groups(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float y = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(y), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

__device__ __forceinline__ mf_f32x4 mma(float a, float b, mf_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The pair tiles of the wave (j = wave, wave + W, ...) against NT query tiles: offsets, sums and outputs in place.
template <int DP, bool BIAS, int QT, int W, int NT>
__device__ __forceinline__ void pair_loop(const float* smem, const unsigned long long* s_bits, int nk, int NP,
                                          const float (&qf)[QT][DP / 4], const float (&gq)[QT], float (&M)[QT],
                                          float (&lsum)[QT], mf_f32x4 (&oa)[QT][DP / 16]) {
  using L = Lay<DP, BIAS, QT, W>;
  constexpr int KS = L::KS, UI = L::UI, NC = DP / 4, ND = DP / 16;
  const int lane = lane_id(), wave = wave_id();
  const int g = lane >> 4, r16 = lane & 15;
  const float* K1s = smem;
  const float* V1s = K1s + NP * KS;
  const float* K2s = V1s + NP * KS;
  const float* V2s = K2s + NP * KS;
  const float* uT = smem + L::operands(NP);
  const float* vS = uT + NP * UI;
  const float* wS = vS + 16 * QT * (NP + 4);
  for (int k0 = 0; k0 < nk; k0 += 16) {
    // k2 of key k0 + r16 at d = NC g + c; v2 of keys k0 + 4 g + r at d = 16 dt + r16
    float k2[NC], v2[4][ND];
#pragma unroll
    for (int c = 0; c < NC; c += 4) {
      const float4 x = *reinterpret_cast<const float4*>(K2s + (k0 + r16) * KS + NC * g + c);
      k2[c] = x.x; k2[c + 1] = x.y; k2[c + 2] = x.z; k2[c + 3] = x.w;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) v2[r][dt] = V2s[(k0 + 4 * g + r) * KS + 16 * dt + r16];
    float vb[NT][4];  // BIAS: v of (query 16 t + r16, key k0 + 4 g + r)
    if constexpr (BIAS) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const float4 x = *reinterpret_cast<const float4*>(vS + (16 * t + r16) * (NP + 4) + k0 + 4 * g);
        vb[t][0] = x.x; vb[t][1] = x.y; vb[t][2] = x.z; vb[t][3] = x.w;
      }
    }
    for (int j = wave; j < nk; j += W) {
      const uint32_t bits = uint32_t(s_bits[j] >> k0) & 0xffffu;
      const bool whole = __builtin_amdgcn_readfirstlane(bits) == 0xffffu;
      float wz[NC];
#pragma unroll
      for (int c = 0; c < NC; c += 4) {
        const float4 x = *reinterpret_cast<const float4*>(K1s + j * KS + NC * g + c);
        wz[c] = x.x * k2[c]; wz[c + 1] = x.y * k2[c + 1]; wz[c + 2] = x.z * k2[c + 2]; wz[c + 3] = x.w * k2[c + 3];
      }
      float v1[ND];
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) v1[dt] = V1s[j * KS + 16 * dt + r16];
      float4 w4{0.f, 0.f, 0.f, 0.f};
      float uj[NT];
      if constexpr (BIAS) {
        w4 = *reinterpret_cast<const float4*>(wS + j * (NP + 4) + k0 + 4 * g);
#pragma unroll
        for (int t = 0; t < NT; ++t) uj[t] = uT[j * UI + 16 * t + r16];
      }
      // natural logits, in two chains of NC / 2 steps: log2 e enters with the offset, in one fma, and not as a
      // rounding of every q
      mf_f32x4 s[NT], sb[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) s[t] = sb[t] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC / 2; ++c)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          s[t] = mma(wz[c], qf[t][c], s[t]);
          sb[t] = mma(wz[NC / 2 + c], qf[t][NC / 2 + c], sb[t]);
        }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[t][r] += sb[t][r];
      if constexpr (BIAS) {
        const float wk[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) s[t][r] = fmaf(gq[t], (uj[t] + vb[t][r]) + wk[r], s[t][r]);
      }
      if (!whole) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool ok = (bits >> (4 * g + r)) & 1u;
#pragma unroll
          for (int t = 0; t < NT; ++t) s[t][r] = ok ? s[t][r] : -INFINITY;
        }
      }
      // move a query's offset when a logit of its four lane groups exceeds it by more than the slack
      float top[NT];
      bool over = false;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        top[t] = fmaxf(fmaxf(s[t][0], s[t][1]), fmaxf(s[t][2], s[t][3]));
        over = over || fmaf(top[t], kLog2e, -M[t]) > kRescaleSlack;
      }
      if (__any(over)) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const float x = max_groups(top[t]) * kLog2e;
          if (x > M[t] + kRescaleSlack) {
            const float alpha = M[t] == -INFINITY ? 0.0f : fast_exp2(M[t] - x);
            M[t] = x;
            lsum[t] *= alpha;
#pragma unroll
            for (int dt = 0; dt < ND; ++dt)
#pragma unroll
              for (int r = 0; r < 4; ++r) oa[t][dt][r] *= alpha;
          }
        }
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const float m = M[t] == -INFINITY ? 0.0f : M[t];
#pragma unroll
        for (int r = 0; r < 4; ++r) s[t][r] = fast_exp2(fmaf(s[t][r], kLog2e, -m));
        lsum[t] += (s[t][0] + s[t][1]) + (s[t][2] + s[t][3]);
      }
      // the tile's pairs are summed on their own, in two chains of 8, then added: not one long chain (error against
      // 64 bits 1.13e-7 instead of 1.8e-7, 1.2e-7 with one chain of 16 and one of logits, at no measured cost)
      mf_f32x4 ot[2][NT][ND];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) ot[0][t][dt] = ot[1][t][dt] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int dt = 0; dt < ND; ++dt) {
          const float z = v1[dt] * v2[r][dt];
#pragma unroll
          for (int t = 0; t < NT; ++t) ot[r & 1][t][dt] = mma(z, s[t][r], ot[r & 1][t][dt]);
        }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
          for (int r = 0; r < 4; ++r) oa[t][dt][r] += ot[0][t][dt][r] + ot[1][t][dt][r];
    }
  }
}

template <int DP, bool BIAS, int QT, int W>
__global__ void __launch_bounds__(W * 64, DP == 32 && W == 4 ? 4 : 2) simplicial_pair_f32_kernel(Params p) {
  constexpr int kWaves = W, kThreads = W * 64;
  using L = Lay<DP, BIAS, QT, W>;
  constexpr int KS = L::KS, UI = L::UI;
  constexpr int NC = DP / 4;    // K steps of S, and a lane's contiguous d
  constexpr int ND = DP / 16;   // 16-d tiles of O
  constexpr int C4 = DP / 4;    // 16-byte chunks per row
  extern __shared__ __attribute__((aligned(16))) float smem[];
  __shared__ int s_k[kMaxN], s_q[kMaxN];
  __shared__ unsigned long long s_bits[kMaxN];   // valid keys of each j (compacted)
  __shared__ float s_m[kWaves][16 * QT], s_l[kWaves][16 * QT];
  const int N = p.N, D = p.D, NP = p.NP;
  const int tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  const int g = lane >> 4, r16 = lane & 15;
  const int bh = blockIdx.x, b = bh / p.H;
  const size_t rbase = size_t(bh) * N;

  // ---- valid keys and queries (every wave forms the same lists) ----
  const bool vk = lane < N && p.pkv[size_t(b) * N + min(lane, N - 1)] != 0;
  const bool vq = lane < N && p.qv[size_t(b) * N + min(lane, N - 1)] != 0;
  const unsigned long long mk = __ballot(vk), mq = __ballot(vq);
  const int nk = __popcll(mk), nq = __popcll(mq);
  const unsigned long long below = (1ull << lane) - 1ull;
  // zero rows: invalid queries, and every query of a molecule without keys (the first query group's workgroup)
  if (blockIdx.y == 0 && (nq < N || nk == 0)) {
    for (int u = tid; u < N * (D / 4); u += kThreads) {
      const int row = u / (D / 4);
      if (nk > 0 && ((mq >> row) & 1ull)) continue;
      const size_t o = (rbase + row) * D + 4 * (u % (D / 4));
      const float4 z{0.f, 0.f, 0.f, 0.f};
      if (p.out) *reinterpret_cast<float4*>(p.out + o) = z;
      if (p.out_f32) *reinterpret_cast<float4*>(p.out_f32 + o) = z;
    }
    if (p.lse && tid < N && (nk == 0 || !((mq >> tid) & 1ull))) p.lse[rbase + tid] = 0.0f;
  }
  const int q0 = blockIdx.y * 16 * QT;
  if (nk == 0 || q0 >= nq) return;
  if (vk) s_k[__popcll(mk & below)] = lane;
  if (vq) s_q[__popcll(mq & below)] = lane;
  __syncthreads();
  const int nqb = min(nq - q0, 16 * QT);

  // ---- stage k1, v1, k2, v2 (compacted rows, zero past the counts and past D) ----
  float* K1s = smem;
  float* V1s = K1s + NP * KS;
  float* K2s = V1s + NP * KS;
  float* V2s = K2s + NP * KS;
  const int nrow = (nk + 15) / 16 * 16;
  for (int u0 = 0; u0 < nrow * C4; u0 += 2 * kThreads) {
    float4 xk1[2], xv1[2], xk2[2], xv2[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = u0 + tid + kThreads * i, row = u / C4, c = u % C4;
      const size_t o = (rbase + s_k[min(row, nk - 1)]) * D + min(4 * c, D - 4);  // clamped: no branch around loads
      xk1[i] = *reinterpret_cast<const float4*>(p.k1 + o);
      xv1[i] = *reinterpret_cast<const float4*>(p.v1 + o);
      xk2[i] = *reinterpret_cast<const float4*>(p.k2 + o);
      xv2[i] = *reinterpret_cast<const float4*>(p.v2 + o);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = u0 + tid + kThreads * i, row = u / C4, c = u % C4;
      if (row < nrow) {
        const int o = row * KS + 4 * c;
        if (row >= nk || 4 * c >= D) xk1[i] = xv1[i] = xk2[i] = xv2[i] = float4{0.f, 0.f, 0.f, 0.f};
        *reinterpret_cast<float4*>(K1s + o) = xk1[i];
        *reinterpret_cast<float4*>(V1s + o) = xv1[i];
        *reinterpret_cast<float4*>(K2s + o) = xk2[i];
        *reinterpret_cast<float4*>(V2s + o) = xv2[i];
      }
    }
  }
  // valid pairs: bit k of word j
  for (int j = wave; j < nk; j += kWaves) {
    const bool on = lane < nk && (p.pv == nullptr || p.pv[(size_t(b) * N + s_k[j]) * N + s_k[min(lane, nk - 1)]] != 0);
    const unsigned long long bits = __ballot(on);
    if (lane == 0) s_bits[j] = bits;
  }
  // bias terms of this query group, compacted
  float* uT = smem + L::operands(NP);
  float* vS = uT + NP * UI;
  float* wS = vS + 16 * QT * (NP + 4);
  if constexpr (BIAS) {
    for (int t = tid; t < 16 * QT * NP; t += kThreads) {
      const int i = t / NP, j = t % NP;
      const size_t o = (rbase + s_q[q0 + min(i, nqb - 1)]) * N + s_k[min(j, nk - 1)];
      uT[j * UI + i] = load_any(p.u, o, p.bias_dtype);
      vS[i * (NP + 4) + j] = load_any(p.v, o, p.bias_dtype);
    }
    for (int t = tid; t < nk * NP; t += kThreads) {
      const int j = t / NP, k = t % NP;
      wS[j * (NP + 4) + k] = load_any(p.w, (rbase + s_k[j]) * N + s_k[min(k, nk - 1)], p.bias_dtype);
    }
  }
  // ---- the queries' operand: q of query 16 t + r16 at d = NC g + c (zero past nqb and D) ----
  float qf[QT][NC], gq[QT];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int i = 16 * t + r16;
    const size_t row = rbase + s_q[q0 + min(i, nqb - 1)];
#pragma unroll
    for (int c = 0; c < NC; c += 4) {
      const int d = NC * g + c;
      const float4 x = *reinterpret_cast<const float4*>(p.q + row * D + min(d, D - 4));
      const bool on = i < nqb && d < D;
      qf[t][c] = on ? x.x : 0.0f;
      qf[t][c + 1] = on ? x.y : 0.0f;
      qf[t][c + 2] = on ? x.z : 0.0f;
      qf[t][c + 3] = on ? x.w : 0.0f;
    }
    gq[t] = BIAS ? load_any(p.gate, row, p.bias_dtype) : 0.0f;
  }
  __syncthreads();

  float M[QT], lsum[QT];
  mf_f32x4 oa[QT][ND];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    M[t] = -INFINITY;
    lsum[t] = 0.0f;
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) oa[t][dt] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (QT == 1 || nqb <= 16) pair_loop<DP, BIAS, QT, W, 1>(smem, s_bits, nk, NP, qf, gq, M, lsum, oa);
  else pair_loop<DP, BIAS, QT, W, QT>(smem, s_bits, nk, NP, qf, gq, M, lsum, oa);

  // ---- the waves' partials: offsets and sums first, then the outputs scaled to the largest offset ----
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const float l = sum_groups(lsum[t]);
    if (g == 0) {
      s_m[wave][16 * t + r16] = M[t];
      s_l[wave][16 * t + r16] = l;
    }
  }
  __syncthreads();  // also: every wave is done with the operands
  float* part = smem;
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int i = 16 * t + r16;
    float mx = s_m[0][i];
#pragma unroll
    for (int w = 1; w < W; ++w) mx = fmaxf(mx, s_m[w][i]);
    const float f = M[t] == -INFINITY ? 0.0f : fast_exp2(M[t] - mx);
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
      *reinterpret_cast<float4*>(part + (wave * 16 * QT + i) * KS + 16 * dt + 4 * g) =
          float4{oa[t][dt][0] * f, oa[t][dt][1] * f, oa[t][dt][2] * f, oa[t][dt][3] * f};
  }
  __syncthreads();
  for (int u = tid; u < nqb * (D / 4); u += kThreads) {
    const int i = u / (D / 4), c = 4 * (u % (D / 4));
    float mx = s_m[0][i];
#pragma unroll
    for (int w = 1; w < W; ++w) mx = fmaxf(mx, s_m[w][i]);
    float l = 0.0f;
    float4 o{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      l += s_m[w][i] == -INFINITY ? 0.0f : s_l[w][i] * fast_exp2(s_m[w][i] - mx);
      const float4 x = *reinterpret_cast<const float4*>(part + (w * 16 * QT + i) * KS + c);
      o.x += x.x; o.y += x.y; o.z += x.z; o.w += x.w;
    }
    const bool mass = l > 0.0f;
    const float inv = mass ? 1.0f / l : (l == l ? 0.0f : l);
    o.x *= inv; o.y *= inv; o.z *= inv; o.w *= inv;
    const size_t row = rbase + s_q[q0 + i];
    if (p.out) *reinterpret_cast<float4*>(p.out + row * D + c) = o;
    if (p.out_f32) *reinterpret_cast<float4*>(p.out_f32 + row * D + c) = o;
    if (p.lse && c == 0) p.lse[row] = mass ? (mx + __log2f(l)) * kLn2 : 0.0f;
  }
}

template <int DP, bool BIAS, int QT, int W>
int launch(const Params& p, int bh, hipStream_t stream) {
  using L = Lay<DP, BIAS, QT, W>;
  const size_t lds = size_t(L::floats(p.NP)) * 4;
  const int st = ensure_dynamic_lds(reinterpret_cast<const void*>(simplicial_pair_f32_kernel<DP, BIAS, QT, W>),
                                    L::floats(kMaxN) * 4);
  if (st != MF_OK) return st;
  hipLaunchKernelGGL((simplicial_pair_f32_kernel<DP, BIAS, QT, W>),
                     dim3(unsigned(bh), unsigned((p.N + 16 * QT - 1) / (16 * QT))), dim3(W * 64), lds, stream, p);
  MF_HIP_CHECK(hipGetLastError());
  return MF_OK;
}

// Two query tiles a workgroup of four waves share each W and Z; where that leaves CUs without work, one tile a
// workgroup of eight waves: twice the workgroups of twice the waves.  8 heads, head_dim 32, one molecule of 32 / 48 /
// 64 tokens 19 / 35 / 59 us -> 11 / 20 / 31; 16 of 32 tokens (256 workgroups) 20 -> 12, 16 of 64 (1024) 62 -> 55, 64
// of 29 tokens (1024) 30 -> 31.  Sixteen waves: 12 / 20 / 30, the matrix cores of a workgroup's CU are busy.
template <int DP, bool BIAS>
int launch_for(const Params& p, int bh, int num_cus, hipStream_t stream) {
  if (long(bh) * ((p.N + 15) / 16) <= kSmallGrid * num_cus) return launch<DP, BIAS, 1, 8>(p, bh, stream);
  return launch<DP, BIAS, 2, 4>(p, bh, stream);
}

}  // namespace spf32

// fp32 operands of at most 64 tokens and head_dim 64, rows of whole 16-byte pieces, with or without a factorized bias.
// (The limit is the LDS that all keys of a molecule take; longer rows and the rank terms stay on the general kernel.)
// A few (molecule, head) of 49 .. 64 tokens without a bias do too: it spreads them over one wave per query where
// the pair form has four workgroups each (8 heads, one molecule of 64 tokens, head_dim 32 / 64: 23 / 39 us
// against 31 / 51; four of 56: 25 / 41 against 29 / 46; eight of 64, 45 / 80 against 32 / 52; 48 tokens 30 / 49 against
// 20 / 31; with a bias, one of 64, 43 / 57 against 36 / 55).
bool simplicial_pair_f32_range(int dtype, int64_t batch_heads, int tokens, int head_dim, bool bias) {
  if (dtype != MF_DTYPE_F32 || tokens > spf32::kMaxN || head_dim > 64 || head_dim % 4 != 0) return false;
  return bias || tokens <= 48 || batch_heads > 32;
}

bool simplicial_pair_f32_serves(const mf_simplicial_fwd_args* a) {
  if (!simplicial_pair_f32_range(a->dtype, int64_t(a->batch) * a->heads, a->tokens, a->head_dim, a->bias_u != nullptr))
    return false;
  if (a->angle_left != nullptr || a->message_left != nullptr) return false;
  if (int64_t(a->batch) * a->heads > 0x7fffffff) return false;
  for (const void* ptr : {a->q, a->k1, a->v1, a->k2, a->v2, (const void*)a->out, (const void*)a->out_f32})
    if (reinterpret_cast<uintptr_t>(ptr) % 16 != 0) return false;
  return true;
}

int simplicial_pair_f32_launch(const mf_simplicial_fwd_args* a, int num_cus, hipStream_t stream) {
  using namespace spf32;
  Params p{};
  p.q = static_cast<const float*>(a->q);
  p.k1 = static_cast<const float*>(a->k1);
  p.v1 = static_cast<const float*>(a->v1);
  p.k2 = static_cast<const float*>(a->k2);
  p.v2 = static_cast<const float*>(a->v2);
  p.qv = a->query_valid; p.pkv = a->pair_key_valid; p.pv = a->pair_valid;
  p.out = static_cast<float*>(a->out); p.out_f32 = a->out_f32; p.lse = a->lse;
  p.u = a->bias_u; p.v = a->bias_v; p.w = a->bias_w; p.gate = a->bias_gate;
  p.bias_dtype = a->bias_dtype;
  p.H = a->heads; p.N = a->tokens; p.D = a->head_dim;
  p.NP = (a->tokens + 15) / 16 * 16;
  const int bh = a->batch * a->heads;
  if (a->head_dim <= 32)
    return a->bias_u ? launch_for<32, true>(p, bh, num_cus, stream) : launch_for<32, false>(p, bh, num_cus, stream);
  return a->bias_u ? launch_for<64, true>(p, bh, num_cus, stream) : launch_for<64, false>(p, bh, num_cus, stream);
}

}  // namespace mf
