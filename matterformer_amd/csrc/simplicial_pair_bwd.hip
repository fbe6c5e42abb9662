// 2-simplicial attention backward, pair formulation, for bf16 operands and
// head_dim 64 on gfx950 (CDNA4), molecules of any size up to 512 tokens,
// deterministic (no floating-point atomics).
//
// The gradient of simplicial_attention.py:206-344 (the quantities of
// triton_simplicial_attention.py:332-782) with the key pairs p = (j, k) as
// the keys of an ordinary attention:
//   W_p = k1_j (.) k2_k,  Z_p = v1_j (.) v2_k,  S_ip = q_i . W_p,
//   P_ip = exp(S_ip - lse_i),  dP_ip = go_i . Z_p,  dS_ip = P_ip (dP_ip - go_i . out_i)
//   dq_i  = sum_p dS_ip W_p                         (contraction over pairs)
//   G_p   = sum_i dS_ip q_i,  H_p = sum_i P_ip go_i   (contractions over queries)
//   dk1_j = sum_k G_jk (.) k2_k,  dk2_k = sum_j G_jk (.) k1_j
//   dv1_j = sum_k H_jk (.) v2_k,  dv2_k = sum_j H_jk (.) v1_j
// Five products of n^3 D multiply-adds, against eleven when every index
// recomputes the scores it owns (simplicial_bwd.hip).
//
// Units.  lse and go . out are given, so every (query block, j block, k block)
// of a molecule is independent work.  A unit (one workgroup of four waves) is
// a run of the j keys of one (molecule, head); it walks its j in blocks of at
// most 24, and for each the query and k blocks of at most 64 rows (48 with a
// bias; one of each for most molecules).  A block triple is staged in LDS
// (78 KB, so two workgroups share a CU and each SIMD holds two waves: with one
// wave a SIMD issued an instruction every ~7 cycles, and one unit's staging
// latency was another's idle time), then
//   for each 16-key tile k0 .. k0 + 15, each wave takes the key pairs
//   (j, j + 1) = (2 jp, 2 jp + 1), jp = wave, wave + 4, ..., in three steps:
//   S, dP   C[i][k] = sum_d A[i][d] B[d][k]   A = q / go rows (LDS), B = W / Z
//           of (j, the tile), formed in registers (MFMA 16x16x32 f16), for
//           every 16-query tile; P and dS are kept as packed fp16
//   G^T, H^T (key x d) += dS^T / P^T [k][i] q / go [i][d], 16 d at a time: the
//           S accumulators of two query tiles are the A operand as they are
//           (K = 32 queries), the B operand (transposed reads) serves both j
//   dq_i   += dS[i][p] W[p][d], K = the 32 pairs, dS turned through a per-wave
//           LDS scratch (transposed read).
// The steps keep a wave's registers under 256 (two waves per SIMD) although
// both j share every row read from LDS.
// dk1_j / dv1_j (sums over the tile's keys) are added to the wave's own LDS
// rows of j: each lane sums 4 keys, and the four lane groups' partials of the
// four 16-d tiles meet in a transposing reduction (3 lane swaps and 3 adds per
// four values) that leaves d = lane in every lane, so a row is updated by one
// full-wave read and write.  dk2 / dv2 of the tile's keys accumulate over the
// wave's j in registers, dq over every pair; the four waves' partials are
// added in a fixed order.  Every sum has a fixed order: two calls give
// identical bits.
//
// Measured (64 GEOM-like molecules of mean 44 atoms, 8 heads, kernel time):
// 117 us without a bias (191 us when one wave per SIMD held both j, the
// products' operands and all query tiles in 470 registers, and a unit had a
// whole CU), 219 us with a bf16 bias and 252 with a fp32 one (365 us and
// 1.88 ms on the kernels that served them before); four molecules of 192
// atoms, 12 heads, bf16 bias: 1.12 ms (5.47 ms on the ownership kernel).
// Registers: a spill waits on memory that two waves per SIMD cannot cover (a
// variant with many in the loop took twice the time); 2 of the 256 are spilled
// without a bias, 11 with one, all in the staging code.
//
// Schedule.  The prepare launch's first workgroup counts every molecule's
// valid keys and queries, picks the j per unit (24, 12 or 6, with a bias 16, 8
// or 4: by an estimate of the time the units take on the chip's 512 slots) and
// writes the unit list longest first (LPT); its other workgroups write the
// zero rows of 16-bit gradients.
// The units of a molecule own their dk1 / dv1 rows; where a molecule has more
// than one block triple, dq, dk2 and dv2 are summed in the unit's slab of the
// workspace (read back by the thread that wrote it) and a finish launch adds
// the slabs, and the units' partial bias sums, in unit order.  (Handing the
// sums over inside the kernel would
// need a device-scope release and acquire per unit, which on this part write
// back and invalidate the whole L2 of the XCD and held each workgroup's CU
// for tens of microseconds.)
//
// Precision.  The rows are staged as fp16 scaled by powers of two, one per
// operand and block, that bring each operand's largest magnitude into [1, 2)
// (bf16 values convert exactly; entries below 2^-14 of the largest lose low
// bits as fp16 subnormals, which moves a dot product by at most 2^-24 of its
// largest term), so that one v_pk_mul_f16 forms two pair products and the
// MFMAs are 16x16x32 f16 with fp32 accumulation.  Infinities and NaN stay what
// they are and do not enter the scales:
//   W for S and for dq: k1 k2 rounded to fp16 (the reference backward rounds
//     the score products to bf16, triton_simplicial_attention.py:546-551);
//   Z for dP: hi + lo, both fp16: hi = v1 v2 rounded, lo = fma(v1, v2, -hi),
//     exact (the product of two bf16 values has at most 16 significant
//     bits), since dP - go . out cancels when one pair dominates the softmax
//     (the reference's dP contraction is fp32, :611-645);
//   dS (scaled by 2^-es) and P (by 2^kPScale) as MFMA operands: rounded once
//     to fp16, to nearest: a softmax spread over n^2 pairs has P near n^-2,
//     below fp16's normal range from 128 atoms on, and truncation's one-sided
//     error does not average out in dv1 and dv2 (512 atoms, flat logits: 8.7e-3
//     unscaled and truncated, 1.7e-3 so).  es is
//     chosen per block triple so that |dS 2^-es| < 2^15 P: from the scales of
//     go, v1 and v2, which bound |dP| in the block, and from the largest
//     |go . out| of its queries, which sums over every key of the molecule
//     and may be far larger;
//   softmax, dS, every accumulator and every bias sum fp32; the scales are
//   undone, exactly, before block triples are added.
//
// Factorized bias (BIAS 1: bf16, 2: fp32 terms): S += gate_i (u_ij + v_ik +
// w_jk) with u staged transposed in LDS as fp32, v read per key tile into
// registers, w per pair (fetched one pair ahead).  du (sum over the tile's
// keys, a transposing reduction over 16 lanes), dv_bias (registers over the
// wave's j), dgate and dw all come from the fp32 dS.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "mf_common.h"

namespace mf {
namespace pbwd {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int DP = 64;            // head_dim
constexpr int KS = DP + 8;        // fp16 row stride of the staged rows (144 B)
constexpr int SS = 16 + 4;        // fp16 row stride of the dS scratch (40 B)
constexpr int PS = DP + 4;        // fp32 row stride of the waves' partial sums
constexpr int kMaxTokens = 512;
constexpr int kMaxPlanBatch = 2048;
constexpr int kPlanThreads = 1024;
constexpr int kPScale = 12;       // P 2^12: exact to fp16's 11 bits down to 2^-26, room to 2^4 above

struct Params {
  const __bf16* q;
  const __bf16* k1;
  const __bf16* v1;
  const __bf16* k2;
  const __bf16* v2;
  const __bf16* go;
  const float* out;
  const float* lse;
  const uint8_t* pv;
  void* dq;               // gradients, fp32 or (gout16) bf16
  void* dk1;
  void* dv1;
  void* dk2;
  void* dv2;
  int gout16;             // dq .. dv2 are bf16
  int bout16;             // du .. dgate are bf16
  const int* head;        // plan: [0] units in the list, [1] j per unit
  const uint32_t* units;  // plan: (b H + h) << 6 | part, longest first
  const int2* counts;     // plan: [B] valid keys, valid queries
  const uint16_t* lists;  // plan: [B][2][N] their atoms
  float* slab;            // [B*H][cap parts][3][N][DP] partial dq, dk2, dv2 (compacted rows)
  // factorized bias (BIAS kernels): S += gate_i (u_ij + v_ik + w_jk), u / v / w [B*H, N, N], gate [B*H, N],
  // bf16 or fp32; gradients fp32 or (gout16) bf16, NULL = not wanted
  const void* bu;
  const void* bv;
  const void* bw;
  const void* bg;
  void* du;
  void* dvb;
  void* dw;
  void* dgate;
  float* dwpart;          // [B*H][N j][N k] dw of the earlier query blocks (compacted)
  float* dvpart;          // [B*H][cap parts][N i][N k] sums over the part's j of dS
  float* dgpart;          // [B*H][cap parts][N i] sums over the part's (j, k) of dS (u + v + w)
  int H, N, cap;
};

// Workspace of the pair path (16-byte aligned regions): what the call uses, no more.  The partial sums of the bias
// gradients are laid out for those that are wanted (dw's only where a molecule can have a second query block).
constexpr size_t kWsTarget = size_t(1) << 30;                   // bytes that any call may take, and per (molecule,
constexpr size_t kWsPerHead = 420 << 10, kWsPerHeadBias = 1 << 20;  // head) what a large one may
constexpr size_t kWsLimit = size_t(48) << 30;                   // calls past it take the ownership kernel
struct Ws {
  int cap;  // units per (molecule, head) at most
  bool dv, dg, dw;
  size_t units, counts, lists, slab, dvpart, dgpart, dwpart, bytes;
  Ws(int B, int H, int N, bool bias, bool dv_, bool dg_, bool dw_);
  explicit Ws(const mf_simplicial_bwd_args* a)
      : Ws(a->batch, a->heads, a->tokens, a->bias_u != nullptr, a->dv_bias != nullptr, a->dgate != nullptr,
           a->dw != nullptr) {}
  size_t layout(int B, size_t bh, size_t n);
};

struct PlanParams {
  const uint8_t* qv;
  const uint8_t* pkv;
  int* head;        // [0] units, [1] j per unit
  uint32_t* units;
  int2* counts;     // [B] (valid keys, valid queries)
  uint16_t* lists;  // [B][2][N] valid key atoms, valid query atoms
  void* dq;         // 16-bit gradients: zero rows are written here (NULL: fp32 gradients, filled by the caller)
  void* dk1;
  void* dv1;
  void* dk2;
  void* dv2;
  int B, H, N, cap;
  int jm;           // j per unit at most
  int bias;
};

// LDS layout (bytes).  A block has at most QM query, JM j and KM k rows: 64, 24 and 64 without a bias; the bias
// terms leave LDS and registers for 48, 16 and 48.  The scratch of the main loop, and between key tiles and at a triple's end the partial
// sums of dk2, dv2 and dq, share one region.
template <bool BIAS>
struct Lay {
  static constexpr int QM = BIAS ? 48 : 64;
  static constexpr int JM = BIAS ? 16 : 24;
  static constexpr int KM = BIAS ? 48 : 64;
  static constexpr int KU = QM + 4;                                             // fp32 row stride of u^T, v^T, du
  static constexpr int KW = KM + 4;                                             // fp32 row stride of w / dw
  static constexpr int kRows = 2 * QM + 2 * JM + 2 * KM;                        // q, go, k1, v1, k2, v2
  static constexpr size_t rows = 0;                                             // [kRows][KS] fp16
  static constexpr size_t acc1 = rows + size_t(kRows) * KS * 2;                 // [2][JM][64] f32 dk1, dv1
  static constexpr size_t scr = acc1 + size_t(2) * JM * DP * 4;                 // [4 waves][16][PS] f32 / scratch
  static constexpr size_t scr_bytes = size_t(kWaves) * (QM / 16 * 32 * SS * 2 > 16 * PS * 4 ? QM / 16 * 32 * SS * 2 : 16 * PS * 4);
  static constexpr size_t ut = scr + scr_bytes;                                 // BIAS: [JM][KU] f32 u^T
  static constexpr size_t dut = ut + (BIAS ? size_t(JM) * KU * 4 : 0);          // BIAS: [JM][KU] f32 sums of dS over k
  static constexpr size_t wd = dut + (BIAS ? size_t(JM) * KU * 4 : 0);          // BIAS: [JM][KW] f32 w, then dw
  static constexpr size_t vt = wd + (BIAS ? size_t(JM) * KW * 4 : 0);           // BIAS: [KM][KU] f32 v^T
  static constexpr size_t gt = vt + (BIAS ? size_t(KM) * KU * 4 : 0);           // BIAS: [QM] f32 gate log2 e
  static constexpr size_t lse2 = gt + (BIAS ? QM * 4 : 0);                      // [QM] f32
  static constexpr size_t dlt = lse2 + QM * 4;                                  // [QM] f32 go . out
  static constexpr size_t dls = dlt + QM * 4;                                   // [QM] f32 go . out 2^(-es - kPScale)
  static constexpr size_t pvb = dls + QM * 4;                                   // [JM][8] bytes: pair bits
  static constexpr size_t jidx = pvb + JM * 8;                                  // [JM] i32
  static constexpr size_t kidx = jidx + JM * 4;                                 // [KM] i32
  static constexpr size_t qidx = kidx + KM * 4;                                 // [QM] i32
  static constexpr size_t red = qidx + QM * 4;                                  // [4 waves][8] u32 operand maxima
  static constexpr size_t bytes = red + kWaves * 8 * 4;
  static_assert(bytes <= 80 * 1024, "two workgroups per CU");
  static_assert(!BIAS || size_t(kWaves) * QM * 16 * 4 <= scr_bytes, "the waves' dv_bias partials of a key tile fit");
};

// ceil(n / d), n below 2^12: (n + d - 1/2) / d is at least 1 / (2 d) from a whole number, far past the rounding of
// the reciprocal.  (An integer division is some forty instructions; the plan makes a chain of them per molecule.)
__device__ __forceinline__ int ceil_div_small(int n, int d) {
  return int((float(n + d) - 0.5f) * __builtin_amdgcn_rcpf(float(d)));
}
inline Ws::Ws(int B, int H, int N, bool bias, bool dv_, bool dg_, bool dw_)
    : dv(dv_), dg(dg_), dw(dw_ && N > Lay<true>::QM) {
  const size_t bh = size_t(B) * H, n = size_t(N);
  // a few units per CU are enough: large batches get four per (molecule, head) (256 molecules of 80 tokens, 8 heads,
  // 1983 us in three of 28 rows, 1850 in four of 20), with a bias, whose blocks of 16 j cost more than their rounds,
  // three (3370 us, in four 3800); small ones as many as give 2048 units (4 j each at the least); fewer where the
  // partial sums would pass the target
  const size_t target = std::max(kWsTarget, bh * (bias ? kWsPerHeadBias : kWsPerHead));
  cap = int(std::min<size_t>(std::min<size_t>(std::max<size_t>(bias ? 3 : 4, 2048 / bh), (n + 3) / 4), 64));
  while (layout(B, bh, n) > target && cap > 1) --cap;
}
inline size_t Ws::layout(int B, size_t bh, size_t n) {
  units = 16;
  counts = units + ((bh * cap * 4 + 15) & ~size_t(15));
  lists = counts + size_t(B) * 8;
  slab = (lists + size_t(B) * 2 * n * 2 + 255) & ~size_t(255);
  dvpart = slab + bh * cap * 3 * n * DP * 4;
  dgpart = dvpart + (dv ? bh * cap * n * n * 4 : 0);
  dwpart = (dgpart + (dg ? bh * cap * n * 4 : 0) + 15) & ~size_t(15);
  bytes = dwpart + (dw ? bh * n * n * 4 : 0);
  return bytes;
}

// Units of a molecule and their j: about `jt` j per unit, at most `cap` units, and no more than their rounds of four key
// pairs ask for (a round takes its time with one pair too: 72 j in four units of 18 are twelve rounds, in three of
// 24 nine); the pairs are shared out evenly.
__device__ __forceinline__ int rounds_of(int pairs, int parts) { return (ceil_div_small(pairs, parts) + kWaves - 1) / kWaves; }
__device__ __forceinline__ int parts_of(int nk, int jt, int cap) {
  const int pairs = (nk + 1) / 2, most = min(cap, ceil_div_small(nk, jt));
  const int parts = ceil_div_small(pairs, kWaves * rounds_of(pairs, most));
  return ceil_div_small(pairs, ceil_div_small(pairs, parts));
}
__device__ __forceinline__ int unit_rows(int nk, int parts) { return 2 * ceil_div_small((nk + 1) / 2, parts); }
// Blocks of a run of n rows, at most m rows (a multiple of 16) each, cut at multiples of 16.
__device__ __forceinline__ int blocks_of(int n, int m) { return (n + m - 1) / m; }
__device__ __forceinline__ int block_rows(int n, int blocks) { return 16 * (((n + 15) / 16 + blocks - 1) / blocks); }

// Relative cost of one unit: for each j block, per key tile and query block the sums that end the tile, and without a
// bias the staging and slab sums of further block triples; for each round of four key pairs, per key tile a fixed part
// for each query block, and the query tiles.  Two units to a CU take about 0.25 us of it without a bias (22 rows of 44
// tokens: 42 us, of 64: 59; of 128: 197 in three rounds, 104 in one), 0.5 us with one (12 rows of 24: 25 us, 16 of 48:
// 45, 16 of 64: 100; 16 of 192: 700, 8 of 192: 530).
struct UnitCost {
  int block, round;
  __device__ __forceinline__ UnitCost(int nk, int nq, int bias) {
    const int nqt = (nq + 15) / 16, nkt = (nk + 15) / 16;
    if (bias) {
      const int nqb = blocks_of(nq, Lay<true>::QM);
      block = nkt * 14 * nqb;
      round = nkt * (nqb + 2 * nqt);
    } else {
      const int nqb = blocks_of(nq, Lay<false>::QM), nkb = blocks_of(nk, Lay<false>::KM);
      block = nkt * 16 * nqb + 25 * (nqb * nkb - 1);
      round = nkt * (6 * nqb + 2 * nqt);
    }
  }
  // a unit of that many rounds
  __device__ __forceinline__ int unit(int rounds, int jm) const {
    return ceil_div_small(rounds, jm / (2 * kWaves)) * block + rounds * round;
  }
};

typedef __attribute__((__vector_size__(4 * sizeof(_Float16)))) _Float16 mf_f16x4;

__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_u16(uint16_t w) { return __uint_as_float(uint32_t(w) << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 mf_bf16x2;

// One gradient element, fp32 or rounded to bf16.
__device__ __forceinline__ void store_grad(void* base, size_t i, float v, int bf16) {
  if (bf16) static_cast<__bf16*>(base)[i] = __bf16(v);
  else static_cast<float*>(base)[i] = v;
}

// Largest magnitude of eight bf16 (as the 15-bit pattern: for positive values bit order is value order); FINITE
// leaves infinities and NaN out.
template <bool FINITE>
__device__ __forceinline__ uint32_t absmax_bits8(const uint4 r) {
  uint32_t m = 0u;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = i == 0 ? r.x : (i == 1 ? r.y : (i == 2 ? r.z : r.w));
    const uint32_t lo = w & 0x7fffu, hi = (w >> 16) & 0x7fffu;
    m = max(m, max(FINITE && lo >= 0x7f80u ? 0u : lo, FINITE && hi >= 0x7f80u ? 0u : hi));
  }
  return m;
}

// Exponent of the largest magnitude (its bf16 pattern), -127 for an all-zero operand: scaling by 2^-e puts the
// largest magnitude in [1, 2).
__device__ __forceinline__ int scale_exp(uint32_t bits) { return int((bits >> 7) & 0xffu) - 127; }

typedef __attribute__((__vector_size__(2 * sizeof(float)))) float mf_f32x2;
typedef __attribute__((__vector_size__(2 * sizeof(_Float16)))) _Float16 mf_f16x2;

// Two fp16, rounded to nearest.
__device__ __forceinline__ uint32_t pack_f16(float a, float b) {
  uint32_t r;
  asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// 2^e for a uniform e (held to the normal range), by scalar operations.
__device__ __forceinline__ float pow2(int e) { return __uint_as_float(uint32_t(min(max(e, -126), 127) + 127) << 23); }

// The exponent of dS, dS 2^-es in fp16.  dP is a sum of 64 products of magnitude below 2^(eg + f1 + f2 + 3), so
// |dP 2^-es| < 2^14 from es = eg + f1 + f2 - 5 on; |go . out| < 2^(ed + 1) needs es = ed - 13 for the same bound.
// Held where 2^-es and 2^es are finite (gradients past either end leave the fp32 range themselves).
__device__ __forceinline__ int ds_exp(int eg, int f1, int f2, int ed) {
  return min(max(max(eg + f1 + f2 - 5, ed - 13), -110), 110);
}

// Eight bf16 times 2^-e (exact) as fp16 (exact in the normal fp16 range).
__device__ __forceinline__ uint4 to_f16x8(const uint4 r, float scale) {
  const auto p0 = __builtin_amdgcn_cvt_pkrtz(bf_lo(r.x) * scale, bf_hi(r.x) * scale);
  const auto p1 = __builtin_amdgcn_cvt_pkrtz(bf_lo(r.y) * scale, bf_hi(r.y) * scale);
  const auto p2 = __builtin_amdgcn_cvt_pkrtz(bf_lo(r.z) * scale, bf_hi(r.z) * scale);
  const auto p3 = __builtin_amdgcn_cvt_pkrtz(bf_lo(r.w) * scale, bf_hi(r.w) * scale);
  return uint4{__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1), __builtin_bit_cast(uint32_t, p2),
               __builtin_bit_cast(uint32_t, p3)};
}

__device__ __forceinline__ mf_f16x8 cat8(const mf_f16x4 a, const mf_f16x4 b) {
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

__device__ __forceinline__ mf_f32x4 mma(const mf_f16x8& a, const mf_f16x8& b, const mf_f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Workgroup barrier that orders LDS accesses only: unlike __syncthreads() it does not wait for this thread's
// outstanding global stores (no workgroup reads back what these kernels store to global memory).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// DPP lane moves within rows of 16 (VALU, no LDS): quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror,
// row_mirror, row_ror 4 and 8.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
  return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), CTRL, 0xf, 0xf, false));
}
constexpr int kDppXor1 = 0xb1, kDppXor2 = 0x4e, kDppHalfMirror = 0x141, kDppMirror = 0x140;
constexpr int kDppRor4 = 0x124, kDppRor8 = 0x128;

// Maximum over the wave in every lane: within rows by DPP, across the four rows by the gfx950 lane swaps.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = max(v, dpp<kDppXor1>(v));
  v = max(v, dpp<kDppXor2>(v));
  v = max(v, dpp<kDppHalfMirror>(v));
  v = max(v, dpp<kDppMirror>(v));
  const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  v = max(uint32_t(a[0]), uint32_t(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return max(uint32_t(b[0]), uint32_t(b[1]));
}

// Sum over each aligned group of 8 lanes, in every lane of the group (pairs, quads, then the two quads).
__device__ __forceinline__ float sum8(float x) {
  x += __uint_as_float(dpp<kDppXor1>(__float_as_uint(x)));
  x += __uint_as_float(dpp<kDppXor2>(__float_as_uint(x)));
  return x + __uint_as_float(dpp<kDppHalfMirror>(__float_as_uint(x)));
}

// Sums over the four 16-lane groups of four values at once: lane group g returns the sum of x[g], added as
// (g0 + g2) + (g1 + g3).  Each lane swap leaves two values' halves where one add joins both.
__device__ __forceinline__ float sum_groups4(const float x0, const float x1, const float x2, const float x3) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x0), __float_as_uint(x2), false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x1), __float_as_uint(x3), false, false);
  const float y = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const float z = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  const auto c = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(z), false, false);
  return __uint_as_float(c[0]) + __uint_as_float(c[1]);
}

// Sum over the four lane groups, in every lane.
__device__ __forceinline__ float sum_groups(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float y = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(y), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Sum over each 16-lane row, in every lane of the row.
__device__ __forceinline__ float row16_sum(float x) {
  x = sum8(x);
  return x + __uint_as_float(dpp<kDppMirror>(__float_as_uint(x)));
}

// Sums over each 16-lane row of four values: lane r16 returns the sum of v[r16 & 3].  Two exchange steps leave that
// value in the lane, two rotations finish the sum.
__device__ __forceinline__ float row16_sum4(const float (&v)[4], int r16) {
  const bool o1 = (r16 & 1) != 0, o2 = (r16 & 2) != 0;
  float w[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float keep = o1 ? v[2 * h + 1] : v[2 * h], send = o1 ? v[2 * h] : v[2 * h + 1];
    w[h] = keep + __uint_as_float(dpp<kDppXor1>(__float_as_uint(send)));
  }
  const float keep = o2 ? w[1] : w[0], send = o2 ? w[0] : w[1];
  float x = keep + __uint_as_float(dpp<kDppXor2>(__float_as_uint(send)));
  x += __uint_as_float(dpp<kDppRor4>(__float_as_uint(x)));
  return x + __uint_as_float(dpp<kDppRor8>(__float_as_uint(x)));
}

// One bias element as fp32 (BIAS 1: bf16, 2: fp32).
template <int BIAS>
__device__ __forceinline__ float load_bias(const void* p, size_t i) {
  if constexpr (BIAS == 2) return static_cast<const float*>(p)[i];
  else return bf_u16(static_cast<const uint16_t*>(p)[i]);
}

// The prepare launch.  Workgroup 0 makes the unit list: mask rows r = 2 b (valid keys of molecule b) and
// 2 b + 1 (valid queries) are read four per wave at a time, every byte load issued before the first ballot; each
// row's count and its list of atoms go to the workspace.  Then the j per unit, the LPT rank of each molecule
// (unit cost descending, ties by index) and its list positions = prefix sums of the units ranked before it.
// Workgroups 1 .. B H (16-bit gradients): the zero rows of one (molecule, head) each -- padded queries (dq) and
// keys (dk1, dv1, dk2, dv2), and every row of a molecule without a valid query or key.
__global__ void __launch_bounds__(kPlanThreads) pair_bwd_prepare(PlanParams pp) {
  __shared__ uint32_t s_cost[kMaxPlanBatch];
  __shared__ int s_units[kMaxPlanBatch];
  __shared__ int s_count[2 * kMaxPlanBatch];
  __shared__ int s_total;
  __shared__ float s_level[kPlanThreads / 64][3][3];  // units, largest cost, sum of costs at each j per unit, by wave
  const int tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  const int B = pp.B, H = pp.H, N = pp.N;
  if (blockIdx.x > 0) {
    const int bh = int(blockIdx.x) - 1, b = bh / H;
    const uint8_t* mq = pp.qv + size_t(b) * N;
    const uint8_t* mk = pp.pkv + size_t(b) * N;
    const int any_q = __syncthreads_or(tid < N && mq[min(tid, N - 1)] != 0);
    const int any_k = __syncthreads_or(tid < N && mk[min(tid, N - 1)] != 0);
    const bool empty = !any_q || !any_k;
    const size_t base = size_t(bh) * N * (DP / 8);
    const uint4 z{0u, 0u, 0u, 0u};
    for (int u = tid; u < N * (DP / 8); u += kPlanThreads) {
      const int row = u / (DP / 8);
      if (empty || mq[row] == 0) static_cast<uint4*>(pp.dq)[base + u] = z;
      if (empty || mk[row] == 0) {
        static_cast<uint4*>(pp.dk1)[base + u] = z;
        static_cast<uint4*>(pp.dv1)[base + u] = z;
        static_cast<uint4*>(pp.dk2)[base + u] = z;
        static_cast<uint4*>(pp.dv2)[base + u] = z;
      }
    }
    return;
  }
  constexpr int kRows = 4;
  for (int r0 = kRows * wave; r0 < 2 * B; r0 += kRows * (kPlanThreads / 64)) {
    uint8_t v[kRows][kMaxTokens / 64];
    // unconditional loads from clamped addresses (issued back to back), then the out-of-range ones zeroed
#pragma unroll
    for (int rr = 0; rr < kRows; ++rr) {
      const int r = min(r0 + rr, 2 * B - 1);
      const uint8_t* row = ((r & 1) ? pp.qv : pp.pkv) + size_t(r >> 1) * N;
#pragma unroll
      for (int sg = 0; sg < kMaxTokens / 64; ++sg) v[rr][sg] = row[min(64 * sg + lane, N - 1)];
    }
#pragma unroll
    for (int rr = 0; rr < kRows; ++rr)
#pragma unroll
      for (int sg = 0; sg < kMaxTokens / 64; ++sg)
        if (64 * sg + lane >= N) v[rr][sg] = uint8_t(0);
#pragma unroll
    for (int rr = 0; rr < kRows; ++rr) {
      const int r = r0 + rr;
      if (r >= 2 * B) break;  // uniform
      uint16_t* list = pp.lists + size_t(r) * N;
      int count = 0;
#pragma unroll
      for (int sg = 0; sg < kMaxTokens / 64; ++sg) {
        const bool on = v[rr][sg] != 0;
        const unsigned long long bal = __ballot(on);
        if (on) list[count + __popcll(bal & ((1ull << lane) - 1ull))] = uint16_t(64 * sg + lane);
        count += __popcll(bal);
      }
      if (lane == 0) s_count[r] = count;
    }
  }
  if (tid == 0) s_total = 0;
  lds_barrier();
  // jm, jm / 2 or jm / 4 j per unit: the one whose units finish first on 512 slots (two per CU; 256 units or fewer
  // left for the last round have a CU each and take 0.5 to 0.8 of their time), in rounds of the mean cost, or by the
  // longest unit; of equals the larger, whose fewer parts are added sooner.  (By the largest j that gives 512 units,
  // 16 molecules of 72 tokens, 8 heads, ran 768 units of 12 rows, 179 us; 384 of 24 rows take one round: 148.)
  {
    // thread 4 b + l: molecule b at jm >> l
    const int l = tid & 3;
    float units = 0.0f, most = 0.0f, sum = 0.0f;
    for (int b = tid >> 2; b < B; b += kPlanThreads / 4) {
      const int nk = s_count[2 * b], nq = s_count[2 * b + 1];
      if (nk <= 0 || nq <= 0 || l == 3) continue;
      const int parts = parts_of(nk, pp.jm >> l, pp.cap);
      const float u = float(H * parts);
      const float c = float(UnitCost(nk, nq, pp.bias).unit(rounds_of((nk + 1) / 2, parts), pp.jm));
      units += u;
      most = fmaxf(most, c);
      sum += u * c;
    }
    if (16 * wave < B) {
#pragma unroll
      for (int off = 4; off < 64; off <<= 1) {
        units += __shfl_xor(units, off, 64);
        most = fmaxf(most, __shfl_xor(most, off, 64));
        sum += __shfl_xor(sum, off, 64);
      }
      if (lane < 3) {
        s_level[wave][lane][0] = units;
        s_level[wave][lane][1] = most;
        s_level[wave][lane][2] = sum;
      }
    }
  }
  lds_barrier();
  int jt = pp.jm;
  {
    float least = INFINITY;
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      float units = 0.0f, most = 0.0f, sum = 0.0f;
      for (int w = 0; w < min(kPlanThreads / 64, (B + 15) / 16); ++w) {
        units += s_level[w][l][0];
        most = fmaxf(most, s_level[w][l][1]);
        sum += s_level[w][l][2];
      }
      if (units == 0.0f) continue;
      const float full = floorf(units / 512.0f), rest = units - 512.0f * full;
      const float last = rest == 0.0f ? 0.0f : (rest <= 256.0f ? 0.5f + 0.3f / 256.0f * rest : 1.0f);
      const float t = fmaxf((full + last) * (sum / units), full == 0.0f ? last * most : most);
      if (t < least) {
        least = t;
        jt = pp.jm >> l;
      }
    }
  }
  for (int b = tid; b < B; b += kPlanThreads) {
    const int nk = s_count[2 * b], nq = s_count[2 * b + 1];
    const bool work = nk > 0 && nq > 0;
    const int parts = work ? parts_of(nk, jt, pp.cap) : 0;
    s_cost[b] = work ? uint32_t(UnitCost(nk, nq, pp.bias).unit(rounds_of((nk + 1) / 2, parts), pp.jm)) : 0u;
    s_units[b] = H * parts;
    pp.counts[b] = int2{nk, nq};
  }
  lds_barrier();
  // rank: tpm threads per molecule, each over every tpm-th other molecule, partial sums added over the
  // thread group (adjacent lanes) by shuffles
  const int tpm = B >= kPlanThreads ? 1 : (B > kPlanThreads / 2 ? 2 : (B > kPlanThreads / 4 ? 4 : (B > kPlanThreads / 8 ? 8 : 16)));
  for (int t0 = 0; t0 < B * tpm; t0 += kPlanThreads) {
    const int t = t0 + tid;
    const int b = t / tpm, sub = t % tpm;
    int pre = 0;
    if (b < B) {
      const uint32_t cb = s_cost[b];
      for (int o = sub; o < B; o += tpm)
        if (s_cost[o] > cb || (s_cost[o] == cb && o < b)) pre += s_units[o];
    }
    for (int off = 1; off < tpm; off <<= 1) pre += __shfl_xor(pre, off, 64);
    if (b < B && s_units[b] > 0) {
      const int parts = s_units[b] / H;
      for (int u = sub; u < s_units[b]; u += tpm)
        pp.units[pre + u] = (uint32_t(b * H + u / parts) << 6) | uint32_t(u % parts);
      if (sub == 0) atomicAdd(&s_total, s_units[b]);
    }
  }
  lds_barrier();
  if (tid == 0) {
    pp.head[0] = s_total;
    pp.head[1] = jt;
  }
}

// The thread index, opaque to the compiler: what is computed from it stays inside the loop that asks, instead of
// being hoisted out of the block loops into registers (and from there into scratch) held throughout.
__device__ __forceinline__ int opaque_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// One block triple of a unit as the kernel staged it: nq queries from q0, nj j keys from j0, nk keys from k0
// (compacted positions), the scale exponents of its operands.
struct Triple {
  int bh, part, q0, nq, j0, nj, k0, nk;
  int eq, eg, e1, e2, f1, f2, ed;   // exponents of q, go, k1, k2, v1, v2 and of the largest |go . out|
  bool direct;                      // the molecule's only triple: gradients written here, not to the slab
  bool first_q, first_k;            // the unit's first triple with these queries (dq) / these keys (dk2, dv2)
  bool first_t;                     // the unit's first triple with these (queries, keys): dv_bias
};

// Row `row`, columns d4 .. d4 + 3 of the four waves' partial sums, added in wave order, times f.
__device__ __forceinline__ float4 sum_partials(const float* slot, int row, int d4, float f) {
  float4 s = *reinterpret_cast<const float4*>(slot + row * PS + d4);
#pragma unroll
  for (int w = 1; w < kWaves; ++w) {
    const float4 x = *reinterpret_cast<const float4*>(slot + (w * 16 + row) * PS + d4);
    s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
  }
  return float4{s.x * f, s.y * f, s.z * f, s.w * f};
}

// Four gradient elements, fp32 or rounded to bf16 (16-byte aligned tensors, whole rows of 64).
__device__ __forceinline__ void store_grad4(void* base, size_t i, const float4 v, int bf16) {
  if (bf16) {
    const uint2 w{__builtin_bit_cast(uint32_t, mf_bf16x2{__bf16(v.x), __bf16(v.y)}),
                  __builtin_bit_cast(uint32_t, mf_bf16x2{__bf16(v.z), __bf16(v.w)})};
    *reinterpret_cast<uint2*>(static_cast<__bf16*>(base) + i) = w;
  } else {
    *reinterpret_cast<float4*>(static_cast<float*>(base) + i) = v;
  }
}

// A unit's running sum of a slab row (this thread wrote what it reads back).
__device__ __forceinline__ void add_slab(float* p, float4 s, bool first) {
  if (!first) {
    const float4 o = *reinterpret_cast<const float4*>(p);
    s.x += o.x; s.y += o.y; s.z += o.z; s.w += o.w;
  }
  *reinterpret_cast<float4*>(p) = s;
}

// The main loop over one triple and its sums.
template <int NQT, int BIAS>
__device__ __forceinline__ void triple_body(const Params& p, unsigned char* smem, const Triple& c) {
  using Ly = Lay<BIAS != 0>;
  constexpr int QM = Ly::QM, JM = Ly::JM, KM = Ly::KM, KU = Ly::KU, KW = Ly::KW;
  const int tid = opaque_tid();
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4;
  const int r16 = lane & 15;
  const int N = p.N;
  const size_t rbase = size_t(c.bh) * N;
  float* slab = p.slab + (size_t(c.bh) * p.cap + c.part) * 3 * N * DP;
  _Float16* Qs = reinterpret_cast<_Float16*>(smem + Ly::rows);
  _Float16* Gs = Qs + QM * KS;
  _Float16* K1s = Gs + QM * KS;
  _Float16* V1s = K1s + JM * KS;
  _Float16* K2s = V1s + JM * KS;
  _Float16* V2s = K2s + KM * KS;
  float* dk1a = reinterpret_cast<float*>(smem + Ly::acc1);
  float* dv1a = dk1a + JM * DP;
  float* slot = reinterpret_cast<float*>(smem + Ly::scr);
  _Float16* scr = reinterpret_cast<_Float16*>(smem + Ly::scr) + wave * (QM / 16) * 32 * SS;
  const float* uT = reinterpret_cast<const float*>(smem + Ly::ut);
  const float* vT = reinterpret_cast<const float*>(smem + Ly::vt);
  float* dut = reinterpret_cast<float*>(smem + Ly::dut);
  float* wd = reinterpret_cast<float*>(smem + Ly::wd);
  const float* cg = reinterpret_cast<const float*>(smem + Ly::gt);
  const float* lse2 = reinterpret_cast<const float*>(smem + Ly::lse2);
  const float* dls = reinterpret_cast<const float*>(smem + Ly::dls);
  const uint32_t* pvb = reinterpret_cast<const uint32_t*>(smem + Ly::pvb);
  const int* kidx = reinterpret_cast<const int*>(smem + Ly::kidx);
  const int* qidx = reinterpret_cast<const int*>(smem + Ly::qidx);
  // dS is carried as dS 2^-es, |dS 2^-es| < 2^15 P, P as P 2^kPScale (staged with lse):  S log2 e = S_c cS,
  // dS 2^-es = P 2^kPScale (dP_c cP - delta 2^(-es - kPScale))
  const int es = ds_exp(c.eg, c.f1, c.f2, c.ed);
  const float cS = ldexpf(kLog2e, c.eq + c.e1 + c.e2);
  const float cP = pow2(c.eg + c.f1 + c.f2 - es - kPScale);
  const float uD = pow2(es);
  const float fk1 = ldexpf(1.0f, c.e2 + es + c.eq), fv1 = ldexpf(1.0f, c.f2 + c.eg - kPScale);

  const int nkt = (c.nk + 15) / 16;
  const int njp = (c.nj + 1) / 2;

  mf_f32x4 dqa[NQT][4];
#pragma unroll
  for (int t = 0; t < NQT; ++t)
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) dqa[t][dt] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
  // BIAS: dgate partial of queries 16 t + 4 g + r over the lane's (j, k)
  float accg[BIAS ? NQT : 1][4];
#pragma unroll
  for (int t = 0; t < (BIAS ? NQT : 1); ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) accg[t][r] = 0.0f;
  for (int kt = 0; kt < nkt; ++kt) {
    const int k0 = kt * 16;
    mf_f32x4 dk2a[4], dv2a[4];  // key k0 + 4 g + r, d = 16 dt + r16
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      dk2a[dt] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
      dv2a[dt] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float dva[BIAS ? NQT : 1][4];  // dv_bias partial of the lane's (query, key) over the wave's j
#pragma unroll
    for (int t = 0; t < (BIAS ? NQT : 1); ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) dva[t][r] = 0.0f;

    for (int jp = wave; jp < njp; jp += kWaves) {
      const int ja = 2 * jp;
      // (BIAS: the LDS addresses are formed again for each pair, a few VALU, instead of living in scratch)
      int ol = lane;
      if constexpr (BIAS != 0) asm volatile("" : "+v"(ol));
      const int g = ol >> 4, r16 = ol & 15;
      mf_f16x8 wb[2][2], zh[2][2], zl[2][2];  // W, Z (hi, lo) of pairs (ja + jn, k0 + r16), d = 32 s + 8 g + e
      bool ok[2];
      auto form = [&](int jn) {
        const int j = ja + jn;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const mf_f16x8 a = *reinterpret_cast<const mf_f16x8*>(K1s + j * KS + 32 * s + 8 * g);
          const mf_f16x8 b = *reinterpret_cast<const mf_f16x8*>(V1s + j * KS + 32 * s + 8 * g);
          const mf_f16x8 k2c = *reinterpret_cast<const mf_f16x8*>(K2s + (k0 + r16) * KS + 32 * s + 8 * g);
          const mf_f16x8 v2c = *reinterpret_cast<const mf_f16x8*>(V2s + (k0 + r16) * KS + 32 * s + 8 * g);
          wb[jn][s] = a * k2c;
          zh[jn][s] = b * v2c;
          zl[jn][s] = __builtin_elementwise_fma(b, v2c, -zh[jn][s]);
        }
        ok[jn] = ((pvb[j * 2 + ((k0 + r16) >> 5)] >> ((k0 + r16) & 31)) & 1u) != 0u;
      };
      // P and dS of (j, query tile) as packed fp16: word r / 2 of query 16 t + 4 g + r, key k0 + r16
      uint2 dsw[2][NQT], pw[2][NQT];
      auto score = [&](int jn, int t, const mf_f16x8 (&aq)[2], const mf_f16x8 (&ag)[2], float wj, float& dwj,
                       float (&dsv)[4]) {
        mf_f32x4 sacc = mf_f32x4{0.f, 0.f, 0.f, 0.f}, pacc = mf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          sacc = mma(aq[s], wb[jn][s], sacc);
          pacc = mma(ag[s], zh[jn][s], pacc);
          pacc = mma(ag[s], zl[jn][s], pacc);
        }
        const float4 l2 = *reinterpret_cast<const float4*>(lse2 + t * 16 + 4 * g);
        const float4 dl = *reinterpret_cast<const float4*>(dls + t * 16 + 4 * g);
        const float l2v[4] = {l2.x, l2.y, l2.z, l2.w};
        const float dlv[4] = {dl.x, dl.y, dl.z, dl.w};
        float cl[4], base[4], pp[4];
        if constexpr (BIAS != 0) {  // gate_i (u_ij + v_ik + w_jk) of the lane's queries and pair
          const float4 c4 = *reinterpret_cast<const float4*>(cg + t * 16 + 4 * g);
          const float4 u4 = *reinterpret_cast<const float4*>(uT + (ja + jn) * KU + t * 16 + 4 * g);
          const float4 v4 = *reinterpret_cast<const float4*>(vT + (k0 + r16) * KU + t * 16 + 4 * g);
          cl[0] = c4.x; cl[1] = c4.y; cl[2] = c4.z; cl[3] = c4.w;
          // (0 at a dropped pair: dS is 0 there, but the terms may be -inf or NaN)
          base[0] = ok[jn] ? (u4.x + v4.x) + wj : 0.0f;
          base[1] = ok[jn] ? (u4.y + v4.y) + wj : 0.0f;
          base[2] = ok[jn] ? (u4.z + v4.z) + wj : 0.0f;
          base[3] = ok[jn] ? (u4.w + v4.w) + wj : 0.0f;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float s2 = fmaf(sacc[r], cS, -l2v[r]);
          if constexpr (BIAS != 0) s2 = fmaf(cl[r], base[r], s2);
          pp[r] = ok[jn] ? fast_exp2(s2) : 0.0f;
          dsv[r] = pp[r] * fmaf(pacc[r], cP, -dlv[r]);
          if constexpr (BIAS != 0) {
            accg[t][r] = fmaf(dsv[r], base[r], accg[t][r]);
            dwj = fmaf(cl[r], dsv[r], dwj);
            dva[t][r] += dsv[r];
          }
        }
        dsw[jn][t] = uint2{pack_f16(dsv[0], dsv[1]), pack_f16(dsv[2], dsv[3])};
        pw[jn][t] = uint2{pack_f16(pp[0], pp[1]), pack_f16(pp[2], pp[3])};
        // dS [pair (jn, key)][query] into the tile's slot of the wave's scratch
        *reinterpret_cast<uint2*>(scr + t * 32 * SS + (jn * 16 + r16) * SS + 4 * g) = dsw[jn][t];
      };
      auto rows_of = [&](const _Float16* base, int t, mf_f16x8 (&a)[2]) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
          a[s] = *reinterpret_cast<const mf_f16x8*>(base + (t * 16 + r16) * KS + 32 * s + 8 * g);
      };
      if constexpr (BIAS == 0 && NQT < 4) {  // both j share the rows of a query tile
        form(0);
        form(1);
#pragma unroll
        for (int t = 0; t < NQT; ++t) {
          mf_f16x8 aq[2], ag[2];
          rows_of(Qs, t, aq);
          rows_of(Gs, t, ag);
          float ds[4], none = 0.0f;
          score(0, t, aq, ag, 0.0f, none, ds);
          score(1, t, aq, ag, 0.0f, none, ds);
        }
        __builtin_amdgcn_sched_barrier(0);
      } else if constexpr (BIAS == 0) {
#pragma unroll
        for (int jn = 0; jn < 2; ++jn) {
          form(jn);
#pragma unroll
          for (int t = 0; t < NQT; ++t) {
            mf_f16x8 aq[2], ag[2];
            rows_of(Qs, t, aq);
            rows_of(Gs, t, ag);
            float ds[4], none = 0.0f;
            score(jn, t, aq, ag, 0.0f, none, ds);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {  // one j at a time: the bias sums leave no registers for two
#pragma unroll
        for (int jn = 0; jn < 2; ++jn) {
          const int j = ja + jn;
          form(jn);
          const float wj = wd[j * KW + k0 + r16];  // its place takes dw below (each pair belongs to one wave)
          // su: the sum over the tile's keys of dS of (j, query 16 (r16 >> 2) + 4 g + (r16 & 3))
          float dwj = 0.0f, su = 0.0f;
#pragma unroll
          for (int t = 0; t < NQT; ++t) {
            mf_f16x8 aq[2], ag[2];
            float dsv[4];
            rows_of(Qs, t, aq);
            rows_of(Gs, t, ag);
            score(jn, t, aq, ag, wj, dwj, dsv);
            const float st = row16_sum4(dsv, r16);
            su = (r16 >> 2) == t ? st : su;
          }
          const int i = 16 * (r16 >> 2) + 4 * g + (r16 & 3);
          if (r16 < 4 * NQT) dut[j * KU + i] = fmaf(su, uD, dut[j * KU + i]);
          // dw of (j, the lane's key): dwj sums gate log2 e dS 2^-es
          const float x = sum_groups(dwj) * (uD * (1.0f / kLog2e));
          if (g == 0) wd[j * KW + k0 + r16] = x;
          __builtin_amdgcn_sched_barrier(0);
        }
      }

      // ---- G^T, H^T (key k0 + 4 g + r, d = 16 dt + r16) and the pairs' key-side gradients, 16 d at a time.  A =
      // dS^T / P^T of two query tiles as the lane holds them (K slot 4 h + r is query (qb + h) 16 + 4 g + r), B =
      // q / go at those queries (transposed reads; the second tile's rows when it exists, else the first's
      // again: its K slots carry zeros) ----
      float x[2][4], y[2][4];
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        mf_f32x4 gt[2], ht[2];
#pragma unroll
        for (int jn = 0; jn < 2; ++jn) {
          gt[jn] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
          ht[jn] = mf_f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int qb = 0; qb < NQT; qb += 2) {
          const bool two = qb + 1 < NQT;
          const int off = (qb * 16 + 4 * g + (r16 >> 2)) * KS + 16 * dt + 4 * (r16 & 3);
          const int off2 = off + (two ? 16 * KS : 0);
          const mf_f16x8 bq = cat8(read_tr16(Qs + off), read_tr16(Qs + off2));
          const mf_f16x8 bg = cat8(read_tr16(Gs + off), read_tr16(Gs + off2));
#pragma unroll
          for (int jn = 0; jn < 2; ++jn) {
            const uint2 d2 = two ? dsw[jn][two ? qb + 1 : qb] : uint2{0u, 0u};
            const uint2 p2 = two ? pw[jn][two ? qb + 1 : qb] : uint2{0u, 0u};
            gt[jn] = mma(__builtin_bit_cast(mf_f16x8, uint4{dsw[jn][qb].x, dsw[jn][qb].y, d2.x, d2.y}), bq, gt[jn]);
            ht[jn] = mma(__builtin_bit_cast(mf_f16x8, uint4{pw[jn][qb].x, pw[jn][qb].y, p2.x, p2.y}), bg, ht[jn]);
          }
        }
        // k2 / v2 of keys k0 + 4 g + r at d = 16 dt + r16 (transposed reads), k1 / v1 of j
        const int roff = (k0 + 4 * g + (r16 >> 2)) * KS + 16 * dt + 4 * (r16 & 3);
        const auto k2t = read_tr16(K2s + roff);
        const auto v2t = read_tr16(V2s + roff);
#pragma unroll
        for (int jn = 0; jn < 2; ++jn) {
          const float k1p = float(K1s[(ja + jn) * KS + 16 * dt + r16]);
          const float v1p = float(V1s[(ja + jn) * KS + 16 * dt + r16]);
          x[jn][dt] = 0.0f;
          y[jn][dt] = 0.0f;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            dk2a[dt][r] = fmaf(k1p, gt[jn][r], dk2a[dt][r]);
            dv2a[dt][r] = fmaf(v1p, ht[jn][r], dv2a[dt][r]);
            x[jn][dt] = fmaf(float(k2t[r]), gt[jn][r], x[jn][dt]);
            y[jn][dt] = fmaf(float(v2t[r]), ht[jn][r], y[jn][dt]);
          }
        }
      }
      // dk1_j / dv1_j at d = lane: rows of j belong to this wave
#pragma unroll
      for (int jn = 0; jn < 2; ++jn) {
        const int o = (ja + jn) * DP + lane;
        const float xs = sum_groups4(x[jn][0], x[jn][1], x[jn][2], x[jn][3]);
        const float ys = sum_groups4(y[jn][0], y[jn][1], y[jn][2], y[jn][3]);
        dk1a[o] = fmaf(xs, fk1, dk1a[o]);
        dv1a[o] = fmaf(ys, fv1, dv1a[o]);
      }
      // ---- dq of queries 16 t + r16: A = dS [query][pairs (ja + (g >> 1), keys 8 (g & 1) + e)] by transposed
      // reads (lane 4 e' + a of a group addresses row e' (+4), columns 4 a .. 4 a + 3), B = W of those pairs at
      // d = 16 dt + r16 ----
      __builtin_amdgcn_wave_barrier();
      mf_f16x8 wc[4];
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const _Float16* pc = K2s + (k0 + 8 * (g & 1) + (r16 >> 2)) * KS + 16 * dt + 4 * (r16 & 3);
        wc[dt] = cat8(read_tr16(pc), read_tr16(pc + 4 * KS)) * K1s[(ja + (g >> 1)) * KS + 16 * dt + r16];
      }
#pragma unroll
      for (int t = 0; t < NQT; ++t) {
        const _Float16* ps = scr + t * 32 * SS + ((g >> 1) * 16 + 8 * (g & 1) + (r16 >> 2)) * SS + 4 * (r16 & 3);
        const mf_f16x8 ads = cat8(read_tr16(ps), read_tr16(ps + 4 * SS));
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) dqa[t][dt] = mma(ads, wc[dt], dqa[t][dt]);
      }
      __builtin_amdgcn_wave_barrier();
    }

    // ---- dk2, then dv2 of the key tile: the four waves' partials in wave order ----
    lds_barrier();  // every wave is done with its scratch
#pragma unroll
    for (int which = 0; which < 2; ++which) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          slot[(wave * 16 + 4 * g + r) * PS + 16 * dt + r16] = which ? dv2a[dt][r] : dk2a[dt][r];
      lds_barrier();
      const int kk = tid / 16, d4 = 4 * (tid % 16);
      if (k0 + kk < c.nk) {
        const float4 s = sum_partials(slot, kk, d4, which ? ldexpf(1.0f, c.f1 + c.eg - kPScale) : ldexpf(1.0f, c.e1 + es + c.eq));
        if (c.direct) {
          store_grad4(which ? p.dv2 : p.dk2, (rbase + kidx[k0 + kk]) * DP + d4, s, p.gout16);
        } else {
          add_slab(slab + (size_t(1 + which) * N + c.k0 + k0 + kk) * DP + d4, s, c.first_k);
        }
      }
      lds_barrier();
    }
    // BIAS: dv_bias partial of the key tile: [t][key r16][query 4 g + r] per wave, a query tile at a time per slot
    if constexpr (BIAS != 0) {
      if (p.dvb != nullptr) {
#pragma unroll
        for (int t = 0; t < NQT; ++t)
          *reinterpret_cast<float4*>(slot + (wave * NQT + t) * 256 + r16 * 16 + 4 * g) =
              float4{dva[t][0], dva[t][1], dva[t][2], dva[t][3]};
        lds_barrier();
        for (int u = tid; u < NQT * 256; u += kThreads) {  // key fastest: 64-byte runs of the rows
          const int kk = u % 16, i16 = (u / 16) % 16, t = u / 256;
          const int i = t * 16 + i16, l = t * 256 + kk * 16 + i16;
          if (i < c.nq && k0 + kk < c.nk) {
            float s = (((slot[l] + slot[NQT * 256 + l]) + slot[2 * NQT * 256 + l]) + slot[3 * NQT * 256 + l]) * uD;
            float* o = p.dvpart + ((size_t(c.bh) * p.cap + c.part) * N + c.q0 + i) * N + c.k0 + k0 + kk;
            *o = c.first_t ? s : s + *o;
          }
        }
        lds_barrier();
      }
    }
  }

  // ---- dq: the four waves' partials in wave order, a query tile at a time ----
#pragma unroll
  for (int t = 0; t < NQT; ++t) {
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) slot[(wave * 16 + 4 * g + r) * PS + 16 * dt + r16] = dqa[t][dt][r];
    lds_barrier();
    const int ii = t * 16 + tid / 16, d4 = 4 * (tid % 16);
    if (ii < c.nq) {
      const float4 s = sum_partials(slot, tid / 16, d4, ldexpf(1.0f, es + c.e1 + c.e2));
      if (c.direct) store_grad4(p.dq, (rbase + qidx[ii]) * DP + d4, s, p.gout16);
      else add_slab(slab + (size_t(c.q0) + ii) * DP + d4, s, c.first_q);
    }
    lds_barrier();
  }
  // BIAS: dgate partials: sums over each lane row's keys, then the four waves in order
  if constexpr (BIAS != 0) {
    if (p.dgate != nullptr) {
#pragma unroll
      for (int t = 0; t < NQT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = row16_sum(accg[t][r]);
          if (r16 == 0) slot[wave * QM + t * 16 + 4 * g + r] = x;
        }
      lds_barrier();
      if (tid < c.nq) {
        const float s = (((slot[tid] + slot[QM + tid]) + slot[2 * QM + tid]) + slot[3 * QM + tid]) * uD;
        float* o = p.dgpart + (size_t(c.bh) * p.cap + c.part) * N + c.q0 + tid;
        *o = c.first_q ? s : s + *o;
      }
      lds_barrier();
    }
  }
}

template <int BIAS>
__global__ void __launch_bounds__(kThreads, 2) pair_bwd_kernel(Params p) {
  using Lk = Lay<BIAS != 0>;
  constexpr int QM = Lk::QM, JM = Lk::JM, KM = Lk::KM, KU = Lk::KU, KW = Lk::KW;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  if (int(blockIdx.x) >= p.head[0]) return;
  const uint32_t unit = p.units[blockIdx.x];
  const int jt = p.head[1];
  const int N = p.N;
  Triple c;
  c.bh = int(unit >> 6);
  c.part = int(unit & 63u);
  const int b = c.bh / p.H;
  const int2 nkq = p.counts[b];
  const int nk = nkq.x, nq = nkq.y;
  const int parts = parts_of(nk, jt, p.cap);
  const int jr = unit_rows(nk, parts);
  const int ju0 = c.part * jr, ju1 = min(nk, ju0 + jr);  // the unit's j
  const size_t rbase = size_t(c.bh) * N;
  const uint16_t* klist = p.lists + size_t(2 * b) * N;
  const uint16_t* qlist = klist + N;
  const int njb = blocks_of(ju1 - ju0, JM), nqb = blocks_of(nq, QM), nkb = blocks_of(nk, KM);
  // (whole rounds of four key pairs in every block but the last)
  const int jrows = 2 * kWaves * (((ju1 - ju0 + 2 * kWaves - 1) / (2 * kWaves) + njb - 1) / njb);
  const int qrows = block_rows(nq, nqb), krows = block_rows(nk, nkb);
  c.direct = parts == 1 && njb == 1 && nqb == 1 && nkb == 1;

  _Float16* Qs = reinterpret_cast<_Float16*>(smem + Lk::rows);
  _Float16* Gs = Qs + QM * KS;
  _Float16* K1s = Gs + QM * KS;
  _Float16* V1s = K1s + JM * KS;
  _Float16* K2s = V1s + JM * KS;
  _Float16* V2s = K2s + KM * KS;
  float* acc1 = reinterpret_cast<float*>(smem + Lk::acc1);
  float* lse2 = reinterpret_cast<float*>(smem + Lk::lse2);
  float* dlt = reinterpret_cast<float*>(smem + Lk::dlt);
  float* dls = reinterpret_cast<float*>(smem + Lk::dls);
  float* ut = reinterpret_cast<float*>(smem + Lk::ut);
  float* dut = reinterpret_cast<float*>(smem + Lk::dut);
  float* wd = reinterpret_cast<float*>(smem + Lk::wd);
  float* vt = reinterpret_cast<float*>(smem + Lk::vt);
  float* cgs = reinterpret_cast<float*>(smem + Lk::gt);
  int* jidx = reinterpret_cast<int*>(smem + Lk::jidx);
  int* kidx = reinterpret_cast<int*>(smem + Lk::kidx);
  int* qidx = reinterpret_cast<int*>(smem + Lk::qidx);
  uint32_t* red = reinterpret_cast<uint32_t*>(smem + Lk::red);

  // FP16_OVFL: fp16 results past the range become the largest fp16 (P where a saturated bias left lse far too small).
  // (Here, after the addresses: at the kernel's top the bias instantiations spilled 45 registers instead of 16.)
  asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 23, 1), 1");
  for (int jb = 0; jb < njb; ++jb) {
    c.j0 = ju0 + jb * jrows;
    c.nj = min(ju1 - c.j0, jrows);
    for (int qb = 0; qb < nqb; ++qb) {
      c.q0 = qb * qrows;
      c.nq = min(nq - c.q0, qrows);
      for (int kb = 0; kb < nkb; ++kb) {
        c.k0 = kb * krows;
        c.nk = min(nk - c.k0, krows);
        c.first_q = jb == 0 && kb == 0;
        c.first_k = jb == 0 && qb == 0;
        c.first_t = jb == 0;
        // ---- stage the rows that changed (compacted, zero past the counts) as fp16 scaled by 2^-e per
        // operand, lse log2 e (less kPScale) and go . out of each query (+inf / 0 on the padding rows: P = 0 there).  A
        // thread has a 16-byte piece of row tid / 8 and, for q and k blocks, of row 32 + tid / 8; every
        // global load is issued before the first LDS store, rows past a count load its last row. ----
        const bool do_j = qb == 0 && kb == 0, do_q = kb == 0, do_k = nkb > 1 || do_j;
        const int tid = opaque_tid(), lane = tid & 63, wave = tid >> 6;
        const int r0 = tid / 8, ch = tid % 8;
        uint4 bq[2], bg[2], b1 = uint4{0u, 0u, 0u, 0u}, d1 = b1, b2[2], d2[2];
        float4 o0[2], o1[2];
        float lv[2];
        int iq[2], ik[2], ij = 0;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          bq[i] = bg[i] = b2[i] = d2[i] = uint4{0u, 0u, 0u, 0u};
          o0[i] = o1[i] = float4{0.f, 0.f, 0.f, 0.f};
          lv[i] = INFINITY;
          iq[i] = qlist[c.q0 + min(r0 + 32 * i, c.nq - 1)];
          ik[i] = klist[c.k0 + min(r0 + 32 * i, c.nk - 1)];
        }
        ij = klist[c.j0 + min(r0, c.nj - 1)];
        if (do_j) {
          b1 = *reinterpret_cast<const uint4*>(p.k1 + (rbase + ij) * DP + 8 * ch);
          d1 = *reinterpret_cast<const uint4*>(p.v1 + (rbase + ij) * DP + 8 * ch);
        }
        if (do_q) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const size_t row = rbase + iq[i];
            bq[i] = *reinterpret_cast<const uint4*>(p.q + row * DP + 8 * ch);
            bg[i] = *reinterpret_cast<const uint4*>(p.go + row * DP + 8 * ch);
            o0[i] = *reinterpret_cast<const float4*>(p.out + row * DP + 8 * ch);
            o1[i] = *reinterpret_cast<const float4*>(p.out + row * DP + 8 * ch + 4);
            lv[i] = fmaf(p.lse[row], kLog2e, -float(kPScale));
          }
        }
        if (do_k) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            b2[i] = *reinterpret_cast<const uint4*>(p.k2 + (rbase + ik[i]) * DP + 8 * ch);
            d2[i] = *reinterpret_cast<const uint4*>(p.v2 + (rbase + ik[i]) * DP + 8 * ch);
          }
        }
        // valid pairs (j, k) of the block, eight keys per byte
        uint32_t bits = 0u;
        const bool do_bits = do_k && tid < JM * (KM / 8);
        if (do_bits) {
          const int j = tid / (KM / 8), k8 = 8 * (tid % (KM / 8));
          const int left = c.nk - k8;
          bits = j >= c.nj || left <= 0 ? 0u : (left >= 8 ? 0xffu : (1u << left) - 1u);
          if (p.pv != nullptr) {
            const uint8_t* row = p.pv + (size_t(b) * N + klist[c.j0 + min(j, c.nj - 1)]) * N;
            uint8_t on[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) on[t] = row[klist[c.k0 + min(k8 + t, c.nk - 1)]];
#pragma unroll
            for (int t = 0; t < 8; ++t) bits &= on[t] != 0 ? 0xffu : ~(1u << t);
          }
        }
        // BIAS: u of (query, j), w of (j, key), v of (query, key) and the gates; thread (tid / 16, tid % 16) of a
        // 16 x 16 grid of entries
        constexpr int kT = BIAS ? QM / 16 : 1;
        static_assert(!BIAS || (JM == 16 && QM == KM), "the 16 x 16 grid covers j; QM / 16 steps cover both others");
        const int jj = tid % 16, ii = tid / 16;
        float ul[kT], wl[kT], vl[kT][kT], ga = 0.0f;
        if constexpr (BIAS != 0) {
          int qx[kT], kx[kT];
          const int jx = klist[c.j0 + min(jj, c.nj - 1)], jy = klist[c.j0 + min(ii, c.nj - 1)];
#pragma unroll
          for (int t = 0; t < kT; ++t) {
            qx[t] = qlist[c.q0 + min(ii + 16 * t, c.nq - 1)];
            kx[t] = klist[c.k0 + min(jj + 16 * t, c.nk - 1)];
          }
          if (do_q) ga = load_bias<BIAS>(p.bg, rbase + qlist[c.q0 + min(tid, c.nq - 1)]);
#pragma unroll
          for (int t = 0; t < kT; ++t) {
            ul[t] = do_q ? load_bias<BIAS>(p.bu, (rbase + qx[t]) * N + jx) : 0.0f;
            wl[t] = load_bias<BIAS>(p.bw, (rbase + jy) * N + kx[t]);
#pragma unroll
            for (int u = 0; u < kT; ++u) vl[t][u] = load_bias<BIAS>(p.bv, (rbase + qx[t]) * N + kx[u]);
          }
        }
        const uint4 zero{0u, 0u, 0u, 0u};
        if (r0 >= c.nj) b1 = d1 = zero;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (r0 + 32 * i >= c.nq) {
            bq[i] = bg[i] = zero;
            lv[i] = INFINITY;
          }
          if (r0 + 32 * i >= c.nk) b2[i] = d2[i] = zero;
        }
        // go . out of the thread's query rows (in the eight threads of a row)
        float go[2] = {0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (!do_q) break;  // uniform
          float s = bf_lo(bg[i].x) * o0[i].x;
          s = fmaf(bf_hi(bg[i].x), o0[i].y, s); s = fmaf(bf_lo(bg[i].y), o0[i].z, s);
          s = fmaf(bf_hi(bg[i].y), o0[i].w, s); s = fmaf(bf_lo(bg[i].z), o1[i].x, s);
          s = fmaf(bf_hi(bg[i].z), o1[i].y, s); s = fmaf(bf_lo(bg[i].w), o1[i].z, s);
          s = fmaf(bf_hi(bg[i].w), o1[i].w, s);
          go[i] = sum8(s);
        }
        // largest magnitude of each operand over the block, and of go . out (its bf16 bits: the exponent is what
        // counts, one that is not finite leaves the others' scale alone): per thread, per wave, then over the four waves
        const uint32_t da = __float_as_uint(go[0]) << 1 >> 17, db = __float_as_uint(go[1]) << 1 >> 17;
        uint32_t mx[7];
        auto magnitudes = [&](auto finite) {
          auto am = [](const uint4& r) { return absmax_bits8<decltype(finite)::value>(r); };
          mx[0] = max(am(bq[0]), am(bq[1]));
          mx[1] = max(am(bg[0]), am(bg[1]));
          mx[2] = am(b1);
          mx[3] = max(am(b2[0]), am(b2[1]));
          mx[4] = am(d1);
          mx[5] = max(am(d2[0]), am(d2[1]));
        };
        magnitudes(std::false_type{});
        // (infinities and NaN stay what they are under any scale and must not decide that of the other rows)
        if (max(max(max(mx[0], mx[1]), max(mx[2], mx[3])), max(mx[4], mx[5])) >= 0x7f80u) magnitudes(std::true_type{});
        mx[6] = max(da < 0x7f80u ? da : 0u, db < 0x7f80u ? db : 0u);
#pragma unroll
        for (int t = 0; t < 7; ++t) {
          mx[t] = wave_max_u32(mx[t]);
          if (lane == 0) red[wave * 8 + t] = mx[t];
        }
        lds_barrier();
        int ex[7];
#pragma unroll
        for (int t = 0; t < 7; ++t)
          ex[t] = __builtin_amdgcn_readfirstlane(scale_exp(max(max(red[t], red[8 + t]), max(red[16 + t], red[24 + t]))));
        if (do_q) {
          c.eq = ex[0];
          c.eg = ex[1];
          c.ed = ex[6];
        }
        if (do_j) {
          c.e1 = ex[2];
          c.f1 = ex[4];
        }
        if (do_k) {
          c.e2 = ex[3];
          c.f2 = ex[5];
        }
        const float dscale = pow2(-ds_exp(c.eg, c.f1, c.f2, c.ed) - kPScale);
        if (do_q) {
          const float sq = ldexpf(1.0f, -ex[0]), sg = ldexpf(1.0f, -ex[1]);
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int r = r0 + 32 * i;
            if (r < QM) {
              *reinterpret_cast<uint4*>(Qs + r * KS + 8 * ch) = to_f16x8(bq[i], sq);
              *reinterpret_cast<uint4*>(Gs + r * KS + 8 * ch) = to_f16x8(bg[i], sg);
              if (ch == 0) {
                dlt[r] = r < c.nq ? go[i] : 0.0f;
                dls[r] = r < c.nq ? go[i] * dscale : 0.0f;
                lse2[r] = lv[i];
                qidx[r] = iq[i];
              }
            }
          }
        } else if (ch == 0) {  // the scale of dS may have changed
#pragma unroll
          for (int i = 0; i < 2; ++i)
            if (r0 + 32 * i < QM) dls[r0 + 32 * i] = dlt[r0 + 32 * i] * dscale;
        }
        if (do_j) {
          if (r0 < JM) {
            *reinterpret_cast<uint4*>(K1s + r0 * KS + 8 * ch) = to_f16x8(b1, ldexpf(1.0f, -ex[2]));
            *reinterpret_cast<uint4*>(V1s + r0 * KS + 8 * ch) = to_f16x8(d1, ldexpf(1.0f, -ex[4]));
            if (ch == 0) jidx[r0] = ij;
          }
          static_assert(2 * JM * DP / 4 % kThreads == 0, "whole passes");
          static_assert(JM <= 32 && QM <= 64 && KM <= 64, "rows of a thread");
#pragma unroll
          for (int u = 0; u < 2 * JM * DP / 4 / kThreads; ++u)
            reinterpret_cast<float4*>(acc1)[tid + kThreads * u] = float4{0.f, 0.f, 0.f, 0.f};
        }
        if (do_bits) (smem + Lk::pvb)[(tid / (KM / 8)) * 8 + tid % (KM / 8)] = uint8_t(bits);
        if constexpr (BIAS != 0) {
          // (1 on the padding rows: there lse = inf makes P = 0 whatever finite or -inf terms it multiplies)
          if (do_q && tid < QM) cgs[tid] = tid < c.nq ? ga * kLog2e : 1.0f;
#pragma unroll
          for (int t = 0; t < kT; ++t) {
            if (do_q) {
              ut[jj * KU + ii + 16 * t] = ii + 16 * t < c.nq && jj < c.nj ? ul[t] : 0.0f;
              dut[jj * KU + ii + 16 * t] = 0.0f;
            }
            wd[ii * KW + jj + 16 * t] = wl[t];
#pragma unroll
            for (int u = 0; u < kT; ++u) vt[(jj + 16 * u) * KU + ii + 16 * t] = vl[t][u];
          }
        }
        if (do_k) {
          const float s2 = ldexpf(1.0f, -ex[3]), t2 = ldexpf(1.0f, -ex[5]);
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int r = r0 + 32 * i;
            if (r < KM) {
              *reinterpret_cast<uint4*>(K2s + r * KS + 8 * ch) = to_f16x8(b2[i], s2);
              *reinterpret_cast<uint4*>(V2s + r * KS + 8 * ch) = to_f16x8(d2[i], t2);
              if (ch == 0) kidx[r] = ik[i];
            }
          }
        }
        lds_barrier();
        switch ((c.nq + 15) / 16) {
          case 1: triple_body<1, BIAS>(p, smem, c); break;
          case 2: triple_body<2, BIAS>(p, smem, c); break;
          case 3: triple_body<3, BIAS>(p, smem, c); break;
          default:
            if constexpr (BIAS == 0) triple_body<4, BIAS>(p, smem, c);
            break;
        }
        if constexpr (BIAS != 0) {  // dw of the triple's (j, k), summed over the query blocks
          if (p.dw != nullptr) {
            const int tid = opaque_tid();
            for (int u = tid; u < c.nj * KM; u += kThreads) {
              const int j = u / KM, k = u % KM;
              if (k >= c.nk) continue;
              float x = wd[j * KW + k];
              // earlier query blocks keep their sum in the workspace (read back by the thread that wrote it)
              float* o = p.dwpart + (rbase + c.j0 + j) * N + c.k0 + k;
              if (qb > 0) x += *o;
              if (qb + 1 < nqb) *o = x;
              else store_grad(p.dw, (rbase + jidx[j]) * N + kidx[k], x, p.bout16);
            }
          }
          if (kb + 1 < nkb) lds_barrier();
        }
      }
      if constexpr (BIAS != 0) {  // du of the block's (query, j): every key is in
        if (p.du != nullptr) {
          for (int u = opaque_tid(); u < c.nq * JM; u += kThreads) {
            const int i = u / JM, j = u % JM;
            if (j < c.nj)
              store_grad(p.du, (rbase + qidx[i]) * N + jidx[j], cgs[i] * (1.0f / kLog2e) * dut[j * KU + i], p.bout16);
          }
        }
        if (qb + 1 < nqb) lds_barrier();
      }
    }
    // ---- dk1 / dv1 rows of the block's j (the barriers that end the body order the waves' rows) ----
    for (int u = opaque_tid(); u < c.nj * (DP / 4); u += kThreads) {
      const int j = u / (DP / 4), d4 = 4 * (u % (DP / 4));
      const size_t o = (rbase + jidx[j]) * DP + d4;
      store_grad4(p.dk1, o, *reinterpret_cast<const float4*>(acc1 + j * DP + d4), p.gout16);
      store_grad4(p.dv1, o, *reinterpret_cast<const float4*>(acc1 + (JM + j) * DP + d4), p.gout16);
    }
    if (jb + 1 < njb) lds_barrier();
  }
}

// Molecules of more than one block triple: dq, dk2, dv2 are in the units' slabs; add them in unit order.  kCombineSplit
// workgroups per (molecule, head); a separate launch, so the stream orders it after the units without any
// cross-workgroup fence.
constexpr int kCombineSplit = 2;
__device__ __forceinline__ void combine(const Params& p, int split, int qm, int jm) {
  const int bh = blockIdx.x;
  const int b = bh / p.H;
  const int2 nkq = p.counts[b];
  const int nk = nkq.x, nq = nkq.y;
  if (nk <= 0 || nq <= 0) return;
  const int parts = parts_of(nk, p.head[1], p.cap);
  if (parts == 1 && nk <= jm && nq <= qm) return;  // one triple
  const size_t rbase = size_t(bh) * p.N;
  const size_t pstride = size_t(3) * p.N * DP;
  const float* slab = p.slab + size_t(bh) * p.cap * pstride;
  const uint16_t* klist = p.lists + size_t(2 * b) * p.N;
  const uint16_t* qlist = klist + p.N;
  // rows: dq of the nq queries, then dk2 and dv2 of the nk keys, 16 float4 each; kAt per thread at a time
  constexpr int kAt = 4;
  const int total = (nq + 2 * nk) * 16;
  for (int u0 = split * kAt * kThreads; u0 < total; u0 += kCombineSplit * kAt * kThreads) {
    float4 a[kAt];
    size_t so[kAt], dst[kAt];
    void* base[kAt];
#pragma unroll
    for (int i = 0; i < kAt; ++i) {
      const int u = min(u0 + int(threadIdx.x) + kThreads * i, total - 1);  // clamped: no branch around loads
      const int row = u / 16, q4 = u % 16;
      const int which = row < nq ? 0 : (row < nq + nk ? 1 : 2);
      const int rr = which == 0 ? row : (which == 1 ? row - nq : row - nq - nk);
      base[i] = which == 0 ? p.dq : (which == 1 ? p.dk2 : p.dv2);
      dst[i] = (rbase + (which == 0 ? qlist[rr] : klist[rr])) * DP + 4 * q4;
      so[i] = (size_t(which) * p.N + rr) * DP + 4 * q4;
      a[i] = *reinterpret_cast<const float4*>(slab + so[i]);
    }
    for (int part = 1; part < parts; ++part) {
#pragma unroll
      for (int i = 0; i < kAt; ++i) {
        const float4 s = *reinterpret_cast<const float4*>(slab + part * pstride + so[i]);
        a[i].x += s.x; a[i].y += s.y; a[i].z += s.z; a[i].w += s.w;
      }
    }
#pragma unroll
    for (int i = 0; i < kAt; ++i) {
      if (u0 + int(threadIdx.x) + kThreads * i < total) store_grad4(base[i], dst[i], a[i], p.gout16);
    }
  }
}

// dv_ik = gate_i sum of the parts and dgate_i = sum of the parts, in part order (du and dw are written by the
// units).  kFinishSplit workgroups per (molecule, head), each thread kFinishAt entries at a time.
constexpr int kFinishSplit = 4, kFinishAt = 4;
template <int BIAS>
__device__ __forceinline__ void bias_finish(const Params& p, int split) {
  const int bh = blockIdx.x;
  const int b = bh / p.H;
  const int2 nkq = p.counts[b];
  const int nk = nkq.x, nq = nkq.y;
  if (nk <= 0 || nq <= 0) return;
  const int tid = threadIdx.x;
  const int N = p.N;
  const size_t rbase = size_t(bh) * N;
  const uint16_t* klist = p.lists + size_t(2 * b) * N;
  const uint16_t* qlist = klist + N;
  const int parts = parts_of(nk, p.head[1], p.cap);
  if (p.dvb != nullptr) {
    const float* dvp = p.dvpart + size_t(bh) * p.cap * N * N;
    const int n = nq * nk, step = kThreads * kFinishSplit;
    for (int u0 = split * kThreads + tid; u0 < n; u0 += kFinishAt * step) {
      float sv[kFinishAt], gate[kFinishAt];
      size_t e[kFinishAt], o[kFinishAt];
#pragma unroll
      for (int t = 0; t < kFinishAt; ++t) {
        const int u = min(u0 + t * step, n - 1), i = u / nk, k = u % nk;  // clamped: loads without branches
        const int qi = qlist[i];
        e[t] = size_t(i) * N + k;
        o[t] = (rbase + qi) * N + klist[k];
        gate[t] = load_bias<BIAS>(p.bg, rbase + qi);
        sv[t] = dvp[e[t]];
      }
      for (int part = 1; part < parts; ++part)
#pragma unroll
        for (int t = 0; t < kFinishAt; ++t) sv[t] += dvp[size_t(part) * N * N + e[t]];
#pragma unroll
      for (int t = 0; t < kFinishAt; ++t)
        if (u0 + t * step < n) store_grad(p.dvb, o[t], gate[t] * sv[t], p.bout16);
    }
  }
  if (p.dgate != nullptr && split == 0) {
    const float* gp = p.dgpart + size_t(bh) * p.cap * N;
    for (int i = tid; i < nq; i += kThreads) {
      float s = gp[i];
      for (int part = 1; part < parts; ++part) s += gp[size_t(part) * N + i];
      store_grad(p.dgate, rbase + qlist[i], s, p.bout16);
    }
  }
}

// Both in one launch, side by side: workgroups 0 .. kCombineSplit - 1 of a (molecule, head) combine, the others (with
// a bias) finish its gradients (one molecule of 56 tokens, fp32 bias, 8 heads: 7 + 6 us as two launches).
template <int BIAS>
__global__ void __launch_bounds__(kThreads) pair_bwd_finish(Params p) {
  const int y = blockIdx.y;
  if (y < kCombineSplit) combine(p, y, Lay<BIAS != 0>::QM, Lay<BIAS != 0>::JM);
  else if constexpr (BIAS != 0) bias_finish<BIAS>(p, y - kCombineSplit);
}

}  // namespace pbwd

static size_t within_limit(size_t bytes) { return bytes <= pbwd::kWsLimit ? bytes : 0; }

size_t simplicial_pair_bwd_workspace_bytes(int batch, int heads, int tokens) {
  if (batch <= 0 || heads <= 0 || tokens <= 0 || batch > pbwd::kMaxPlanBatch || tokens > pbwd::kMaxTokens) return 0;
  // (with fewer bias gradients there may be more units per molecule)
  size_t most = 0;
  for (int w = 0; w < 9; ++w)
    most = std::max(most, within_limit(pbwd::Ws(batch, heads, tokens, w < 8, w & 1, w & 2, w & 4).bytes));
  return most;
}

// Bytes that this call uses, 0 when it is not one of the pair kernel's (its buffers' alignment aside).
size_t simplicial_pair_bwd_workspace_bytes(const mf_simplicial_bwd_args* a) {
  if (a->dtype != MF_DTYPE_BF16 || a->grad_dtype != MF_DTYPE_BF16 || a->head_dim != pbwd::DP) return 0;
  if (a->batch <= 0 || a->heads <= 0 || a->tokens <= 0 || a->batch > pbwd::kMaxPlanBatch || a->tokens > pbwd::kMaxTokens)
    return 0;
  if (a->angle_left != nullptr || a->message_left != nullptr) return 0;
  if (a->bias_u != nullptr && a->bias_dtype != MF_DTYPE_BF16 && a->bias_dtype != MF_DTYPE_F32) return 0;
  return within_limit(pbwd::Ws(a).bytes);
}

bool simplicial_pair_bwd_serves(const mf_simplicial_bwd_args* a) {
  const size_t need = simplicial_pair_bwd_workspace_bytes(a);
  if (need == 0 || a->workspace == nullptr || reinterpret_cast<uintptr_t>(a->workspace) % 256 != 0 ||
      a->workspace_bytes < need)
    return false;
  if (int64_t(a->batch) * a->heads >= (1 << 26)) return false;  // unit codes are 32 bits
  if (a->bias_u != nullptr && (!a->bias_v || !a->bias_w || !a->bias_gate)) return false;
  if (!a->dq || !a->dk1 || !a->dv1 || !a->dk2 || !a->dv2) return false;
  for (const void* ptr : {(const void*)a->q, (const void*)a->k1, (const void*)a->v1, (const void*)a->k2,
                          (const void*)a->v2, (const void*)a->grad_out, (const void*)a->out, (const void*)a->dq,
                          (const void*)a->dk1, (const void*)a->dv1, (const void*)a->dk2, (const void*)a->dv2})
    if (reinterpret_cast<uintptr_t>(ptr) % 16 != 0) return false;
  return true;
}

template <int BIAS>
static int launch_units(const pbwd::Params& p, int blocks, int bh, hipStream_t stream) {
  using namespace pbwd;
  constexpr size_t lds = Lay<BIAS != 0>::bytes;
  const int st = ensure_dynamic_lds(reinterpret_cast<const void*>(pair_bwd_kernel<BIAS>), int(lds));
  if (st != MF_OK) return st;
  hipLaunchKernelGGL(pair_bwd_kernel<BIAS>, dim3(unsigned(blocks)), dim3(kThreads), lds, stream, p);
  MF_HIP_CHECK(hipGetLastError());
  const bool finish = BIAS != 0 && (p.dvb != nullptr || p.dgate != nullptr);
  hipLaunchKernelGGL(pair_bwd_finish<BIAS>, dim3(unsigned(bh), kCombineSplit + (finish ? kFinishSplit : 0)), dim3(kThreads),
                     0, stream, p);
  MF_HIP_CHECK(hipGetLastError());
  return MF_OK;
}

int simplicial_pair_bwd_launch(const mf_simplicial_bwd_args* a, bool bias16, hipStream_t stream) {
  using namespace pbwd;
  const Ws ws(a);
  unsigned char* wsp = static_cast<unsigned char*>(a->workspace);
  const bool g16 = a->grads_dtype == MF_DTYPE_BF16;
  PlanParams pp{};
  pp.qv = a->query_valid;
  pp.pkv = a->pair_key_valid;
  pp.head = reinterpret_cast<int*>(wsp);
  pp.units = reinterpret_cast<uint32_t*>(wsp + ws.units);
  pp.counts = reinterpret_cast<int2*>(wsp + ws.counts);
  pp.lists = reinterpret_cast<uint16_t*>(wsp + ws.lists);
  pp.dq = a->dq; pp.dk1 = a->dk1; pp.dv1 = a->dv1; pp.dk2 = a->dk2; pp.dv2 = a->dv2;
  pp.B = a->batch;
  pp.H = a->heads;
  pp.N = a->tokens;
  pp.cap = ws.cap;
  pp.bias = a->bias_u != nullptr ? 1 : 0;
  pp.jm = pp.bias ? Lay<true>::JM : Lay<false>::JM;
  Params p{};
  p.head = pp.head;
  p.units = pp.units;
  p.counts = pp.counts;
  p.lists = pp.lists;
  p.slab = reinterpret_cast<float*>(wsp + ws.slab);
  p.q = static_cast<const __bf16*>(a->q);
  p.k1 = static_cast<const __bf16*>(a->k1);
  p.v1 = static_cast<const __bf16*>(a->v1);
  p.k2 = static_cast<const __bf16*>(a->k2);
  p.v2 = static_cast<const __bf16*>(a->v2);
  p.go = static_cast<const __bf16*>(a->grad_out);
  p.out = a->out;
  p.lse = a->lse;
  p.pv = a->pair_valid;
  p.dq = a->dq; p.dk1 = a->dk1; p.dv1 = a->dv1; p.dk2 = a->dk2; p.dv2 = a->dv2;
  p.gout16 = g16 ? 1 : 0;
  p.bout16 = bias16 ? 1 : 0;
  p.H = a->heads;
  p.N = a->tokens;
  p.cap = ws.cap;
  const bool bias = a->bias_u != nullptr;
  if (bias) {
    p.bu = a->bias_u; p.bv = a->bias_v; p.bw = a->bias_w; p.bg = a->bias_gate;
    p.du = a->du; p.dvb = a->dv_bias; p.dw = a->dw; p.dgate = a->dgate;
    p.dvpart = reinterpret_cast<float*>(wsp + ws.dvpart);
    p.dgpart = reinterpret_cast<float*>(wsp + ws.dgpart);
    p.dwpart = reinterpret_cast<float*>(wsp + ws.dwpart);
  }
  const int64_t bh = int64_t(a->batch) * a->heads;
  const int64_t blocks = bh * ws.cap;  // the most units a plan can list
  if (blocks > 0x7fffffffLL) return fail(MF_ERR_UNSUPPORTED, "mf_simplicial_bwd: grid too large");
  hipLaunchKernelGGL(pair_bwd_prepare, dim3(unsigned(g16 ? 1 + bh : 1)), dim3(kPlanThreads), 0, stream, pp);
  MF_HIP_CHECK(hipGetLastError());
  if (!bias) return launch_units<0>(p, int(blocks), int(bh), stream);
  if (a->bias_dtype == MF_DTYPE_BF16) return launch_units<1>(p, int(blocks), int(bh), stream);
  return launch_units<2>(p, int(blocks), int(bh), stream);
}

}  // namespace mf
