// DGDA prefill for per-channel gates (decay, erase and write gates [B,H,L,d] with
// unit or zero channel stride): the layer's gate layout, and every head size the
// reference's GPU prefill takes (d_k, d_v in {32, 64, 128}, triton_dgda.py:389-396):
// the kernels are instantiated for d_k in {32, 64, 128} and 32 or 64 value columns;
// d_v = 128 runs as two groups of 64 columns in the same launches (the recurrence is
// separable over value columns).  q, k, v in bf16, fp16 or fp32.
//
// Sub-chunks of SC = 16 tokens.  With Lam_i the inclusive cumulative log-decay of
// token i within the sub-chunk (a d_k-vector over key channels) and S the state at the
// sub-chunk start (reference math: cpu_dgda.py:101-146, common.py:229-268):
//   L_ij = sum_c (b*k)_ic k_jc e^{Lam_ic - Lam_jc}      i > j
//   A_ij = sum_c  q_ic    k_jc e^{Lam_ic - Lam_jc}      i >= j
//   (I + L) u = w*v - (b*k*e^Lam) S
//   o    = (q*e^Lam) S + A u
//   S'   = diag(e^{Lam_15}) (S + (k*e^-Lam)^T u)
// L and A are formed as (b*k*e^Lam)(k*e^-Lam)^T and (q*e^Lam)(k*e^-Lam)^T.  All of this
// holds while |Lam| <= 64 at every token and channel of the sub-chunk (e^{+-Lam} stay
// far inside fp32); in a sub-chunk with a wider range L and A are summed pair by pair on
// the VALU with exact exponentials and the update takes k*e^{Lam_15 - Lam}.  Decays above
// one are taken as the recurrence takes them.
// Products with fp32 operands split them into bf16 hi + lo (three or four MFMA products),
// so they carry ~16 mantissa bits; the triangular solve and the state are fp32.
//
// One wave runs one segment of one (b, h) sequence on its own: no workgroup barriers, no
// operand staged twice.  (Four waves per segment, 16 state columns each, share the key side but
// spend most of a sub-chunk in three barriers, a triangular inverse on one of them and reading
// every shared operand from LDS four times.)  The waves of a SIMD hide each other's latencies, and
// the operand layouts below keep the value side out of LDS altogether.  What bounds a wave is
// instruction issue: per sub-chunk at d_k = d_v = 64 about 1,000 VALU instructions with 64 columns
// and 800 with 32 (fused layer 1,800 and 1,500, 230 and 200 of them transcendental) beside 100 and
// 56 MFMAs, so that a wave alone on its SIMD takes 4.6 us with 64 columns and 3.0 with 32 (fused
// layer 32: 4.2), and two hardly less time each.  Whole calls, four waves per segment / one: B=4 H=10
// T=8192 d=128 fp16 1,383 / 364 us; B=1 H=10 T=2048 fp32 212 / 45 us; the fused layer's launches at
// B=4 T=32768 1,150 / 640 us, at B=1 T=1000 310 / 74 us.
//
// Layouts.  NKT = d_k / 16, NCT = columns / 16.  Lane (c = lane & 15, g = lane >> 4):
//  * staging: tokens 4g .. 4g+3, key channels NKT c .. NKT c + NKT-1, value channels
//    NCT c .. NCT c + NCT-1: every row load is 16 lanes on consecutive bytes;
//  * state: rows (key channels) (d_k/4) g .. (d_k/4) g + d_k/4 - 1, columns NCT c ..: the
//    accumulator tile (kt, t) has rows NKT m + kt (m = 0..15) and columns NCT n + t, so
//    element i of lane (c, g) is row (d_k/4) g + NKT i + kt, column NCT c + t;
//  * with that choice the staged k*e^-Lam are the A operand of the state update and the
//    staged w*v and the stored outputs are accumulator fragments, all without moving
//    between lanes; only the row operands b*k*e^Lam, q*e^Lam and k*e^-Lam (rows = tokens)
//    pass through LDS, written 8 and read 16 bytes at a time in the natural order;
//  * the solve wants one column per lane: a 4 x 4 transpose between registers and lane
//    groups with permlane swaps, then 120 FMAs against rows of L broadcast from LDS.
//
// Sequence parallelism.  A sequence is cut into nseg segments of equal length (see
// sub_cut).  One launch runs every segment from a zero state (the first from the initial
// state) and, as further waves, every later segment's transition M (S <- M S + N) from
// the identity, until M is exactly zero.  scan (three segments or more): start states of
// segments whose predecessor's M survived.  fix: every later segment from its true start
// state, over the sub-chunks until its M vanished, or in full.
//
// Fused layer prologue (PRO, d_k = d_v = 64; maba_hip_dgda_layer_prefill; reference layers/dgda.py:103-121,
// 186-207): the kernels read the layer's six bf16 projections instead of q, k, v and the
// gates, and form the op inputs in the staging step: the causal depthwise conv (kernel 4)
// + SiLU of q, k, v over [history, projections], the per-head L2 norm of k, the decay
// max(-softplus, -14) and the sigmoid erase and write gates, all in fp32 and never
// written back.  The decays e^max(-softplus(x), -14) = max(sigmoid(-x), e^-14) enter as they
// are and e^Lam as their running product, which saves a logarithm and an exponential per
// element.  A lane loads the seven rows its four tokens' taps cover.
#pragma once
#include "dgda_common.h"
#include "dgda_rows.h"

namespace maba {

constexpr int SUB_MAX_SEG = 256;         // segments per sequence at most
constexpr float LOG2E = 1.4426950408889634f;
constexpr float SUB_MFMA_RANGE = 64.f * LOG2E;   // largest |Lam| within a sub-chunk on the MFMA path, in log2 units
constexpr float SUB_MFMA_MIN = 1.6038108e-28f;   // e^-64, the same limit for the prologue's decay products
constexpr float DECAY_MIN = 8.3152872e-7f;       // e^-14
enum { SUB_MAIN = 0, SUB_FIX = 1 };

struct SubArgs {
  const void* q; int qs0, qs1, qs2;         // [B,H,L,dk], channel stride 1 (16-bit or fp32, see F32IN)
  const void* k; int ks0, ks1, ks2;
  const void* vp; int vs0, vs1, vs2;
  // gates: fp32, or 16-bit in q's format (see G16); channel stride 0 or 1 (all 1: GCH)
  const void* gp; int gs0, gs1, gs2, gs3;   // log_alpha (use_log) or alpha
  const void* bp; int bs0, bs1, bs2, bs3;   // erase gate b
  const void* wp; int ws0, ws1, ws2, ws3;   // write gate w
  View4 s0;
  void* op; int odt; int os0, os1, os2;     // output [B,H,L,dv], channel stride 1
  int ovec;        // output rows allow one vector store per lane and token
  MView4 sf;
  // [BH, nseg, dk (dv + dk)]: a slot per segment.  First N as the waves hold it, [column group]
  // [tile t][lane][tile kt][4]; then M, rows of dk bf16 hi and dk lo parts.  The scan turns N
  // into start states.
  float* agg;
  int* zc;         // [BH, nseg, 2]: sub-chunks after which the segment's M (64 columns each) is zero, -1 if never
  int H, L, BH, nseg, seglen, nchunks, nvh, dvt, use_log, has_s0;
  int mode;        // SUB_MAIN or SUB_FIX
  // fused prologue (PRO): the six bf16 projections [B, L, C] (q, k, v, decay, erase, write;
  // unit channel stride, head h at channels 64h ..), conv taps [C, 1, 4] (f32/bf16), the
  // bf16 conv history [B, C, 3] (null: zeros), the new history and the key-norm eps
  const uint16_t* px[6]; int pxs0[6], pxs1[6];
  const void* cw[3]; int cwdt; int cwsc[3], cwst[3];
  const uint16_t* ph[3]; int phs0[3], phs1[3], phs2[3];
  void* nh[3]; int nhdt[3]; int64_t nhs0[3], nhs1[3], nhs2[3];
  float eps;
  int f16;         // 16-bit q, k, v are fp16 (else bf16)
};

template <int N> using fvec = float __attribute__((ext_vector_type(N)));

// N consecutive row elements as loaded (16-bit pairs or fp32 words).  Prefetched rows stay
// raw until they are staged, so that no conversion waits for the loads.
template <bool F32, int N>
struct Row { uint32_t w[F32 ? N : N / 2]; };

// Rows start at a multiple of four elements (checked on the host).
template <bool F32, int N>
__device__ __forceinline__ Row<F32, N> load_row(const char* p) {
  constexpr int NW = F32 ? N : N / 2;
  Row<F32, N> r;
  if constexpr (NW == 1) {
    r.w[0] = *(const uint32_t*)p;
  } else if constexpr (NW == 2) {
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    const u2 v = *(const u2*)p;
    r.w[0] = v[0]; r.w[1] = v[1];
  } else {
    typedef uint32_t u4 __attribute__((ext_vector_type(4), aligned(8)));
#pragma unroll
    for (int i = 0; i < NW / 4; ++i) {
      const u4 v = ((const u4*)p)[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) r.w[4 * i + j] = v[j];
    }
  }
  return r;
}
// Element j; 16-bit ones are fp16 (F16) or bf16.
template <bool F16, bool F32, int N>
__device__ __forceinline__ float row_at(const Row<F32, N>& r, int j) {
  if constexpr (F32) return __uint_as_float(r.w[j]);
  else if constexpr (F16) return __half2float(__ushort_as_half((unsigned short)(r.w[j / 2] >> (16 * (j & 1)))));
  else return __uint_as_float((j & 1) ? r.w[j / 2] & 0xffff0000u : r.w[j / 2] << 16);
}
// N gate values of one token at channel stride cs (0 or 1), p at the first, as raw elements.
template <bool G16, bool GCH, int N>
__device__ __forceinline__ Row<!G16, N> load_gate(const char* p, int cs) {
  if constexpr (GCH) {
    return load_row<!G16, N>(p);
  } else {
    Row<!G16, N> r;
    if constexpr (G16) {
#pragma unroll
      for (int j = 0; j < N / 2; ++j)
        r.w[j] = (uint32_t)((const uint16_t*)p)[2 * j * cs] | ((uint32_t)((const uint16_t*)p)[(2 * j + 1) * cs] << 16);
    } else {
#pragma unroll
      for (int j = 0; j < N; ++j) r.w[j] = ((const uint32_t*)p)[j * cs];
    }
    return r;
  }
}

// ------------------------------------------------------------------ lane-group moves

// x[t] of lane group g  <->  x[g] of lane group t (4 x 4 transpose; its own inverse).
__device__ __forceinline__ void transpose4(uint32_t (&x)[4]) {
  swap32(x[0], x[2]);
  swap32(x[1], x[3]);
  swap16(x[0], x[1]);
  swap16(x[2], x[3]);
}
// Exclusive prefix over the lane groups (g = 0: the neutral element) and the total, of sums or
// (MUL) products.
template <bool MUL>
__device__ __forceinline__ void group_prefix(float x, int g, float& excl, float& tot) {
  auto op = [](float p, float q) { return MUL ? p * q : p + q; };
  const float one = MUL ? 1.f : 0.f;
  uint32_t a = __float_as_uint(x), b = a;
  swap16(a, b);                                    // a: x0 x0 x2 x2, b: x1 x1 x3 x3
  uint32_t lo = __float_as_uint(op(__uint_as_float(a), __uint_as_float(b))), hi = lo;
  swap32(lo, hi);                                  // lo: x0, x1 and hi: x2, x3 together, in every lane
  excl = op((g & 1) ? __uint_as_float(a) : one, (g & 2) ? __uint_as_float(lo) : one);
  tot = op(__uint_as_float(lo), __uint_as_float(hi));
}
// Sum over the 16 lanes of a row, in every lane (row_ror 8, 4, 2, 1).
__device__ __forceinline__ float row16_sum(float x) {
  auto ror = [](float v, auto ctrl_c) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl_c)::value, 0xf, 0xf, true));
  };
  using std::integral_constant;
  x = ror(x, integral_constant<int, 0x128>{});
  x = ror(x, integral_constant<int, 0x124>{});
  x = ror(x, integral_constant<int, 0x122>{});
  return ror(x, integral_constant<int, 0x121>{});
}
// LDS traffic of the wave so far is ordered before what follows (a wave's LDS operations
// execute in order; this keeps the compiler from moving them across).
__device__ __forceinline__ void wave_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// bf16 hi and lo parts of a pair, packed (x ~= hi + lo).
__device__ __forceinline__ void split2(float x0, float x1, uint32_t& h, uint32_t& l) {
  h = cvt_pk_bf16(x0, x1);
  l = cvt_pk_bf16(bf16_rem<0>(h, x0), bf16_rem<1>(h, x1));
}
// The same of a pair that stays in use: bf16_rem's dot product overwrites its operand, so it would
// cost a copy, and wait states on either side.
__device__ __forceinline__ void split2_kept(float x0, float x1, uint32_t& h, uint32_t& l) {
  h = cvt_pk_bf16(x0, x1);
  l = cvt_pk_bf16(x0 - __uint_as_float(h << 16), x1 - __uint_as_float(h & 0xffff0000u));
}
__device__ __forceinline__ i16x8 pack8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const u4 v = {a, b, c, d};
  return __builtin_bit_cast(i16x8, v);
}

// ------------------------------------------------------------------ the wave's LDS

template <bool PRO, int DK>
struct SubSmem {
  static constexpr int PK = DK + 8;   // row pitch of the bf16 row operands (16-byte aligned rows that shift banks)
  union {
    struct {   // rows = tokens
      __attribute__((aligned(16))) short BKh[SC * PK], BKl[SC * PK];   // -(b k e^Lam)
      __attribute__((aligned(16))) short QEh[SC * PK], QEl[SC * PK];   // q e^Lam
      __attribute__((aligned(16))) short KIh[SC * PK], KIl[SC * PK];   // k e^-Lam
      __attribute__((aligned(16))) float Lm[SC][SC];         // -L, rows i, zero for j >= i
      __attribute__((aligned(16))) float elast[DK];          // e^{Lam_15}
    } r;
    struct {   // pair-by-pair sums, fp32
      __attribute__((aligned(16))) float k[SC][DK], bk[SC][DK], q[SC][DK], lam[SC][DK];
    } f;
  };
  __attribute__((aligned(16))) float cw[PRO ? 3 : 1][4][PRO ? 64 : 1];   // the head's conv taps [stream][tap][channel]
};

// ------------------------------------------------------------------ one segment

// Sub-chunks [c_begin, c_end) of sequence bh.  ROLE OUT: from the state in Sr, outputs
// stored, state left in Sr.  ROLE MAP: the transition, v = 0 and no outputs; returns the
// sub-chunks after which Sr is exactly zero (-1: never).  col: the lane's first value
// column (of dvt); key-side work is the same for every column group.
template <bool MAP, bool F32IN, bool G16, bool GCH, bool PRO, int DK, int DV>
__device__ __forceinline__ int sub_run(const SubArgs& a, SubSmem<PRO, DK>& sm, int lane, int bh, int col,
                                       int c_begin, int c_end, f32x4 (&Sr)[DK / 16][MAP ? (DK < 64 ? DK : 64) / 16 : DV / 16]) {
  constexpr int NKT = DK / 16, NCT = MAP ? (DK < 64 ? DK : 64) / 16 : DV / 16, NVT = DV / 16;
  constexpr int NP = DK / 32;              // K = 32 steps over the key channels
  constexpr int PK = SubSmem<PRO, DK>::PK;
  constexpr int NL = DK / 4;               // state rows of a lane: channel NL g + l, l = NKT i + kt
  constexpr int ES = F32IN ? 4 : 2, EG = G16 ? 2 : 4;
  const int g = lane >> 4, c = lane & 15;
  const int bi = bh / a.H, hi = bh % a.H;
  const int kch = NKT * c;                 // the lane's first key channel

  // ---- row sources: a uniform base per sub-chunk plus a 32-bit lane offset
  auto base = [&](const void* p, int s0, int s1, int s2, int es, int t0) {
    return (const char*)p + ((int64_t)bi * s0 + (int64_t)hi * s1 + (int64_t)t0 * s2) * es;
  };
  // Output waves of the fused layer and of 32 columns keep pointers to the rows to load next (a
  // twentieth of a sub-chunk's instructions otherwise); elsewhere their registers cost more (64
  // columns at 160 heads T=1000 135 us without, 137 with).
  constexpr bool HOIST = !MAP && DK == 64 && (PRO || DV == 32);
  const char* src[6] = {};
  if constexpr (HOIST) {
    const int t0 = c_begin * SC;
    if constexpr (PRO) {
#pragma unroll
      for (int s = 0; s < 6; ++s) src[s] = base(a.px[s], a.pxs0[s], 0, a.pxs1[s], 2, max(t0 - 3, 0));
    } else {
      src[0] = base(a.q, a.qs0, a.qs1, a.qs2, ES, t0);
      src[1] = base(a.k, a.ks0, a.ks1, a.ks2, ES, t0);
      src[2] = base(a.vp, a.vs0, a.vs1, a.vs2, ES, t0);
      src[3] = base(a.gp, a.gs0, a.gs1, a.gs2, EG, t0);
      src[4] = base(a.bp, a.bs0, a.bs1, a.bs2, EG, t0);
      src[5] = base(a.wp, a.ws0, a.ws1, a.ws2, EG, t0);
    }
  }
  Row<F32IN, NKT> pq[4], pk[4];
  Row<F32IN, NVT> pv[4];
  Row<!G16, NKT> pg[4], pb[4];
  Row<!G16, NVT> pw[4];
  // fused prologue: rows 4g-3 .. 4g+3 of q, k, v, and the gates' rows (key side, value side)
  Row<false, 4> tq[7], tk[7], xg[2][4];
  Row<false, NVT> tv[7], xw[4];
  // rows past the end re-read the last one, as do rows before the first (replaced by the history)
  auto prefetch = [&](int cc) {
    const int t0 = cc * SC;
    if constexpr (PRO) {
      const int d = min(t0, 3);   // rows are counted from token t0 - d
      auto rows = [&](int s, auto& x, int ch, int m0, auto n_c) {
        constexpr int N = sizeof(x[0]) / 2;
        const char* p = !HOIST ? base(a.px[s], a.pxs0[s], 0, a.pxs1[s], 2, t0 - d) : src[s];
        const int S = 2 * a.pxs1[s], chb = 2 * (hi * 64 + ch);
        const uint32_t lane0 = 4u * g * S + chb, end = row_end(a.L - 1 - (t0 - d), SC - 1 + d, S, chb);
#pragma unroll
        for (int m = 0; m < decltype(n_c)::value; ++m)
          x[m] = load_row<false, N>(p + row_offset(lane0, m + m0 + d, S, end));
        if (HOIST) src[s] += (int64_t)(cc + 1 < c_end ? SC - 3 + d : 0) * S;
      };
      using std::integral_constant;
      if (!MAP) rows(0, tq, kch, -3, integral_constant<int, 7>{});
      rows(1, tk, kch, -3, integral_constant<int, 7>{});
      if (!MAP) rows(2, tv, col, -3, integral_constant<int, 7>{});
      rows(3, xg[0], kch, 0, integral_constant<int, 4>{});
      rows(4, xg[1], kch, 0, integral_constant<int, 4>{});
      if (!MAP) rows(5, xw, col, 0, integral_constant<int, 4>{});
    } else {
      auto rows = [&](int s, const void* b, int s0, int s1, int s2, int es, int chb, auto& x, auto load) {
        const int S = s2 * es;
        const char* p = !HOIST ? base(b, s0, s1, s2, es, t0) : src[s];
        const uint32_t lane0 = 4 * g * S + chb, end = row_end(a.L - 1 - t0, SC - 1, S, chb);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = load(p + row_offset(lane0, i, S, end));
        if (HOIST) src[s] += cc + 1 < c_end ? SC * S : 0;
      };
      auto lk = [](const char* p) { return load_row<F32IN, NKT>(p); };
      auto lv = [](const char* p) { return load_row<F32IN, NVT>(p); };
      // a gate's rows at channel stride 1, or its element at stride 0 (then chb is zero)
      const int ck = kch * EG, cv = col * EG;
      rows(1, a.k, a.ks0, a.ks1, a.ks2, ES, kch * ES, pk, lk);
      rows(3, a.gp, a.gs0, a.gs1, a.gs2, EG, GCH ? ck : ck * a.gs3, pg, [&](const char* p) { return load_gate<G16, GCH, NKT>(p, a.gs3); });
      rows(4, a.bp, a.bs0, a.bs1, a.bs2, EG, GCH ? ck : ck * a.bs3, pb, [&](const char* p) { return load_gate<G16, GCH, NKT>(p, a.bs3); });
      if (!MAP) {
        rows(0, a.q, a.qs0, a.qs1, a.qs2, ES, kch * ES, pq, lk);
        rows(2, a.vp, a.vs0, a.vs1, a.vs2, ES, col * ES, pv, lv);
        rows(5, a.wp, a.ws0, a.ws1, a.ws2, EG, GCH ? cv : cv * a.ws3, pw, [&](const char* p) { return load_gate<G16, GCH, NVT>(p, a.ws3); });
      }
    }
  };
  // fused prologue: taps before token 0 come from the history, or are zero
  auto hist_rows = [&](int s, auto& t, int ch) {
    constexpr int N = sizeof(t[0]) / 2;
    if (g != 0) return;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      uint32_t h[N] = {};
      if (a.ph[s]) {
        const uint16_t* hp = a.ph[s] + (int64_t)bi * a.phs0[s] + (int64_t)(hi * 64 + ch) * a.phs1[s] + (int64_t)m * a.phs2[s];
#pragma unroll
        for (int e = 0; e < N; ++e) h[e] = hp[(int64_t)e * a.phs1[s]];
      }
#pragma unroll
      for (int e = 0; e < N; e += 2) t[m].w[e / 2] = h[e] | (h[e + 1] << 16);
    }
  };
  // fused prologue: SiLU(depthwise conv) of the lane's four tokens and N channels from ch on
  auto conv = [&](int s, const auto& t, int ch, auto& y) {
    constexpr int N = sizeof(y[0]) / sizeof(float);
    fvec<N> w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = *(const fvec<N>*)&sm.cw[s][j][PRO ? ch : 0];
#pragma unroll
    for (int e = 0; e < N; ++e) {
      float x[7];
#pragma unroll
      for (int m = 0; m < 7; ++m) x[m] = row_at<false>(t[m], e);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float acc = w[3][e] * x[i + 3];
        acc = fmaf(w[2][e], x[i + 2], acc);
        acc = fmaf(w[1][e], x[i + 1], acc);
        acc = fmaf(w[0][e], x[i], acc);
        y[i][e] = pro_silu(acc);
      }
    }
  };

  // ---- outputs of a sub-chunk are stored during the next one's staging, before its
  // prefetch: the wait for the prefetched rows then does not cover the stores
  f32x4 ob[NVT];
  int ot0 = -1;
  auto flush = [&]() {
    if (MAP || ot0 < 0) return;
    const int nt = a.L - ot0;
    const int64_t ub = (int64_t)bi * a.os0 + (int64_t)hi * a.os1 + (int64_t)ot0 * a.os2;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 4 * g + i;
      if (t >= nt) continue;
      const int64_t off = ub + (int64_t)t * a.os2 + col;
      if (a.ovec && a.odt == MABA_BF16) {
        uint32_t* p = (uint32_t*)((uint16_t*)a.op + off);
        if constexpr (NVT == 4) *(uint2*)p = make_uint2(cvt_pk_bf16(ob[0][i], ob[1][i]), cvt_pk_bf16(ob[2][i], ob[3][i]));
        else p[0] = cvt_pk_bf16(ob[0][i], ob[1][i]);
      } else if (a.ovec && a.odt == MABA_F16) {
        auto pk = [](float x, float y) {
          return (uint32_t)__half_as_ushort(__float2half(x)) | ((uint32_t)__half_as_ushort(__float2half(y)) << 16);
        };
        uint32_t* p = (uint32_t*)((uint16_t*)a.op + off);
        if constexpr (NVT == 4) *(uint2*)p = make_uint2(pk(ob[0][i], ob[1][i]), pk(ob[2][i], ob[3][i]));
        else p[0] = pk(ob[0][i], ob[1][i]);
      } else if (a.ovec) {
        float* p = (float*)a.op + off;
        if constexpr (NVT == 4) *(f32x4*)p = f32x4{ob[0][i], ob[1][i], ob[2][i], ob[3][i]};
        else *(float2*)p = make_float2(ob[0][i], ob[1][i]);
      } else {
#pragma unroll
        for (int t2 = 0; t2 < NVT; ++t2) store_elem(a.op, a.odt, off + t2, ob[t2][i]);   // unaligned rows
      }
    }
  };

  if (c_begin < c_end) prefetch(c_begin);
  for (int cc = c_begin; cc < c_end; ++cc) {
    const int t0 = cc * SC, nt = a.L - t0;
    // ---- staging: the op inputs of tokens 4g + i
    float kk[4][NKT], la[4][NKT], be[4][NKT], qq[4][NKT];
    f32x4 ve[NCT];                         // w*v, then the solve's right-hand side
    if constexpr (PRO) {
      if (cc == 0) {
        if (!MAP) hist_rows(0, tq, kch);
        hist_rows(1, tk, kch);
        if (!MAP) hist_rows(2, tv, col);
      }
      conv(1, tk, kch, kk);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float ss = row16_sum(kk[i][0] * kk[i][0] + kk[i][1] * kk[i][1] + kk[i][2] * kk[i][2] + kk[i][3] * kk[i][3]);
        const float inv = pro_knorm_inv(ss, a.eps);
#pragma unroll
        for (int j = 0; j < NKT; ++j) {
          kk[i][j] *= inv;
          // the decay e^max(-softplus(x), -14) = max(1 / (1 + e^x), e^-14)
          la[i][j] = fmaxf(fast_rcp(1.f + fast_exp(row_at<false>(xg[0][i], j))), DECAY_MIN);
          be[i][j] = pro_sigmoid(row_at<false>(xg[1][i], j));
        }
      }
      if (!MAP) {
        float vv[4][NVT];
        conv(2, tv, col, vv);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < NVT; ++j) ve[j][i] = pro_sigmoid(row_at<false>(xw[i], j)) * vv[i][j];
        conv(0, tq, kch, qq);
      }
    } else {
      auto convert = [&](auto f16_c) {
        constexpr bool F16 = decltype(f16_c)::value;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int j = 0; j < NKT; ++j) {
            kk[i][j] = row_at<F16>(pk[i], j);
            be[i][j] = row_at<F16>(pb[i], j);
            la[i][j] = row_at<F16>(pg[i], j);
            if (!MAP) qq[i][j] = row_at<F16>(pq[i], j);
          }
          if (!MAP) {
#pragma unroll
            for (int j = 0; j < NVT; ++j) ve[j][i] = row_at<F16>(pw[i], j) * row_at<F16>(pv[i], j);
          }
        }
      };
      if (!F32IN && a.f16) convert(std::true_type{});   // one branch, not one per element
      else convert(std::false_type{});
      if (a.use_log) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < NKT; ++j) la[i][j] *= LOG2E;
      } else {
        asm volatile("");   // keeps this a branch
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < NKT; ++j) la[i][j] = __builtin_amdgcn_logf(fmaxf(la[i][j], 1e-20f));
      }
    }
    if (MAP) {
#pragma unroll
      for (int t = 0; t < NCT; ++t) ve[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (nt < SC) {   // tokens past the end: no decay, no key, no write
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool on = 4 * g + i < nt;
#pragma unroll
        for (int j = 0; j < NKT; ++j) {
          kk[i][j] = on ? kk[i][j] : 0.f;
          la[i][j] = on ? la[i][j] : PRO ? 1.f : 0.f;
          be[i][j] = on ? be[i][j] : 0.f;
          if (!MAP) qq[i][j] = on ? qq[i][j] : 0.f;
        }
#pragma unroll
        for (int t = 0; t < NCT; ++t) ve[t][i] = on ? ve[t][i] : 0.f;
      }
    }
    flush();
    // ---- Lam (PRO: e^Lam): prefix over the lane's tokens, then over the lane groups
    float lam[4][NKT], tot[NKT];
    auto prefix = [&](auto mul_c) {
      constexpr bool MUL = decltype(mul_c)::value;
#pragma unroll
      for (int j = 0; j < NKT; ++j) {
        lam[0][j] = la[0][j];
#pragma unroll
        for (int i = 1; i < 4; ++i) lam[i][j] = MUL ? lam[i - 1][j] * la[i][j] : lam[i - 1][j] + la[i][j];
        float ex;
        group_prefix<MUL>(lam[3][j], g, ex, tot[j]);
#pragma unroll
        for (int i = 0; i < 4; ++i) lam[i][j] = MUL ? lam[i][j] * ex : lam[i][j] + ex;
      }
    };
    prefix(std::integral_constant<bool, PRO>{});
    float mx = PRO ? 1.f : 0.f;
    bool over = false;
#pragma unroll
    for (int j = 0; j < NKT; ++j) {
#pragma unroll
      for (int i = 0; i < 4; ++i) mx = PRO ? fminf(mx, lam[i][j]) : fmaxf(mx, fabsf(lam[i][j]));
      if (!PRO) over |= !(tot[j] == tot[j]);   // fmaxf drops NaN, which every prefix that meets one carries to the total
    }
    over |= PRO ? !(mx >= SUB_MFMA_MIN) : !(mx <= SUB_MFMA_RANGE);
    const bool wide = __ballot(over) != 0ull;   // the same in every lane
    wave_fence();   // the previous sub-chunk's LDS reads come first
    // the row factors e^Lam and the keys scaled for the column side (wide: for the update only)
    float e[4][NKT], kx[4][NKT];
    f32x4 lt = {0.f, 0.f, 0.f, 0.f}, at = lt;    // -L and A: lane (c, g), element r: row i = c, column j = 4g + r
    if (!wide) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NKT; ++j) {
          e[i][j] = PRO ? lam[i][j] : __builtin_amdgcn_exp2f(lam[i][j]);
          kx[i][j] = kk[i][j] * (PRO ? fast_rcp(lam[i][j]) : __builtin_amdgcn_exp2f(-lam[i][j]));
          if (!PRO && i == 0) tot[j] = __builtin_amdgcn_exp2f(tot[j]);
        }
    } else {
      if constexpr (PRO) {   // in logarithms here: the products may have left fp32's range
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < NKT; ++j) la[i][j] = __builtin_amdgcn_logf(la[i][j]);
        prefix(std::false_type{});
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NKT; ++j) {
          sm.f.k[4 * g + i][kch + j] = kk[i][j];
          sm.f.bk[4 * g + i][kch + j] = be[i][j] * kk[i][j];
          if (!MAP) sm.f.q[4 * g + i][kch + j] = qq[i][j];
          sm.f.lam[4 * g + i][kch + j] = lam[i][j];
          e[i][j] = __builtin_amdgcn_exp2f(lam[i][j]);
          kx[i][j] = kk[i][j] * __builtin_amdgcn_exp2f(tot[j] - lam[i][j]);
        }
#pragma unroll
      for (int j = 0; j < NKT; ++j) tot[j] = __builtin_amdgcn_exp2f(tot[j]);
      wave_fence();
#pragma unroll 1
      for (int ch = 0; ch < DK; ch += 4) {
        const f32x4 li = *(const f32x4*)&sm.f.lam[c][ch], bi4 = *(const f32x4*)&sm.f.bk[c][ch];
        const f32x4 qi = MAP ? li : *(const f32x4*)&sm.f.q[c][ch];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const f32x4 lj = *(const f32x4*)&sm.f.lam[4 * g + r][ch], kj = *(const f32x4*)&sm.f.k[4 * g + r][ch];
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const float d = __builtin_amdgcn_exp2f(4 * g + r <= c ? li[x] - lj[x] : 0.f) * kj[x];   // later tokens' pairs are dropped below
            lt[r] = fmaf(-bi4[x], d, lt[r]);
            if (!MAP) at[r] = fmaf(qi[x], d, at[r]);
          }
        }
      }
      wave_fence();
    }
    {
      // ---- row operands to LDS; the update's A operand kf stays in registers
      i16x8 kf[NKT];
      {
        uint32_t kh_[4][NKT / 2], kl_[4][NKT / 2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int tk_ = 4 * g + i;
          uint32_t bh_[NKT / 2], bl_[NKT / 2], qh_[NKT / 2], ql_[NKT / 2];
#pragma unroll
          for (int j = 0; j < NKT; j += 2) {
            split2(-(be[i][j] * kk[i][j]) * e[i][j], -(be[i][j + 1] * kk[i][j + 1]) * e[i][j + 1], bh_[j / 2], bl_[j / 2]);
            split2(kx[i][j], kx[i][j + 1], kh_[i][j / 2], kl_[i][j / 2]);
            if (!MAP) split2(qq[i][j] * e[i][j], qq[i][j + 1] * e[i][j + 1], qh_[j / 2], ql_[j / 2]);
          }
          auto put = [&](short* dst, const uint32_t (&v)[NKT / 2]) {
            uint32_t* p = (uint32_t*)(dst + tk_ * PK + kch);
            if constexpr (NKT == 2) p[0] = v[0];
            else if constexpr (NKT == 4) *(uint2*)p = make_uint2(v[0], v[1]);
            else *(uint4*)p = make_uint4(v[0], v[1], v[2], v[3]);
          };
          put(sm.r.BKh, bh_);
          put(sm.r.BKl, bl_);
          put(sm.r.KIh, kh_[i]);
          put(sm.r.KIl, kl_[i]);
          if (!MAP) {
            put(sm.r.QEh, qh_);
            put(sm.r.QEl, ql_);
          }
        }
#pragma unroll
        for (int j = 0; j < NKT; ++j) {
          // [hi | lo] of tokens 4g .. 4g+3, channel kch + j, from the pairs of channels
          const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
          auto two = [&](const uint32_t (&v)[4][NKT / 2], int i) { return __builtin_amdgcn_perm(v[i + 1][j / 2], v[i][j / 2], sel); };
          kf[j] = pack8(two(kh_, 0), two(kh_, 2), two(kl_, 0), two(kl_, 2));
        }
        if (g == 3) {
#pragma unroll
          for (int j = 0; j < NKT; ++j) sm.r.elast[kch + j] = tot[j];
        }
      }
      wave_fence();
      // ---- -L and A as products, and the row operands for those with S
      i16x8 bh8[NP], bl8[NP], qh8[NP], ql8[NP];
      i16x8 af = {};
      {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const int off = c * PK + NL * g + 8 * p;
          bh8[p] = *(const i16x8*)(sm.r.BKh + off);
          bl8[p] = *(const i16x8*)(sm.r.BKl + off);
          if (!MAP) {
            qh8[p] = *(const i16x8*)(sm.r.QEh + off);
            ql8[p] = *(const i16x8*)(sm.r.QEl + off);
          }
        }
        if (!wide) {
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            const int off = c * PK + NL * g + 8 * p;
            const i16x8 kh8 = *(const i16x8*)(sm.r.KIh + off), kl8 = *(const i16x8*)(sm.r.KIl + off);
            lt = mma32(lt, kh8, bh8[p]);
            lt = mma32(lt, kh8, bl8[p]);
            lt = mma32(lt, kl8, bh8[p]);
            if (!MAP) {
              at = mma32(at, kh8, qh8[p]);
              at = mma32(at, kh8, ql8[p]);
              at = mma32(at, kl8, qh8[p]);
            }
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) lt[r] = 4 * g + r < c ? lt[r] : 0.f;
        *(f32x4*)&sm.r.Lm[c][4 * g] = lt;
        if (!MAP) {
#pragma unroll
          for (int r = 0; r < 4; ++r) at[r] = 4 * g + r <= c ? at[r] : 0.f;
          uint32_t h0, h1, l0, l1;
          split2(at[0], at[1], h0, l0);
          split2(at[2], at[3], h1, l1);
          af = pack8(h0, h1, l0, l1);
        }
      }
      // ---- v_e = w*v - (b k e^Lam) S and q S, both tokens 4g + i of the lane's columns
      f32x4 qs[NVT];
#pragma unroll
      for (int t = 0; t < NCT; ++t) {
        if (!MAP) qs[t < NVT ? t : 0] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          uint32_t h[4], l[4];
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            const int l0 = 8 * p + e, l1 = l0 + 1;
            split2_kept(Sr[l0 % NKT][t][l0 / NKT], Sr[l1 % NKT][t][l1 / NKT], h[e / 2], l[e / 2]);
          }
          const i16x8 sh = pack8(h[0], h[1], h[2], h[3]), sl = pack8(l[0], l[1], l[2], l[3]);
          ve[t] = mma32(ve[t], bh8[p], sh);
          ve[t] = mma32(ve[t], bh8[p], sl);
          ve[t] = mma32(ve[t], bl8[p], sh);
          if (!MAP) {
            f32x4& q_ = qs[t < NVT ? t : 0];
            q_ = mma32(q_, qh8[p], sh);
            q_ = mma32(q_, qh8[p], sl);
            q_ = mma32(q_, ql8[p], sh);
          }
        }
      }
      f32x4 el[NL / 4];
#pragma unroll
      for (int l = 0; l < NL / 4; ++l) el[l] = *(const f32x4*)&sm.r.elast[NL * g + 4 * l];
      if (wide) {   // S' = e^{Lam_15} S + (k e^{Lam_15 - Lam})^T u
        asm volatile("");   // keeps this a branch
#pragma unroll
        for (int t = 0; t < NCT; ++t)
#pragma unroll
          for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) Sr[kt][t][i] *= el[(NKT * i + kt) / 4][(NKT * i + kt) % 4];
#pragma unroll
        for (int l = 0; l < NL / 4; ++l) el[l] = f32x4{1.f, 1.f, 1.f, 1.f};
      }
      wave_fence();
      // ---- (I + L) u = v_e: one column per lane, u[4G + i] = token 4G + i
      float u[SC];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t x[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) x[t] = t < NCT ? __float_as_uint(ve[t < NCT ? t : 0][i]) : 0u;
        transpose4(x);
#pragma unroll
        for (int t = 0; t < 4; ++t) u[4 * t + i] = __uint_as_float(x[t]);
      }
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
#pragma unroll
        for (int i = 4 * jb + 1; i < SC; ++i) {
          const f32x4 lr = *(const f32x4*)&sm.r.Lm[i][4 * jb];   // broadcast
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (4 * jb + r < i) u[i] = fmaf(lr[r], u[4 * jb + r], u[i]);
        }
      }
      // the next rows: from here on the registers have room for them
      prefetch(min(cc + 1, c_end - 1));
      // ---- u as B operands: hi and lo pairs back to tokens 4g + i of the lane's columns
      uint32_t uh[2][4], ul[2][4];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
#pragma unroll
        for (int G = 0; G < 4; ++G) split2(u[4 * G + 2 * m], u[4 * G + 2 * m + 1], uh[m][G], ul[m][G]);
        transpose4(uh[m]);
        transpose4(ul[m]);
      }
#pragma unroll
      for (int t = 0; t < NCT; ++t) {
        const i16x8 uh8 = pack8(uh[0][t], uh[1][t], uh[0][t], uh[1][t]);
        const i16x8 ul8 = pack8(ul[0][t], ul[1][t], ul[0][t], ul[1][t]);
        if (!MAP) {
          f32x4 o = qs[t < NVT ? t : 0];
          o = mma32(o, af, uh8);
          ob[t < NVT ? t : 0] = mma32(o, af, ul8);
        }
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
          f32x4 s = Sr[kt][t];
          s = mma32(s, kf[kt], uh8);
          s = mma32(s, kf[kt], ul8);
#pragma unroll
          for (int i = 0; i < 4; ++i) s[i] *= el[(NKT * i + kt) / 4][(NKT * i + kt) % 4];
          Sr[kt][t] = s;
        }
      }
    }
    ot0 = t0;
    if (MAP) {
      uint32_t nz = 0;
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int t = 0; t < NCT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) nz |= __float_as_uint(Sr[kt][t][i]);
      if (__ballot((nz << 1) != 0u) == 0ull) return cc + 1 - c_begin;
    }
  }
  flush();
  return -1;
}

// The new conv history of head hi: the last three conv inputs, from the projections or, for
// fewer than three tokens, the old history (all read before any is written: the two may be
// the same buffers).
__device__ __forceinline__ void sub_new_history(const SubArgs& a, int lane, int bi, int hi) {
  const int ch = hi * 64 + lane;
  float x[3][3];
#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const int t = a.L - 3 + m;
      x[s][m] = 0.f;
      if (t >= 0) x[s][m] = bf16_bits_to_f32(a.px[s][(int64_t)bi * a.pxs0[s] + (int64_t)t * a.pxs1[s] + ch]);
      else if (a.ph[s])
        x[s][m] = bf16_bits_to_f32(a.ph[s][(int64_t)bi * a.phs0[s] + (int64_t)ch * a.phs1[s] + (int64_t)(t + 3) * a.phs2[s]]);
    }
#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int m = 0; m < 3; ++m)
      store_elem(a.nh[s], a.nhdt[s], bi * a.nhs0[s] + ch * a.nhs1[s] + m * a.nhs2[s], x[s][m]);
}

// One wave per workgroup.  SUB_MAIN: BH * nseg * nvh output waves, then BH * (nseg - 1) *
// (d_k / 64) transition waves of the segments k >= 1.  SUB_FIX: the output waves of the
// segments k >= 1.  Two waves per SIMD (256 VGPRs); d_k = 128 holds twice the state per
// lane and runs one.
template <bool F32IN, bool G16, bool GCH, bool PRO, int DK, int DV>
__global__ __launch_bounds__(64, DK == 128 ? 1 : 2) void dgda_sub_kernel(SubArgs a) {
  static_assert(!PRO || DK == 64, "the fused prologue takes 64-channel heads");
  static_assert((DK == 32 || DK == 64 || DK == 128) && (DV == 32 || DV == 64), "head sizes");
  constexpr int NKT = DK / 16, NVT = DV / 16;
  constexpr int MC = DK < 64 ? DK : 64, NMT = MC / 16, NCG = DK / MC;   // transition columns per wave, waves per map
  __shared__ SubSmem<PRO, DK> sm;
  const int lane = threadIdx.x;
  const int g = lane >> 4, c = lane & 15;
  const int nout = a.mode == SUB_FIX ? a.BH * (a.nseg - 1) * a.nvh : a.BH * a.nseg * a.nvh;
  const int AW = a.dvt + DK;
  int id = blockIdx.x;
  const bool map = id >= nout;
  int k, bh, part;
  if (map) {
    id -= nout;
    part = id % NCG;
    id /= NCG;
    bh = id / (a.nseg - 1);
    k = id % (a.nseg - 1) + 1;
  } else {
    part = id % a.nvh;
    id /= a.nvh;
    if (a.mode == SUB_FIX) {
      bh = id / (a.nseg - 1);
      k = id % (a.nseg - 1) + 1;
    } else {
      bh = id / a.nseg;
      k = id % a.nseg;
    }
  }
  const int c0 = k * a.seglen;
  int c1 = min(c0 + a.seglen, a.nchunks);
  const bool last = k == a.nseg - 1;
  const int bi = bh / a.H, hi = bh % a.H;
  int* zc = a.zc + 2 * ((int64_t)bh * a.nseg + k);
  if constexpr (PRO) {
    for (int i = lane; i < 3 * 4 * 64; i += 64) {
      const int s = i >> 8, j = (i >> 6) & 3, cl = i & 63;
      sm.cw[s][j][cl] = load_elem(a.cw[s], a.cwdt, (int64_t)(hi * 64 + cl) * a.cwsc[s] + j * a.cwst[s]);
    }
    wave_fence();
  }

  if (map) {
    const int col = MC * part + NMT * c;
    f32x4 Sr[NKT][NMT];
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
      for (int t = 0; t < NMT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) Sr[kt][t][i] = (DK / 4) * g + NKT * i + kt == col + t ? 1.f : 0.f;
    const int z = sub_run<true, F32IN, G16, GCH, PRO, DK, DV>(a, sm, lane, bh, 0, c0, c1, Sr);
    if (lane == 0) {
      zc[part] = z;
      if (NCG == 1) zc[1] = z;
    }
    if (z < 0 && !last) {
      uint32_t* dst = (uint32_t*)(a.agg + ((int64_t)bh * a.nseg + k) * DK * AW + DK * a.dvt) + col / 2;
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int t = 0; t < NMT; t += 2) {
            uint32_t* row = dst + ((DK / 4) * g + NKT * i + kt) * DK + t / 2;
            split2(Sr[kt][t][i], Sr[kt][t + 1][i], row[0], row[DK / 2]);
          }
    }
    return;
  }

  const int col = DV * part + NVT * c;
  f32x4 Sr[NKT][NVT];
  auto fill = [&](auto load) {
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < NVT; ++t) Sr[kt][t][i] = load((DK / 4) * g + NKT * i + kt, t);
  };
  // the state in slot s of the sequence
  auto slot = [&](int s) {
    return (f32x4*)(a.agg + ((int64_t)bh * a.nseg + s) * DK * AW + DK * DV * part) + lane * NKT;
  };
  auto fetch = [&](const f32x4* src) {
#pragma unroll
    for (int t = 0; t < NVT; ++t)
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt) Sr[kt][t] = src[64 * NKT * t + kt];
  };
  int z = -1;
  if (a.mode == SUB_FIX) {
    z = zc[0] < 0 || zc[1] < 0 ? -1 : max(zc[0], zc[1]);
    if (z >= 0) c1 = c0 + z;
    fetch(slot(k - 1));
  } else if (k == 0 && a.has_s0) {
    const int64_t o = bi * a.s0.s0 + hi * a.s0.s1 + col * a.s0.s3, rs = a.s0.s2, cs = a.s0.s3;
    if (a.s0.dt == MABA_F32) fill([&](int r, int t) { return ((const float*)a.s0.p)[o + r * rs + t * cs]; });
    else if (a.s0.dt == MABA_BF16) fill([&](int r, int t) { return bf16_bits_to_f32(((const uint16_t*)a.s0.p)[o + r * rs + t * cs]); });
    else fill([&](int r, int t) { return __half2float(((const __half*)a.s0.p)[o + r * rs + t * cs]); });
  } else {
    fill([&](int, int) { return 0.f; });
  }
  sub_run<false, F32IN, G16, GCH, PRO, DK, DV>(a, sm, lane, bh, col, c0, c1, Sr);
  if constexpr (PRO) {
    // after the sequence's first segment has read the old history, which this may overwrite
    if (last && part == 0 && (a.nseg == 1 || a.mode == SUB_FIX)) sub_new_history(a, lane, bi, hi);
  }
  auto drain = [&](auto put) {
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < NVT; ++t) put((DK / 4) * g + NKT * i + kt, t, Sr[kt][t][i]);
  };
  if (last && (a.nseg == 1 || a.mode == SUB_FIX)) {
    // (never in the launch that reads the initial state from another wave: the two may be one buffer)
    if (z >= 0) fetch(slot(k));   // the zero start's end state is the true one
    const int64_t o = bi * a.sf.s0 + hi * a.sf.s1 + col * a.sf.s3, rs = a.sf.s2, cs = a.sf.s3;
    if (a.sf.dt == MABA_F32) drain([&](int r, int t, float v) { ((float*)a.sf.p)[o + r * rs + t * cs] = v; });
    else if (a.sf.dt == MABA_BF16)
      drain([&](int r, int t, float v) { ((uint16_t*)a.sf.p)[o + r * rs + t * cs] = f32_to_bf16_bits(v); });
    else drain([&](int r, int t, float v) { ((__half*)a.sf.p)[o + r * rs + t * cs] = __float2half(v); });
  } else if (a.mode == SUB_MAIN) {   // N_k
    f32x4* dst = slot(k);
#pragma unroll
    for (int t = 0; t < NVT; ++t)
#pragma unroll
      for (int kt = 0; kt < NKT; ++kt) dst[64 * NKT * t + kt] = Sr[kt][t];
  }
}

// Start states: slot k of a sequence holds N_k, segment k's end state from a zero start
// (from the initial state for k = 0), and becomes the true one, S_{k+1} = M_k S_k + N_k,
// where M_k survived (else N_k already is it).  One wave per 16 columns of one sequence
// walks its slots in order; M (stored split) and S as bf16 hi + lo, three products.  A
// slot's loads do not depend on the walk, so they run DEPTH slots ahead (what a wave may
// have outstanding, 63 operations, allows no more).
template <int DK>
__global__ __launch_bounds__(64, 1) void dgda_sub_scan_kernel(SubArgs a) {
  constexpr int NKT = DK / 16, NP = DK / 32, NL = DK / 4;
  constexpr int DEPTH = DK == 128 ? 1 : 3;
  const int lane = threadIdx.x;
  const int g = lane >> 4, c = lane & 15;
  const int bh = blockIdx.x, AW = a.dvt + DK;
  const int* zc = a.zc + 2 * (int64_t)bh * a.nseg;
  float* agg = a.agg + (int64_t)bh * a.nseg * DK * AW;
  const int64_t slot = (int64_t)DK * AW;
  const int own = blockIdx.y * 64 * 4 * NKT + lane * 4 * NKT;   // a tile of 16 columns, as sub_run's waves hold it
  const int kend = a.nseg - 1;   // slots 1 .. kend - 1 (the last segment's end state starts nothing)

  // which slots survived; most calls have none and end here
  __shared__ uint8_t alive[SUB_MAX_SEG];
  int any = 0;
  for (int k = threadIdx.x; k < kend; k += blockDim.x) {
    alive[k] = k < 1 ? 0 : (zc[2 * k] < 0 ? 1 : 0) | (zc[2 * k + 1] < 0 ? 2 : 0);   // M's column halves
    any |= alive[k];
  }
  if (!__syncthreads_or(any)) return;

  // tile kt: rows NKT m + kt, so element i of the lane is row NL g + NKT i + kt, as in sub_run
  struct Slot { f32x4 n[NKT]; i16x8 mh[NKT][NP], ml[NKT][NP]; } buf[DEPTH];
  auto load = [&](Slot& s, int k) {
    const float* X = agg + min(k, kend - 1) * slot;
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt) {
      s.n[kt] = *(const f32x4*)(X + own + 4 * kt);
      const short* mrow = (const short*)(X + DK * a.dvt + (NKT * c + kt) * DK) + NL * g;
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        s.mh[kt][p] = *(const i16x8*)(mrow + 8 * p);
        s.ml[kt][p] = *(const i16x8*)(mrow + DK + 8 * p);
      }
    }
  };
  f32x4 Sr[NKT];
#pragma unroll
  for (int kt = 0; kt < NKT; ++kt) Sr[kt] = *(const f32x4*)(agg + own + 4 * kt);
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load(buf[d], 1 + d);
  // The step is straight-line code (a vanished slot's products are dropped and its N stored
  // back), so that the wait for one slot's loads is not a wait for the later slots'.
  auto step = [&](Slot& b, int k, int alive) {
    if constexpr (DK == 128) {
      // one half of M's columns vanished: its wave stored nothing there
      if (alive == 1 || alive == 2) {
        const bool drop = alive == (g < 2 ? 2 : 1);   // lane groups 0, 1 hold columns 0 .. 63
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            b.mh[kt][p] = drop ? i16x8{} : b.mh[kt][p];
            b.ml[kt][p] = drop ? i16x8{} : b.ml[kt][p];
          }
      }
    }
    i16x8 sh[NP], sl[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      uint32_t h[4], l[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const int l0 = 8 * p + e, l1 = l0 + 1;
        split2(Sr[l0 % NKT][l0 / NKT], Sr[l1 % NKT][l1 / NKT], h[e / 2], l[e / 2]);
      }
      sh[p] = pack8(h[0], h[1], h[2], h[3]);
      sl[p] = pack8(l[0], l[1], l[2], l[3]);
    }
    float* X = agg + k * slot;
#pragma unroll
    for (int kt = 0; kt < NKT; ++kt) {
      f32x4 acc = b.n[kt];
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        acc = mma32(acc, b.mh[kt][p], sh[p]);
        acc = mma32(acc, b.mh[kt][p], sl[p]);
        acc = mma32(acc, b.ml[kt][p], sh[p]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) Sr[kt][i] = alive ? acc[i] : b.n[kt][i];
      *(f32x4*)(X + own + 4 * kt) = Sr[kt];
    }
  };
  int k = 1;
  for (; k + DEPTH <= kend; k += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      step(buf[d], k + d, alive[k + d]);
      load(buf[d], k + d + DEPTH);
    }
  }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    if (k + d >= kend) break;
    step(buf[d], k + d, alive[k + d]);
  }
}

// The launches of one prefill.  PRO: the fused-prologue inputs (bf16 projections).  f32in:
// fp32 q, k, v; g16: 16-bit gates in q's format (only with 16-bit q, k, v); gch: every gate
// per channel.
template <bool PRO, int DK, int DV>
int run_sub_passes(SubArgs& a, bool f32in, bool g16, bool gch, hipStream_t stream) {
  constexpr int NCG = DK > 64 ? DK / 64 : 1;
  auto launch = [&](int mode) {
    a.mode = mode;
    const int64_t per = (int64_t)a.BH * a.nvh;
    const dim3 grid((unsigned)(mode == SUB_MAIN ? per * a.nseg + (int64_t)a.BH * (a.nseg - 1) * NCG : per * (a.nseg - 1)));
#define MABA_SUB_K(F, G, C) hipLaunchKernelGGL((dgda_sub_kernel<F, G, C, PRO, DK, DV>), grid, dim3(64), 0, stream, a)
    if constexpr (PRO) {
      MABA_SUB_K(false, false, true);
    } else if (f32in) {
      if (gch) MABA_SUB_K(true, false, true);
      else MABA_SUB_K(true, false, false);
    } else if (g16) {
      if (gch) MABA_SUB_K(false, true, true);
      else MABA_SUB_K(false, true, false);
    } else {
      if (gch) MABA_SUB_K(false, false, true);
      else MABA_SUB_K(false, false, false);
    }
#undef MABA_SUB_K
    return check_launch("dgda_prefill/sub-chunk");
  };
  int rc = launch(SUB_MAIN);
  if (rc || a.nseg == 1) return rc;
  if (a.nseg > 2) {
    hipLaunchKernelGGL((dgda_sub_scan_kernel<DK>), dim3((unsigned)a.BH, (unsigned)(a.dvt / 16)), dim3(64), 0, stream, a);
    if ((rc = check_launch("dgda_prefill/sub-chunk scan"))) return rc;
  }
  return launch(SUB_FIX);
}

// One translation unit per d_k instantiates the kernels (dgda_sub_k32.hip, dgda_sub.hip,
// dgda_sub_k128.hip), so that they compile in parallel; dv is 32 or 64 columns.
int run_sub_k32(SubArgs& a, int dv, bool f32in, bool g16, bool gch, hipStream_t stream);
int run_sub_k64(SubArgs& a, int dv, bool f32in, bool g16, bool gch, hipStream_t stream);
int run_sub_k128(SubArgs& a, int dv, bool f32in, bool g16, bool gch, hipStream_t stream);

}  // namespace maba
