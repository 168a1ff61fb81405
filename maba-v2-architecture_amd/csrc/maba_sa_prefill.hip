// MABA-SA prefill: the three attention streams for every query of a sequence and their
// gate superposition, without the reference's dense [Lq, Lkv] masks.
//
// Reference semantics (maba_sparse/layers/sparse_attention.py), per batch b, head h and
// query t at position pos = (Lkv - Lq) + t, with per-head keys/values k, v [Lkv, dh]:
//   local  (:95-105)  keys j <= pos with pos - j < window or j < min(n_sink, Lkv)
//   sparse (:145-171) the tokens of the blocks idx[b, t, :] that are < Lkv and <= pos
//                     (a block listed twice counts twice, as the reference's gather does)
//   HCA    (:173-219) pos >= pool - 1: the complete-block means e with (e+1) pool - 1 <= pos,
//                     keys kh / values vh (up-projected means); pos < pool - 1: the caller's
//                     running-mean row early[t]
//   gate   (:275)     out = sum_s softmax(logits)_s o_s; a stream with no valid key gives 0
//
// One workgroup per 64 consecutive queries of one (b, h), one wave per 16 of them.  The
// workgroup walks one list of 64-key tiles -- local (sinks, then the window of all 64
// queries), sparse (the union of the 64 queries' blocks, from an LDS bitmap compacted in
// ascending block order), HCA (the means any of them sees) -- staging each key and value tile
// once into double-buffered LDS, the next tile's loads in flight while the current one
// computes, one barrier per tile.  Per tile and wave, on bf16 MFMA with fp32 accumulation:
//   scores  S^T[key][query] = K Q^T     (A: key rows from the LDS tile, B: the wave's
//                                        16 queries in registers)
//   values  O^T[dim][query] += V^T P    (A: V^T fragments read transposed from the LDS
//                                        tile, B: the probabilities in bf16 hi + lo)
// with an online softmax per query and stream; each sparse key is weighted by how often the
// lane's query lists its block.  A wave skips the tiles none of its queries weights.
//
// The kernel is bound by VALU issue, not by its products (a tile's 24 MFMAs are 384 cycles of
// the matrix unit), so the softmax is kept to one FMA, one maximum, one exp2, one addition and
// the hi/lo split per score:
//  * the running reference m of a query moves only when a score passes it by 2^PF_SLACK; only
//    then do lanes exchange maxima and the sums rescale;
//  * a key's weight is folded into the exponent as its log2, so an unlisted block is a bias of
//    -inf and a block listed once costs nothing.  Where that score is infinite or NaN the sum is
//    NaN; the tile's largest score is therefore taken with the maximum that carries NaN, and only
//    a tile that has one masks its rows with selects (no cost per score: v_maximum3_f32, two
//    scores each; with a slack of 8, 2.66 -> 2.57 ms at the first size below against fmaxf);
//  * the probabilities' sum is a product with a row of ones, on the matrix unit;
//  * which union entries a query lists is a row of bits in LDS, one word per 32 entries, in
//    place of comparing the entry with all of the query's slots (which remains for unions
//    beyond PF_QWORDS words and for queries that list a block twice);
//  * a tile inside every query's range skips the row masks, and the staging addresses are a
//    uniform base and a 32-bit lane offset.
// Measured at B=1 H=10 dh=64 T=32768, top-32 (first of each pair: a maximum and a rescale per
// tile, counted slots, 64-bit addresses, padded rows): random queries, 5.1 K distinct blocks
// per 16 of them, 3.82 -> 2.62 ms; neighbouring queries alike 1.13 -> 0.83 ms.  VALU
// instructions per call 1,234 M -> 605 M, a quarter of the SIMDs' cycles MFMA, LDS bank conflicts 390
// M -> 12 M cycles.  Tiles loaded straight to LDS three ahead, with 64 or 128 queries per workgroup,
// measured the same on random queries and 12 to 20 % slower on alike ones (two workgroups per CU
// instead of three): issue bounds it, not latency.
#include <algorithm>

#include "dgda_common.h"

namespace maba {

constexpr int PF_MAXK = 64;          // index slots per query
constexpr int PF_WORDS = 512;        // bitmap words per workgroup: blocks below 16384
constexpr int PF_LIST = 64 * PF_MAXK;   // the union of a workgroup's 64 queries' slots
constexpr int PF_QWORDS = 16;        // words of a query's row of union bits (512 entries)
// A score may pass the running reference by 2^PF_SLACK.  The heaviest key's probability is exact in
// bf16 hi + lo while the reference is its score; the more the reference lags, the larger that key's
// rounding: error against 64 bits before the output's rounding (queries of twice unit variance,
// T=2048) 9.43e-7 at 0, 9.50e-7 at 0.5, 9.6e-7 at 1, 1.30e-6 at 8 (a maximum per tile, the sums on
// the VALU: 9.86e-7); time at T=32768 2.71, 2.65, 2.63 and 2.56 ms
// (2.61 with no sums rescaled at a stream's first tile).
constexpr float PF_SLACK = 0.5f;

// The workgroup's union of blocks; behind a list of at most 32 PF_QWORDS of them, the rows of bits.
union PfList {
  uint16_t block[PF_LIST];
  struct {
    uint16_t list[32 * PF_QWORDS];
    uint32_t qbits[64][PF_QWORDS];   // per query, the list entries it lists
  } behind;
};
static_assert(sizeof(PfList) == PF_LIST * 2, "the rows of bits fit behind the list");

typedef __attribute__((ext_vector_type(8))) short pf16x8;
typedef __attribute__((ext_vector_type(4))) short pf16x4;

struct PfArgs {
  const uint16_t* q; int64_t qsb, qsh, qst;       // [B,H,Lq,dh] bf16, unit channel stride
  const uint16_t* k; int64_t ksb, ksh, kst;       // [B,H,Lkv,dh]
  const uint16_t* v; int64_t vsb, vsh, vst;
  const uint16_t* kh; int64_t khb, khh, khe;      // [B,H,nc,dh] (unused when nc == 0)
  const uint16_t* vh; int64_t vhb, vhh, vhe;
  const void* early; int edt; int64_t esb, esh, est, esd;   // [B,H,n_early,dh] or null
  const int64_t* idx; int64_t isb, ist, isk;      // [B,Lq,K] (ist = 0 for one shared row)
  const void* gate; int gdt; int64_t gsb, gsh, gst, gsm;    // [B,Lq,3] (gsh = 0) or [B,H,Lq,3]
  void* out; int odt; int64_t osb, osh, ost;      // [B,H,Lq,dh], unit channel stride
  int64_t Lq, Lkv, nc, n_early, nb;
  int K, window, n_sink, pool;
  float scale;
};

// LDS tiles: rows of dh without padding, the 16-byte chunks of row r exchanged so that neither
// the staging writes, nor a b128 read of one chunk of 16 consecutive rows (keys), nor a
// transposed b64 read of two chunks of 8 consecutive rows (values) meets a bank twice: NP rows
// of 64 banks hold 4 NP chunks; keys xor the chunk with r / (4 / NP), values with twice that.
// (With rows padded by 8 elements the conflicts were a quarter of the LDS's time.)
template <int NP>
__device__ __forceinline__ constexpr int pf_kswz(int r) { return (r / (4 / NP)) & (4 * NP - 1); }
template <int NP>
__device__ __forceinline__ constexpr int pf_vswz(int r) { return 2 * ((r / (4 / NP)) & (2 * NP - 1)); }

// Bits 4 rb + i of the lane's 16 tile rows j = 16 rb + 4 g + i that lie in [lo, hi]
// (tile-relative, either bound may fall outside [0, 63]).
__device__ __forceinline__ uint32_t pf_range_bits(int lo, int hi, int g) {
  auto lowmask = [](int n) -> uint32_t { return n <= 0 ? 0u : n >= 32 ? 0xffffffffu : (1u << n) - 1u; };
  const uint32_t m0 = lowmask(hi + 1) & ~lowmask(lo);
  const uint32_t m1 = lowmask(hi - 31) & ~lowmask(lo - 32);
  const int sh = 4 * g;
  return ((m0 >> sh) & 0xfu) | (((m0 >> (16 + sh)) & 0xfu) << 4) | (((m1 >> sh) & 0xfu) << 8) |
         (((m1 >> (16 + sh)) & 0xfu) << 12);
}

// Running softmax state of one stream for the lane's query: the reference m (log2 units), the
// sum l of the probabilities (in each element), the values.
template <int NDT>
struct PfAcc {
  float m;
  f32x4 l;
  f32x4 z[NDT];   // O^T[16 dt + 4g + i][query c16]
};

// dh = 32 NP.  FAR: rows 2^24 bytes apart or more, whose offsets take 64 bits.
template <int NP, bool FAR>
__global__ __launch_bounds__(256, NP == 4 ? 2 : 3) void maba_sa_prefill_kernel(PfArgs a) {
  constexpr int DH = 32 * NP;
  constexpr int NDT = DH / 16;
  constexpr int NC = 4 * NP;      // 16-byte chunks per row
  constexpr int RP = 256 / NC;    // rows per staging pass of the workgroup
  constexpr int TE = 64 * DH;
  __shared__ __attribute__((aligned(16))) short s_k[2][TE];
  __shared__ __attribute__((aligned(16))) short s_v[2][TE];
  __shared__ uint32_t s_bits[PF_WORDS];
  __shared__ PfList s_union;
  uint16_t* s_list = s_union.block;
  __shared__ uint32_t s_need[4][PF_LIST / 32];    // per wave: the list entries its queries list
  // Set-up only, in value buffer 1 (first written by the first tile's prefetch, after the
  // set-up's last barrier): the list position of each bitmap word's first block, the list length.
  int* s_wpre = (int*)&s_v[1][0];
  int* s_nlist = s_wpre + PF_WORDS;
  int* s_count = s_nlist + 1;   // some query lists a block twice: slots are counted
  static_assert((PF_WORDS + 2) * 4 <= TE * 2, "set-up tables fit one value buffer");
  // per query, the list entries it lists, behind the entries of a list that short
  uint32_t (*s_qbits)[PF_QWORDS] = s_union.behind.qbits;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, c16 = lane & 15;
  const int64_t b = blockIdx.z;
  const int h = blockIdx.y;
  // the workgroup's first query (< Lq): the last groups see the most keys and start first
  const int64_t tw0 = (int64_t)(gridDim.x - 1 - blockIdx.x) * 64;
  const int64_t tq0 = tw0 + wave * 16;                         // the wave's first query
  const bool qvalid = tq0 + c16 < a.Lq;
  const int64_t tq = qvalid ? tq0 + c16 : a.Lq - 1;            // extra columns repeat the last query
  const int64_t off = a.Lkv - a.Lq;
  const int pos = (int)(off + tq);   // key positions fit 32 bits: Lkv <= PF_WORDS * 32 * 64
  const int64_t wpos_lo = off + tw0;
  // the wave's own first and last position: a tile inside every query's range needs no row masks
  const int vpos_lo = __builtin_amdgcn_readfirstlane((int)(off + min(tq0, a.Lq - 1)));
  const int vpos_hi = __builtin_amdgcn_readfirstlane((int)(off + min(tq0 + 15, a.Lq - 1)));
  const int64_t wpos_hi = off + min(tw0 + 63, a.Lq - 1);

  pf16x8 qb[NP];   // lane (query c16, group g): dims 32 p + 8 g .. +7
#pragma unroll
  for (int p = 0; p < NP; ++p) qb[p] = *(const pf16x8*)(a.q + b * a.qsb + h * a.qsh + tq * a.qst + 32 * p + 8 * g);

  // gate weights of the lane's query
  const int64_t gb = b * a.gsb + h * a.gsh + tq * a.gst;
  float g0 = load_elem(a.gate, a.gdt, gb), g1 = load_elem(a.gate, a.gdt, gb + a.gsm),
        g2 = load_elem(a.gate, a.gdt, gb + 2 * a.gsm);
  {
    const float gm = fmaxf(g0, fmaxf(g1, g2));
    g0 = __expf(g0 - gm); g1 = __expf(g1 - gm); g2 = __expf(g2 - gm);
    const float gi = 1.f / (g0 + g1 + g2);
    g0 *= gi; g1 *= gi; g2 *= gi;
  }
  f32x4 o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- the workgroup's tiles, in stream order: local (sink tiles below the first window
  // tile, then the window tiles of all 64 queries), sparse (the union of the 64 queries'
  // blocks, ascending), HCA (the means any of the 64 queries can see).
  const int64_t ns = min((int64_t)a.n_sink, a.Lkv);
  const int64_t lo = max((int64_t)0, wpos_lo - a.window + 1);
  const int64_t wt0 = (lo / 64) * 64;
  const int64_t sink_end = min(ns, wt0);
  const int n_st = (int)((sink_end + 63) / 64);
  const int n_loc = n_st + (wpos_hi >= wt0 ? (int)((wpos_hi - wt0) / 64 + 1) : 0);

  // this lane's share of its query's index slots, k = g + 4 r, two per register (slot 2 m in
  // the low half): the block, or 0xffff for an empty or out-of-range slot (blocks are below
  // PF_WORDS * 32 = 16384)
  uint32_t myblk[PF_MAXK / 8];
#pragma unroll
  for (int m = 0; m < PF_MAXK / 8; ++m) {
    uint32_t pr = 0u;
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const int kk = g + 4 * (2 * m + hf);
      const int64_t v = kk < a.K ? a.idx[b * a.isb + tq * a.ist + kk * a.isk] : -1;
      pr |= (uint32_t)((v >= 0 && v < a.nb) ? (int)v : 0xffff) << (16 * hf);
    }
    myblk[m] = pr;
  }
  const int64_t nbl = min(a.nb, wpos_hi / 64 + 1);   // blocks that hold a key <= wpos_hi
  const int nwords = (int)((nbl + 31) / 32);
  for (int wd = tid; wd < nwords; wd += 256) s_bits[wd] = 0u;
  __syncthreads();
  if (qvalid) {
#pragma unroll
    for (int r = 0; r < PF_MAXK / 4; ++r) {
      const int bk = (int)((myblk[r >> 1] >> (16 * (r & 1))) & 0xffffu);
      if (bk < nbl) atomicOr(&s_bits[bk >> 5], 1u << (bk & 31));
    }
  }
  __syncthreads();
  if (wave == 0) {   // compaction in ascending block order: word wd's set bits at base + (bits before it)
    int nlist = 0;
    for (int w0 = 0; w0 < nwords; w0 += 64) {
      const int wd = w0 + lane;
      const uint32_t word = wd < nwords ? s_bits[wd] : 0u;
      const int cnt = __popc(word);
      int incl = cnt;
#pragma unroll
      for (int o2 = 1; o2 < 64; o2 <<= 1) {
        const int y = __shfl_up(incl, o2);
        if (lane >= o2) incl += y;
      }
      int at = nlist + incl - cnt;
      if (wd < nwords) s_wpre[wd] = at;
      uint32_t rest = word;
      while (rest) {
        const int bit = __ffs(rest) - 1;
        s_list[at++] = (uint16_t)(wd * 32 + bit);
        rest &= rest - 1;
      }
      nlist += __shfl(incl, 63);
    }
    if (lane == 0) *s_nlist = nlist;
  }
  const int64_t e_hi = min(a.nc - 1, (wpos_hi + 1) / a.pool - 1);
  const int n_hca = e_hi >= 0 ? (int)(e_hi / 64 + 1) : 0;
  for (int wd = tid; wd < 4 * (PF_LIST / 32); wd += 256) (&s_need[0][0])[wd] = 0u;
  if (tid == 0) *s_count = 0;
  __syncthreads();
  const int n_sp = __builtin_amdgcn_readfirstlane(*s_nlist);
  const bool is_short = n_sp <= 32 * PF_QWORDS;
  if (is_short) {
    for (int wd = tid; wd < 64 * PF_QWORDS; wd += 256) (&s_qbits[0][0])[wd] = 0u;
  }
  __syncthreads();
  if (qvalid) {   // mark the list entries of the lane's slots for its wave
#pragma unroll
    for (int r = 0; r < PF_MAXK / 4; ++r) {
      const int bk = (int)((myblk[r >> 1] >> (16 * (r & 1))) & 0xffffu);
      if (bk < nbl) {
        const int u = s_wpre[bk >> 5] + __popc(s_bits[bk >> 5] & ((1u << (bk & 31)) - 1u));
        const uint32_t bit = 1u << (u & 31);
        atomicOr(&s_need[wave][u >> 5], bit);
        if (is_short && (atomicOr(&s_qbits[16 * wave + c16][u >> 5], bit) & bit)) *s_count = 1;
      }
    }
  }
  __syncthreads();
  const bool by_bits = is_short && *s_count == 0;
  const int n_ls = n_loc + n_sp;
  const int nt = n_ls + n_hca;

  // ---- tile staging: thread tid copies chunk tid % NC of rows tid / NC + RP p of the key and
  // value tiles; the next tile's loads are in flight while the current one computes.  Tile
  // bases are uniform, a lane adds its byte offset, its row clamped to the last one (such rows
  // are masked).
  const uint16_t* kbase = a.k + b * a.ksb + h * a.ksh;
  const uint16_t* vbase = a.v + b * a.vsb + h * a.vsh;
  const uint16_t* khbase = a.kh ? a.kh + b * a.khb + h * a.khh : nullptr;
  const uint16_t* vhbase = a.vh ? a.vh + b * a.vhb + h * a.vhh : nullptr;
  const int srow = tid / NC, sch = tid % NC;
  short* kw = &s_k[0][0] + (srow * NC + (sch ^ pf_kswz<NP>(srow))) * 8;
  short* vw = &s_v[0][0] + (srow * NC + (sch ^ pf_vswz<NP>(srow))) * 8;
  pf16x8 pk[NP], pv[NP];
  auto fetch = [&](int i) {
    const uint16_t* kr;
    const uint16_t* vr;
    int64_t ks, vs;
    int last;
    if (i < n_ls) {
      const int64_t tb = i < n_st ? 64 * (int64_t)i
                       : i < n_loc ? wt0 + 64 * (int64_t)(i - n_st)
                                   : 64 * (int64_t)__builtin_amdgcn_readfirstlane((int)s_list[i - n_loc]);
      kr = kbase + tb * a.kst;
      vr = vbase + tb * a.vst;
      ks = a.kst; vs = a.vst;
      last = (int)min(a.Lkv - 1 - tb, (int64_t)63);
    } else {
      const int64_t e0 = 64 * (int64_t)(i - n_ls);
      kr = khbase + e0 * a.khe;
      vr = vhbase + e0 * a.vhe;
      ks = a.khe; vs = a.vhe;
      last = (int)min(a.nc - 1 - e0, (int64_t)63);
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int r = min(srow + RP * p, last);
      if constexpr (FAR) {
        pk[p] = *(const pf16x8*)(kr + r * ks + 8 * sch);
        pv[p] = *(const pf16x8*)(vr + r * vs + 8 * sch);
      } else {
        pk[p] = *(const pf16x8*)((const char*)kr + (__umul24(r, (uint32_t)ks * 2u) + 16u * sch));
        pv[p] = *(const pf16x8*)((const char*)vr + (__umul24(r, (uint32_t)vs * 2u) + 16u * sch));
      }
    }
  };
  auto stash = [&](int buf) {   // pf_kswz and pf_vswz repeat every RP rows
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      *(pf16x8*)(kw + buf * TE + RP * p * DH) = pk[p];
      *(pf16x8*)(vw + buf * TE + RP * p * DH) = pv[p];
    }
  };
  // the lane's read addresses: key rows 16 rb + c16, chunk 4 p + g; value rows
  // 16 rb + 4 g + c16 / 4, columns 16 dt + 4 (c16 % 4) .. (transposed: the lane receives column
  // c16 of rows 4 g .. 4 g + 3)
  const short* kl[NP];
  const short* vl[NDT];
#pragma unroll
  for (int p = 0; p < NP; ++p) kl[p] = &s_k[0][0] + (c16 * NC + ((4 * p + g) ^ pf_kswz<NP>(c16))) * 8;
  {
    const int r = 4 * g + (c16 >> 2);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
      vl[dt] = &s_v[0][0] + (r * NC + ((2 * dt + ((c16 >> 1) & 1)) ^ pf_vswz<NP>(r))) * 8 + 4 * (c16 & 1);
  }
  auto vT = [](const short* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) pf16x4*)p);
  };

  // One 64-key tile from LDS buffer buf: the lane's rows with bit 4 rb + i of vmask set
  // (row 16 rb + 4 g + i) have weight 2^lw, the others 0 (lw = -inf: all of them).  A wave none
  // of whose queries weights any row skips the tile: for such a lane the tile would leave its
  // state exactly as it is.  Scores are taken in log2 units (scale * log2 e); rows are masked one
  // by one only where some lane weights a part of the tile.
  const float sl2 = a.scale * 1.4426950408889634f;
  auto tile = [&](PfAcc<NDT>& st, int buf, float lw, uint32_t vmask) {
    if (!qvalid || lw == -INFINITY) vmask = 0u;
    if (vmask == 0u) lw = -INFINITY;
    if (__ballot(vmask != 0u) == 0ull) return;   // wave-uniform
    const bool part = __ballot(vmask != 0u && vmask != 0xffffu) != 0ull;
    f32x4 sc[4], x[4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const pf16x8 kv = *(const pf16x8*)(kl[p] + buf * TE + 16 * rb * DH);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kv),
                                                      __builtin_bit_cast(bf16x8, qb[p]), acc, 0, 0, 0);
      }
      sc[rb] = acc;
    }
    // lane (query c16, g) holds the scores of keys 16 rb + 4 g + i; x: relative to the reference
    auto drop = [&]() {   // the rows without weight, one by one
      uint32_t vm = vmask;
      asm volatile("" : "+v"(vm));   // the bit tests stay in the callers' branches
#pragma unroll
      for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int i = 0; i < 4; ++i) x[rb][i] = ((vm >> (4 * rb + i)) & 1u) ? x[rb][i] : -INFINITY;
    };
    auto relative = [&]() {
      const float bias = lw == -INFINITY ? -INFINITY : st.m == -INFINITY ? lw : lw - st.m;
#pragma unroll
      for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int i = 0; i < 4; ++i) x[rb][i] = fmaf(sc[rb][i], sl2, bias);
      if (part) drop();
    };
    auto largest = [&](auto max2) {
      float mx = -INFINITY;
#pragma unroll
      for (int rb = 0; rb < 4; ++rb)
        mx = max2(max2(max2(max2(mx, x[rb][0]), x[rb][1]), x[rb][2]), x[rb][3]);
      return mx;
    };
    relative();
    float mx = largest([](float p, float q) { return __builtin_elementwise_maximum(p, q); });   // NaN if any x is
    if (__ballot(!(mx <= PF_SLACK) || (st.m == -INFINITY && lw != -INFINITY)) != 0ull) {
      // Some query's reference moves: to the largest score so far, in all of its lanes.  Or a score
      // is NaN: of a query that weights the row, whose result it is, or an infinity (or NaN) that the
      // bias of -inf did not take away from the other queries, which the rows' masks then do.
      const bool nan = __ballot(mx != mx) != 0ull;
      if (nan) {
        drop();
        mx = largest([](float p, float q) { return fmaxf(p, q); });   // a NaN moves no reference
      }
      const float base = st.m == -INFINITY ? 0.f : st.m;
      float top = lw == -INFINITY ? -INFINITY : mx - lw + base;
      top = group_max(top);
      const float m_new = fmaxf(st.m, top);
      if (__ballot(st.l[0] != 0.f) != 0ull) {   // not at a stream's first tile: there is no sum yet
        const float corr = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(st.m - m_new);
        st.l *= corr;   // every element is the query's sum
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) st.z[dt] *= corr;
      }
      st.m = m_new;
      relative();
      if (nan) drop();
    }
    i16x4 ph[4], pl[4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      f32x4 pe;
#pragma unroll
      for (int i = 0; i < 4; ++i) pe[i] = __builtin_amdgcn_exp2f(x[rb][i]);   // exp2(-inf) = 0 for masked keys
      split4(pe, ph[rb], pl[rb]);
    }
    // l += the probabilities' sum, as a product with a row of ones
    {
      const short one = 0x3f80;
      const pf16x8 ones = {one, one, one, one, one, one, one, one};
#pragma unroll
      for (int p2 = 0; p2 < 2; ++p2) {
        st.l = mma32(st.l, ones, cat8(ph[2 * p2], ph[2 * p2 + 1]));
        st.l = mma32(st.l, ones, cat8(pl[2 * p2], pl[2 * p2 + 1]));
      }
    }
    // O^T[dim][query] += V^T P over the 64 keys as two 32-key steps whose key order
    // (16 rb + 4 g + i, rb in {2 p2, 2 p2 + 1}) matches the probabilities this lane holds
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      f32x4 acc = st.z[dt];
#pragma unroll
      for (int p2 = 0; p2 < 2; ++p2) {
        const pf16x4 a0 = vT(vl[dt] + buf * TE + 32 * p2 * DH);
        const pf16x4 a1 = vT(vl[dt] + buf * TE + (32 * p2 + 16) * DH);
        const pf16x8 av = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
        const i16x8 bh = cat8(ph[2 * p2], ph[2 * p2 + 1]), bl = cat8(pl[2 * p2], pl[2 * p2 + 1]);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), __builtin_bit_cast(bf16x8, bh),
                                                      acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), __builtin_bit_cast(bf16x8, bl),
                                                      acc, 0, 0, 0);
      }
      st.z[dt] = acc;
    }
  };
  auto reset = [&](PfAcc<NDT>& st) {
    st.m = -INFINITY;
    st.l = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) st.z[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto fold = [&](const PfAcc<NDT>& st, float gs) {   // o += g_s z_s / l_s
    const float w = st.l[0] > 0.f ? gs / st.l[0] : 0.f;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[dt] += st.z[dt] * w;
  };
  // tiles [i, i_end): prefetch tile i + 1 (of whichever stream), compute tile i, stage the
  // prefetched tile into the other buffer, one barrier per tile.  weight_of(i) gives the log2 of
  // tile i's weight for the lane's query and mask_of(i) its row mask (pf_range_bits).
  int i = 0;
  auto run = [&](PfAcc<NDT>& st, int i_end, auto weight_of, auto mask_of) {
    for (; i < i_end; ++i) {
      if (i + 1 < nt) fetch(i + 1);
      const float lw = weight_of(i);
      tile(st, i & 1, lw, lw != -INFINITY ? mask_of(i) : 0u);
      if (i + 1 < nt) stash((i + 1) & 1);
      __syncthreads();
    }
  };
  if (nt > 0) {
    fetch(0);
    stash(0);
  }
  __syncthreads();
  PfAcc<NDT> st;

  // ---- local stream: sink tiles hold keys [0, min(sink_end, pos + 1)); window tiles the keys
  // in (pos - window, pos] and the sinks below min(ns, pos + 1)
  reset(st);
  run(st, n_loc, [](int) { return 0.f; }, [&](int ti) {
    if (ti < n_st) return pf_range_bits(-64 * ti, min((int)sink_end - 1, pos) - 64 * ti, g);
    const int tb = (int)wt0 + 64 * (ti - n_st);
    if (tb + 63 <= vpos_lo && tb > vpos_hi - a.window) return 0xffffu;
    return pf_range_bits(pos - a.window + 1 - tb, pos - tb, g) |
           pf_range_bits(-tb, min((int)ns - 1, pos) - tb, g);
  });
  fold(st, g0);

  // ---- sparse stream: each key weighted by how often the lane's query lists its block; a
  // wave skips the entries none of its queries lists
  reset(st);
  uint32_t word = 0u;
  run(st, n_ls, [&](int ti) {
    const int u = ti - n_loc;
    if (by_bits) {
      if ((u & 31) == 0) word = s_qbits[16 * wave + c16][u >> 5];
      return ((word >> (u & 31)) & 1u) ? 0.f : -INFINITY;
    }
    if (((s_need[wave][u >> 5] >> (u & 31)) & 1u) == 0u) return -INFINITY;   // wave-uniform
    const int blk = s_list[u];
    int cnt = 0;
#pragma unroll
    for (int m = 0; m < PF_MAXK / 8; ++m)
      cnt += (int)((myblk[m] & 0xffffu) == (uint32_t)blk) + (int)((myblk[m] >> 16) == (uint32_t)blk);
    cnt += __shfl_xor(cnt, 16);
    cnt += __shfl_xor(cnt, 32);
    return cnt > 0 ? __builtin_amdgcn_logf((float)cnt) : -INFINITY;
  }, [&](int ti) {
    const int tb = 64 * __builtin_amdgcn_readfirstlane((int)s_list[ti - n_loc]);
    return tb + 63 <= vpos_lo ? 0xffffu : pf_range_bits(0, pos - tb, g);
  });
  fold(st, g1);

  // ---- HCA stream: means e <= e_max, the last complete block's mean before the lane's query;
  // early queries take their row
  reset(st);
  const int e_max = (int)min(a.nc - 1, (int64_t)((pos + 1) / a.pool) - 1);
  const int ve_max = (int)min(a.nc - 1, (int64_t)((vpos_lo + 1) / a.pool) - 1);
  run(st, nt, [](int) { return 0.f; }, [&](int ti) {
    const int e0 = 64 * (ti - n_ls);
    return e0 + 63 <= ve_max ? 0xffffu : pf_range_bits(0, e_max - e0, g);
  });
  if (pos < a.pool - 1) {   // running mean of c[0..pos] through W_v (the caller's row)
    const bool have = a.early && tq < a.n_early;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i2 = 0; i2 < 4; ++i2) {
        const int d = 16 * dt + 4 * g + i2;
        const float x = have ? load_elem(a.early, a.edt, b * a.esb + h * a.esh + tq * a.est + d * a.esd) : 0.f;
        o[dt][i2] += g2 * x;
      }
  } else {
    fold(st, g2);
  }

  if (!qvalid) return;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
    const int64_t oo = b * a.osb + h * a.osh + tq * a.ost + 16 * dt + 4 * g;
    if (a.odt == MABA_F32) {
      *(f32x4*)((float*)a.out + oo) = o[dt];
    } else {
      uint2 u;
      u.x = (uint32_t)f32_to_bf16_bits(o[dt][0]) | ((uint32_t)f32_to_bf16_bits(o[dt][1]) << 16);
      u.y = (uint32_t)f32_to_bf16_bits(o[dt][2]) | ((uint32_t)f32_to_bf16_bits(o[dt][3]) << 16);
      *(uint2*)((uint16_t*)a.out + oo) = u;
    }
  }
}

// How many distinct blocks each 16 consecutive queries list, summed per workgroup: what the choice
// between this kernel and the latent one goes by.  A wave takes 16 queries at a time and marks
// their slots in its LDS bitmap; the lane that sets a bit counts it, and afterwards the words it
// touched are cleared.  Latency-bound: 10 us for the 6.3 MB of indices at T=24571 K=32 (a segmented
// sort of the 16 K slots 48 us, beside the compare of neighbours, its sum and their mean).
struct PfUnionArgs {
  const int64_t* idx; int64_t isb, ist, isk;
  int32_t* out;                       // one count per workgroup
  int64_t gpb, groups;                // 16-query groups per batch element, in all
  int K;
};

__global__ __launch_bounds__(256) void prefill_union_kernel(PfUnionArgs a) {
  __shared__ uint32_t s_bits[4][PF_WORDS + 1];   // the last word: indices that are no block
  __shared__ int s_sum[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t* bits = s_bits[wave];
  for (int w = lane; w <= PF_WORDS; w += 64) bits[w] = 0u;
  __syncthreads();
  int n = 0;
  const int slots = 16 * a.K;
  for (int64_t gi = (int64_t)blockIdx.x * 4 + wave; gi < a.groups; gi += (int64_t)gridDim.x * 4) {
    const int64_t base = (gi / a.gpb) * a.isb + (gi % a.gpb) * 16 * a.ist;
    int blk[PF_MAXK / 4];
#pragma unroll
    for (int r = 0; r < PF_MAXK / 4; ++r) {   // all loads in flight
      const int sl = lane + 64 * r;
      const int64_t v = sl < slots ? a.idx[base + (sl / a.K) * a.ist + (sl % a.K) * a.isk] : -1;
      blk[r] = sl >= slots ? -1 : v >= 0 && v < PF_WORDS * 32 ? (int)v : PF_WORDS * 32;
    }
#pragma unroll
    for (int r = 0; r < PF_MAXK / 4; ++r)
      if (blk[r] >= 0) n += (atomicOr(&bits[blk[r] >> 5], 1u << (blk[r] & 31)) >> (blk[r] & 31) & 1u) == 0u;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < PF_MAXK / 4; ++r)   // after every mark: a wave's LDS operations stay in order
      if (blk[r] >= 0) bits[blk[r] >> 5] = 0u;
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
  if (lane == 0) s_sum[wave] = n;
  __syncthreads();
  if (threadIdx.x == 0) a.out[blockIdx.x] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
}

static bool pf_rows_ok(const maba_tensor* t, int64_t B, int64_t H, int64_t n, int64_t dh) {
  if (!t || t->ndim != 4 || t->dtype != MABA_BF16) return false;
  if (t->shape[0] != B || t->shape[1] != H || t->shape[2] != n || t->shape[3] != dh) return false;
  if (t->stride[3] != 1 || (uintptr_t)t->data % 16 != 0) return false;
  for (int d = 0; d < 3; ++d)
    if (t->shape[d] > 1 && t->stride[d] % 8 != 0) return false;
  return true;
}

}  // namespace maba

using namespace maba;

extern "C" int maba_hip_maba_sa_prefill(const maba_tensor* q, const maba_tensor* k, const maba_tensor* v,
                                        const maba_tensor* kh, const maba_tensor* vh,
                                        const maba_tensor* early, const maba_tensor* idx,
                                        const maba_tensor* gate, float scale, int window, int n_sink,
                                        int block_size, int pool, maba_tensor* out, void* stream) {
  if (!q || q->ndim != 4) return fail(MABA_ERR_INVALID, "maba_sa_prefill: q must be [B,H,Lq,dh]");
  const int64_t B = q->shape[0], H = q->shape[1], Lq = q->shape[2], dh = q->shape[3];
  if (!k || k->ndim != 4 || !v || v->ndim != 4)
    return fail(MABA_ERR_INVALID, "maba_sa_prefill: k and v must be [B,H,Lkv,dh]");
  const int64_t Lkv = k->shape[2];
  if (Lq > Lkv) return fail(MABA_ERR_INVALID, "maba_sa_prefill: more queries than keys");
  if (window < 0 || n_sink < 0 || pool <= 0) return fail(MABA_ERR_INVALID, "maba_sa_prefill: bad window/sink/pool");
  if (block_size != 64) return fail(MABA_ERR_UNSUPPORTED, "maba_sa_prefill: block_size 64 only");
  if (dh != 32 && dh != 64 && dh != 128) return fail(MABA_ERR_UNSUPPORTED, "maba_sa_prefill: dh in {32, 64, 128}");
  if (!pf_rows_ok(q, B, H, Lq, dh) || !pf_rows_ok(k, B, H, Lkv, dh) || !pf_rows_ok(v, B, H, Lkv, dh))
    return fail(MABA_ERR_UNSUPPORTED, "maba_sa_prefill: q, k, v must be bf16 with unit channel stride and "
                "16-byte aligned rows");
  const int64_t nc = Lkv / pool;
  if (nc > 0 && (!pf_rows_ok(kh, B, H, nc, dh) || !pf_rows_ok(vh, B, H, nc, dh)))
    return fail(MABA_ERR_UNSUPPORTED, "maba_sa_prefill: kh, vh must be bf16 [B,H,Lkv/pool,dh], unit channel stride");
  const int64_t off = Lkv - Lq;
  const int64_t n_early = off < pool - 1 ? std::min(Lq, (int64_t)(pool - 1) - off) : 0;
  if (n_early > 0) {
    const int64_t se[4] = {B, H, n_early, dh};
    if (!expect_shape(early, "early", 4, se) || !expect_float(early, "early")) return MABA_ERR_INVALID;
  }
  if (!idx || idx->ndim != 3 || idx->shape[0] != B || (idx->shape[1] != Lq && idx->shape[1] != 1))
    return fail(MABA_ERR_INVALID, "maba_sa_prefill: idx must be [B,Lq|1,K]");
  if (idx->dtype != MABA_I64) return fail(MABA_ERR_DTYPE, "maba_sa_prefill: idx must be int64");
  const int64_t K = idx->shape[2];
  if (K > PF_MAXK) return fail(MABA_ERR_UNSUPPORTED, "maba_sa_prefill: at most %d index slots", PF_MAXK);
  const int64_t nb = (Lkv + 63) / 64;
  if (nb > (int64_t)PF_WORDS * 32) return fail(MABA_ERR_UNSUPPORTED, "maba_sa_prefill: Lkv up to %d", PF_WORDS * 32 * 64);
  if (!gate || !((gate->ndim == 3 && gate->shape[0] == B && gate->shape[1] == Lq && gate->shape[2] == 3) ||
                 (gate->ndim == 4 && gate->shape[0] == B && gate->shape[1] == H && gate->shape[2] == Lq &&
                  gate->shape[3] == 3)))
    return fail(MABA_ERR_INVALID, "maba_sa_prefill: gate must be [B,Lq,3] or [B,H,Lq,3]");
  if (!expect_float(gate, "gate")) return MABA_ERR_DTYPE;
  const int64_t so[4] = {B, H, Lq, dh};
  if (!expect_shape(out, "out", 4, so)) return MABA_ERR_INVALID;
  if ((out->dtype != MABA_F32 && out->dtype != MABA_BF16) || out->stride[3] != 1 ||
      (uintptr_t)out->data % 16 != 0 || out->stride[0] % 4 != 0 || out->stride[1] % 4 != 0 ||
      out->stride[2] % 4 != 0)
    return fail(MABA_ERR_UNSUPPORTED, "maba_sa_prefill: out must be f32/bf16 with unit channel stride");
  if (B * H * Lq == 0) return MABA_OK;
  PfArgs a;
  a.q = (const uint16_t*)q->data; a.qsb = q->stride[0]; a.qsh = q->stride[1]; a.qst = q->stride[2];
  a.k = (const uint16_t*)k->data; a.ksb = k->stride[0]; a.ksh = k->stride[1]; a.kst = k->stride[2];
  a.v = (const uint16_t*)v->data; a.vsb = v->stride[0]; a.vsh = v->stride[1]; a.vst = v->stride[2];
  a.kh = nc > 0 ? (const uint16_t*)kh->data : nullptr;
  a.khb = nc > 0 ? kh->stride[0] : 0; a.khh = nc > 0 ? kh->stride[1] : 0; a.khe = nc > 0 ? kh->stride[2] : 0;
  a.vh = nc > 0 ? (const uint16_t*)vh->data : nullptr;
  a.vhb = nc > 0 ? vh->stride[0] : 0; a.vhh = nc > 0 ? vh->stride[1] : 0; a.vhe = nc > 0 ? vh->stride[2] : 0;
  a.early = n_early > 0 ? early->data : nullptr; a.edt = n_early > 0 ? early->dtype : MABA_F32;
  a.esb = n_early > 0 ? early->stride[0] : 0; a.esh = n_early > 0 ? early->stride[1] : 0;
  a.est = n_early > 0 ? early->stride[2] : 0; a.esd = n_early > 0 ? early->stride[3] : 0;
  a.idx = (const int64_t*)idx->data; a.isb = idx->stride[0];
  a.ist = idx->shape[1] == 1 ? 0 : idx->stride[1]; a.isk = idx->stride[2];
  a.gate = gate->data; a.gdt = gate->dtype; a.gsb = gate->stride[0];
  if (gate->ndim == 3) { a.gsh = 0; a.gst = gate->stride[1]; a.gsm = gate->stride[2]; }
  else { a.gsh = gate->stride[1]; a.gst = gate->stride[2]; a.gsm = gate->stride[3]; }
  a.out = out->data; a.odt = out->dtype; a.osb = out->stride[0]; a.osh = out->stride[1]; a.ost = out->stride[2];
  a.Lq = Lq; a.Lkv = Lkv; a.nc = nc; a.n_early = n_early; a.nb = nb;
  a.K = (int)K; a.window = window; a.n_sink = n_sink; a.pool = pool; a.scale = scale;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)ceil_div(Lq, 64), (unsigned)H, (unsigned)B);
  auto far = [](int64_t st) { return st < 0 || st >= (1 << 23); };   // elements
  auto launch = [&](auto far_c) {
    constexpr bool FAR = decltype(far_c)::value;
    switch (dh) {
      case 32: hipLaunchKernelGGL((maba_sa_prefill_kernel<1, FAR>), grid, dim3(256), 0, s, a); break;
      case 64: hipLaunchKernelGGL((maba_sa_prefill_kernel<2, FAR>), grid, dim3(256), 0, s, a); break;
      default: hipLaunchKernelGGL((maba_sa_prefill_kernel<4, FAR>), grid, dim3(256), 0, s, a); break;
    }
  };
  if (far(a.kst) || far(a.vst) || far(a.khe) || far(a.vhe)) launch(std::true_type{});
  else launch(std::false_type{});
  return check_launch("maba_sa_prefill");
}

extern "C" int maba_hip_prefill_union(const maba_tensor* idx, maba_tensor* out, void* stream) {
  if (!idx || idx->ndim != 3) return fail(MABA_ERR_INVALID, "prefill_union: idx must be [B,Lq,K]");
  if (!out || out->ndim != 1) return fail(MABA_ERR_INVALID, "prefill_union: out must be 1D");
  if (idx->dtype != MABA_I64 || out->dtype != MABA_I32)
    return fail(MABA_ERR_DTYPE, "prefill_union: idx must be int64 and out int32");
  const int64_t B = idx->shape[0], Lq = idx->shape[1], K = idx->shape[2], n = out->shape[0];
  if (K < 1 || K > PF_MAXK) return fail(MABA_ERR_UNSUPPORTED, "prefill_union: 1 to %d index slots", PF_MAXK);
  if (n < 1 || n > 65535 || (n > 1 && out->stride[0] != 1))
    return fail(MABA_ERR_INVALID, "prefill_union: out must hold 1 to 65535 contiguous counts");
  PfUnionArgs a;
  a.idx = (const int64_t*)idx->data; a.isb = idx->stride[0]; a.ist = idx->stride[1]; a.isk = idx->stride[2];
  a.out = (int32_t*)out->data;
  a.gpb = Lq / 16; a.groups = B * a.gpb; a.K = (int)K;
  hipLaunchKernelGGL(prefill_union_kernel, dim3((unsigned)n), dim3(256), 0, (hipStream_t)stream, a);
  return check_launch("prefill_union");
}
