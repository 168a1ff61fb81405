// Host side of the sub-chunk DGDA prefill for per-channel gates (kernels and their math
// in dgda_sub.h): operand checks, workspace sizing, the d_v = 128 split, the kernels for
// d_k = 64 and the fused layer prologue entry point (maba_hip_dgda_layer_prefill).
#include "dgda_sub.h"

#include <algorithm>

namespace maba {

// ------------------------------------------------------------------ host side

static bool al16s(const void* p) { return ((uintptr_t)p & 15) == 0; }
static bool fits32s(const maba_tensor* t) {
  for (int d = 0; d < t->ndim; ++d)
    if (t->stride[d] < 0 || t->stride[d] > INT32_MAX) return false;
  return true;
}
// the kernels address the 16 rows of a sub-chunk with 32-bit byte offsets (row_end)
static bool rows_fit(int64_t row_stride) { return row_stride <= (INT32_MAX - 4096) / (SC * 4); }
// gate with channel stride 0 (per token) or 1 (per channel, 16-byte aligned rows), fp32 or
// (16-bit q, k, v) in q's dtype
static bool sub_gate_ok(const maba_tensor* t, int gdt) {
  if (!t || t->dtype != gdt || !fits32s(t) || !rows_fit(t->stride[2])) return false;
  if (t->stride[3] == 0) return true;
  if (t->stride[3] != 1 || !al16s(t->data)) return false;
  for (int d = 0; d < 3; ++d)
    if (t->shape[d] > 1 && t->stride[d] % 4 != 0) return false;
  return true;
}

static bool sub_head_size(int64_t d) { return d == 32 || d == 64 || d == 128; }
static bool sub_io_dtype(int dt) { return dt == MABA_BF16 || dt == MABA_F16 || dt == MABA_F32; }

bool dgda_sub_supported(const maba_tensor* q, const maba_tensor* k, const maba_tensor* v,
                        const maba_tensor* gate, const maba_tensor* b, const maba_tensor* w,
                        const maba_tensor* out) {
  if (!q || !k || !v || !gate || !b) return false;
  if (!sub_head_size(q->shape[3]) || !sub_head_size(v->shape[3])) return false;
  const int dt = q->dtype;
  if (!sub_io_dtype(dt) || k->dtype != dt || v->dtype != dt) return false;
  for (const maba_tensor* t : {q, k, v}) {   // 4-element (8- or 16-byte) loads
    if (t->stride[3] != 1 || !al16s(t->data) || !fits32s(t) || !rows_fit(t->stride[2])) return false;
    for (int d = 0; d < 3; ++d)
      if (t->shape[d] > 1 && t->stride[d] % 4 != 0) return false;
  }
  // the three gates share one dtype: fp32, or q's 16-bit dtype
  const int gdt = gate->dtype;
  if (gdt != MABA_F32 && (gdt != dt || dt == MABA_F32)) return false;
  if (!sub_gate_ok(gate, gdt) || !sub_gate_ok(b, gdt)) return false;
  if (w && !sub_gate_ok(w, gdt)) return false;
  if (out && (out->stride[3] != 1 || !fits32s(out) || !sub_io_dtype(out->dtype))) return false;
  return q->shape[2] <= ((int64_t)1 << 30);
}

// ---- segments per sequence
// Sub-chunks per segment at least.  Shorter ones no longer gain: a segment's end costs a step
// of the scan where transitions survive (0.7 us against 4.6 us per sub-chunk twice), and where
// they vanish it costs up to their 3 to 10 sub-chunks again.  At 16, 8, 6, 5, 4, 3: B=1 H=10 T=2048
// fp32 69, 49, 45, 46, 48, 83 us; decay that remembers, T=4096 bf16 129, 98, 103, 105, 112, 125.
constexpr int64_t SUB_MIN_LEN = 5;
// Sub-chunks per segment from which two waves per SIMD pay: the second wave gains a little (B=4
// H=10 T=32768 per-channel bf16: 436 us against 445), and twice as many segments cost their re-runs
// (the fused layer at B=1 T=32768, 10 sub-chunks each: 283 us against 208).
constexpr int64_t SUB_LEN_2 = 32;
// Segments per sequence at most.  Where transitions survive the scan takes a step per segment (0.7 us
// at d_k = 64, 4 at 128, 0.4 at 32), and every sub-chunk is run twice, so few heads over a long sequence
// are not cut until every SIMD has a wave: with these bounds no decay is slower than in segments of 64
// sub-chunks on four waves each.  One head, four waves / 6 sqrt(sub-chunks) segments / these bounds, us,
// log-decay per token 2.1 (and 0.2, 0.01): d_k = 64 T=32768 232 / 51 / 59 (402 / 337 / 236, 663 / 336 / 236),
// T=131072 233 / 95 / 158 (403 / 570 / 245, 926 / 570 / 445); d_k = 128 T=65536 880 / 136 / 255 (1685 /
// 1495 / 397, 4015 / 1495 / 770); the fused layer T=65536 344 / 94 / 137 (571 / 447 / 367, 926 / 446 / 367).
static int64_t seg_most(int64_t dk) { return dk == 128 ? 96 : dk == 64 ? 192 : 256; }
// A short sequence stays whole where cutting it does not pay if its transitions survive: every
// sub-chunk is run twice, on SIMDs that segments and transitions share once these are more than
// half as many as the SIMDs (below that segments always paid), and joining them takes as long as
// SUB_ENDS sub-chunks.  B H = 160, T=200, cut into three / whole, us, decay that remembers (and that
// vanishes): 67 / 50 (53 / 50); BH = 320, T=320 110 / 76 (73 / 76), T=500 154 / 117 (90 / 117); d_k =
// 128, d_v = 64, BH = 160, T=170 101 / 61 (fp32).  At d_k = 32 a sub-chunk takes 2.2 us and the three
// launches of a cut call 34 us of the host's time: T=170 35 / 30.  d_k = d_v = 128 always gained.
// Beyond SUB_SHORT sub-chunks the segments of vanishing transitions gain more than that.
constexpr int64_t SUB_SHORT = 64;
constexpr int SUB_ENDS = 8, SUB_ENDS_32 = 5;

static int64_t sub_chunks(int64_t L) { return ceil_div(L, SC); }
static size_t sub_slot_bytes(int64_t dk, int64_t dv) { return (size_t)(dk * (dv + dk)) * sizeof(float) + 2 * sizeof(int); }

// How a call is cut: nseg segments of seglen sub-chunks, cols value columns per wave.
struct SubCut { int nseg, seglen, cols; };

// As many segments as fill one wave per SIMD, or two (see SUB_LEN_2; always at d_k = 32, whose
// waves hold a quarter of the state, never at d_k = 128, whose state leaves registers for one),
// no more than a scan should walk (seg_most), and no more than the workspace holds.  Where that
// leaves half the SIMDs without work a wave takes 32 columns instead of 64 (narrow): the key side is
// done twice, but a sub-chunk takes a wave less time (B=2 H=10 bf16: T=160 41 -> 34 us, T=1000 45 ->
// 44 us; the fused layer at H=10, T=100 49 -> 42 us, T=160 64 -> 55, T=1000 83 -> 72).
static SubCut sub_cut(int64_t BH, int64_t L, int64_t dk, int64_t dv, size_t ws_bytes, bool narrow) {
  const int64_t nch = sub_chunks(L);
  const int64_t simds = 4 * (int64_t)device_cu_count();
  const int64_t waves = (BH > 0 ? BH : 1) * (dv == 128 ? 2 : 1);
  const bool two = dk == 32 || (dk == 64 && nch * waves >= SUB_LEN_2 * 2 * simds);
  int64_t n = (two ? 2 : 1) * simds / waves;
  if (n > ceil_div(nch, SUB_MIN_LEN)) n = ceil_div(nch, SUB_MIN_LEN);
  if (n > seg_most(dk)) n = seg_most(dk);
  const int64_t fit = (int64_t)(ws_bytes / ((size_t)(BH > 0 ? BH : 1) * sub_slot_bytes(dk, dv)));
  if (n > fit) n = fit;
  static_assert(SUB_MAX_SEG >= 256, "the scan's table holds seg_most");
  // two short segments take no less time one after the other (the second's re-run) than one
  if (n < 2 || (n == 2 && nch < 4 * SUB_MIN_LEN)) n = 1;
  auto cut = [&](int64_t n) {
    const int64_t len = nch > 0 ? ceil_div(nch, n) : 0;
    SubCut c;
    c.seglen = (int)len;
    c.nseg = len > 0 ? (int)ceil_div(nch, len) : 1;
    c.cols = dv == 32 || (narrow && 2 * waves * c.nseg <= simds) ? 32 : 64;
    return c;
  };
  const SubCut c = cut(n);
  if (c.nseg > 1 && nch <= SUB_SHORT && (dk < 128 || dv < 128)) {
    // the first launch's waves: 32 or 64 output columns each, 64 columns of a transition
    const int64_t main = waves * (c.cols < dv ? 64 / c.cols : 1) * c.nseg + BH * (c.nseg - 1) * (dk == 128 ? 2 : 1);
    const double share = std::max(1.0, (double)main / (dk == 32 ? 2 * simds : simds));
    if ((dk == 32 || 2 * main > simds) && 2 * c.seglen * share + (dk == 32 ? SUB_ENDS_32 : SUB_ENDS) > nch) return cut(1);
  }
  return c;
}

// The size the query promises to be enough; what fits in it, sub_cut works out.
size_t dgda_sub_workspace(int64_t BH, int64_t L, int64_t dk, int64_t dv) {
  const SlotGeom gm = slot_geom(BH, sub_chunks(L) > 0 ? sub_chunks(L) : 1, 64, device_cu_count());
  if (gm.nseg_max <= 1) return 16;
  const int64_t dvc = dv == 128 ? 64 : dv;
  return (size_t)(BH * gm.nseg_max * dk * (dvc + dk)) * sizeof(float) + (size_t)(BH * gm.nseg_max) * sizeof(int);
}

// The size with which a call is cut as finely as pays.
size_t dgda_sub_workspace_preferred(int64_t BH, int64_t L, int64_t dk, int64_t dv) {
  const SubCut c = sub_cut(BH, L, dk, dv, SIZE_MAX, true);
  return c.nseg == 1 ? 16 : (size_t)(BH * c.nseg) * sub_slot_bytes(dk, dv);
}

// Returns the columns per wave.
static int sub_place(SubArgs& a, int64_t BH, int64_t L, int64_t dk, int64_t dv, void* ws, size_t ws_bytes, bool narrow) {
  const SubCut c = sub_cut(BH, L, dk, dv, ws_bytes, narrow);
  a.nseg = c.nseg;
  a.seglen = c.seglen;
  a.nchunks = (int)sub_chunks(L);
  a.nvh = (int)(dv / c.cols);
  a.dvt = (int)dv;
  a.agg = (float*)ws;
  a.zc = (int*)(a.agg + BH * a.nseg * dk * (dv + dk));
  return c.cols;
}

// No byte of the new history belongs to the old one.
static bool histories_apart(const maba_tensor* const* hist, maba_tensor* const* new_hist) {
  auto range = [](const maba_tensor* t, uintptr_t& lo, uintptr_t& hi) {
    lo = hi = (uintptr_t)t->data;
    for (int d = 0; d < 3; ++d) {
      const int64_t span = (t->shape[d] - 1) * t->stride[d] * (t->dtype == MABA_F32 ? 4 : 2);
      (span < 0 ? lo : hi) += span;
    }
    hi += 4;
  };
  for (int s = 0; s < 3; ++s)
    for (int n = 0; n < 3; ++n) {
      uintptr_t l0, h0, l1, h1;
      range(hist[s], l0, h0);
      range(new_hist[n], l1, h1);
      if (l0 < h1 && l1 < h0) return false;
    }
  return true;
}

// One vector store per lane and token: aligned rows.
static int sub_out_vec(const maba_tensor* out) {
  return al16s(out->data) && out->stride[0] % 4 == 0 && out->stride[1] % 4 == 0 && out->stride[2] % 4 == 0;
}

int launch_dgda_sub(const maba_tensor* q, const maba_tensor* k, const maba_tensor* v,
                    const maba_tensor* gate, int use_log, const maba_tensor* b,
                    const maba_tensor* w, const maba_tensor* s0, maba_tensor* out,
                    maba_tensor* sf, void* ws, size_t ws_bytes, hipStream_t stream) {
  const int64_t B = q->shape[0], H = q->shape[1], L = q->shape[2], dk = q->shape[3], dv = v->shape[3];
  const int64_t BH = B * H;
  SubArgs a = {};
  // strides fit in int32 (dgda_sub_supported checks every operand)
  a.q = q->data; a.qs0 = (int)q->stride[0]; a.qs1 = (int)q->stride[1]; a.qs2 = (int)q->stride[2];
  a.k = k->data; a.ks0 = (int)k->stride[0]; a.ks1 = (int)k->stride[1]; a.ks2 = (int)k->stride[2];
  a.vp = v->data; a.vs0 = (int)v->stride[0]; a.vs1 = (int)v->stride[1]; a.vs2 = (int)v->stride[2];
  a.gp = gate->data; a.gs0 = (int)gate->stride[0]; a.gs1 = (int)gate->stride[1];
  a.gs2 = (int)gate->stride[2]; a.gs3 = (int)gate->stride[3];
  a.bp = b->data; a.bs0 = (int)b->stride[0]; a.bs1 = (int)b->stride[1];
  a.bs2 = (int)b->stride[2]; a.bs3 = (int)b->stride[3];
  a.wp = w->data; a.ws0 = (int)w->stride[0]; a.ws1 = (int)w->stride[1];
  a.ws2 = (int)w->stride[2]; a.ws3 = (int)w->stride[3];
  a.s0 = view4(s0);
  a.op = out->data; a.odt = out->dtype;
  a.os0 = (int)out->stride[0]; a.os1 = (int)out->stride[1]; a.os2 = (int)out->stride[2];
  a.ovec = sub_out_vec(out);
  a.sf = mview4(sf);
  a.H = (int)H; a.L = (int)L; a.BH = (int)BH;
  a.use_log = use_log; a.has_s0 = s0 != nullptr;
  a.f16 = q->dtype == MABA_F16;
  const int cols = sub_place(a, BH, L, dk, dv, ws, ws_bytes, true);
  const bool f32in = q->dtype == MABA_F32, g16 = gate->dtype != MABA_F32;
  const bool gch = a.gs3 == 1 && a.bs3 == 1 && a.ws3 == 1;
  if (dk == 32) return run_sub_k32(a, cols, f32in, g16, gch, stream);
  if (dk == 64) return run_sub_k64(a, cols, f32in, g16, gch, stream);
  return run_sub_k128(a, cols, f32in, g16, gch, stream);
}

int run_sub_k64(SubArgs& a, int dv, bool f32in, bool g16, bool gch, hipStream_t stream) {
  return dv == 32 ? run_sub_passes<false, 64, 32>(a, f32in, g16, gch, stream)
                  : run_sub_passes<false, 64, 64>(a, f32in, g16, gch, stream);
}

}  // namespace maba

using namespace maba;

extern "C" size_t maba_hip_dgda_layer_prefill_workspace_size(int64_t B, int64_t H, int64_t L) {
  return std::max(dgda_sub_workspace(B * H, L, 64, 64), dgda_sub_workspace_preferred(B * H, L, 64, 64));
}

extern "C" int maba_hip_dgda_layer_prefill(const maba_tensor* const* xs, const maba_tensor* const* conv_w,
                                           const maba_tensor* const* hist, float eps,
                                           const maba_tensor* initial_state, maba_tensor* out,
                                           maba_tensor* final_state, maba_tensor* const* new_hist, void* workspace,
                                           size_t workspace_bytes, void* stream) {
  if (!xs || !conv_w || !new_hist || !out || !final_state)
    return fail(MABA_ERR_INVALID, "dgda_layer_prefill: null argument");
  for (int s = 0; s < 6; ++s)
    if (!xs[s] || xs[s]->ndim != 3) return fail(MABA_ERR_INVALID, "dgda_layer_prefill: projection %d must be [B,L,C]", s);
  const int64_t B = xs[0]->shape[0], L = xs[0]->shape[1], C = xs[0]->shape[2];
  if (C % 64 != 0 || C == 0) return fail(MABA_ERR_UNSUPPORTED, "dgda_layer_prefill: C must be 64 * H");
  if (L < 1) return fail(MABA_ERR_INVALID, "dgda_layer_prefill: at least one token");
  if (L > ((int64_t)1 << 30)) return fail(MABA_ERR_UNSUPPORTED, "dgda_layer_prefill: L too large");
  const int64_t H = C / 64, BH = B * H;
  for (int s = 0; s < 6; ++s) {
    const maba_tensor* t = xs[s];
    if (t->shape[0] != B || t->shape[1] != L || t->shape[2] != C || t->dtype != MABA_BF16 || t->stride[2] != 1 ||
        ((uintptr_t)t->data & 7) || t->stride[0] % 4 || t->stride[1] % 4 || !fits32s(t))
      return fail(MABA_ERR_UNSUPPORTED, "dgda_layer_prefill: projections must be bf16 [B,L,C], unit channel "
                  "stride, 8-byte aligned rows");
    // the kernels address the 19 rows under a sub-chunk's conv taps with 32-bit byte offsets
    if ((L + SC) * t->stride[1] + C > INT32_MAX)
      return fail(MABA_ERR_UNSUPPORTED, "dgda_layer_prefill: L * row stride must stay below 2^31 elements");
  }
  const int64_t sw[3] = {C, 1, 4}, sh[3] = {B, C, 3};
  for (int s = 0; s < 3; ++s) {
    if (!expect_shape(conv_w[s], "conv weight", 3, sw) || !expect_float(conv_w[s], "conv weight"))
      return MABA_ERR_INVALID;
    if (conv_w[s]->dtype != conv_w[0]->dtype) return fail(MABA_ERR_DTYPE, "dgda_layer_prefill: conv weights differ in dtype");
    if (!fits32s(conv_w[s])) return fail(MABA_ERR_UNSUPPORTED, "dgda_layer_prefill: conv weight strides");
    if (hist) {
      if (!expect_shape(hist[s], "conv history", 3, sh)) return MABA_ERR_INVALID;
      if (hist[s]->dtype != MABA_BF16 || !fits32s(hist[s]))
        return fail(MABA_ERR_DTYPE, "dgda_layer_prefill: the conv history must be bf16");
    }
    if (!expect_shape(new_hist[s], "new conv history", 3, sh) || !expect_float(new_hist[s], "new conv history"))
      return MABA_ERR_INVALID;
  }
  const int64_t so[4] = {B, H, L, 64}, ss[4] = {B, H, 64, 64};
  if (!expect_shape(out, "out", 4, so) || !expect_shape(final_state, "final_state", 4, ss)) return MABA_ERR_INVALID;
  if (out->stride[3] != 1 || !fits32s(out) || (out->dtype != MABA_BF16 && out->dtype != MABA_F32))
    return fail(MABA_ERR_UNSUPPORTED, "dgda_layer_prefill: out must be f32/bf16 with unit channel stride");
  if (!expect_float(final_state, "final_state")) return MABA_ERR_DTYPE;
  if (initial_state && (!expect_shape(initial_state, "initial_state", 4, ss) || !expect_float(initial_state, "initial_state")))
    return MABA_ERR_INVALID;
  const size_t need = dgda_sub_workspace(BH, L, 64, 64);
  if (!workspace || workspace_bytes < need)
    return fail(MABA_ERR_WORKSPACE, "dgda_layer_prefill: workspace of %zu bytes required", need);
  if (B == 0) return MABA_OK;
  SubArgs a = {};
  for (int s = 0; s < 6; ++s) {
    a.px[s] = (const uint16_t*)xs[s]->data; a.pxs0[s] = (int)xs[s]->stride[0]; a.pxs1[s] = (int)xs[s]->stride[1];
  }
  a.cwdt = conv_w[0]->dtype;
  for (int s = 0; s < 3; ++s) {
    a.cw[s] = conv_w[s]->data; a.cwsc[s] = (int)conv_w[s]->stride[0]; a.cwst[s] = (int)conv_w[s]->stride[2];
    a.ph[s] = hist ? (const uint16_t*)hist[s]->data : nullptr;
    a.phs0[s] = hist ? (int)hist[s]->stride[0] : 0; a.phs1[s] = hist ? (int)hist[s]->stride[1] : 0;
    a.phs2[s] = hist ? (int)hist[s]->stride[2] : 0;
  }
  a.eps = eps;
  a.s0 = view4(initial_state);
  for (int s = 0; s < 3; ++s) {
    a.nh[s] = new_hist[s]->data; a.nhdt[s] = new_hist[s]->dtype;
    a.nhs0[s] = new_hist[s]->stride[0]; a.nhs1[s] = new_hist[s]->stride[1]; a.nhs2[s] = new_hist[s]->stride[2];
  }
  a.op = out->data; a.odt = out->dtype;
  a.os0 = (int)out->stride[0]; a.os1 = (int)out->stride[1]; a.os2 = (int)out->stride[2];
  a.ovec = sub_out_vec(out);
  a.sf = mview4(final_state);
  a.H = (int)H; a.L = (int)L; a.BH = (int)BH;
  a.use_log = 1; a.has_s0 = initial_state != nullptr;
  // the new history is written by the last launch, after the first one has read the old: it may
  // overwrite it in place; where one launch is all, by the one wave per head that read it
  const int cols = sub_place(a, BH, L, 64, 64, workspace, workspace_bytes,
                             !hist || sub_cut(BH, L, 64, 64, workspace_bytes, true).nseg > 1 || histories_apart(hist, new_hist));
  return cols == 32 ? run_sub_passes<true, 64, 32>(a, false, false, true, (hipStream_t)stream)
                    : run_sub_passes<true, 64, 64>(a, false, false, true, (hipStream_t)stream);
}
