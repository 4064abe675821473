// A whole decoder layer per call: the launches of a decode step or of a mixed prompt + decode step issued
// from native code, in the order and with the choices of jitengine_amd/model.py's op-by-op path
// (Q36/model/model.py:65-80).  Host code only; every launch is an entry point of this library.
//
// What it is for: the host.  Issued op by op from Python a one-token layer costs ~95 us of host time (7
// launches, ~15 us each with the tensors, checks and argument conversion) against ~45 us of GPU time at 4,096
// keys, so a lone sequence's step waited for the host; one call costs ~30 us.
#include <cstdint>

#include "jit_moe.h"

namespace jit {
int fail(int code, const char *fmt, ...);
}

namespace {

// The layer's intermediates inside the caller's scratch (256-byte aligned pieces, in this order).
struct Scratch {
  uint16_t *x, *xn, *qkv, *q, *attn, *o, *h, *hn, *logits, *scores, *hh, *r;
  uint32_t *inds;
  int32_t *order, *pair_row, *inv, *cnt, *off, *seg_expert, *seg_start, *seg_cnt, *meta;
  void *pack_ws;
  int64_t pack_ws_bytes, bytes;

  Scratch(const jit_layer &L, int rows, bool mixed, void *base) {
    uint8_t *p = (uint8_t *)base;
    int64_t at = 0;
    auto take = [&](int64_t n) {
      uint8_t *q = p + at;
      at += (n + 255) / 256 * 256;
      return q;
    };
    auto bf = [&](int64_t n) { return (uint16_t *)take(2 * n); };
    const int64_t B = rows, P = B * L.k, heads = (int64_t)L.H * JIT_HEAD_DIM;
    // (what a deferred combine reads -- r, inv, scores, h -- comes first: its place depends on D and k alone)
    r = bf(P * L.D);
    h = bf(B * L.D);
    scores = bf(P);
    int32_t *t = (int32_t *)take(4 * (3 * P + 5 * (int64_t)L.E + 4));
    order = t;
    pair_row = t + P;
    inv = t + 2 * P;
    cnt = t + 3 * P;
    off = cnt + L.E;
    seg_expert = off + L.E;
    seg_start = seg_expert + L.E;
    seg_cnt = seg_start + L.E;
    meta = seg_cnt + L.E;
    x = bf(B * L.D);
    xn = bf(B * L.D);
    qkv = bf(B * (L.H + 2 * (int64_t)L.Hkv) * JIT_HEAD_DIM);
    q = mixed ? bf(B * heads) : nullptr;
    attn = bf(B * heads);
    o = bf(B * L.D);
    hn = bf(B * L.D);
    logits = bf(B * L.E);
    inds = (uint32_t *)take(4 * P);
    hh = bf(P * L.I);
    pack_ws_bytes = jit_moe_pack_workspace_bytes((int)P, L.E);
    pack_ws = take(pack_ws_bytes);
    bytes = at;
  }
};

bool row_prologue_fits(int N, int D) { return D % 256 == 0 && D <= 2048 && N % 16 == 0; }

// x . W^T on the tile GEMM of long batches or the decode kernel (ops.qmm's rule).
int project(const uint16_t *x, int T, int K, const void *w, int N, uint16_t *y, bool prompt, void *st) {
  if (prompt && T >= 192 && N % 256 == 0 && K % 128 == 0) return jit_qmm_seg(x, T, K, w, N, y, st);
  return jit_qmm_packed(x, T, K, w, N, y, st);
}

#define JIT_TRY(call)         \
  do {                        \
    if (int rc_ = (call)) return rc_; \
  } while (0)

// From the attention's rows on: o projection, residual + norm, router, experts, combine.
int layer_tail(const jit_layer &L, int B, bool prompt, const uint16_t *x, const Scratch &s, int defer,
               const uint16_t *next_norm, uint16_t *y, uint16_t *xn_next, void *st) {
  const int D = L.D, E = L.E, k = L.k, I = L.I, P = B * k;
  JIT_TRY(project(s.attn, B, L.H * JIT_HEAD_DIM, L.o, D, s.o, prompt, st));
  if (!prompt && B == 1 && row_prologue_fits(E, D)) {
    JIT_TRY(jit_qmm_packed_add_rmsnorm(s.o, x, L.post_norm, L.eps, D, L.router, E, s.h, s.hn, s.logits, st));
  } else {
    JIT_TRY(jit_rmsnorm(s.o, x, B, D, L.post_norm, L.eps, s.h, s.hn, st));
    JIT_TRY(project(s.hn, B, D, L.router, E, s.logits, prompt, st));
  }
  if (!prompt && B == 1 && E % 32 == 0 && E <= 128 && k < E && k <= 64) {
    JIT_TRY(jit_moe_gate_up_swiglu_routed_packed(s.hn, D, s.logits, E, k, L.norm_topk, L.gate_up, I, s.hh, s.inds,
                                                 s.scores, s.order, s.pair_row, s.inv, s.cnt, s.off, s.seg_expert,
                                                 s.seg_start, s.seg_cnt, s.meta, st));
    JIT_TRY(jit_moe_down_packed(s.hh, I, s.cnt, s.off, E, L.down, D, P, s.r, st));
  } else {
    if (!prompt && B <= 4 && E <= 128) {
      JIT_TRY(jit_route_pack(s.logits, B, E, k, L.norm_topk, s.inds, s.scores, s.order, s.pair_row, s.inv, s.cnt,
                             s.off, s.seg_expert, s.seg_start, s.seg_cnt, s.meta, st));
    } else {
      JIT_TRY(jit_router_topk(s.logits, B, E, k, L.norm_topk, s.inds, s.scores, nullptr, st));
      if (s.pack_ws_bytes)
        JIT_TRY(jit_moe_pack_ws(s.inds, P, k, E, s.order, s.pair_row, s.inv, s.cnt, s.off, s.seg_expert, s.seg_start,
                                s.seg_cnt, s.meta, s.pack_ws, s.pack_ws_bytes, st));
      else
        JIT_TRY(jit_moe_pack(s.inds, P, k, E, s.order, s.pair_row, s.inv, s.cnt, s.off, s.seg_expert, s.seg_start,
                             s.seg_cnt, s.meta, st));
    }
    if (prompt && P >= 16 && P / E >= 4) {  // (MoEBlock.use_seg)
      JIT_TRY(jit_moe_gate_up_swiglu_seg(s.hn, D, s.pair_row, s.cnt, s.off, E, L.gate_up, I, P, s.hh, st));
      JIT_TRY(jit_moe_down_seg(s.hh, I, s.cnt, s.off, E, L.down, D, P, s.r, st));
    } else {
      JIT_TRY(jit_moe_gate_up_swiglu_packed(s.hn, D, s.pair_row, s.cnt, s.off, E, L.gate_up, I, P, s.hh, st));
      JIT_TRY(jit_moe_down_packed(s.hh, I, s.cnt, s.off, E, L.down, D, P, s.r, st));
    }
  }
  if (defer) return JIT_OK;
  if (next_norm)
    return jit_moe_combine_rmsnorm(s.r, s.inv, s.scores, B, k, D, s.h, y, next_norm, L.eps, xn_next, st);
  return jit_moe_combine(s.r, s.inv, s.scores, B, k, D, s.h, y, st);
}

int layer_check(const jit_layer *L, int rows, const char *what) {
  if (!L || rows < 1 || L->D <= 0 || L->H <= 0 || L->Hkv <= 0 || L->E <= 0 || L->k <= 0 || L->I <= 0)
    return jit::fail(JIT_EINVAL, "%s: bad geometry or %d rows", what, rows);
  if (!L->input_norm || !L->q_norm || !L->k_norm || !L->post_norm || !L->inv_freq || !L->qkv || !L->o || !L->router ||
      !L->gate_up || !L->down)
    return jit::fail(JIT_EINVAL, "%s: null weight", what);
  if ((long long)rows * L->k > 0x7fffffffLL) return jit::fail(JIT_EUNSUPPORTED, "%s: %d rows", what, rows);
  return JIT_OK;
}

}  // namespace

extern "C" int64_t jit_layer_scratch_bytes(const jit_layer *layer, int rows, int mixed) {
  if (layer_check(layer, rows, "layer_scratch_bytes")) return -1;
  return Scratch(*layer, rows, mixed != 0, nullptr).bytes;
}

extern "C" int jit_decode_layer(const jit_layer *layer, const jit_decode_rows *d, uint16_t *pool, const uint16_t *x,
                                const uint16_t *xn, const jit_layer *prev_layer, const void *prev, int defer,
                                const uint16_t *next_norm, void *scratch, uint16_t *y, uint16_t *xn_next, void *stream) {
  if (!d) return jit::fail(JIT_EINVAL, "decode_layer: null step");
  JIT_TRY(layer_check(layer, d->B, "decode_layer"));
  const jit_layer &L = *layer;
  const int B = d->B, D = L.D, nqkv = (L.H + 2 * L.Hkv) * JIT_HEAD_DIM;
  if ((prev || defer) && B != 1) return jit::fail(JIT_EINVAL, "decode_layer: a deferred combine takes one row");
  if (!scratch || (!prev && !x) || (!defer && !y) || (next_norm && !defer && !xn_next))
    return jit::fail(JIT_EINVAL, "decode_layer: null pointer");
  if (prev) {
    JIT_TRY(layer_check(prev_layer, 1, "decode_layer: previous layer"));
    if (prev_layer->D != D)
      return jit::fail(JIT_EINVAL, "decode_layer: a deferred row of %d for a layer of %d", prev_layer->D, D);
  }
  const Scratch s(L, B, false, scratch);
  if (prev) {
    // (the row's combine is the previous layer's: its tables, top-k and places in its scratch)
    const Scratch p(*prev_layer, 1, false, (void *)prev);
    JIT_TRY(jit_qmm_packed_combine_rmsnorm(p.r, p.inv, p.scores, prev_layer->k, p.h, L.input_norm, L.eps, D, L.qkv, nqkv, s.x,
                                           s.qkv, stream));
    x = s.x;
  } else {
    if (!xn) {
      JIT_TRY(jit_rmsnorm(x, nullptr, B, D, L.input_norm, L.eps, nullptr, s.xn, stream));
      xn = s.xn;
    }
    JIT_TRY(jit_qmm_packed(xn, B, D, L.qkv, nqkv, s.qkv, stream));
  }
  JIT_TRY(jit_paged_decode_attn_qkv_ws(s.qkv, L.q_norm, L.k_norm, L.eps, L.inv_freq, pool, d->page_table,
                                       d->max_pages, d->lens, d->chunk_start, d->chunk_seq, B, L.H, L.Hkv, L.scale,
                                       d->total_chunks, d->workspace, d->workspace_bytes, s.attn, stream));
  return layer_tail(L, B, false, x, s, defer, next_norm, y, xn_next, stream);
}

extern "C" int jit_mixed_layer(const jit_layer *layer, const jit_prompt_rows *p, const jit_decode_rows *d,
                               uint16_t *pool, const uint16_t *x, void *scratch, uint16_t *y, void *stream) {
  if (!p || !d) return jit::fail(JIT_EINVAL, "mixed_layer: null step");
  const int T = p->rows + d->B;
  if (p->rows < 0 || d->B < 0) return jit::fail(JIT_EINVAL, "mixed_layer: %d prompt and %d decode rows", p->rows, d->B);
  JIT_TRY(layer_check(layer, T, "mixed_layer"));
  if (!x || !scratch || !y) return jit::fail(JIT_EINVAL, "mixed_layer: null pointer");
  const jit_layer &L = *layer;
  const int D = L.D, nqkv = (L.H + 2 * L.Hkv) * JIT_HEAD_DIM;
  const Scratch s(L, T, true, scratch);
  JIT_TRY(jit_rmsnorm(x, nullptr, T, D, L.input_norm, L.eps, nullptr, s.xn, stream));
  JIT_TRY(project(s.xn, T, D, L.qkv, nqkv, s.qkv, true, stream));
  JIT_TRY(jit_qk_norm_rope_append(s.qkv, T, L.H, L.Hkv, L.q_norm, L.k_norm, L.eps, L.inv_freq, p->pos, p->table_rows,
                                  p->table_rows_pages, pool, s.q, stream));
  // (both halves write their rows of one buffer: no concatenation)
  if (p->rows)
    JIT_TRY(jit_paged_prefill_attn(s.q, pool, p->seq_table, p->seq_pages, p->chunk_seq, p->chunk_ctx, p->chunk_len,
                                   p->chunk_row, p->C, p->blk_chunk, p->blk_q0, p->blk_part, p->nblk, p->pmax,
                                   p->max_len, L.H, L.Hkv, L.scale, p->workspace, s.attn, stream));
  if (d->B) {
    const int64_t at = (int64_t)p->rows * L.H * JIT_HEAD_DIM;
    JIT_TRY(jit_paged_decode_attn_ws(s.q + at, pool, d->page_table, d->max_pages, d->lens, d->chunk_start,
                                     d->chunk_seq, d->B, L.H, L.Hkv, L.scale, d->total_chunks, d->workspace,
                                     d->workspace_bytes, s.attn + at, stream));
  }
  return layer_tail(L, T, true, x, s, 0, nullptr, y, nullptr, stream);
}
