// One call per pass: the launch sequences of the ops (host code only; the
// kernels behind the C ABI entry points it calls live in the other files).
//
// A pass of the smallest shapes is bound by the host: at 8 heads x 2 048 tokens
// the forward's kernels take 24 us and the launches, allocations and argument
// conversions of four separate calls from Python took 52.  Here a pass costs
// one call, one allocation per workspace and its launches.
#include <hip/hip_runtime.h>

#include "vsa_launch.h"

namespace vsa {
namespace {

// Hands out 256-byte aligned pieces of a workspace (base may be null: only the
// size is wanted).
struct Carve {
  char* base;
  int64_t used = 0;
  template <typename P = void>
  P* take(int64_t bytes) {
    const int64_t at = used;
    used += (bytes + 255) / 256 * 256;
    return base ? reinterpret_cast<P*>(base + at) : nullptr;
  }
};

struct Dims {
  bool full, raster, padded;
  int qb, kb, D, be, es, gate_es, gate_width;
  int64_t sq, skv;   // as the kernels see them
  int gate_layout;   // gate_mode without its type flag
};

int dims_of(const vsa_op* op, Dims& d) {
  if (!op || (op->dtype != VSA_BF16 && op->dtype != VSA_F16 && op->dtype != VSA_F32))
    return op ? VSA_ERR_DTYPE : VSA_ERR_NULL;
  d.full = op->selected == nullptr;
  d.raster = op->slot_rows != nullptr;
  if (op->bh <= 0 || op->block <= 0 || op->sq <= 0 || op->skv <= 0 || op->topk < 1 ||
      op->sq % op->block || op->skv % op->block || op->sq > (1LL << 31) / 256 ||
      op->skv > (1LL << 31) / 256 || op->block > op->kernel_block ||
      op->head_dim <= 0 || op->head_dim > op->kernel_dim || (d.raster && !d.full))
    return VSA_ERR_SHAPE;
  d.D = op->kernel_dim;
  d.be = op->kernel_block;
  d.padded = d.D != op->head_dim || d.be != op->block;
  if (d.padded && d.raster) return VSA_ERR_SHAPE;
  d.qb = (int)(op->sq / op->block);
  d.kb = (int)(op->skv / op->block);
  d.sq = (int64_t)d.qb * d.be;
  d.skv = (int64_t)d.kb * d.be;
  d.es = op->dtype == VSA_F32 ? 4 : 2;
  d.gate_layout = d.full ? op->gate_mode & ~VSA_GATE_F32 : 0;
  d.gate_es = op->gate_mode & VSA_GATE_F32 ? 4 : d.es;
  d.gate_width = d.gate_layout == VSA_GATE_PER_TOKEN ? 1 : d.D;
  // the padded copies of a token-major gate would need its own layout
  if (d.padded && d.gate_layout == VSA_GATE_TOKEN_MAJOR) return VSA_ERR_SHAPE;
  return VSA_OK;
}

// What a forward produces for its own later steps and for the backward.
struct Kept {
  void *q = nullptr, *k = nullptr, *v = nullptr, *gate = nullptr;  // padded / tiled copies
  void *qc = nullptr, *kc = nullptr, *vc = nullptr, *outc = nullptr;
  float* probs = nullptr;
  int32_t* sel = nullptr;
  void* fine = nullptr;   // fine output (full op; the padded route op's result)
  float* lse = nullptr;
};

Kept carve_kept(Carve& c, const vsa_op* op, const Dims& d, bool keep) {
  Kept k;
  const int64_t bh = op->bh, row = (int64_t)d.D * d.es;
  if (d.padded || d.raster) {
    k.q = c.take(bh * d.sq * row);
    k.k = c.take(bh * d.skv * row);
    k.v = c.take(bh * d.skv * row);
    if (d.padded && d.gate_layout) k.gate = c.take(bh * d.sq * d.gate_width * d.gate_es);
  }
  if (d.full) {
    k.qc = c.take(bh * d.qb * row);
    k.kc = c.take(bh * d.kb * row);
    k.vc = c.take(bh * d.kb * row);
    k.outc = c.take(bh * d.qb * row);
    k.probs = c.take<float>(bh * d.qb * d.kb * 4);
    k.sel = c.take<int32_t>(bh * d.qb * (int64_t)op->topk * 4);
  }
  if (keep) {
    if (d.full || d.padded) k.fine = c.take(bh * d.sq * row);
    k.lse = c.take<float>(bh * d.sq * 4);
  }
  return k;
}

// Scratch of the forward: with nothing kept, its intermediates too.
struct FwdScratch {
  float* scores = nullptr;
  void* out = nullptr;  // the padded op's result before its rows are taken back
};

FwdScratch carve_fwd(Carve& c, const vsa_op* op, const Dims& d) {
  FwdScratch s;
  if (d.full) s.scores = c.take<float>(op->bh * d.qb * d.kb * 4);
  if (d.padded && (d.full || !op->keep)) s.out = c.take(op->bh * d.sq * d.D * d.es);
  return s;
}

struct BwdScratch {
  float *delta, *ds;
  void *d_outc, *dqc, *dkc, *dvc;
  int32_t *counts, *offsets, *inverse, *order;
  int64_t order_len;
  void *dout, *dq, *dk, *dv, *dgate;  // tiled dout; padded dout and gradients
};

BwdScratch carve_bwd(Carve& c, const vsa_op* op, const Dims& d) {
  BwdScratch s = {};
  const int64_t bh = op->bh, row = (int64_t)d.D * d.es;
  s.delta = c.take<float>(bh * d.sq * 4);
  if (d.full) {
    s.d_outc = c.take(bh * d.qb * row);
    s.dqc = c.take(bh * d.qb * row);
    s.dkc = c.take(bh * d.kb * row);
    s.dvc = c.take(bh * d.kb * row);
    s.ds = c.take<float>(bh * d.qb * d.kb * 4);
  }
  s.counts = c.take<int32_t>(bh * d.kb * 4);
  s.offsets = c.take<int32_t>(bh * d.kb * 4);
  s.inverse = c.take<int32_t>(bh * d.qb * (int64_t)op->topk * 4);
  if (op->dtype != VSA_F32) {
    // the smallest tiles any dK/dV kernel takes: 64 keys, in two halves at head dim 256
    const int64_t tiles = bh * (d.skv / 64) * (d.D > 128 ? 2 : 1);
    s.order_len = 8 * ((tiles + 7) / 8) + 16;
    s.order = c.take<int32_t>(s.order_len * 4);
  }
  if (d.padded || d.raster) s.dout = c.take(bh * d.sq * row);
  if (d.padded) {
    s.dq = c.take(bh * d.sq * row);
    s.dk = c.take(bh * d.skv * row);
    s.dv = c.take(bh * d.skv * row);
    if (d.gate_layout) s.dgate = c.take(bh * d.sq * d.gate_width * d.gate_es);
  }
  return s;
}

// A list of block moves between the caller's shapes and the padded ones.
struct Moves {
  BlockMove m = {};
  const vsa_op* op;
  const Dims& d;
  bool pad;
  Moves(const vsa_op* o, const Dims& dd, bool p) : op(o), d(dd), pad(p) {
    m.be = o->block;
    m.kbe = dd.be;
  }
  void add(const void* src, void* dst, int nb, int width, int kwidth, int es) {
    const int i = m.n++;
    m.src[i] = src;
    m.dst[i] = dst;
    m.rows[i] = op->bh * nb * (pad ? d.be : op->block);
    m.src_bytes[i] = (pad ? width : kwidth) * es;
    m.dst_bytes[i] = (pad ? kwidth : width) * es;
  }
  void rows(const void* src, void* dst, int nb) {
    add(src, dst, nb, op->head_dim, d.D, d.es);
  }
  void gate(const void* src, void* dst) {
    const bool tok = d.gate_layout == VSA_GATE_PER_TOKEN;
    add(src, dst, d.qb, tok ? 1 : op->head_dim, d.gate_width, d.gate_es);
  }
  int run(hipStream_t s) { return block_move(m, pad, s); }
};

#define VSA_TRY(call)                 \
  do {                                \
    const int rc_ = (call);           \
    if (rc_ != VSA_OK) return rc_;    \
  } while (0)

}  // namespace
}  // namespace vsa

using namespace vsa;

extern "C" int vsa_op_sizes(const vsa_op* op, int64_t* saved, int64_t* scratch_fwd,
                            int64_t* scratch_bwd) {
  Dims d;
  VSA_TRY(dims_of(op, d));
  if (!saved || !scratch_fwd || !scratch_bwd) return VSA_ERR_NULL;
  Carve kept{nullptr}, fwd{nullptr}, bwd{nullptr};
  carve_kept(op->keep ? kept : fwd, op, d, op->keep != 0);
  carve_fwd(fwd, op, d);
  if (op->keep) carve_bwd(bwd, op, d);
  *saved = kept.used;
  *scratch_fwd = fwd.used;
  *scratch_bwd = bwd.used;
  return VSA_OK;
}

extern "C" int vsa_op_fwd(const vsa_op* op, void* out, void* saved, void* scratch, void* stream) {
  Dims d;
  VSA_TRY(dims_of(op, d));
  if (!op->q || !op->k || !op->v || !op->kv_vbs || !out || (d.full && !op->q_vbs) ||
      (op->keep && !saved) || (d.gate_layout && !op->gate))
    return VSA_ERR_NULL;
  if (!vsa_aligned<16>(op->q, op->k, op->v, op->gate, out) || !vsa_aligned<256>(saved, scratch))
    return VSA_ERR_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  Carve kept{(char*)saved}, fwd{(char*)scratch};
  const Kept k = carve_kept(op->keep ? kept : fwd, op, d, op->keep != 0);
  const FwdScratch f = carve_fwd(fwd, op, d);
  if (fwd.used && !scratch) return VSA_ERR_NULL;

  const void *q = op->q, *kk = op->k, *v = op->v, *gate = d.gate_layout ? op->gate : nullptr;
  void* res = out;
  if (d.padded) {
    Moves mv(op, d, true);
    mv.rows(q, k.q, d.qb);
    mv.rows(kk, k.k, d.kb);
    mv.rows(v, k.v, d.kb);
    if (gate) mv.gate(gate, k.gate);
    VSA_TRY(mv.run(s));
    q = k.q;
    kk = k.k;
    v = k.v;
    if (gate) gate = k.gate;
    res = d.full || !op->keep ? f.out : k.fine;
  }
  const int32_t* sel = op->selected;
  if (d.full) {
    if (d.raster) {
      VSA_TRY(vsa_tile_pool_qkv(q, kk, v, op->slot_rows, op->q_vbs, op->kv_vbs, k.q, k.k, k.v,
                                k.qc, k.kc, k.vc, op->bh, op->s_out, op->heads, d.qb, d.D, d.be,
                                op->dtype, stream));
      q = k.q;
      kk = k.k;
      v = k.v;
    } else {
      VSA_TRY(vsa_pool_qkv(q, kk, v, op->q_vbs, op->kv_vbs, k.qc, k.kc, k.vc, op->bh, d.sq,
                           d.skv, d.D, d.be, op->dtype, stream));
    }
    VSA_TRY(vsa_coarse_fwd(k.qc, k.kc, k.vc, f.scores, k.probs, k.outc, k.sel, op->bh, d.qb, d.kb,
                           d.D, op->topk, op->scale, op->dtype, stream));
    sel = k.sel;
  }
  if (d.raster)
    return vsa_sparse_fwd_tiled(q, kk, v, sel, op->kv_vbs, res, k.fine, k.lse, k.outc, gate,
                                op->gate_mode, op->slot_rows, op->s_out, op->heads, op->bh, d.sq,
                                d.skv, d.D, d.be, op->topk, op->scale, op->dtype, stream);
  VSA_TRY(sparse_fwd_rows(op->block, q, kk, v, sel, op->kv_vbs, res, d.full ? k.fine : nullptr,
                          k.lse, k.outc, gate, d.full ? op->gate_mode : 0, op->gate_heads, op->bh,
                          d.sq, d.skv, d.D, d.be, op->topk, op->scale, op->dtype, stream));
  if (d.padded) {
    Moves mv(op, d, false);
    mv.rows(res, out, d.qb);
    return mv.run(s);
  }
  return VSA_OK;
}

extern "C" int vsa_op_bwd(const vsa_op* op, const void* out, const void* dout, void* saved,
                          void* scratch, void* dq, void* dk, void* dv, void* d_gate,
                          void* stream) {
  Dims d;
  VSA_TRY(dims_of(op, d));
  const bool copies = d.padded || d.raster;
  if (!op->kv_vbs || !dout || !saved || !scratch || !dq || !dk || !dv ||
      (!copies && (!op->q || !op->k || !op->v)) || (d.full && !op->q_vbs) ||
      (!d.full && !d.padded && !out) || (d.gate_layout && !d_gate) ||
      (d.gate_layout && !d.padded && !op->gate) || !op->keep)
    return VSA_ERR_NULL;
  if (!vsa_aligned<16>(op->q, op->k, op->v, op->gate, out, dout, dq, dk, dv, d_gate) ||
      !vsa_aligned<256>(saved, scratch))
    return VSA_ERR_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  Carve kept{(char*)saved}, bwd{(char*)scratch};
  const Kept k = carve_kept(kept, op, d, true);
  const BwdScratch b = carve_bwd(bwd, op, d);

  const void* q = copies ? k.q : op->q;
  const void* kk = copies ? k.k : op->k;
  const void* v = copies ? k.v : op->v;
  const void* gate = !d.gate_layout ? nullptr : d.padded ? k.gate : op->gate;
  const int32_t* sel = d.full ? k.sel : op->selected;
  void *gq = d.padded ? b.dq : dq, *gk = d.padded ? b.dk : dk, *gv = d.padded ? b.dv : dv;
  void* gg = !d.gate_layout ? nullptr : d.padded ? b.dgate : d_gate;
  const void* g = dout;
  if (d.padded) {
    Moves mv(op, d, true);
    mv.rows(dout, b.dout, d.qb);
    VSA_TRY(mv.run(s));
    g = b.dout;
  }
  if (d.raster) {
    VSA_TRY(vsa_bwd_prep_tiled(k.fine, dout, k.outc, gate, op->gate_mode, op->slot_rows,
                               op->s_out, op->heads, b.delta, b.d_outc, gg, b.dout, op->bh, d.sq,
                               d.D, d.be, op->dtype, stream));
    g = b.dout;
  } else {
    VSA_TRY(vsa_bwd_prep(k.fine ? k.fine : out, g, k.outc, gate, d.full ? op->gate_mode : 0,
                         op->gate_heads, b.delta, b.d_outc, gg, op->bh, d.sq, d.D, d.be,
                         op->dtype, stream));
  }
  if (d.full)
    VSA_TRY(vsa_coarse_bwd(k.qc, k.kc, k.vc, k.probs, b.d_outc, b.ds, b.dqc, b.dkc, b.dvc, op->bh,
                           d.qb, d.kb, d.D, op->scale, op->dtype, stream));
  VSA_TRY(vsa_csr_build(sel, b.counts, b.offsets, b.inverse, op->bh, d.qb, d.kb, op->topk,
                        stream));
  if (b.order)
    VSA_TRY(vsa_dkdv_tile_order(b.counts, b.order, b.order_len, op->bh, d.skv, d.D, d.be, stream));
  if (d.raster) {
    VSA_TRY(vsa_sparse_bwd_dq_tiled(q, kk, v, g, k.lse, b.delta, sel, op->kv_vbs, gq, b.dqc,
                                    op->q_vbs, op->slot_rows, op->s_out, op->heads, op->bh, d.sq,
                                    d.skv, d.D, d.be, op->topk, op->scale, op->dtype, stream));
    return vsa_sparse_bwd_dkdv_tiled(q, kk, v, g, k.lse, b.delta, b.counts, b.offsets, b.inverse,
                                     op->kv_vbs, gk, gv, b.dkc, b.dvc, op->slot_rows, op->s_out,
                                     op->heads, op->bh, d.sq, d.skv, d.D, d.be, op->topk,
                                     op->scale, b.order, op->dtype, stream);
  }
  VSA_TRY(sparse_bwd_dq_rows(op->block, q, kk, v, g, k.lse, b.delta, sel, op->kv_vbs, gq, b.dqc,
                            d.full ? op->q_vbs : nullptr, op->bh, d.sq, d.skv, d.D, d.be,
                            op->topk, op->scale, op->dtype, stream));
  VSA_TRY(sparse_bwd_dkdv_rows(op->block, q, kk, v, g, k.lse, b.delta, b.counts, b.offsets, b.inverse,
                              op->kv_vbs, gk, gv, b.dkc, b.dvc, op->bh, d.sq, d.skv, d.D, d.be,
                              op->topk, op->scale, b.order, op->dtype, stream));
  if (d.padded) {
    Moves mv(op, d, false);
    mv.rows(gq, dq, d.qb);
    mv.rows(gk, dk, d.kb);
    mv.rows(gv, dv, d.kb);
    if (gg) mv.gate(gg, d_gate);
    return mv.run(s);
  }
  return VSA_OK;
}
