// One call for the whole no / scalar decay chunk forward: chunk_simple_gla_int8 (linquant/kernels/zoo/simple_gla.py:175-212)
// as one C entry over one caller-supplied workspace that holds what the Python wrapper would otherwise allocate per call.
// 64-token chunks where linear_scan says so: two launches, the operand pre-pass (zoo_lin_prep.hip; with it the operand rotations, if
// asked for) and recurrence with output (zoo_scan.hip).  Otherwise: the four stand-alone stages (cumsum, write-operand pre-pass or
// rotate-quantize, state recurrence, output) back to back.  The bits of the stage entry points in either case.
#include <initializer_list>

#include "zoo_params.h"

namespace {

constexpr int64_t kAlign = 256;
int64_t up(int64_t n) { return (n + kAlign - 1) / kAlign * kAlign; }

struct Layout {
  int64_t gc, kqT, vqT, vcT, qc, kc, A, gpk, ev, gam, h_i8, cross, total;
  bool scan;  // operand pre-pass, then recurrence and output in one launch
};

// No / scalar decay, linear family, 64-token chunks: recurrence and output in one launch (zoo_scan.hip), or state and output one after the other?
// The chain is NT steps either way, and a step that shares its SIMDs with the output is the longer one; the launch of its own has the
// whole chip for the output.  What the one launch saves is launches (4 .. 6 us a call, which decides short calls), the stored states
// (2 K V bytes a chunk and head) and the second reading of raw operands (with a prologue: of their token-major codes), against A
// (16 KB) and one more set of codes.
// With a prologue, up to 128 tiles of 32 columns: there the one launch runs a chain in segments side by side (zoo_scan.hip), and is the
// faster but for K = V = 64 on more than 80 tiles, where the chain is long.  GPU time of the two launches over that of the one, no decay ..
// scalar decay (B = 1, 16 to 128 tiles; graph replays of two sets of inputs in turn):
//                                T = 2048      4096          8192          32768
//   K = V = 128                  1.14 .. 1.54  1.15 .. 1.55  1.10 .. 1.73  1.12 .. 1.77
//   K 128, V 64                  1.16 .. 1.64  1.07 .. 1.65  1.05 .. 1.65  1.05 .. 1.66
//   K 64, V 128                  1.27 .. 1.72  1.26 .. 1.80  1.19 .. 1.82  1.01 .. 1.94
//   K = V = 64, to 80 tiles      1.09 .. 1.44  1.08 .. 1.43  1.00 .. 1.55  1.02 .. 1.61
//     96 .. 128                  1.05 .. 1.11  0.98 .. 1.05  0.91 .. 1.01  0.97 .. 1.19
// Otherwise, bytes saved > 0 (K = V = 128; with a prologue all but K = V = 64): one launch, while 16 KB are saved or there is no second
// tile per compute unit (more than 256) or no more than 32 steps; else: one launch for short chains whose operands stay in the last-level
// cache.  Time of the two launches over that of the one, three sets of inputs in turn, geometric mean over no and scalar decay, before the
// operand pre-pass took the last chunks first (zoo_params.h), by which the one launch gains: T = 2048 .. 8192, B*H = 4 .. 256 (where fewer
// tiles ran their chains in one piece): K = V = 128 0.91 .. 1.27, with prologue 1.00 .. 1.25; K 128, V 64 0.81 .. 1.11, with prologue
// 0.97 .. 1.18; K 64, V 128 0.78 .. 1.15 (B*H*NT <= 4096 0.99 .. 1.15), with prologue 0.89 .. 1.27; K = V = 64 0.67 .. 1.08, with
// prologue 0.83 .. 1.07 (B*H*NT <= 2048 0.98 .. 1.07).
// Without a prologue the lines of few tiles are still those of chains in one piece, also where segments have moved them (two launches over
// the one, measured as in the table above, K = V = 128, 128 tiles or fewer, past 128 steps 1.08 .. 1.79): the workspace that a caller asks
// for follows the route (lq_zoo_simple_gla_workspace_bytes), and that of few long chains grows by the one launch's operands.
bool linear_scan(bool prologue, int64_t B, int64_t T, int64_t H, int64_t K, int64_t V) {
  const int64_t NT = T / 64, chunks = B * H * NT, tiles = B * H * (V / 32);
  if (prologue && tiles <= 128) return K + V > 128 || NT <= 64 || tiles <= 80;
  if (NT > 128 && tiles < 128) return false;
  const int64_t saved = 2 * K * V - 16384 + (prologue ? 128 * K : 0);  // bytes a chunk and head
  if (saved >= 16384) return true;
  if (saved > 0) return NT <= 32 || tiles <= 256;
  return saved == 0 ? NT <= V / 2 && chunks <= 32 * V : NT <= 32 && chunks <= 1024;
}

// What the launches over 64-token chunks (operand pre-pass, zoo_scan.hip) ask of a call, checked in front of the first of them; the
// same calls that the stage entry points take
int check_scan(const void* q, const void* k, const void* v, const void* o, const void* ss, const void* svl, int B, int T, int H, int K,
               int V, int qmax, int dt) {
  if ((K != 64 && K != 128) || V % 64 != 0 || qmax < 1 || qmax > 127) return LQ_ERR_SHAPE;
  if (dt != LQ_DT_F16 && dt != LQ_DT_BF16) return LQ_ERR_SHAPE;
  for (const void* x : {q, k, v, o, ss, svl})
    if (!zoo_al(x, 16)) return LQ_ERR_SHAPE;
  if ((int64_t)B * H > 65535 || T / 64 > 65535 || (int64_t)(T / 64) * B * H > 0x7fffffff) return LQ_ERR_SHAPE;
  return LQ_OK;
}

// Does lq_zoo_rotate_quant, the staged route's operand launch, take this call?  (the one-launch route takes any V that is a multiple
// of 64, and tables at any address)
bool staged_prologue(const lq_zoo_simple_gla_args* a) {
  if (a->vdim != 64 && a->vdim != 128) return false;
  for (const void* x : {a->dq, a->dq_rcp, a->skw, a->svw})
    if (!zoo_al(x, 16)) return false;
  return true;
}

bool has_prologue(const lq_zoo_simple_gla_args* a) { return a->signs_qk || a->signs_v || a->dq; }

int check_dims(const lq_zoo_simple_gla_args* a) {
  if (a->batch <= 0 || a->seqlen <= 0 || a->nheads <= 0 || a->kdim <= 0 || a->vdim <= 0) return LQ_ERR_SHAPE;
  const int cs = a->chunk_size;
  if (cs != 64 && cs != 128 && cs != 192 && cs != 256) return LQ_ERR_SHAPE;
  return a->seqlen % cs == 0 ? LQ_OK : LQ_ERR_SHAPE;
}

// Offsets of the intermediates for the dims in `a` (chunk sizes above 64 keep the 64-token layouts)
Layout plan(const lq_zoo_simple_gla_args* a, bool scan) {
  Layout l;
  const int cs = a->chunk_size;
  const int64_t B = a->batch, T = a->seqlen, H = a->nheads, K = a->kdim, V = a->vdim, NT = T / 64;
  const bool codes = !scan && has_prologue(a);  // token-major local codes of q, k, v
  l.scan = scan;
  int64_t off = 0;
  auto take = [&](int64_t& slot, int64_t n) { slot = off, off += up(n); };
  take(l.kqT, B * NT * H * K * 64);
  take(l.vqT, B * NT * H * V * 64);
  take(l.gam, B * NT * H * K * 4);
  take(l.vcT, scan || codes ? B * NT * H * V * 64 : 0);
  take(l.qc, scan || codes ? B * NT * H * K * 64 : 0);
  take(l.kc, codes ? B * NT * H * K * 64 : 0);
  take(l.A, scan ? B * NT * H * 8192 : 0);
  take(l.gpk, scan ? B * NT * H * 256 : 0);
  take(l.gc, scan ? 0 : B * T * H * 4);
  take(l.ev, scan ? 0 : B * T * H * 4);
  take(l.h_i8, scan ? 0 : B * (T / cs) * H * V * K);
  take(l.cross, cs == 64 ? 0 : B * T * H * V * 4);
  l.total = off;
  return l;
}

bool scan_route(const lq_zoo_simple_gla_args* a) {
  return a->chunk_size == 64 && linear_scan(has_prologue(a), a->batch, a->seqlen, a->nheads, a->kdim, a->vdim);
}

}  // namespace

extern "C" int lq_zoo_simple_gla_workspace_bytes(const lq_zoo_simple_gla_args* a, int64_t* bytes) {
  if (!a || !bytes) return LQ_ERR_NULL;
  if (const int rc = check_dims(a)) return rc;
  *bytes = plan(a, scan_route(a)).total;
  if (a->chunk_size == 64 && has_prologue(a)) {  // its route depends on the tables' addresses too: enough for either
    const int64_t other = plan(a, !scan_route(a)).total;
    if (other > *bytes) *bytes = other;
  }
  return LQ_OK;
}

extern "C" int lq_zoo_simple_gla(const lq_zoo_simple_gla_args* a, hipStream_t stream) {
  if (!a || !a->q || !a->k || !a->v || !a->o || !a->workspace) return LQ_ERR_NULL;
  if (!a->sq || !a->sk || !a->skw || !a->svw || !a->svl || !a->ss) return LQ_ERR_NULL;
  if ((a->dq != nullptr) != (a->dq_rcp != nullptr)) return LQ_ERR_NULL;
  // what a call with a prologue may be does not depend on its route: checked here, in front of the first launch of either
  const bool prologue = has_prologue(a);
  if (prologue && a->chunk_size != 64) return LQ_ERR_SHAPE;
  if (!zoo_al(a->signs_qk, 16) || !zoo_al(a->signs_v, 16) || (a->signs_v && a->vdim != 64 && a->vdim != 128)) return LQ_ERR_SHAPE;
  int rc = check_dims(a);
  if (rc != LQ_OK) return rc;
  const Layout l = plan(a, scan_route(a) || (prologue && !staged_prologue(a)));
  if (a->workspace_bytes < l.total || ((uintptr_t)a->workspace % kAlign) != 0) return LQ_ERR_SHAPE;
  char* ws = (char*)a->workspace;
  const int decay = a->g ? LQ_DECAY_SCALAR : LQ_DECAY_NONE;
  if (a->chunk_size == 64 && (rc = check_scan(a->q, a->k, a->v, a->o, a->ss, a->svl, a->batch, a->seqlen, a->nheads, a->kdim, a->vdim, a->qmax, a->act_dtype)) != LQ_OK)
    return rc;
  if (l.scan) {
    const bool bf = a->act_dtype == LQ_DT_BF16;
    ZooLinPrepParams w = {};
    w.q = (const _Float16*)a->q, w.k = (const _Float16*)a->k, w.v = (const _Float16*)a->v, w.g = a->g;
    w.signs_qk = a->signs_qk, w.signs_v = a->signs_v, w.dq = a->dq, w.dq_rcp = a->dq_rcp;
    w.kqT = (int8_t*)(ws + l.kqT), w.vqT = (int8_t*)(ws + l.vqT), w.vcT = (int8_t*)(ws + l.vcT), w.qc = (int8_t*)(ws + l.qc);
    w.A = (_Float16*)(ws + l.A), w.gam = (float*)(ws + l.gam), w.gpk = (float*)(ws + l.gpk);
    w.sq = a->sq, w.sk = a->sk, w.skw = a->skw, w.svw = a->svw, w.svl = a->svl, w.eta = a->eta, w.scale = a->scale, w.qmax = a->qmax;
    w.B = a->batch, w.T = a->seqlen, w.H = a->nheads, w.V = a->vdim, w.NT = a->seqlen / 64;
    if ((rc = zoo_lin_prep_launch(w, a->kdim, bf, stream)) != LQ_OK) return rc;
    ZooScanParams s = {};
    s.kqT = w.kqT, s.vqT = w.vqT, s.vcT = w.vcT, s.gam = w.gam, s.qc = w.qc, s.A = w.A, s.gpk = w.gpk;
    s.o = a->o, s.o_is_f32 = a->o_is_f32, s.ht = a->ht;
    s.skw = a->skw, s.svw = a->svw, s.ss = a->ss, s.sq = a->sq, s.svl = a->svl;
    s.qmax = a->qmax, s.bf = bf, s.B = w.B, s.T = w.T, s.H = w.H, s.V = w.V, s.NT = w.NT;
    return zoo_scan_launch(s, false, decay, a->kdim, stream);
  }
  float* gc = a->g ? (float*)(ws + l.gc) : nullptr;

  // every stage validates its own arguments before it launches; the stages share the dims, so what the first accepts the
  // later ones accept as well, except for pointer alignment, which each checks on its own operands: a call refused by a
  // later stage has queued the earlier ones (they only write the workspace)
  if (a->g) {
    lq_zoo_cumsum_args c = {};
    c.g = a->g, c.gc = gc, c.batch = a->batch, c.seqlen = a->seqlen, c.nheads = a->nheads, c.kdim = 0, c.chunk_size = a->chunk_size;
    if ((rc = lq_zoo_cumsum(&c, stream)) != LQ_OK) return rc;
  }
  if (prologue) {
    lq_zoo_rotate_quant_args w = {};
    w.q = a->q, w.k = a->k, w.v = a->v, w.g = gc, w.qc = (int8_t*)(ws + l.qc), w.kc = (int8_t*)(ws + l.kc), w.vc = (int8_t*)(ws + l.vcT);
    w.kqT = (int8_t*)(ws + l.kqT), w.vqT = (int8_t*)(ws + l.vqT), w.ev = (float*)(ws + l.ev), w.gam = (float*)(ws + l.gam);
    w.dq = a->dq, w.dk = a->dq_rcp, w.signs_qk = a->signs_qk, w.signs_v = a->signs_v;
    w.sq = a->sq, w.sk = a->sk, w.svl = a->svl, w.skw = a->skw, w.svw = a->svw, w.eta = a->eta, w.scale = a->scale, w.qmax = a->qmax;
    w.batch = a->batch, w.seqlen = a->seqlen, w.nheads = a->nheads, w.kdim = a->kdim, w.vdim = a->vdim, w.chunk_size = 64;
    w.act_dtype = a->act_dtype;
    if ((rc = lq_zoo_rotate_quant(&w, stream)) != LQ_OK) return rc;
  } else {
    lq_zoo_write_codes_args w = {};
    w.key = a->k, w.val = a->v, w.g = gc, w.kqT = (int8_t*)(ws + l.kqT), w.vqT = (int8_t*)(ws + l.vqT);
    w.ev = (float*)(ws + l.ev), w.gam = (float*)(ws + l.gam), w.skw = a->skw, w.svw = a->svw, w.eta = a->eta, w.qmax = a->qmax;
    w.batch = a->batch, w.seqlen = a->seqlen, w.nheads = a->nheads, w.kdim = a->kdim, w.vdim = a->vdim, w.chunk_size = a->chunk_size;
    w.decay = decay, w.act_dtype = a->act_dtype;
    if ((rc = lq_zoo_write_codes(&w, stream)) != LQ_OK) return rc;
  }
  {
    lq_zoo_state_args s = {};
    s.kqT = (const int8_t*)(ws + l.kqT), s.vqT = (const int8_t*)(ws + l.vqT), s.gam = (const float*)(ws + l.gam);
    s.h_i8 = (int8_t*)(ws + l.h_i8), s.ht = a->ht, s.skw = a->skw, s.svw = a->svw, s.ss = a->ss, s.qmax = a->qmax;
    s.batch = a->batch, s.seqlen = a->seqlen, s.nheads = a->nheads, s.kdim = a->kdim, s.vdim = a->vdim, s.chunk_size = a->chunk_size;
    s.family = LQ_FAMILY_LINEAR, s.vtile = 0, s.act_dtype = a->act_dtype;
    if ((rc = lq_zoo_state(&s, stream)) != LQ_OK) return rc;
  }
  {
    lq_zoo_output_args o = {};
    o.q = a->q, o.k = a->k, o.v = a->v, o.h_i8 = (const int8_t*)(ws + l.h_i8), o.g = gc;
    if (prologue) o.qc = (const int8_t*)(ws + l.qc), o.kc = (const int8_t*)(ws + l.kc), o.vc = (const int8_t*)(ws + l.vcT);
    o.o = a->o, o.o_is_f32 = a->o_is_f32;
    o.sq = a->sq, o.sk = a->sk, o.svl = a->svl, o.ss = a->ss, o.scale = a->scale, o.qmax = a->qmax;
    o.batch = a->batch, o.seqlen = a->seqlen, o.nheads = a->nheads, o.kdim = a->kdim, o.vdim = a->vdim, o.chunk_size = a->chunk_size;
    o.decay = decay, o.act_dtype = a->act_dtype, o.cross = a->chunk_size == 64 ? nullptr : (float*)(ws + l.cross);
    if ((rc = lq_zoo_output(&o, stream)) != LQ_OK) return rc;
  }
  return LQ_OK;
}

// ---- the other cells: chunk_gla_int8 (linquant/kernels/zoo/gla.py:235-279), chunk_delta_int8
// (gated_delta_rule.py:159-203) and chunk_kda_int8 (kda.py:154-203) as one C entry over one workspace.  128-token chunks: the stage
// entry points in the order the Python wrappers issue them.  64-token chunks: recurrence and output in one launch (zoo_scan.hip: the bits
// of the stages, no stored states, no E in memory); in front of it under per-channel decay one launch for everything (zoo_diag_prep.h),
// otherwise the WY prep, which also cumulates a scalar decay and makes the write codes.  Neither family needs a rule.
// Delta: its step is two rendezvous and two dependent products with or without the output beside it, and the one launch was the faster at
// every size measured (B*H = 4 .. 256, T = 256 .. 16384, K = V = 64 and 128: 1.0 to 1.7 times with scalar decay and without, 1.0 to 1.56
// with per-channel decay; the most on few long chains).  GLA: more than 128 steps
// on less than half of the compute units took four launches while the pre-pass was two of them; against all four the two launches are,
// at T = 16384, K = V = 128, H = 4 / 12 / 28: 164 -> 152, 308 -> 229, 558 -> 389 us, K = V = 64, H = 4 / B2 H16: 115 -> 113, 326 -> 300; at
// T = 65536, K = V = 128, H = 1 / 4: 452 -> 445, 678 -> 655.  The slower ones are those of one or two heads of 64 key channels from 512
// steps on, by 2 to 7 % (T = 65536, V = 64, H = 1 / 2 / 4: 338 -> 362, 361 -> 382, 423 -> 423).
namespace {

struct FLayout {
  int64_t gc, logenv, kqT, vqT, vcT, wq, ev, gam, pack, gpk, A, Ax, qg, Hw, W, U, fw, e_out, h_i8, cross, total;
};

int fplan(const lq_zoo_chunk_forward_args* a, FLayout* l) {
  if (a->batch <= 0 || a->seqlen <= 0 || a->nheads <= 0 || a->kdim <= 0 || a->vdim <= 0) return LQ_ERR_SHAPE;
  const int cs = a->chunk_size;
  if ((cs != 64 && cs != 128) || a->seqlen % cs != 0) return LQ_ERR_SHAPE;
  if (a->family != LQ_FAMILY_LINEAR && a->family != LQ_FAMILY_DELTA) return LQ_ERR_SHAPE;
  if (a->decay < LQ_DECAY_NONE || a->decay > LQ_DECAY_DIAGONAL) return LQ_ERR_SHAPE;
  if (a->family == LQ_FAMILY_LINEAR && a->decay != LQ_DECAY_DIAGONAL) return LQ_ERR_SHAPE;  // lq_zoo_simple_gla serves those
  const bool delta = a->family == LQ_FAMILY_DELTA, diag = a->decay == LQ_DECAY_DIAGONAL, big = cs == 128;
  const int64_t B = a->batch, T = a->seqlen, H = a->nheads, K = a->kdim, V = a->vdim, NT = T / 64;
  int64_t off = 0;
  auto take = [&](int64_t& slot, int64_t n) { slot = off, off += up(n); };
  // (one launch in front of the recurrence: gc, logenv and Hw stay on the chip.  Scalar decay keeps gc's place, 4 bytes a token and
  // head, all the same: the size of a caller's workspace is part of the interface)
  take(l->gc, a->decay == LQ_DECAY_NONE || (diag && !big) ? 0 : B * T * H * (diag ? K : 1) * 4);
  take(l->logenv, diag && big ? B * T * H * 4 : 0);
  take(l->kqT, B * NT * H * K * 64);
  take(l->vqT, delta ? 0 : B * NT * H * V * 64);
  take(l->wq, delta ? B * T * H * K : 0);
  take(l->ev, big ? B * T * H * 4 : 0);
  take(l->gam, !big && delta ? 0 : B * NT * H * K * 4);  // (delta family: zoo_scan.hip reads them and fw from the pack)
  take(l->pack, delta && !big ? B * NT * H * (128 + K) * 4 : 0);
  take(l->A, diag || !big ? B * T * H * 64 * 2 : 0);
  take(l->Ax, diag && big ? B * T * H * 64 * 2 : 0);
  take(l->qg, diag || !big ? B * T * H * K : 0);
  take(l->gpk, a->decay == LQ_DECAY_SCALAR && !big ? B * NT * H * 64 * 4 : 0);
  take(l->vcT, !big && !delta ? B * NT * H * V * 64 : 0);
  take(l->Hw, delta && big ? B * T * H * K * 2 : 0);
  take(l->W, delta && big ? B * T * H * K * 2 : 0);
  take(l->U, delta ? B * T * H * V * 2 : 0);
  take(l->fw, delta && big ? B * T * H * 4 : 0);
  take(l->e_out, delta && big ? B * T * H * V * 2 : 0);
  take(l->h_i8, big ? B * (T / cs) * H * V * K : 0);
  take(l->cross, big ? B * T * H * V * 4 : 0);
  l->total = off;
  return LQ_OK;
}

// R_QK laid out as operands by a launch of its own (2 us in a stream of launches), or read by every chunk and head as the caller holds it (32
// requests of 4 or, fp32, 8 bytes a lane at K = 128, rows apart, in the place of eight of 16)?  GPU us of the whole call, as it is / laid out
// (H 16 or 32, 64 value columns):
//   chunks and heads     1024            2048            4096            8192
//   GLA fp32, K = 64     41.0 / 41.8     64.7 / 62.5     118 / 111       233 / 216
//             K = 128    58.4 / 57.1     98.3 / 91.7     185 / 169       349 / 312
//   KDA fp32, K = 64     75.2 / 76.3     104.6 / 103.9   179 / 172       342 / 323
//             K = 128    100.9 / 100.1   146.1 / 143.0   269 / 253       489 / 455
//   GLA fp16, K = 64     40.0 / 41.7     61.0 / 62.5     110.2 / 111.3   218.0 / 215.6
//             K = 128    55.1 / 57.1     90.6 / 92.1     169.5 / 168.5   315.2 / 311.9
//   KDA fp16, K = 64     74.5 / 76.3     103.0 / 104.0   172.0 / 171.6   326.2 / 322.2
//             K = 128    99.2 / 100.4    142.8 / 143.0   254.9 / 252.2   460.5 / 455.2
bool rot_operand(const lq_zoo_chunk_forward_args* a) {
  return (int64_t)a->batch * a->nheads * (a->seqlen / 64) >= (a->rot_f32 ? 1024 : 4096);
}

}  // namespace

extern "C" int lq_zoo_chunk_forward_workspace_bytes(const lq_zoo_chunk_forward_args* a, int64_t* bytes) {
  if (!a || !bytes) return LQ_ERR_NULL;
  FLayout l;
  const int rc = fplan(a, &l);
  if (rc != LQ_OK) return rc;
  *bytes = l.total;
  return LQ_OK;
}

extern "C" int lq_zoo_chunk_forward(const lq_zoo_chunk_forward_args* a, hipStream_t stream) {
  if (!a || !a->q || !a->k || !a->v || !a->o || !a->workspace) return LQ_ERR_NULL;
  if (!a->sq || !a->skw || !a->svw || !a->svl || !a->ss) return LQ_ERR_NULL;
  FLayout l;
  int rc = fplan(a, &l);
  if (rc != LQ_OK) return rc;
  const bool delta = a->family == LQ_FAMILY_DELTA, diag = a->decay == LQ_DECAY_DIAGONAL, big = a->chunk_size == 128;
  if (a->decay != LQ_DECAY_NONE && !a->g) return LQ_ERR_NULL;
  if (delta && (!a->beta || !a->sw)) return LQ_ERR_NULL;
  if (!a->sk) return LQ_ERR_NULL;
  if ((a->dq != nullptr) != (a->dq_rcp != nullptr)) return LQ_ERR_NULL;
  if ((a->dq || a->dqk) && (!delta || !diag || big)) return LQ_ERR_SHAPE;  // D_QK at load: KDA, 64-token chunks
  if (a->rot && !diag) return LQ_ERR_SHAPE;
  if (a->rot_f32 && (!diag || big)) return LQ_ERR_SHAPE;  // rounded in the launch in front of the recurrence
  if ((a->rot && a->rot_f32) || (a->dq && a->dqk)) return LQ_ERR_SHAPE;
  if (!big && (rc = check_scan(a->q, a->k, a->v, a->o, a->ss, a->svl, a->batch, a->seqlen, a->nheads, a->kdim, a->vdim, a->qmax, a->act_dtype)) != LQ_OK)
    return rc;
  if (a->workspace_bytes < l.total || ((uintptr_t)a->workspace % kAlign) != 0) return LQ_ERR_SHAPE;
  char* ws = (char*)a->workspace;
  float* gc = a->decay != LQ_DECAY_NONE && big ? (float*)(ws + l.gc) : nullptr;
  float* logenv = diag && big ? (float*)(ws + l.logenv) : nullptr;
  int8_t* kqT = (int8_t*)(ws + l.kqT);
  int8_t* vqT = delta ? nullptr : (int8_t*)(ws + l.vqT);
  int8_t* wq = delta ? (int8_t*)(ws + l.wq) : nullptr;
  float* ev = big ? (float*)(ws + l.ev) : nullptr;
  float* gam = !big && delta ? nullptr : (float*)(ws + l.gam);
  float* pack = delta && !big ? (float*)(ws + l.pack) : nullptr;
  void* Hw = delta && big ? ws + l.Hw : nullptr;
  void* W = delta && big ? ws + l.W : nullptr;
  void* U = delta ? ws + l.U : nullptr;
  float* fw = delta && big ? (float*)(ws + l.fw) : nullptr;
  void* e_out = delta && big ? ws + l.e_out : nullptr;
  int8_t* h_i8 = (int8_t*)(ws + l.h_i8);
  void* A = diag || !big ? ws + l.A : nullptr;
  void* Ax = diag && big ? ws + l.Ax : nullptr;
  int8_t* qg = diag || !big ? (int8_t*)(ws + l.qg) : nullptr;
  float* gpk = a->decay == LQ_DECAY_SCALAR && !big ? (float*)(ws + l.gpk) : nullptr;
  int8_t* vcT = !big && !delta ? (int8_t*)(ws + l.vcT) : nullptr;
  float* cross = big ? (float*)(ws + l.cross) : nullptr;

  if (diag && !big) {  // everything in front of the recurrence in one launch
    for (const void* x : {(const void*)a->rot, (const void*)a->rot_f32, (const void*)a->dq, (const void*)a->dq_rcp, (const void*)a->dqk,
                          (const void*)a->rot_ws, delta ? (const void*)a->skw : nullptr})
      if (!zoo_al(x, 16)) return LQ_ERR_SHAPE;
    ZooDiagParams d = {};
    d.q = (const _Float16*)a->q, d.k = (const _Float16*)a->k, d.v = (const _Float16*)a->v, d.g = a->g, d.beta = a->beta;
    if ((a->rot || a->rot_f32) && a->rot_ws && rot_operand(a)) {
      if ((rc = zoo_rot_operand_launch(a->rot_f32 ? a->rot_f32 : a->rot, a->rot_f32, (_Float16*)a->rot_ws, a->kdim, stream)) != LQ_OK) return rc;
      d.rot_op = (const _Float16*)a->rot_ws;
    }
    d.rot = (const _Float16*)a->rot, d.rot_f = a->rot_f32, d.dq = d.dk_div = a->dqk ? a->dqk : a->dq, d.dk_rcp = a->dq_rcp;
    d.sq = a->sq, d.sk = a->sk, d.skw = a->skw, d.sw = a->sw, d.svw = a->svw, d.svl = a->svl;
    d.A = (_Float16*)A, d.qc = qg, d.kqT = kqT, d.wq = wq, d.vqT = vqT, d.vcT = vcT, d.U = (_Float16*)U, d.gam = gam, d.pack = pack;
    d.sigma = a->sigma, d.tau = a->tau, d.eta = a->eta, d.scale = a->scale, d.qmax = a->qmax, d.bf = a->act_dtype == LQ_DT_BF16;
    d.B = a->batch, d.T = a->seqlen, d.H = a->nheads, d.V = a->vdim, d.NT = a->seqlen / 64;
    rc = delta ? zoo_diag_kda_launch(d, a->kdim, stream) : zoo_diag_gla_launch(d, a->kdim, stream);
    if (rc != LQ_OK) return rc;
  }
  // (every stage validates its own arguments before it launches: see lq_zoo_simple_gla)
  if (a->decay != LQ_DECAY_NONE && big) {
    lq_zoo_cumsum_args c = {};
    c.g = a->g, c.gc = gc, c.logenv = logenv, c.batch = a->batch, c.seqlen = a->seqlen, c.nheads = a->nheads;
    c.kdim = diag ? a->kdim : 0, c.chunk_size = a->chunk_size;
    if ((rc = lq_zoo_cumsum(&c, stream)) != LQ_OK) return rc;
  }
  if (delta && (big || !diag)) {
    lq_zoo_wy_prep_args w = {};
    w.k = a->k, w.v = a->v, w.beta = a->beta, w.g = big ? gc : a->g, w.Hw = Hw, w.W = W, w.U = U, w.fw = fw, w.sigma = a->sigma, w.tau = a->tau;
    w.batch = a->batch, w.seqlen = a->seqlen, w.nheads = a->nheads, w.kdim = a->kdim, w.vdim = a->vdim, w.chunk_size = a->chunk_size;
    w.decay = a->decay, w.act_dtype = a->act_dtype;
    if (!big) {  // the write operands come with the transform
      w.kqT = kqT, w.wq = wq, w.ev = ev, w.gam = gam, w.skw = a->skw, w.sw = a->sw, w.eta = a->eta, w.qmax = a->qmax, w.pack = pack;
    }
    const ZooWyLocal local = {a->q, qg, A, gpk, a->sq, a->sk, a->scale};
    if ((rc = zoo_wy_prep_launch(&w, !big, big ? nullptr : &local, stream)) != LQ_OK) return rc;
  }
  if (big) {
    lq_zoo_write_codes_args w = {};
    w.key = delta ? Hw : a->k, w.val = delta ? nullptr : a->v, w.w = W, w.g = gc, w.logenv = logenv, w.kqT = kqT, w.vqT = vqT, w.wq = wq;
    w.ev = ev, w.gam = gam, w.skw = a->skw, w.svw = delta ? nullptr : a->svw, w.sw = a->sw, w.eta = a->eta, w.qmax = a->qmax;
    w.batch = a->batch, w.seqlen = a->seqlen, w.nheads = a->nheads, w.kdim = a->kdim, w.vdim = a->vdim, w.chunk_size = a->chunk_size;
    w.decay = a->decay, w.act_dtype = a->act_dtype;
    if ((rc = lq_zoo_write_codes(&w, stream)) != LQ_OK) return rc;
  }
  if (diag && big) {
    lq_zoo_gla_A_args g = {};
    g.q = a->q, g.k = delta ? Hw : a->k, g.g = gc, g.A = A, g.qg = qg, g.rot = a->rot, g.sq = a->sq, g.sk = a->sk, g.scale = a->scale;
    g.qmax = a->qmax, g.batch = a->batch, g.seqlen = a->seqlen, g.nheads = a->nheads, g.kdim = a->kdim, g.chunk_size = a->chunk_size;
    g.act_dtype = a->act_dtype, g.dq = a->dq, g.A_cross = Ax;
    if ((rc = lq_zoo_gla_A(&g, stream)) != LQ_OK) return rc;
  }
  if (!big) {
    ZooScanParams s = {};
    s.kqT = kqT, s.vqT = vqT, s.vcT = vcT, s.wq = wq, s.u = (const _Float16*)U, s.pack = pack, s.gam = gam;
    s.qc = qg, s.A = (const _Float16*)A, s.gpk = gpk, s.o = a->o, s.o_is_f32 = a->o_is_f32, s.ht = a->ht;
    s.skw = a->skw, s.svw = a->svw, s.sw = a->sw, s.ss = a->ss, s.sq = a->sq, s.svl = a->svl;
    s.qmax = a->qmax, s.bf = a->act_dtype == LQ_DT_BF16;
    s.B = a->batch, s.T = a->seqlen, s.H = a->nheads, s.V = a->vdim, s.NT = a->seqlen / 64;
    return zoo_scan_launch(s, delta, a->decay, a->kdim, stream);
  }
  {
    lq_zoo_state_args s = {};
    s.kqT = kqT, s.vqT = vqT, s.wq = wq, s.u = U, s.fw = fw, s.ev = delta ? ev : nullptr, s.gam = gam, s.h_i8 = h_i8, s.e_out = e_out;
    s.ht = a->ht, s.skw = a->skw, s.svw = a->svw, s.sw = a->sw, s.ss = a->ss, s.qmax = a->qmax;
    s.batch = a->batch, s.seqlen = a->seqlen, s.nheads = a->nheads, s.kdim = a->kdim, s.vdim = a->vdim, s.chunk_size = a->chunk_size;
    s.family = a->family, s.vtile = 0, s.act_dtype = a->act_dtype, s.pack = pack;
    if ((rc = lq_zoo_state(&s, stream)) != LQ_OK) return rc;
  }
  {
    lq_zoo_output_args o = {};
    o.q = diag ? nullptr : a->q, o.qg = qg, o.k = diag ? nullptr : (delta ? Hw : a->k), o.v = delta ? e_out : a->v, o.h_i8 = h_i8;
    o.g = diag ? nullptr : gc, o.A = A, o.o = a->o, o.o_is_f32 = a->o_is_f32, o.sq = a->sq, o.sk = a->sk, o.svl = a->svl, o.ss = a->ss;
    o.scale = a->scale, o.qmax = a->qmax;
    o.batch = a->batch, o.seqlen = a->seqlen, o.nheads = a->nheads, o.kdim = a->kdim, o.vdim = a->vdim, o.chunk_size = a->chunk_size;
    o.decay = a->decay, o.act_dtype = a->act_dtype, o.cross = cross, o.A_cross = Ax;
    if ((rc = lq_zoo_output(&o, stream)) != LQ_OK) return rc;
  }
  return LQ_OK;
}
