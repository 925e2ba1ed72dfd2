// Entry point of the intra-chunk product under per-channel (diagonal) decay, 16-token sub-blocks: _gla_A_inter
// (linquant/kernels/zoo/gla.py:27-63) and _gla_A_intra (gla.py:66-99).  The kernel is the DIAG_A form of zoo_diag_prep.h; 128-token
// chunks take their blocks between the halves from zoo_gla_A_cross.hip.
#include "zoo_params.h"
#include "../../include/linquant_hip.h"

extern "C" int lq_zoo_gla_A(const lq_zoo_gla_A_args* a, hipStream_t stream) {
  if (!a || !a->q || !a->k || !a->g || !a->A || !a->sq || !a->sk) return LQ_ERR_NULL;
  if (a->batch <= 0 || a->seqlen <= 0 || a->nheads <= 0) return LQ_ERR_SHAPE;
  // 128-token chunks: the blocks inside either half are those of 64-token chunks (g cumulated over the 128 tokens), the
  // blocks between the halves come from a second launch into A_cross
  const bool pair = a->chunk_size == 128;
  if (pair && !a->A_cross) return LQ_ERR_NULL;
  if (pair && !zoo_al(a->A_cross, 16)) return LQ_ERR_SHAPE;
  if ((a->chunk_size != 64 && !pair) || a->seqlen % a->chunk_size != 0) return LQ_ERR_SHAPE;
  if (a->kdim != 64 && a->kdim != 128) return LQ_ERR_SHAPE;
  if (a->qmax < 1 || a->qmax > 127) return LQ_ERR_SHAPE;
  if (a->act_dtype != LQ_DT_F16 && a->act_dtype != LQ_DT_BF16) return LQ_ERR_SHAPE;
  if (!zoo_al(a->q, 16) || !zoo_al(a->k, 16) || !zoo_al(a->g, 16) || !zoo_al(a->A, 16) || (a->qg && !zoo_al(a->qg, 8)))
    return LQ_ERR_SHAPE;
  if (a->rot && !zoo_al(a->rot, 16)) return LQ_ERR_SHAPE;
  if (a->dq && !zoo_al(a->dq, 16)) return LQ_ERR_SHAPE;
  if ((int64_t)a->batch * a->nheads > 65535) return LQ_ERR_SHAPE;
  if ((int64_t)(a->seqlen / 64) * a->batch * a->nheads > 0x7fffffff) return LQ_ERR_SHAPE;
  ZooDiagParams p = {};
  p.q = (const _Float16*)a->q, p.k = (const _Float16*)a->k, p.g = a->g, p.A = (_Float16*)a->A, p.qc = a->qg;
  p.dq = a->dq, p.sq = a->sq, p.sk = a->sk, p.rot = (const _Float16*)a->rot, p.scale = a->scale, p.qmax = a->qmax;
  p.bf = a->act_dtype == LQ_DT_BF16;
  p.B = a->batch, p.T = a->seqlen, p.H = a->nheads, p.NT = a->seqlen / 64;
  const int rc = zoo_diag_a_launch(p, a->kdim, stream);
  if (rc || !pair) return rc;
  ZooACrossParams c = {};
  c.q = p.q, c.k = p.k, c.g = p.g, c.Ax = (_Float16*)a->A_cross, c.sq = p.sq, c.sk = p.sk, c.rot = p.rot, c.dq = p.dq;
  c.scale = p.scale, c.qmax = p.qmax, c.bf = p.bf, c.B = p.B, c.T = p.T, c.H = p.H;
  return zoo_gla_A_cross_launch(c, a->kdim, stream);
}
