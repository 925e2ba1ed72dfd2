// The dt pipeline of the Mamba-2 SSD (mamba2_cumsum.hip) as a workgroup's function, shared by its stand-alone launch and the one that
// runs C.B^T beside it (mamba2_cumsum_bmm.hip).
#pragma once

#include "lq_common.h"
#include "../../include/linquant_hip.h"

namespace {

constexpr int kMaxE = 16;  // chunk sizes up to 1024

LQ_DEV float load_dt(const void* p, int64_t off, int dtype) {
  if (dtype == LQ_DT_F16) return (float)((const _Float16*)p)[off];
  if (dtype == LQ_DT_F32) return ((const float*)p)[off];
  return (float)((const int8_t*)p)[off];
}

constexpr int kHG = 16;   // heads per workgroup: one token row of the tile is 16 adjacent heads (32 bytes of fp16 dt)
constexpr int kWaves = 8;  // two heads per wave

// Which (head group, chunk, batch) a workgroup of the flat grid works on.  Workgroups are dealt to the 8 XCDs round-robin
// in launch order, and the head groups of one (chunk, batch) read the same 128-byte lines of dt (a token row of 80 heads
// is 160 bytes): on consecutive workgroups every XCD's L2 fetched those lines from HBM for itself (21 MB read for 5 MB
// of dt).  Workgroup 8 j + x takes head group j % hg of unit 8 (j / hg) + x, so a unit's head groups share one XCD.
struct Where {
  int h0, c, b;
};
LQ_DEV Where where(uint32_t block, int hg, int nchunks, int by_xcd) {
  uint32_t unit, grp;
  if (by_xcd) {
    const uint32_t x = block & 7u, j = block >> 3;
    const uint32_t uh = j / (uint32_t)hg;
    grp = j - uh * (uint32_t)hg, unit = uh * 8u + x;
  } else {
    unit = block / (uint32_t)hg, grp = block - unit * (uint32_t)hg;
  }
  Where w;
  w.b = (int)(unit / (uint32_t)nchunks), w.c = (int)(unit - (uint32_t)w.b * (uint32_t)nchunks), w.h0 = (int)grp * kHG;
  return w;
}

// A workgroup's tile for chunk sizes of 64 E tokens with E known at compile time (1, 2, 4, 8): every dt of the tile, A_log and
// the bias are requested before the first use, outside any branch (in the generic kernel of mamba2_cumsum.hip each staging iteration and each
// head waits for its own load), the element loops have no run-time bounds, and a lane's E outputs leave as one vector
// store when E is 2 or 4.
struct CumsumParams {
  const void* dt_in;
  int dt_dtype;
  int64_t sdt_b, sdt_l, sdt_h;
  const float* dt_scale;
  const int8_t* a_log;
  int64_t sa_h;
  const float* a_log_scale;
  const float* dt_bias;
  int64_t sbias_h;
  float* dt_out;
  float* dA_cs;
  int seqlen, nheads, nchunks, softplus;
  float dt_min, dt_max;
  int hg, by_xcd;
};

// tile: [Q][kHG + 1] raw dt as float, in LDS
template <int E>
LQ_DEV void chunk_cumsum_fixed(const CumsumParams& p, uint32_t block, float* tile) {
  constexpr int Q = 64 * E, NIT = Q * kHG / (kWaves * 64);
  const Where wh = where(block, p.hg, p.nchunks, p.by_xcd);
  const int h0 = wh.h0, c = wh.c, b = wh.b;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int limit = min(Q, p.seqlen - c * Q);
  // ---- requests: the (token, head) tile (consecutive lanes read consecutive heads of one token; positions past the
  // sequence end or the last head re-read a valid neighbour and are zeroed below), then the per-head constants
  // The tile's first element is a scalar; a lane's offset from it fits 32 bits in bytes and its factors 24 (cumsum_fixed_e), a multiply of
  // full rate: 64-bit products for each request were 47 vector instructions of a quarter of it.
  float raw[NIT];
  uint32_t offs[NIT];
  const int64_t first = (int64_t)b * p.sdt_b + (int64_t)c * Q * p.sdt_l + (int64_t)h0 * p.sdt_h;
  const uint32_t hoff = __umul24((uint32_t)min(tid % kHG, p.nheads - 1 - h0), (uint32_t)p.sdt_h);
#pragma unroll
  for (int i = 0; i < NIT; ++i) offs[i] = __umul24((uint32_t)min((tid + i * kWaves * 64) / kHG, limit - 1), (uint32_t)p.sdt_l) + hoff;
  if (p.dt_dtype == LQ_DT_F16) {  // one uniform branch around all requests of a dtype, not one per request
    _Float16 r[NIT];
#pragma unroll
    for (int i = 0; i < NIT; ++i) r[i] = *(const _Float16*)((const char*)((const _Float16*)p.dt_in + first) + 2u * offs[i]);
#pragma unroll
    for (int i = 0; i < NIT; ++i) raw[i] = (float)r[i];
  } else if (p.dt_dtype == LQ_DT_F32) {
#pragma unroll
    for (int i = 0; i < NIT; ++i) raw[i] = *(const float*)((const char*)((const float*)p.dt_in + first) + 4u * offs[i]);
  } else {
    int8_t r[NIT];
#pragma unroll
    for (int i = 0; i < NIT; ++i) r[i] = *((const int8_t*)p.dt_in + first + offs[i]);
#pragma unroll
    for (int i = 0; i < NIT; ++i) raw[i] = (float)r[i];
  }
  int8_t alog[kHG / kWaves];
  float bias[kHG / kWaves];
#pragma unroll
  for (int hw = 0; hw < kHG / kWaves; ++hw) {
    const int h = min(h0 + wave * (kHG / kWaves) + hw, p.nheads - 1);
    alog[hw] = p.a_log[(int64_t)h * p.sa_h];
    bias[hw] = p.dt_bias ? p.dt_bias[(int64_t)h * p.sbias_h] : 0.0f;
  }
  const float dt_scale = *p.dt_scale;
  const float a_scale = *p.a_log_scale;
#pragma unroll
  for (int i = 0; i < NIT; ++i) {
    const int it = tid + i * kWaves * 64;
    const int pos = it / kHG, hh = it % kHG;
    tile[pos * (kHG + 1) + hh] = (pos < limit && h0 + hh < p.nheads) ? raw[i] : 0.0f;
  }
  __syncthreads();
#pragma unroll
  for (int hw = 0; hw < kHG / kWaves; ++hw) {
    const int hh = wave * (kHG / kWaves) + hw;
    const int h = h0 + hh;
    if (h >= p.nheads) continue;
    const float A = -lq_expf(a_scale * (float)alog[hw]);
    float dtv[E], pre[E];
    float run = 0.0f;
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int pos = lane * E + i;
      float v = dt_scale * tile[pos * (kHG + 1) + hh];
      if (p.dt_bias) v = v + bias[hw];
      if (p.softplus) v = (v > 20.0f) ? v : lq_logf(1.0f + lq_expf(v));
      v = fminf(fmaxf(v, p.dt_min), p.dt_max);
      v = pos < limit ? v : 0.0f;
      dtv[i] = v;
      const float dA = v * A;
      run = (i == 0) ? dA : run + dA;
      pre[i] = run;
    }
    float t = run;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float up = __shfl_up(t, off, 64);
      if (lane >= off) t = t + up;
    }
    float ex = __shfl_up(t, 1, 64);
    if (lane == 0) ex = 0.0f;
    const int64_t base = (((int64_t)b * p.nheads + h) * p.nchunks + c) * Q;
    char* const dto = (char*)(p.dt_out + base);
    char* const dAo = (char*)(p.dA_cs + base);
    const uint32_t at = 4u * E * lane;
    if constexpr (E == 4) {
      *(lq_v4f*)(dto + at) = lq_v4f{dtv[0], dtv[1], dtv[2], dtv[3]};
      *(lq_v4f*)(dAo + at) = lq_v4f{ex + pre[0], ex + pre[1], ex + pre[2], ex + pre[3]};
    } else {
#pragma unroll
      for (int i = 0; i < E; ++i) {
        *(float*)(dto + (at + 4u * i)) = dtv[i];
        *(float*)(dAo + (at + 4u * i)) = ex + pre[i];
      }
    }
  }
}

// Parameters of a call and its workgroups, or the reason to refuse it
inline int cumsum_plan(const lq_chunk_cumsum_args* a, CumsumParams* p, uint32_t* blocks) {
  if (!a || !a->dt || !a->dt_scale || !a->A_log || !a->A_log_scale || !a->dt_out || !a->dA_cumsum) return LQ_ERR_NULL;
  if (a->batch <= 0 || a->seqlen <= 0 || a->nheads <= 0 || a->batch > 65535) return LQ_ERR_SHAPE;
  const int Q = a->chunk_size;
  if (Q < 64 || Q % 64 != 0 || Q > 64 * kMaxE) return LQ_ERR_SHAPE;
  if (a->dt_dtype != LQ_DT_F16 && a->dt_dtype != LQ_DT_F32 && a->dt_dtype != LQ_DT_I8) return LQ_ERR_SHAPE;
  const int nchunks = (a->seqlen + Q - 1) / Q;
  if (nchunks > 65535) return LQ_ERR_SHAPE;
  const int hg = (a->nheads + kHG - 1) / kHG;
  const int64_t units = (int64_t)nchunks * a->batch;
  if (units * hg >= (1ll << 31)) return LQ_ERR_SHAPE;
  const int by_xcd = units % 8 == 0;
  *p = CumsumParams{a->dt, a->dt_dtype, a->dt_stride_b, a->dt_stride_l, a->dt_stride_h, a->dt_scale, a->A_log, a->A_log_stride_h,
                    a->A_log_scale, a->dt_bias, a->dt_bias_stride_h, a->dt_out, a->dA_cumsum, a->seqlen, a->nheads, nchunks,
                    a->dt_softplus, a->dt_min, a->dt_max, hg, by_xcd};
  *blocks = (uint32_t)(units * hg);
  return LQ_OK;
}

// E = Q / 64 where chunk_cumsum_fixed takes the call, else 0
inline int cumsum_fixed_e(const lq_chunk_cumsum_args* a) {
  const int Q = a->chunk_size;
  const bool vec_ok = ((uintptr_t)a->dt_out % 16 == 0) && ((uintptr_t)a->dA_cumsum % 16 == 0);
  // lane offsets of the tile: 24-bit factors, 32 bits of bytes
  const int64_t sl = a->dt_stride_l, sh = a->dt_stride_h;
  if (sl < 0 || sh < 0 || sl >= (1 << 24) || sh >= (1 << 24) || (Q - 1) * sl + (kHG - 1) * sh >= (1ll << 30)) return 0;
  return Q == 64 || Q == 128 || Q == 512 || (Q == 256 && vec_ok) ? Q / 64 : 0;
}

}  // namespace
