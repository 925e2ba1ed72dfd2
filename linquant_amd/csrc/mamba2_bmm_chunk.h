// The C.B^T tile of the Mamba-2 SSD (mamba2_bmm_chunk.hip) as a wave's function, shared by its stand-alone launch and the one that
// runs it beside the cumulative sum (mamba2_cumsum_bmm.hip).
#pragma once

#include "lq_common.h"
#include "../../include/linquant_hip.h"

namespace {

typedef uint32_t lq_v2u __attribute__((ext_vector_type(2)));

// clamp to [-127, 127] then round half even; returns a dword whose low byte is the INT8 code
LQ_DEV uint32_t rint_code(float y) {
  const float c = __builtin_amdgcn_fmed3f(y, -127.0f, 127.0f);
  return __float_as_uint(c + 12582912.0f);
}

LQ_DEV uint32_t pack_low_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  const uint32_t lo = __builtin_amdgcn_perm(b, a, 0x0c0c0400u);  // {a.b0, b.b0, 0, 0}
  const uint32_t hi = __builtin_amdgcn_perm(d, c, 0x04000c0cu);  // {0, 0, c.b0, d.b0}
  return lo | hi;
}

// One wavefront per 64 x 64 output tile.  N64 = N / 64 contraction steps, all of whose operands are requested before
// the first is used, from clamped (always valid) rows: a request inside `if (row < limit)` is waited for where the
// branches join, and a run-time loop over N put a second memory round trip behind the first.  Rows past the sequence
// end are zeroed after the fact.  The epilogue transposes each lane's 4 x 4 block of code dwords across the four lane
// groups so that a lane stores 16 contiguous bytes: 4 stores per lane instead of 16, 64 contiguous bytes per row.
struct BmmParams {
  const int8_t* a;
  int64_t sa_b, sa_l, sa_g;
  const void* bv;
  int64_t sb_b, sb_l, sb_g;
  const float* a_scale;
  const float* b_scale;
  const float* cb_scale;
  int8_t* out;
  int seqlen, G, Q, nchunks;
  uint32_t tiles_magic, g_magic, tpc, tpc_magic, ncg, ncg_magic;
  int by_xcd;
  int causal;      // only the tiles on and below the diagonal
  uint32_t tiles;  // in all
};

// Tile number j of XCD x where the units are dealt to the XCDs (by_xcd), else tile number j of all
template <bool B_IS_FP, int N64>
LQ_DEV void bmm_chunk_tile(const BmmParams& p, uint32_t x, uint32_t j, int lane) {
  const int rl = lane & 15, kg = lane >> 4;
  const int Q = p.Q, G = p.G;
  // floor(2^32 / d) + 1 multipliers (0 for d == 1) stand in for the run-time divisions (exact while x * d < 2^32, which
  // the launcher checks).
  // Workgroups are dealt to the 8 XCDs round-robin in launch order, and the tpc tiles of one (batch, chunk, group) read
  // the same C and B rows: with consecutive workgroups on consecutive tiles every XCD's L2 fetched those rows from HBM
  // for itself (33.7 MB read for 12.6 MB of operands).  Workgroup 8 j + x takes tile j % tpc of unit 8 (j / tpc) + x, so
  // a unit's tiles run on one XCD, one after the other.
  const uint32_t uh = p.tpc_magic ? __umulhi(j, p.tpc_magic) : j;
  const uint32_t tile = j - uh * p.tpc, unit = p.by_xcd ? uh * 8u + x : uh;
  int mt64, kt64;
  if (p.causal) {  // (wave-uniform, at most eight rows of tiles)
    mt64 = 0, kt64 = (int)tile;
    while (kt64 > mt64) kt64 -= ++mt64;
  } else {
    mt64 = p.tiles_magic ? (int)__umulhi(tile, p.tiles_magic) : (int)tile;
    kt64 = (int)tile - mt64 * (Q >> 6);
  }
  const int b = p.ncg_magic ? (int)__umulhi(unit, p.ncg_magic) : (int)unit;
  const uint32_t cg = unit - (uint32_t)b * p.ncg;
  const int c = p.g_magic ? (int)__umulhi(cg, p.g_magic) : (int)cg;
  const int g = (int)cg - c * G;
  const int limit = min(Q, p.seqlen - c * Q);
  const float a_sc = p.a_scale[g], b_sc = p.b_scale[g], cb_sc = p.cb_scale[g];

  const int8_t* ap = p.a + (int64_t)b * p.sa_b + (int64_t)c * Q * p.sa_l + (int64_t)g * p.sa_g;
  const char* bp = (const char*)p.bv + ((int64_t)b * p.sb_b + (int64_t)c * Q * p.sb_l + (int64_t)g * p.sb_g) * (B_IS_FP ? 2 : 1);
  const uint32_t sal = (uint32_t)p.sa_l, sbl = (uint32_t)p.sb_l * (B_IS_FP ? 2u : 1u);
  lq_v4i cop[N64][4], braw[N64][4][B_IS_FP ? 2 : 1];
  bool mlive[4], klive[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = mt64 * 64 + i * 16 + rl, k = kt64 * 64 + i * 16 + rl;
    mlive[i] = m < limit, klive[i] = k < limit;
    const uint32_t mo = __umul24((uint32_t)min(m, limit - 1), sal) + (uint32_t)kg * 16u;
    const uint32_t ko = __umul24((uint32_t)min(k, limit - 1), sbl) + (uint32_t)kg * (B_IS_FP ? 32u : 16u);
#pragma unroll
    for (int n = 0; n < N64; ++n) {
      cop[n][i] = *(const lq_v4i*)(ap + mo + 64u * n);
      braw[n][i][0] = *(const lq_v4i*)(bp + ko + (B_IS_FP ? 128u : 64u) * n);
      if (B_IS_FP) braw[n][i][1] = *(const lq_v4i*)(bp + ko + 128u * n + 16u);
    }
  }
  const float b_inv = 1.0f / b_sc;
  const float inv_scb = (a_sc * b_sc) / cb_sc;

  lq_v4i acc[4][4];  // [k tile][m tile]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = lq_v4i{0, 0, 0, 0};
#pragma unroll
  for (int n = 0; n < N64; ++n) {
    lq_v4i bop[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (!mlive[i]) cop[n][i] = lq_v4i{0, 0, 0, 0};
      if (B_IS_FP) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const lq_v8h hv = __builtin_bit_cast(lq_v8h, braw[n][i][d >> 1]);
          uint32_t cd[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) cd[e] = rint_code((float)hv[4 * (d & 1) + e] * b_inv);
          bop[i][d] = (int)pack_low_bytes(cd[0], cd[1], cd[2], cd[3]);
        }
      } else {
        bop[i] = braw[n][i][0];
      }
      if (!klive[i]) bop[i] = lq_v4i{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = lq_mfma_i8(bop[i], cop[n][j], acc[i][j]);
  }

  int8_t* op = p.out + ((((int64_t)b * p.nchunks + c) * G + g) * Q) * Q + (int64_t)(mt64 * 64) * Q + kt64 * 64;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    // accumulator rows = k (4 consecutive per lane: k = 16 i + 4 kg + r), column = m = 16 j + rl
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t cd[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) cd[r] = rint_code((float)acc[i][j][r] * inv_scb);
      d[i] = pack_low_bytes(cd[0], cd[1], cd[2], cd[3]);
    }
    // dword i of lane group kg covers k = 16 i + 4 kg ..: transposing register index with lane group leaves lane group
    // kg with the four dwords of k = 16 kg .. 16 kg + 15
    lq_v2u t;
    t = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false), d[0] = t[0], d[2] = t[1];
    t = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false), d[1] = t[0], d[3] = t[1];
    t = __builtin_amdgcn_permlane16_swap(d[0], d[1], false, false), d[0] = t[0], d[1] = t[1];
    t = __builtin_amdgcn_permlane16_swap(d[2], d[3], false, false), d[2] = t[0], d[3] = t[1];
    *(lq_v4i*)(op + (uint32_t)((16 * j + rl) * Q + 16 * kg)) = lq_v4i{(int)d[0], (int)d[1], (int)d[2], (int)d[3]};
  }
}

inline bool bmm_al(const void* q, int n) { return ((uintptr_t)q % n) == 0; }

// Parameters of a call (causal: for a caller that reads nothing above the diagonal tiles), or the reason to refuse it
inline int bmm_plan(const lq_bmm_chunk_args* a, BmmParams* p, bool causal = false) {
  if (!a || !a->a || !a->b || !a->a_scale || !a->b_scale || !a->cb_scale || !a->out) return LQ_ERR_NULL;
  if (a->batch <= 0 || a->seqlen <= 0 || a->ngroups <= 0 || a->batch > 65535) return LQ_ERR_SHAPE;
  const int Q = a->chunk_size, N = a->dstate;
  if (Q < 64 || Q % 64 != 0 || Q > 4096 || N < 64 || N % 64 != 0 || N > 256) return LQ_ERR_SHAPE;
  if (a->a_stride_b % 16 || a->a_stride_l % 16 || a->a_stride_g % 16 || !bmm_al(a->a, 16)) return LQ_ERR_SHAPE;
  const int bal = 16;  // 16 int8 or 8 fp16 per vector load
  const int bmod = a->b_is_fp ? 8 : 16;
  if (a->b_stride_b % bmod || a->b_stride_l % bmod || a->b_stride_g % bmod || !bmm_al(a->b, bal) || !bmm_al(a->out, 16))
    return LQ_ERR_SHAPE;
  // 24-bit row * pitch products and 32-bit lane offsets inside a chunk
  if (a->a_stride_l < 0 || a->b_stride_l < 0 || a->a_stride_l >= (1 << 23) || a->b_stride_l >= (1 << 22) ||
      (int64_t)Q * a->a_stride_l >= (1ll << 31) || (int64_t)Q * a->b_stride_l * 2 >= (1ll << 31))
    return LQ_ERR_SHAPE;
  const int nchunks = (a->seqlen + Q - 1) / Q;
  if ((int64_t)nchunks * a->ngroups > 65535) return LQ_ERR_SHAPE;
  const uint32_t shift = Q == 64 ? 0u : (uint32_t)(0x100000000ull / (uint32_t)(Q / 64)) + 1u;  // tiles per row, as a multiplier
  const uint32_t g_magic = a->ngroups == 1 ? 0u : (uint32_t)(0x100000000ull / (uint32_t)a->ngroups) + 1u;
  const uint32_t tpc = (uint32_t)(causal ? (Q / 64) * (Q / 64 + 1) / 2 : (Q / 64) * (Q / 64)), ncg = (uint32_t)(nchunks * a->ngroups);
  const uint64_t units = (uint64_t)a->batch * ncg, total = units * tpc;
  if (total >= (1ull << 31) || total * tpc >= (1ull << 32) || units * ncg >= (1ull << 32)) return LQ_ERR_SHAPE;
  auto magic = [](uint32_t d) { return d == 1 ? 0u : (uint32_t)(0x100000000ull / d) + 1u; };
  const int by_xcd = units % 8 == 0;
  *p = BmmParams{a->a, a->a_stride_b, a->a_stride_l, a->a_stride_g, a->b, a->b_stride_b, a->b_stride_l, a->b_stride_g, a->a_scale,
                 a->b_scale, a->cb_scale, a->out, a->seqlen, a->ngroups, Q, nchunks, shift, g_magic, tpc, magic(tpc), ncg, magic(ncg),
                 by_xcd, causal, (uint32_t)total};
  return LQ_OK;
}

}  // namespace
