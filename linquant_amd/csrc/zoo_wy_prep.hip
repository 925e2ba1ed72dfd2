// WY / UT transform of the delta family, per chunk, in fp32: the entry point, and the kernel for 128-token chunks (every decay kind);
// 64-token chunks are zoo_diag_prep.h (per-channel decay) and zoo_wy_ns.hip (no / scalar decay).
// Replaces the torch prep linquant/kernels/zoo/kda.py:22-53 and gated_delta_rule.py:20-47; the reference's default route through
// fla-core's prep kernels for sigma = tau = 1 is served by the same native prep.
//   L = beta^sigma k,  Hg = beta^(1-sigma) k
//   G[i][j] = sum_n L[i][n] Hg[j][n] * decay(i,j,n)  for i > j, decay = 1 | exp(g_i - g_j) | exp(g_in - g_jn)
//   T = (I + G)^-1  (unit lower triangular, forward substitution)
//   W = T (L * exp(g)),  U = T (beta^sigma v),  Hw = beta^((1-sigma) tau) k,  fw = beta^((1-sigma)(1-tau))
//
#include "zoo_params.h"

namespace {

using WyParams = ZooWyParams;

LQ_DEV float powb(float b, float e) {
  if (e == 0.0f) return 1.0f;
  if (e == 1.0f) return b;
  return __builtin_amdgcn_exp2f(e * __builtin_amdgcn_logf(b));
}

LQ_DEV lq_v4f mfma_f32(float a, float b, lq_v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

LQ_DEV float wy_wave_max(float m) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  return m;
}

// Gram of row block I with the per-channel decay factorized around the first row of the row block: operands straight from
// global memory, lane (rl, kg) supplies 16 contiguous channels of token rl per 64-channel pass; off-diagonal blocks: both
// factors <= 1; diagonal block: only when the spread inside the block is small, otherwise one exponential per (i, j, channel).
// NB = row blocks of the chunk, GS = floats per row of the G tile.
template <int DECAY, int K, bool BF, int NB, int GS>
LQ_DEV void gram_rowblock(const WyParams& p, float* G_s, const float* bs_s, const float* bh_s, const float* gs_s, int I,
                          int rl, int kg, int64_t t0, int h) {
  const int H = p.H;
  constexpr bool bf = BF;
    const int64_t irow = ((t0 + 16 * I + rl) * H + h) * K;
    const int64_t arow = ((t0 + 16 * I) * H + h) * K;
    const float bs_i = bs_s[16 * I + rl];
    lq_v4f acc[NB];
#pragma unroll
    for (int J = 0; J < NB; ++J) acc[J] = lq_v4f{0.f, 0.f, 0.f, 0.f};
    bool exact_diag = false;
    if (DECAY == LQ_DECAY_DIAGONAL) {
      float spread = 0.0f;
      for (int c = 16 * kg; c < K; c += 64)
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
          const lq_v4f g4 = *(const lq_v4f*)(p.g + irow + c + 4 * e4), a4 = *(const lq_v4f*)(p.g + arow + c + 4 * e4);
#pragma unroll
          for (int e = 0; e < 4; ++e) spread = fmaxf(spread, __builtin_fabsf(g4[e] - a4[e]));
        }
      exact_diag = wy_wave_max(spread) > 40.0f;
    }
#pragma unroll
    for (int ps = 0; ps < K / 64; ++ps) {
      const int c0 = 64 * ps + 16 * kg;
      float Lr[16], gi[16], an[16];
      {
        float k0[8];
        zoo_ld8(p.k + irow + c0, bf, k0);
        float k1[8];
        zoo_ld8(p.k + irow + c0 + 8, bf, k1);
#pragma unroll
        for (int e = 0; e < 16; ++e) Lr[e] = bs_i * (float)(e < 8 ? k0[e & 7] : k1[e & 7]);
        if (DECAY == LQ_DECAY_DIAGONAL) {
#pragma unroll
          for (int e4 = 0; e4 < 4; ++e4) {
            const lq_v4f g4 = *(const lq_v4f*)(p.g + irow + c0 + 4 * e4), a4 = *(const lq_v4f*)(p.g + arow + c0 + 4 * e4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              gi[4 * e4 + e] = g4[e];
              an[4 * e4 + e] = a4[e];
            }
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) Lr[e] = Lr[e] * zoo_exp(gi[e] - an[e]);
        }
      }
#pragma unroll
      for (int J = 0; J < NB; ++J) {
        if (J > I) continue;
        if (DECAY == LQ_DECAY_DIAGONAL && J == I && exact_diag) continue;
        const int64_t jrow = ((t0 + 16 * J + rl) * H + h) * K;
        const float bh_j = bh_s[16 * J + rl];
        float k0[8];
        zoo_ld8(p.k + jrow + c0, bf, k0);
        float k1[8];
        zoo_ld8(p.k + jrow + c0 + 8, bf, k1);
        float Hr[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) Hr[e] = bh_j * (float)(e < 8 ? k0[e & 7] : k1[e & 7]);
        if (DECAY == LQ_DECAY_DIAGONAL) {
#pragma unroll
          for (int e4 = 0; e4 < 4; ++e4) {
            const lq_v4f g4 = *(const lq_v4f*)(p.g + jrow + c0 + 4 * e4);
#pragma unroll
            for (int e = 0; e < 4; ++e) Hr[4 * e4 + e] = Hr[4 * e4 + e] * zoo_exp(an[4 * e4 + e] - g4[e]);
          }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[J] = mfma_f32(Lr[e], Hr[e], acc[J]);
      }
    }
    // lane holds column j = rl of block J, rows i = 4kg + r of block I
#pragma unroll
    for (int J = 0; J < NB; ++J) {
      if (J > I) continue;
      if (DECAY == LQ_DECAY_DIAGONAL && J == I && exact_diag) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * I + 4 * kg + r, j = 16 * J + rl;
        float v = 0.0f;
        if (i > j) {
          v = acc[J][r];
          if (DECAY == LQ_DECAY_SCALAR) v = v * zoo_exp(gs_s[i] - gs_s[j]);
        }
        G_s[i * GS + j] = v;
      }
    }
    if (DECAY == LQ_DECAY_DIAGONAL && exact_diag) {
      // lane (i = rl, j = 4kg + jj) of the diagonal block, one exponential per (i, j, channel)
      float sacc[4] = {0.f, 0.f, 0.f, 0.f};
      for (int n8 = 0; n8 < K; n8 += 8) {
        float ki[8];
        zoo_ld8(p.k + irow + n8, bf, ki);
        const lq_v4f gi0 = *(const lq_v4f*)(p.g + irow + n8), gi1 = *(const lq_v4f*)(p.g + irow + n8 + 4);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int j = 4 * kg + jj;
          const int64_t jrow = ((t0 + 16 * I + j) * H + h) * K;
          float kj[8];
          zoo_ld8(p.k + jrow + n8, bf, kj);
          const lq_v4f gj0 = *(const lq_v4f*)(p.g + jrow + n8), gj1 = *(const lq_v4f*)(p.g + jrow + n8 + 4);
          const float bh_j = bh_s[16 * I + j];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float gi_ = e < 4 ? gi0[e & 3] : gi1[e & 3], gj_ = e < 4 ? gj0[e & 3] : gj1[e & 3];
            const float w = (rl > j) ? zoo_exp(gi_ - gj_) : 0.0f;
            sacc[jj] = fmaf((bs_i * ki[e]) * (bh_j * kj[e]), w, sacc[jj]);
          }
        }
      }
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) G_s[(16 * I + rl) * GS + 16 * I + 4 * kg + jj] = (rl > 4 * kg + jj) ? sacc[jj] : 0.0f;
    }
}

// ---- 128-token chunks: the same transform over a 128 x 128 Gram matrix (gated_delta_rule.py:20-47, kda.py:22-53 with
// chunk_size = 128), written for reach, not for speed: one workgroup per (chunk, batch*head) with the G tile in 67 KB of LDS
// (two workgroups per compute unit), inverted in place, everything on the fp32 MFMA.
//   Gram: wave w takes row blocks w and 7 - w (equal numbers of 16 x 16 blocks), per-channel decay anchored at the row
//     block's first row (both factors <= 1), operands straight from global memory (gram_rowblock).
//   Inverse, in place (row I of the tile holds G until block row I is done, T after): the eight diagonal blocks by forward
//     substitution, then block rows 1..7, every block of a row formed in registers before the row is overwritten.
//   W, U: T . X with X staged as fp32 in LDS 16 columns at a time.
// No write codes (lq_zoo_write_codes makes them from the stored Hw and W), no D_QK at load.
constexpr int kGS2 = 130;  // floats per row of the 128-row G / T tile (an A-operand read, 16 rows of 4 adjacent slots, takes one LDS pass at 2 mod 4)
constexpr int kXS2 = 20;   // floats per token row of the X slab (16 columns + pad); with the tile and the tables 77 KB

template <int DECAY, int K, bool BF>
__global__ __launch_bounds__(256, 2) void zoo_wy_prep128_kernel(WyParams p) {
  __shared__ __align__(16) float G_s[128 * kGS2];
  __shared__ __align__(16) float X_s[128 * kXS2];
  __shared__ float gs_s[128], bs_s[128], bh_s[128], bw_s[128];
  float* T_s = G_s;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int rl = lane & 15, kg = lane >> 4;
  const int H = p.H, V = p.V;
  const int h = blockIdx.x % H;
  const int64_t grp = blockIdx.x / H;  // b * (T / 128) + chunk
  const int64_t t0 = grp * 128;        // (b * T + chunk * 128: T is a multiple of 128)
  const float sigma = p.sigma, tau = p.tau;
  constexpr bool bf = BF;

  if (tid < 128) {
    const float bt = p.beta[(t0 + tid) * H + h];
    bs_s[tid] = powb(bt, sigma);
    bh_s[tid] = powb(bt, 1.0f - sigma);
    bw_s[tid] = powb(bt, (1.0f - sigma) * tau);
    p.fw[(t0 + tid) * H + h] = powb(bt, (1.0f - sigma) * (1.0f - tau));
    gs_s[tid] = DECAY == LQ_DECAY_SCALAR ? p.g[(t0 + tid) * H + h] : 0.0f;
  }
  __syncthreads();

  // ---- Gram
#pragma unroll 1
  for (int u = 0; u < 2; ++u)
    gram_rowblock<DECAY, K, BF, 8, kGS2>(p, G_s, bs_s, bh_s, gs_s, u ? 7 - wave : wave, rl, kg, t0, h);
  __syncthreads();

  // ---- T = (I + G)^-1: diagonal blocks (wave w: blocks w and w + 4; lane c < 16 holds column c)
  if (lane < 16) {
#pragma unroll 1
    for (int u = 0; u < 2; ++u) {
      const int o = 16 * (wave + 4 * u);
      float tc[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float a = (i == lane) ? 1.0f : 0.0f;
#pragma unroll
        for (int j = 0; j < i; ++j) a = fmaf(-G_s[(o + i) * kGS2 + o + j], tc[j], a);
        tc[i] = a;
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) T_s[(o + i) * kGS2 + o + lane] = tc[i];
    }
  }
  __syncthreads();
  // block rows 1..7: T_IJ = -T_II . sum_{J <= M < I} G_IM . T_MJ, the J of a row dealt to the waves
#pragma unroll 1
  for (int I = 1; I < 8; ++I) {
    lq_v4f tnew[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) tnew[u] = lq_v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int J = wave + 4 * u;
      if (J >= I) continue;
      lq_v4f sacc = {0.f, 0.f, 0.f, 0.f};
      for (int M = J; M < I; ++M)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int m = 16 * M + 4 * s + kg;
          sacc = mfma_f32(G_s[(16 * I + rl) * kGS2 + m], T_s[m * kGS2 + 16 * J + rl], sacc);
        }
      // sacc: lane (rl = column, kg) holds rows 4kg + r, which is contraction index 4kg + s of the next product
      lq_v4f tacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) tacc = mfma_f32(T_s[(16 * I + rl) * kGS2 + 16 * I + 4 * kg + s], sacc[s], tacc);
      tnew[u] = tacc;
    }
    __syncthreads();  // every wave has read what it needs of row I's G blocks
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int J = wave + 4 * u;
      if (J < I) {
#pragma unroll
        for (int r = 0; r < 4; ++r) T_s[(16 * I + 4 * kg + r) * kGS2 + 16 * J + rl] = -tnew[u][r];
      }
    }
    __syncthreads();
  }

  // ---- W = T . X (X = beta^sigma k exp(g)) and U = T . (beta^sigma v), 16 columns at a time; Hw goes straight out.
  // Staging: thread (token = tid / 2, half = tid % 2) forms 8 columns of its token.
  const int tok = tid >> 1, hf = tid & 1;
  const int nslab = (K + V) / 16;
#pragma unroll 1
  for (int sl = 0; sl < nslab; ++sl) {
    const bool isk = sl < K / 16;
    const int cc = isk ? 16 * sl : 16 * sl - K;  // first column of the slab in k (or v)
    const int c0 = cc + 8 * hf;                  // first column of this thread
    __syncthreads();  // the slab is no longer read
    {
      float x[8];
      if (isk) {
        const int64_t off = ((t0 + tok) * H + h) * K + c0;
        float kk[8];
        zoo_ld8(p.k + off, bf, kk);
        float bl = bs_s[tok];
        if (DECAY == LQ_DECAY_SCALAR) bl = bl * zoo_exp(gs_s[tok]);
        const float bw = bw_s[tok];
        float hw[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          x[e] = bl * kk[e];
          hw[e] = bw * kk[e];
        }
        if (DECAY == LQ_DECAY_DIAGONAL) {
          const lq_v4f g0 = *(const lq_v4f*)(p.g + off), g1 = *(const lq_v4f*)(p.g + off + 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = x[e] * zoo_exp(g0[e]), x[4 + e] = x[4 + e] * zoo_exp(g1[e]);
        }
        lq_v4i o;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] = (int)zoo_enc2(hw[2 * d], hw[2 * d + 1], bf);
        *(lq_v4i*)(p.Hw + off) = o;
      } else {
        float vv[8];
        zoo_ld8(p.v + ((t0 + tok) * H + h) * V + c0, bf, vv);
        const float bsr = bs_s[tok];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = bsr * vv[e];
      }
      *(lq_v4f*)(X_s + tok * kXS2 + 8 * hf) = lq_v4f{x[0], x[1], x[2], x[3]};
      *(lq_v4f*)(X_s + tok * kXS2 + 8 * hf + 4) = lq_v4f{x[4], x[5], x[6], x[7]};
    }
    __syncthreads();
    _Float16* dst = isk ? p.W : p.U;
    const int C = isk ? K : V;
#pragma unroll 1
    for (int u = 0; u < 2; ++u) {
      const int I = u ? 7 - wave : wave;
      lq_v4f acc = {0.f, 0.f, 0.f, 0.f};
      for (int s = 0; s < 4 * (I + 1); ++s)
        acc = mfma_f32(T_s[(16 * I + rl) * kGS2 + 4 * s + kg], X_s[(4 * s + kg) * kXS2 + rl], acc);
      // lane holds column rl of the slab, rows 16I + 4kg + r
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *(uint16_t*)(dst + ((t0 + 16 * I + 4 * kg + r) * H + h) * C + cc + rl) = (uint16_t)zoo_enc1(acc[r], bf);
    }
  }
}

template <int DECAY, int K>
int launch128(const WyParams& p, hipStream_t stream) {
  const dim3 grid((uint32_t)((int64_t)(p.T / 128) * p.B * p.H));
  if (p.bf)
    hipLaunchKernelGGL((zoo_wy_prep128_kernel<DECAY, K, true>), grid, dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL((zoo_wy_prep128_kernel<DECAY, K, false>), grid, dim3(256), 0, stream, p);
  return lq_check_launch();
}

template <int K>
int launch128_decay(const WyParams& p, int decay, hipStream_t stream) {
  switch (decay) {
    case LQ_DECAY_NONE: return launch128<LQ_DECAY_NONE, K>(p, stream);
    case LQ_DECAY_SCALAR: return launch128<LQ_DECAY_SCALAR, K>(p, stream);
    case LQ_DECAY_DIAGONAL: return launch128<LQ_DECAY_DIAGONAL, K>(p, stream);
  }
  return LQ_ERR_SHAPE;
}

}  // namespace

int zoo_wy_prep_launch(const lq_zoo_wy_prep_args* a, bool scan, const ZooWyLocal* local, hipStream_t stream) {
  const bool no_hw = scan && local;  // Hw itself is not wanted
  if (!a || !a->k || !a->v || !a->beta || (!a->Hw && !no_hw) || !a->U || (!a->fw && !scan)) return LQ_ERR_NULL;
  if (a->decay != LQ_DECAY_NONE && !a->g) return LQ_ERR_NULL;
  const bool codes = a->kqT != nullptr;
  if (scan && (!codes || !a->pack || !local || a->decay == LQ_DECAY_DIAGONAL)) return LQ_ERR_SHAPE;
  if (local && (!local->q || !local->qc || !local->A || !local->sq || !local->sk || (a->decay == LQ_DECAY_SCALAR && !local->gpk)))
    return LQ_ERR_NULL;
  if (local && !zoo_al(local->q, 16)) return LQ_ERR_SHAPE;
  if (!codes && !a->W) return LQ_ERR_NULL;
  if (codes && (!a->wq || (!scan && (!a->ev || !a->gam)) || !a->skw || !a->sw)) return LQ_ERR_NULL;
  if (codes && a->decay == LQ_DECAY_DIAGONAL && !a->logenv) return LQ_ERR_NULL;
  if (codes && (a->qmax < 1 || a->qmax > 127)) return LQ_ERR_SHAPE;
  if (codes && (!zoo_al(a->kqT, 16) || !zoo_al(a->wq, 4) || !zoo_al(a->skw, 16))) return LQ_ERR_SHAPE;
  if ((a->dk_div != nullptr) != (a->dk_rcp != nullptr)) return LQ_ERR_NULL;
  if (a->pack && (!codes || !zoo_al(a->pack, 16))) return LQ_ERR_SHAPE;
  if (a->dk_div && !codes) return LQ_ERR_SHAPE;  // built for the launch that also makes the write operands
  if (a->dk_div && (!zoo_al(a->dk_div, 16) || !zoo_al(a->dk_rcp, 16))) return LQ_ERR_SHAPE;
  if (a->batch <= 0 || a->seqlen <= 0 || a->nheads <= 0) return LQ_ERR_SHAPE;
  // 128-token chunks: a kernel of their own, without the write codes and without D_QK at load
  const bool big = a->chunk_size == 128;
  if (big && (codes || a->dk_div || !a->W)) return LQ_ERR_SHAPE;
  if ((a->chunk_size != 64 && !big) || a->seqlen % a->chunk_size != 0) return LQ_ERR_SHAPE;
  if ((a->kdim != 64 && a->kdim != 128) || a->vdim % 64 != 0 || a->vdim <= 0) return LQ_ERR_SHAPE;
  if (a->act_dtype != LQ_DT_F16 && a->act_dtype != LQ_DT_BF16) return LQ_ERR_SHAPE;
  if (a->decay < LQ_DECAY_NONE || a->decay > LQ_DECAY_DIAGONAL) return LQ_ERR_SHAPE;
  if (!zoo_al(a->k, 16) || !zoo_al(a->v, 16) || (!no_hw && !zoo_al(a->Hw, 16))) return LQ_ERR_SHAPE;
  if (a->decay == LQ_DECAY_DIAGONAL && !zoo_al(a->g, 16)) return LQ_ERR_SHAPE;
  if ((int64_t)a->batch * a->nheads > 65535) return LQ_ERR_SHAPE;
  WyParams p = {};
  p.k = (const _Float16*)a->k, p.v = (const _Float16*)a->v, p.beta = a->beta, p.g = a->g;
  p.Hw = (_Float16*)a->Hw, p.W = (_Float16*)a->W, p.U = (_Float16*)a->U, p.fw = a->fw;
  p.sigma = a->sigma, p.tau = a->tau, p.bf = a->act_dtype == LQ_DT_BF16;
  p.B = a->batch, p.T = a->seqlen, p.H = a->nheads, p.V = a->vdim;
  p.kqT = a->kqT, p.wq = a->wq, p.ev = a->ev, p.gam = a->gam, p.logenv = a->logenv, p.skw = a->skw, p.sw = a->sw;
  p.eta = a->eta, p.qmax = a->qmax, p.NT = a->seqlen / 64;
  p.dk_div = a->dk_div, p.dk_rcp = a->dk_rcp;
  p.pack = a->pack;
  if (local) {
    p.q = (const _Float16*)local->q, p.qc = local->qc, p.A = (_Float16*)local->A, p.gpk = local->gpk;
    p.sq = local->sq, p.sk = local->sk, p.scale = local->scale;
  }
  if ((int64_t)(a->seqlen / 64) * a->batch * a->nheads > 0x7fffffff) return LQ_ERR_SHAPE;
  if (big) return a->kdim == 128 ? launch128_decay<128>(p, a->decay, stream) : launch128_decay<64>(p, a->decay, stream);
  if (a->decay != LQ_DECAY_DIAGONAL) return zoo_wy_ns_launch(p, a->decay == LQ_DECAY_SCALAR, a->kdim, scan, stream);
  ZooDiagParams d = {};
  d.k = p.k, d.v = p.v, d.beta = p.beta, d.g = p.g, d.logenv = p.logenv, d.dk_div = p.dk_div, d.dk_rcp = p.dk_rcp;
  d.skw = p.skw, d.sw = p.sw, d.kqT = p.kqT, d.wq = p.wq, d.Hw = p.Hw, d.W = p.W, d.U = p.U, d.fw = p.fw, d.ev = p.ev, d.gam = p.gam;
  d.pack = p.pack, d.sigma = p.sigma, d.tau = p.tau, d.eta = p.eta, d.qmax = p.qmax, d.bf = p.bf;
  d.B = p.B, d.T = p.T, d.H = p.H, d.V = p.V, d.NT = p.NT;
  return zoo_diag_wy_launch(d, a->kdim, stream);
}

extern "C" int lq_zoo_wy_prep(const lq_zoo_wy_prep_args* a, hipStream_t stream) { return zoo_wy_prep_launch(a, false, nullptr, stream); }
