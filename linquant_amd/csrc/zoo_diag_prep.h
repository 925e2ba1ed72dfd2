// Everything in front of the chunk recurrence under per-channel (diagonal) decay, 64-token chunks: cumulative log decay and its
// envelope, key (and value) write codes, state-read codes of the queries, the intra-chunk product A and, for the delta rule, the
// WY / UT transform.  One kernel in four forms:
//   DIAG_GLA, DIAG_KDA  all of it in one launch, from the model's tensors to the operands of zoo_scan.hip
//   DIAG_A              lq_zoo_gla_A: A and the state-read codes, from the cumulative decay
//   DIAG_WY             lq_zoo_wy_prep: the transform (and its write codes), from the cumulative decay
// The stage forms run the code of the fused ones, so one call and the stages one after the other give the same bits.
// Replaces the torch prep of the reference's wrappers (linquant/kernels/zoo/gla.py:249-251, kda.py:22-53, 168-170) and its kernels
// _gla_A_inter (gla.py:27-63) and _gla_A_intra (gla.py:66-99).  With g the cumulative log decay, a_J its row 16J:
//   A   off-diagonal block (I > J):  q8(q_i e^(g_i - a_I) scale . R, 1/sq) . q8(Hw_j e^(a_I - g_j) . R, 1/sk) * (sq sk)
//       diagonal block:              sum_n q8(q_i scale)[n] q8(Hw_j)[n] e^(g_i - g_j)[n] * (sq sk),  j <= i
//   G[i][j] = beta_i^sigma beta_j^(1-sigma) sum_n k_i[n] k_j[n] e^(g_i - g_j)[n] for i > j,  T = (I + G)^-1
//   W = T (beta^sigma k e^g),  U = T (beta^sigma v),  Hw = beta^((1-sigma) tau) k,  fw = beta^((1-sigma)(1-tau))
//
// The exponentials are what a separate kernel per product repeats (and what the vector unit issues at a quarter of its rate):
// here an element takes e+ = e^(g - a_J) and e- = e^(a_J - g), J its own 16-token sub-block, the key write code's, and e^(a_I - g) for each
// later sub-block I.  (e- times a factor per channel, e^(a_I - a_J), in the latter's place took 390 us where this takes 381, and put two
// to five times as many entries of A beside the fp16 of their float64 value: its operands are rounded next.)  The state read and W's
// operand are e+ times e^(a_J), the latter with the rounding of its argument made good.  The diagonal blocks are products of e+ and e- where the decay inside
// the sub-block spreads over no more than e^40 (each wave decides for its half of the channels), otherwise they take one exponential per
// (i, j, channel).
//
// One 8-wave workgroup per (chunk, batch*head), two to a compute unit (80 KB of LDS, 128 registers).  Two waves own sub-block J, half of
// the channels each; lane (rl, kg) holds its token rl, channels 32ks + 8kg + e, which is the layout of every MFMA operand built from them.
//   1  running sums in fp64, 16 tokens of a channel per thread, into LDS
//   2  own rows: codes, diagonal blocks, e+ k into LDS          3  key operands of the later sub-blocks, Gram blocks
//   4  rotation: 9 operands x 32 channels per wave, R in registers   5  INT8 products; inverse of the diagonal blocks
//   6  block columns of T                                       7  W, U: T and the rows in three bf16 pieces, six products
//
// Measured (kernel us, against a kernel each for cumsum, WY prep and A), fp16 unless said, with rotation: KDA B2 T8192 H32 K = V = 128,
// sigma = 1, 82 + 266 + 208 -> 380 (with D_QK 82 + 303 + 208 -> 381, bf16 377); sigma = 0.5, 82 + 268 + 208 -> 454 (with D_QK 82 + 303
// + 208 -> 451, bf16 81 + 276 + 203 -> 454); GLA B4 T4096 H16 K = V = 128 cumsum with codes 87 + 117 -> 139; KDA B1 T2048 H8 bf16
// 8 + 21 + 24 -> 23.
// On the way, KDA / GLA: 4 waves of 256 registers with W and U on the fp32 MFMA 501 / 165; on the bf16 MFMA 475; eight waves 467 / 148;
// the inverse one instruction a term, the key operands read ahead of their products 443; no gate arithmetic where Hw is k, bf16 rounded
// by the conversion 409 / 141; one exponential for a key operand (above).
// Bound by vector issue and the waits at its rendezvous, of which two workgroups cover part of each other's.  By counters, KDA B2 T8192 /
// GLA B4 T4096: vector unit busy 74 / 73 % of the time, matrix unit 26 / 11 %, waves waiting 38 % of theirs, LDS conflicts 2.5 / 3.5 %,
// memory 1093 / 507 MB at 2.9 / 3.6 TB/s; KDA B1 T2048, one workgroup to a compute unit: 31, 12, 24 %.  The vector work is the
// exponentials, the quantizations and what the products of phases 2 and 3 hold up: these stay on the fp32 MFMA, 33 cycles a 16x16x4,
// during which its SIMD issues no vector instruction (the half-precision MFMA costs them only its issue), yet splitting their operands in
// three would cost more.  Persistent workgroups with the next chunk's requests ahead spilled (KDA 714), three workgroups a compute unit for
// GLA too (194).
// R_QK comes in fp16, in fp32 or (larger calls) laid out as operands; D_QK's reciprocals are formed here.  As launches in front these were
// 4.6 us for R_QK and 9.3 for the reciprocals.  On one card in turn, with the steps of zoo_scan.hip since: whole calls KDA B1 T2048 H8 47.3
// -> 45.1 (this kernel 23.0 -> 23.6, R_QK read as fp32), KDA B2 T8192 H32 with D_QK 566 -> 558, GLA B4 T4096 H16 207 -> 204 (there R_QK is
// laid out as operands in the place of converted, a launch of 4.6 as before).
// Spilled registers: DIAG_KDA at K = 128 with the gate (sigma < 1, tau > 0) keeps Hw beside k over the key operands and spills 13 to 19
// of its 128 in fp16 and up to 15 in bf16 (56 to 80 and up to 64 bytes a lane; about 300 of the 972 MB read and of the 730 MB written at
// sigma = 0.5 above); without the gate at most one (bf16 with D_QK); the other forms and K = 64 none.
#pragma once

#include <type_traits>

#include "zoo_params.h"

enum { DIAG_A = 0, DIAG_WY = 1, DIAG_GLA = 2, DIAG_KDA = 3 };

namespace zoo_diag {

LQ_DEV lq_v4f mfma_f32(float a, float b, lq_v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

LQ_DEV float powb(float b, float e) {
  if (e == 0.0f) return 1.0f;
  if (e == 1.0f) return b;
  return __builtin_amdgcn_exp2f(e * __builtin_amdgcn_logf(b));
}

// float index of (token, channel) in the 64 x K tile.  Sub-block J and 32 channels are 2 KB: piece p of four channels of token rl is
// 16-byte slot 16p + (rl xor p), so that a lane's reads (pieces 2kg, 2kg + 1 of token rl), the running sums' writes (one token, 64
// channels) and the transposed reads of W's operand (16 channels, tokens 4kg + s) all spread over the banks.
template <int K>
LQ_DEV int at(int token, int ch) {
  const int p = (ch >> 2) & 7;
  return (((token >> 4) * (K / 32) + (ch >> 5)) * 128 + p * 16 + ((token & 15) ^ p)) * 4 + (ch & 3);
}

// byte of the transposed write codes [channel][64 tokens]: 16 bytes of pad after every eight channels
LQ_DEV int ct_at(int ch, int token) { return ch * 64 + (ch >> 3) * 16 + token; }

// 16 x 16 blocks of T (lower triangle; the diagonal ones hold G first) and of G below the diagonal, rows of 20 floats
constexpr int kBP = 20;
constexpr int kBlk = 16 * kBP;
LQ_DEV int t_blk(int I, int J) { return (I * (I + 1) / 2 + J) * kBlk; }
LQ_DEV int g_blk(int I, int J) { return I == J ? t_blk(I, I) : (10 + I * (I - 1) / 2 + J) * kBlk; }

// T as three bf16 pieces in the order of the bf16 MFMA's operand: step (I, st) is row block I, tokens 32st .. (what
// lies right of the diagonal block is zero, steps that are zero altogether are left out); its slot 8kg + 4m + s is token 32st + 16m +
// 4kg + s, so that the other operand is what a lane reads of one column
constexpr int kSteps = 6;
LQ_DEV int t_step(int I, int st) { return I < 2 ? I : 2 * (I - 1) + st; }

// two fp32 values -> one dword each of their upper, middle and lower 8 bits as bf16 (first value in the low half)
LQ_DEV void split3(float x0, float x1, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  const uint32_t b0 = __float_as_uint(x0), b1 = __float_as_uint(x1);
  hi = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
  const float r0 = x0 - __uint_as_float(b0 & 0xffff0000u), r1 = x1 - __uint_as_float(b1 & 0xffff0000u);  // exact
  const uint32_t c0 = __float_as_uint(r0), c1 = __float_as_uint(r1);
  mid = __builtin_amdgcn_perm(c1, c0, 0x07060302u);
  const float q0 = r0 - __uint_as_float(c0 & 0xffff0000u), q1 = r1 - __uint_as_float(c1 & 0xffff0000u);  // exact
  lo = __builtin_amdgcn_perm(__float_as_uint(q1), __float_as_uint(q0), 0x07060302u);
}

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
LQ_DEV lq_v4f mfma_bf16(lq_v4i a, lq_v4i b, lq_v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

// pair (J, I), J < I, of sub-blocks: (0,1) (0,2) (0,3) (1,2) (1,3) (2,3)
LQ_DEV int pair_of(int J, int I) { return (J == 0 ? -1 : (J == 1 ? 1 : 2)) + I; }

constexpr int maxi(int a, int b) { return a > b ? a : b; }

template <int K, bool ROT, int MODE, bool DK>
struct Lds {
  static constexpr bool DO_A = MODE != DIAG_WY, DELTA = MODE == DIAG_WY || MODE == DIAG_KDA, KQ = MODE != DIAG_A;
  static constexpr int OP = 16 * K * 2, CD = 16 * K;  // bytes of an fp16 operand and of its codes
  static constexpr int r1 = 0;                        // decay tile, then e+ k; GLA: value codes; U: v
  static constexpr int r2 = 64 * K * 4;
  static constexpr int X = ROT ? OP : CD;             // an operand as its waves leave it
  static constexpr int F_bytes = 3 * K * 4, GT_bytes = DELTA ? 16 * kBlk * 4 : 0, KQ_bytes = KQ ? K * 64 + K * 2 : 0;
  // operands (3 queries, 6 keys) | then their codes, then the pieces of T; blocks of G and T behind them.  The write codes pass
  // through the key operands' place, the fp64 totals through the queries'; the rows a_1 .. a_3 (F) lie at the end, dead when G is written.
  static constexpr int kq = r2 + (DO_A ? 3 * X : 0);
  static constexpr int TP_bytes = DELTA ? 3 * kSteps * 1024 : 0;
  static constexpr int gt = r2 + maxi(DO_A ? 9 * CD : 0, TP_bytes);
  static constexpr int area = maxi(maxi((DO_A ? maxi(9 * X, 3 * X + KQ_bytes) : KQ_bytes) + F_bytes, gt - r2 + GT_bytes), 4 * K * 8);
  static constexpr int F = r2 + area - F_bytes;
  static constexpr int E = r2 + area;                 // e^(a_J)
  static constexpr int bs = E + 4 * K * 4;
  static constexpr int le = bs + 64 * 4;              // envelope over either half of the channels
  // tables of phase 2, then the second half's share of the diagonal blocks of A
  static constexpr int an = le + 2 * 64 * 4;          // decay rows 0, 16, 32, 48, 63
  static constexpr int iskw = an + 5 * K * 4;
  static constexpr int dq = iskw + (KQ ? K * 4 : 0);
  static constexpr int dkd = dq + (DK && DO_A ? K * 4 : 0);
  static constexpr int dkr = dkd + (DK && DELTA ? K * 4 : 0);
  static constexpr int bytes = maxi(dkr + (DK && DELTA ? K * 4 : 0), an + (DO_A ? 4 * 64 * 16 : 0));
};

// GATE (delta rule): beta^((1-sigma) tau) is not one for every token (otherwise Hw is k)
template <int K, bool ROT, bool BF, int MODE, bool DK, bool GATE>
__global__ __launch_bounds__(512, 4) void zoo_diag_prep_kernel(ZooDiagParams p) {
  using L = Lds<K, ROT, MODE, DK>;
  constexpr bool FUSED = MODE == DIAG_GLA || MODE == DIAG_KDA, DO_A = L::DO_A, DELTA = L::DELTA;
  constexpr int KS = K / 32;      // steps of 32 channels
  constexpr int KW = KS / 2;      // of one wave
  constexpr int SEG = K / 8;      // tokens per thread where all threads take one value channel
  __shared__ __align__(16) unsigned char lds[L::bytes];
  float* const R1 = (float*)(lds + L::r1);
  float* const F_s = (float*)(lds + L::F);
  float* const AN = (float*)(lds + L::an);
  float* const E_s = (float*)(lds + L::E);
  float* const iskw_s = (float*)(lds + L::iskw);
  float* const dq_s = (float*)(lds + L::dq);
  float* const dkd_s = (float*)(lds + L::dkd);
  float* const dkr_s = (float*)(lds + L::dkr);
  float* const bs_s = (float*)(lds + L::bs);  // beta^sigma per token; GLA: e^(eta * envelope)
  float* const le_s = (float*)(lds + L::le);
  float* const GT = (float*)(lds + L::gt);
  uint16_t* const TP = (uint16_t*)(lds + L::r2);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rl = lane & 15, kg = lane >> 4;
  ZooUnit unit;
  if (!zoo_unit(p.B, p.NT, p.H, unit)) return;
  const int h = unit.h, H = p.H, V = p.V, qmax = p.qmax;
  const int64_t group = (int64_t)unit.b * p.NT + unit.ct;
  const int64_t t0 = group * 64;                 // (b * T + chunk * 64: T is a multiple of 64)
  const int64_t cb = group * H + h;
  constexpr bool bf = BF;
  // sub-block and half of the channels of this wave (the two waves of a SIMD, w and w + 4, share the work of sub-blocks J and 3 - J:
  // the earlier a sub-block, the more later ones take its keys)
  const int half = wave >> 2, J = half ? 7 - wave : wave;
  const int tok = 16 * J + rl;                   // token of this lane
  const int ks0 = KW * half, n0 = 32 * ks0 + 8 * kg;  // first step, first channel of this lane

  // ---- requests of the chunk
  const int col = tid % K, seg = wave / (K / 64);  // running sums: one channel, 16 tokens (seg: uniform over the wave)
  const bool scans = K == 128 || wave < 4;
  float gv[FUSED ? 16 : 1];
  if constexpr (FUSED) {
    if (scans) {
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        const float* row = p.g + ((t0 + 16 * seg + t) * H + h) * K;  // (a scalar: the lane adds 32 bits)
        gv[t] = row[(uint32_t)col];
      }
    }
  }
  const int64_t roff = ((t0 + tok) * H + h) * K + n0;
  lq_v4i kraw[KW], qraw[DO_A ? KW : 1];
#pragma unroll
  for (int i = 0; i < KW; ++i) {
    kraw[i] = *(const lq_v4i*)(p.k + roff + 32 * i);
    if constexpr (DO_A) qraw[i] = *(const lq_v4i*)(p.q + roff + 32 * i);
  }
  float bt = 0.0f;
  if constexpr (DELTA) bt = p.beta[(t0 + tok) * H + h];
  const bool codes = FUSED || (MODE == DIAG_WY && p.kqT);
  if (tid < K) {
    if constexpr (L::KQ) iskw_s[tid] = codes ? 1.0f / p.skw[h * K + tid] : 0.0f;
    if constexpr (DK && DO_A) dq_s[tid] = p.dq[h * K + tid];
    if constexpr (DK && DELTA) {
      const float d = p.dk_div[h * K + tid];
      dkd_s[tid] = d, dkr_s[tid] = p.dk_rcp ? p.dk_rcp[h * K + tid] : 1.0f / d;
    }
  }

  // ---- 1: cumulative log decay of the chunk into LDS
  if constexpr (FUSED) {
    double* part = (double*)(lds + L::r2);  // totals of the four 16-token quarters [4][K]
    double pre[16];
    if (scans) {
      double run = 0.0;
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        run += (double)gv[t];
        pre[t] = run;
      }
      part[seg * K + col] = run;
    }
    __syncthreads();
    if (scans) {
      double off = 0.0;
      for (int Q = 0; Q < seg; ++Q) off += part[Q * K + col];
      float x = 0.0f;
      float* const dst = R1 + at<K>(16 * seg, col);
      const int p4 = 4 * ((col >> 2) & 7);  // (slot t xor p of the piece's sixteen)
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        x = (float)(off + pre[t]);
        dst[((4 * t) ^ p4) - p4] = x;
        if (t == 0) AN[seg * K + col] = x;
      }
      if (seg == 3) {
        AN[4 * K + col] = x;
        const float gm = zoo_exp(x);
        if constexpr (DELTA) p.pack[cb * (128 + K) + 128 + col] = gm; else p.gam[cb * K + col] = gm;
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < K / 32; ++i) {
      const int it = tid + 512 * i, t = it / (K / 4), n = 4 * (it % (K / 4));
      const lq_v4f x = *(const lq_v4f*)(p.g + ((t0 + t) * H + h) * K + n);
      *(lq_v4f*)(R1 + at<K>(t, n)) = x;
      if ((t & 15) == 0) *(lq_v4f*)(AN + (t >> 4) * K + n) = x;
      if (t == 63) {
        *(lq_v4f*)(AN + 4 * K + n) = x;
        if constexpr (DELTA) {
          if (codes) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float gm = zoo_exp(x[e]);
              p.gam[cb * K + n + e] = gm;
              if (p.pack) p.pack[cb * (128 + K) + 128 + n + e] = gm;
            }
          }
        }
      }
    }
  }
  __syncthreads();

  // ---- 2: own rows.  gem: the decay of the lane's elements
  const float* const an_s = AN + J * K;
  float gem[KW][8];
  float spread = 0.0f, le = -__builtin_inff();
#pragma unroll
  for (int i = 0; i < KW; ++i)
#pragma unroll
    for (int e4 = 0; e4 < 2; ++e4) {
      const int n = n0 + 32 * i + 4 * e4;
      const lq_v4f g4 = *(const lq_v4f*)(R1 + at<K>(tok, n)), a4 = *(const lq_v4f*)(an_s + n);
      lq_v4f l4;
      if constexpr (FUSED) l4 = *(const lq_v4f*)(AN + 4 * K + n);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        gem[i][4 * e4 + e] = g4[e];
        spread = fmaxf(spread, __builtin_fabsf(g4[e] - a4[e]));
        if constexpr (FUSED) le = fmaxf(le, l4[e] - g4[e]);
      }
    }
  const bool slow = __any(spread > 40.0f);  // (uniform over the wave: a sub-block's halves decide for themselves)
  if constexpr (FUSED) {
    le = fmaxf(le, __shfl_xor(le, 16));
    le = fmaxf(le, __shfl_xor(le, 32));
    if (kg == 0) le_s[64 * half + tok] = le;
  }
  // e^(a_J) of this sub-block, and a_J for the earlier ones (the tables that hold it are overwritten behind this phase)
  if (lane < K / 2) {
    const int n = K / 2 * half + lane;
    const float a = an_s[n];
    E_s[J * K + n] = zoo_exp_acc(a);
    if (J > 0) F_s[(J - 1) * K + n] = a;
  }
  float bs = 1.0f, bh = 1.0f, bw = 1.0f, el = 0.0f;
  if constexpr (DELTA) {
    bs = powb(bt, p.sigma);
    bh = powb(bt, 1.0f - p.sigma);
    if constexpr (GATE) bw = powb(bt, (1.0f - p.sigma) * p.tau);
  }
  if constexpr (FUSED) {
    __syncthreads();
    el = p.eta * fmaxf(le, le_s[64 * (1 - half) + tok]);
  } else if constexpr (MODE == DIAG_WY) {
    if (codes) el = p.eta * p.logenv[(t0 + tok) * H + h];
  }
  __builtin_amdgcn_wave_barrier();
  if (half == 0 && kg == 0) {
    if constexpr (DELTA) {
      const float fwv = powb(bt, (1.0f - p.sigma) * (1.0f - p.tau)), evv = zoo_exp(el);
      bs_s[tok] = bs;
      if constexpr (!FUSED) {
        p.fw[(t0 + tok) * H + h] = fwv;
        if (codes) p.ev[(t0 + tok) * H + h] = evv;
      }
      if (codes && p.pack) p.pack[cb * (128 + K) + tok] = fwv, p.pack[cb * (128 + K) + 64 + tok] = evv;
    } else if constexpr (MODE == DIAG_GLA) {
      bs_s[tok] = zoo_exp(el);
    }
  }

  float sq = 0.0f, sk = 0.0f, inv_sq = 0.0f, inv_sk = 0.0f;
  if constexpr (DO_A) sq = p.sq[h], sk = p.sk[h], inv_sq = 1.0f / sq, inv_sk = 1.0f / sk;
  // eight channels of a key row: the caller's k, rescaled by D_QK
  auto load_k = [&](lq_v4i raw, int n, float (&o)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int d = 0; d < 4; ++d) zoo_dec2((uint32_t)raw[d], bf, o[2 * d], o[2 * d + 1]);
    if constexpr (DK && DELTA) {
      const lq_v4f d0 = *(const lq_v4f*)(dkd_s + n), d1 = *(const lq_v4f*)(dkd_s + n + 4);
      const lq_v4f r0 = *(const lq_v4f*)(dkr_s + n), r1 = *(const lq_v4f*)(dkr_s + n + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = zoo_round_act(zoo_div_rn(o[e], e < 4 ? d0[e & 3] : d1[e & 3], e < 4 ? r0[e & 3] : r1[e & 3]), bf);
    }
  };
  auto load_q = [&](lq_v4i raw, int n, float (&o)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int d = 0; d < 4; ++d) zoo_dec2((uint32_t)raw[d], bf, o[2 * d], o[2 * d + 1]);
    if constexpr (DK) {
      const lq_v4f d0 = *(const lq_v4f*)(dq_s + n), d1 = *(const lq_v4f*)(dq_s + n + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = zoo_round_act(zoo_mul_rn(o[e], e < 4 ? d0[e & 3] : d1[e & 3]), bf);
    }
  };
  // Hw = beta^((1-sigma) tau) k as it would be stored
  auto hw_of = [&](const float (&k)[8], float w, float (&o)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = k[e];
    if constexpr (GATE) {
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = zoo_round_act(zoo_mul_rn(w, k[e]), bf);
    }
  };

  // diagonal blocks, this half's channels: A transposed (lane: row rl, columns 4kg + r), G (lane: column rl, rows 4kg + r)
  lq_v4f dacc = {0.f, 0.f, 0.f, 0.f}, gacc = {0.f, 0.f, 0.f, 0.f};
  lq_v4f dslow = dacc, gslow = gacc;
  if (slow) {  // every (i, j, channel) weight on its own, masked before use
#pragma unroll 1
    for (int n = K / 2 * half; n < K / 2 * (half + 1); n += 8) {
      float ko[8], qo[8], go[8];
      load_k(*(const lq_v4i*)(p.k + ((t0 + tok) * H + h) * K + n), n, ko);
      if constexpr (DO_A) load_q(*(const lq_v4i*)(p.q + ((t0 + tok) * H + h) * K + n), n, qo);
#pragma unroll
      for (int e = 0; e < 8; ++e) go[e] = R1[at<K>(tok, n + e)];
#pragma unroll 1
      for (int r = 0; r < 4; ++r) {
        const int o = 4 * kg + r;  // the other token of the pair
        float kj[8], hj[8];
        load_k(*(const lq_v4i*)(p.k + ((t0 + 16 * J + o) * H + h) * K + n), n, kj);
        float w = 1.0f;
        if constexpr (GATE) w = powb(p.beta[(t0 + 16 * J + o) * H + h], (1.0f - p.sigma) * p.tau);
        hw_of(kj, w, hj);
        float sd = 0.0f, sg = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float gj = R1[at<K>(16 * J + o, n + e)];
          if constexpr (DO_A) {
            const float wd = o <= rl ? zoo_exp(go[e] - gj) : 0.0f;
            sd += ((float)zoo_q8(qo[e] * p.scale, inv_sq, qmax) * (float)zoo_q8(hj[e], inv_sk, qmax)) * wd;
          }
          if constexpr (DELTA) {
            const float wg = o > rl ? zoo_exp(gj - go[e]) : 0.0f;
            sg += (kj[e] * ko[e]) * wg;
          }
        }
#pragma unroll
        for (int r2 = 0; r2 < 4; ++r2)
          if (r2 == r) dslow[r2] += sd, gslow[r2] += sg;
      }
    }
  }

  unsigned char* const xq = lds + L::r2 + L::X * (J - 1);  // this sub-block's query operand (none for the first)
#pragma unroll
  for (int i = 0; i < KW; ++i) {
    const int ks = ks0 + i, n = n0 + 32 * i;
    float kf[8], qf[8], hf[8];
    load_k(kraw[i], n, kf);
    if constexpr (DO_A) load_q(qraw[i], n, qf);
    if constexpr (DK && DELTA) {
#pragma unroll
      for (int d = 0; d < 4; ++d) kraw[i][d] = (int)zoo_enc2(kf[2 * d], kf[2 * d + 1], bf);
    }
    hw_of(kf, bw, hf);
    if constexpr (MODE == DIAG_WY) {
      lq_v4i o;
#pragma unroll
      for (int d = 0; d < 4; ++d) o[d] = (int)zoo_enc2(hf[2 * d], hf[2 * d + 1], bf);
      *(lq_v4i*)(p.Hw + roff + 32 * i) = o;
    }
    int ck[8], cs[8], cx[8];
    lq_v8h x;
    lq_v4f kp[2];
#pragma unroll
    for (int e4 = 0; e4 < 2; ++e4) {
      const lq_v4f a4 = *(const lq_v4f*)(an_s + n + 4 * e4);
      lq_v4f l4, is4, E4;
      if constexpr (L::KQ) l4 = *(const lq_v4f*)(AN + 4 * K + n + 4 * e4), is4 = *(const lq_v4f*)(iskw_s + n + 4 * e4);
      if constexpr (DO_A) E4 = *(const lq_v4f*)(E_s + J * K + n + 4 * e4);
#pragma unroll
      for (int e_ = 0; e_ < 4; ++e_) {
        const int e = 4 * e4 + e_;
        const float g = gem[i][e], d = g - a4[e_];
        const float dl = d * 1.44269504088896340736f;
        const float ep = __builtin_amdgcn_exp2f(dl), em = __builtin_amdgcn_exp2f(-dl);
        if constexpr (DELTA) {
          kp[e4][e_] = kf[e] * ep;
          gacc = mfma_f32(kp[e4][e_], kf[e] * em, gacc);
        }
        if constexpr (DO_A) {
          const float cq = (float)zoo_q8(qf[e] * p.scale, inv_sq, qmax), chw = (float)zoo_q8(hf[e], inv_sk, qmax);
          dacc = mfma_f32(chw * em, cq * ep, dacc);
          const float xv = zoo_mul_rn(qf[e] * ep, p.scale);
          if constexpr (ROT) x[e] = (_Float16)xv; else cx[e] = zoo_q8(xv, inv_sq, qmax);
          cs[e] = zoo_q8(xv * E4[e_], inv_sq, qmax);
        }
        if constexpr (L::KQ) ck[e] = zoo_q8(hf[e] * zoo_exp(l4[e_] - g - el), is4[e_], qmax);
      }
    }
    if constexpr (DELTA) {
      *(lq_v4f*)(R1 + at<K>(tok, n)) = kp[0];
      *(lq_v4f*)(R1 + at<K>(tok, n + 4)) = kp[1];
      asm volatile("" : "+v"(gacc));
    }
    if constexpr (DO_A) {
      if (FUSED || p.qc) {
        const lq_v2i o = {(int)zoo_pack_codes(cs[0], cs[1], cs[2], cs[3]), (int)zoo_pack_codes(cs[4], cs[5], cs[6], cs[7])};
        *(lq_v2i*)(FUSED ? p.qc + cb * 64 * K + zoo_op_codes(tok, n, K) : p.qc + roff + 32 * i) = o;
      }
      if (J > 0) {
        if constexpr (ROT)
          *(lq_v8h*)(xq + (ks * 64 + lane) * 16) = x;
        else
          *(lq_v2i*)(xq + (ks >> 1) * 1024 + lane * 16 + 8 * (ks & 1)) =
              lq_v2i{(int)zoo_pack_codes(cx[0], cx[1], cx[2], cx[3]), (int)zoo_pack_codes(cx[4], cx[5], cx[6], cx[7])};
      }
      asm volatile("" : "+v"(dacc));
    }
    if constexpr (L::KQ) {
      if (codes) {
        // four adjacent lanes hold tokens 4Q .. 4Q+3 of the same eight channels: bytes are transposed among them, lane j of the
        // four keeps channels j and 4 + j, four tokens each
        uint32_t w[2] = {zoo_pack_codes(ck[0], ck[1], ck[2], ck[3]), zoo_pack_codes(ck[4], ck[5], ck[6], ck[7])};
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const uint32_t o1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w[q], 0xB1, 0xf, 0xf, true);  // lane ^ 1
          // even lane: channels 0, 2 of (own, other); odd lane: channels 1, 3 of (other, own)
          const uint32_t m = __builtin_amdgcn_perm(rl & 1 ? w[q] : o1, rl & 1 ? o1 : w[q], rl & 1 ? 0x07030501u : 0x06020400u);
          const uint32_t o2 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4E, 0xf, 0xf, true);  // lane ^ 2
          w[q] = __builtin_amdgcn_perm(rl & 2 ? m : o2, rl & 2 ? o2 : m, rl & 2 ? 0x07060302u : 0x05040100u);
        }
        unsigned char* dst = lds + L::kq;
        *(uint32_t*)(dst + ct_at(n + (rl & 3), 16 * J + (rl & 12))) = w[0];
        *(uint32_t*)(dst + ct_at(n + 4 + (rl & 3), 16 * J + (rl & 12))) = w[1];
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // one step after the other
  }
  if (slow) dacc = dslow, gacc = gslow;
  const float sqk = sq * sk;
  // elements (row, column ..) of A: sums of products of codes, scaled as they are rounded
  auto a_store = [&](int row, int c, lq_v4f v) __attribute__((always_inline)) {
    _Float16* dst = FUSED ? p.A + cb * 4096 + zoo_op_A(row, c) : p.A + ((t0 + row) * H + h) * 64 + c;
    *(lq_v2i*)dst = lq_v2i{(int)zoo_mul_h2(v[0], v[1], sqk), (int)zoo_mul_h2(v[2], v[3], sqk)};
  };
  // GLA: value rows, requested a phase ahead of their codes
  uint16_t vr[MODE == DIAG_GLA ? SEG : 1];
  auto request_values = [&](int c0) __attribute__((always_inline)) {
    if constexpr (MODE == DIAG_GLA) {
      const uint32_t c = (uint32_t)min(c0 + col, V - 1);
#pragma unroll
      for (int t = 0; t < SEG; ++t) {
        const uint16_t* row = (const uint16_t*)p.v + ((t0 + SEG * seg + t) * H + h) * V;
        vr[t] = row[c];
      }
    }
  };
  request_values(0);
  __syncthreads();

  // ---- the write codes leave as whole rows; the second half's share of the diagonal blocks of A passes through the dead tables
  lq_v4f* const dg = (lq_v4f*)(lds + L::an) + J * 64 + lane;
  if constexpr (DO_A) {
    if (half) *dg = dacc;
  }
  if constexpr (L::KQ) {
    if (codes && tid < 4 * K) *(lq_v4i*)(p.kqT + cb * K * 64 + 16 * tid) = *(const lq_v4i*)(lds + L::kq + ct_at(tid >> 2, 16 * (tid & 3)));
    if constexpr (DO_A) __syncthreads();  // the key operands take their place
  }

  // ---- 3: key rows of this sub-block anchored at the first row of each later one: Gram blocks, operands of A
  lq_v4f goff[3];
#pragma unroll
  for (int di = 0; di < 3; ++di) {
    goff[di] = lq_v4f{0.f, 0.f, 0.f, 0.f};
    const int I = J + 1 + di;
    if (I > 3) continue;  // (wave-uniform)
    const int pr = pair_of(J, I);
    unsigned char* const xk = lds + L::r2 + L::X * (3 + pr);
    lq_v4f fr[KW][2], ki[KW][2];  // all of the pair's reads ahead of its products
#pragma unroll
    for (int i = 0; i < KW; ++i)
#pragma unroll
      for (int e4 = 0; e4 < 2; ++e4) {
        const int n = n0 + 32 * i + 4 * e4;
        fr[i][e4] = *(const lq_v4f*)(F_s + (I - 1) * K + n);
        if constexpr (DELTA) ki[i][e4] = *(const lq_v4f*)(R1 + at<K>(16 * I + rl, n));
      }
#pragma unroll
    for (int i = 0; i < KW; ++i) {
      const int ks = ks0 + i;
      float kf[8], hf[8];
#pragma unroll
      for (int d = 0; d < 4; ++d) zoo_dec2((uint32_t)kraw[i][d], bf, kf[2 * d], kf[2 * d + 1]);
      if constexpr (DO_A) hw_of(kf, bw, hf);
      lq_v8h x;
      int cx[8];
      float we[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) we[e] = zoo_exp(fr[i][e >> 2][e & 3] - gem[i][e]);
#pragma unroll
      for (int e4 = 0; e4 < 2; ++e4) {
#pragma unroll
        for (int e_ = 0; e_ < 4; ++e_) {
          const int e = 4 * e4 + e_;
          const float kv = zoo_mul_rn(kf[e], we[e]);
          if constexpr (DELTA) goff[di] = mfma_f32(ki[i][e4][e_], kv, goff[di]);
          if constexpr (DO_A) {
            const float xv = GATE ? zoo_mul_rn(hf[e], we[e]) : kv;
            if constexpr (ROT) x[e] = (_Float16)xv; else cx[e] = zoo_q8(xv, inv_sk, qmax);
          }
        }
      }
      if constexpr (DO_A) {
        if constexpr (ROT)
          *(lq_v8h*)(xk + (ks * 64 + lane) * 16) = x;
        else
          *(lq_v2i*)(xk + (ks >> 1) * 1024 + lane * 16 + 8 * (ks & 1)) =
              lq_v2i{(int)zoo_pack_codes(cx[0], cx[1], cx[2], cx[3]), (int)zoo_pack_codes(cx[4], cx[5], cx[6], cx[7])};
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  // GLA: value codes, one channel per thread, through the dead decay tile; K channels at a time
  auto value_codes = [&](int c0) __attribute__((always_inline)) {
    const int c = c0 + col, vt = SEG * seg;
    if (c >= V) return;
    const float inv_svw = 1.0f / p.svw[h * V + c], inv_svl = 1.0f / p.svl[h * V + c];
    unsigned char* const vb = lds + L::r1;
    unsigned char* const lb = vb + K * 64;
#pragma unroll
    for (int t8 = 0; t8 < SEG; t8 += 8) {
      int cw[8], cl[8];
#pragma unroll
      for (int e4 = 0; e4 < 2; ++e4) {
        const lq_v4f ev4 = *(const lq_v4f*)(bs_s + vt + t8 + 4 * e4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = zoo_dec1(vr[t8 + 4 * e4 + e], bf);
          cw[4 * e4 + e] = zoo_q8(x * ev4[e], inv_svw, qmax), cl[4 * e4 + e] = zoo_q8(x, inv_svl, qmax);
        }
      }
      *(lq_v2i*)(vb + col * 64 + vt + t8) = lq_v2i{(int)zoo_pack_codes(cw[0], cw[1], cw[2], cw[3]), (int)zoo_pack_codes(cw[4], cw[5], cw[6], cw[7])};
      *(lq_v2i*)(lb + zoo_op_values(col, vt + t8)) = lq_v2i{(int)zoo_pack_codes(cl[0], cl[1], cl[2], cl[3]), (int)zoo_pack_codes(cl[4], cl[5], cl[6], cl[7])};
    }
  };
  auto value_copy = [&](int c0) __attribute__((always_inline)) {
    const int o = 16 * tid;
    if (o < min(K, V - c0) * 64) {
      *(lq_v4i*)(p.vqT + (cb * V + c0) * 64 + o) = *(const lq_v4i*)(lds + L::r1 + o);
      *(lq_v4i*)(p.vcT + (cb * V + c0) * 64 + o) = *(const lq_v4i*)(lds + L::r1 + K * 64 + o);
    }
  };
  // R in MFMA operand order: this wave rotates into channels 32 strip .., tile t takes the even / odd ones of them (a lane then
  // ends up with eight adjacent channels)
  constexpr int NS = K / 32, WPS = 8 / NS;
  const int strip = wave % NS, part_of = wave / NS;
  lq_v4i rop[ROT ? 2 : 1][KS];
  if constexpr (ROT) {
    auto operand = [&](const uint32_t (&w)[8], int ks) __attribute__((always_inline)) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        rop[0][ks][d] = (int)__builtin_amdgcn_perm(w[2 * d + 1], w[2 * d], 0x05040100u);
        rop[1][ks][d] = (int)__builtin_amdgcn_perm(w[2 * d + 1], w[2 * d], 0x07060302u);
      }
    };
    const int at0 = 8 * kg * K + 32 * strip + 2 * rl;
    if (FUSED && p.rot_op) {  // (uniform over the launch)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) rop[t][ks] = *(const lq_v4i*)(p.rot_op + (((strip * 2 + t) * KS + ks) * 64 + lane) * 8);
    } else if (FUSED && p.rot_f) {  // fp32, rounded here
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const zoo_v2f x = *(const zoo_v2f*)(p.rot_f + at0 + (32 * ks + e) * K);
          w[e] = zoo_pack_h2(x[0], x[1]);
        }
        operand(w, ks);
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = *(const uint32_t*)(p.rot + at0 + (32 * ks + e) * K);
        operand(w, ks);
      }
    }
  }
  if constexpr (MODE == DIAG_GLA) value_codes(0);
  __syncthreads();
  if constexpr (MODE == DIAG_GLA) value_copy(0);
  if constexpr (DO_A) {
    if (half == 0) {
      const lq_v4f d1 = *dg;
      lq_v4f o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = 4 * kg + r <= rl ? dacc[r] + d1[r] : 0.0f;
      a_store(tok, 16 * J + 4 * kg, o);
    }
  }

  // ---- 4: rotation of the nine operands into this wave's 32 channels, codes
  if constexpr (DO_A && ROT) {
    constexpr int NO = (9 + WPS - 1) / WPS;
    lq_v2i cd[NO];
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      const int o = part_of + WPS * i;
      if (o >= 9) continue;
      lq_v4f r[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const lq_v8h x = *(const lq_v8h*)(lds + L::r2 + L::X * o + (ks * 64 + lane) * 16);
        r[0] = lq_mfma_f16(__builtin_bit_cast(lq_v8h, rop[0][ks]), x, r[0]);
        r[1] = lq_mfma_f16(__builtin_bit_cast(lq_v8h, rop[1][ks]), x, r[1]);
      }
      const float inv = o < 3 ? inv_sq : inv_sk;
      int c[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) c[q] = zoo_q8(r[q & 1][q >> 1], inv, qmax);
      cd[i] = lq_v2i{(int)zoo_pack_codes(c[0], c[1], c[2], c[3]), (int)zoo_pack_codes(c[4], c[5], c[6], c[7])};
    }
    __syncthreads();  // the operands have been read
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      const int o = part_of + WPS * i;
      if (o >= 9) continue;
      *(lq_v2i*)(lds + L::r2 + L::CD * o + (strip >> 1) * 1024 + lane * 16 + 8 * (strip & 1)) = cd[i];
    }
  }
  // G: the second half's share, then the sum with the factors of its rows and columns
  if constexpr (DELTA) {
    if (half) {
#pragma unroll
      for (int di = -1; di < 3; ++di) {
        const int I = J + 1 + di;
        if (I > 3) continue;
        float* G = GT + g_blk(I, J) + rl;
#pragma unroll
        for (int r = 0; r < 4; ++r) G[(4 * kg + r) * kBP] = di < 0 ? gacc[r] : goff[di < 0 ? 0 : di][r];
      }
    }
  }
  __syncthreads();

  // ---- 5: INT8 products of the six off-diagonal blocks (transposed: lane: row rl of I, columns 4kg + r of J), zeros above
  if constexpr (DELTA) {
    if (half == 0) {
#pragma unroll
      for (int di = -1; di < 3; ++di) {
        const int I = J + 1 + di;
        if (I > 3) continue;
        const lq_v4f b4 = *(const lq_v4f*)(bs_s + 16 * I + 4 * kg);
        float* G = GT + g_blk(I, J) + rl;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = (di < 0 ? gacc[r] : goff[di < 0 ? 0 : di][r]) + G[(4 * kg + r) * kBP];
          G[(4 * kg + r) * kBP] = di >= 0 || 4 * kg + r > rl ? (b4[r] * bh) * v : 0.0f;
        }
      }
    }
  }
  if constexpr (DO_A) {
    // GLA: one to a wave; KDA: the first half's waves are busy with G, the others take one or two
#pragma unroll
    for (int s = 0; s < (DELTA ? 2 : 1); ++s) {
      const int pr = DELTA ? wave - 4 + 4 * s : wave;
      if (pr < 0 || pr >= 6 || (DELTA && wave < 4)) continue;
      const int Jp = pr < 3 ? 0 : (pr < 5 ? 1 : 2), Ip = pr < 3 ? pr + 1 : (pr < 5 ? pr - 1 : 3);
      lq_v4i acc = {0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < K / 64; ++ks)
        acc = lq_mfma_i8(*(const lq_v4i*)(lds + L::r2 + L::CD * (3 + pr) + ks * 1024 + lane * 16),
                         *(const lq_v4i*)(lds + L::r2 + L::CD * (Ip - 1) + ks * 1024 + lane * 16), acc);
      lq_v4f o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = (float)acc[r];
      a_store(16 * Ip + rl, 16 * Jp + 4 * kg, o);
      a_store(16 * Jp + rl, 16 * Ip + 4 * kg, lq_v4f{0.f, 0.f, 0.f, 0.f});
    }
  }
  if constexpr (MODE == DIAG_GLA) {
    for (int c0 = K; c0 < V; c0 += K) {  // further value channels
      request_values(c0);
      __syncthreads();
      value_codes(c0);
      __syncthreads();
      value_copy(c0);
    }
  }
  if constexpr (DELTA) {
    // first v columns, requested ahead of the inverse
    constexpr int VP = K / 64;  // 16-byte pieces of a pass per thread
    lq_v4i vraw[VP];
    auto request_v = [&](int vb) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < VP; ++i) {
        const int it = tid + 512 * i, t = it / (K / 8), c = vb + 8 * (it % (K / 8));
        vraw[i] = *(const lq_v4i*)(p.v + ((t0 + t) * H + h) * V + (c < V ? c : 0));
      }
    };
    request_v(0);
    // ---- T = (I + G)^-1: diagonal block J in the wave that has just written it
    if (half == 0) {
      float* B = GT + t_blk(J, J);
      float gr[16], tc[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) gr[i] = B[i * kBP + rl];
      zoo_substitute(gr, tc, rl);
      if (lane < 16) {
#pragma unroll
        for (int i = 1; i < 16; ++i) B[i * kBP + lane] = tc[i];
        B[lane] = tc[0];
      }
    }
    __syncthreads();
    // ---- 6: block column J of T by wave J: T_IJ = -T_II . sum_{J <= M < I} G_IM . T_MJ.  A block of the column is used as it comes
    // out of the MFMA (rows 4kg + s of column rl is the contraction slot 4kg + s of the next product)
    if (wave < 3) {
      lq_v4f tcol[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) tcol[0][s] = GT[t_blk(J, J) + (4 * kg + s) * kBP + rl];
#pragma unroll
      for (int di = 1; di < 4; ++di) {
        const int I = J + di;
        if (I > 3) break;
        lq_v4f sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dm = 0; dm < di; ++dm) {
          const lq_v4f g4 = *(const lq_v4f*)(GT + g_blk(I, J + dm) + rl * kBP + 4 * kg);
#pragma unroll
          for (int s = 0; s < 4; ++s) sacc = mfma_f32(g4[s], tcol[dm][s], sacc);
        }
        const lq_v4f t4 = *(const lq_v4f*)(GT + t_blk(I, I) + rl * kBP + 4 * kg);
        lq_v4f tacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s) tacc = mfma_f32(t4[s], sacc[s], tacc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          tcol[di][r] = -tacc[r];
          GT[t_blk(I, J) + (4 * kg + r) * kBP + rl] = -tacc[r];
        }
      }
    }
    __syncthreads();
    // T in pieces: twelve blocks of 16 columns (two of them zero) over the waves
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int n = wave + 8 * q;  // (step, M parity): steps (0,0) (1,0) (2,0) (2,1) (3,0) (3,1)
      if (n >= 2 * kSteps) continue;
      const int step = n >> 1, I = step < 2 ? step : 1 + (step >> 1), M = (step < 2 ? 0 : 2 * (step & 1)) + (n & 1);
      lq_v4f t = {0.f, 0.f, 0.f, 0.f};
      if (M <= I) t = *(const lq_v4f*)(GT + t_blk(I, M) + rl * kBP + 4 * kg);
      uint32_t pc[2][3];
      split3(t[0], t[1], pc[0][0], pc[0][1], pc[0][2]);
      split3(t[2], t[3], pc[1][0], pc[1][1], pc[1][2]);
#pragma unroll
      for (int i = 0; i < 3; ++i) *(lq_v2i*)(TP + (i * kSteps + step) * 512 + lane * 8 + 4 * (n & 1)) = lq_v2i{(int)pc[0][i], (int)pc[1][i]};
    }
    __syncthreads();

    // ---- 7: W = T (beta^sigma k e^g), U = T (beta^sigma v), transposed: lane: token 16I + rl, channels 16nt + 4kg + r.  Row blocks
    // 0, 3 and then 1, 2 (three steps each) of a column tile to a wave, or, where there are fewer tiles than waves, either to one of two
    // x: tokens 16M + 4kg + s of the lane's column
    auto split_x = [&](const float (&x)[4][4], lq_v4i (&xp)[3][2]) __attribute__((always_inline)) {
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          uint32_t pc[3];
          split3(x[2 * st + (d >> 1)][2 * (d & 1)], x[2 * st + (d >> 1)][2 * (d & 1) + 1], pc[0], pc[1], pc[2]);
#pragma unroll
          for (int i = 0; i < 3; ++i) xp[i][st][d] = (int)pc[i];
        }
    };
    // row blocks u and 3 - u; six of the nine products of pieces: the others are 2^-21 of the leading one at most
    auto product = [&](int u, const lq_v4i (&xp)[3][2], lq_v4f (&acc)[2]) __attribute__((always_inline)) {
      acc[0] = acc[1] = lq_v4f{0.f, 0.f, 0.f, 0.f};
      const uint16_t* const t_at = TP + lane * 8;
#pragma unroll
      for (int sum = 2; sum >= 0; --sum)  // smallest first
#pragma unroll
        for (int i = 0; i <= sum; ++i) {
          const uint16_t* const tq = t_at + (sum - i) * (kSteps * 512);
          acc[0] = mfma_bf16(xp[i][0], *(const lq_v4i*)(tq + u * 512), acc[0]);
          acc[1] = mfma_bf16(xp[i][0], *(const lq_v4i*)(tq + (u ? 2 : 4) * 512), acc[1]);
          acc[1] = mfma_bf16(xp[i][1], *(const lq_v4i*)(tq + (u ? 3 : 5) * 512), acc[1]);
        }
    };
    // places of tokens 4kg + s (of sub-block 0) of column 16nt + rl in the tile
    auto column = [&](int nt, int (&xi)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 4; ++s) xi[s] = at<K>(4 * kg + s, 16 * nt + rl);
    };
    constexpr bool SPLIT = K == 64;  // four column tiles: two waves to each
    const int ntile = SPLIT ? wave & 3 : wave;
    const float inv_sw = codes ? 1.0f / p.sw[h] : 0.0f;
    {
      int xi[4];
      column(ntile, xi);
      float x[4][4];
#pragma unroll
      for (int M = 0; M < 4; ++M) {
        const float E = E_s[M * K + 16 * ntile + rl];
        const lq_v4f b4 = *(const lq_v4f*)(bs_s + 16 * M + 4 * kg);
#pragma unroll
        for (int s = 0; s < 4; ++s) x[M][s] = (R1[xi[s] + M * (KS * 512)] * E) * b4[s];
      }
      lq_v4i xp[3][2];
      split_x(x, xp);
#pragma unroll
      for (int q = 0; q < (SPLIT ? 1 : 2); ++q) {
        const int u = SPLIT ? half : q;
        lq_v4f acc[2];
        product(u, xp, acc);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int I = i ? 3 - u : u;
          lq_v2i o;
          o[0] = (int)zoo_enc2(acc[i][0], acc[i][1], bf);
          o[1] = (int)zoo_enc2(acc[i][2], acc[i][3], bf);
          const int64_t woff = FUSED ? cb * 64 * K + zoo_op_codes(16 * I + rl, 16 * ntile + 4 * kg, K)
                                     : ((t0 + 16 * I + rl) * H + h) * K + 16 * ntile + 4 * kg;
          if constexpr (!FUSED) {
            if (p.W) *(lq_v2i*)(p.W + woff) = o;
          }
          if (codes) {  // state-read codes of the rounded W
            float w0, w1, w2, w3;
            zoo_dec2((uint32_t)o[0], bf, w0, w1);
            zoo_dec2((uint32_t)o[1], bf, w2, w3);
            *(uint32_t*)(p.wq + woff) = zoo_pack_codes(zoo_q8(w0, inv_sw, qmax), zoo_q8(w1, inv_sw, qmax), zoo_q8(w2, inv_sw, qmax),
                                                       zoo_q8(w3, inv_sw, qmax));
          }
        }
      }
    }
#pragma unroll 1
    for (int vb = 0; vb < V; vb += K) {
      if (vb > 0) request_v(vb);
      __syncthreads();  // the tile has been read
#pragma unroll
      for (int i = 0; i < VP; ++i) {
        const int it = tid + 512 * i, t = it / (K / 8), c = 8 * (it % (K / 8));
        float x[8];
#pragma unroll
        for (int d = 0; d < 4; ++d) zoo_dec2((uint32_t)vraw[i][d], bf, x[2 * d], x[2 * d + 1]);
        const float bt_ = bs_s[t];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = bt_ * x[e];
        *(lq_v4f*)(R1 + at<K>(t, c)) = lq_v4f{x[0], x[1], x[2], x[3]};
        *(lq_v4f*)(R1 + at<K>(t, c + 4)) = lq_v4f{x[4], x[5], x[6], x[7]};
      }
      __syncthreads();
      // a pass of K columns as above; of 64 out of 128: two waves to a tile
      const bool pairs = SPLIT || V - vb < 128;
      const int nt = pairs ? wave & 3 : wave;
      int xi[4];
      column(nt, xi);
      float x[4][4];
#pragma unroll
      for (int M = 0; M < 4; ++M)
#pragma unroll
        for (int s = 0; s < 4; ++s) x[M][s] = R1[xi[s] + M * (KS * 512)];
      lq_v4i xp[3][2];
      split_x(x, xp);
#pragma unroll 1
      for (int u = pairs ? half : 0; u < (pairs ? half + 1 : 2); ++u) {
        lq_v4f acc[2];
        product(u, xp, acc);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int I = i ? 3 - u : u;
          lq_v2i o;
          o[0] = (int)zoo_enc2(acc[i][0], acc[i][1], bf);
          o[1] = (int)zoo_enc2(acc[i][2], acc[i][3], bf);
          *(lq_v2i*)(FUSED ? p.U + cb * 64 * V + zoo_op_U(16 * I + rl, vb + 16 * nt + 4 * kg)
                           : p.U + ((t0 + 16 * I + rl) * H + h) * V + vb + 16 * nt + 4 * kg) = o;
        }
      }
    }
  }
}

template <int K, bool ROT, bool BF, int MODE, bool DK, bool GATE>
int launch_one(const ZooDiagParams& p, hipStream_t stream) {
  const dim3 grid = zoo_unit_grid(p.B, p.NT, p.H);
  hipLaunchKernelGGL((zoo_diag_prep_kernel<K, ROT, BF, MODE, DK, GATE>), grid, dim3(512), 0, stream, p);
  return lq_check_launch();
}

template <int K, bool ROT, int MODE, bool DK>
int launch_bf(const ZooDiagParams& p, hipStream_t stream) {
  if constexpr (MODE == DIAG_WY || MODE == DIAG_KDA) {
    if ((1.0f - p.sigma) * p.tau != 0.0f)
      return p.bf ? launch_one<K, ROT, true, MODE, DK, true>(p, stream) : launch_one<K, ROT, false, MODE, DK, true>(p, stream);
  }
  return p.bf ? launch_one<K, ROT, true, MODE, DK, false>(p, stream) : launch_one<K, ROT, false, MODE, DK, false>(p, stream);
}

template <int K, int MODE, bool DK>
int launch_rot(const ZooDiagParams& p, hipStream_t stream) {
  if constexpr (MODE != DIAG_WY) {
    if (p.rot || p.rot_f || p.rot_op) return launch_bf<K, true, MODE, DK>(p, stream);
  }
  return launch_bf<K, false, MODE, DK>(p, stream);
}

template <int K, int MODE>
int launch_dk(const ZooDiagParams& p, hipStream_t stream) {
  if constexpr (MODE != DIAG_GLA) {
    if (MODE == DIAG_WY ? p.dk_div != nullptr : p.dq != nullptr) return launch_rot<K, MODE, true>(p, stream);
  }
  return launch_rot<K, MODE, false>(p, stream);
}

template <int MODE>
int launch(const ZooDiagParams& p, int K, hipStream_t stream) {
  return K == 128 ? launch_dk<128, MODE>(p, stream) : launch_dk<64, MODE>(p, stream);
}

}  // namespace zoo_diag
