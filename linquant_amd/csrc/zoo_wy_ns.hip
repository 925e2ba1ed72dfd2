// WY / UT transform of the delta family with no or scalar decay (DeltaNet, Gated DeltaNet), 64-token chunks, with everything the
// chunk recurrence wants of a chunk made in the same launch.
// Replaces the torch prep linquant/kernels/zoo/gated_delta_rule.py:20-47 and the operand preparation of the state and output
// bodies (gated_delta_rule.py:85-105, simple_gla.py:125-140):
//   G[i][j] = bs_i bh_j (k_i . k_j) * exp(g_i - g_j) for i > j,  bs = beta^sigma, bh = beta^(1-sigma);  T = (I + G)^-1
//   W = T (bs k exp(g)),  U = T (bs v),  Hw = beta^((1-sigma) tau) k,  fw = beta^((1-sigma)(1-tau))
//
// Nothing but per-token factors separates the operands of these products from k and v themselves, and a per-token factor is an
// index of T's columns.  So the half-precision rows stay exact and all arithmetic goes to T:
//   Gram: k . k^T on the half-precision MFMA (exact products, fp32 accumulation), the factors applied to the 64 x 64 result;
//   W, U: (T . diag(bs exp(g))) . k and (T . diag(bs)) . v with k and v as they are and only T split, in three half-precision
//     pieces that together hold the 24 bits of an fp32 entry.  bf16 pieces have fp32's range.  fp16 pieces: each row is scaled by a
//     power of two to just below fp16's range and the third piece by another 2^22, in an accumulator that is scaled back before
//     the other two are added: what is left of an entry is below 2^-51 of its row's largest (two pieces left 2^-39, which behind a
//     strong decay and in front of a large value cost half of an entry's bits).
//     Share of W, U entries on the other side of a rounding boundary than the float64 result (B4 T2048 H16 K = V = 128, unit keys;
//     two fp16 pieces, and the fp32 form below, in brackets): fp16 2.6e-4, 2.9e-4 (2.9e-4, 3.3e-4; 4.5e-4, 5.4e-4), with scalar decay
//     1.1e-4, 0.9e-4 (1.2e-4, 1.2e-4; 1.3e-4, 1.6e-4); bf16 5.0e-5, 4.5e-5 (fp32 form 9.5e-5, 8.7e-5).  The third fp16 piece costs 6
//     us of 256 (Gated DeltaNet B4 T4096 H16, whole call).
// An fp32 form of the same (operands scaled and staged as fp32, 32 fp32 MFMA steps per Gram block, T and X split in three bf16
// pieces, six products) took 121 us at B4 T4096 H16 K = V = 128, of which the splitting and the fp32 steps were two thirds, and left
// the codes of q and the product A to the output kernel; this one takes 117 us with them and with scalar decay.
//
// One 8-wave workgroup per (chunk, batch*head), three to a compute unit (49 KB of LDS, 80 registers): load and quantize | Gram blocks and,
// MODE_SCAN, the blocks of the intra-chunk product A (20 blocks over the 8 waves) | G; keys transposed | inverse of the four diagonal
// blocks by forward substitution | block columns of T, one wave each, in registers | W | values transposed | U.  Keys and then values
// pass through one transposed tile, the rows waiting in registers (every row is read once), and G and T lie in 16 blocks in the place of
// the raw keys and codes.  With a tile each for keys and values and square G and T (77 KB) two workgroups fitted, which did not cover each
// other's waits between eight barriers: on one card in turn 130.4 -> 116 to 120 us at B4 T4096 H16 with scalar decay (fp16), 61.3 -> 56.5 at B8
// T2048 H8 without (bf16; 2.7 rounds of the chip for four), although there are two barriers more.  Bound by no unit alone: 410 MB are 81 us
// at the rate of a large copy and the vector instructions 82 us.
#include "zoo_params.h"

namespace {

enum { MODE_PLAIN = 0, MODE_CODES = 1, MODE_SCAN = 2 };
// MODE_PLAIN: Hw, W, U, fw.  MODE_CODES: also the write operands of the state kernel (W stored only when p.W is set).
// MODE_SCAN: what zoo_scan.hip wants: the write operands, wq and U in operand order, the codes of q and the product A; no Hw.  The log
// decay per token comes in as it is and is cumulated here, while the rows are on their way (the others: cumulated): a launch of 4.8 us for
// 2 MB less at B4 T4096 H16, whole call 248.7 -> 238.

LQ_DEV lq_v4f wn_mfma_f32(float a, float b, lq_v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

typedef __bf16 wn_v8bf __attribute__((ext_vector_type(8)));

template <bool BF>
LQ_DEV lq_v4f wn_mfma(lq_v4i a, lq_v4i b, lq_v4f c) {
  if constexpr (BF) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wn_v8bf, a), __builtin_bit_cast(wn_v8bf, b), c, 0, 0, 0);
  return lq_mfma_f16(__builtin_bit_cast(lq_v8h, a), __builtin_bit_cast(lq_v8h, b), c);
}

// 16 x 16 blocks of T (lower triangle; the diagonal ones hold G first) and of G below the diagonal, rows of 20 floats
constexpr int kBP = 20;
constexpr int kBlk = 16 * kBP;
LQ_DEV int wn_t(int I, int J) { return (I * (I + 1) / 2 + J) * kBlk; }
LQ_DEV int wn_g(int I, int J) { return I == J ? wn_t(I, I) : (10 + I * (I - 1) / 2 + J) * kBlk; }
constexpr int kXP = 36;   // dwords per column of the transposed tiles (32 token pairs + pad)
// byte of the transposed write codes [channel][64 tokens]: 16 bytes of pad after every eight channels, so that the 16 channel
// groups of a wave's writes fall on different banks (rows of 80 bytes put them on two: Gated DeltaNet B4 T4096 H16 260 -> 256 us,
// DeltaNet B8 T2048 H8 bf16 101 -> 99 for the whole call)
LQ_DEV int wn_ct(int ch, int token) { return ch * 64 + (ch >> 3) * 16 + token; }

// dword of the transposed tile [column][token pair]; the pairs are permuted in groups of four (one 16-byte operand piece) so that
// the writes of a wave (16 groups of eight columns x 4 pairs) fall on 64 different banks
LQ_DEV int wn_xt(int col, int pair) { return col * kXP + (pair ^ (((col >> 4) & 7) << 2)); }

LQ_DEV float wn_powb(float b, float e) {
  if (e == 0.0f) return 1.0f;
  if (e == 1.0f) return b;
  return __builtin_amdgcn_exp2f(e * __builtin_amdgcn_logf(b));
}

// T operand of one row block and contraction step: eight values of a row (fp16: scaled) as three pieces (fp16: the third
// times 2^22)
template <bool BF>
struct TPieces {
  lq_v4i p[3];
};

template <bool BF>
LQ_DEV void wn_split(const float (&x)[8], TPieces<BF>& t) {
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const float x0 = x[2 * d], x1 = x[2 * d + 1];
    if constexpr (BF) {  // upper 16 bits of what the pieces before leave: 24 significant bits in all
      const uint32_t b0 = __float_as_uint(x0), b1 = __float_as_uint(x1);
      t.p[0][d] = (int)__builtin_amdgcn_perm(b1, b0, 0x07060302u);
      const float r0 = x0 - __uint_as_float(b0 & 0xffff0000u), r1 = x1 - __uint_as_float(b1 & 0xffff0000u);
      const uint32_t c0 = __float_as_uint(r0), c1 = __float_as_uint(r1);
      t.p[1][d] = (int)__builtin_amdgcn_perm(c1, c0, 0x07060302u);
      const float q0 = r0 - __uint_as_float(c0 & 0xffff0000u), q1 = r1 - __uint_as_float(c1 & 0xffff0000u);
      t.p[2][d] = (int)__builtin_amdgcn_perm(__float_as_uint(q1), __float_as_uint(q0), 0x07060302u);
    } else {
      const _Float16 b0 = (_Float16)x0, b1 = (_Float16)x1;
      t.p[0][d] = __builtin_bit_cast(int, lq_v2h{b0, b1});
      const float r0 = x0 - (float)b0, r1 = x1 - (float)b1;
      const _Float16 c0 = (_Float16)r0, c1 = (_Float16)r1;
      t.p[1][d] = __builtin_bit_cast(int, lq_v2h{c0, c1});
      t.p[2][d] = (int)zoo_pack_h2((r0 - (float)c0) * 0x1p22f, (r1 - (float)c1) * 0x1p22f);
    }
  }
}

template <bool SCALAR, int K, bool BF, int MODE>
__global__ __launch_bounds__(512, 6) void zoo_wy_ns_kernel(ZooWyParams p) {
  constexpr bool CODES = MODE != MODE_PLAIN, SCAN = MODE == MODE_SCAN;
  constexpr int FS = K + 16;                      // halves per row of the raw key tile (72 or 40 dwords: two-pass operand reads)
  constexpr int QS = K == 128 ? 160 : 80;         // bytes per row of the code tiles
  constexpr int kF_bytes = 64 * FS * 2, kQ_bytes = 2 * 64 * QS;                 // raw keys, codes of q and k, and behind them the transposed
  constexpr int kP1 = kF_bytes + kQ_bytes + (CODES ? K * 66 : 0);               // write codes; then
  constexpr int kGT = 16 * kBlk * 4, kP2 = kGT + 128 * kXP * 4;                 // G and T, and keys, then values, transposed
  __shared__ __align__(16) unsigned char lds[kP1 > kP2 ? kP1 : kP2];
  _Float16* kF = (_Float16*)lds;
  unsigned char* qI = lds + kF_bytes;
  unsigned char* kI = qI + 64 * QS;
  unsigned char* cT = lds + kF_bytes + kQ_bytes;
  float* GT = (float*)lds;
  uint32_t* X = (uint32_t*)(lds + kGT);
  __shared__ float bs_s[64], bh_s[64], bw_s[64], el_s[64], fW_s[64], gs_s[64], iskw_s[CODES ? K : 1];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rl = lane & 15, kg = lane >> 4;
  ZooUnit unit;
  if (!zoo_unit(p.B, p.NT, p.H, unit)) return;
  const int h = unit.h, b = unit.b, ct = unit.ct;
  const int H = p.H, V = p.V, qmax = p.qmax;
  const int64_t t0 = (int64_t)b * p.T + (int64_t)ct * 64;
  const int64_t cb = ((int64_t)b * p.NT + ct) * H + h;
  constexpr bool bf = BF;

  // ---- requests: a thread takes two adjacent tokens x 8 channels of k, q and (first 128 columns) v
  constexpr int KP = K / 8;  // 16-byte pieces of a key row
  const int krp = tid / KP, kc = tid % KP;
  const bool kact = K == 128 || tid < 256;
  const int vsh = V >= 128 ? 4 : 3;  // (V is a multiple of 64: 16 or 8 pieces of a value row per pass)
  const int vrp = tid >> vsh, vc8 = tid & ((1 << vsh) - 1);
  const bool vact = vrp < 32;
  lq_v4i kraw[2], qraw[2], vraw[2];
  const int64_t head = (t0 * H + h) * K, vstep = (int64_t)H * V;  // (uniform)
  const _Float16* const vrow = p.v + (t0 * vstep + (int64_t)h * V) + (vact ? 2 * vrp : 0) * vstep + 8 * vc8;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const uint32_t at = 2 * (zoo_rows(2 * (kact ? krp : 0) + u, H, K) + 8 * kc);
    kraw[u] = zoo_at<lq_v4i>(p.k + head, at);
    if constexpr (SCAN) qraw[u] = zoo_at<lq_v4i>(p.q + head, at);
    vraw[u] = *(const lq_v4i*)(vrow + u * vstep);
  }
  // ---- per-token factors
  if (tid < 64) {
    const float bt = zoo_at<float>(p.beta + t0 * H + h, 4 * zoo_rows(tid, H, 1));
    const float bs = wn_powb(bt, p.sigma);
    const float fwv = wn_powb(bt, (1.0f - p.sigma) * (1.0f - p.tau));
    float gv = 0.0f, gl = 0.0f;
    if constexpr (SCALAR && SCAN) {
      gv = zoo_cumsum64(zoo_at<float>(p.g + t0 * H + h, 4 * zoo_rows(tid, H, 1)));
      gl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gv), 63));
    } else if constexpr (SCALAR) {
      gv = p.g[(t0 + tid) * H + h], gl = p.g[(t0 + 63) * H + h];
    }
    bs_s[tid] = bs;
    bh_s[tid] = wn_powb(bt, 1.0f - p.sigma);
    bw_s[tid] = wn_powb(bt, (1.0f - p.sigma) * p.tau);
    gs_s[tid] = gv;
    fW_s[tid] = SCALAR ? bs * zoo_exp_acc(gv) : bs;
    el_s[tid] = SCALAR ? zoo_exp((1.0f - p.eta) * (gl - gv)) : 1.0f;
    float* pk = p.pack ? p.pack + cb * (128 + K) : nullptr;
    if (!SCAN) p.fw[(t0 + tid) * H + h] = fwv;
    if constexpr (CODES) {
      const float evv = SCALAR ? zoo_exp(p.eta * (gl - gv)) : 1.0f;
      if (!SCAN) p.ev[(t0 + tid) * H + h] = evv;
      if (pk) pk[tid] = fwv, pk[64 + tid] = evv;
      if (SCAN && SCALAR) p.gpk[cb * 64 + tid] = gv;
    }
  } else if (CODES && tid >= 128 && tid < 128 + K) {
    const int n = tid - 128;
    if constexpr (!SCAN) {
      const float gm = SCALAR ? zoo_exp(p.g[(t0 + 63) * H + h]) : 1.0f;
      p.gam[cb * K + n] = gm;
      if (p.pack) p.pack[cb * (128 + K) + 128 + n] = gm;
    }
    iskw_s[n] = 1.0f / p.skw[h * K + n];
  }
  __syncthreads();
  if constexpr (SCAN) {
    if (tid < K) p.pack[cb * (128 + K) + 128 + tid] = SCALAR ? zoo_exp(gs_s[63]) : 1.0f;
  }

  // ---- rows into LDS: raw keys by token (Gram), codes of q and Hw, transposed write codes
  if (kact) {
    if (p.dk_div) {  // D_QK at load: k' = act(k / D), the quotient rounded once (uniform over the launch)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const int n = h * K + 8 * kc + 2 * d;
          float x0, x1;
          zoo_dec2((uint32_t)kraw[u][d], bf, x0, x1);
          kraw[u][d] = (int)zoo_enc2(zoo_div_rn(x0, p.dk_div[n], p.dk_rcp[n]), zoo_div_rn(x1, p.dk_div[n + 1], p.dk_rcp[n + 1]), bf);
        }
    }
    float inv_sq = 0.0f, inv_sk = 0.0f;
    if constexpr (SCAN) inv_sq = 1.0f / p.sq[h], inv_sk = 1.0f / p.sk[h];
    uint32_t wc[2][8];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = 2 * krp + u;
      *(lq_v4i*)(kF + t * FS + 8 * kc) = kraw[u];
      const float bw = bw_s[t], el = el_s[t];
      lq_v2i ok, oq;
      lq_v4i hw;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        float x0, x1;
        zoo_dec2((uint32_t)kraw[u][d], bf, x0, x1);
        // Hw as it would be stored, rounded to fp32 first (folded into one rounding, a product next to a midpoint went the other
        // way than the stored Hw in some of the instantiations, and its code with it)
        hw[d] = (int)zoo_enc2(zoo_mul_rn(bw, x0), zoo_mul_rn(bw, x1), bf);
      }
      if constexpr (!SCAN) zoo_put(p.Hw + head, 2 * (zoo_rows(t, H, K) + 8 * kc), hw);
      if constexpr (CODES) {
        int ck[8], cq[8];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          float x0, x1;
          zoo_dec2((uint32_t)hw[d], bf, x0, x1);
          if constexpr (SCAN) ck[2 * d] = zoo_q8(x0, inv_sk, qmax), ck[2 * d + 1] = zoo_q8(x1, inv_sk, qmax);
          if (SCALAR) x0 = x0 * el, x1 = x1 * el;
          wc[u][2 * d] = (uint32_t)zoo_q8(x0, iskw_s[8 * kc + 2 * d], qmax);
          wc[u][2 * d + 1] = (uint32_t)zoo_q8(x1, iskw_s[8 * kc + 2 * d + 1], qmax);
          if constexpr (SCAN) {
            zoo_dec2((uint32_t)qraw[u][d], bf, x0, x1);
            cq[2 * d] = zoo_q8(x0 * p.scale, inv_sq, qmax), cq[2 * d + 1] = zoo_q8(x1 * p.scale, inv_sq, qmax);
          }
        }
        if constexpr (SCAN) {
          ok[0] = (int)zoo_pack_codes(ck[0], ck[1], ck[2], ck[3]), ok[1] = (int)zoo_pack_codes(ck[4], ck[5], ck[6], ck[7]);
          oq[0] = (int)zoo_pack_codes(cq[0], cq[1], cq[2], cq[3]), oq[1] = (int)zoo_pack_codes(cq[4], cq[5], cq[6], cq[7]);
          *(lq_v2i*)(kI + t * QS + 8 * kc) = ok;
          *(lq_v2i*)(qI + t * QS + 8 * kc) = oq;
        }
      }
    }
    if constexpr (CODES) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        *(uint16_t*)(cT + wn_ct(8 * kc + e, 2 * krp)) = (uint16_t)__builtin_amdgcn_perm(wc[1][e], wc[0][e], 0x0c0c0400u);
    }
  }
  __syncthreads();

  // ---- the write codes leave as whole rows
  if constexpr (CODES) {
    if (tid < K * 4) zoo_put(p.kqT + cb * K * 64, 16 * tid, *(const lq_v4i*)(cT + wn_ct(tid >> 2, 16 * (tid & 3))));
  }
  // ---- Gram blocks (tasks 0..9) and, MODE_SCAN, A blocks (tasks 10..19): task t belongs to wave t % 8
  // block n of the lower triangle: (0,0) (1,0) (1,1) (2,0) (2,1) (2,2) (3,0) ..
  auto blk_i = [](int n) { return n < 1 ? 0 : (n < 3 ? 1 : (n < 6 ? 2 : 3)); };
  auto blk_j = [](int n) { return n < 1 ? 0 : (n < 3 ? n - 1 : (n < 6 ? n - 3 : n - 6)); };
  lq_v4f gacc[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    gacc[s] = lq_v4f{0.f, 0.f, 0.f, 0.f};
    const int n = wave + 8 * s;
    if (n >= 10) continue;
    const _Float16* ra = kF + (16 * blk_i(n) + rl) * FS + 8 * kg;
    const _Float16* rb = kF + (16 * blk_j(n) + rl) * FS + 8 * kg;
#pragma unroll
    for (int ks = 0; ks < K / 32; ++ks) gacc[s] = wn_mfma<BF>(*(const lq_v4i*)(ra + 32 * ks), *(const lq_v4i*)(rb + 32 * ks), gacc[s]);
  }
  if constexpr (SCAN) {
    const float sqk = p.sq[h] * p.sk[h];
#pragma unroll
    for (int s = 1; s < 3; ++s) {
      const int n = wave + 8 * s - 10;  // (A blocks: tasks 10 .. 19)
      if (n < 0 || n >= 10) continue;
      const int I = blk_i(n), J = blk_j(n);
      lq_v4i acc = {0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < K / 64; ++ks)  // transposed: lane (rl, kg) holds row 16I + rl, columns 16J + 4kg + r
        acc = lq_mfma_i8(*(const lq_v4i*)(kI + (16 * J + rl) * QS + 64 * ks + 16 * kg), *(const lq_v4i*)(qI + (16 * I + rl) * QS + 64 * ks + 16 * kg), acc);
      const int i = 16 * I + rl, j0 = 16 * J + 4 * kg;
      float x[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[r] = (float)acc[r] * sqk;
        if (SCALAR) x[r] = x[r] * zoo_exp(gs_s[i] - gs_s[j0 + r]);
        x[r] = j0 + r <= i ? x[r] : 0.0f;
      }
      zoo_put(p.A + cb * 4096, 2 * zoo_op_A(i, j0), lq_v2i{(int)zoo_pack_h2(x[0], x[1]), (int)zoo_pack_h2(x[2], x[3])});
    }
    // zero blocks above the diagonal (waves 4 .. 7, which have a task less) and the codes of q, operand by operand (waves 0 .. 3)
    if (wave >= 4) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int n = wave - 4 + 4 * s;  // (0,1) (0,2) (0,3) (1,2) (1,3) (2,3)
        if (n >= 6) continue;
        const int I = n < 3 ? 0 : (n < 5 ? 1 : 2), J = n < 3 ? n + 1 : (n < 5 ? n - 1 : 3);
        zoo_put(p.A + cb * 4096, 2 * zoo_op_A(16 * I + rl, 16 * J + 4 * kg), lq_v2i{0, 0});
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < K / 64; ++ks)
        zoo_put(p.qc + cb * 64 * K, ((wave * (K / 64) + ks) * 64 + lane) * 16, *(const lq_v4i*)(qI + (16 * wave + rl) * QS + 64 * ks + 16 * kg));
    }
  }
  __syncthreads();  // raw keys, codes and transposed codes are dead

  // ---- G, with the factors of its rows and columns; k transposed
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int n = wave + 8 * s;
    if (n >= 10) continue;
    const int j = 16 * blk_j(n) + rl;  // lane holds column j, rows i = 4kg + r of the block
    const float bh = bh_s[j], gj = gs_s[j];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * blk_i(n) + 4 * kg + r;
      float x = (bs_s[i] * bh) * gacc[s][r];
      if (SCALAR) x = x * zoo_exp(gs_s[i] - gj);
      GT[wn_g(blk_i(n), blk_j(n)) + (4 * kg + r) * kBP + rl] = i > j ? x : 0.0f;
    }
  }
  // two rows of eight channels -> transposed tile
  auto stage = [&](const lq_v4i (&raw)[2], int c8, int pair) __attribute__((always_inline)) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      X[wn_xt(8 * c8 + 2 * d, pair)] = __builtin_amdgcn_perm((uint32_t)raw[1][d], (uint32_t)raw[0][d], 0x05040100u);
      X[wn_xt(8 * c8 + 2 * d + 1, pair)] = __builtin_amdgcn_perm((uint32_t)raw[1][d], (uint32_t)raw[0][d], 0x07060302u);
    }
  };
  if (kact) stage(kraw, kc, krp);
  __syncthreads();

  // ---- T = (I + G)^-1: diagonal blocks by forward substitution (wave w < 4, lane c of every 16 holds column c of block w)
  if (wave < 4) {
    float* B = GT + wn_t(wave, wave);
    float gr[16], tc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) gr[i] = B[i * kBP + rl];
    zoo_substitute(gr, tc, rl);
    if (lane < 16) {
#pragma unroll
      for (int i = 0; i < 16; ++i) B[i * kBP + lane] = tc[i];
    }
  }
  __syncthreads();
  // block column J of T by wave J: T_IJ = -T_II . sum_{J <= M < I} G_IM . T_MJ.  A block of the column is used as it comes out of
  // the MFMA (rows 4kg + s of column rl is the contraction slot 4kg + s of the next product), so the column stays in registers.
  if (wave < 3) {
    const int J = wave;
    lq_v4f tcol[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) tcol[0][s] = GT[wn_t(J, J) + (4 * kg + s) * kBP + rl];
#pragma unroll
    for (int di = 1; di < 4; ++di) {
      const int I = J + di;
      if (I > 3) break;
      lq_v4f sacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dm = 0; dm < di; ++dm) {
        const lq_v4f g4 = *(const lq_v4f*)(GT + wn_g(I, J + dm) + rl * kBP + 4 * kg);
#pragma unroll
        for (int s = 0; s < 4; ++s) sacc = wn_mfma_f32(g4[s], tcol[dm][s], sacc);
      }
      const lq_v4f t4 = *(const lq_v4f*)(GT + wn_t(I, I) + rl * kBP + 4 * kg);
      lq_v4f tacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) tacc = wn_mfma_f32(t4[s], sacc[s], tacc);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        tcol[di][r] = -tacc[r];
        GT[wn_t(I, J) + (4 * kg + r) * kBP + rl] = -tacc[r];
      }
    }
  }
  __syncthreads();

  // ---- W and U: wave w takes row block I (w, or 7 - w: the two waves of a SIMD have the same work as any other two) and half of
  // the column tiles of both
  const int I = wave < 4 ? wave : 7 - wave, half = wave >> 2;
  const int NST = (I >> 1) + 1;  // 32-token contraction steps that are not zero
  // T . diag(f) for this row block in pieces; un: what the sums are to be multiplied by
  auto t_pieces = [&](const float* f, TPieces<BF> (&t)[2], float& un) __attribute__((always_inline)) {
    float x[2][8];
    float m = 0.0f;
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      if (st >= NST) continue;  // (wave-uniform)
      const int m0 = 32 * st + 8 * kg, M = 2 * st + (kg >> 1);
      const bool live = M <= I;  // blocks right of the diagonal were never written
      const float* row = GT + wn_t(I, live ? M : I) + rl * kBP + 8 * (kg & 1);
      const lq_v4f lo = *(const lq_v4f*)row, hi = *(const lq_v4f*)(row + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = live ? (e < 4 ? lo[e & 3] : hi[e & 3]) : 0.0f;
        x[st][e] = v * f[m0 + e];
        m = fmaxf(m, __builtin_fabsf(x[st][e]));
      }
    }
    un = 1.0f;
    if constexpr (!BF) {
      // each row scaled so that its largest entry lies in [2^14, 2^15)
      m = fmaxf(m, __shfl_xor(m, 16));
      m = fmaxf(m, __shfl_xor(m, 32));
      const int e = min(max((int)(__float_as_uint(m) >> 23), 16), 254);  // largest entry 2^(e - 127) .. 2^(e - 126)
      un = __uint_as_float((uint32_t)(e - 14) << 23);
      const float s = __uint_as_float((uint32_t)(268 - e) << 23);  // 2^(141 - e)
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (st < NST) x[st][e] = x[st][e] * s;
    }
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      if (st >= NST) continue;
      wn_split<BF>(x[st], t[st]);
    }
  };
  TPieces<BF> t[2];
  float un;
  t_pieces(fW_s, t, un);
  // D^T tile: lane (rl = token of block I, kg) gets columns 16nt + 4kg + r
  auto tile = [&](int nt) __attribute__((always_inline)) {
    lq_v4f acc = {0.f, 0.f, 0.f, 0.f};
    lq_v4i x[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      if (st >= NST) continue;
      x[st] = *(const lq_v4i*)(X + wn_xt(16 * nt + rl, 16 * st + 4 * kg));
#pragma unroll
      for (int i = 2; i >= (BF ? 0 : 2); --i) acc = wn_mfma<BF>(x[st], t[st].p[i], acc);
    }
    if constexpr (!BF) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] = acc[r] * 0x1p-22f;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        if (st >= NST) continue;
#pragma unroll
        for (int i = 1; i >= 0; --i) acc = wn_mfma<BF>(x[st], t[st].p[i], acc);
      }
    }
    return acc;
  };
  const float inv_sw = CODES ? 1.0f / p.sw[h] : 0.0f;
#pragma unroll
  for (int q = 0; q < K / 32; ++q) {
    const int nt = half * (K / 32) + q;
    const lq_v4f a = tile(nt);
    lq_v2i o;
    o[0] = (int)zoo_enc2(a[0] * un, a[1] * un, bf);
    o[1] = (int)zoo_enc2(a[2] * un, a[3] * un, bf);
    const uint32_t wat = zoo_rows(16 * I + rl, H, K) + 16 * nt + 4 * kg;  // (token-major forms)
    if (!SCAN && (!CODES || p.W)) zoo_put(p.W + head, 2 * wat, o);
    if constexpr (CODES) {  // state-read codes of the rounded W
      float w0, w1, w2, w3;
      zoo_dec2((uint32_t)o[0], bf, w0, w1);
      zoo_dec2((uint32_t)o[1], bf, w2, w3);
      zoo_put(p.wq + (SCAN ? cb * 64 * K : head), SCAN ? (uint32_t)zoo_op_codes(16 * I + rl, 16 * nt + 4 * kg, K) : wat,
              zoo_pack_codes(zoo_q8(w0, inv_sw, qmax), zoo_q8(w1, inv_sw, qmax), zoo_q8(w2, inv_sw, qmax), zoo_q8(w3, inv_sw, qmax)));
    }
  }
  if constexpr (SCALAR) t_pieces(bs_s, t, un);  // (no decay: W and U share T . diag(bs))
  for (int vb = 0; vb < V; vb += 128) {  // passes of up to 128 value columns
    if (vb > 0 && vact && vc8 < min(V - vb, 128) / 8) {
#pragma unroll
      for (int u = 0; u < 2; ++u) vraw[u] = *(const lq_v4i*)(vrow + u * vstep + vb);
    }
    __syncthreads();  // the tile has been read
    if (vact && vc8 < min(V - vb, 128) / 8) stage(vraw, vc8, vrp);
    __syncthreads();
    const int ntiles = min(V - vb, 128) / 32;  // column tiles per half
    for (int q = 0; q < ntiles; ++q) {
      const int nt = half * ntiles + q;
      const lq_v4f a = tile(nt);
      lq_v2i o;
      o[0] = (int)zoo_enc2(a[0] * un, a[1] * un, bf);
      o[1] = (int)zoo_enc2(a[2] * un, a[3] * un, bf);
      if constexpr (SCAN)
        zoo_put(p.U + cb * 64 * V + zoo_op_U(0, vb), 2 * zoo_op_U(16 * I + rl, 16 * nt + 4 * kg), o);
      else
        *(lq_v2i*)(p.U + ((t0 + 16 * I + rl) * H + h) * V + vb + 16 * nt + 4 * kg) = o;
    }
  }
}

template <bool SCALAR, int K, bool BF>
void launch_mode(const ZooWyParams& p, bool scan, dim3 grid, hipStream_t stream) {
  if (scan)
    hipLaunchKernelGGL((zoo_wy_ns_kernel<SCALAR, K, BF, MODE_SCAN>), grid, dim3(512), 0, stream, p);
  else if (p.kqT)
    hipLaunchKernelGGL((zoo_wy_ns_kernel<SCALAR, K, BF, MODE_CODES>), grid, dim3(512), 0, stream, p);
  else
    hipLaunchKernelGGL((zoo_wy_ns_kernel<SCALAR, K, BF, MODE_PLAIN>), grid, dim3(512), 0, stream, p);
}

template <bool SCALAR, int K>
void launch_bf(const ZooWyParams& p, bool scan, dim3 grid, hipStream_t stream) {
  if (p.bf) launch_mode<SCALAR, K, true>(p, scan, grid, stream); else launch_mode<SCALAR, K, false>(p, scan, grid, stream);
}

}  // namespace

int zoo_wy_ns_launch(const ZooWyParams& p, bool scalar, int K, bool scan, hipStream_t stream) {
  const dim3 grid = zoo_unit_grid(p.B, p.NT, p.H);
  if (scalar) {
    if (K == 128) launch_bf<true, 128>(p, scan, grid, stream); else launch_bf<true, 64>(p, scan, grid, stream);
  } else {
    if (K == 128) launch_bf<false, 128>(p, scan, grid, stream); else launch_bf<false, 64>(p, scan, grid, stream);
  }
  return lq_check_launch();
}
