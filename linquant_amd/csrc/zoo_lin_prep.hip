// Operand pre-pass of the linear family with no or scalar decay (linear attention, the Mamba-2 cell), 64-token chunks: everything
// that zoo_scan.hip wants of a chunk, from the rows as the model produced them, in one launch.
// Replaces the chunk-local cumsum (linquant/kernels/zoo/simple_gla.py:191), the operand preparation inside _state_body
// (simple_gla.py:55-66), the operand quantization and the intra-chunk product of _output_body (simple_gla.py:125-140) and, where the
// caller asks for them, the operand rotations and the D_QK rescaling (bench/zoo_kernels.py:135-140, linquant/harness.py:68-88), with
// the arithmetic of lq_zoo_cumsum, lq_zoo_rotate_quant and lq_zoo_output in their order: the same bits.
//
// One 8-wave workgroup per (chunk, batch*head), three to a compute unit (80 registers, 49 KB of LDS): load (a thread takes four adjacent
// tokens x 8 channels; every row is read once) while one wave forms the cumulative decay | rotate and quantize q and k into LDS, then v,
// requested when their rows have left the registers | operands out as whole 1 KB tiles and 64-byte rows, blocks of A on the INT8 MFMA.
// What holds the registers at 80: one token after the other, with the tables of its channels (scales, signs) read from LDS anew for each,
// and one copy of the pass over value columns, with nothing that follows from the thread's number kept across it.  Linear attention with
// the rotations, B4 T4096 H16 K = V = 128: 95.3 -> 84 to 87 us for 201 MB read and 168 MB written (4.3 TB/s; two workgroups to a compute
// unit at 127 registers before), vector instructions 70 us of it; whole call 146.6 -> 136 to 138.
// B4 T4096 H16 K 64, V 128: whole call 106.2 -> 93.2 (100.6 with two workgroups and v requested first), Mamba-2 cell K = V = 64 of the same
// size even.
#include <type_traits>

#include "zoo_params.h"

namespace {

// dword of the transposed code tile [channel][16 token quads]; four dwords of pad after every eight channels, so that the writes of
// a wave (16 groups of eight channels, four quads) fall on 64 different banks and rows stay 16-byte aligned
LQ_DEV int lp_ct(int ch, int quad) { return ch * 16 + (ch >> 3) * 4 + quad; }
constexpr int lp_ct_size(int channels) { return channels * 16 + channels / 8 * 4; }

// w with byte T replaced by the code's (the bytes above it undefined until their turn)
template <int T>
LQ_DEV uint32_t lp_put(uint32_t w, int code) {
  if constexpr (T == 0) return (uint32_t)code;
  return __builtin_amdgcn_perm((uint32_t)code, w, T == 1 ? 0x0c0c0400u : (T == 2 ? 0x0c040100u : 0x04020100u));
}

template <typename F>
LQ_DEV void lp_quad(const F& f) {
  f(std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 1>{});
  f(std::integral_constant<int, 2>{});
  f(std::integral_constant<int, 3>{});
}

// clamp(rha(x * inv), -qmax, qmax) with the clamp as one median instruction (same value as zoo_q8)
LQ_DEV int lp_q8(float x, float inv, int qmax) {
  int r;
  asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(lq_rha_i32(x * inv)), "v"(-qmax), "v"(qmax));
  return r;
}

// tokens one after the other, the tables of the eight channels read anew for each
LQ_DEV void token_end() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// rotation of a row of 128 (wide: uniform over the workgroup) or 64 channels, as lq_zoo_rotate_qkv forms it before it rounds
LQ_DEV void lp_rotate(float (&x)[8], int sub, const float* signs, bool wide) {
  const float norm = wide ? 0.08838834764831845f : 0.125f;  // 1 / sqrt(128), 1 / sqrt(64)
  zoo_fwht<8>(x, sub);
  if (wide) zoo_fwht_stage<8>(x, sub);
  const lq_v4f s0 = *(const lq_v4f*)(signs + 8 * sub), s1 = *(const lq_v4f*)(signs + 8 * sub + 4);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (x[e] * norm) * (e < 4 ? s0[e & 3] : s1[e & 3]);
}

// rounded to the activation dtype and back
template <bool BF>
LQ_DEV void lp_round(float (&x)[8]) {
#pragma unroll
  for (int d = 0; d < 4; ++d) zoo_dec2(zoo_enc2(x[2 * d], x[2 * d + 1], BF), BF, x[2 * d], x[2 * d + 1]);
}

template <bool BF>
LQ_DEV void lp_dec(lq_v4i raw, float (&x)[8]) {
#pragma unroll
  for (int d = 0; d < 4; ++d) zoo_dec2((uint32_t)raw[d], BF, x[2 * d], x[2 * d + 1]);
}

LQ_DEV lq_v2i lp_pack8(const int (&c)[8]) {
  return lq_v2i{(int)zoo_pack_codes(c[0], c[1], c[2], c[3]), (int)zoo_pack_codes(c[4], c[5], c[6], c[7])};
}

template <bool SCALAR, int K, bool BF>
__global__ __launch_bounds__(512, 6) void zoo_lin_prep_kernel(ZooLinPrepParams p) {
  constexpr int QS = K == 128 ? 160 : 80;  // bytes per row of the code tiles
  __shared__ __align__(16) unsigned char qI[64 * QS], kI[64 * QS];
  __shared__ __align__(16) uint32_t cK[lp_ct_size(K)], cW[lp_ct_size(128)], cL[lp_ct_size(128)];
  __shared__ float fk_s[64], fv_s[64], gs_s[64], iskw_s[K], isvw_s[128], isvl_s[128];
  __shared__ __align__(16) float sqk_s[K], sv_s[128];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rl = lane & 15, kg = lane >> 4;
  ZooUnit unit;
  if (!zoo_unit(p.B, p.NT, p.H, unit)) return;
  const int h = unit.h, b = unit.b, ct = unit.ct;
  const int H = p.H, V = p.V, qmax = p.qmax;
  const int64_t t0 = (int64_t)b * p.T + (int64_t)ct * 64;
  const int64_t cb = ((int64_t)b * p.NT + ct) * H + h;

  // ---- requests: a thread takes a token quad x 8 channels of q or k (the first or second half of the first K / 16 waves)
  constexpr int KP = K / 8;
  const bool is_k = wave >= K / 32;
  const int kt = tid & (16 * KP - 1), kq = kt / KP, kc = kt % KP;
  const bool kact = wave < K / 16;
  lq_v4i kraw[4];
  const _Float16* src = is_k ? p.k : p.q;
#pragma unroll
  for (int u = 0; u < 4; ++u) kraw[u] = zoo_at<lq_v4i>(src + (t0 * H + h) * K, 2 * (zoo_rows(4 * kq + u, H, K) + 8 * kc));
  // ---- per-token factors
  if (wave == 0) {
    float fk = 1.0f, fv = 1.0f;
    if constexpr (SCALAR) {
      const float gc = zoo_cumsum64(zoo_at<float>(p.g + t0 * H + h, 4 * zoo_rows(lane, H, 1)));
      const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gc), 63)) - gc;
      fk = zoo_exp((1.0f - p.eta) * d), fv = zoo_exp(p.eta * d);
      gs_s[lane] = gc;
      p.gpk[cb * 64 + lane] = gc;
    }
    fk_s[lane] = fk, fv_s[lane] = fv;
  } else if (wave == 1 || wave == 2) {
    const int n = tid - 64;
    if (n < K) {
      iskw_s[n] = 1.0f / p.skw[(int64_t)h * K + n];
      if (p.signs_qk) sqk_s[n] = p.signs_qk[n];
    }
  } else if (wave == 3 || wave == 4) {
    const int n = tid - 192;
    if (n < V) {
      isvw_s[n] = 1.0f / p.svw[(int64_t)h * V + n];
      if (p.signs_v) sv_s[n] = p.signs_v[n];
    }
  } else if (wave == 5 || wave == 6) {
    const int n = tid - 320;
    if (n < V) isvl_s[n] = 1.0f / p.svl[(int64_t)h * V + n];
  }
  __syncthreads();
  for (int n = tid; n < K; n += 512) p.gam[cb * K + n] = SCALAR ? zoo_exp(gs_s[63]) : 1.0f;

  // ---- queries and keys: local codes by token; keys: write codes by channel
  if (kact) {
    const float inv = 1.0f / (is_k ? p.sk : p.sq)[h];
    unsigned char* codes = is_k ? kI : qI;
    uint32_t wc[8];
    lp_quad([&](auto u_c) __attribute__((always_inline)) {
      constexpr int u = decltype(u_c)::value;
      const int t = 4 * kq + u;
      float x[8];
      lp_dec<BF>(kraw[u], x);
      if (p.dq) {  // (uniform over the launch)
        const int64_t n = (int64_t)h * K + 8 * kc;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = is_k ? zoo_div_rn(x[e], p.dq[n + e], p.dq_rcp[n + e]) : zoo_mul_rn(x[e], p.dq[n + e]);
      }
      if (p.signs_qk) lp_rotate(x, kc, sqk_s, K == 128);
      if (p.dq || p.signs_qk) lp_round<BF>(x);
      int c[8];
      if (is_k) {  // (wave-uniform)
        const float f = fk_s[t];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          c[e] = lp_q8(x[e], inv, qmax);
          wc[e] = lp_put<u>(wc[e], lp_q8(SCALAR ? x[e] * f : x[e], iskw_s[8 * kc + e], qmax));
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e] = lp_q8(x[e] * p.scale, inv, qmax);
      }
      *(lq_v2i*)(codes + t * QS + 8 * kc) = lp_pack8(c);
      token_end();
    });
    if (is_k) {
#pragma unroll
      for (int e = 0; e < 8; ++e) cK[lp_ct(8 * kc + e, kq)] = wc[e];
    }
  }
  // ---- values, up to 128 columns a pass: write and local codes by channel.  A thread takes a token quad x 8 channels, from wave 0 on
  // beside 128 keys, from wave 4 on beside 64.
#pragma unroll 1
  for (int vb = 0; vb < V; vb += 128) {
    int own = tid;
    asm volatile("" : "+v"(own));  // (nothing that follows from it is to wait in registers from in front of the loop on)
    const int tid = own, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), rl = lane & 15, kg = lane >> 4;
    const int vt = K == 128 ? tid : max(tid - 256, 0);
    const int vsh = V - vb >= 128 ? 4 : 3, vp = 1 << vsh;  // 16-byte pieces of a value row (V is a multiple of 64)
    const bool vact = (K == 128 || wave >= 4) && vt < 16 * vp;  // (wave-uniform)
    const int vq = (vt >> vsh) & 15, vc = vt & (vp - 1);
    __builtin_amdgcn_sched_barrier(0);  // (requested behind the codes of q and k, whose rows leave their registers)
    lq_v4i vraw[4];
    const int64_t vstep = (int64_t)H * V;  // (uniform)
    const _Float16* const vrow = p.v + (t0 * vstep + (int64_t)h * V + vb) + 4 * vq * vstep + 8 * vc;
#pragma unroll
    for (int u = 0; u < 4; ++u) vraw[u] = *(const lq_v4i*)(vrow + u * vstep);
    if (vb > 0) {
      __syncthreads();  // the tiles have been read
      if (tid < 8 * vp) {
        isvw_s[tid] = 1.0f / p.svw[(int64_t)h * V + vb + tid];
        isvl_s[tid] = 1.0f / p.svl[(int64_t)h * V + vb + tid];
      }
      __syncthreads();
    }
    if (vact) {
      uint32_t ww[8], wl[8];
      lp_quad([&](auto u_c) __attribute__((always_inline)) {
        constexpr int u = decltype(u_c)::value;
        float x[8];
        lp_dec<BF>(vraw[u], x);
        if (p.signs_v) {  // (V is 64 or 128: one pass)
          lp_rotate(x, vc, sv_s, vp == 16);
          lp_round<BF>(x);
        }
        const float f = fv_s[4 * vq + u];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          wl[e] = lp_put<u>(wl[e], lp_q8(x[e], isvl_s[8 * vc + e], qmax));
          ww[e] = lp_put<u>(ww[e], lp_q8(SCALAR ? x[e] * f : x[e], isvw_s[8 * vc + e], qmax));
        }
        token_end();
      });
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int at = lp_ct(8 * vc + e, vq);
        cW[at] = ww[e], cL[at] = wl[e];
      }
    }
    __syncthreads();
    if (tid < 32 * vp) {  // four 16-byte pieces per channel (wave-uniform)
      zoo_put(p.vqT + (cb * V + vb) * 64, 16 * tid, *(const lq_v4i*)(cW + lp_ct(tid >> 2, 4 * (tid & 3))));
      // operand order: wave w has the even or odd channels of tile w >> 1, tokens 8 kg .. and 32 + 8 kg ..
      const uint32_t* row = cL + lp_ct(32 * (wave >> 1) + 2 * rl + (wave & 1), 2 * kg);
      const lq_v2i lo = *(const lq_v2i*)row, hi = *(const lq_v2i*)(row + 8);
      zoo_put(p.vcT + cb * 64 * V + 64 * vb, 16 * tid, lq_v4i{lo[0], lo[1], hi[0], hi[1]});
    }
  }

  // ---- operands out
  if (tid < 4 * K) {
    zoo_put(p.kqT + cb * K * 64, 16 * tid, *(const lq_v4i*)(cK + lp_ct(tid >> 2, 4 * (tid & 3))));
    const int tb = wave / (K / 64), ks = wave % (K / 64);  // 16 tokens x 64 channels
    zoo_put(p.qc + cb * 64 * K, 16 * tid, *(const lq_v4i*)(qI + (16 * tb + rl) * QS + 64 * ks + 16 * kg));
  }
  // ---- blocks of A: (0,0) (1,0) (1,1) (2,0) .. (3,3) of the lower triangle, then zeros above it
  const float sqk = p.sq[h] * p.sk[h];
  for (int n = wave; n < 16; n += 8) {
    int I, J;
    if (n < 10) {
      I = n < 1 ? 0 : (n < 3 ? 1 : (n < 6 ? 2 : 3)), J = n - I * (I + 1) / 2;
    } else {
      const int m = n - 10;  // (0,1) (0,2) (0,3) (1,2) (1,3) (2,3)
      I = m < 3 ? 0 : (m < 5 ? 1 : 2), J = m < 3 ? m + 1 : (m < 5 ? m - 1 : 3);
    }
    lq_v2i out = {0, 0};
    const int i = 16 * I + rl, j0 = 16 * J + 4 * kg;
    if (n < 10) {
      lq_v4i acc = {0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < K / 64; ++ks)  // transposed: lane (rl, kg) holds row 16I + rl, columns 16J + 4kg + r
        acc = lq_mfma_i8(*(const lq_v4i*)(kI + (16 * J + rl) * QS + 64 * ks + 16 * kg), *(const lq_v4i*)(qI + (16 * I + rl) * QS + 64 * ks + 16 * kg), acc);
      float x[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[r] = (float)acc[r] * sqk;
        if (SCALAR) x[r] = x[r] * zoo_exp(gs_s[i] - gs_s[j0 + r]);
        x[r] = j0 + r <= i ? x[r] : 0.0f;
      }
      out = lq_v2i{(int)zoo_pack_h2(x[0], x[1]), (int)zoo_pack_h2(x[2], x[3])};
    }
    zoo_put(p.A + cb * 4096, 2 * zoo_op_A(i, j0), out);
  }
}

template <bool SCALAR, int K>
void launch(const ZooLinPrepParams& p, bool bf, dim3 grid, hipStream_t stream) {
  if (bf)
    hipLaunchKernelGGL((zoo_lin_prep_kernel<SCALAR, K, true>), grid, dim3(512), 0, stream, p);
  else
    hipLaunchKernelGGL((zoo_lin_prep_kernel<SCALAR, K, false>), grid, dim3(512), 0, stream, p);
}

}  // namespace

int zoo_lin_prep_launch(const ZooLinPrepParams& p, int K, bool bf, hipStream_t stream) {
  const dim3 grid = zoo_unit_grid(p.B, p.NT, p.H);
  if (p.g) {
    if (K == 128) launch<true, 128>(p, bf, grid, stream); else launch<true, 64>(p, bf, grid, stream);
  } else {
    if (K == 128) launch<false, 128>(p, bf, grid, stream); else launch<false, 64>(p, bf, grid, stream);
  }
  return lq_check_launch();
}
