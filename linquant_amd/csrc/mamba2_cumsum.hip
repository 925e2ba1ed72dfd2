// Mamba-2 SSD stage 1: dt pipeline + chunk-local cumulative sum of dt*A.
// Replaces the reference stage linquant/kernels/mamba2/chunk_cumsum.py:27-74 (launcher :77-100).
//
// One 8-wave workgroup per (16 heads, chunk, batch): the (token, head) tile of raw dt is staged through LDS with
// head-contiguous reads (dt is laid out (B, L, H): a head's tokens are H elements apart), then each wavefront
// scans two heads.  Lane l owns the E = Q/64 consecutive positions l*E .. l*E+E-1 of the chunk.  The prefix sum is: sequential inside the lane, Hillis-Steele
// inclusive scan of the lane totals over the wave (offsets 1,2,4,...,32, "t = t + up"), then
// exclusive lane prefix + local prefix.  The CPU checker restates exactly this order.
#include "mamba2_cumsum.h"

namespace {

__global__ __launch_bounds__(kWaves * 64) void chunk_cumsum_kernel(
    const void* __restrict__ dt_in, int dt_dtype, int64_t sdt_b, int64_t sdt_l, int64_t sdt_h,
    const float* __restrict__ dt_scale_p, const int8_t* __restrict__ a_log, int64_t sa_h,
    const float* __restrict__ a_log_scale_p, const float* __restrict__ dt_bias, int64_t sbias_h,
    float* __restrict__ dt_out, float* __restrict__ dA_cs, int seqlen, int nheads, int nchunks, int Q,
    int softplus, float dt_min, float dt_max, int hg, int by_xcd) {
  extern __shared__ float tile[];  // [Q][kHG + 1] raw dt as float
  const Where wh = where(blockIdx.x, hg, nchunks, by_xcd);
  const int h0 = wh.h0, c = wh.c, b = wh.b;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int E = Q >> 6;
  const int limit = min(Q, seqlen - c * Q);
  // ---- stage the (token, head) tile: consecutive lanes read consecutive heads of one token
  for (int it = tid; it < Q * kHG; it += kWaves * 64) {
    const int pos = it / kHG, hh = it % kHG;
    float v = 0.0f;
    if (pos < limit && h0 + hh < nheads)
      v = load_dt(dt_in, (int64_t)b * sdt_b + (int64_t)(c * Q + pos) * sdt_l + (int64_t)(h0 + hh) * sdt_h, dt_dtype);
    tile[pos * (kHG + 1) + hh] = v;
  }
  __syncthreads();
  const float dt_scale = *dt_scale_p;
  const float a_scale = *a_log_scale_p;
#pragma unroll
  for (int hw = 0; hw < kHG / kWaves; ++hw) {
    const int hh = wave * (kHG / kWaves) + hw;
    const int h = h0 + hh;
    if (h >= nheads) continue;
    const float A = -lq_expf(a_scale * (float)a_log[(int64_t)h * sa_h]);
    const float bias = dt_bias ? dt_bias[(int64_t)h * sbias_h] : 0.0f;
    float dtv[kMaxE], pre[kMaxE];
    float run = 0.0f;
#pragma unroll
    for (int i = 0; i < kMaxE; ++i) {
      if (i < E) {
        const int pos = lane * E + i;
        float v = 0.0f;
        if (pos < limit) {
          v = dt_scale * tile[pos * (kHG + 1) + hh];
          if (dt_bias) v = v + bias;
          if (softplus) v = (v > 20.0f) ? v : lq_logf(1.0f + lq_expf(v));
          v = fminf(fmaxf(v, dt_min), dt_max);
        }
        dtv[i] = v;
        const float dA = v * A;
        run = (i == 0) ? dA : run + dA;
        pre[i] = run;
      }
    }
    float t = run;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float up = __shfl_up(t, off, 64);
      if (lane >= off) t = t + up;
    }
    float ex = __shfl_up(t, 1, 64);
    if (lane == 0) ex = 0.0f;
    const int64_t base = (((int64_t)b * nheads + h) * nchunks + c) * Q + lane * E;
#pragma unroll
    for (int i = 0; i < kMaxE; ++i) {
      if (i < E) {
        dt_out[base + i] = dtv[i];
        dA_cs[base + i] = ex + pre[i];
      }
    }
  }
}

template <int E>
__global__ __launch_bounds__(kWaves * 64) void chunk_cumsum_fixed_kernel(CumsumParams p) {
  extern __shared__ float tile[];
  chunk_cumsum_fixed<E>(p, blockIdx.x, tile);
}

}  // namespace

extern "C" int lq_chunk_cumsum(const lq_chunk_cumsum_args* a, hipStream_t stream) {
  CumsumParams p;
  uint32_t blocks;
  if (const int rc = cumsum_plan(a, &p, &blocks)) return rc;
  const int Q = a->chunk_size;
  const dim3 grid(blocks);
  const size_t lds = (size_t)Q * (kHG + 1) * sizeof(float);
  if (lds > 65536 && hipFuncSetAttribute(reinterpret_cast<const void*>(&chunk_cumsum_kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return LQ_ERR_LAUNCH;
  switch (cumsum_fixed_e(a)) {
    case 1: hipLaunchKernelGGL(chunk_cumsum_fixed_kernel<1>, grid, dim3(kWaves * 64), lds, stream, p); break;
    case 2: hipLaunchKernelGGL(chunk_cumsum_fixed_kernel<2>, grid, dim3(kWaves * 64), lds, stream, p); break;
    case 4: hipLaunchKernelGGL(chunk_cumsum_fixed_kernel<4>, grid, dim3(kWaves * 64), lds, stream, p); break;
    case 8: hipLaunchKernelGGL(chunk_cumsum_fixed_kernel<8>, grid, dim3(kWaves * 64), lds, stream, p); break;
    default:
      hipLaunchKernelGGL(chunk_cumsum_kernel, grid, dim3(kWaves * 64), lds, stream, a->dt, a->dt_dtype, a->dt_stride_b,
                         a->dt_stride_l, a->dt_stride_h, a->dt_scale, a->A_log, a->A_log_stride_h, a->A_log_scale, a->dt_bias,
                         a->dt_bias_stride_h, a->dt_out, a->dA_cumsum, a->seqlen, a->nheads, p.nchunks, Q, a->dt_softplus, a->dt_min,
                         a->dt_max, p.hg, p.by_xcd);
  }
  return lq_check_launch();
}
