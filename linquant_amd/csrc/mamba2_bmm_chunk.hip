// Mamba-2 SSD stage 4: INT8 C.B^T per (batch, chunk, group), requantized to INT8 on a static scale.
// Replaces linquant/kernels/mamba2/bmm_chunk.py:49-139 (launcher :142-217):
//   acc = C_i8[m,:] . B_i8[k,:]        (key side: B_i8 = clamp(rint(B_fp * (1/sB)), +-127) in-loop)
//   CB_i8[m,k] = clamp(rint(float(acc) * ((sC*sB)/S_cb)), +-127)      full QxQ, no causal mask here.
//
// Both operands are contraction-contiguous (N is the unit-stride axis), so MFMA operands are plain
// 16-byte loads.  One wavefront computes a 64x64 output tile as the transposed product (rows = B tokens,
// cols = C tokens) so that every lane ends up with 4 consecutive k of one m: one 32-bit store each.
#include "mamba2_bmm_chunk.h"

namespace {

template <bool B_IS_FP, int N64>
__global__ __launch_bounds__(64, 2) void bmm_chunk_kernel(BmmParams p) {
  if (p.by_xcd)
    bmm_chunk_tile<B_IS_FP, N64>(p, blockIdx.x & 7u, blockIdx.x >> 3, threadIdx.x);
  else
    bmm_chunk_tile<B_IS_FP, N64>(p, 0, blockIdx.x, threadIdx.x);
}

}  // namespace

extern "C" int lq_bmm_chunk(const lq_bmm_chunk_args* a, hipStream_t stream) {
  BmmParams p;
  if (const int rc = bmm_plan(a, &p)) return rc;
#define LQ_BMM_LAUNCH(FP, NN) hipLaunchKernelGGL((bmm_chunk_kernel<FP, NN>), dim3(p.tiles), dim3(64), 0, stream, p)
  switch (a->dstate / 64) {
    case 1: if (a->b_is_fp) LQ_BMM_LAUNCH(true, 1); else LQ_BMM_LAUNCH(false, 1); break;
    case 2: if (a->b_is_fp) LQ_BMM_LAUNCH(true, 2); else LQ_BMM_LAUNCH(false, 2); break;
    case 3: if (a->b_is_fp) LQ_BMM_LAUNCH(true, 3); else LQ_BMM_LAUNCH(false, 3); break;
    default: if (a->b_is_fp) LQ_BMM_LAUNCH(true, 4); else LQ_BMM_LAUNCH(false, 4); break;
  }
#undef LQ_BMM_LAUNCH
  return lq_check_launch();
}
