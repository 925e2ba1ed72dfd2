// The local R_QK in the order in which zoo_diag_prep.h wants it: 16 bytes of operand (strip, tile t, step ks) for lane (rl, kg) are
// R[32ks + 8kg + 0 .. 7][32 strip + 2rl + t], the operands one after the other.  A launch of 32 KB in front of the one that reads them.
#include "zoo_params.h"

namespace {

template <typename T>
__global__ __launch_bounds__(256) void rot_operand_kernel(const T* rot, _Float16* op, int K) {
  const int i = blockIdx.x * 256 + threadIdx.x, lane = i & 63, KS = K / 32;  // (K * K / 8 threads)
  const int ks = (i >> 6) % KS, st = (i >> 6) / KS;
  const T* src = rot + (32 * ks + 8 * (lane >> 4)) * K + 32 * (st >> 1) + 2 * (lane & 15) + (st & 1);
  lq_v8h o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = (_Float16)src[e * K];
  *(lq_v8h*)(op + 8 * i) = o;
}

}  // namespace

int zoo_rot_operand_launch(const void* rot, bool f32, _Float16* op, int K, hipStream_t stream) {
  const dim3 grid(K * K / 2048);
  if (f32)
    hipLaunchKernelGGL(rot_operand_kernel<float>, grid, dim3(256), 0, stream, (const float*)rot, op, K);
  else
    hipLaunchKernelGGL(rot_operand_kernel<_Float16>, grid, dim3(256), 0, stream, (const _Float16*)rot, op, K);
  return lq_check_launch();
}
