// Cumulative sum and C.B^T of the Mamba-2 SSD in one launch: neither reads what the other writes, and both are a few microseconds of
// work behind a launch and a memory round trip.  The first workgroups take the dt tiles (mamba2_cumsum.h, the longer chain), the others
// one to eight C.B^T tiles each (mamba2_bmm_chunk.h), the bits of the two stand-alone launches.
// The scan reads nothing above the diagonal 64 x 64 tiles of C.B^T: those (6 of 16 at 256-token chunks) are not formed here.  With them, and
// with 64-bit lane offsets for dt (mamba2_cumsum.h), kernel us on one card in turn: B4 L8192 H80 20.5 -> 19.6, B3 L5000 H80 13.3 -> 11.9, B8
// L2048 H64 value side 9.7 -> 9.3, B4 L2048 H80 8.7 -> 8.5, B1 L512 H80 even (6.4).
// Bound by latency.  Kernel us before that, two launches -> one: B1 L512 H80 6.4 + 5.9 -> 6.4, B3 L5000 H80 11.0 + 7.5 -> 13.2, B4 L2048 H80
// 7.0 + 6.0 -> 8.3, B8 L2048 H64 value side 7.1 + 6.0 -> 9.8, B4 L8192 H80 12.6 + 10.2 -> 19.6 .. 22.7.
#include "mamba2_bmm_chunk.h"
#include "mamba2_cumsum.h"

namespace {

// cblocks: workgroups of the sum (cpad: rounded up to a multiple of 8, so that both halves keep their place on the XCDs); per: tiles of
// a workgroup, one to a wave
template <int E, bool B_IS_FP, int N64>
__global__ __launch_bounds__(kWaves * 64, 4) void cumsum_bmm_kernel(CumsumParams c, BmmParams b, uint32_t cblocks, uint32_t cpad, uint32_t per) {
  extern __shared__ float tile[];
  if (blockIdx.x < cpad) {
    if (blockIdx.x < cblocks) chunk_cumsum_fixed<E>(c, blockIdx.x, tile);
    return;
  }
  const uint32_t w = blockIdx.x - cpad, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wave >= per) return;
  if (b.by_xcd) {  // (units and with them tiles are a multiple of 8 then)
    const uint32_t j = (w >> 3) * per + wave;
    if (j < b.tiles / 8u) bmm_chunk_tile<B_IS_FP, N64>(b, w & 7u, j, threadIdx.x & 63);
  } else {
    const uint32_t j = w * per + wave;
    if (j < b.tiles) bmm_chunk_tile<B_IS_FP, N64>(b, 0, j, threadIdx.x & 63);
  }
}

template <int E, bool B_IS_FP>
void launch(int N64, dim3 grid, hipStream_t stream, const CumsumParams& c, const BmmParams& b, uint32_t cblocks, uint32_t cpad, uint32_t per) {
  const size_t lds = (size_t)(64 * E) * (kHG + 1) * sizeof(float);
  if (N64 == 1)
    hipLaunchKernelGGL((cumsum_bmm_kernel<E, B_IS_FP, 1>), grid, dim3(kWaves * 64), lds, stream, c, b, cblocks, cpad, per);
  else
    hipLaunchKernelGGL((cumsum_bmm_kernel<E, B_IS_FP, 2>), grid, dim3(kWaves * 64), lds, stream, c, b, cblocks, cpad, per);
}

template <int E>
void launch(bool fp, int N64, dim3 grid, hipStream_t stream, const CumsumParams& c, const BmmParams& b, uint32_t cblocks, uint32_t cpad, uint32_t per) {
  if (fp) launch<E, true>(N64, grid, stream, c, b, cblocks, cpad, per); else launch<E, false>(N64, grid, stream, c, b, cblocks, cpad, per);
}

}  // namespace

// Both stages, in one launch where there is a form for the sizes (chunks of 64 .. 512 tokens, d_state 64 or 128), else one after the other
int lq_cumsum_bmm(const lq_chunk_cumsum_args* cs, const lq_bmm_chunk_args* bm, hipStream_t stream) {
  CumsumParams c;
  BmmParams b;
  uint32_t cblocks;
  int rc;
  if ((rc = cumsum_plan(cs, &c, &cblocks)) != LQ_OK || (rc = bmm_plan(bm, &b, true)) != LQ_OK) return rc;
  const int E = cumsum_fixed_e(cs), N64 = bm->dstate / 64;
  const uint32_t cpad = (cblocks + 7u) / 8u * 8u;
  // as few tiles to a workgroup as keep everything in the 512 places of one round (two workgroups per compute unit): 32 tiles eight to
  // a workgroup took 9.7 us, one to a workgroup 6.4; 960 beside 300 workgroups of the sum took 13.9 us by eights, 15.4 by fours
  // (a second round), and 2048 by eights 19.3 (the two launches 22.8)
  uint32_t per = 1;
  while (per < kWaves && (uint64_t)cpad + (b.tiles + per - 1) / per > 512) ++per;
  const uint64_t grid = (uint64_t)cpad + (b.by_xcd ? 8u * ((b.tiles / 8u + per - 1) / per) : (b.tiles + per - 1) / per);
  if (!E || N64 > 2 || grid >= (1ull << 31)) {
    if ((rc = lq_chunk_cumsum(cs, stream)) != LQ_OK) return rc;
    return lq_bmm_chunk(bm, stream);
  }
  const bool fp = bm->b_is_fp;
  const dim3 g((uint32_t)grid);
  switch (E) {
    case 1: launch<1>(fp, N64, g, stream, c, b, cblocks, cpad, per); break;
    case 2: launch<2>(fp, N64, g, stream, c, b, cblocks, cpad, per); break;
    case 4: launch<4>(fp, N64, g, stream, c, b, cblocks, cpad, per); break;
    default: launch<8>(fp, N64, g, stream, c, b, cblocks, cpad, per); break;
  }
  return lq_check_launch();
}
