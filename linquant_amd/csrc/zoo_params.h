// Kernel parameter blocks of the zoo state / output kernels, shared by the rotated-storage kernels and the
// canonical-storage (in-kernel un-rotation) variants.
#pragma once

#include "zoo_common.h"
#include "../../include/linquant_hip.h"

struct ZooStateParams {
  const int8_t* kqT;
  const int8_t* vqT;
  const int8_t* wq;
  const _Float16* u;
  const float* fw;
  const float* ev;
  const float* gam;
  const float* pack;  // fw | ev | gam per (batch, chunk, head), 64 + 64 + K floats, or nullptr
  int8_t* h_i8;
  _Float16* e_out;
  float* ht;
  const float* skw;
  const float* svw;
  const float* sw;
  const float* ss;
  const _Float16* unrot;
  int qmax;
  int bf;  // activations are bf16
  int T, H, V, NT;
  int S;  // 64-token pieces per chunk (1; 2..4 in the kernels' PAIR mode)
};

struct ZooOutParams {
  const _Float16* q;
  const _Float16* k;
  const _Float16* v;
  const int8_t* h_i8;
  const float* g;
  const _Float16* A;
  const int8_t* qg;
  const int8_t* qc;  // ready-made local codes of q, k (B,T,H,K) and v (B,T,H,V): q, k, v are then not read
  const int8_t* kc;
  const int8_t* vc;
  void* o;
  int o_is_f32;
  const float* sq;
  const float* sk;
  const float* svl;
  const float* ss;
  const _Float16* unrot;
  float scale;
  int qmax;
  int bf;  // activations (and a 16-bit output) are bf16
  int B, T, H, V, NT;
  const _Float16* Ax;  // 128-token chunks under per-channel decay: (B,T,H,64) fp16 from the cross launch of the A kernel
  float* cross;  // chunks of S > 1 pieces: fp32 (B,T,H,V) partial local products of the later pieces, else nullptr
  int S;         // 64-token pieces per chunk (and per stored state): 1, or 2..4
  int cross_j;   // cross launch j = 1 .. S-1: piece s >= j of a chunk takes its product with the tokens of piece j - 1
};

// 128-token chunks under per-channel decay: the second halves' blocks of the intra-chunk product with the first halves' tokens
struct ZooACrossParams {
  const _Float16* q;
  const _Float16* k;
  const float* g;
  _Float16* Ax;  // (B,T,H,64) fp16, rows of the second halves
  const float* sq;
  const float* sk;
  const _Float16* rot;
  const float* dq;
  float scale;
  int qmax;
  int bf;
  int B, T, H;
};
int zoo_gla_A_cross_launch(const ZooACrossParams& p, int K, hipStream_t stream);  // defined in zoo_gla_A_cross.hip

// canonical storage: one workgroup spans all V value channels (V = 64 or 128); defined in zoo_unrot.hip
int zoo_state_unrot_launch(const ZooStateParams& p, bool delta, int K, int batch, bool pair, hipStream_t stream);
int zoo_output_unrot_launch(const ZooOutParams& p, int decay, int K, hipStream_t stream);

// ---- Grid of the per-channel decay pre-pass: one workgroup per (batch, chunk) and head.  Workgroups are dealt to the 8 XCDs round-robin in launch
// order (x first): x = XCD + 8 head, y counts (batch, chunk)s by eights.  The workgroups resident on one XCD at a time then cover all heads
// of a few (batch, chunk)s, so rows and (B, T, H) tensors (a head's values 4 H bytes apart) are fetched and written as whole lines, and
// the eight XCDs work on neighbouring chunks.  Two dimensions and not one: no division stands
// in front of a workgroup's first request (GLA B4 T4096 H16 141 -> 136.5 us; KDA even; the no / scalar decay pre-passes were 1 % slower).
static inline dim3 zoo_unit_grid(int64_t groups, int H) {
  const int64_t n = groups % 8 ? groups : groups / 8, y = n < 32768 ? n : 32768;
  return dim3((uint32_t)(groups % 8 ? H : 8 * H), (uint32_t)y, (uint32_t)((n + y - 1) / y));
}
// false: beyond the last (batch, chunk) (uniform over the workgroup)
LQ_DEV bool zoo_unit(uint32_t groups, int& h, uint32_t& group) {
  const uint32_t y = blockIdx.y + gridDim.y * blockIdx.z;
  const bool by8 = (groups & 7u) == 0;
  h = (int)(by8 ? blockIdx.x >> 3 : blockIdx.x);
  group = by8 ? (blockIdx.x & 7u) + 8u * y : y;
  return group < groups;
}

// ---- Operand order: the layouts in which the pre-pass kernels leave the operands of zoo_scan.hip.  Tiles of one (batch, chunk,
// head) are contiguous, and inside a tile the 16 bytes that lane l of a wave wants as its MFMA operand (row l & 15, contraction
// group l >> 4) lie at 16 l: a wave's request is 1 KB of whole cache lines.  From token-major rows (16 rows of 64 bytes, H * K
// bytes apart) the same requests kept the vector memory pipeline of a compute unit busy for 1055 of a step's 2790 cycles, in this
// order for 640 of 2100 (linear family, K = V = 128).
// INT8 codes of 64 tokens x K channels: element (token, ch)
LQ_DEV int zoo_op_codes(int token, int ch, int K) {
  return ((token >> 4) * (K >> 6) + (ch >> 6)) * 1024 + ((ch >> 4) & 3) * 256 + (token & 15) * 16 + (ch & 15);
}
// fp16 A of 64 x 64: element (row, col), in halves
LQ_DEV int zoo_op_A(int row, int col) {
  return ((row >> 4) * 2 + (col >> 5)) * 512 + ((col >> 3) & 3) * 128 + (row & 15) * 8 + (col & 7);
}
// INT8 local value codes of V channels x 64 tokens: element (channel, token)
LQ_DEV int zoo_op_values(int ch, int token) {
  return (ch >> 5) * 2048 + (ch & 1) * 1024 + ((token >> 3) & 3) * 256 + ((ch >> 1) & 15) * 16 + (token >> 5) * 8 + (token & 7);
}
// 16-bit U of 64 tokens x V channels, in elements: element (token, channel)
LQ_DEV int zoo_op_U(int token, int ch) { return (ch >> 5) * 2048 + token * 32 + (ch & 31); }

// recurrence and output in one launch (rotated storage, 64-token chunks); defined in zoo_scan.hip
struct ZooScanParams {
  const int8_t* kqT;    // key write codes (B,NT,H,K,64)
  const int8_t* vqT;    // linear: value write codes (B,NT,H,V,64)
  const int8_t* vcT;    // linear: local value codes (B,NT,H, zoo_op_values)
  const int8_t* wq;     // delta: state-read codes of W (B,NT,H, zoo_op_codes)
  const _Float16* u;    // delta: (B,NT,H, zoo_op_U)
  const float* pack;    // delta: fw[64] | ev[64] | gam[K] per (batch, chunk, head)
  const float* gam;     // linear: (B,NT,H,K)
  const int8_t* qc;     // codes of q that read the state (B,NT,H, zoo_op_codes)
  const _Float16* A;    // intra-chunk product (B,NT,H, zoo_op_A), zeros above the diagonal
  const float* gpk;     // scalar decay: cumulative log decay (B,NT,H,64)
  void* o;
  int o_is_f32;
  float* ht;
  const float* skw;
  const float* svw;
  const float* sw;
  const float* ss;
  const float* sq;
  const float* svl;
  int qmax;
  int bf;
  int B, T, H, V, NT;
};
int zoo_scan_launch(const ZooScanParams& p, bool delta, bool scalar, int K, hipStream_t stream);

// WY prep, no / scalar decay.  scan (with the write codes and `local`): wq and U in operand order, the codes of q and A, no Hw
struct ZooWyLocal {
  const void* q;
  int8_t* qc;   // zoo_op_codes
  void* A;      // zoo_op_A
  float* gpk;   // scalar decay: (B,NT,H,64)
  const float* sq;
  const float* sk;
  float scale;
};
int zoo_wy_prep_launch(const lq_zoo_wy_prep_args* a, bool scan, const ZooWyLocal* local, hipStream_t stream);

struct ZooWyParams {
  const _Float16* k;
  const _Float16* v;
  const float* beta;
  const float* g;
  _Float16* Hw;
  _Float16* W;
  _Float16* U;
  float* fw;
  float sigma, tau;
  int bf;
  int B, T, H, V;
  // write-operand codes of the state kernel, made here when kqT is set (otherwise lq_zoo_write_codes makes them from the
  // stored Hw and W)
  int8_t* kqT;
  int8_t* wq;
  float* ev;
  float* gam;
  const float* logenv;
  const float* skw;
  const float* sw;
  float eta;
  int qmax;
  int NT;
  const float* dk_div;  // (H,K) D_QK applied to k at load (k' = act(k / D)), with its reciprocal; or nullptr
  const float* dk_rcp;
  float* pack;  // fw | ev | gam per (batch, chunk, head), 64 + 64 + K floats, or nullptr
  // ZooWyLocal
  const _Float16* q;
  int8_t* qc;
  _Float16* A;
  float* gpk;
  const float* sq;
  const float* sk;
  float scale;
};
// no / scalar decay; defined in zoo_wy_ns.hip
int zoo_wy_ns_launch(const ZooWyParams& p, bool scalar, int K, bool scan, dim3 grid, hipStream_t stream);

// Per-channel decay, 64-token chunks (zoo_diag_prep.h); defined in zoo_diag_{a,wy,gla,kda}.hip
struct ZooDiagParams {
  const _Float16* q;
  const _Float16* k;      // DIAG_A: Hw
  const _Float16* v;
  const float* g;         // DIAG_GLA, DIAG_KDA: log decay per token; DIAG_A, DIAG_WY: cumulated over the chunk
  const float* beta;
  const float* logenv;    // DIAG_WY with write codes
  const _Float16* rot;    // (K,K) local R_QK, or nullptr
  const float* dq;        // (H,K) D_QK for q, and for k with its reciprocal, or nullptr
  const float* dk_div;
  const float* dk_rcp;
  const float* sq;
  const float* sk;
  const float* skw;
  const float* sw;
  const float* svw;       // DIAG_GLA
  const float* svl;
  // fused forms: operand order (above); stage forms: token-major
  _Float16* A;
  int8_t* qc;
  int8_t* kqT;
  int8_t* wq;
  int8_t* vqT;
  int8_t* vcT;
  _Float16* Hw;           // DIAG_WY
  _Float16* W;            // DIAG_WY, may be nullptr
  _Float16* U;
  float* fw;              // DIAG_WY
  float* ev;              // DIAG_WY with write codes
  float* gam;             // DIAG_WY with write codes, DIAG_GLA
  float* pack;            // fw | ev | gam per (batch, chunk, head); DIAG_WY: may be nullptr
  float sigma, tau, eta, scale;
  int qmax;
  int bf;
  int B, T, H, V, NT;
};
int zoo_diag_a_launch(const ZooDiagParams& p, int K, hipStream_t stream);
int zoo_diag_wy_launch(const ZooDiagParams& p, int K, hipStream_t stream);
int zoo_diag_gla_launch(const ZooDiagParams& p, int K, hipStream_t stream);
int zoo_diag_kda_launch(const ZooDiagParams& p, int K, hipStream_t stream);

// Operand pre-pass of the linear family with no / scalar decay for zoo_scan.hip; defined in zoo_lin_prep.hip
struct ZooLinPrepParams {
  const _Float16* q;
  const _Float16* k;
  const _Float16* v;
  const float* g;         // (B,T,H) log decay per token (not cumulated), or nullptr
  const float* signs_qk;  // (K,), (V,) column signs of R_QK, R_V, or nullptr: no rotation
  const float* signs_v;
  const float* dq;        // (H,K) D_QK and its reciprocal, or nullptr
  const float* dq_rcp;
  int8_t* kqT;            // what zoo_scan.hip reads (ZooScanParams)
  int8_t* vqT;
  int8_t* vcT;
  int8_t* qc;
  _Float16* A;
  float* gam;
  float* gpk;
  const float* sq;
  const float* sk;
  const float* skw;
  const float* svw;
  const float* svl;
  float eta, scale;
  int qmax;
  int B, T, H, V, NT;
};
int zoo_lin_prep_launch(const ZooLinPrepParams& p, int K, bool bf, hipStream_t stream);
