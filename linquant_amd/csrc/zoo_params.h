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

// ---- Grid of the kernels in front of zoo_scan.hip: one workgroup per (batch, chunk) and head.  Workgroups are dealt to the 8 XCDs
// round-robin in launch order (x first): x = XCD + 8 head, y and z count the batches and chunks that an XCD takes.  The workgroups
// resident on one XCD at a time then cover all heads of a few (batch, chunk)s, so rows and (B, T, H) tensors (a head's values 4 H bytes
// apart) are fetched and written as whole lines, and the eight XCDs work on neighbouring chunks.
// The last chunks come first, all sequences side by side: the recurrence starts from the first ones, which have then just been
// written and are still in the 256 MB last-level cache (in the other order it finds none of a larger call there, each line having been
// displaced by those behind it).  B4 T4096 H16 K = V = 128, recurrence: Gated DeltaNet 91 -> 82.5 us, linear attention 71 -> 63, GLA the
// same, DeltaNet 86 -> 77, KDA 79 -> 74; KDA B2 T8192 H32 137 -> 135; calls that fit the cache even.  (The launches that write: up to 3 us
// slower.  With the sequences one after the other, last chunk first, the recurrence gains nothing: 90.6.)
struct ZooUnit {
  int h, b, ct;
};
constexpr uint32_t kZooUnitZ = 32768;
__host__ __device__ inline uint32_t zoo_unit_chunks(uint32_t B, uint32_t NT) {  // of the eight (batch, chunk)s side by side; 0: they do not come in eights
  const uint32_t c = (NT & 7u) == 0 ? 8u : NT & (0u - NT);
  return (B & (8u / c - 1u)) == 0 ? c : 0u;
}
static inline dim3 zoo_unit_grid(int B, int NT, int H) {
  const uint32_t c = zoo_unit_chunks((uint32_t)B, (uint32_t)NT), z = c ? NT / c : NT, fold = (z + kZooUnitZ - 1) / kZooUnitZ;
  return dim3((c ? 8 : 1) * H * fold, c ? B / (8 / c) : B, fold > 1 ? kZooUnitZ : z);
}
// false: beyond the last chunk (uniform over the workgroup)
LQ_DEV bool zoo_unit(int B, int NT, int H, ZooUnit& u) {
  const uint32_t c = zoo_unit_chunks((uint32_t)B, (uint32_t)NT);
  uint32_t hx = blockIdx.x, z = blockIdx.z;
  if (c) hx >>= 3;
  if (hx >= (uint32_t)H) z += kZooUnitZ * (hx / (uint32_t)H), hx %= (uint32_t)H;
  u.h = (int)hx;
  u.b = (int)blockIdx.y, u.ct = (int)z;
  if (c) {
    const uint32_t x = blockIdx.x & 7u, lc = (uint32_t)__builtin_ctz(c);
    u.b = (int)((blockIdx.y << (3 - lc)) + (x >> lc)), u.ct = (int)((z << lc) + (x & (c - 1)));
  }
  u.ct = NT - 1 - u.ct;
  return u.ct >= 0;
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
int zoo_scan_launch(const ZooScanParams& p, bool delta, int decay, int K, hipStream_t stream);  // decay: LQ_DECAY_*

// WY prep, no / scalar decay.  scan (with the write codes and `local`): wq and U in operand order, the codes of q and A, no Hw; its g
// is not cumulated
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
  const float* g;  // scalar decay: cumulated over the chunk; what zoo_scan.hip wants made: log decay per token
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
int zoo_wy_ns_launch(const ZooWyParams& p, bool scalar, int K, bool scan, hipStream_t stream);

// Per-channel decay, 64-token chunks (zoo_diag_prep.h); defined in zoo_diag_{a,wy,gla,kda}.hip
struct ZooDiagParams {
  const _Float16* q;
  const _Float16* k;      // DIAG_A: Hw
  const _Float16* v;
  const float* g;         // DIAG_GLA, DIAG_KDA: log decay per token; DIAG_A, DIAG_WY: cumulated over the chunk
  const float* beta;
  const float* logenv;    // DIAG_WY with write codes
  const _Float16* rot;    // (K,K) local R_QK, or nullptr
  const float* rot_f;     // fused forms: the same in fp32, to be rounded to fp16 (instead of rot), or nullptr
  const _Float16* rot_op; // fused forms: the same as zoo_rot_operand_launch leaves it (before the others), or nullptr
  const float* dq;        // (H,K) D_QK for q, and for k with its reciprocal (nullptr: formed here), or nullptr
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
// R_QK (fp16, or fp32: rounded) in the operand order of the fused forms, K * K halves; defined in zoo_rot_operand.hip
int zoo_rot_operand_launch(const void* rot, bool f32, _Float16* op, int K, hipStream_t stream);

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
