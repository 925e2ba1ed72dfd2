// The chunk recurrence and the output of a zoo cell in one launch (rotated storage, 64-token chunks): what zoo_state.hip and
// zoo_output.hip do one after the other, without the stored states and the pseudo-values E ever reaching memory.
// Covers the state bodies linquant/kernels/zoo/simple_gla.py:23-75, gla.py:102-148, gated_delta_rule.py:50-115, kda.py:68-130
// and the output bodies simple_gla.py:98-153, gla.py:170-213, with the arithmetic of the two kernels named above in their
// order, so the outputs are theirs bit for bit.
//
// What bounds it: the chain of chunk steps (64 at T = 4096).  One 8-wave workgroup per (BV-column V tile, batch*head); per
// step
//   waves 0..3 (chain) quantize the fp32 carry they hold in registers (wave w owns K/4 rows) into LDS, read the state for
//     the delta family, form E and its write codes, and apply the INT8 write product to the carry;
//   waves 4..7 (output; wave 4 + w owns token rows 16w .. 16w + 15) read the same stored copy from LDS with the codes of q,
//     and add the intra-chunk product of A with the local codes of v (linear family) or E (delta family).
// Every SIMD holds one wave of each kind, so the output's instructions fill the issue slots that the chain leaves while it
// waits for its rendezvous.  The output's operands do not depend on the carry; it has no rendezvous of its own: the chain's
// (one per step for the linear family, two for the delta family) hand it the stored copy and E.  The delta family's output
// runs half a step behind: E of a chunk becomes local codes between the chain's second and the next first rendezvous, and the
// chunk's local product and store follow after that one.
//
// Measured (kernel time; before = zoo_state + zoo_output): GLA B4 T4096 H16 K = V = 128 47 + 66 -> 67 us (63 since the launch in front
// of it takes the last chunks first: zoo_params.h), KDA B2 T8192 H32 157 + 128 -> 135 us, KDA B1 T2048 H8 41 + 7 -> 36 us (24 with 16 columns).  A step (1.0 us at KDA) is now the chain's own: about 900 cycles to quantize the
// carry, 300 to issue its requests, 1000 for state read and E, 300 for the update; one workgroup of 32 columns per compute unit
// at the first two shapes.
//
// Nothing inside an output step branches (A holds zeros above the diagonal and both 32-token slabs are always multiplied, the
// output type is a template parameter, the first step is peeled off): memory operations retire in issue order and the compiler
// derives each wait from a count of those issued since, merged over all paths, so a branch around a store or a product made
// every step wait for the operands it had just requested (seen in its assembly: vmcnt(2) .. vmcnt(4)
// where vmcnt(27) is meant).
//
// An output wave's products take the local value codes of all 64 tokens as fp16.  Converted by each of the four waves they were 40 of its
// vector instructions a step; an operand to a wave, handed on through LDS at the rendezvous that is there, they are 10: linear attention
// and GLA B4 T4096 H16 K = V = 128, kernel 64.7 -> 62.1 us, whole calls 136.9 -> 133.8 and 196.8 -> 194.8.
//
// Addresses are a scalar base and a lane's 32-bit offset, and an output's place is formed once: kernel 62.1 -> 59.0 us for the linear family
// (its output waves multiplied by H V in the vector unit for each store), 86.2 -> 83.7 for Gated DeltaNet B4 T4096 H16.
//
// The linear family keeps two operand sets and at most 128 registers, so that two workgroups fit a compute unit.  With five sets
// (199 .. 236 registers, one workgroup) 257 to 511 workgroups took two rounds of the chip, the second nearly empty, and lost to the
// two launches that this one replaces; the second workgroup hides more than the three further sets did.  Linear attention K = V = 128,
// us per call with two launches / five sets / two sets: B*H = 80 T1024 54 / 63 / 54, B*H = 192 T1024 112 / 116 / 106, B*H = 96 T2048
// 112 / 118 / 106, B*H = 64 T4096 (one full round) 151 / 145 / 146.  The delta family's sets hold more per step (three sets, 142 ..
// 165 registers at K = 128): its step is longer, and with one workgroup per compute unit it was faster than its two launches at every
// size measured (B*H = 4 .. 256, T = 256 .. 16384: 1.04 to 1.7 times).
#include <algorithm>
#include <type_traits>

#include "zoo_params.h"

namespace {

using ScanParams = ZooScanParams;

// ---- Segments (linear family).  Its carry reads neither the stored copy nor anything else of a step but the write codes and the
// decay, so a workgroup can start in the middle of a chain: it first runs the updates of the chunks in front (one MFMA a tile and five
// vector instructions a value, no rendezvous, three or four operand sets in rotation), with the order and the arithmetic of the whole
// chain and so with its bits, and then its own steps.  An update takes about 0.3 of a step; segments that shrink by that share, first to
// last, end together.  One workgroup per compute unit: as many segments as keep all of them at 256 or fewer (a second workgroup per
// compute unit repeats updates faster than it hides waits: B4 T4096 H16 K = V = 128, 256 tiles, one / two segments 150 / 156 us).
// GPU time of the whole call, one segment or two launches (zoo_combined.hip), whichever was taken before -> segments: linear attention
// with R_QK, K = V = 128, H4 T4096 / T16384 49.3 -> 30.3 / 132 -> 75.5 us, H16 60.3 -> 49.9 / 231 -> 187; K = V = 64 H8 T2048 / T16384
// 24.2 -> 16.6 / 110 -> 67.4; GLA K = V = 128 H4 T16384 162 -> 90, H5 T8192 96.3 -> 59.4.  Decay of the segments' lengths by 0.2 or 0.4
// in the place of 0.3: at most 4 % slower.
// All of this takes the compute units that one call leaves idle for free.  Where other work fills them, the repeated updates cost it: GPU us
// a call, one segment or two launches -> segments, with 1 / 2 / 4 / 8 streams of the same call: Mamba-2 cell H8 T16384 116 -> 65 / 63 -> 63 /
// 45 -> 60 / 45 -> 60, H8 T2048 24 -> 18 / 17 -> 12 / 9.5 -> 7.6 / 9.3 -> 7.4; linear attention H4 T16384 132 -> 71 / 76 -> 66 / 55 -> 63 /
// 67 -> 64, H4 T4096 46 -> 29 / 30 -> 19 / 18 -> 15 / 17 -> 15; GLA H4 T16384 155 -> 91 / 107 -> 79 / 84 -> 76 / 95 -> 80, H8 T4096 56 -> 41 /
// 55 -> 40 / 24 -> 29.  A call cannot see what else runs; the lines are those of one call at a time.
constexpr int scan_update_sets(int K, int BV) { return K == 128 && BV == 32 ? 3 : 4; }  // (four spill there)
constexpr int kMaxCuts = 16;
struct ScanCuts {
  int n;                 // segments of a chain (1 for the delta family)
  int at[kMaxCuts + 1];  // first chunk of each (multiples of scan_update_sets), then NT
};

// BV: value columns per workgroup.  32, and 16 where 32 would leave half of the 256 compute units or more without a workgroup: a
// step is bound by the vector instructions of the two waves of a SIMD, and half the columns are little more than half of them
// (32 -> 16 columns: scalar decay B1 T2048 H8 K = V = 64 21.4 -> 15.9 us, 14 with two operand sets; KDA B1 T2048 H8 K = V = 128 36.7 ->
// 25.2 us).  From
// more than half of the compute units on, a second workgroup of 16 columns would only repeat what does not depend on the columns.
// The linear family, whose chains come in segments (below), takes 16 columns for up to 42 tiles of 32, and for more where the chain is
// too short for segments that make up for it.  GPU us of the whole call with 16 / 32 columns, both in segments, scalar decay: K = V =
// 128 with R_QK, T = 2048 / 8192 / 32768: 32 tiles 24.1 / 26.2, 61.8 / 68.5, 234 / 252; 44 tiles 32.1 / 32.4, 80.9 / 79.8, 365 / 312; 60
// tiles 31.3 / 32.1, 95.1 / 96.3, 430 / 380; K = V = 64: 34 tiles 27.7 / 28.5, 63.5 / 61.8, 284 / 254; 48 tiles 28.2 / 26.9, 85.5 / 76.1,
// 401 / 334; K = V = 128, 96 tiles, T = 512 / 1024 / 2048 / 8192: 17.4 / 17.7, 27.3 / 27.4, 38.9 / 37.2, 131 / 121.
template <bool DELTA, int K, int BV>
struct ChainOps {
  lq_v4i kop[K / 64];                 // key write codes: rows of this wave, 16 token slots of the lane's group
  lq_v4i vop[DELTA ? 1 : BV / 16];    // linear: value write codes
  lq_v4i wop[DELTA ? K / 64 : 1];     // delta: state-read codes of token 16*wave + (lane & 15)
  typename std::conditional<BV == 32, lq_v4i, lq_v2i>::type uraw;  // delta: U of token 16*wave + (lane >> 2), a quarter of the columns
  float misc;                         // lanes 0..15 fw, 16..31 ev of the wave's tokens (delta), 32.. decay of the carry rows
};

template <bool DELTA, bool SCALAR, int K, int BV>
struct OutOps {
  lq_v4i qop[K / 64];                     // codes of q: token 16*w + (lane & 15)
  lq_v4i aop[2];                          // A (fp16): the same token, columns 32 js + 8 kg ..
  lq_v4f g;                               // scalar decay: cumulative log decay of tokens 16*w + 4 kg ..
};

template <int I, int N, typename F>
LQ_DEV void scan_for_from(const F& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    scan_for_from<I + 1, N>(f);
  }
}
template <int N, typename F>
LQ_DEV void scan_for(const F& f) {
  scan_for_from<0, N>(f);
}

// eight int8 codes -> eight exact fp16 values
LQ_DEV lq_v8h scan_i8x8_to_f16x8(lq_v2i c) {
  uint32_t w[4];
  zoo_i8x4_to_f16x4((uint32_t)c[0], w[0], w[1]);
  zoo_i8x4_to_f16x4((uint32_t)c[1], w[2], w[3]);
  return __builtin_bit_cast(lq_v8h, lq_v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]});
}

// Operand sets in rotation: a set is requested D - 1 steps ahead of its use, and the loop is unrolled by D so that the sets
// keep their registers.  Its body has no exit in it (what does not fill D steps follows behind): an exit inside merged, in the
// compiler's count of outstanding requests, paths that had requested less, and the first step of every trip waited for all.
constexpr int scan_sets(bool delta) { return delta ? 3 : 2; }

template <bool DELTA, int DECAY, int K, int BV, bool BF, bool OF32>
__global__ __launch_bounds__(512, DELTA ? 2 : 4) void zoo_scan_kernel(ScanParams p, ScanCuts cuts) {
  constexpr bool SCALAR = DECAY == LQ_DECAY_SCALAR;
  constexpr int D = scan_sets(DELTA), DU = scan_update_sets(K, BV);
  constexpr int KR = K / 4;        // carry rows per chain wave
  constexpr int KT = K / 64;       // 16-row tiles per chain wave
  constexpr int VT = BV / 16;      // 16-column tiles
  constexpr int NJ = BV / 16;      // adjacent value columns per lane in the state reads
  constexpr int HS = K + 16;       // byte stride of a stored-state row in LDS
  constexpr int ES = 64 + 16;      // byte stride of a pseudo-value write-code row
  constexpr int US = 2 * BV + 16;  // byte stride of a token row of the chain's wave-private U tile
  constexpr int LS = 128 + 16;     // byte stride of a channel row of E / of its local codes (64 tokens, 2 bytes each)

  __shared__ __align__(16) unsigned char hT[(DELTA ? 1 : 2) * BV * HS];
  __shared__ __align__(16) unsigned char eT[DELTA ? BV * ES : 16];
  __shared__ __align__(16) unsigned char eB[DELTA ? BV * LS : 16];  // E in the activation dtype, channel-major
  __shared__ __align__(16) unsigned char eL[DELTA ? BV * LS : 16];  // its local codes as fp16, channel-major
  __shared__ __align__(16) unsigned char vL[DELTA ? 16 : 2 * BV * 128];  // linear: local value codes as fp16, operand by operand
  __shared__ __align__(16) unsigned char ue_lds[DELTA ? 4 * 16 * US : 16];
  __shared__ __align__(16) float misc_lds[256];                     // 64 floats per chain wave

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rl = lane & 15, kg = lane >> 4;
  // The V tiles of one (batch, head) read the same key, query, state-read and decay operands at the same time: all of them run on one
  // XCD (workgroups are dealt to the 8 XCDs round-robin, blockIdx.x counts to 8 times the V tiles), and the (batch, head)s, each with
  // its segments, are dealt to the XCDs as evenly as they go; blockIdx.y counts to the most that one XCD has.  (When only grids that
  // divide evenly were renumbered, the operands of the others were fetched by up to eight L2s: T4096 H28 K = V = 128, DeltaNet 145 ->
  // 107 us, KDA 226 -> 187.  Four heads of sixteen tiles with all segments of a head on one XCD left four XCDs idle: T16384 115 us.)
  const uint32_t xcd = blockIdx.x & 7u, mine = blockIdx.y, nseg = DELTA ? 1u : (uint32_t)cuts.n;
  const uint32_t units = (uint32_t)p.B * (uint32_t)p.H * nseg, each = units >> 3, extra = units & 7u;
  if (mine >= each + (xcd < extra ? 1u : 0u)) return;  // (uniform over the workgroup)
  const uint32_t unit = xcd * each + min(xcd, extra) + mine;
  const int vtile = (int)(blockIdx.x >> 3), bh = (int)(DELTA ? unit : unit / nseg);
  const int v0 = vtile * BV;
  const int b = bh / p.H, h = bh % p.H;
  const int H = p.H, V = p.V, T = p.T, NT = p.NT;
  const int qmax = p.qmax;
  constexpr bool bf = BF;
  // linear family: chunks c0 .. c1 - 1 of this workgroup's segment
  const int seg = DELTA ? 0 : (int)(unit - (uint32_t)bh * nseg);
  const int c0 = DELTA ? 0 : cuts.at[seg], c1 = DELTA ? NT : cuts.at[seg + 1];

  if (wv < 4) {
    // ------------------------------------------------------------------------------------------------------- chain
    const int wave = wv;
    __builtin_amdgcn_s_setprio(2);  // the chain is what the launch lasts: it issues first where both waves of a SIMD can
    float skw_r[KT][4], svw_c[VT], inv_ss_c[VT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r) skw_r[kt][r] = p.skw[h * K + KR * wave + 16 * kt + 4 * kg + r];
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      svw_c[vt] = p.svw[h * V + v0 + 16 * vt + rl];
      inv_ss_c[vt] = 1.0f / p.ss[h * V + v0 + 16 * vt + rl];
    }
    float ss_d[NJ], inv_ew_d[NJ], sw = 0.f;
    if (DELTA) {
      sw = p.sw[h];
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj) {
        ss_d[jj] = p.ss[h * V + v0 + NJ * rl + jj];
        inv_ew_d[jj] = 1.0f / p.svw[h * V + v0 + NJ * rl + jj];
      }
    }
    using Ops = ChainOps<DELTA, K, BV>;
    using URaw = decltype(Ops::uraw);
    // float of a lane: per-token factors (delta) in lanes 0 .. 31, chunk decays of the wave's carry rows behind
    const uint32_t misc_at = 4 * (DELTA ? (lane < 32 ? 64 * (lane >> 4) + 16 * wave + (lane & 15) : 128 + KR * wave + min(lane - 32, KR - 1))
                                        : KR * wave + min(max(lane - 32, 0), KR - 1));
    // part: 0 = everything, 1 = key codes, decays and per-token factors, 2 = state-read codes and U
    auto load_part = [&](auto part_c, int ct, Ops& o) __attribute__((always_inline)) {
      constexpr int part = decltype(part_c)::value;
      const int64_t cb = ((int64_t)b * NT + ct) * H + h;
      if constexpr (part == 0 || part == 1) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) o.kop[kt] = zoo_at<lq_v4i>(p.kqT + cb * K * 64, (KR * wave + 16 * kt + rl) * 64 + 16 * kg);
        if constexpr (DELTA) {  // fw[64] | ev[64] | gam[K]
          o.misc = zoo_at<float>(p.pack + cb * (128 + K), misc_at);
        } else {
          if constexpr (DECAY != LQ_DECAY_NONE) o.misc = zoo_at<float>(p.gam + cb * K, misc_at);
#pragma unroll
          for (int vt = 0; vt < VT; ++vt) o.vop[vt] = zoo_at<lq_v4i>(p.vqT + (cb * V + v0) * 64, (16 * vt + rl) * 64 + 16 * kg);
        }
      }
      if constexpr (DELTA && (part == 0 || part == 2)) {
#pragma unroll
        for (int ks = 0; ks < K / 64; ++ks)
          o.wop[ks] = zoo_at<lq_v4i>(p.wq + cb * 64 * K, ((wave * (K / 64) + ks) * 64 + lane) * 16);
        o.uraw = zoo_at<URaw>(p.u + cb * 64 * V + zoo_op_U(0, v0), 2 * zoo_op_U(16 * wave + (lane >> 2), BV / 4 * (lane & 3)));
      }
    };
    float hc[KT][VT][4];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
#pragma unroll
        for (int r = 0; r < 4; ++r) hc[kt][vt][r] = 0.0f;
    float* misc_s = misc_lds + 64 * wave;
    unsigned char* ue_s = ue_lds + wave * 16 * US;

    // write product and carry update
    auto update = [&](const Ops& cur) __attribute__((always_inline)) {
      if constexpr (!DELTA && DECAY != LQ_DECAY_NONE) misc_s[lane] = cur.misc;  // (no earlier: with one set in flight the step would start with this wait)
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        lq_v4i bop;
        if constexpr (DELTA)
          bop = *(const lq_v4i*)(eT + (16 * vt + rl) * ES + 16 * kg);
        else
          bop = cur.vop[vt];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
          const lq_v4i a = lq_mfma_i8(cur.kop[kt], bop, lq_v4i{0, 0, 0, 0});
          lq_v4f gam4;
          if constexpr (DECAY != LQ_DECAY_NONE) gam4 = *(const lq_v4f*)(misc_s + 32 + 16 * kt + 4 * kg);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float prod = (float)a[r] * skw_r[kt][r];
            prod = prod * svw_c[vt];
            if constexpr (DECAY != LQ_DECAY_NONE) hc[kt][vt][r] = hc[kt][vt][r] * gam4[r];  // (no decay: times one)
            hc[kt][vt][r] = hc[kt][vt][r] + prod;
          }
        }
      }
    };

    // one chunk step; the operands of chunk ct + D - 1 are requested into `pre` (unconditionally: the last chunks re-request the
    // final one, so that the compiler's count of outstanding requests does not depend on the path)
    auto do_step = [&](int ct, Ops& cur, Ops& pre) __attribute__((always_inline)) {
      __builtin_amdgcn_sched_barrier(0);  // a request hoisted over the last use of its set would need registers of its own
      unsigned char* hTb = hT + (DELTA ? 0 : (ct & 1) * BV * HS);
      if constexpr (DELTA) {
        misc_s[lane] = cur.misc;
        *(URaw*)(ue_s + (lane >> 2) * US + BV / 2 * (lane & 3)) = cur.uraw;
      }
      // stored copy of the incoming state -> LDS (V-major)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          int cd[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) cd[r] = zoo_q8(hc[kt][vt][r], inv_ss_c[vt], 127);
          *(uint32_t*)(hTb + (16 * vt + rl) * HS + KR * wave + 16 * kt + 4 * kg) = zoo_pack_codes(cd[0], cd[1], cd[2], cd[3]);
        }
      const int ctn = min(ct + D - 1, c1 - 1);
      load_part(std::integral_constant<int, 1>{}, ctn, pre);
      __syncthreads();

      if constexpr (DELTA) {
        // state read against the stored copy, pseudo-values E, their write codes
        lq_v4i aw[NJ];
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) aw[jj] = lq_v4i{0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < K / 64; ++ks)
#pragma unroll
          for (int jj = 0; jj < NJ; ++jj) {
            const lq_v4i hop = *(const lq_v4i*)(hTb + (NJ * rl + jj) * HS + 64 * ks + 16 * kg);
            aw[jj] = lq_mfma_i8(cur.wop[ks], hop, aw[jj]);
          }
        load_part(std::integral_constant<int, 2>{}, ctn, pre);
        uint32_t ecode[NJ][4];
        float ef[NJ][4];
        const lq_v4f fw4 = *(const lq_v4f*)(misc_s + 4 * kg), ev4 = *(const lq_v4f*)(misc_s + 16 + 4 * kg);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const unsigned char* cell = ue_s + (4 * kg + r) * US + 2 * NJ * rl;
          uint32_t uw;
          if constexpr (NJ == 2) uw = *(const uint32_t*)cell; else uw = *(const uint16_t*)cell;
#pragma unroll
          for (int jj = 0; jj < NJ; ++jj) {
            float ws = (float)aw[jj][r] * sw;
            ws = ws * ss_d[jj];
            const float u = zoo_dec1(jj ? uw >> 16 : uw & 0xffffu, bf);
            ef[jj][r] = (u - ws) * fw4[r];
            ecode[jj][r] = (uint32_t)zoo_q8(ef[jj][r] * ev4[r], inv_ew_d[jj], qmax);
          }
        }
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
          *(uint32_t*)(eT + (NJ * rl + jj) * ES + 16 * wave + 4 * kg) =
              zoo_pack_codes((int)ecode[jj][0], (int)ecode[jj][1], (int)ecode[jj][2], (int)ecode[jj][3]);
          lq_v2i eo;
          eo[0] = (int)zoo_enc2(ef[jj][0], ef[jj][1], bf);
          eo[1] = (int)zoo_enc2(ef[jj][2], ef[jj][3], bf);
          *(lq_v2i*)(eB + (NJ * rl + jj) * LS + 2 * (16 * wave + 4 * kg)) = eo;
        }
        __syncthreads();
      }

      update(cur);
    };

    // everything requested so far is waited for once, in front of a loop (a load still outstanding at loop entry would make
    // every iteration wait until almost nothing is in flight)
    auto arrive = [&]() __attribute__((always_inline)) {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      asm volatile("" ::: "memory");
    };
    Ops st[DELTA ? D : DU];
    load_part(std::integral_constant<int, 0>{}, 0, st[0]);
    scan_for<(DELTA ? D : DU) - 1>([&](auto i) __attribute__((always_inline)) { st[i + 1] = st[0]; });
    if constexpr (!DELTA) {
      // the carry that enters the segment: the updates of all chunks in front of it, in their order and with their arithmetic (so
      // with their bits).  No rendezvous: a wave updates its own rows.  The sets hold DU - 1 chunks in flight, and as cuts are
      // multiples of DU, chunk c0 ends up in the first.
      if (c0 > 0) {
        scan_for<DU - 2>([&](auto i) __attribute__((always_inline)) { load_part(std::integral_constant<int, 0>{}, i + 1, st[i + 1]); });
        arrive();
        for (int cu = 0; cu < c0; cu += DU)
          scan_for<DU>([&](auto i) __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            load_part(std::integral_constant<int, 0>{}, min(cu + i + DU - 1, c0), st[(i + DU - 1) % DU]);
            update(st[i]);
          });
      }
    } else {
      scan_for<D - 2>([&](auto i) __attribute__((always_inline)) { load_part(std::integral_constant<int, 0>{}, min(i + 1, NT - 1), st[i + 1]); });
    }
    arrive();
    int ct = c0;
    for (; ct + D <= c1; ct += D) scan_for<D>([&](auto i) __attribute__((always_inline)) { do_step(ct + i, st[i], st[(i + D - 1) % D]); });
    scan_for<D - 1>([&](auto i) __attribute__((always_inline)) {
      if (ct + i < c1) do_step(ct + i, st[i], st[(i + D - 1) % D]);
    });
    if constexpr (DELTA) __syncthreads();  // the output's last local codes (its rendezvous below)

    if (p.ht && c1 == NT) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int vt = 0; vt < VT; ++vt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            p.ht[(((int64_t)b * H + h) * K + KR * wave + 16 * kt + 4 * kg + r) * V + v0 + 16 * vt + rl] = hc[kt][vt][r];
    }
  } else {
    // ------------------------------------------------------------------------------------------------------ output
    const int w = wv - 4;      // token rows 16w .. 16w + 15 of every chunk
    const int ot = tid - 256;  // thread of the output waves
    const float sq = p.sq[h];
    float ss_o[NJ], svl_o[NJ], inv_el = 0.0f;
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) ss_o[jj] = p.ss[h * V + v0 + NJ * rl + jj], svl_o[jj] = p.svl[h * V + v0 + NJ * rl + jj];
    if constexpr (DELTA) inv_el = 1.0f / p.svl[h * V + v0 + ot / (256 / BV)];  // E -> local codes: this thread's column
    using Ops = OutOps<DELTA, SCALAR, K, BV>;
    auto load = [&](int ct, Ops& o) __attribute__((always_inline)) {
      const int64_t cb = ((int64_t)b * NT + ct) * H + h;
#pragma unroll
      for (int ks = 0; ks < K / 64; ++ks) o.qop[ks] = zoo_at<lq_v4i>(p.qc + cb * 64 * K, ((w * (K / 64) + ks) * 64 + lane) * 16);
#pragma unroll
      for (int js = 0; js < 2; ++js) o.aop[js] = zoo_at<lq_v4i>(p.A + cb * 4096, ((w * 2 + js) * 64 + lane) * 16);
      if constexpr (SCALAR) o.g = zoo_at<lq_v4f>(p.gpk + cb * 64, 4 * (16 * w + 4 * kg));
    };
    float of[NJ][4];
    // outputs: elements between tokens, this lane's place in a chunk (once: formed anew for each store, the products by H V took 16 to 25
    // instructions of a quarter of the rate a step)
    const int64_t orow = (int64_t)H * V;
    int64_t olane = (16 * w + 4 * kg) * orow + (int64_t)h * V + v0 + NJ * rl;
    asm volatile("" : "+v"(olane));
    // state read of chunk ct
    auto read_state = [&](int ct, const Ops& o) __attribute__((always_inline)) {
      const unsigned char* hTb = hT + (DELTA ? 0 : (ct & 1) * BV * HS);
      lq_v4i a[NJ];
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj) a[jj] = lq_v4i{0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < K / 64; ++ks)
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
          const lq_v4i hop = *(const lq_v4i*)(hTb + (NJ * rl + jj) * HS + 64 * ks + 16 * kg);
          a[jj] = lq_mfma_i8(o.qop[ks], hop, a[jj]);
        }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float eg = SCALAR ? zoo_exp(o.g[r]) : 1.0f;
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
          float x = (float)a[jj][r] * sq;
          x = x * ss_o[jj];
          of[jj][r] = SCALAR ? x * eg : x;
        }
      }
    };
    // local product of chunk ct on the fp16 MFMA, output
    auto finish = [&](int ct, const Ops& o) __attribute__((always_inline)) {
      lq_v4f loc[NJ];
#pragma unroll
      for (int jj = 0; jj < NJ; ++jj) loc[jj] = lq_v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int js = 0; js < 2; ++js) {
        const lq_v8h aop = __builtin_bit_cast(lq_v8h, o.aop[js]);
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
          lq_v8h x;
          if constexpr (DELTA)
            x = *(const lq_v8h*)(eL + (NJ * rl + jj) * LS + 2 * (32 * js + 8 * kg));
          else
            x = *(const lq_v8h*)(vL + (ct & 1) * BV * 128 + ((jj * 2 + js) * 64 + lane) * 16);
          loc[jj] = lq_mfma_f16(aop, x, loc[jj]);
        }
      }
      const int64_t chunk = ((int64_t)b * T + (int64_t)ct * 64) * orow;  // (uniform)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t off = chunk + r * orow + olane;
        float res[NJ];
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) res[jj] = of[jj][r] + loc[jj][r] * svl_o[jj];
        if constexpr (OF32) {
          float* op = (float*)p.o + off;
          if constexpr (NJ == 2) *(lq_v2i*)op = lq_v2i{__float_as_int(res[0]), __float_as_int(res[1])}; else *op = res[0];
        } else {
          _Float16* op = (_Float16*)p.o + off;
          if constexpr (NJ == 2) *(uint32_t*)op = zoo_enc2(res[0], res[1], bf); else *(uint16_t*)op = zoo_enc1(res[0], bf);
        }
      }
    };
    // E of the chunk the chain has just formed -> its local codes (fp16), BV / 4 tokens of a column per thread
    auto convert = [&]() __attribute__((always_inline)) {
      using Raw = typename std::conditional<BV == 32, lq_v4i, lq_v2i>::type;
      const int at = ot / (256 / BV) * LS + BV / 2 * (ot % (256 / BV));
      const Raw raw = *(const Raw*)(eB + at);
      Raw o;
#pragma unroll
      for (int d = 0; d < BV / 8; ++d) {
        float e0, e1;
        zoo_dec2((uint32_t)raw[d], bf, e0, e1);
        o[d] = (int)zoo_pack_h2((float)zoo_q8(e0, inv_el, qmax), (float)zoo_q8(e1, inv_el, qmax));
      }
      *(Raw*)(eL + at) = o;
    };
    // linear family: the local value codes become fp16 once for all four waves, an operand to a wave (column NJ rl + jj, tokens 32 js + 8 kg
    // .., of jj = w & 1, js = w >> 1; 16 columns: an operand to two of them), a step ahead of their use and requested two
    const int ojj = NJ == 2 ? w & 1 : 0, ojs = w >> 1;
    const int vcol = zoo_op_values(v0 & ~31, 0);
    const uint32_t vlane = zoo_op_values((v0 & 31) + NJ * rl + ojj, 8 * kg) + 8 * ojs;
    lq_v2i vraw[2];
    auto load_v = [&](int ct, lq_v2i& o) __attribute__((always_inline)) {
      if constexpr (!DELTA)
        o = zoo_at<lq_v2i>(p.vcT + (((int64_t)b * NT + ct) * H + h) * 64 * V + vcol, vlane);
    };
    auto convert_v = [&](int ct, const lq_v2i& raw) __attribute__((always_inline)) {
      if constexpr (!DELTA) *(lq_v8h*)(vL + (ct & 1) * BV * 128 + ((ojj * 2 + ojs) * 64 + lane) * 16) = scan_i8x8_to_f16x8(raw);
    };
    // One step: `cur` holds chunk ct, `prev` chunk ct - 1, into which chunk ct + D - 1 is requested once its last use is past.
    auto do_step = [&](auto first_c, int ct, Ops& cur, Ops& prev, lq_v2i& vnext, lq_v2i& vafter) __attribute__((always_inline)) {
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();  // the stored copy of chunk ct is in LDS
      if constexpr (DELTA && !decltype(first_c)::value) finish(ct - 1, prev);
      load(min(ct + D - 1, c1 - 1), prev);
      load_v(min(ct + 2, c1 - 1), vafter);
      read_state(ct, cur);
      if constexpr (DELTA) {
        __syncthreads();  // E of chunk ct is in LDS
        convert();
      } else {
        finish(ct, cur);
        convert_v(ct + 1, vnext);
      }
    };
    Ops st[D];
    load_v(c0, vraw[0]);
    load_v(min(c0 + 1, c1 - 1), vraw[1]);
    load(c0, st[0]);
    scan_for<D - 1>([&](auto i) __attribute__((always_inline)) { st[i + 1] = st[0]; });
    scan_for<D - 2>([&](auto i) __attribute__((always_inline)) { load(min(c0 + i + 1, c1 - 1), st[i + 1]); });
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), as above
    asm volatile("" ::: "memory");
    // (linear family, D = 2: the value codes of chunk c0 + n are requested into vraw[n % 2])
    convert_v(c0, vraw[0]);
    do_step(std::true_type{}, c0, st[0], st[D - 1], vraw[1], vraw[0]);
    int ct = c0 + 1;
    for (; ct + D <= c1; ct += D)
      scan_for<D>([&](auto i) __attribute__((always_inline)) { do_step(std::false_type{}, ct + i, st[(i + 1) % D], st[i], vraw[i % 2], vraw[(i + 1) % 2]); });
    scan_for<D - 1>([&](auto i) __attribute__((always_inline)) {
      if (ct + i < c1) do_step(std::false_type{}, ct + i, st[(i + 1) % D], st[i], vraw[i % 2], vraw[(i + 1) % 2]);
    });
    if constexpr (DELTA) {
      __syncthreads();  // the local codes of the last chunk, written by all four output waves
      scan_for<D>([&](auto i) __attribute__((always_inline)) {
        if ((NT - 1) % D == i) finish(NT - 1, st[i]);
      });
    }
  }
}

// Segments of a chain of NT chunks where `tiles` workgroups of them would run side by side, cut at multiples of `step`
ScanCuts scan_cuts(int64_t tiles, int NT, int step) {
  const int n = (int)std::min((int64_t)kMaxCuts, 256 / tiles);
  ScanCuts c = {};
  double len = 1.0, all = 0.0, at = 0.0;
  for (int s = 0; s < n; ++s) all += len, len *= 0.7;
  len = NT / all;
  for (int s = 1; s < n; ++s) {
    at += len, len *= 0.7;
    const int cut = (int)(at / step + 0.5) * step;
    if (cut > c.at[c.n] && cut < NT) c.at[++c.n] = cut;
  }
  c.at[++c.n] = NT;
  return c;
}

template <bool DELTA, int DECAY, int K, int BV>
int launch(const ScanParams& p, hipStream_t stream) {
  const int64_t tiles = (int64_t)p.B * p.H * (p.V / BV);
  const ScanCuts cuts = DELTA || tiles > 128 ? ScanCuts{1, {0, p.NT}} : scan_cuts(tiles, p.NT, scan_update_sets(K, BV));
  const dim3 grid(8 * (p.V / BV), (p.B * p.H * cuts.n + 7) / 8), block(512);
  if (DELTA && p.o_is_f32 && p.bf)  // (the linear family reads codes only: the activation dtype is that of the output)
    hipLaunchKernelGGL((zoo_scan_kernel<DELTA, DECAY, K, BV, DELTA, true>), grid, block, 0, stream, p, cuts);
  else if (p.o_is_f32)
    hipLaunchKernelGGL((zoo_scan_kernel<DELTA, DECAY, K, BV, false, true>), grid, block, 0, stream, p, cuts);
  else if (p.bf)
    hipLaunchKernelGGL((zoo_scan_kernel<DELTA, DECAY, K, BV, true, false>), grid, block, 0, stream, p, cuts);
  else
    hipLaunchKernelGGL((zoo_scan_kernel<DELTA, DECAY, K, BV, false, false>), grid, block, 0, stream, p, cuts);
  return lq_check_launch();
}

template <bool DELTA, int DECAY, int K>
int launch_bv(const ScanParams& p, hipStream_t stream) {
  const int64_t tiles = (int64_t)p.B * p.H * (p.V / 32);
  // linear family: a tile of 32 columns in more segments is the better use of the same compute units once the chain is long
  const bool few = tiles <= (DELTA || p.NT <= 12 ? 128 : (p.NT <= 32 ? 64 : (p.NT <= 256 ? 42 : 32)));
  return few ? launch<DELTA, DECAY, K, 16>(p, stream) : launch<DELTA, DECAY, K, 32>(p, stream);
}

template <bool DELTA, int DECAY>
int launch_k(const ScanParams& p, int K, hipStream_t stream) {
  return K == 128 ? launch_bv<DELTA, DECAY, 128>(p, stream) : launch_bv<DELTA, DECAY, 64>(p, stream);
}

}  // namespace

int zoo_scan_launch(const ZooScanParams& p, bool delta, int decay, int K, hipStream_t stream) {
  if (decay == LQ_DECAY_NONE) return delta ? launch_k<true, LQ_DECAY_NONE>(p, K, stream) : launch_k<false, LQ_DECAY_NONE>(p, K, stream);
  if (decay == LQ_DECAY_SCALAR) return delta ? launch_k<true, LQ_DECAY_SCALAR>(p, K, stream) : launch_k<false, LQ_DECAY_SCALAR>(p, K, stream);
  return delta ? launch_k<true, LQ_DECAY_DIAGONAL>(p, K, stream) : launch_k<false, LQ_DECAY_DIAGONAL>(p, K, stream);
}
