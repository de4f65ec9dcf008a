// The 16-wave chunked scan of the 16-bit activation types.
#pragma once

#include "scan_common.hpp"

namespace m3 {

// scan16_kernel<T, R, F, SO>: 16-bit activations, ranks 1, 2, 4 and 8, up to N = 128, P = 64 and
// 32 angles, forwards or backwards, with 1024 threads, so that four waves share each SIMD to hide
// one another's LDS, MFMA and transcendental latency. A sub-chunk is 64 rows (token, rank), rank
// minor: 64 / R tokens, whose decay weights, phases and scalars are per token and whose output
// sums the token's R rows (times mimo_out). The work of a sub-chunk c, between workgroup barriers:
//   staging   every wave: row qt's q / k (norm, bias and rotation; waves 0-7 the slots
//             that can rotate, waves 8-15 the others) -> Qs, Ks; row vt's values scaled for the
//             carry -> VS;
//   start     row vt's gate and value -> ZR, VR; the wave's two state tiles, rounded -> Sb, decayed;
//   scores    ten waves one causal tile each (Sc^T = K Q^T) and its decay weights W -> WS;
//   carry     every wave the products of its two state tiles;
//   output    wave w the output tile (row tile w / 4, P tile w % 4): intra V^T W^T from WS, inter
//             rnd(S) Q^T, epilogue, store;
//   phases    of c + 1, on the first waves: a long dependent chain per wave.
// Rank 1, three intervals: staging and start | scores and carry | output and phases (whose waves
// 0-7 have the shortest intra products). Above rank 1, two: start, phases, scores (on the waves
// without phases) and carry of c | staging of c + 1 (Qs has two tiles; Ks and VS were last read in
// the first interval) and output of c. VALU, LDS and MFMA work then share both intervals, and a
// sub-chunk's four waves per SIMD overlap them: 8 x 4096 tokens, 32 heads at rank 4 792 -> 686 us
// per call, the rank-2 hook (4 x 2048) 186 -> 172. Rank 1 in two intervals measured 388 -> 402 (8 x
// 8192): its phases are four times as long, and no wave is left to hide them. The interval
// lengths are set by the SIMD's lowest-priority waves (12-15), not by the first to finish: raising
// the priority of the later waves (s_setprio) measured 2-5% slower.
// Same mathematics and rounding points as scan_kernel (whose header lists them).
//
// Slots. The columns are taken in slot order: the rotation's pairs first, a pair's two columns side
// by side (slots 2j, 2j + 1 of angle j), then the other columns, zeros up to 128. The products sum
// over the columns, so any common order of q, k and the state gives the same result, and one
// staging code serves both rotations (adjacent pairs, and above rank 1 the MIMO pairs (j, j + 2S))
// and every d_state; slot_col() maps a slot back to its column. Slots 0-63 go through the rotation
// with phase 0 past the call's angles (cos 1, sin 0: the value itself).
//
// Forms (F), by where the q / k rows come from:
//   kModel  the model's own shape (N = 128, P = 64, 32 angles, ranks 1 and 4) in projection form:
//           prep's rows in slot order, rounded after the RMSNorm (the reference's rounding point,
//           model.py:48-55);
//   kRows   the other shapes in projection form above rank 1: prep's rows in slot order in FP32, of
//           d_state slots, rounded once after the rotation;
//   kProj   those at rank 1, and any that have no workspace for rows: the caller's rows, normalized
//           in FP32 by prep's factors;
//   kCopy   the hook form (normed rows, phases given or none) above rank 1 where 16 heads or more
//           share a row: prep's copies in slot order;
//   kHook   the hook form elsewhere, and with no workspace for rows: the caller's rows.
// The caller's rows are read as they lie, above rank 1 by two loads of two columns where prep's take
// one of four slots. Measured (32 heads, d_state 128): hook form, rank 2, one group (4 x 2048)
// kCopy 172 us, kHook 192; 32 groups (2 x 1024) 102 and 85; rank 4, 32 groups (4 x 2048) 511 and
// 362; 8 heads at rank 4 (1 x 32768) 355 and 304. Projection form (8 x 1024) kRows 121 us at rank 2
// and 384 at rank 8, kProj, whose normalization at every head spills registers, 147 and 494; at rank
// 1 and d_state 64 73 and 74, with 13.6 and 5.7 MiB of workspace.
//
// LO: d_state no power of 2. Those calls are the recurrent scan's on rows that are not aligned, and
// came from it: it holds the decay weights and the scaled values in FP32, rounding neither. Here
// each becomes two 16-bit operands, the rounded value and the rounding error (for FP16 times 2^11,
// in accumulators of its own, so that it stays a normal number; above 65504 it overflows, as at a
// power of 2), and two products. Output error
// against 64 bits (bf16, 2 x 500 tokens; recurrent scan, one operand each, two weights alone, two
// each): hook form d_state 96 rank 1 2.00e-3, 2.43e-3, 2.04e-3, 1.85e-3; projection form d_state
// 112 rank 2 3.18e-3, 3.28e-3, 3.26e-3, 3.10e-3.

constexpr int k16Threads = 1024;

// LDS layout, 16-bit elements unless noted. The strides and swizzles make every access pattern
// of the kernel conflict-free under the measured gfx950 LDS behaviour: 16-byte reads of 16 rows
// at one 16-byte chunk (the MFMA operands) with 288-byte rows or an XOR swizzle of 256-byte rows;
// 8-byte accesses (stores, transposing reads) 32 lanes at a time over 64 banks of 4 bytes, so
// the 32 lanes' 8-byte pieces must cover 256 distinct bytes.
//   Qs, Ks  [64 tokens][144]: 288-byte rows
//   Sb      [64 p][128]: 256-byte rows, 16-byte chunk c of row p at c ^ (p % 16) (sb_off)
//   VR, VS  [64 tokens][64]: 128-byte rows, 32-byte pair and chunk half swizzled (v_off)
//   ZR      rank 1 the same; above it [64 rows][64] FP32: 256-byte rows, 16-byte chunks
//           XOR-swizzled by row (z_off)
//   WS      [64 t][80]: 160-byte rows
//   WL, VL  (LO) the second operands of WS and VS, laid out as they are; ZR is 16-bit at every rank
struct Lay16Rows {
  static constexpr int ROWS = 64, LQ = kNPad + 16, LS = kNPad, LV = kPPad, LW = kPPad + 16, ES = 2;
};
template <int R, bool LO>
struct Lay16 : Lay16Rows {
  static constexpr bool TWO = R > 1;              // the two-interval schedule
  static constexpr bool ZF32 = TWO && !LO;        // ZR holds the FP32 gate
  static constexpr int QS = 0, QB = ROWS * LQ;    // one or two Qs tiles, QB elements apart
  static constexpr int KS = QS + (TWO ? 2 : 1) * QB * ES;
  static constexpr int VR = KS + ROWS * LQ * ES;
  static constexpr int ZR = VR + ROWS * LV * ES;
  static constexpr int VS = ZR + ROWS * LV * (ZF32 ? 4 : ES);
  static constexpr int SB = VS + ROWS * LV * ES;
  static constexpr int WS = SB + kPPad * LS * ES;  // decay weights [t][s'] (s' permuted, below)
  static constexpr int FB = WS + ROWS * LW * ES;
  // floats from FB: the side blocks (scalar blocks) of two or three sub-chunks, the angle tile, the
  // cos / sin tables (two at rank 1, whose phases run while the staging's table is still needed),
  // the phase block sum and carry per angle
  static constexpr int SCB = 5 * ROWS + 8, SC0 = 0, NSC = TWO ? 3 : 2;
  static constexpr int ANG = SC0 + NSC * SCB;
  static constexpr int CST = 2 * kSMax + 4, CSB = ROWS * CST, NCS = TWO ? 1 : 2;
  static constexpr int CS0 = ANG + ROWS * kSMax, PBASE = CS0 + NCS * CSB, POFF = PBASE + kSMax;
  // ranks above 1: the rounded mimo_x, mimo_z and mimo_out [R][P]
  static constexpr int MP = TWO ? R * kPPad : 0;
  static constexpr int MX = POFF + kSMax, MZ = MX + MP, MO = MZ + MP;
  static constexpr int NW = MO + MP;  // form kProj: the rounded norm weights of q and k, by slot
  static constexpr int WL = FB + 4 * (NW + 2 * kNPad);
  static constexpr int VL = WL + (LO ? ROWS * LW * ES : 0);
  static constexpr int BYTES = VL + (LO ? ROWS * LV * ES : 0);
  static_assert(BYTES <= 160 * 1024, "scan16 LDS layout exceeds 160 KiB");
  static_assert(FB % 16 == 0 && WS % 16 == 0 && SB % 16 == 0 && WL % 16 == 0 && VL % 16 == 0 &&
                    (ANG * 4) % 16 == 0 &&
                    (CS0 * 4) % 16 == 0 && (MX * 4) % 16 == 0 &&
                    (NW * 4) % 16 == 0,
                "alignment");
};

// Element offset of column `col` of state row p in Sb (16-byte chunks XOR-swizzled by row).
__device__ __forceinline__ int sb_off(int p, int col) {
  return p * Lay16Rows::LS + 8 * ((col >> 3) ^ (p & 15)) + (col & 7);
}

// Element offset of column `col` of row r in the FP32 ZR.
__device__ __forceinline__ int z_off(int r, int col) {
  return r * Lay16Rows::LV + 4 * ((col >> 2) ^ (r & 15)) + (col & 3);
}

// Element offset of column `col` of token row r in VR, VS and rank 1's ZR: the row's 32-byte pair
// (col / 16) XOR (r / 2) % 4 and the chunk within it flipped by (r / 8) % 2. Eight consecutive
// rows then place one pair in eight distinct 32-byte bank groups (the transposing reads), and
// sixteen consecutive rows one chunk in sixteen distinct 16-byte groups (the epilogue reads).
__device__ __forceinline__ int v_off(int r, int col) {
  const int c = col >> 3;
  const int pc = 2 * ((c >> 1) ^ ((r >> 1) & 3)) + ((c & 1) ^ ((r >> 3) & 1));
  return r * Lay16Rows::LV + 8 * pc + (col & 7);
}

// The causal score tiles (row tile it, column tile sj <= it) of waves 0-9: the diagonal tiles,
// whose decay weights take the most arithmetic, on waves 0-3 (one per SIMD).
__device__ __forceinline__ void score_tile16(int w, int& it, int& sj) {
  // w: 0 1 2 3 | 4 5 6 7 8 9  ->  (0,0) (1,1) (2,2) (3,3) | (1,0) (2,0) (2,1) (3,0) (3,1) (3,2)
  const int k = w - 4;
  it = w < 4 ? w : (k < 1 ? 1 : (k < 3 ? 2 : 3));
  sj = w < 4 ? w : (k < 1 ? 0 : (k < 3 ? k - 1 : k - 3));
}

template <typename T, int R, Form16 F, bool SO, bool LO>
__global__ __launch_bounds__(k16Threads) void scan16_kernel(const m3_scan_args a,
                                                            const ScanGeom g,
                                                            const float* __restrict__ prep) {
  static_assert(R == 1 || R == 2 || R == 4 || R == 8, "scan16_kernel: ranks 1, 2, 4 and 8");
  static_assert(F != kModel || R == 1 || R == 4, "scan16_kernel: the model's shape");
  using M = Mma<T>;
  static_assert(F != kModel || !LO, "scan16_kernel: the model's d_state is a power of 2");
  using Ly = Lay16<R, LO>;
  constexpr int TOK = 64 / R;  // tokens per 64-row sub-chunk (rows (token, rank), rank minor)
  using SB_ = ScBlk<TOK>;
  constexpr int LQ = Ly::LQ, LW = Ly::LW, CST = Ly::CST, ES = 2;
  constexpr bool PREP = F == kModel || F == kRows || F == kCopy;  // prep's rows; else the caller's
  constexpr bool ROWF = F == kRows;   // in FP32
  constexpr bool NORM = F == kProj;   // to be normalized here
  constexpr bool GIVEN = F == kHook || F == kCopy;  // phases given (or none), no increments
  const int N = F == kModel ? kNPad : a.d_state;
  const int RB = ROWF ? N * 4 : kNPad * 2;  // bytes of one of prep's rows
  const int P = F == kModel ? kPPad : a.head_dim;
  const int S = F == kModel ? kSMax : a.num_angles;
  // phase: PG lanes per angle, TPL tokens per lane, on the first PG / 2 waves (32 angles)
  constexpr int TPL = F == kModel && R == 4 ? 1 : 4;
  constexpr int PG = TOK / TPL, PW = PG * kSMax / 64;
  const int H = a.heads;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;

  int bid = blockIdx.x;
  if (g.xcd_map) {
    const int per = gridDim.x >> 3;
    bid = (bid & 7) * per + (bid >> 3);
  }
  // segment sgi of batch row b (one unless the call is split): tokens tok0 .. tok0 + L - 1, its
  // sub-chunks from the row's sub-chunk c0 on
  const int bs = bid / H, h = bid - bs * H;
  const int b = g.segs > 1 ? bs / g.segs : bs, sgi = bs - b * g.segs;
  const int tok0 = sgi * g.seg_len, c0 = tok0 / TOK;
  const int L = min(g.seg_len, a.length - tok0);
  const int nsub = (L + TOK - 1) / TOK;
  const int GRP = F == kModel ? 1 : a.groups;
  const int grp = F == kModel ? 0 : h / (H / GRP);
  const int perm = R == 1 ? 0 : F == kModel ? 1 : g.perm;
  auto col = [&](int slot) { return slot_col(slot, perm, S); };

  extern __shared__ __attribute__((aligned(16))) char smem[];
  T* Qs = lds_t<T>(smem, Ly::QS);
  T* Ks = lds_t<T>(smem, Ly::KS);
  T* VR = lds_t<T>(smem, Ly::VR);
  T* ZR = lds_t<T>(smem, Ly::ZR);
  float* ZF = lds_t<float>(smem, Ly::ZR);  // Ly::ZF32
  T* VS = lds_t<T>(smem, Ly::VS);
  T* Sb = lds_t<T>(smem, Ly::SB);
  T* WS = lds_t<T>(smem, Ly::WS);
  T* WL = lds_t<T>(smem, Ly::WL);
  T* VL = lds_t<T>(smem, Ly::VL);
  // LO: the factor of the second operands; other than 1 they have accumulators of their own
  constexpr float kLo = sizeof(T) == 2 && std::is_same<T, _Float16>::value ? 2048.f : 1.f;
  constexpr bool LOA = LO && kLo != 1.f;
  auto low = [](f4 x) {
    f4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = (x[i] - rnd<T>(x[i])) * kLo;
    return y;
  };
  float* F_ = lds_t<float>(smem, Ly::FB);

  // ---- lane roles
  // q / k: rows qt and qt + 32 (rank qr), slots n0 .. n0 + 3 (waves 0-7 the slots 0-63)
  const bool rot = w < 8;
  const int qt = (tid & 511) >> 4, qr = qt & (R - 1);
  const int n0 = 64 * (tid >> 9) + 4 * (tid & 15);
  // value / gate: row vt (token vt / R, rank vt % R), columns p0 .. p0+3
  const int vt = tid >> 4, p0 = 4 * (tid & 15);
  // phase (the first PW waves): angle ps, tokens TPL pg .. TPL pg + TPL - 1
  const int ps = tid / PG, pg = tid & (PG - 1);
  const bool ph_wave = w < PW;
  // state tiles (ni, pj), k = 0, 1: ni = w / 2, pj = 2 (w % 2) + k; lane holds
  // n = 16 ni + 4 lg + i, p = 16 pj + l16 (S^T in MFMA accumulator layout)
  const int sni = w >> 1, spj0 = 2 * (w & 1);

  // ---- global reads: one buffer resource per tensor and (batch, head) whose extent ends with
  // token L - 1, so rows of tokens past it read zero and stores past it are dropped (a token's
  // row ends below the next token's: the host's check); backwards, logical token t is the
  // physical row L - 1 - t and the resource starts at physical row 0. Per-lane byte offsets at
  // logical token 0.
  struct Rows {
    __amdgpu_buffer_rsrc_t rs;
    int step, o0;  // bytes from a token to the next, offset of logical token 0
  };
  auto rows_of = [&](const m3_tensor& t, int64_t head_off, int span, int es) {
    const int64_t s1 = t.stride[1];
    const int64_t back = s1 < 0 ? (L - 1) * s1 : 0;
    Rows r;
    r.rs = make_rsrc(static_cast<const char*>(t.ptr) +
                         (b * t.stride[0] + tok0 * s1 + head_off + back) * es,
                     static_cast<int>(((L - 1) * (s1 < 0 ? -s1 : s1) + span) * es));
    r.step = static_cast<int>(s1) * es;
    r.o0 = static_cast<int>(-back) * es;
    return r;
  };
  const Rows gv = rows_of(a.value, h * a.value.stride[2], P, ES);
  const Rows gz = rows_of(a.gate, h * a.gate.stride[2], P, ES);
  const Rows go = rows_of(a.out, h * a.out.stride[2], P, ES);
  // lanes past column P read columns 0-3: their VR / VS / ZR columns and state rows are never
  // stored to memory
  const int p0c = p0 < P ? p0 : 0;
  const int o_v = gv.o0 + (vt / R) * gv.step + p0c * ES;
  const int o_z = gz.o0 + (vt / R) * gz.step + p0c * ES;
  // prep's q / k rows of batch row b: row (token, group, rank) at 2 RB bytes, k after q; 32 rows on: 32
  // / R tokens
  const int tok_qk = GRP * R * 2 * RB;
  const __amdgpu_buffer_rsrc_t rs_qk =
      PREP ? make_rsrc(reinterpret_cast<const char*>(prep) + g.ws_qk +
                           (static_cast<int64_t>(b) * a.length + tok0) * tok_qk,
                       L * tok_qk)
           : make_rsrc(nullptr, 0);
  // the caller's rows: the columns of slots n0 .. n0 + 3, which above rank 1 are two words `d2`
  // bytes apart (a MIMO pair's columns; the words of two pairs are put side by side at the staging,
  // v_perm selectors selA and selB); lanes past column N read past every extent (kOut: not moved
  // with the token). prep's norm factors (q, k) of the same row.
  constexpr int kOut = INT32_MIN;  // as an unsigned offset 2^31, the extents are below it
  const bool in_n = (PREP && !ROWF) || n0 < N;
  // (prep's rows run forwards, less than 2^31 bytes: a lane may start at kOut and move with the token)
  const int o_qk =
      in_n ? (qt / R) * tok_qk + (grp * R + qr) * 2 * RB + n0 * (ROWF ? 4 : ES) : kOut;
  const bool pair = !PREP && perm && n0 < 2 * S;
  const int c0q = col(n0), d2 = (pair ? 2 * S : 2) * ES;
  const uint32_t selA = pair ? 0x05040100u : 0x03020100u, selB = pair ? 0x07060302u : 0x07060504u;
  const int qr_s = PREP ? 0 : static_cast<int>(a.q.stride[3]);
  const int kr_s = PREP ? 0 : static_cast<int>(a.k.stride[3]);
  const Rows none{make_rsrc(nullptr, 0), 0, 0};
  const Rows gq = PREP ? none : rows_of(a.q, grp * a.q.stride[2], (R - 1) * qr_s + N, ES);
  const Rows gk = PREP ? none : rows_of(a.k, grp * a.k.stride[2], (R - 1) * kr_s + N, ES);
  const int o_q = gq.o0 + (qt / R) * gq.step + (qr * qr_s + c0q) * ES;
  const int o_k = gk.o0 + (qt / R) * gk.step + (qr * kr_s + c0q) * ES;
  const int tok_n = GRP * R * 8;
  const __amdgpu_buffer_rsrc_t rs_n =
      NORM ? make_rsrc(prep + g.ws_norm + (static_cast<int64_t>(b) * a.length + tok0) * GRP * R * 2,
                       L * tok_n)
           : make_rsrc(nullptr, 0);
  const int o_n = (qt / R) * tok_n + (grp * R + qr) * 8;
  const int scw = g.scw;
  // side words (waves 0-3, one float pair per lane): the scalar block
  const int q2 = 2 * tid;
  const bool side_on = q2 < scw;
  const __amdgpu_buffer_rsrc_t rs_s =
      make_rsrc(prep + g.ws_sc + (static_cast<int64_t>(b * H + h) * g.nsub + c0) * scw, nsub * scw * 4);
  const int side_o = side_on ? q2 * 4 : 0;
  const int side_s = scw * 4;
  // angle words: 4 tokens of angle tid % 32 each, in the tile order [TOK / 4][32][4]; prep's
  // increments [L4][S][4], or the given phases. Lanes past angle S read past the extent (zero).
  const bool ang_on = tid < TOK * kSMax / 4;
  const int agq = tid / kSMax, asl = tid & (kSMax - 1);
  constexpr int kPast = 0x40000000;  // beyond every extent (below 2^30 bytes), also advanced
  const __amdgpu_buffer_rsrc_t rs_a =
      GIVEN ? make_rsrc(nullptr, 0)
            : make_rsrc(prep + g.ws_ang + (static_cast<int64_t>(b) * g.L4 + tok0 / 4) * S * 4,
                        (L + 3) / 4 * S * 16);
  const int ang_o = asl < S ? (agq * S + asl) * 16 : kPast;
  const int ang_s = (TOK / 4) * S * 16;
  const bool phases_in = GIVEN && a.phase_mode == M3_PHASE_GIVEN;
  const Rows gx = phases_in ? rows_of(a.phase, h * a.phase.stride[2],
                                      (S - 1) * static_cast<int>(a.phase.stride[3]) + 1, 4)
                            : Rows{make_rsrc(nullptr, 0), 0, 0};
  const int o_x = gx.o0 + 4 * agq * gx.step + asl * static_cast<int>(a.phase.stride[3]) * 4;

  // where the end state, phase and k go: the segment's own slots (pass 1 of a split call), or the
  // call's outputs, written by the last segment alone
  const bool fin = !g.last_only || sgi == g.segs - 1;
  const int bo = g.last_only ? b : bs;
  float* fph = a.final_phase.ptr != nullptr && fin && ph_wave && ps < S
                   ? static_cast<float*>(a.final_phase.ptr) + bo * a.final_phase.stride[0] +
                         h * a.final_phase.stride[1] + ps * a.final_phase.stride[2]
                   : nullptr;
  float* fblk = a.block_phase.ptr != nullptr && ph_wave && ps < S
                    ? static_cast<float*>(a.block_phase.ptr) + b * a.block_phase.stride[0] +
                          h * a.block_phase.stride[1] + (tok0 >> 6) * a.block_phase.stride[2] +
                          ps * a.block_phase.stride[3]
                    : nullptr;
  const int64_t blk_stride = a.block_phase.stride[2];

  // q / k words: rows qt and qt + 32, q and k, 4 slots each; their norm factors
  using RowT = std::conditional_t<ROWF, float, T>;
  constexpr int QW = ROWF ? 4 : 2;
  uint32_t rq[2][QW], rk[2][QW], rv[2], rz[2];
  u32x2 fac[2];
  float2 side = make_float2(0.f, 0.f);
  float4 ang = make_float4(0.f, 0.f, 0.f, 0.f);
  auto load_qk = [&](int t0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int tj = t0 + (32 / R) * j;
      if constexpr (PREP) {
        const int o = o_qk + tj * tok_qk;
        bload_words<QW>(rq[j], rs_qk, o);
        bload_words<QW>(rk[j], rs_qk, o + RB);
      } else {
        auto row = [&](uint32_t (&w2)[2], const Rows& x, int o) {
          const int oo = in_n ? o + tj * x.step : kOut;
          if constexpr (R == 1) {
            bload_words<2>(w2, x.rs, oo);
          } else {
            w2[0] = __builtin_amdgcn_raw_buffer_load_b32(x.rs, oo, 0, 0);
            w2[1] = __builtin_amdgcn_raw_buffer_load_b32(x.rs, oo + d2, 0, 0);
          }
        };
        row(rq[j], gq, o_q);
        row(rk[j], gk, o_k);
        if constexpr (NORM) {
          fac[j] = __builtin_bit_cast(
              u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs_n, o_n + tj * tok_n, 0, 0));
        }
      }
    }
  };
  auto load_vz = [&](int t0) {
    bload_words<2>(rv, gv.rs, o_v + t0 * gv.step);
    bload_words<2>(rz, gz.rs, o_z + t0 * gz.step);
  };
  auto load_side = [&](int c) {
    if (w < 4) {
      const u32x2 v = __builtin_bit_cast(
          u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs_s, side_o + c * side_s, 0, 0));
      side = make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
    }
    if (w < 8) {
      if constexpr (GIVEN) {
        // lanes past the call's angles stay at kPast: moved on with the others, backwards (a
        // negative step) they would come back into an extent above half of 2^30 bytes. The host
        // keeps 256 tokens between every extent and 2^30, so the 4 steps below stay past it too.
        const int o = asl < S ? o_x + c * TOK * gx.step : kPast;
        ang = make_float4(bload_f32(gx.rs, o), bload_f32(gx.rs, o + gx.step),
                          bload_f32(gx.rs, o + 2 * gx.step), bload_f32(gx.rs, o + 3 * gx.step));
      } else {
        const u32x4 v = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_a, ang_o + c * ang_s, 0, 0));
        ang = make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]),
                          __uint_as_float(v[3]));
      }
    }
  };
  float* ANG = F_ + Ly::ANG;
  // angle tile slot of 4-token group gq and angle s (XOR-keyed by the group's phase lane)
  auto ang_slot = [&](int gq, int s) { return gq * kSMax + (s ^ gq); };
  // side block slots (floats from F_) of sub-chunks c, c + 1 and c + 2, rotated once per sub-chunk
  int sc0 = Ly::SC0, sc1 = sc0 + Ly::SCB, sc2 = sc1 + Ly::SCB;
  auto put_side = [&](int slot) {
    if (w < 4 && side_on) *reinterpret_cast<float2*>(F_ + slot + q2) = side;
    if (w < 8 && ang_on) *reinterpret_cast<float4*>(ANG + 4 * ang_slot(agq, asl)) = ang;
  };
  auto cst = [&](int c) { return F_ + Ly::CS0 + (Ly::NCS == 2 ? c & 1 : 0) * Ly::CSB; };
  auto phases = [&](int c, int slot) {
    // phases of sub-chunk c (the phase waves), from the angle tile and the dt of its side block
    if (ph_wave && c < nsub) {
      float pa[TPL];
      if constexpr (TPL == 4) {
        const float4 v = *reinterpret_cast<const float4*>(ANG + 4 * ang_slot(pg, ps));
        pa[0] = v.x;
        pa[1] = v.y;
        pa[2] = v.z;
        pa[3] = v.w;
      } else {
        pa[0] = ANG[4 * ang_slot(pg >> 2, ps) + (pg & 3)];  // token pg of its 4-token group
      }
      phase_stage<PG, TPL, CST, true, false, GIVEN && LO ? kWide : kFast>(
          cst(c), ps, F_ + Ly::PBASE + ps, F_ + Ly::POFF + ps,
                                             F_ + slot + SB_::DTV, c * TOK, L, pg, lane, !GIVEN, pa,
                                             fph, fblk, blk_stride);
    }
  };

  // ---- prologue. A short sequence, or one segment of a split one, is a few sub-chunks, and 16
  // waves issue every instruction of this: the parameters are read through buffer resources at
  // 32-bit offsets, a dtype tested once for a whole group of loads, what a call does not have
  // skipped. First the words of sub-chunk 0, then everything else, waited for afterwards.
  load_side(0);
  load_qk(0);
  load_vz(0);
  __builtin_amdgcn_sched_barrier(0);
  // E elements of a parameter row at element offsets o[]: raw bits, decoded after the waits
  auto ld_raw = [&](__amdgpu_buffer_rsrc_t rs, int dtype, const auto& o, auto& raw) {
    constexpr int E = sizeof(raw) / 4;
    if (dtype == M3_F32) {
#pragma unroll
      for (int i = 0; i < E; ++i) raw[i] = __builtin_amdgcn_raw_buffer_load_b32(rs, o[i] * 4, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < E; ++i) raw[i] = __builtin_amdgcn_raw_buffer_load_b16(rs, o[i] * 2, 0, 0);
    }
  };
  auto decode_raw = [&](int dtype, const auto& raw, auto& v) {
    constexpr int E = sizeof(raw) / 4;
    if (dtype == M3_F32) {
#pragma unroll
      for (int i = 0; i < E; ++i) v[i] = __uint_as_float(raw[i]);
    } else if (dtype == M3_BF16) {
#pragma unroll
      for (int i = 0; i < E; ++i) v[i] = __uint_as_float(raw[i] << 16);
    } else {
#pragma unroll
      for (int i = 0; i < E; ++i) v[i] = bits_to_f(raw[i], static_cast<_Float16*>(nullptr));
    }
  };
  // head h's slice of a parameter [H, ..] whose rows end `n` elements after its start
  auto head_rs = [&](const m3_tensor& t, int n) {
    const int es = t.dtype == M3_F32 ? 4 : 2;
    return make_rsrc(static_cast<const char*>(t.ptr) + h * t.stride[0] * es, n * es);
  };
  // biases of the lane's 4 slots, rank qr (slots past the call's columns read past the extent)
  const bool bias = !GIVEN || a.q_bias.ptr != nullptr;
  uint32_t bq_r[4] = {0u, 0u, 0u, 0u}, bk_r[4] = {0u, 0u, 0u, 0u};
  if (bias) {
    const int qs = static_cast<int>(a.q_bias.stride[1]), ks = static_cast<int>(a.k_bias.stride[1]);
    int oq[4], ok[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool on = F == kModel || n0 + i < N;
      oq[i] = on ? qr * qs + col(n0 + i) : kPast / 4;
      ok[i] = on ? qr * ks + col(n0 + i) : kPast / 4;
    }
    ld_raw(head_rs(a.q_bias, (R - 1) * qs + N), a.q_bias.dtype, oq, bq_r);
    ld_raw(head_rs(a.k_bias, (R - 1) * ks + N), a.k_bias.dtype, ok, bk_r);
  }
  uint32_t mx_r[1], mz_r[1], mo_r[1];
  if constexpr (R > 1) {
    // mimo_x / mimo_z and mimo_out of this head, element tid of [R][P] (ops.py:700-714, 869-877)
    const int r = tid / kPPad, p = min(tid & (kPPad - 1), P - 1);
    auto ld_mimo = [&](const m3_tensor& t, uint32_t (&raw)[1]) {
      const int rs = static_cast<int>(t.stride[1]);
      const int o[1] = {r < R ? r * rs + p : kPast / 4};
      ld_raw(head_rs(t, (R - 1) * rs + P), t.dtype, o, raw);
    };
    ld_mimo(a.mimo_x, mx_r);
    ld_mimo(a.mimo_z, mz_r);
    ld_mimo(a.mimo_out, mo_r);
  }
  const float Dh = ldx(a.D.ptr, a.D.dtype, h * a.D.stride[0]);
  float po = 0.f;  // the phase carry of angle tid
  if (a.initial_phase.ptr != nullptr && tid < S) {
    po = static_cast<const float*>(a.initial_phase.ptr)
        [bs * a.initial_phase.stride[0] + h * a.initial_phase.stride[1] +
         tid * a.initial_phase.stride[2]];
  }
  // the lane's state elements: offsets of (p, column) in floats, row stride `sp`, and its [P, N]
  // slice's resource (the final state is stored the same way)
  auto state_rs = [&](const m3_tensor& t, int row) {
    const int sp = static_cast<int>(t.stride[2]);
    return make_rsrc(static_cast<const float*>(t.ptr) + row * t.stride[0] + h * t.stride[1],
                     ((P - 1) * sp + N) * 4);
  };
  auto state_off = [&](int k, int i, int sp) {
    const int p = 16 * (spj0 + k) + l16, sl = 16 * sni + 4 * lg + i;
    return F == kModel || (p < P && sl < N) ? (p * sp + col(sl)) * 4 : kPast;
  };
  f4 st[2] = {zero4(), zero4()};
  if (a.initial_state.ptr != nullptr) {
    const __amdgpu_buffer_rsrc_t rs = state_rs(a.initial_state, bs);
    const int sp = static_cast<int>(a.initial_state.stride[2]);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int i = 0; i < 4; ++i) st[k][i] = bload_f32(rs, state_off(k, i, sp));
    }
  }
  // Endpoint continuation (ops.py:681-686): S += dt_0 (1 - trap_0) sum_r (v_prev mx_r) k_prev_r^T.
  if (a.initial_k.ptr != nullptr) {
    const RawX dt_r = ldraw(a.dt.ptr, a.dt.dtype,
                            b * a.dt.stride[0] + tok0 * a.dt.stride[1] + h * a.dt.stride[2]);
    const RawX tr_r = ldraw(a.trap.ptr, a.trap.dtype,
                            b * a.trap.stride[0] + tok0 * a.trap.stride[1] + h * a.trap.stride[2]);
    const RawX db_r = GIVEN ? RawX{0u, 0u}
                                 : ldraw(a.dt_bias.ptr, a.dt_bias.dtype, h * a.dt_bias.stride[0]);
    const int kr_s = static_cast<int>(a.initial_k.stride[2]);
    const __amdgpu_buffer_rsrc_t rs_v =
        make_rsrc(static_cast<const T*>(a.initial_value.ptr) + bs * a.initial_value.stride[0] +
                      h * a.initial_value.stride[1],
                  P * ES);
    const __amdgpu_buffer_rsrc_t rs_k =
        make_rsrc(static_cast<const T*>(a.initial_k.ptr) + bs * a.initial_k.stride[0] +
                      h * a.initial_k.stride[1],
                  ((R - 1) * kr_s + N) * ES);
    auto b16 = [&](__amdgpu_buffer_rsrc_t r, int i) {
      return bits_to_f(__builtin_amdgcn_raw_buffer_load_b16(r, i * ES, 0, 0),
                       static_cast<T*>(nullptr));
    };
    float v0[2], k0[R][4], mxv[2][R];
#pragma unroll
    for (int k = 0; k < 2; ++k) v0[k] = b16(rs_v, 16 * (spj0 + k) + l16);
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int sl = 16 * sni + 4 * lg + i;
        k0[r][i] = b16(rs_k, F == kModel || sl < N ? r * kr_s + col(sl) : kPast / ES);
      }
      if constexpr (R > 1) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          mxv[k][r] = rnd<T>(ldx(a.mimo_x.ptr, a.mimo_x.dtype,
                                 h * a.mimo_x.stride[0] + r * a.mimo_x.stride[1] +
                                     min(16 * (spj0 + k) + l16, P - 1)));
        }
      }
    }
    float dt0, adt0;
    dt_adt(!GIVEN, decode(dt_r, a.dt.dtype), 0.f, decode(db_r, GIVEN ? 0 : a.dt_bias.dtype),
           dt0, adt0);
    const float c0 = dt0 * (1.f - sigmoidf(decode(tr_r, a.trap.dtype)));
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float outer = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          outer += (R > 1 ? mul_r<T>(v0[k], mxv[k][r]) : v0[k]) * k0[r][i];
        }
        st[k][i] += c0 * outer;
      }
    }
  }
  // norm weights, slot tid % 128 of q (threads 0-127) or k
  float nw = 0.f;
  if constexpr (NORM) {
    const m3_tensor& t = tid < kNPad ? a.q_norm_w : a.k_norm_w;
    const int sl = tid & (kNPad - 1);
    if (tid < 2 * kNPad && sl < N) nw = rnd<T>(ldx(t.ptr, t.dtype, col(sl) * t.stride[0]));
  }
  __builtin_amdgcn_sched_barrier(0);
  put_side(sc0);
  load_side(1);
  if (NORM && tid < 2 * kNPad) F_[Ly::NW + tid] = nw;
  if (tid < kSMax) {
    F_[Ly::PBASE + tid] = 0.f;
    F_[Ly::POFF + tid] = po;
  }
  float bq[4], bk[4];
  decode_raw(a.q_bias.dtype, bq_r, bq);
  decode_raw(a.k_bias.dtype, bk_r, bk);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    bq[i] = rnd<T>(bq[i]);
    bk[i] = rnd<T>(bk[i]);
  }
  if constexpr (R > 1) {
    if (tid < R * kPPad) {
      float x[1], z[1], o[1];
      decode_raw(a.mimo_x.dtype, mx_r, x);
      decode_raw(a.mimo_z.dtype, mz_r, z);
      decode_raw(a.mimo_out.dtype, mo_r, o);
      F_[Ly::MX + tid] = rnd<T>(x[0]);
      F_[Ly::MZ + tid] = rnd<T>(z[0]);
      F_[Ly::MO + tid] = o[0];
    }
  }
  __syncthreads();
  phases(0, sc0);
  // q / k of the coming sub-chunk -> its Qs tile and Ks
  // (`qo`: the Qs tile's element offset). Rank 1 addresses q and k, and the two state tiles, from
  // one base each, so that two stores are one instruction: 404 -> 390 us at 8 x 8192; at rank 4 the
  // same measured 686 -> 701 (8 x 4096).
  auto stage_qk = [&](int qo, const float* CSt) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      // row rw (token tt): q = q^ + bias, k = k^ + bias, rotated: pairs (n0, n0 + 1) and
      // (n0 + 2, n0 + 3), angles n0 / 2 and n0 / 2 + 1, adjacent in the cos / sin table row
      const int rw = qt + 32 * j, tt = rw / R;
      f4 q, k;
      if constexpr (!PREP && R > 1) {
        const uint32_t q0 = rq[j][0], q1 = rq[j][1], k0 = rk[j][0], k1 = rk[j][1];
        rq[j][0] = __builtin_amdgcn_perm(q1, q0, selA);
        rq[j][1] = __builtin_amdgcn_perm(q1, q0, selB);
        rk[j][0] = __builtin_amdgcn_perm(k1, k0, selA);
        rk[j][1] = __builtin_amdgcn_perm(k1, k0, selB);
      }
      if constexpr (NORM) {
        const float fq = __uint_as_float(fac[j][0]), fk = __uint_as_float(fac[j][1]);
        const f4 wq = *reinterpret_cast<const f4*>(F_ + Ly::NW + n0);
        const f4 wk = *reinterpret_cast<const f4*>(F_ + Ly::NW + kNPad + n0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          q[i] = fmaf(raw_get<T>(rq[j], i) * fq, wq[i], bq[i]);
          k[i] = fmaf(raw_get<T>(rk[j], i) * fk, wk[i], bk[i]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          q[i] = raw_get<RowT>(rq[j], i) + bq[i];
          k[i] = raw_get<RowT>(rk[j], i) + bk[i];
        }
      }
      if (rot) {
        const f4 cv = *reinterpret_cast<const f4*>(CSt + tt * CST + 2 * cs_col<true>(n0 >> 1, tt));
#pragma unroll
        for (int pp = 0; pp < 2; ++pp) {
          const float cc = cv[2 * pp], ss = cv[2 * pp + 1];
          const float q0 = q[2 * pp], q1 = q[2 * pp + 1];
          const float k0 = k[2 * pp], k1 = k[2 * pp + 1];
          q[2 * pp] = fmaf(q0, cc, -(q1 * ss));
          q[2 * pp + 1] = fmaf(q0, ss, q1 * cc);
          k[2 * pp] = fmaf(k0, cc, -(k1 * ss));
          k[2 * pp + 1] = fmaf(k0, ss, k1 * cc);
        }
      }
      T* qd = R == 1 ? Qs + qt * LQ + n0 + 32 * j * LQ : Qs + rw * LQ + n0;
      T* kd = R == 1 ? Qs + qt * LQ + n0 + (Ly::KS - Ly::QS) / ES + 32 * j * LQ : Ks + rw * LQ + n0;
      if constexpr (!SO) st_quad<T>(qd + qo, q);
      st_quad<T>(kd, k);
    }
  };
  // its values scaled for the carry -> VS: value (above rank 1 times the rounded mimo_x of the
  // row's rank, rounded, kept in rv) * scale * exp(cum_last - cum)
  auto stage_vs = [&](const float* SN) {
    const int tv = vt / R;
    const float ev = SN[SB_::SCL + tv] * __expf(SN[SB_::CL] - SN[SB_::CUM + tv]);
    f4 vq;
#pragma unroll
    for (int i = 0; i < 4; ++i) vq[i] = raw_get<T>(rv, i);
    if constexpr (R > 1) {
      const f4 mx = *reinterpret_cast<const f4*>(F_ + Ly::MX + (vt & (R - 1)) * kPPad + p0);
#pragma unroll
      for (int i = 0; i < 4; ++i) vq[i] *= mx[i];
      rv[0] = pack2<T>(vq[0], vq[1]);
      rv[1] = pack2<T>(vq[2], vq[3]);
#pragma unroll
      for (int i = 0; i < 4; ++i) vq[i] = raw_get<T>(rv, i);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) vq[i] *= ev;
    st_quad<T>(VS + v_off(vt, p0), vq);
    if constexpr (LO) st_quad<T>(VL + v_off(vt, p0), low(vq));
  };
  // the gate of row vt -> ZR (rank 1 as loaded; above it silu of the rounded z * mimo_z in FP32, so
  // that the interval with the staging has less of the transcendental work, LO the product itself),
  // its values -> VR,
  // the state at the sub-chunk's start, rounded -> Sb
  auto stage_out = [&] {
    if constexpr (!SO) {
      if constexpr (R == 1) {
        *reinterpret_cast<u32x2*>(ZR + v_off(vt, p0)) = (u32x2){rz[0], rz[1]};
      } else {
        const f4 mz = *reinterpret_cast<const f4*>(F_ + Ly::MZ + (vt & (R - 1)) * kPPad + p0);
        f4 zq;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float zm = mul_r<T>(raw_get<T>(rz, i), mz[i]);
          zq[i] = Ly::ZF32 ? silu_fast(zm) : zm;
        }
        if constexpr (Ly::ZF32) {
          *reinterpret_cast<f4*>(ZF + z_off(vt, p0)) = zq;
        } else {
          st_quad<T>(ZR + v_off(vt, p0), zq);
        }
      }
      *reinterpret_cast<u32x2*>(VR + v_off(vt, p0)) = (u32x2){rv[0], rv[1]};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int so = R == 1 ? sb_off(16 * spj0 + l16, 16 * sni + 4 * lg) + 16 * k * Ly::LS
                              : sb_off(16 * (spj0 + k) + l16, 16 * sni + 4 * lg);
        st_quad<T>(Sb + so, st[k]);
      }
    }
  };
  float log_decay = 0.f;
  auto decay_state = [&](const float* SC) {
    {
      const float ecl = SC[SB_::ECL];
      log_decay += SC[LO ? SB_::DEC : SB_::CL];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) st[k][i] *= ecl;
      }
    }
  };
  // causal score tile `tile` (score_tile16) and its decay weights -> WS
  auto scores = [&](int tile, const T* Qc, const float* SC) {
    if constexpr (!SO) {
      int it, sj;
      score_tile16(tile, it, sj);
      const int tq = 16 * it + l16;
      f4 acc = zero4();
      // (four waves per SIMD hide the operand latency: one k-step's operands in registers at a
      // time keeps the kernel within 128 VGPRs)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const typename M::v8 av = *reinterpret_cast<const typename M::v8*>(
            Ks + (16 * sj + l16) * LQ + 32 * kk + 8 * lg);
        const typename M::v8 bv =
            *reinterpret_cast<const typename M::v8*>(Qc + tq * LQ + 32 * kk + 8 * lg);
        acc = M::mma(av, bv, acc);
        __builtin_amdgcn_sched_barrier(0);
      }
      // decay weights by token: row tq is token tq / R, column rows 16 sj + 4 lg + i are
      // tokens (16 sj + 4 lg + i) / R: TS tokens, 4 / TS of the rows each
      constexpr int TS = R >= 4 ? 1 : 4 / R;
      const int tqt = tq / R;
      const float cum_t = SC[SB_::CUM + tqt];
      f4 wv;
      if (sj < it) {
        // d = exp(cum_t - cend) * (scale_s exp(cend - cum_s)), both factors <= 1
        const float at = __expf(cum_t - SC[SB_::CEND + sj]);
        if constexpr (R == 1) {
          const f4 bs = *reinterpret_cast<const f4*>(SC + SB_::BSC + 16 * sj + 4 * lg);
#pragma unroll
          for (int i = 0; i < 4; ++i) wv[i] = acc[i] * (at * bs[i]);
        } else {
          float bs[TS];
#pragma unroll
          for (int j = 0; j < TS; ++j) bs[j] = SC[SB_::BSC + (16 * sj + 4 * lg) / R + j];
#pragma unroll
          for (int i = 0; i < 4; ++i) wv[i] = acc[i] * (at * bs[i * TS / 4]);
        }
      } else {
        const float gam_t = SC[SB_::GAM + tqt];
        int tq_m = tqt;
        __asm__ volatile("" : "+v"(tq_m));
        if constexpr (R == 1) {
          const f4 c4 = *reinterpret_cast<const f4*>(SC + SB_::CUM + 16 * sj + 4 * lg);
          const f4 s4 = *reinterpret_cast<const f4*>(SC + SB_::SCL + 16 * sj + 4 * lg);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int ts = 16 * sj + 4 * lg + i;
            const float lower = s4[i] * __expf(cum_t - c4[i]);
            const float d = tq_m > ts ? lower : (tq_m == ts ? gam_t : 0.f);
            wv[i] = acc[i] * d;
          }
        } else {
          // same token (every rank pair): gamma; an earlier token: the decayed scale
          float d[TS];
#pragma unroll
          for (int j = 0; j < TS; ++j) {
            const int ts = (16 * sj + 4 * lg) / R + j;
            const float lower = SC[SB_::SCL + ts] * __expf(cum_t - SC[SB_::CUM + ts]);
            d[j] = tq_m > ts ? lower : (tq_m == ts ? gam_t : 0.f);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) wv[i] = acc[i] * d[i * TS / 4];
        }
      }
      // W[t][s], s = 16 sj + 4 lg + i, at s' = 32 (sj / 2) + 8 lg + 4 (sj % 2) + i: the order of
      // the intra product's K axis (below)
      const int wo = tq * LW + 32 * (sj >> 1) + 8 * lg + 4 * (sj & 1);
      st_quad<T>(WS + wo, wv);
      if constexpr (LO) st_quad<T>(WL + wo, low(wv));
    }
  };
  auto carry = [&] {
    {
      // carry: S^T(ni, pj) += K~^T V~ over the 64 tokens. A: 8 tokens of column n from the
      // row-major Ks by two transposing reads (in each 16-lane group, lane 4a + b receives
      // element b of the 8-byte vectors of lanes a, a + 4, a + 8, a + 12); B: the same from VS.
      // The K axis of k-step kk, lane group lg: tokens kk + 4 lg + j (slots j) and
      // kk + 16 + 4 lg + j (slots 4 + j), so the 32 lanes of each read take 8 consecutive tokens
      const int xr = l16 >> 2, xc = 4 * (l16 & 3);
      f4 sl[2] = {zero4(), zero4()};
#pragma unroll
      for (int kk = 0; kk < 64; kk += 32) {  // the 64 rows
        const int r0 = kk + 4 * lg + xr;
        const T* k0 = Ks + r0 * LQ + 16 * sni + xc;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)(k0));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)(k0 + 16 * LQ));
        const typename M::v8 av = __builtin_bit_cast(
            typename M::v8, (i16x8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int vc = 16 * (spj0 + k) + xc;
          auto rows8 = [&](const T* v) {
            const i16x4 vlo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) i16x4*)(v + v_off(r0, vc)));
            const i16x4 vhi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) i16x4*)(v + v_off(r0 + 16, vc)));
            return __builtin_bit_cast(
                typename M::v8,
                (i16x8){vlo[0], vlo[1], vlo[2], vlo[3], vhi[0], vhi[1], vhi[2], vhi[3]});
          };
          st[k] = M::mma(av, rows8(VS), st[k]);
          if constexpr (LO) (LOA ? sl[k] : st[k]) = M::mma(av, rows8(VL), LOA ? sl[k] : st[k]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (LOA) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
#pragma unroll
          for (int i = 0; i < 4; ++i) st[k][i] = fmaf(sl[k][i], 1.f / kLo, st[k][i]);
        }
      }
    }
  };
  // output tile (row tile it, P tile pj) of the sub-chunk at token t0
  auto output = [&](int t0, const T* Qc, const float* SC) {
    if constexpr (!SO) {
      const int it = w >> 2, pj = w & 3;
      const int tq = 16 * it + l16;
      f4 yi = zero4(), ye = zero4(), yl = zero4();
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if (2 * m > it) continue;
        // intra: V^T W^T over tokens s = 32 m + 4 lg + i and 32 m + 16 + 4 lg + i
        const int vrow = 32 * m + 4 * lg + (l16 >> 2), vcol = 16 * pj + 4 * (l16 & 3);
        const typename M::v4 b0 = __builtin_bit_cast(
            typename M::v4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                (__attribute__((address_space(3))) i16x4*)(VR + v_off(vrow, vcol))));
        const typename M::v4 b1 = __builtin_bit_cast(
            typename M::v4,
            __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) i16x4*)(VR + v_off(vrow + 16, vcol))));
        typename M::v8 av, bv = *reinterpret_cast<const typename M::v8*>(WS + tq * LW + 32 * m + 8 * lg);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          av[i] = b0[i];
          av[4 + i] = b1[i];
        }
        auto causal = [&](typename M::v8 x) {
          if (2 * m + 1 > it) {
            // column tile 2m + 1 lies above it: the operand's upper half (two words) is zero
            // (element-wise 16-bit zeroing took a select and a permute per element)
            u32x4 bw = __builtin_bit_cast(u32x4, x);
            bw[2] = 0u;
            bw[3] = 0u;
            x = __builtin_bit_cast(typename M::v8, bw);
          }
          return x;
        };
        bv = causal(bv);
        yi = M::mma(av, bv, yi);
        if constexpr (LO) {
          const typename M::v8 bl =
              *reinterpret_cast<const typename M::v8*>(WL + tq * LW + 32 * m + 8 * lg);
          (LOA ? yl : yi) = M::mma(av, causal(bl), LOA ? yl : yi);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (LOA) {
#pragma unroll
        for (int i = 0; i < 4; ++i) yi[i] = fmaf(yl[i], 1.f / kLo, yi[i]);
      }
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        // inter: rnd(S) Q^T
        const typename M::v8 av = *reinterpret_cast<const typename M::v8*>(
            Sb + sb_off(16 * pj + l16, 32 * kk + 8 * lg));
        const typename M::v8 bv =
            *reinterpret_cast<const typename M::v8*>(Qc + tq * LQ + 32 * kk + 8 * lg);
        ye = M::mma(av, bv, ye);
        __builtin_amdgcn_sched_barrier(0);
      }
      // epilogue: row tq (token tq / R), columns pb .. pb+3
      const int pb = 16 * pj + 4 * lg, tqt = tq / R;
      const float ecum_t = __expf(SC[SB_::CUM + tqt]);
      const typename M::v4 v4 = *reinterpret_cast<const typename M::v4*>(VR + v_off(tq, pb));
      typename M::v4 z4;
      f4 sz;
      if constexpr (!Ly::ZF32) {
        z4 = *reinterpret_cast<const typename M::v4*>(ZR + v_off(tq, pb));
      } else {
        sz = *reinterpret_cast<const f4*>(ZF + z_off(tq, pb));
      }
      f4 y;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float gate = Ly::ZF32 ? sz[i] : silu_fast(to_f(z4[i]));
        y[i] = (fmaf(ye[i], ecum_t, yi[i]) + Dh * to_f(v4[i])) * gate;
      }
      if constexpr (R > 1) {
        // times mimo_out of the row's rank, summed over the token's R rows, consecutive lanes
        // of the 16-lane group: DPP quad permutes (lane ^ 1, lane ^ 2) and a swizzle (lane ^ 4)
        const f4 mo = *reinterpret_cast<const f4*>(F_ + Ly::MO + (tq & (R - 1)) * kPPad + pb);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float t = y[i] * mo[i];
          t += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                                             0, __builtin_bit_cast(int, t), 0xb1, 0xf, 0xf, false));
          if constexpr (R >= 4) {
            t += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                                               0, __builtin_bit_cast(int, t), 0x4e, 0xf, 0xf, false));
          }
          if constexpr (R >= 8) {
            t += __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, t),
                                                                       0x101f));
          }
          y[i] = t;
        }
      }
      if ((R == 1 || (tq & (R - 1)) == 0) && (F == kModel || pb < P)) {
        bstore_quad<T>(y, go.rs, (tqt * go.step + go.o0 + pb * ES) +
                                     __builtin_amdgcn_readfirstlane(t0 * go.step));
      }
    }
  };
  auto pin = [] { __builtin_amdgcn_sched_barrier(0); };

  if constexpr (R == 1) {
    // three intervals per sub-chunk
    __syncthreads();
    for (int c = 0; c < nsub; ++c) {
      const int t0 = c * TOK;
      const float* SC = F_ + sc0;
      if (c + 1 < nsub) put_side(sc1);
      stage_qk(0, cst(c));
      stage_vs(SC);
      stage_out();
      decay_state(SC);
      __syncthreads();
      pin();
      load_qk(t0 + TOK);
      pin();
      if (w < 10) scores(w, Qs, SC);
      carry();
      pin();
      load_vz(t0 + TOK);
      pin();
      load_side(c + 2);
      pin();
      __syncthreads();
      output(t0, Qs, SC);
      phases(c + 1, sc1);
      __syncthreads();
      const int sct = sc0;
      sc0 = sc1;
      sc1 = sct;
    }
  } else {
    // two intervals per sub-chunk; the first sub-chunk's staging ahead of the loop
    __syncthreads();
    stage_qk(0, cst(0));
    stage_vs(F_ + sc0);
    if (nsub > 1) put_side(sc1);
    load_qk(TOK);
    load_side(2);
    __syncthreads();
    for (int c = 0; c < nsub; ++c) {
      const int t0 = c * TOK;
      const float* SC = F_ + sc0;
      const T* Qc = Qs + (c & 1) * Ly::QB;
      stage_out();
      pin();
      load_vz(t0 + TOK);
      pin();
      decay_state(SC);
      phases(c + 1, sc1);
      if (w < 2 || w >= 8) scores((w - 8) & 15, Qc, SC);  // waves 8-15 and 0, 1
      carry();
      __syncthreads();
      if (c + 1 < nsub) {
        stage_qk(((c + 1) & 1) * Ly::QB, cst(c + 1));
        stage_vs(F_ + sc1);
        if (c + 2 < nsub) put_side(sc2);
      }
      pin();
      load_qk(t0 + 2 * TOK);
      load_side(c + 3);
      pin();
      output(t0, Qc, SC);
      __syncthreads();
      const int sct = sc0;
      sc0 = sc1;
      sc1 = sc2;
      sc2 = sct;
    }
  }

  // ---- final k: the biased, rotated k rows of token L-1, still in Ks from the last sub-chunk
  if (a.final_k.ptr != nullptr && fin) {
    const int tl = (L - 1) - (nsub - 1) * TOK;
    for (int i = tid; i < R * kNPad; i += k16Threads) {
      const int r = i / kNPad, sl = i - r * kNPad;
      if (sl < N) {
        static_cast<T*>(a.final_k.ptr)[bo * a.final_k.stride[0] + h * a.final_k.stride[1] +
                                       r * a.final_k.stride[2] + col(sl)] =
            Ks[(tl * R + r) * LQ + sl];
      }
    }
  }
  if (a.final_decay.ptr != nullptr && tid == 0) {
    static_cast<float*>(a.final_decay.ptr)[bo * a.final_decay.stride[0] +
                                           h * a.final_decay.stride[1]] = log_decay;
  }
  if (a.block_phase.ptr != nullptr) {
    for (int i = tid; i < S; i += k16Threads) {
      static_cast<float*>(a.block_phase.ptr)[b * a.block_phase.stride[0] +
                                             h * a.block_phase.stride[1] +
                                             ((tok0 + L - 1) >> 6) * a.block_phase.stride[2] +
                                             i * a.block_phase.stride[3]] = F_[Ly::PBASE + i];
    }
  }
  if (fin) {
    const __amdgpu_buffer_rsrc_t rs = state_rs(a.final_state, bo);
    const int sp = static_cast<int>(a.final_state.stride[2]);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(st[k][i]), rs, state_off(k, i, sp), 0,
                                              0);
      }
    }
  }
}

template <typename T, int R, Form16 F, bool SO, bool LO>
static int launch_one16(const m3_scan_args& a, const ScanGeom& g, const float* prep,
                        unsigned grid, hipStream_t stream) {
  constexpr int kBytes = Lay16<R, LO>::BYTES;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(&scan16_kernel<T, R, F, SO, LO>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kBytes);
    if (e != hipSuccess) {
      return fail(M3_ELAUNCH, "m3_scan_fwd: hipFuncSetAttribute: %s", hipGetErrorString(e));
    }
    attr_set = true;
  }
  hipLaunchKernelGGL((scan16_kernel<T, R, F, SO, LO>), dim3(grid), dim3(k16Threads), kBytes,
                     stream, a, g, prep);
  return check_launch("m3_scan_fwd");
}

template <typename T, int R, Form16 F>
static int launch_form16(const m3_scan_args& a, const ScanGeom& g, const float* prep, bool so,
                         unsigned grid, hipStream_t stream) {
  if constexpr (F != kModel) {
    if (g.lo) {
      return so ? launch_one16<T, R, F, true, true>(a, g, prep, grid, stream)
                : launch_one16<T, R, F, false, true>(a, g, prep, grid, stream);
    }
  }
  return so ? launch_one16<T, R, F, true, false>(a, g, prep, grid, stream)
            : launch_one16<T, R, F, false, false>(a, g, prep, grid, stream);
}

template <typename T, int R>
static int launch_rank16(const m3_scan_args& a, const ScanGeom& g, const float* prep, bool so,
                         unsigned grid, hipStream_t stream) {
  if constexpr (R == 1 || R == 4) {
    if (g.form16 == kModel) return launch_form16<T, R, kModel>(a, g, prep, so, grid, stream);
  }
  if constexpr (R > 1) {
    if (g.form16 == kRows) return launch_form16<T, R, kRows>(a, g, prep, so, grid, stream);
    if (g.form16 == kCopy) return launch_form16<T, R, kCopy>(a, g, prep, so, grid, stream);
  }
  if (g.form16 == kProj) return launch_form16<T, R, kProj>(a, g, prep, so, grid, stream);
  return launch_form16<T, R, kHook>(a, g, prep, so, grid, stream);
}

// One instantiation per activation type (scan16_bf16.hip, scan16_f16.hip).
template <typename T>
int launch_scan16(const m3_scan_args& a, const ScanGeom& g, const float* prep, bool state_only,
                  hipStream_t stream) {
  const unsigned grid = static_cast<unsigned>(a.batch) * g.segs * a.heads;
  switch (a.rank) {
    case 1: return launch_rank16<T, 1>(a, g, prep, state_only, grid, stream);
    case 2: return launch_rank16<T, 2>(a, g, prep, state_only, grid, stream);
    case 4: return launch_rank16<T, 4>(a, g, prep, state_only, grid, stream);
    default: return launch_rank16<T, 8>(a, g, prep, state_only, grid, stream);
  }
}

}  // namespace m3
