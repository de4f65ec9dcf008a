// Chunked Mamba-3 SSD for CDNA4 (gfx950).
//
// Two launches per call:
//   prep_kernel  head-independent per-token work, once per token instead of once per head:
//                the RMSNorm factors of the raw B / C rows (model.py:190-191) and
//                pi * tanh(angle) of the phase increments (model.py:225-228), into a workspace.
//   scan16_kernel (scan16_kernel.hpp) the 16-bit calls whose rows can be read as vectors;
//   scan_kernel  the others. One persistent workgroup per (batch, head) walks the sequence in
//                sub-chunks of ROWS flattened (token, rank) rows. The FP32 state lives in MFMA
//                accumulator registers for the whole sequence (stored transposed, S^T [N, P],
//                as 16x16 tiles spread over the waves), so the per-chunk state update that the
//                reference launches once per chunk (_triton.py:294-413 from ops.py:444-504) is
//                fused and the state never round-trips through HBM.
//
// Per sub-chunk of scan_kernel (the global loads of sub-chunk c+1 are issued into registers
// before the MFMA work of sub-chunk c, so their latency hides behind it):
//   scalars  dt, adt, trap from the raw projection or given (model.py:195-198), the
//            exp-trapezoid gamma and scale (ops.py:659-671), within-chunk cumsum of adt.
//   phase    bounded phase (model.py:215-256): 64-token blocks of fmod-reduced increments with
//            an fmod-reduced carry, 4 tokens per lane plus a cross-lane scan; cos / sin.
//   q / k    RMSNorm, head bias, rotation (ops.py:35-84, 700-714) -> Q, K (row-major) and K^T.
//   v / z    rank values v * mimo_x, z * mimo_z, and v * scale * end_decay -> V^T, Vs^T, Z^T.
//   scores   Sc^T = K Q^T                                  (MFMA, FP32 accumulate) ops.py:763
//   weights  W = rnd(Sc * d), d[t,s] = scale_s exp(cum_t - cum_s) for s < t, gamma_t at s = t:
//            the reference's K * scale and diagonal gamma / scale fold (ops.py:743, 770-787).
//   intra    W V   (W stays in registers: the K axis is permuted alike in both operands)
//   inter    Q rnd(S)^T * exp(cum)                                               ops.py:753
//   epilogue (inter + intra + D v) silu(z), MIMO rank sum                    ops.py:792-802
//   carry    S^T = exp(cum_last) S^T + K^T Vs                                ops.py:806-816
//
// Products and sums are evaluated in FP32 and rounded to the activation dtype once, where the
// data become MFMA operands; the reference rounds some intermediates (bias add, rotation,
// k * scale) separately in the activation dtype.
//
// Replaces ops._fused_chunk_scan (ops.py:253-367) / its driver (ops.py:370-505) and the Triton
// kernels _chunk_main_kernel (_triton.py:74-291) and _chunk_state_kernel (_triton.py:294-413);
// the same kernel serves the portable entry ops.mamba3_scan (ops.py:544-822).
#include "scan_common.hpp"

#include <algorithm>

namespace m3 {

// Global reads of one (batch, head). Per sub-chunk: the q / k and value / gate words of each
// lane's rows, and the side data the block stages through LDS: its scalar block followed by the
// RMSNorm factors of its rows (SIDE floats, one 8-byte word per lane) and its angle tile (4
// consecutive tokens of one angle per 16-byte word, TOK * S floats). FULL: every per-token input
// is a slice of one projection row (host-checked), read at per-lane byte offsets through one
// buffer resource per batch row whose extent ends at token L, so rows of tokens >= L read as
// zero without guards; the workspace likewise through one resource. BUF (the model's shape with
// the generic inputs, host-checked): the same guard-free reads through one resource per input
// tensor and (batch, head), whose extent ends at token L, at 32-bit per-lane offsets. Otherwise
// element pointers with explicit guards.
template <typename T, int R, bool FULL, bool BUF = false>
struct Feed {
  static constexpr int ES = sizeof(T), W8 = Words<T>::W8, W4 = Words<T>::W4;
  static constexpr int ROWS = Mma<T>::ROWS, TOK = ROWS / R;
  static constexpr int VJ = R == 1 ? 2 : 1;  // value / gate tokens per lane
  static constexpr int kPast = 0x7f000000;   // beyond the workspace (below 2^30 bytes there)
  // FULL
  __amdgpu_buffer_rsrc_t rs_p, rs_w;
  int o_qk, o_vz, d_q1, d_k, d_z, tok_b;  // per-lane byte offsets at token 0, uniform deltas
  int side_o, side_s, ang_o, ang_s;        // per-lane workspace byte offsets at sub-chunk 0, strides
  // BUF: resources of q, k, value, gate and the given phases; per-lane byte offsets at token 0,
  // the byte strides of a token and the second row's delta
  __amdgpu_buffer_rsrc_t rs_q, rs_k, rs_v, rs_z, rs_x;
  int o_q, o_k, o_v, o_z, o_x, tq_b, tk_b, tv_b, tz_b, tx_b, d_q2, d_k2;
  // generic
  const T *q_row, *k_row, *v_row, *z_row;
  const float *side_p, *ang_p;  // this lane's side / angle word at sub-chunk 0 (null: none)
  const float* ph_row;          // given phases of (b, h): [L][S] with strides ph_t, ph_s
  int64_t side_ps, ang_ps;      // per-sub-chunk strides (floats)
  int q_t, q_r, k_t, k_r, v_t, z_t, ph_t, ph_s, qk_n, vz_n;
  int side_tok, side_lim;       // norm words: token of the word (sub-chunk 0), last valid
  int ang_grp;                  // angle words: 4-token group of the word (sub-chunk 0)
  bool vec_qk, vec_vz, given;
  int rp, vp, nsub, L, S, L4;

  __device__ __forceinline__ void init(const m3_scan_args& a, const ScanGeom& g,
                                       const float* prep, int b, int h, int grp, int rp_,
                                       int n0, int vp_, int p0, int N, int P, bool norm) {
    L = a.length;
    S = a.num_angles;
    L4 = g.L4;
    rp = rp_;
    vp = vp_;
    nsub = g.nsub;
    const int GR = a.groups * a.rank, H = a.heads, tid = threadIdx.x;
    const int tt0 = (2 * rp) / R, r0 = (2 * rp) % R;
    const int scw = g.scw;
    // side word of this lane: floats 2 tid, 2 tid + 1 of [scalar block (scw) | norms (2 ROWS)]
    const int q2 = 2 * tid;
    const int64_t sc0 = g.ws_sc + static_cast<int64_t>(b * H + h) * nsub * scw + q2;
    const int nrow = (q2 - scw) >> 1;  // norm word: row of the sub-chunk (token nrow / R)
    // FULL, BUF: the norm word's token at sub-chunk 0 (other words: none) and the angle word's
    // 4-token group; past the row's end they are not the row's any more and read as zero
    side_tok = q2 >= scw ? nrow / R : INT32_MIN / 2;
    ang_grp = tid / max(S, 1);
    if constexpr (FULL) {
      tok_b = g.tok_b;
      rs_p = make_rsrc(g.proj + b * g.proj_b, L * (tok_b < 0 ? -tok_b : tok_b));
      rs_w = make_rsrc(prep, g.ws_bytes);
      o_qk = g.o_q + grp * g.qk_g + r0 * g.qk_r + tt0 * tok_b + n0 * ES;
      o_vz = g.o_v + h * g.vz_h + (R == 1 ? 2 * vp : (2 * vp) / R) * tok_b + p0 * ES;
      d_q1 = R == 1 ? tok_b : g.qk_r;  // row 2rp + 1: the next token (R = 1) or the next rank
      d_k = g.o_k - g.o_q;
      d_z = g.o_z - g.o_v;
      // groups == 1: the norm pairs of a sub-chunk's rows are 2 ROWS contiguous floats
      if (q2 < scw) {
        side_o = static_cast<int>(sc0) * 4;
        side_s = scw * 4;
      } else if (q2 < scw + 2 * ROWS) {
        side_o = static_cast<int>(g.ws_norm + static_cast<int64_t>(b) * L * GR * 2 + q2 - scw) * 4;
        side_s = TOK * GR * 2 * 4;
      } else {
        side_o = side_s = 0;
      }
      ang_o = static_cast<int>(g.ws_ang + static_cast<int64_t>(b) * g.L4 * S * 4 + 4 * tid) * 4;
      ang_s = (TOK / 4) * S * 16;
    } else if constexpr (BUF) {
      rs_w = make_rsrc(prep, g.ws_bytes);
      // every token stride is positive and a token's row ends below the next token's (host),
      // so rows of tokens >= L lie past the extent L * stride and read as zero
      const char* q0 = static_cast<const char*>(a.q.ptr) + b * a.q.stride[0] * ES;
      const char* k0 = static_cast<const char*>(a.k.ptr) + b * a.k.stride[0] * ES;
      const char* v0 = static_cast<const char*>(a.value.ptr) +
                       (b * a.value.stride[0] + h * a.value.stride[2]) * ES;
      const char* z0 = static_cast<const char*>(a.gate.ptr) +
                       (b * a.gate.stride[0] + h * a.gate.stride[2]) * ES;
      tq_b = static_cast<int>(a.q.stride[1]) * ES;
      tk_b = static_cast<int>(a.k.stride[1]) * ES;
      tv_b = static_cast<int>(a.value.stride[1]) * ES;
      tz_b = static_cast<int>(a.gate.stride[1]) * ES;
      rs_q = make_rsrc(q0, L * tq_b);
      rs_k = make_rsrc(k0, L * tk_b);
      rs_v = make_rsrc(v0, L * tv_b);
      rs_z = make_rsrc(z0, L * tz_b);
      const int qr_b = static_cast<int>(a.q.stride[3]) * ES, kr_b = static_cast<int>(a.k.stride[3]) * ES;
      o_q = tt0 * tq_b + r0 * qr_b + n0 * ES;
      o_k = tt0 * tk_b + r0 * kr_b + n0 * ES;
      d_q2 = R == 1 ? tq_b : qr_b;  // row 2rp + 1: the next token (R = 1) or the next rank
      d_k2 = R == 1 ? tk_b : kr_b;
      const int tv = R == 1 ? 2 * vp : (2 * vp) / R;
      o_v = tv * tv_b + p0 * ES;
      o_z = tv * tz_b + p0 * ES;
      // side and angle words as in the projection form (groups == 1); no norm: unused words
      if (q2 < scw) {
        side_o = static_cast<int>(sc0) * 4;
        side_s = scw * 4;
      } else if (q2 < scw + 2 * ROWS && g.ws_norm >= 0) {
        side_o = static_cast<int>(g.ws_norm + static_cast<int64_t>(b) * L * GR * 2 + q2 - scw) * 4;
        side_s = TOK * GR * 2 * 4;
      } else {
        side_o = side_s = 0;
      }
      ang_o = g.ws_ang >= 0
                  ? static_cast<int>(g.ws_ang + static_cast<int64_t>(b) * g.L4 * S * 4 + 4 * tid) * 4
                  : 0;
      ang_s = (TOK / 4) * S * 16;
      given = a.phase_mode == M3_PHASE_GIVEN;
      if (given) {
        // tile word tid = (group, angle): tokens 4 group .. + 3 of that angle
        const char* x0 = static_cast<const char*>(a.phase.ptr) +
                         (b * a.phase.stride[0] + h * a.phase.stride[2]) * 4;
        tx_b = static_cast<int>(a.phase.stride[1]) * 4;
        rs_x = make_rsrc(x0, L * tx_b);
        const int grp4 = tid / S, sa = tid - grp4 * S;
        o_x = 4 * grp4 * tx_b + sa * static_cast<int>(a.phase.stride[3]) * 4;
      }
    } else {
      q_row = static_cast<const T*>(a.q.ptr) + b * a.q.stride[0] + grp * a.q.stride[2] + n0;
      k_row = static_cast<const T*>(a.k.ptr) + b * a.k.stride[0] + grp * a.k.stride[2] + n0;
      q_t = static_cast<int>(a.q.stride[1]);
      q_r = static_cast<int>(a.q.stride[3]);
      k_t = static_cast<int>(a.k.stride[1]);
      k_r = static_cast<int>(a.k.stride[3]);
      v_row = static_cast<const T*>(a.value.ptr) + b * a.value.stride[0] +
              h * a.value.stride[2] + p0;
      z_row = static_cast<const T*>(a.gate.ptr) + b * a.gate.stride[0] + h * a.gate.stride[2] +
              p0;
      v_t = static_cast<int>(a.value.stride[1]);
      z_t = static_cast<int>(a.gate.stride[1]);
      qk_n = max(0, min(8, N - n0));
      vz_n = max(0, min(4, P - p0));
      vec_qk = g.vec_qk;
      vec_vz = g.vec_vz;
      side_p = nullptr;
      side_tok = 0;
      side_lim = INT32_MAX;
      if (q2 < scw) {
        side_p = prep + sc0;
        side_ps = scw;
      } else if (q2 < scw + 2 * ROWS && norm) {
        // rows are (token, rank); a word holds the (q, k) pair of one row
        const int tr = nrow / R, rr = nrow - tr * R;
        side_p = prep + g.ws_norm + (static_cast<int64_t>(b) * L * GR + tr * GR + grp * R + rr) * 2;
        side_ps = static_cast<int64_t>(TOK) * GR * 2;
        side_tok = tr;
        side_lim = L - 1;
      }
      given = a.phase_mode == M3_PHASE_GIVEN;
      ang_p = nullptr;
      ph_row = nullptr;
      if (a.phase_mode == M3_PHASE_ANGLES && 4 * tid < TOK * S) {
        ang_p = prep + g.ws_ang + static_cast<int64_t>(b) * g.L4 * S * 4 + 4 * tid;
        ang_ps = (TOK / 4) * S * 4;
      } else if (given && 4 * tid < TOK * S) {
        ph_row = static_cast<const float*>(a.phase.ptr) + b * a.phase.stride[0] +
                 h * a.phase.stride[2];
        ph_t = static_cast<int>(a.phase.stride[1]);
        ph_s = static_cast<int>(a.phase.stride[3]);
      }
    }
  }

  // q / k rows 2rp, 2rp+1 and the value / gate of rows 2vp, 2vp+1 of the sub-chunk at token t0
  // (nw valid tokens): tokens 2vp, 2vp+1 for R = 1, else token 2vp / R (both rows' ranks)
  __device__ __forceinline__ void words(int t0, int nw, bool qk_on, bool vz_on,
                                        uint32_t (&rq)[2][W8], uint32_t (&rk)[2][W8],
                                        uint32_t (&rv)[2][W4], uint32_t (&rz)[2][W4]) const {
    words_qk(t0, nw, qk_on, rq, rk);
    words_vz(t0, nw, vz_on, rv, rz);
  }

  __device__ __forceinline__ void words_qk(int t0, int nw, bool qk_on, uint32_t (&rq)[2][W8],
                                           uint32_t (&rk)[2][W8]) const {
    if constexpr (FULL) {
      // unconditional, also for lanes without a q/k or v/z role: every offset stays inside a
      // buffer or past its extent, where the load returns zero
      const int tb = t0 * tok_b;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        bload_words<W8>(rq[j], rs_p, o_qk + tb + j * d_q1);
        bload_words<W8>(rk[j], rs_p, o_qk + tb + j * d_q1 + d_k);
      }
    } else if constexpr (BUF) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        bload_words<W8>(rq[j], rs_q, o_q + t0 * tq_b + j * d_q2);
        bload_words<W8>(rk[j], rs_k, o_k + t0 * tk_b + j * d_k2);
      }
    } else {
      if (qk_on) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int row = 2 * rp + j, tt = row / R, r = row - tt * R;
          const bool ok = tt < nw;
          const int tg = t0 + tt;
          load_words<T, 8>(rq[j], q_row + tg * q_t + r * q_r, ok ? qk_n : 0, vec_qk);
          load_words<T, 8>(rk[j], k_row + tg * k_t + r * k_r, ok ? qk_n : 0, vec_qk);
        }
      }
    }
  }

  __device__ __forceinline__ void words_vz(int t0, int nw, bool vz_on, uint32_t (&rv)[2][W4],
                                           uint32_t (&rz)[2][W4]) const {
    if constexpr (FULL) {
      const int tb = t0 * tok_b;
#pragma unroll
      for (int j = 0; j < VJ; ++j) {
        bload_words<W4>(rv[j], rs_p, o_vz + tb + j * tok_b);
        bload_words<W4>(rz[j], rs_p, o_vz + tb + j * tok_b + d_z);
      }
    } else if constexpr (BUF) {
#pragma unroll
      for (int j = 0; j < VJ; ++j) {
        bload_words<W4>(rv[j], rs_v, o_v + (t0 + j) * tv_b);
        bload_words<W4>(rz[j], rs_z, o_z + (t0 + j) * tz_b);
      }
    } else {
      if (vz_on) {
#pragma unroll
        for (int j = 0; j < VJ; ++j) {
          const int tt = R == 1 ? 2 * vp + j : (2 * vp) / R;
          const bool ok = tt < nw;
          const int tg = t0 + tt;
          load_words<T, 4>(rv[j], v_row + tg * v_t, ok ? vz_n : 0, vec_vz);
          load_words<T, 4>(rz[j], z_row + tg * z_t, ok ? vz_n : 0, vec_vz);
        }
      }
    }
  }

  // this lane's side word of sub-chunk c (FULL: unconditional; unused words read anything)
  __device__ __forceinline__ float2 side_in(int c) const {
    if constexpr (FULL || BUF) {
      const int o = side_tok + c * TOK < L ? side_o + c * side_s : kPast;
      const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs_w, o, 0, 0));
      return make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
    } else {
      float2 v = make_float2(1.f, 1.f);
      if (side_p != nullptr && c < nsub && side_tok + c * TOK <= side_lim) {
        v = *reinterpret_cast<const float2*>(side_p + c * side_ps);
      }
      return v;
    }
  }

  // this lane's angle word of sub-chunk c: in the tile order [TOK/4][S][4], 4-token group
  // tid / S of angle tid % S
  __device__ __forceinline__ float4 ang_in(int c) const {
    if constexpr (BUF) {
      if (given) {
        const int o = o_x + c * TOK * tx_b;
        return make_float4(bload_f32(rs_x, o), bload_f32(rs_x, o + tx_b),
                           bload_f32(rs_x, o + 2 * tx_b), bload_f32(rs_x, o + 3 * tx_b));
      }
    }
    if constexpr (FULL || BUF) {
      const int o = ang_grp + c * (TOK / 4) < L4 ? ang_o + c * ang_s : kPast;
      const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs_w, o, 0, 0));
      return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]),
                         __uint_as_float(v[3]));
    } else {
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (c >= nsub) return v;
      if (ang_p != nullptr) {
        if (c * (TOK / 4) + static_cast<int>(threadIdx.x) / S < L4) {  // groups past L4: none
          v = *reinterpret_cast<const float4*>(ang_p + c * ang_ps);
        }
      } else if (ph_row != nullptr) {
        // tile word tid = (group, angle): tokens 4 group .. + 3 of that angle
        const int tid = threadIdx.x;
        const int grp4 = tid / S, sa = tid - grp4 * S;
        float e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = c * TOK + 4 * grp4 + i;
          e[i] = t < L ? ph_row[static_cast<int64_t>(t) * ph_t + sa * ph_s] : 0.f;
        }
        v = make_float4(e[0], e[1], e[2], e[3]);
      }
      return v;
    }
  }
};

// ------------------------------------------------------------------ prep

// The scalar functions of a call, LO (d_state no power of 2: the calls that came from the recurrent
// scan) that scan's library functions, else the hardware's.
template <bool LO>
__device__ __forceinline__ float exp_x(float x) {
  return LO ? expf(x) : __expf(x);
}
template <bool LO>
__device__ __forceinline__ float sigmoid_x(float x) {
  return LO ? sigmoidf(x) : sigmoid_fast(x);
}
template <bool LO>
__device__ __forceinline__ float silu_x(float x) {
  return LO ? siluf(x) : silu_fast(x);
}
template <bool LO>
__device__ __forceinline__ void dt_adt_x(bool raw, float dt_in, float a_in, float dt_bias, float& dt,
                                         float& adt) {
  if constexpr (LO) {
    dt_adt(raw, dt_in, a_in, dt_bias, dt, adt);
  } else {
    dt_adt_fast(raw, dt_in, a_in, dt_bias, dt, adt);
  }
}

// The scalar block of sub-chunk c of (batch, head) bh (one wave, lane = token): dt, adt, trap
// from the raw projection or given (model.py:195-198), gamma = dt sigmoid(trap), scale = gamma +
// dt' (1 - sigmoid(trap')) of the next token, 0 at the last token (ops.py:659-671) and, `cut`, at
// the last of a segment (the next segment starts with it as its endpoint term), the within-chunk
// cumsum of adt by a wave scan, and the decay products the scan uses.
template <int TOK, int TPT, bool LO>
__device__ __forceinline__ void scalar_block(const m3_scan_args& a, float* __restrict__ o,
                                             int c, int lane, float dt_bias, float dt_in,
                                             float a_in, float tr_in, float dtn_in,
                                             float trn_in, bool cut) {
  using B = ScBlk<TOK>;
  const int L = a.length;
  const int tb = c * TOK, t = tb + lane;
  const int wn = min(TOK, L - tb);
  const bool tv = lane < wn;
  const bool nv = lane < TOK && t + 1 < L && !(cut && lane == TOK - 1);
  const bool raw_dt = a.raw_dt != 0;
  float dt = 0.f, adt = 0.f, tr = 0.f;
  if (tv) {
    dt_adt_x<LO>(raw_dt, dt_in, a_in, dt_bias, dt, adt);
    tr = sigmoid_x<LO>(tr_in);
  }
  // right = dt' (1 - sigmoid(trap')) of the next token: lane + 1's; the last lane's from the
  // token after the sub-chunk (dtn_in, trn_in)
  const float own = dt * (1.f - tr);
  float right = __shfl_down(own, 1);
  if (lane == TOK - 1) {
    float dn, an;
    dt_adt_x<LO>(raw_dt, dtn_in, 0.f, dt_bias, dn, an);
    right = dn * (1.f - sigmoid_x<LO>(trn_in));
  }
  if (!nv) right = 0.f;
  const float gamma = dt * tr;
  const float scale = gamma + right;
  const float cum = wave_incl_scan(LO && adt < kDecayLow ? kDecayLow : adt, lane);
  const float cum_last = readlane_f(cum, wn - 1);
  const float cv = tv ? cum : cum_last;
  // cum at the end of this lane's 16-row tile (TPT tokens), clamped to the last valid token
  float cend;
  if constexpr (TPT == 16) {
    const float e0 = readlane_f(cv, 15), e1 = readlane_f(cv, 31), e2 = readlane_f(cv, 47);
    const float e3 = readlane_f(cv, 63);
    const int q = lane >> 4;
    cend = q == 0 ? e0 : (q == 1 ? e1 : (q == 2 ? e2 : e3));
  } else {
    cend = __shfl(cv, min(lane | (TPT - 1), wn - 1));
  }
  if (lane < TOK) {
    o[B::DTV + lane] = dt;
    o[B::CUM + lane] = cv;
    o[B::SCL + lane] = tv ? scale : 0.f;
    o[B::GAM + lane] = gamma;
    o[B::BSC + lane] = tv ? scale * exp_x<LO>(cend - cv) : 0.f;
    if ((lane & (TPT - 1)) == 0) o[B::CEND + lane / TPT] = cend;
  }
  if constexpr (LO) {
    const float sum = readlane_f(wave_incl_scan(adt, lane), wn - 1);
    if (lane == 0) o[B::DEC] = sum;
  }
  if (lane == 0) {
    o[B::ECL] = exp_x<LO>(cum_last);
    o[B::CL] = cum_last;
  }
}

// The same for sub-chunks of TOK <= 16 tokens, 64 / TOK heads per wave: lane = (head lane / TOK,
// token lane % TOK), `o` the lane's head's block, `live` false for lanes past the last head
// (they compute on a valid head's inputs and store nothing). The arithmetic and its order are
// scalar_block's (a segment's scan is the wave scan's first row), so the blocks are identical.
template <int TOK, int TPT, bool LO>
__device__ __forceinline__ void scalar_block_seg(const m3_scan_args& a, float* __restrict__ o,
                                                 int c, int lane, bool live, float dt_bias,
                                                 float dt_in, float a_in, float tr_in,
                                                 float dtn_in, float trn_in, bool cut) {
  static_assert(TOK <= 16 && (TOK & (TOK - 1)) == 0, "segments of at most 16 lanes");
  using B = ScBlk<TOK>;
  const int L = a.length;
  const int j = lane & (TOK - 1), s0 = lane - j;  // token in the sub-chunk, segment's lane 0
  const int tb = c * TOK, t = tb + j;
  const int wn = min(TOK, L - tb);
  const bool tv = j < wn;
  const bool nv = t + 1 < L && !(cut && j == TOK - 1);
  const bool raw_dt = a.raw_dt != 0;
  float dt = 0.f, adt = 0.f, tr = 0.f;
  if (tv) {
    dt_adt_x<LO>(raw_dt, dt_in, a_in, dt_bias, dt, adt);
    tr = sigmoid_x<LO>(tr_in);
  }
  const float own = dt * (1.f - tr);
  float right = __shfl_down(own, 1);
  if (j == TOK - 1) {
    float dn, an;
    dt_adt_x<LO>(raw_dt, dtn_in, 0.f, dt_bias, dn, an);
    right = dn * (1.f - sigmoid_x<LO>(trn_in));
  }
  if (!nv) right = 0.f;
  const float gamma = dt * tr;
  const float scale = gamma + right;
  const float cum = seg_incl_scan<TOK>(LO && adt < kDecayLow ? kDecayLow : adt, lane);
  const float cum_last = __shfl(cum, s0 + wn - 1);
  const float cv = tv ? cum : cum_last;
  const float cend = __shfl(cv, s0 + min(j | (TPT - 1), wn - 1));
  if constexpr (LO) {
    const float sum = __shfl(seg_incl_scan<TOK>(adt, lane), s0 + wn - 1);
    if (live && j == 0) o[B::DEC] = sum;
  }
  if (live) {
    o[B::DTV + j] = dt;
    o[B::CUM + j] = cv;
    o[B::SCL + j] = tv ? scale : 0.f;
    o[B::GAM + j] = gamma;
    o[B::BSC + j] = tv ? scale * exp_x<LO>(cend - cv) : 0.f;
    if ((j & (TPT - 1)) == 0) o[B::CEND + j / TPT] = cend;
    if (j == 0) {
      o[B::ECL] = exp_x<LO>(cum_last);
      o[B::CL] = cum_last;
    }
  }
}

// Head-independent and per-(head, sub-chunk) work ahead of the scan, three block ranges:
//  [0, nb_norm)  one 16-lane group per norm_rows() raw q / k rows (token, group, rank, q|k), 8
//                elements per lane: each row's RMSNorm factor 1 / sqrt(mean(x^2) + eps)
//                (model.py:190-191), or for the 16-wave scan the finished row in slot order;
//  [.., +nb_ang) one lane per kAngQuads (4-token group, angle) pairs, tokens padded to a multiple
//                of 4: pi * tanh(angle) (model.py:225-228), 0 in the padding;
// The first two give each workgroup several rows' loads in flight: with one round trip per
// workgroup they were bound by workgroup turnover (the scalar blocks' LDS allows 6 workgroups per
// CU). The scalar blocks, the longest workgroups, are dispatched first.
//  [.., +nb_sc)  one workgroup per (batch, sub-chunk, head group): the dt / a / trap of its TOK
//                tokens and the next sub-chunk's first, loaded with consecutive lanes on
//                consecutive heads (32 heads per pass, or 8 in groups that small) into LDS; then one wave per head computes
//                that head's scalar block (sub-chunks of 16 tokens or fewer: one 16- or 8-lane
//                segment per head, 4 or 8 heads per wave).
// q / k rows per 16-lane group of prep_kernel: 16 for the 16-bit single-rank rows (their fewer,
// longer workgroups measured faster at config 2: 37.5 -> 34.8 us per prep), else 8 (16 measured
// slower at rank 4, and FP32 rows would not fit the registers)
template <typename T, int R>
constexpr int norm_rows() {
  return sizeof(T) == 2 && R == 1 ? 16 : 8;
}
constexpr int kAngQuads = 4;  // (4-token group, angle) pairs per lane of prep_kernel

template <typename T, int R, bool LO>
__global__ __launch_bounds__(256) void prep_kernel(const m3_scan_args a, const ScanGeom g,
                                                   float* __restrict__ ws, int nb_norm,
                                                   int nb_ang, int head_groups) {
  // every index below fits 31 bits (checked by the host)
  constexpr int TOK = Mma<T>::ROWS / R, TPT = 16 / R;
  constexpr int kNormRows = norm_rows<T, R>();
  // the longest-running range (scalar blocks) is dispatched first: block ids [0, nb_sc) map to
  // it, the rest to the norm and angle ranges in order
  const int nb_sc = a.batch * g.nsub * head_groups;
  const int tid = threadIdx.x;
  const int blk = static_cast<int>(blockIdx.x) < nb_sc ? static_cast<int>(blockIdx.x) + nb_norm + nb_ang
                                                       : static_cast<int>(blockIdx.x) - nb_sc;
  const int L = a.length, tokens = a.batch * L;
  if (blk < nb_norm) {
    // rows blk * 16 kNormRows + (tid >> 4) + 16 k, k < kNormRows: every row's loads first
    const int gr_n = a.groups * a.rank;
    const int nrows = tokens * gr_n * 2;
    const int l16 = tid & 15, row0 = blk * 16 * kNormRows + (tid >> 4);
    const int N = a.d_state;
    const bool in = 8 * l16 < N;  // lanes past column N load column 0 and count zeros
    // rows_out (the 16-wave scan's forms kModel, kRows and kCopy): the finished rows; lane l16 holds the slots 8 l16 ..
    // 8 l16 + 7 (slot_col) instead of the columns, as two 4-column chunks at ca and cb (a pair's two
    // columns with the MIMO rotation, interleaved below). Form kProj, whose factors alone are
    // written, reads the same chunks where the rows start on 8 bytes only; a chunk past column N
    // counts zeros.
    const bool rows_out = sizeof(T) == 2 && g.ws_qk >= 0;
    const int perm = R > 1 && rows_out ? g.perm : 0;
    const bool pairs = perm && 8 * l16 < 2 * a.num_angles;
    const bool in_b = 8 * l16 + 4 < N;
    const int ca = !in ? 0 : pairs ? 4 * l16 : slot_col(8 * l16, perm, a.num_angles);
    const int cb = !in_b ? 0 : pairs ? 4 * l16 + 2 * a.num_angles
                                     : slot_col(8 * l16 + 4, perm, a.num_angles);
    const bool chunks = sizeof(T) == 2 && g.form16 >= 0 && (perm || !g.vec_qk);
    // Rows (token, group, rank, q | k): a lane's rows row0 + 16 k all have row0's parity, so one
    // tensor (q or k). When 2 gr_n divides 16 they also share its (group, rank), the token
    // advancing by 8 / gr_n per k: the addresses follow from row0's by additions (a division
    // per row and a select per tensor field, unrolled over the rows, were most of this range's
    // instructions). Rows past the end re-read the last batch row's last token.
    const int which = row0 & 1;
    const m3_tensor& xt = which ? a.k : a.q;
    // (the chunks are added to the row's start below)
    const T* xbase = static_cast<const T*>(xt.ptr) + (in && !chunks ? 8 * l16 : 0);
    const int64_t xs0 = xt.stride[0], xs1 = xt.stride[1];
    const bool step_rows = 16 % (2 * gr_n) == 0;
    const int dtok = step_rows ? 8 / gr_n : 0;
    int tk = row0 / (2 * gr_n);
    const int gr = (row0 - tk * 2 * gr_n) >> 1;
    const int gi = gr / a.rank, rk = gr - gi * a.rank;
    const T* xgr = xbase + gi * xt.stride[2] + rk * xt.stride[3];
    int bk = tk / L, tt = tk - bk * L;
    auto row_ptr = [&](int k) -> const T* {
      if (step_rows) {
        if (k > 0) {
          tt += dtok;
          while (tt >= L) {
            tt -= L;
            ++bk;
          }
        }
        const bool live = bk < a.batch;
        return xgr + (live ? bk : a.batch - 1) * xs0 + (live ? tt : L - 1) * xs1;
      }
      const int row = min(row0 + 16 * k, nrows - 1);
      const int tok = row / (2 * gr_n);
      const int rem = row - tok * 2 * gr_n;
      const int g2 = rem >> 1, wh = rem & 1;
      const int g2i = g2 / a.rank, r2 = g2 - g2i * a.rank;
      const int b2 = tok / L, t2 = tok - b2 * L;
      const m3_tensor& x = wh ? a.k : a.q;
      return static_cast<const T*>(x.ptr) + b2 * x.stride[0] + t2 * x.stride[1] +
             g2i * x.stride[2] + r2 * x.stride[3] + (in && !chunks ? 8 * l16 : 0);
    };
    float ss[kNormRows];
    uint32_t w8[kNormRows][Words<T>::W8];
    // the rows' weights for this lane's two chunks, raw, issued with the rows (after the factor
    // stores below they would be a second round trip)
    const bool nw_vec = rows_out && g.vec_nw;
    Raw4 nw_r[2][2] = {};
    if (nw_vec) {
      nw_r[0][0] = ldraw4(a.q_norm_w, ca);
      nw_r[0][1] = ldraw4(a.q_norm_w, cb);
      nw_r[1][0] = ldraw4(a.k_norm_w, ca);
      nw_r[1][1] = ldraw4(a.k_norm_w, cb);
    }
    if (chunks) {
      if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int k = 0; k < kNormRows; ++k) {
          const T* p = row_ptr(k);
          const uint2 x = *reinterpret_cast<const uint2*>(p + ca);
          const uint2 y = *reinterpret_cast<const uint2*>(p + cb);
          w8[k][0] = in ? x.x : 0u;
          w8[k][1] = in ? x.y : 0u;
          w8[k][2] = in_b ? y.x : 0u;
          w8[k][3] = in_b ? y.y : 0u;
        }
#pragma unroll
        for (int k = 0; k < kNormRows; ++k) {
          ss[k] = 0.f;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float v = raw_get<T>(w8[k], i);
            ss[k] = fmaf(v, v, ss[k]);
          }
        }
      }
    } else if (g.vec_qk) {
#pragma unroll
      for (int k = 0; k < kNormRows; ++k) {
        // rows past the end re-read an earlier row; their sums are not stored
        const T* p = row_ptr(k);
#pragma unroll
        for (int j = 0; j < Words<T>::W8; j += 4) {
          const uint4 q = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint32_t*>(p) + j);
          w8[k][j] = in ? q.x : 0u;
          w8[k][j + 1] = in ? q.y : 0u;
          w8[k][j + 2] = in ? q.z : 0u;
          w8[k][j + 3] = in ? q.w : 0u;
        }
      }
#pragma unroll
      for (int k = 0; k < kNormRows; ++k) {
        ss[k] = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float v = raw_get<T>(w8[k], i);
          ss[k] = fmaf(v, v, ss[k]);
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < kNormRows; ++k) {
        const T* p = row_ptr(k);
        ss[k] = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (in && 8 * l16 + i < N) {
            const float v = to_f(p[i]);
            ss[k] = fmaf(v, v, ss[k]);
          }
        }
      }
    }
    float fac[kNormRows];
#pragma unroll
    for (int k = 0; k < kNormRows; ++k) {
      ss[k] = row16_sum(ss[k]);  // the row's 16 lanes
      const int row = row0 + 16 * k;
      fac[k] = 1.f / sqrtf(ss[k] / static_cast<float>(N) + a.norm_eps);
      if (l16 == 0 && row < nrows && !rows_out) ws[g.ws_norm + static_cast<int64_t>(row)] = fac[k];
    }
    if constexpr (sizeof(T) == 2) {
      if (rows_out) {
        // the rows themselves: rnd(x * factor * rnd(w)) (model.py:48-55: F.rms_norm with the weight
        // in the activation dtype, the result in it), in FP32 unrounded (kRows), or x, zeros past
        // column N (kCopy). Rows (token, group, rank, q | k).
        // The lane's tensor's weights (every row of the lane is q, or every row k) are chosen by
        // bit masks on the raw words: a select between two weight arrays by `which` became a
        // dynamically indexed array in scratch memory
        const bool norm = R == 1 || a.q_norm_w.ptr != nullptr;
        float wl[8] = {};
        if (nw_vec) {
          const uint32_t msk = 0u - static_cast<uint32_t>(which);
          const int wdt = which ? a.k_norm_w.dtype : a.q_norm_w.dtype;
#pragma unroll
          for (int h2 = 0; h2 < 2; ++h2) {
            Raw4 r;
#pragma unroll
            for (int j = 0; j < 4; ++j) r.w[j] = (nw_r[0][h2].w[j] & ~msk) | (nw_r[1][h2].w[j] & msk);
            const f4 v4 = decode4(r, wdt);
#pragma unroll
            for (int e = 0; e < 4; ++e) wl[4 * h2 + e] = rnd<T>(v4[e]);
          }
        } else if (norm) {
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int n = (i < 4 ? ca : cb) + (i & 3);  // (a chunk past column N: column 0's)
            const float wq = ldx(a.q_norm_w.ptr, a.q_norm_w.dtype, n * a.q_norm_w.stride[0]);
            const float wk = ldx(a.k_norm_w.ptr, a.k_norm_w.dtype, n * a.k_norm_w.stride[0]);
            wl[i] = rnd<T>(which ? wk : wq);
          }
        }
        char* qk = reinterpret_cast<char*>(ws) + g.ws_qk;
#pragma unroll
        for (int k = 0; k < kNormRows; ++k) {
          const int row = row0 + 16 * k;
          if (row >= nrows) continue;
          float x[8], y[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float v = raw_get<T>(w8[k], i);
            x[i] = norm ? v * fac[k] * wl[i] : v;
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            // a pair's two columns side by side
            y[2 * i] = pairs ? x[i] : x[2 * i];
            y[2 * i + 1] = pairs ? x[4 + i] : x[2 * i + 1];
          }
          if (R > 1 && g.form16 == kRows) {
            float* o = reinterpret_cast<float*>(qk) + static_cast<int64_t>(row) * N + 8 * l16;
            if (in) *reinterpret_cast<f4*>(o) = (f4){y[0], y[1], y[2], y[3]};
            if (in_b) *reinterpret_cast<f4*>(o + 4) = (f4){y[4], y[5], y[6], y[7]};
          } else {
            st_row8<T>(reinterpret_cast<T*>(qk) + static_cast<int64_t>(row) * kNPad + 8 * l16, y);
          }
        }
      }
    }
  } else if (blk < nb_norm + nb_ang) {
    // (b, t4, s) quads blk * 256 kAngQuads + tid + 256 k: the angle s of tokens 4 t4 .. 4 t4 + 3,
    // written as the angle region's 4 consecutive elements (b, t4, s, i); 0 past token L - 1
    const int S = a.num_angles;
    const int nq = a.batch * g.L4 * S;
    const int q0 = (blk - nb_norm) * 256 * kAngQuads + tid;
    RawX raw[kAngQuads][4];
#pragma unroll
    for (int k = 0; k < kAngQuads; ++k) {
      const int quad = min(q0 + 256 * k, nq - 1);
      const int sa = quad % S, bt4 = quad / S;
      const int b = bt4 / g.L4, t4 = bt4 - b * g.L4;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = min(4 * t4 + i, L - 1);
        raw[k][i] = ldraw(a.phase.ptr, a.phase.dtype,
                          b * a.phase.stride[0] + t * a.phase.stride[1] + sa * a.phase.stride[2]);
      }
    }
#pragma unroll
    for (int k = 0; k < kAngQuads; ++k) {
      const int quad = q0 + 256 * k;
      if (quad >= nq) continue;
      const int bt4 = quad / S;
      const int t4 = bt4 - (bt4 / g.L4) * g.L4;
      float4 v;
      float* vv = reinterpret_cast<float*>(&v);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float th = decode(raw[k][i], a.phase.dtype);
        vv[i] = 4 * t4 + i < L ? __fmul_rn(kPi, tanhf(th)) : 0.f;
      }
      *reinterpret_cast<float4*>(ws + g.ws_ang + 4 * static_cast<int64_t>(quad)) = v;
    }
  } else {
    const int hgi = (blk - nb_norm - nb_ang) % head_groups, bc = (blk - nb_norm - nb_ang) / head_groups;
    if (bc >= a.batch * g.nsub) return;  // whole workgroups leave together
    const int b = bc / g.nsub, c = bc - b * g.nsub;
    const bool cut = (c + 1) * TOK % g.seg_len == 0;  // the sub-chunk ends a segment
    const int hpg = (a.heads + head_groups - 1) / head_groups;  // heads of this workgroup
    const int h_end = min(a.heads, (hgi + 1) * hpg);
    constexpr int HG_MAX = 32;
    __shared__ float s_in[3][TOK + 1][HG_MAX + 1];
    __shared__ float s_db[HG_MAX];  // dt_bias of the group's heads
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const char* base_dt = static_cast<const char*>(offx(a.dt.ptr, a.dt.dtype, b * a.dt.stride[0]));
    const char* base_a = static_cast<const char*>(offx(a.a.ptr, a.a.dtype, b * a.a.stride[0]));
    const char* base_tr =
        static_cast<const char*>(offx(a.trap.ptr, a.trap.dtype, b * a.trap.stride[0]));
    const int s1_dt = static_cast<int>(a.dt.stride[1]), s2_dt = static_cast<int>(a.dt.stride[2]);
    const int s1_a = static_cast<int>(a.a.stride[1]), s2_a = static_cast<int>(a.a.stride[2]);
    const int s1_tr = static_cast<int>(a.trap.stride[1]), s2_tr = static_cast<int>(a.trap.stride[2]);
    // the inputs of heads h0 .. h0 + hn - 1, hg at a time, into LDS (the scalar blocks below are one
    // copy of code for both sizes; with one each, and the copies of MIMO rows in rank 1's code, prep
    // took 34.8 us instead of 34.1 at 8 x 8192 tokens of 32 heads, and 40.9 instead of 40.0 at rank 4,
    // 8 x 4096)
    auto stage = [&](auto hg, int h0, int hn) {
      constexpr int HG = decltype(hg)::value, NE = (TOK + 1) * HG, NIT = (NE + 255) / 256;
      // raw loads of every element first (clamped to valid tokens / heads), then decode and store
      RawX rd[NIT], ra[NIT], rt[NIT];
      // dt_bias with the batch (inside the per-head loop below, after its stores, each head's
      // load would be a round trip of its own)
      const RawX rdb = a.raw_dt != 0
                           ? ldraw(a.dt_bias.ptr, a.dt_bias.dtype,
                                   (h0 + min(tid & (HG - 1), hn - 1)) * a.dt_bias.stride[0])
                           : RawX{0u, 0u};
#pragma unroll
      for (int k = 0; k < NIT; ++k) {
        const int e = min(tid + 256 * k, NE - 1);
        const int j = e / HG, hh = e - j * HG;
        const int t = min(c * TOK + j, L - 1), h = h0 + min(hh, hn - 1);
        rd[k] = ldraw(base_dt, a.dt.dtype, t * s1_dt + h * s2_dt);
        ra[k] = ldraw(base_a, a.a.dtype, t * s1_a + h * s2_a);
        rt[k] = ldraw(base_tr, a.trap.dtype, t * s1_tr + h * s2_tr);
      }
#pragma unroll
      for (int k = 0; k < NIT; ++k) {
        const int e = tid + 256 * k;
        if (e < NE) {
          const int j = e / HG, hh = e - j * HG;
          s_in[0][j][hh] = decode(rd[k], a.dt.dtype);
          s_in[1][j][hh] = decode(ra[k], a.a.dtype);
          s_in[2][j][hh] = decode(rt[k], a.trap.dtype);
        }
      }
      if (tid < HG) s_db[tid] = a.raw_dt != 0 ? decode(rdb, a.dt_bias.dtype) : 0.f;
    };
    const int hg = hpg <= 8 ? 8 : HG_MAX;
    for (int h0 = hgi * hpg; h0 < h_end; h0 += hg) {
      const int hn = min(hg, h_end - h0);
      if (hg == 8) {
        stage(std::integral_constant<int, 8>{}, h0, hn);
      } else {
        stage(std::integral_constant<int, HG_MAX>{}, h0, hn);
      }
      __syncthreads();
      if constexpr (TOK <= 16) {
        // 64 / TOK heads per wave (one wave per head would leave most lanes idle)
        constexpr int HPW = 64 / TOK;
        const int j = lane & (TOK - 1);
        for (int hb = w * HPW; hb < hn; hb += 4 * HPW) {
          const int hh = hb + lane / TOK, hc = min(hh, hn - 1);
          scalar_block_seg<TOK, TPT, LO>(
              a, ws + g.ws_sc + (static_cast<int64_t>(b * a.heads + h0 + hc) * g.nsub + c) * g.scw,
              c, lane, hh < hn, s_db[hc], s_in[0][j][hc], s_in[1][j][hc], s_in[2][j][hc],
              s_in[0][TOK][hc], s_in[2][TOK][hc], cut);
        }
      } else {
        for (int hh = w; hh < hn; hh += 4) {
          const int h = h0 + hh, j = min(lane, TOK - 1);
          scalar_block<TOK, TPT, LO>(
              a, ws + g.ws_sc + (static_cast<int64_t>(b * a.heads + h) * g.nsub + c) * g.scw, c,
              lane, s_db[hh], s_in[0][j][hh], s_in[1][j][hh], s_in[2][j][hh], s_in[0][TOK][hh],
              s_in[2][TOK][hh], cut);
        }
      }
      __syncthreads();
    }
  }
}

// FULL and SHAPE are FP32 forms (16-bit calls of those shapes take scan16_kernel). SHAPE: the
// model's shape (N = 128, P = 64, 32 angles when rotating, aligned 16-byte rows) with the generic inputs (the hook form): the dimensions and the vector-load
// choice are compile-time constants, the features stay runtime; every read and the output go
// through buffer resources at per-lane offsets, issued unconditionally as in the FULL form.
//
// SO (state only, FP32): the segmented scan's first pass, which needs the end state, log decay,
// last k and phase block sums but no outputs: the stores of Qs, VR, ZR, Sb and the output are left
// out, and with them (dead code) the q math, the scores, the decay weights, the intra and inter
// products and the epilogue.
// LO (FP32): d_state no power of 2. Those calls came from the recurrent scan and are no further from
// 64 bits than there: its functions (exp_x, sincos_of), the carry's sum taken apart from the state it
// is added to (a matrix instruction rounds at the size of its accumulator four times), and the
// scores' and the inter product's in two halves. Errors of 2 x 500 tokens, hook form, output and
// state: d_state 96 rank 1 recurrent 1.5e-7 and 2.4e-7, without these 1.9e-7 and 1.5e-7, with them
// 1.4e-7 and 1.2e-7; rank 8 1.4e-7 and 2.4e-7, 1.3e-7 and 3.2e-7, 0.9e-7 and 1.4e-7; given phases of
// 10^5 at rank 1 1.8e-7 and 2.5e-7, 3e-4 and 1.5e-3, 1.4e-7 and 1.3e-7. Time, 16 x 2048 tokens, 32
// heads: 985 us without, 1,220 with; 1,367 with eight sums each, whose registers spill (output 1.2e-7).
template <typename T, int R, bool FULL, bool SHAPE = false, bool SO = false, bool LO = false>
__global__ __launch_bounds__(kThreads) void scan_kernel(const m3_scan_args a, const ScanGeom g,
                                                        const float* __restrict__ prep) {
  using M = Mma<T>;
  using Lay = Layout<T>;
  constexpr int ROWS = M::ROWS;
  constexpr int RT = ROWS / 16;        // 16-row tiles per sub-chunk
  constexpr int WPR = kWaves / RT;     // waves sharing one query row tile
  constexpr int TOK = ROWS / R;        // tokens per sub-chunk
  constexpr bool F32 = sizeof(T) == 4;
  static_assert(F32 || !(FULL || SHAPE || SO || LO), "16-bit calls of those forms take scan16_kernel");
  static_assert(!LO || !(FULL || SHAPE), "the model's d_state is a power of 2");
  constexpr int ES = sizeof(T);
  constexpr int LQ = Lay::LQ, LR = Lay::LR, LP = Lay::LP, NP = kNPad, CST = Lay::CST;
  using SB_ = ScBlk<TOK>;
  constexpr int TPL = 4;               // tokens per phase lane
  constexpr int PG = TOK / TPL;        // phase lanes per angle
  // swizzle keys of the FP32 transposed tiles, n >> KSH for KT and p >> VSH for VT
  constexpr int KSH = F32 ? 3 : 4, VSH = F32 ? 2 : 4;
  // 16-bit: no transposed copies. The carry reads K~^T from the row-major Ks and V from the
  // row-major VS (the rank values with each token's scale * end decay, in KT's place), the
  // intra product V^T from VR, all through transposing LDS reads
  constexpr bool KTR = !F32;
  // FULL: the model's shape (N = 128, P = 64, S = 32) in projection form with vector loads
  constexpr bool FIX = FULL || SHAPE;  // the model's shape, fixed at compile time
  const int N = FIX ? kNPad : a.d_state;
  const int P = FIX ? kPPad : a.head_dim;
  const int S = FIX ? kSMax : a.num_angles;
  const bool norm = FULL || g.ws_norm >= 0;
  const bool bias = FULL || a.q_bias.ptr != nullptr;
  const bool rotate = FULL || a.phase_mode != M3_PHASE_NONE;
  const bool angles = FULL || a.phase_mode == M3_PHASE_ANGLES;
  const bool raw_dt = FULL || a.raw_dt != 0;
  const bool mimo_rot = FULL ? (R > 1) : (a.mimo_rotation != 0);
  const int H = a.heads;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave index (wave-uniform)
  const int l16 = lane & 15, lg = lane >> 4;

  // ---- block -> (b, h): with xcd_map the blocks of one XCD (blockIdx % 8) take consecutive
  // (b, h), so the heads of one batch row share that XCD's L2 for q, k and the angles.
  int bid = blockIdx.x;
  if (g.xcd_map) {
    const int per = gridDim.x >> 3;
    bid = (bid & 7) * per + (bid >> 3);
  }
  // segment sgi of batch row b (one unless the call is split): tokens tok0 .. tok0 + L - 1, the
  // row's sub-chunks c0 .. c0 + nsub - 1
  const int bs = bid / H, h = bid - bs * H;
  const int b = g.segs > 1 ? bs / g.segs : bs, sgi = bs - b * g.segs;
  const int tok0 = sgi * g.seg_len, c0 = tok0 / TOK;
  const int L = min(g.seg_len, a.length - tok0);
  const int nsub = (L + TOK - 1) / TOK;
  const bool fin = !g.last_only || sgi == g.segs - 1;
  const int bo = g.last_only ? b : bs;
  const int grp = h / (H / a.groups);

  extern __shared__ __attribute__((aligned(16))) char smem[];
  T* Qs = lds_t<T>(smem, Lay::QS);
  T* Ks = lds_t<T>(smem, Lay::KS);
  T* KT = lds_t<T>(smem, Lay::KT);  // FP32: [n][row] K~, transposed and scaled (carry)
  T* VS = KT;                        // 16-bit: [row][p] rank values scaled per token (carry)
  T* VT = lds_t<T>(smem, Lay::VT);  // FP32: [p][row] rank values v mx_r, transposed
  T* VR = lds_t<T>(smem, Lay::VR);  // [row][p] the same, row-major (epilogue D v)
  T* ZR = lds_t<T>(smem, Lay::ZR);  // [row][p] rank gates z mz_r, row-major (epilogue)
  T* Sb = lds_t<T>(smem, Lay::SB);
  float* F = lds_t<float>(smem, Lay::FB);
  const float Dh = ldx(a.D.ptr, a.D.dtype, h * a.D.stride[0]);

  // ---- lane roles
  // q / k: row pair rp (rows 2rp, 2rp+1), columns n0 .. n0+7
  const int rp = tid >> 4, n0 = 8 * (tid & 15);
  const bool qk_on = rp < ROWS / 2 && n0 < N;
  // v / z: row pair vp (rows 2vp, 2vp+1; tokens 2vp, 2vp+1 for R = 1), columns p0 .. p0+3
  // (FP32's 32 rows are 256 lanes' work each: q / k on waves 0-3, value / gate on waves 4-7)
  constexpr int P4 = kPPad / 4;
  const int vp = (F32 ? tid ^ 256 : tid) / P4, p0 = 4 * (tid % P4);
  const bool vz_on = 2 * vp < TOK * R && p0 < P;
  // phase: angle ps, token group pg (tokens TPL pg .. TPL pg + TPL-1)
  const int pg = tid % PG, ps = tid / PG;
  const bool ph_on = rotate && ps < S;

  // ---- one-time LDS setup: zero the operand regions (padding), MIMO parameters, phase carry
  for (int i = tid; i < Lay::FB / 4; i += kThreads) reinterpret_cast<uint32_t*>(smem)[i] = 0u;
  for (int i = tid; i < R * P; i += kThreads) {
    const int r = i / P, p = i - r * P;
    const int o = r * kPPad + p;
    if (R > 1) {
      F[Lay::MX + o] = rnd<T>(ldx(a.mimo_x.ptr, a.mimo_x.dtype,
                                  h * a.mimo_x.stride[0] + r * a.mimo_x.stride[1] + p));
      F[Lay::MZ + o] = rnd<T>(ldx(a.mimo_z.ptr, a.mimo_z.dtype,
                                  h * a.mimo_z.stride[0] + r * a.mimo_z.stride[1] + p));
      F[Lay::MO + o] = ldx(a.mimo_out.ptr, a.mimo_out.dtype,
                           h * a.mimo_out.stride[0] + r * a.mimo_out.stride[1] + p);
    } else {
      F[Lay::MX + o] = 1.f;
      F[Lay::MZ + o] = 1.f;
      F[Lay::MO + o] = 1.f;
    }
  }
  for (int s = tid; s < S; s += kThreads) {
    F[Lay::PBASE + s] = 0.f;
    F[Lay::POFF + s] = a.initial_phase.ptr != nullptr
                           ? static_cast<const float*>(a.initial_phase.ptr)
                                 [bs * a.initial_phase.stride[0] + h * a.initial_phase.stride[1] +
                                  s * a.initial_phase.stride[2]]
                           : 0.f;
  }

  // per-lane constants of the value / gate role (R > 1): the rounded mimo_x / mimo_z of its rows
  // ranks, (2 vp) % R and the next, at columns p0 .. p0+3, read once here instead of from LDS
  // in every sub-chunk
  float mxl[2][4], mzl[2][4];
#pragma unroll
  for (int jr = 0; jr < 2; ++jr) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = (2 * vp + jr) % R, p = min(p0 + i, P - 1);
      mxl[jr][i] = R > 1 ? rnd<T>(ldx(a.mimo_x.ptr, a.mimo_x.dtype,
                                      h * a.mimo_x.stride[0] + r * a.mimo_x.stride[1] + p))
                         : 1.f;
      mzl[jr][i] = R > 1 ? rnd<T>(ldx(a.mimo_z.ptr, a.mimo_z.dtype,
                                      h * a.mimo_z.stride[0] + r * a.mimo_z.stride[1] + p))
                         : 1.f;
    }
  }

  // per-lane constants of the q / k role: rounded norm weights and the biases of its rows
  // (rows 2rp, 2rp+1 have ranks (2rp) % R, (2rp+1) % R: one set suffices when R == 1)
  constexpr int NB = R == 1 ? 1 : 2;
  float wq[8], wk[8], bq[NB][8], bk[NB][8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int n = n0 + i;
    const bool ok = qk_on && n < N;
    wq[i] = (ok && norm) ? rnd<T>(ldx(a.q_norm_w.ptr, a.q_norm_w.dtype, n * a.q_norm_w.stride[0]))
                         : 1.f;
    wk[i] = (ok && norm) ? rnd<T>(ldx(a.k_norm_w.ptr, a.k_norm_w.dtype, n * a.k_norm_w.stride[0]))
                         : 1.f;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int r = (2 * rp + j) % R;
      bq[j][i] = (ok && bias) ? rnd<T>(ldx(a.q_bias.ptr, a.q_bias.dtype,
                                           h * a.q_bias.stride[0] + r * a.q_bias.stride[1] + n))
                              : 0.f;
      bk[j][i] = (ok && bias) ? rnd<T>(ldx(a.k_bias.ptr, a.k_bias.dtype,
                                           h * a.k_bias.stride[0] + r * a.k_bias.stride[1] + n))
                              : 0.f;
    }
  }

  // ---- the state: S^T tiles (ni, pj), tile u = w + 8k; lane holds n = 16 ni + 4 lg + i,
  // p = 16 pj + l16.
  constexpr int n_tiles = kNT * kPT;
  static_assert(n_tiles <= kWaves * kTiles, "state tiles exceed the waves' share");
  constexpr bool all_tiles = n_tiles == kWaves * kTiles;  // every (wave, k) holds a tile
  f4 st[kTiles];
#pragma unroll
  for (int k = 0; k < kTiles; ++k) {
    st[k] = zero4();
    const int u = w + kWaves * k;
    if (u < n_tiles && a.initial_state.ptr != nullptr) {
      const int ni = u / kPT, pj = u - ni * kPT;
      const int p = 16 * pj + l16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = 16 * ni + 4 * lg + i;
        if (p < P && n < N) {
          st[k][i] = static_cast<const float*>(a.initial_state.ptr)
              [bs * a.initial_state.stride[0] + h * a.initial_state.stride[1] +
               p * a.initial_state.stride[2] + n];
        }
      }
    }
  }
  // Endpoint continuation (ops.py:681-686): S += dt_0 (1 - trap_0) sum_r (v_prev mx_r) k_prev_r.
  if (a.initial_k.ptr != nullptr && L > 0) {
    float dt0, adt0;
    dt_adt(raw_dt,
           ldx(a.dt.ptr, a.dt.dtype,
               b * a.dt.stride[0] + tok0 * a.dt.stride[1] + h * a.dt.stride[2]),
           ldx(a.a.ptr, a.a.dtype, b * a.a.stride[0] + tok0 * a.a.stride[1] + h * a.a.stride[2]),
           raw_dt ? ldx(a.dt_bias.ptr, a.dt_bias.dtype, h * a.dt_bias.stride[0]) : 0.f, dt0,
           adt0);
    const float tr0 = sigmoidf(ldx(a.trap.ptr, a.trap.dtype,
                                   b * a.trap.stride[0] + tok0 * a.trap.stride[1] +
                                       h * a.trap.stride[2]));
    const float ce = dt0 * (1.f - tr0);
#pragma unroll
    for (int k = 0; k < kTiles; ++k) {
      const int u = w + kWaves * k;
      if (u >= n_tiles) continue;
      const int ni = u / kPT, pj = u - ni * kPT;
      const int p = 16 * pj + l16;
      if (p >= P) continue;
      const float v0 = to_f(static_cast<const T*>(a.initial_value.ptr)
                                [bs * a.initial_value.stride[0] + h * a.initial_value.stride[1] + p]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = 16 * ni + 4 * lg + i;
        if (n >= N) continue;
        float outer = 0.f;
        for (int r = 0; r < R; ++r) {
          const float pv = R > 1 ? mul_r<T>(v0, rnd<T>(ldx(a.mimo_x.ptr, a.mimo_x.dtype,
                                                             h * a.mimo_x.stride[0] +
                                                                 r * a.mimo_x.stride[1] + p)))
                                 : v0;
          const float k0 = to_f(static_cast<const T*>(a.initial_k.ptr)
                                    [bs * a.initial_k.stride[0] + h * a.initial_k.stride[1] +
                                     r * a.initial_k.stride[2] + n]);
          outer += pv * k0;
        }
        st[k][i] += ce * outer;
      }
    }
  }

  // ---- per-token reads
  Feed<T, R, FULL, SHAPE> fd;
  fd.init(a, g, prep, b, h, grp, rp, n0, vp, p0, N, P, norm);
  float* fph = a.final_phase.ptr != nullptr && fin
                   ? static_cast<float*>(a.final_phase.ptr) + bo * a.final_phase.stride[0] +
                         h * a.final_phase.stride[1] + ps * a.final_phase.stride[2]
                   : nullptr;
  float* fblk = a.block_phase.ptr != nullptr
                    ? static_cast<float*>(a.block_phase.ptr) + b * a.block_phase.stride[0] +
                          h * a.block_phase.stride[1] + (tok0 >> 6) * a.block_phase.stride[2] +
                          ps * a.block_phase.stride[3]
                    : nullptr;
  const int64_t blk_stride = a.block_phase.stride[2];
  const __amdgpu_buffer_rsrc_t rs_o =
      make_rsrc(FIX ? const_cast<char*>(g.out_base) + b * g.out_b : nullptr,
                FIX ? a.length * (g.out_t < 0 ? -g.out_t : g.out_t) : 0);
  T* out_row = nullptr;
  int out_t = 0, o_out = 0;
  if constexpr (FIX) {
    out_t = g.out_t;
    o_out = h * g.out_h + g.out_o0;
  } else {
    out_row = static_cast<T*>(a.out.ptr) + b * a.out.stride[0] + h * a.out.stride[2];
    out_t = static_cast<int>(a.out.stride[1]);
  }

  // rotation roles of the q / k lane's 8 columns n0 + i: partner element, cos / sin table
  // column and the sign of the sine term; columns outside the rotated range keep cos 1, sin 0
  int rcol[8];
  float rsgn[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int n = n0 + i;
    if (!mimo_rot) {
      const int jn = n >> 1;
      rcol[i] = min(jn, max(S - 1, 0));
      rsgn[i] = jn < S ? ((i & 1) ? 1.f : -1.f) : 0.f;
    } else {
      const bool first = n < S, third = n >= 2 * S && n < 3 * S;
      rcol[i] = first ? n : (third ? n - 2 * S : 0);
      rsgn[i] = first ? -1.f : (third ? 1.f : 0.f);
    }
  }

  // ---- registers the global data of coming sub-chunks is loaded into
  constexpr int W8 = Words<T>::W8, W4 = Words<T>::W4;
  uint32_t rq[2][W8], rk[2][W8], rv[2][W4], rz[2][W4];
  float2 side;   // this lane's side word of a coming sub-chunk
  float4 ang;    // this lane's angle word of a coming sub-chunk
  const int scw = g.scw;
  const int side_n = scw + 2 * ROWS;  // floats of a side block
  float* ANG = F + Lay::ANG;
  // angle tile slot (16 bytes) of 4-token group g and angle s: rows of kSMax slots, the angle
  // XOR-keyed by the group's phase lane, so the PG lanes reading one angle and the lanes writing
  // one group hit distinct banks (key < 16, so s ^ key < kSMax)
  static_assert(16 % PG == 0 && 16 / PG * (PG - 1) < kSMax, "angle tile key");
  auto ang_slot = [&](int g, int s) { return g * kSMax + (s ^ ((g / (TPL / 4)) * (16 / PG))); };
  auto ang_store = [&](const float4& v) {
    if (4 * tid < TOK * S) {
      const int g = tid / S;
      *reinterpret_cast<float4*>(ANG + 4 * ang_slot(g, tid - g * S)) = v;
    }
  };
  // the angle inputs of this phase lane's tokens, from the angle tile
  auto angles_of = [&](float (&pa)[TPL]) {
#pragma unroll
    for (int q = 0; q < TPL / 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(ANG + 4 * ang_slot((TPL / 4) * pg + q, ps));
      pa[4 * q] = v.x;
      pa[4 * q + 1] = v.y;
      pa[4 * q + 2] = v.z;
      pa[4 * q + 3] = v.w;
    }
  };
  auto scb = [&](int c) { return F + Lay::SC0 + (c & 1) * Lay::SCB; };
  auto csb = [&](int c) { return F + Lay::CS0 + (c & 1) * Lay::CSB; };

  // Pipeline: iteration c stages sub-chunk c into LDS and writes the side block and angle tile of
  // c + 1 there (interval 1), then computes the outputs and state carry of c while the phases of
  // c + 1 are computed and the loads of c + 1 (words) and c + 2 (side, angles) are in flight
  // (interval 2). Side blocks and cos / sin tables alternate between two LDS buffers each.
  // prologue: side block and angle tile of 0 to LDS, phases of 0
  side = fd.side_in(c0);
  ang = fd.ang_in(c0);
  fd.words(tok0, min(TOK, L), qk_on, vz_on, rq, rk, rv, rz);
  if (2 * tid < side_n) *reinterpret_cast<float2*>(scb(0) + 2 * tid) = side;
  ang_store(ang);
  side = fd.side_in(c0 + 1);
  ang = fd.ang_in(c0 + 1);
  __syncthreads();
  if (ph_on && nsub > 0) {
    float pa[TPL];
    angles_of(pa);
    phase_stage<PG, TPL, CST, false, F32, LO ? kFull : kFast>(csb(0), ps, F + Lay::PBASE + ps, F + Lay::POFF + ps,
                                     scb(0) + SB_::DTV, 0, L, pg, lane, angles, pa, fph, fblk,
                                     blk_stride);
  }
  __syncthreads();

  float log_decay = 0.f;  // sum of adt so far: the log of the state's decay over the sequence
  for (int c = 0; c < nsub; ++c) {
    const int t0 = c * TOK;
    const int width = min(TOK, L - t0);
    const float* SC = scb(c);
    const float* CSt = csb(c);

    // ---- interval 1: stage sub-chunk c; the scalar block of c + 1 to LDS
    if (c + 1 < nsub) {
      if (2 * tid < side_n) *reinterpret_cast<float2*>(scb(c + 1) + 2 * tid) = side;
      ang_store(ang);
    }
    // q / k rows -> Qs, Ks (row-major), FP32 KT (transposed, swizzled); rows 2rp, 2rp+1.
    if (qk_on) {
      // (q, k) RMSNorm factors of rows 2rp, 2rp+1
      float fq[2] = {1.f, 1.f}, fk[2] = {1.f, 1.f};
      if (norm) {
        const float4 f = *reinterpret_cast<const float4*>(SC + scw + 4 * rp);
        fq[0] = f.x;
        fk[0] = f.y;
        fq[1] = f.z;
        fk[1] = f.w;
      }
      float kt[2][8];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int row = 2 * rp + j, tt = row / R;
        float q[8], k[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          q[i] = fmaf(raw_get<T>(rq[j], i), fq[j] * wq[i], bq[R == 1 ? 0 : j][i]);
          k[i] = fmaf(raw_get<T>(rk[j], i), fk[j] * wk[i], bk[R == 1 ? 0 : j][i]);
        }
        if (rotate && !mimo_rot) {
          // pairs (2j, 2j+1): one cos / sin per pair (cos 1, sin 0 past the call's angles)
#pragma unroll
          for (int pp = 0; pp < 4; ++pp) {
            const float2 cs = *reinterpret_cast<const float2*>(CSt + tt * CST + 2 * rcol[2 * pp]);
            const bool on = rsgn[2 * pp] != 0.f;
            const float cc = on ? cs.x : 1.f, ss = on ? cs.y : 0.f;
            const float q0 = q[2 * pp], q1 = q[2 * pp + 1], k0 = k[2 * pp], k1 = k[2 * pp + 1];
            q[2 * pp] = fmaf(q1, -ss, q0 * cc);
            q[2 * pp + 1] = fmaf(q0, ss, q1 * cc);
            k[2 * pp] = fmaf(k1, -ss, k0 * cc);
            k[2 * pp + 1] = fmaf(k0, ss, k1 * cc);
          }
        } else if (rotate) {
          // x' = x cos + sgn partner sin: MIMO pairs (n, n + N/2)
          float qp[8], kp[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int half = N >> 1;
            if (FULL) {
              // N = 128: the partner lane is lane ^ 8, a rotation by 8 in the 16-lane row
              qp[i] = dpp_shr<0x128>(q[i]);
              kp[i] = dpp_shr<0x128>(k[i]);
            } else if (half >= 8) {
              // (half is a multiple of 8: the host's check)
              const int l = tid & 15, src = 8 * l < half ? l + (half >> 3) : l - (half >> 3);
              qp[i] = __shfl(q[i], src, 16);
              kp[i] = __shfl(k[i], src, 16);
            } else {
              qp[i] = q[i ^ half];
              kp[i] = k[i ^ half];
            }
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float2 cs = *reinterpret_cast<const float2*>(CSt + tt * CST + 2 * rcol[i]);
            const float cc = rsgn[i] != 0.f ? cs.x : 1.f;
            const float ss = rsgn[i] * cs.y;
            q[i] = fmaf(qp[i], ss, q[i] * cc);
            k[i] = fmaf(kp[i], ss, k[i] * cc);
          }
        }
        if constexpr (!SO) st_row8<T>(Qs + row * LQ + n0, q);
        st_row8<T>(Ks + row * LQ + n0, k);
#pragma unroll
        for (int i = 0; i < 8; ++i) kt[j][i] = k[i];
      }
      // (FP32) K^T for the carry, each row scaled by its token's scale * end decay (the
      // carry's K~ e^{cum_last - cum}, ops.py:806-816)
      if constexpr (!KTR) {
        const int r0 = (2 * rp) / R, r1 = (2 * rp + 1) / R;
        const float cl = SC[SB_::CL];
        const float e0 = SC[SB_::SCL + r0] * exp_x<LO>(cl - SC[SB_::CUM + r0]);
        const float e1 = SC[SB_::SCL + r1] * exp_x<LO>(cl - SC[SB_::CUM + r1]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int n = n0 + i;
          if (FIX || n < N) {
            st_pair<T>(KT + n * LR + swz<ROWS>(2 * rp, n >> KSH), kt[0][i] * e0, kt[1][i] * e1);
          }
        }
      }
    }
    // value / gate of tokens 2vp, 2vp+1, columns p0 .. p0+3: rank values v mx_r -> VR
    // (row-major; 16-bit also VS, scaled; FP32 VT, transposed and swizzled), rank gates z mz_r
    // -> ZR (row-major)
    if (vz_on) {
      constexpr int VJ = Feed<T, R, FULL>::VJ;
      float v[VJ][4], z[VJ][4];
#pragma unroll
      for (int j = 0; j < VJ; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[j][i] = raw_get<T>(rv[j], i);
          z[j][i] = raw_get<T>(rz[j], i);
        }
      }
      // (16-bit) rows 2vp, 2vp+1 of VS: the token's scale * end decay (the carry's
      // e^{cum_last - cum} K~ factor, ops.py:806-816, moved onto V)
      float ev0 = 0.f, ev1 = 0.f;
      if constexpr (KTR) {
        const int u0 = (2 * vp) / R, u1 = (2 * vp + 1) / R;
        const float cl = SC[SB_::CL];
        ev0 = SC[SB_::SCL + u0] * __expf(cl - SC[SB_::CUM + u0]);
        ev1 = SC[SB_::SCL + u1] * __expf(cl - SC[SB_::CUM + u1]);
      }
      if (R == 1 && !F32) {
        // the loaded 16-bit words go to LDS unchanged as VR / ZR rows; VS rows scaled
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          f4 sv;
#pragma unroll
          for (int i = 0; i < 4; ++i) sv[i] = v[j][i] * (j ? ev1 : ev0);
          st_quad<T>(VS + (2 * vp + j) * LP + p0, sv);
          *reinterpret_cast<u32x2*>(VR + (2 * vp + j) * LP + p0) = (u32x2){rv[j][0], rv[j][1]};
          *reinterpret_cast<u32x2*>(ZR + (2 * vp + j) * LP + p0) = (u32x2){rz[j][0], rz[j][1]};
        }
      } else if (R == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int p = p0 + i;
          if (FIX || p < P) st_pair<T>(VT + p * LR + swz<ROWS>(2 * vp, p >> VSH), v[0][i], v[1][i]);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if constexpr (SO) break;
          f4 vq, zq;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            vq[i] = v[j][i];
            zq[i] = z[j][i];
          }
          st_quad<T>(VR + (2 * vp + j) * LP + p0, vq);
          st_quad<T>(ZR + (2 * vp + j) * LP + p0, zq);
        }
      } else {
        // rows 2vp, 2vp+1: ranks r0, r0 + 1 of token 2vp / R (every lane of the workgroup has a
        // row pair, as for R = 1)
        f4 vq[2];
#pragma unroll
        for (int jr = 0; jr < 2; ++jr) {
          const int row = 2 * vp + jr;
          f4 zq;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            vq[jr][i] = mul_r<T>(v[0][i], mxl[jr][i]);
            zq[i] = mul_r<T>(z[0][i], mzl[jr][i]);
          }
          if constexpr (!SO) {
            st_quad<T>(VR + row * LP + p0, vq[jr]);
            st_quad<T>(ZR + row * LP + p0, zq);
          }
        }
        if constexpr (KTR) {
#pragma unroll
          for (int jr = 0; jr < 2; ++jr) {
            f4 sv;
#pragma unroll
            for (int i = 0; i < 4; ++i) sv[i] = vq[jr][i] * (jr ? ev1 : ev0);
            st_quad<T>(VS + (2 * vp + jr) * LP + p0, sv);
          }
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int p = p0 + i;
            if (FIX || p < P) st_pair<T>(VT + p * LR + swz<ROWS>(2 * vp, p >> VSH), vq[0][i], vq[1][i]);
          }
        }
      }
    }
    // the state at the start of this sub-chunk, rounded to the activation dtype -> Sb[p][n]
#pragma unroll
    for (int k = 0; k < kTiles; ++k) {
      const int u = w + kWaves * k;
      if (!SO && (all_tiles || u < n_tiles)) {
        const int ni = u / kPT, pj = u - ni * kPT;
        st_quad<T>(Sb + (16 * pj + l16) * LQ + 16 * ni + 4 * lg, st[k]);
      }
    }
    // the carry's decay of the state, exp(cum_last) S^T: the carry products below accumulate
    // onto it
    {
      const float ecl = SC[SB_::ECL];
      log_decay += SC[LO ? SB_::DEC : SB_::CL];
#pragma unroll
      for (int k = 0; k < kTiles; ++k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) st[k][i] *= ecl;
      }
    }
    __syncthreads();

    // ---- interval 2
    // words of sub-chunk c + 1 into registers; they fly while sub-chunk c computes. FULL issues
    // every load of the loop unconditionally (reads past token L return zero), which keeps the
    // compiler's in-order wait counts exact: no load is waited for before its use. FULL spreads
    // them over the interval in three groups (q / k at its start, value / gate after the
    // scores, side and angle words after the phases) pinned between the compute stages, so the
    // eight waves do not queue all their loads at once.
    auto loads_qk = [&] {
      __builtin_amdgcn_sched_barrier(0);
      fd.words_qk(tok0 + t0 + TOK, min(TOK, L - t0 - TOK), qk_on, rq, rk);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto loads_vz = [&] {
      __builtin_amdgcn_sched_barrier(0);
      fd.words_vz(tok0 + t0 + TOK, min(TOK, L - t0 - TOK), vz_on, rv, rz);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto loads_side = [&] {
      __builtin_amdgcn_sched_barrier(0);
      side = fd.side_in(c0 + c + 2);
      ang = fd.ang_in(c0 + c + 2);
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (!FULL && !SHAPE) {
      if (c + 1 < nsub) fd.words(tok0 + t0 + TOK, min(TOK, L - t0 - TOK), qk_on, vz_on, rq, rk, rv, rz);
      side = fd.side_in(c0 + c + 2);
      ang = fd.ang_in(c0 + c + 2);
    }

    // (q / k words first: they are waited for first, at the top of the next iteration)
    if constexpr (FULL || SHAPE) loads_qk();

    // outputs for query row tile `it` and P tiles pj = wp, wp + WPR, ...
    const int it = w / WPR, wp = w - it * WPR;
    const int trow = 16 * it + l16;
    const int tq = trow / R;
    // 16-bit: the query rows of this tile, B operand of the scores and A operand of inter
    typename M::v8 qv[F32 ? 1 : NP / 32];
    if constexpr (!F32) {
#pragma unroll
      for (int kk = 0; kk < NP / 32; ++kk) {
        qv[kk] = *reinterpret_cast<const typename M::v8*>(Qs + trow * LQ + 32 * kk + 8 * lg);
      }
    }
    // FP32 operands are read 4 elements of K per lane (a 16-byte LDS read feeds 4 MFMAs): MFMA i of
    // a 16-element step takes elements 4 lg + i from both operands, K's own order permuted alike
    // (2 x 1024 tokens of 8 heads, 256-token segments: 71 us a pass with one 4-byte read per
    // operand and MFMA, 28 us so; 8 x 1000 tokens, 32 heads 253 -> 225). The query rows serve the scores and inter.
    f4 qf[F32 ? NP / 16 : 1];
    if constexpr (F32 && !SO) {
#pragma unroll
      for (int kk = 0; kk < NP / 16; ++kk) {
        qf[kk] = *reinterpret_cast<const f4*>(Qs + trow * LQ + 16 * kk + 4 * lg);
      }
    }
    // scores Sc^T tiles (rows s, column t), issued before the phase work below
    f4 acc[RT];
#pragma unroll
    for (int sj = 0; sj < RT; ++sj) {
      acc[sj] = zero4();
      if (SO || sj > it) continue;
      if constexpr (!F32) {
#pragma unroll
        for (int kk = 0; kk < NP / 32; ++kk) {
          const typename M::v8 av = *reinterpret_cast<const typename M::v8*>(
              Ks + (16 * sj + l16) * LQ + 32 * kk + 8 * lg);
          acc[sj] = M::mma(av, qv[kk], acc[sj]);
        }
      } else {
        f4 half = zero4();
#pragma unroll
        for (int kk = 0; kk < NP / 16; ++kk) {
          const f4 kv = *reinterpret_cast<const f4*>(Ks + (16 * sj + l16) * LQ + 16 * kk + 4 * lg);
          f4& sum = LO && kk < NP / 32 ? half : acc[sj];
#pragma unroll
          for (int i = 0; i < 4; ++i) sum = M::mma(kv[i], qf[kk][i], sum);
        }
        if constexpr (LO) acc[sj] += half;
      }
    }
    // K~^T V products of the state carry, issued early (they depend only on staged tiles),
    // accumulated onto the decayed state
#pragma unroll
    for (int k = 0; k < kTiles; ++k) {
      const int u = w + kWaves * k;
      if (!all_tiles && u >= n_tiles) continue;
      const int ni = u / kPT, pj = u - ni * kPT;
      const int nrow = 16 * ni + l16, prow = 16 * pj + l16;
      if constexpr (KTR) {
        // A: 8 tokens of column nrow from the row-major Ks, two transposing reads of 4 tokens
        // (in each 16-lane group, lane 4a + b receives element b of the 8-byte vectors of lanes
        // a, a + 4, a + 8, a + 12: lane x addresses token x / 4, columns 4 (x % 4) ..)
        const T* kc = Ks + (l16 >> 2) * LQ + 16 * ni + 4 * (l16 & 3);
        const T* vc = VS + (l16 >> 2) * LP + 16 * pj + 4 * (l16 & 3);  // B: the same from VS
#pragma unroll
        for (int kk = 0; kk < ROWS; kk += 32) {
          const T* k0 = kc + (kk + 8 * lg) * LQ;
          const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) i16x4*)(k0));
          const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) i16x4*)(k0 + 4 * LQ));
          const typename M::v8 av = __builtin_bit_cast(
              typename M::v8, (i16x8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
          const T* v0 = vc + (kk + 8 * lg) * LP;
          const i16x4 vlo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) i16x4*)(v0));
          const i16x4 vhi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) i16x4*)(v0 + 4 * LP));
          const typename M::v8 bv = __builtin_bit_cast(
              typename M::v8, (i16x8){vlo[0], vlo[1], vlo[2], vlo[3], vhi[0], vhi[1], vhi[2], vhi[3]});
          st[k] = M::mma(av, bv, st[k]);
        }
      } else {
        f4 sum = LO ? zero4() : st[k];
#pragma unroll
        for (int kk = 0; kk < ROWS; kk += 16) {
          const f4 kv = *reinterpret_cast<const f4*>(KT + nrow * LR + swz<ROWS>(kk + 4 * lg, nrow >> KSH));
          const f4 vv = *reinterpret_cast<const f4*>(VT + prow * LR + swz<ROWS>(kk + 4 * lg, prow >> VSH));
#pragma unroll
          for (int i = 0; i < 4; ++i) sum = M::mma(kv[i], vv[i], sum);
        }
        if constexpr (LO) {
#pragma unroll
          for (int i = 0; i < 4; ++i) sum[i] += st[k][i];
        }
        st[k] = sum;
      }
    }
    if constexpr (FULL || SHAPE) loads_vz();
    // phases of sub-chunk c + 1 (its dt block was computed two iterations ago)
    if (ph_on && c + 1 < nsub) {
      float pa[TPL];
      angles_of(pa);
      phase_stage<PG, TPL, CST, false, F32, LO ? kFull : kFast>(csb(c + 1), ps, F + Lay::PBASE + ps, F + Lay::POFF + ps,
                                       scb(c + 1) + SB_::DTV, t0 + TOK, L, pg, lane, angles, pa,
                                       fph, fblk, blk_stride);
    }
    if constexpr (FULL || SHAPE) loads_side();
    if constexpr (SO) {
      __syncthreads();
      continue;
    }
    // decayed scores W[t, s] = Sc[t, s] d[t, s] in FP32
    const float cum_t = SC[SB_::CUM + tq];
    const float gam_t = SC[SB_::GAM + tq];
    // the causal masks below compare a copy of tq the compiler cannot see through, so they are
    // evaluated here as vector compares, not hoisted out of the loop into scalar mask registers
    int tq_m = tq;
    __asm__ volatile("" : "+v"(tq_m));
    f4 wsc[RT];
#pragma unroll
    for (int sj = 0; sj < RT; ++sj) {
      wsc[sj] = zero4();
      if (sj > it) continue;
      if (sj < it) {
        // strictly earlier tile: d = exp(cum_t - cend) * (scale_s exp(cend - cum_s)), both <= 1
        const float at = exp_x<LO>(cum_t - SC[SB_::CEND + sj]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int ts = (16 * sj + 4 * lg + i) / R;
          wsc[sj][i] = acc[sj][i] * (at * SC[SB_::BSC + ts]);
        }
      } else {
        // diagonal tile: every term is read and computed, then selected (no per-lane branches)
        float cs[4], sc[4];
        if constexpr (R == 1) {
          const f4 c4 = *reinterpret_cast<const f4*>(SC + SB_::CUM + 16 * sj + 4 * lg);
          const f4 s4 = *reinterpret_cast<const f4*>(SC + SB_::SCL + 16 * sj + 4 * lg);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            cs[i] = c4[i];
            sc[i] = s4[i];
          }
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int ts = (16 * sj + 4 * lg + i) / R;
            cs[i] = SC[SB_::CUM + ts];
            sc[i] = SC[SB_::SCL + ts];
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int ts = (16 * sj + 4 * lg + i) / R;
          const float lower = sc[i] * exp_x<LO>(cum_t - cs[i]);
          const float d = tq_m > ts ? lower : (tq_m == ts ? gam_t : 0.f);
          wsc[sj][i] = acc[sj][i] * d;
        }
      }
    }
    // Outputs, computed transposed (Y^T tiles, rows p, columns the row tile's 16 (token, rank)
    // rows): a lane holds 4 consecutive p of one row, stored as one vector.
    const float ecum_t = exp_x<LO>(cum_t);
    const int rr = trow - tq * R;  // the lane's rank
#pragma unroll
    for (int pq = 0; pq < kPT / WPR; ++pq) {
      const int pj = wp + pq * WPR;
      const int pcol = 16 * pj + l16;  // the A-operand row of V^T / rnd(S)
      const int key = pcol >> VSH;
      f4 yi = zero4(), ye = zero4();
      if constexpr (!F32) {
        // intra: V^T W^T, the K axis permuted as the D-layout of wsc
#pragma unroll
        for (int m = 0; m < (RT + 1) / 2; ++m) {
          if (2 * m > it) continue;
          typename M::v8 av, bv;
          // 4 tokens of column pcol from the row-major VR by a transposing read each
          const T* vr0 = VR + (32 * m + 4 * lg + (l16 >> 2)) * LP + 16 * pj + 4 * (l16 & 3);
          const typename M::v4 b0 = __builtin_bit_cast(
              typename M::v4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                  (__attribute__((address_space(3))) i16x4*)(vr0)));
          const typename M::v4 b1 = __builtin_bit_cast(
              typename M::v4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                  (__attribute__((address_space(3))) i16x4*)(vr0 + 16 * LP)));
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            bv[i] = from_f<T>(wsc[2 * m][i]);
            bv[4 + i] = from_f<T>(2 * m + 1 < RT ? wsc[2 * m + 1][i] : 0.f);
            av[i] = b0[i];
            av[4 + i] = b1[i];
          }
          yi = M::mma(av, bv, yi);
        }
        // inter: rnd(S) Q^T
#pragma unroll
        for (int kk = 0; kk < NP / 32; ++kk) {
          const typename M::v8 av =
              *reinterpret_cast<const typename M::v8*>(Sb + pcol * LQ + 32 * kk + 8 * lg);
          ye = M::mma(av, qv[kk], ye);
        }
      } else {
#pragma unroll
        for (int sj = 0; sj < RT; ++sj) {
          if (sj > it) continue;
          const f4 vv = *reinterpret_cast<const f4*>(VT + pcol * LR + swz<ROWS>(16 * sj + 4 * lg, key));
#pragma unroll
          for (int i = 0; i < 4; ++i) yi = M::mma(vv[i], wsc[sj][i], yi);
        }
        f4 half = zero4();
#pragma unroll
        for (int kk = 0; kk < NP / 16; ++kk) {
          const f4 sv = *reinterpret_cast<const f4*>(Sb + pcol * LQ + 16 * kk + 4 * lg);
          f4& sum = LO && kk < NP / 32 ? half : ye;
#pragma unroll
          for (int i = 0; i < 4; ++i) sum = M::mma(sv[i], qf[kk][i], sum);
        }
        if constexpr (LO) ye += half;
      }
      // epilogue: row trow (token tq, rank rr), columns pb .. pb+3
      const int pb = 16 * pj + 4 * lg;
      float vv[4], zz[4];
      if constexpr (!F32) {
        const typename M::v4 v4 = *reinterpret_cast<const typename M::v4*>(VR + trow * LP + pb);
        const typename M::v4 z4 = *reinterpret_cast<const typename M::v4*>(ZR + trow * LP + pb);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          vv[i] = to_f(v4[i]);
          zz[i] = to_f(z4[i]);
        }
      } else {
        const f4 v4 = *reinterpret_cast<const f4*>(VR + trow * LP + pb);
        const f4 z4 = *reinterpret_cast<const f4*>(ZR + trow * LP + pb);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          vv[i] = v4[i];
          zz[i] = z4[i];
        }
      }
      f4 y;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        y[i] = (fmaf(ye[i], ecum_t, yi[i]) + Dh * vv[i]) * silu_x<LO>(zz[i]);
        if (R > 1) y[i] *= F[Lay::MO + rr * kPPad + pb + i];
      }
      if constexpr (R > 1) {
        // MIMO rank sum over the R consecutive lanes of one token (within a 16-lane row): DPP
        // quad permutes for lane ^ 1 and lane ^ 2, a swizzle for lane ^ 4 (no LDS access)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float t = y[i];
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
      if (rr == 0) {
        if constexpr (FIX) {
          // rows of tokens >= L fall outside the buffer extent: the store is dropped
          bstore_quad<T>(y, rs_o,
                         (tq * out_t + o_out + pb * ES) +
                             __builtin_amdgcn_readfirstlane((tok0 + t0) * out_t));
        } else {
          if (tq < width) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              if (pb + i < P) out_row[(tok0 + t0 + tq) * out_t + pb + i] = from_f<T>(y[i]);
            }
          }
        }
      }
    }

    // (the state carry S^T = exp(cum_last) S^T + K~^T V was accumulated above)
    __syncthreads();
  }

  // ---- final k: the biased, rotated k of token L-1, still in Ks from the last sub-chunk
  if (a.final_k.ptr != nullptr && fin) {
    const int tl = (L - 1) - (nsub - 1) * TOK;  // its row in the last sub-chunk
    for (int i = tid; i < R * N; i += kThreads) {
      const int r = i / N, n = i - r * N;
      static_cast<T*>(a.final_k.ptr)[bo * a.final_k.stride[0] + h * a.final_k.stride[1] +
                                     r * a.final_k.stride[2] + n] =
          Ks[(tl * R + r) * LQ + n];
    }
  }

  if (a.final_decay.ptr != nullptr && tid == 0) {
    static_cast<float*>(a.final_decay.ptr)[bo * a.final_decay.stride[0] +
                                           h * a.final_decay.stride[1]] = log_decay;
  }
  // the last block's increment sum (the earlier blocks' were written as each one ended)
  if (a.block_phase.ptr != nullptr && rotate && angles) {
    for (int i = tid; i < S; i += kThreads) {
      static_cast<float*>(a.block_phase.ptr)[b * a.block_phase.stride[0] +
                                             h * a.block_phase.stride[1] +
                                             ((tok0 + L - 1) >> 6) * a.block_phase.stride[2] +
                                             i * a.block_phase.stride[3]] = F[Lay::PBASE + i];
    }
  }

  // ---- final state
#pragma unroll
  for (int k = 0; k < kTiles; ++k) {
    const int u = w + kWaves * k;
    if (u >= n_tiles || !fin) continue;
    const int ni = u / kPT, pj = u - ni * kPT;
    const int p = 16 * pj + l16;
    if (p >= P) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 16 * ni + 4 * lg + i;
      if (n < N) {
        static_cast<float*>(a.final_state.ptr)[bo * a.final_state.stride[0] +
                                               h * a.final_state.stride[1] +
                                               p * a.final_state.stride[2] + n] = st[k][i];
      }
    }
  }
}


// ------------------------------------------------------------ segmented scan (composition)

// A sequence split into G segments is scanned twice (pass 1: every segment from a zero state and
// zero phase; pass 2: every segment from its true start), each segment a workgroup per head over
// the row's own tensors and prep results (ScanGeom::segs). Between them, compose_kernel walks
// each (b, h)'s segments in order. The scan is linear in its initial state and a rotation by
// phi + psi is the rotation by psi followed by phi, so with pass 1's local end state U_g (built
// from k rotated by local phases), log-decay l_g = sum adt and last k k_g:
//   S_{g+1} = e^{l_g} (S_g + c_g sum_r (v_prev mx_r) k_prev_r^T) + U_g Rot(phi_g)^T,
//   k_prev <- Rot(phi_g) k_g,  v_prev <- v at the segment's last token,
// where c_g = dt (1 - trap) at the segment's first token (the endpoint continuation the kernel
// applies to initial_k / initial_value; here it is part of the state pass 2 starts from, whose
// workgroups then skip it). The phase carry phi is the kernel's own walk over
// 64-token blocks, off <- fmod(off + block sum) (segments start on block boundaries), redone
// from pass 1's block sums: bit for bit the carry the unsplit scan reaches there, the fmod
// representative (sign) included. Pass 2 then starts segment g from S_g and phi_g; its last segment writes the call's final
// state, phase and k, and its block sums, which do not depend on the carry, are the call's.
struct SegGeom {
  int G, Ls, nblk;        // segments per batch row, tokens per segment, 64-token blocks per row
  float* seg_state;       // [B*G][H][P][N] pass 1's end states
  float* seg_decay;       // [B*G][H]
  float* seg_blk;         // [B][H][nblk][S] pass 1's phase block sums (phase mode ANGLES)
  void* seg_k;            // [B*G][H][R][N] pass 1's last k (activation dtype)
  float* in_state;        // [B*G][H][P][N] pass-2 initial states
  float* in_phase;        // [B*G][H][S]
};

constexpr int kCompThreads = 256;                         // state-row threads
constexpr int kCompBlock = 64 + kCompThreads;             // compose_kernel: phase walker + state rows
constexpr int kCompRows = 8;                              // state rows per workgroup
constexpr int kCompPer = kCompRows * kNPad / kCompThreads;  // state elements per thread
constexpr int kWalkBatch = 32;                          // block sums per walker load batch
constexpr int kMaxSegments = 256;                       // bounds compose_kernel's LDS

// Dynamic LDS of compose_kernel (floats): per segment the phase carry at its start [G][S], the
// endpoint coefficient, e^{sum adt} and sum adt [3][G].
static size_t compose_lds_bytes(int G, int S) {
  return sizeof(float) * (static_cast<size_t>(G) * S + static_cast<size_t>(3) * G);
}

// One workgroup per (batch, head, group of kCompRows state rows): the rows are independent in the
// composition (rotations pair columns within a row, the endpoint term is an outer product).
// Wave 0 walks the phase carry through every 64-token block in order; the other four waves
// update the state rows segment by segment behind it. Everything the state update reads except
// the carry (the local end states, last k and last values of pass 1) is loaded segments ahead,
// so the call's critical path is the walk itself. The waves meet through s_ready in LDS, never
// at a barrier: the walker publishes each segment's carry and moves on.
template <typename T, int R>
__global__ __launch_bounds__(kCompBlock) void compose_kernel(const m3_scan_args a,
                                                             const SegGeom sg) {
  const int H = a.heads, N = a.d_state, P = a.head_dim, S = a.num_angles, G = sg.G;
  const int nrg = (P + kCompRows - 1) / kCompRows;  // row groups per (b, h)
  const int bh = blockIdx.x / nrg, rg = blockIdx.x - bh * nrg;
  const int b = bh / H, h = bh - b * H;
  const int p0 = rg * kCompRows, np = min(kCompRows, P - p0);
  const int tid = threadIdx.x;
  const bool angles = a.phase_mode == M3_PHASE_ANGLES;
  const bool walk = angles && S > 0;
  const bool mimo = a.mimo_rotation != 0;
  const bool raw_dt = a.raw_dt != 0;
  const bool lead = rg == 0;  // writes the per-(b, h) outputs: phases, k, decay
  extern __shared__ float dyn[];
  float* s_phig = dyn;             // [G][S] phase carry at each segment's start
  float* s_c0g = s_phig + G * S;   // [G] endpoint coefficient dt (1 - trap)
  float* s_decg = s_c0g + G;       // [G] e^{sum adt}
  float* s_draw = s_decg + G;      // [G] sum adt
  __shared__ int s_ready;          // segments whose starting carry is in s_phig
  auto row = [&](int g) { return (static_cast<int64_t>(b) * G + g) * H + h; };

  // per segment, in parallel: the endpoint coefficient and the decay (raw loads of segment tid,
  // decoded after the other loads are out)
  const int gc0 = min(tid, G - 1);
  const int64_t tc0 = static_cast<int64_t>(gc0) * sg.Ls;
  const RawX dt_r = ldraw(a.dt.ptr, a.dt.dtype,
                          b * a.dt.stride[0] + tc0 * a.dt.stride[1] + h * a.dt.stride[2]);
  const RawX tr_r = ldraw(a.trap.ptr, a.trap.dtype,
                          b * a.trap.stride[0] + tc0 * a.trap.stride[1] + h * a.trap.stride[2]);
  const RawX db_r = raw_dt ? ldraw(a.dt_bias.ptr, a.dt_bias.dtype, h * a.dt_bias.stride[0])
                           : RawX{0u, 0u};
  const float lg_dec = sg.seg_decay[row(gc0)];
  static_assert(kMaxSegments <= kCompBlock, "a thread per segment");
  auto coefficients = [&]() __attribute__((always_inline)) {
    if (tid < G) {
      float dt0, adt0;
      dt_adt(raw_dt, decode(dt_r, a.dt.dtype), 0.f, raw_dt ? decode(db_r, a.dt_bias.dtype) : 0.f, dt0,
             adt0);
      s_c0g[tid] = dt0 * (1.f - sigmoidf(decode(tr_r, a.trap.dtype)));
      s_draw[tid] = lg_dec;
      s_decg[tid] = expf(lg_dec);
    }
    if (tid == 0) s_ready = walk ? 0 : G;
    __syncthreads();
  };

  if (tid < 64) {
    // ---- wave 0: the phase carry, the kernel's own recurrence off <- fmod(off + block sum)
    // over the blocks of segments 0 .. G-2 in order, published at each segment's start. Lanes
    // s < S walk angle s; block sums are loaded a batch ahead of the fmod chain.
    const bool walker = walk && tid < S;
    const int tw = walker ? tid : 0;  // lanes without an angle load angle 0 and do nothing else
    float off = 0.f;
    if (a.initial_phase.ptr != nullptr && walk) {
      off = static_cast<const float*>(a.initial_phase.ptr)
          [b * a.initial_phase.stride[0] + h * a.initial_phase.stride[1] +
           tw * a.initial_phase.stride[2]];
    }
    auto publish = [&](int g) __attribute__((always_inline)) {
      s_phig[g * S + tid] = off;
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the carry is in LDS before the count
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      if (tid == 0) __hip_atomic_store(&s_ready, g + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    // (segments 0 .. G - 2 are whole: nbs blocks each)
    const int nbs = sg.Ls >> 6, gend = G - 1;
    const int64_t seg_stride = static_cast<int64_t>(nbs) * S;  // floats from segment to segment
    const float* blk = sg.seg_blk + static_cast<int64_t>(bh) * sg.nblk * S + tw;
    // batches never cross a segment's end; every load is issued (the last one repeated past a
    // short batch's end) so the waits stay exact
    auto load = [&](float (&buf)[kWalkBatch], int g, int k0) __attribute__((always_inline)) {
      const int n = min(kWalkBatch, nbs - k0);
      const float* p = blk + g * seg_stride + static_cast<int64_t>(k0) * S;
#pragma unroll
      for (int u = 0; u < kWalkBatch; ++u) buf[u] = p[min(u, n - 1) * S];
    };
    auto advance = [&](int& g, int& k0) __attribute__((always_inline)) {
      k0 += kWalkBatch;
      if (k0 >= nbs) {
        k0 = 0;
        ++g;
      }
    };
    auto walk_batch = [&](const float (&buf)[kWalkBatch], int g, int k0)
                          __attribute__((always_inline)) {
      const int n = min(kWalkBatch, nbs - k0);
#pragma unroll
      for (int u = 0; u < kWalkBatch; ++u) {
        if (u >= n) break;
        off = m3_fmod_2pi_small(__fadd_rn(off, buf[u]));
      }
      if (k0 + n == nbs) publish(g + 1);  // segment g walked: the carry at segment g + 1's start
    };
    float bufA[kWalkBatch], bufB[kWalkBatch];
    int gA = 0, kA = 0;
    if (walk && gend > 0) load(bufA, gA, kA);
    coefficients();
    if (!walker) return;
    publish(0);
    if (gend > 0) {
      for (;;) {
        int gB = gA, kB = kA;
        advance(gB, kB);
        const bool moreB = gB < gend;
        load(bufB, moreB ? gB : gA, moreB ? kB : kA);
        walk_batch(bufA, gA, kA);
        if (!moreB) break;
        int gC = gB, kC = kB;
        advance(gC, kC);
        const bool moreC = gC < gend;
        load(bufA, moreC ? gC : gB, moreC ? kC : kB);
        walk_batch(bufB, gB, kB);
        if (!moreC) break;
        gA = gC;
        kA = kC;
      }
    }
    return;
  }

  // ---- waves 1-4: this workgroup's state rows, segment by segment
  const int tb = tid - 64;
  // thread tb holds column tb % 2^lgN (2^lgN: N rounded up to a power of 2, which divides
  // kCompThreads; threads past column N do nothing) of the rows (tb + kCompThreads i) >> lgN
  const int lgN = N > 1 ? 32 - __builtin_clz(N - 1) : 0;
  const int n = min(tb & ((1 << lgN) - 1), N - 1);
  const bool col_on = (tb & ((1 << lgN) - 1)) < N;
  // rotation partner of column n (-1: not rotated), whether n is the pair's first element, and
  // the pair's angle: SISO pairs (2j, 2j+1), j < S; MIMO pairs (j, j + 2S), j < S
  const int S2 = 2 * S;
  bool lo;
  int j;
  int part;
  if (!mimo) {
    lo = (n & 1) == 0;
    j = n >> 1;
    part = (angles && n < S2) ? (n ^ 1) : -1;
  } else {
    lo = n < S2;
    j = lo ? n : n - S2;
    part = (angles && j < S) ? (lo ? n + S2 : j) : -1;
  }
  const int np_n = part >= 0 ? part : n;
  auto rot = [&](float x, float xp, float c, float sn) {
    return lo ? x * c - xp * sn : xp * sn + x * c;
  };
  const T* seg_k = static_cast<const T*>(sg.seg_k);
  const T* value = static_cast<const T*>(a.value.ptr);
  int pl[kCompPer];
  bool on[kCompPer];
#pragma unroll
  for (int i = 0; i < kCompPer; ++i) {
    const int p = (tb + kCompThreads * i) >> lgN;
    on[i] = col_on && p < np;
    pl[i] = min(p, np - 1);
  }

  // the start: the caller's state, k and value (zero without them)
  float st[kCompPer], vp[kCompPer], kp[R], mxr[R][kCompPer];
#pragma unroll
  for (int i = 0; i < kCompPer; ++i) {
    st[i] = (on[i] && a.initial_state.ptr != nullptr)
                ? static_cast<const float*>(a.initial_state.ptr)
                      [b * a.initial_state.stride[0] + h * a.initial_state.stride[1] +
                       (p0 + pl[i]) * a.initial_state.stride[2] + n]
                : 0.f;
    vp[i] = a.initial_k.ptr != nullptr
                ? to_f(static_cast<const T*>(a.initial_value.ptr)
                           [b * a.initial_value.stride[0] + h * a.initial_value.stride[1] +
                            p0 + pl[i]])
                : 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      mxr[r][i] = R > 1 ? rnd<T>(ldx(a.mimo_x.ptr, a.mimo_x.dtype,
                                     h * a.mimo_x.stride[0] + r * a.mimo_x.stride[1] + p0 + pl[i]))
                        : 1.f;
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    kp[r] = a.initial_k.ptr != nullptr
                ? to_f(static_cast<const T*>(a.initial_k.ptr)
                           [b * a.initial_k.stride[0] + h * a.initial_k.stride[1] +
                            r * a.initial_k.stride[2] + n])
                : 0.f;
  }

  // a ring of D segments' inputs: local end state (the element and its rotation partner), last
  // k (column n and its partner, every rank) and the value of the last token (the thread's rows)
  constexpr int D = R <= 4 ? 4 : 2;
  float ru[D][kCompPer], rup[D][kCompPer], rk[D][R], rkp[D][R], rv[D][kCompPer];
  auto fetch = [&](int d, int g) __attribute__((always_inline)) {
    const int gc = min(g, G - 1);  // past the end: a repeat of the last segment, unused
    const int64_t sh = row(gc);
    const float* U = sg.seg_state + (sh * P + p0) * N;
#pragma unroll
    for (int i = 0; i < kCompPer; ++i) {
      ru[d][i] = U[pl[i] * N + n];
      rup[d][i] = U[pl[i] * N + np_n];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      rk[d][r] = to_f(seg_k[sh * R * N + r * N + n]);
      rkp[d][r] = to_f(seg_k[sh * R * N + r * N + np_n]);
    }
    const int tl = min(gc * sg.Ls + sg.Ls, a.length) - 1;
#pragma unroll
    for (int i = 0; i < kCompPer; ++i) {
      rv[d][i] = to_f(value[b * a.value.stride[0] + tl * a.value.stride[1] +
                            h * a.value.stride[2] + p0 + pl[i]]);
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d) fetch(d, d);
  coefficients();

  for (int g0 = 0; g0 < G; g0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int g = g0 + d;
      if (g >= G) break;
      const int64_t sh = row(g);
      float u[kCompPer], up[kCompPer], kx[R], kxp[R], vl[kCompPer];
#pragma unroll
      for (int i = 0; i < kCompPer; ++i) {
        u[i] = ru[d][i];
        up[i] = rup[d][i];
        vl[i] = rv[d][i];
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        kx[r] = rk[d][r];
        kxp[r] = rkp[d][r];
      }
      fetch(d, g + D);

      // (1) segment g's start for pass 2: the state with the endpoint term (ops.py:681-686)
      const float c0 = s_c0g[g], dec = s_decg[g];
#pragma unroll
      for (int i = 0; i < kCompPer; ++i) {
        float endpoint = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) endpoint += (R > 1 ? mul_r<T>(vp[i], mxr[r][i]) : vp[i]) * kp[r];
        st[i] += c0 * endpoint;
        if (on[i]) sg.in_state[(sh * P + p0 + pl[i]) * N + n] = st[i];
      }
      // the carry at segment g's start, once the walker has published it. The walker is a wave
      // of this workgroup (resident with it) and publishes every segment without waiting on
      // anything, so the wait always ends; the spin cap (seconds) only keeps a defect from
      // becoming a hang. LDS operations of one wave complete in order and the walker drains its
      // carry stores before the count, so a count above g means the carry is readable.
      float cs = 1.f, sn = 0.f;
      if (walk) {
        for (int spin = 0;
             __hip_atomic_load(&s_ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <= g &&
             spin < (1 << 24);
             ++spin) {
          __builtin_amdgcn_s_sleep(2);
        }
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        if (part >= 0) {
          if (sizeof(T) == 4 && (N & (N - 1)) != 0) {
            sincos_of<kFull>(s_phig[g * S + j], &sn, &cs);
          } else {
            __sincosf(s_phig[g * S + j], &sn, &cs);
          }
        }
        if (lead && tb < S) sg.in_phase[sh * S + tb] = s_phig[g * S + tb];
      }

      // (2) the state at the segment's end: e^l S + Rot U
#pragma unroll
      for (int i = 0; i < kCompPer; ++i) {
        if (on[i]) st[i] = dec * st[i] + (part >= 0 ? rot(u[i], up[i], cs, sn) : u[i]);
      }
      // (3) the next segment's endpoint: this segment's last k, rotated by its carry, and value
#pragma unroll
      for (int r = 0; r < R; ++r) {
        kp[r] = part >= 0 ? rnd<T>(rot(kx[r], kxp[r], cs, sn)) : rnd<T>(kx[r]);
      }
#pragma unroll
      for (int i = 0; i < kCompPer; ++i) vp[i] = vl[i];
    }
  }

  // the call's decay (its final state, phase and k come from pass 2)
  if (lead && tb == 0 && a.final_decay.ptr != nullptr) {
    float decay_sum = 0.f;
    for (int g = 0; g < G; ++g) decay_sum += s_draw[g];
    static_cast<float*>(a.final_decay.ptr)[b * a.final_decay.stride[0] +
                                           h * a.final_decay.stride[1]] = decay_sum;
  }
}

// ------------------------------------------------------------------ host side

static bool pow2(int x) { return x > 0 && (x & (x - 1)) == 0; }

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The form in which scan16_kernel takes a call (Form16), -1 when it does not: a 16-bit call of up
// to 128 columns, 64 values and 32 angles at ranks 1, 2, 4 and 8, whose q / k / value / gate /
// out rows can be read and written 4 elements at a time, each token's row (of one group or head)
// below the next token's, and whose offsets within a batch row fit 32 bits (the loads run up to
// two sub-chunks, 128 tokens, and a token group ahead). Projection form: norm weights, biases, raw
// dt, angle increments; hook form: none of the norms, phases given or none. Rank 1 with the MIMO
// rotation takes the other kernels. `rows` false: without the workspace for prep's rows (kModel's
// shape and the ranks above 1 then take kProj and kHook, which read the caller's). A required tensor
// that is not set yet (a workspace query ahead of the buffers) counts as one that fits; at a d_state
// no power of 2, whose other route needs no workspace, as one that does not.
// Every such call is faster on it than on the kernel it took before (per call, scan_kernel then
// scan16_kernel, 8 x 1024 tokens, 32 heads): hook form rank 1 80 -> 71 us, rank 2 184 -> 120,
// rank 4 332 -> 200, rank 8 628 -> 359; projection form rank 2 140 -> 120, rank 8 487 -> 381,
// d_state 64 rank 1 114 -> 73; hook form of 32 groups, 4 x 4096 tokens, 518 -> 235, of 64 groups at
// rank 8, 64 heads, 1,678 -> 858; the recurrent scan at d_state 96, 4 x 1500 tokens, 16 heads: 21.6
// ms -> 77 us.
static int form16_of(const m3_scan_args& a, bool rows) {
  if (a.act_dtype != M3_BF16 && a.act_dtype != M3_F16) return -1;
  if (a.rank != 1 && a.rank != 2 && a.rank != 4 && a.rank != 8) return -1;
  const int N = a.d_state, P = a.head_dim, S = a.num_angles;
  if (N < 4 || N > kNPad || N % 4 != 0 || P <= 0 || P > kPPad || P % 4 != 0 || S > kSMax ||
      a.length <= 0 || a.batch <= 0 || a.groups <= 0 || a.heads % a.groups != 0) {
    return -1;
  }
  const bool rotates = a.phase_mode != M3_PHASE_NONE;
  // the MIMO pairs' columns come in chunks of 4 (4 S == N there, 2 S <= N otherwise: validated)
  if (rotates && (a.mimo_rotation ? S % 4 != 0 || 4 * S != N : 2 * S > N)) return -1;
  if (rotates && (S <= 0 || (a.rank == 1 && a.mimo_rotation))) return -1;
  const bool norm = a.q_norm_w.ptr != nullptr && a.k_norm_w.ptr != nullptr;
  const bool proj = norm && a.q_bias.ptr != nullptr && a.k_bias.ptr != nullptr &&
                    a.raw_dt != 0 && a.phase_mode == M3_PHASE_ANGLES;
  const bool hook = a.q_norm_w.ptr == nullptr && a.k_norm_w.ptr == nullptr && a.raw_dt == 0 &&
                    a.phase_mode != M3_PHASE_ANGLES;
  if (!proj && !hook) return -1;
  const int64_t len = a.length, ahead = len + 256;
  // rows of `dims` outer axes (extents in `ext`) read `span` elements at a time
  auto rows_ok = [&](const m3_tensor& t, std::initializer_list<int64_t> ext, int64_t span) {
    if (t.ptr == nullptr) return pow2(N);
    if (reinterpret_cast<uintptr_t>(t.ptr) % 8 != 0) return false;
    int i = 0;
    for (int64_t e : ext) {
      if (e > 1 && t.stride[i] % 4 != 0) return false;
      ++i;
    }
    const int64_t s1 = t.stride[1] < 0 ? -t.stride[1] : t.stride[1];
    return (len == 1 || s1 >= span) && ahead * s1 * 2 < INT32_MAX;
  };
  if (!rows_ok(a.q, {a.batch, len, a.groups, a.rank}, N) ||
      !rows_ok(a.k, {a.batch, len, a.groups, a.rank}, N) ||
      !rows_ok(a.value, {a.batch, len, a.heads}, P) || !rows_ok(a.gate, {a.batch, len, a.heads}, P) ||
      !rows_ok(a.out, {a.batch, len, a.heads}, P)) {
    return -1;
  }
  // one token: its stride is never used to reach another, and must not take the offsets out of
  // range or make a second token alias the first
  if (len == 1) {
    for (const m3_tensor* t : {&a.value, &a.gate, &a.out}) {
      if (t->ptr != nullptr && (t->stride[1] < 0 ? -t->stride[1] : t->stride[1]) < P) return -1;
    }
  }
  const int64_t tok = 64 / a.rank, nsub = (len + tok - 1) / tok;
  if ((proj && ahead * a.groups * a.rank * 8 >= INT32_MAX) || (nsub + 3) * (5 * tok + 8) * 4 >= INT32_MAX) {
    return -1;
  }
  if (a.phase_mode == M3_PHASE_ANGLES && ahead * S * 4 >= (int64_t{1} << 30)) return -1;
  if (a.phase_mode == M3_PHASE_GIVEN && (a.phase.ptr != nullptr || !pow2(N))) {
    const int64_t s1 = a.phase.stride[1] < 0 ? -a.phase.stride[1] : a.phase.stride[1];
    const int64_t span = (S - 1) * a.phase.stride[3] + 1;
    if (a.phase.ptr == nullptr || a.phase.stride[3] < 0 || s1 < span ||
        ahead * s1 * 4 >= (int64_t{1} << 30)) {
      return -1;
    }
  }
  // offsets within one (batch, head) of the states and within one head of the parameters, in
  // 32 bits
  for (const m3_tensor* t : {&a.initial_state, &a.final_state}) {
    if (t->ptr != nullptr && (t->stride[2] < 0 || (P * t->stride[2] + N) * 4 >= (int64_t{1} << 30))) {
      return -1;
    }
  }
  for (const m3_tensor* t : {&a.q_bias, &a.k_bias, &a.mimo_x, &a.mimo_z, &a.mimo_out}) {
    if (t->ptr != nullptr && (t->stride[1] < 0 || (a.rank * t->stride[1] + N) * 4 >= (int64_t{1} << 30))) {
      return -1;
    }
  }
  if (a.initial_k.ptr != nullptr &&
      (a.initial_k.stride[2] < 0 || (a.rank * a.initial_k.stride[2] + N) * 2 >= (int64_t{1} << 30))) {
    return -1;
  }
  if (proj && rows && N == kNPad && P == kPPad && S == kSMax && a.groups == 1 &&
      (a.rank == 1 || a.rank == 4) && (a.mimo_rotation != 0) == (a.rank > 1) &&
      ahead * a.rank * 2 * kNPad * 2 < INT32_MAX) {
    return kModel;
  }
  // prep's rows of one batch row, in 32 bits
  const int64_t row_bytes = proj ? N * 4 : kNPad * 2;
  if (rows && a.rank > 1 && ahead * a.groups * a.rank * 2 * row_bytes < INT32_MAX) {
    if (proj) return kRows;
    if (a.heads >= 16 * a.groups && int64_t{2} * a.batch * len * a.groups * a.rank < INT32_MAX) return kCopy;
  }
  // the caller's rows: the ranks of a token's row below the next token's (also of one token: the
  // rows after it are read, as zeros, past the extent)
  for (const m3_tensor* t : {&a.q, &a.k}) {
    if (t->ptr == nullptr) continue;
    const int64_t s1 = t->stride[1] < 0 ? -t->stride[1] : t->stride[1];
    const int64_t span = (a.rank - 1) * t->stride[3] + N;
    if ((a.rank > 1 && t->stride[3] < 0) || s1 < span) return -1;
  }
  return proj ? kProj : kHook;
}

// Prep workspace regions (floats, each 16-byte aligned) and the sub-chunk geometry; returns the
// workspace size in bytes. `form16`: form16_of(a).
static size_t ws_layout(const m3_scan_args& a, ScanGeom& g, int form16) {
  const int rows = a.act_dtype == M3_F32 ? Mma<float>::ROWS : Mma<__bf16>::ROWS;
  const int rank = a.rank > 0 ? a.rank : 1;
  g.tok = rows / rank > 0 ? rows / rank : 1;
  const int64_t len = a.length > 0 ? a.length : 0;
  g.nsub = static_cast<int>((len + g.tok - 1) / g.tok);
  g.scw = 5 * g.tok + 8;  // ScBlk<tok>::SIZE
  g.L4 = static_cast<int>((len + 3) / 4);
  g.form16 = form16;
  g.segs = 1;
  g.seg_len = static_cast<int>((len + 63) / 64 * 64);
  g.last_only = 0;
  g.perm = a.phase_mode != M3_PHASE_NONE && a.mimo_rotation != 0;
  g.lo = !pow2(a.d_state);
  const bool norm = a.q_norm_w.ptr != nullptr && form16 != kModel && form16 != kRows;
  const bool angles = a.phase_mode == M3_PHASE_ANGLES;
  const int64_t batch = a.batch > 0 ? a.batch : 0;
  int64_t off = 0;
  auto take = [&](int64_t n) {
    const int64_t o = off;
    off += (n + 3) / 4 * 4;
    return o;
  };
  g.ws_norm = norm ? take(batch * len * a.groups * a.rank * 2) : -1;
  g.ws_ang = angles ? take(batch * g.L4 * a.num_angles * 4) : -1;
  g.ws_sc = take(batch * a.heads * g.nsub * g.scw);
  const int64_t bytes = off * static_cast<int64_t>(sizeof(float));
  // the projection form's 32-bit offsets run up to two sub-chunk strides past the end
  g.ws_bytes = bytes < (int64_t{1} << 30) ? static_cast<int>(bytes) : -1;
  g.ws_qk = -1;
  if (form16 != kModel && form16 != kRows && form16 != kCopy) return static_cast<size_t>(bytes);
  g.ws_qk = (bytes + 255) / 256 * 256;  // 256-byte aligned
  return static_cast<size_t>(g.ws_qk + batch * len * a.groups * a.rank * 2 *
                                           (form16 == kRows ? a.d_state * 4 : kNPad * 2));
}

template <typename T>
static ScanGeom make_geom(const m3_scan_args& a, int form16) {
  ScanGeom g{};
  const int es = sizeof(T);
  const int total = a.batch * a.heads;
  g.xcd_map = (total % 8 == 0) ? 1 : 0;
  // vector loads need every row start aligned: base pointers and all outer strides
  auto vec_ok = [&](const m3_tensor& t, int dims, int need) {
    if ((reinterpret_cast<uintptr_t>(t.ptr) % need) != 0) return false;
    for (int i = 0; i < dims - 1; ++i) {
      if ((t.stride[i] * es) % need != 0) return false;
    }
    return true;
  };
  g.vec_qk = (a.d_state % 8 == 0) && vec_ok(a.q, 5, 16) && vec_ok(a.k, 5, 16);
  auto nw_ok = [](const m3_tensor& t) {
    return t.ptr != nullptr && t.stride[0] == 1 && reinterpret_cast<uintptr_t>(t.ptr) % 8 == 0;
  };
  g.vec_nw = (a.d_state % 8 == 0) && nw_ok(a.q_norm_w) && nw_ok(a.k_norm_w);
  const int vneed = es * 4;  // 4 elements per v / z load
  g.vec_vz = (a.head_dim % 4 == 0) && vec_ok(a.value, 4, vneed) && vec_ok(a.gate, 4, vneed);
  ws_layout(a, g, form16);
  return g;
}

// Projection form: q, k, value, gate, dt, a, trap all of the activation dtype and slices of one
// projection row (same batch and token strides, every slice's per-token extent inside one token
// row), out token-major, and every offset the kernel forms below 2^31 bytes. Fills the byte
// geometry of `g`.
static bool projection_form(const m3_scan_args& a, ScanGeom& g, int es) {
  const m3_tensor* ts[7] = {&a.q, &a.k, &a.value, &a.gate, &a.dt, &a.a, &a.trap};
  for (const m3_tensor* t : ts) {
    if (t->dtype != a.act_dtype || t->stride[0] != a.q.stride[0] ||
        t->stride[1] != a.q.stride[1]) {
      return false;
    }
  }
  for (int i = 2; i < 5; ++i) {
    if (a.k.stride[i] != a.q.stride[i]) return false;
  }
  for (int i = 2; i < 4; ++i) {
    if (a.gate.stride[i] != a.value.stride[i]) return false;
  }
  if (a.a.stride[2] != a.dt.stride[2] || a.trap.stride[2] != a.dt.stride[2]) return false;
  const int64_t lim = INT32_MAX;
  const bool rev = a.q.stride[1] < 0;  // every per-token tensor runs the same way (validated)
  const int64_t tok = (rev ? -a.q.stride[1] : a.q.stride[1]) * es;
  const int64_t ext_q = ((a.groups - 1) * a.q.stride[2] + (a.rank - 1) * a.q.stride[3] +
                         a.d_state) * es;
  const int64_t ext_v = ((a.heads - 1) * a.value.stride[2] + a.head_dim) * es;
  const int64_t ext_s = ((a.heads - 1) * a.dt.stride[2] + 1) * es;
  const int64_t ext[7] = {ext_q, ext_q, ext_v, ext_v, ext_s, ext_s, ext_s};
  const char* base = static_cast<const char*>(a.q.ptr);
  for (const m3_tensor* t : ts) base = std::min(base, static_cast<const char*>(t->ptr));
  int64_t off[7];
  for (int i = 0; i < 7; ++i) {
    off[i] = static_cast<const char*>(ts[i]->ptr) - base;
    if (off[i] + ext[i] > tok) return false;
  }
  const int64_t out_tok = (rev ? -a.out.stride[1] : a.out.stride[1]) * es;
  if (((a.heads - 1) * a.out.stride[2] + a.head_dim) * es > out_tok) return false;
  const int64_t len = a.length;
  if (len * tok >= lim || len * out_tok >= lim || len * a.groups * a.rank * 8 >= lim ||
      static_cast<int64_t>(g.L4) * a.num_angles * 16 >= lim ||
      static_cast<int64_t>(g.nsub) * g.scw * 4 >= lim) {
    return false;
  }
  // backwards: the slices' pointers address logical token 0, the physical row L - 1; the buffer
  // starts at physical row 0 and logical token t sits (L - 1 - t) rows above it
  const int64_t shift = rev ? (len - 1) * tok : 0;
  g.proj = base - shift;
  g.proj_b = a.q.stride[0] * es;
  g.tok_b = static_cast<int>(rev ? -tok : tok);
  g.o_q = static_cast<int>(off[0] + shift);
  g.o_k = static_cast<int>(off[1] + shift);
  g.o_v = static_cast<int>(off[2] + shift);
  g.o_z = static_cast<int>(off[3] + shift);
  g.o_dt = static_cast<int>(off[4] + shift);
  g.o_a = static_cast<int>(off[5] + shift);
  g.o_tr = static_cast<int>(off[6] + shift);
  g.qk_g = static_cast<int>(a.q.stride[2] * es);
  g.qk_r = static_cast<int>(a.q.stride[3] * es);
  g.vz_h = static_cast<int>(a.value.stride[2] * es);
  g.sc_h = static_cast<int>(a.dt.stride[2] * es);
  g.out_b = a.out.stride[0] * es;
  g.out_t = static_cast<int>(rev ? -out_tok : out_tok);
  g.out_h = static_cast<int>(a.out.stride[2] * es);
  g.out_o0 = static_cast<int>(rev ? (len - 1) * out_tok : 0);
  g.out_base = static_cast<const char*>(a.out.ptr) - g.out_o0;
  return true;
}

// The model's own shape (N = 128, P = 64, S = 32, norm, bias, raw dt, angle phases, the rank's
// rotation) in projection form: the specialization with every shape and mode a compile-time
// constant and guard-free buffer addressing.
static bool full_shape(const m3_scan_args& a, ScanGeom& g, int R) {
  return a.length > 0 && a.groups == 1 && g.ws_bytes > 0 && a.d_state == kNPad &&
         a.head_dim == kPPad &&
         a.num_angles == kSMax &&
         a.q_norm_w.ptr != nullptr && a.q_bias.ptr != nullptr && a.raw_dt != 0 &&
         a.phase_mode == M3_PHASE_ANGLES && (a.mimo_rotation != 0) == (R > 1) && g.vec_qk &&
         g.vec_vz && projection_form(a, g, a.act_dtype == M3_F32 ? 4 : 2);
}

// The model's shape with the generic inputs (scan_kernel's SHAPE form): N = 128, P = 64, 32
// angles when rotating, one group, vector-aligned q / k and value / gate rows, a workspace
// below 2^30 bytes. Its reads and the output go through one buffer resource per tensor and
// (batch, head) at 32-bit byte offsets, so every token stride is positive, each token's row
// (ranks, or heads for the output) ends below the next token's, and L + 256 rows (the loads
// run up to two sub-chunks and a token group ahead) stay below 2^31 bytes. Sets the output
// geometry.
static bool model_shape(const m3_scan_args& a, ScanGeom& g, int es) {
  // (rank 1 rotates the pairs (2j, 2j+1) only)
  if (!(a.d_state == kNPad && a.head_dim == kPPad && a.groups == 1 && g.vec_qk && g.vec_vz &&
        (a.phase_mode == M3_PHASE_NONE || a.num_angles == kSMax) && g.ws_bytes > 0 &&
        (a.rank > 1 || a.mimo_rotation == 0) &&
        g.ws_bytes < (1 << 30))) {
    return false;
  }
  const int64_t rows = static_cast<int64_t>(a.length) + 256;
  // a token's row of `span` elements below the next token's, L + 256 rows in 32 bits
  auto fits = [&](const m3_tensor& t, int64_t span, int64_t esz) {
    return t.stride[1] > 0 && span <= t.stride[1] && rows * t.stride[1] * esz < INT32_MAX;
  };
  for (const m3_tensor* t : {&a.q, &a.k}) {
    if (t->stride[3] < 0 || !fits(*t, (a.rank - 1) * t->stride[3] + a.d_state, es)) return false;
  }
  // the output is stored 4 elements at a time
  const int64_t o4 = 4 * es;
  if (reinterpret_cast<uintptr_t>(a.out.ptr) % o4 != 0 || (a.out.stride[0] * es) % o4 != 0 ||
      (a.out.stride[1] * es) % o4 != 0 || (a.out.stride[2] * es) % o4 != 0) {
    return false;
  }
  if (!fits(a.value, a.head_dim, es) || !fits(a.gate, a.head_dim, es) ||
      !fits(a.out, (a.heads - 1) * a.out.stride[2] + a.head_dim, es) || a.out.stride[2] < 0) {
    return false;
  }
  if (a.phase_mode == M3_PHASE_GIVEN &&
      (a.phase.stride[3] < 0 || !fits(a.phase, (a.num_angles - 1) * a.phase.stride[3] + 1, 4))) {
    return false;
  }
  g.out_base = static_cast<const char*>(a.out.ptr);
  g.out_b = a.out.stride[0] * es;
  g.out_t = static_cast<int>(a.out.stride[1] * es);
  g.out_h = static_cast<int>(a.out.stride[2] * es);
  g.out_o0 = 0;
  return true;
}

template <typename T, int R, bool FULL, bool SHAPE = false, bool SO = false, bool LO = false>
static int launch_kernel(const m3_scan_args& a, const ScanGeom& g, const float* prep, dim3 grid,
                         dim3 block, hipStream_t stream) {
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&scan_kernel<T, R, FULL, SHAPE, SO, LO>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       Layout<T>::BYTES);
    if (e != hipSuccess) {
      return fail(M3_ELAUNCH, "m3_scan_fwd: hipFuncSetAttribute: %s", hipGetErrorString(e));
    }
    attr_set = true;
  }
  hipLaunchKernelGGL((scan_kernel<T, R, FULL, SHAPE, SO, LO>), grid, block, Layout<T>::BYTES, stream,
                     a, g, prep);
  return check_launch("m3_scan_fwd");
}

// One pass: the prep kernel (unless `run_prep` is false: its workspace already holds this
// geometry's results) and the scan kernel over `split`'s segments (one per batch row without).
// `form16`: the call's (form16_of, -1 without the 16-wave kernel; a pass of a split call has the
// call's own). `state_only`: the caller needs only the end state, decay, last k and phase block sums (the
// outputs are not written where the kernel has a state-only form).
struct Split {
  int segs, seg_len, last_only;
};

template <typename T, int R>
static int launch_pass(const m3_scan_args& a, hipStream_t stream, bool run_prep, int form16,
                       const Split* split = nullptr, bool state_only = false) {
  ScanGeom g = make_geom<T>(a, form16);
  const size_t need = ws_layout(a, g, g.form16);
  if (split != nullptr) {
    g.segs = split->segs;
    g.seg_len = split->seg_len;
    g.last_only = split->last_only;
    g.xcd_map = static_cast<int64_t>(a.batch) * g.segs * a.heads % 8 == 0;
  }
  static_assert(Layout<T>::BYTES <= 160 * 1024, "LDS layout exceeds 160 KiB");
  const float* prep = nullptr;
  if (need > 0) {
    if (a.workspace == nullptr || a.workspace_bytes < need || !aligned16(a.workspace)) {
      return fail(M3_EWORKSPACE, "m3_scan_fwd: needs a 16-byte aligned workspace of %zu bytes",
                  need);
    }
    prep = static_cast<const float*>(a.workspace);
    const int64_t tokens = static_cast<int64_t>(a.batch) * a.length;
    const int64_t nrow = g.ws_norm >= 0 || g.ws_qk >= 0 ? tokens * 2 * a.groups * a.rank : 0;
    const int64_t ang = g.ws_ang >= 0 ? static_cast<int64_t>(a.batch) * g.L4 * a.num_angles * 4 : 0;
    // scalar-block workgroups: one per sub-chunk and group of heads. A call of many sub-chunks
    // fills the GPU with all its heads in one group (8 heads each there, 4 times the workgroups,
    // took 33 -> 44 us at 1024 sub-chunks); one of few is a chain of one workgroup's loads and
    // scans, which groups of 8 heads shorten (28 sub-chunks of 64 heads: prep 15.5 -> 13.0 us)
    const int64_t subs = static_cast<int64_t>(a.batch) * g.nsub;
    const int head_groups = (a.heads + 31) / 32 * subs < 256 ? (a.heads + 7) / 8 : 1;
    const int64_t blocks = subs * head_groups;
    if (nrow >= INT32_MAX || ang >= INT32_MAX || blocks >= INT32_MAX || tokens >= INT32_MAX) {
      return fail(M3_EUNSUPPORTED, "m3_scan_fwd: too many tokens for one launch");
    }
    constexpr int kNormRows = norm_rows<T, R>();
    const int64_t nb_norm = (nrow + 16 * kNormRows - 1) / (16 * kNormRows);
    const int64_t nb_ang = (ang / 4 + 256 * kAngQuads - 1) / (256 * kAngQuads), nb_sc = blocks;
    if (run_prep && nb_norm + nb_ang + nb_sc > 0) {
      const dim3 pgrid(static_cast<unsigned>(nb_norm + nb_ang + nb_sc)), pblock(256);
      auto launch_prep = [&](auto lo) {
        hipLaunchKernelGGL((prep_kernel<T, R, decltype(lo)::value>), pgrid, pblock, 0, stream, a, g,
                           static_cast<float*>(a.workspace), static_cast<int>(nb_norm),
                           static_cast<int>(nb_ang), head_groups);
      };
      if (g.lo) {
        launch_prep(std::true_type{});
      } else {
        launch_prep(std::false_type{});
      }
      int rc = check_launch("m3_scan_fwd (prep)");
      if (rc != M3_OK) return rc;
    }
  }
  if constexpr (sizeof(T) == 2) {
    if (g.form16 >= 0) return launch_scan16<T>(a, g, prep, state_only, stream);
  }
  const dim3 grid(static_cast<unsigned>(a.batch) * g.segs * a.heads), block(kThreads);
  if constexpr (sizeof(T) == 4) {
    if (full_shape(a, g, R) && prep != nullptr) {
      if (state_only) return launch_kernel<T, R, true, false, true>(a, g, prep, grid, block, stream);
      return launch_kernel<T, R, true>(a, g, prep, grid, block, stream);
    }
    if (prep != nullptr && model_shape(a, g, static_cast<int>(sizeof(T)))) {
      if (state_only) return launch_kernel<T, R, false, true, true>(a, g, prep, grid, block, stream);
      return launch_kernel<T, R, false, true>(a, g, prep, grid, block, stream);
    }
    if (g.lo) {
      if (state_only) return launch_kernel<T, R, false, false, true, true>(a, g, prep, grid, block, stream);
      return launch_kernel<T, R, false, false, false, true>(a, g, prep, grid, block, stream);
    }
    if (state_only) return launch_kernel<T, R, false, false, true>(a, g, prep, grid, block, stream);
  }
  return launch_kernel<T, R, false>(a, g, prep, grid, block, stream);
}

// Sub-chunk length of a call's geometry.
static int sub_chunk_tokens(const m3_scan_args& a) {
  ScanGeom g{};
  ws_layout(a, g, -1);
  return g.tok;
}

// Segments a call's sequence is split into (-1: an explicit request that cannot be met) and their
// length: a multiple of the sub-chunk, and of the 64-token phase blocks with angle increments; the
// last segment may be shorter.
//
// Automatic (segments == 0): the G of least estimated time. With one workgroup per (b, h,
// segment), a pass takes ceil(B H G c / 256) rounds over the 256 CUs (c calls of this shape
// sharing the GPU, 1 alone), each of the segment's sub-chunks plus a prologue. In units of a
// sub-chunk (2.7 us): the state-only first pass takes kStateOnly of the second, a
// workgroup's start 3 (without phases less), the split's extra launches and composition kCompose, kPerSeg per segment and kWalk per 64-token block
// walked. A further segment is a serial step of the composition, so more than a few must be
// longer: 16-bit segments of 4 sub-chunks up to 8 segments, else 8; FP32's (three times as long a
// sub-chunk) 2 up to 16, else 4. Measured (bf16, angle increments, graph-timed, us):
//   1 x 1792, 64 heads:  unsplit 91, G = 2 93, 4 71, 7 87     1 x 1792, 32 heads: 90; 4 67, 7 59, 14 73
//   1 x 8192, 32 heads:  348; 4 170, 8 110, 16 124            3 x 3072, 24 heads: 144; 2 138, 3 109, 6 122
//   1 x 61440, 24 heads: 2528; 8 596, 10 500, 16 609, 32 506  4 x 2048, 32 heads: 104; 2 112
//   1 x 512, 64 heads:   38; 2 52, 4 52                       FP32 2 x 1024, 8 heads: 240; 4 149, 8 100, 16 84
//
// A count that does not divide the sequence is taken back as an explicit request only where it is
// the choice for one of 1 .. kOwnCalls concurrent calls; for more calls the choice is among the
// counts that divide it, which every request may name.
constexpr int kOwnCalls = 4;
constexpr double kStateOnly = 0.53, kCompose = 4.5, kPerSeg = 0.11, kWalk = 0.02;

struct Segments {
  int count, len;
};

static Segments cut(int64_t len, int64_t unit, int64_t count) {
  const int64_t ls = (len + count * unit - 1) / (count * unit) * unit;
  return Segments{static_cast<int>((len + ls - 1) / ls), static_cast<int>(ls)};
}

// Whether `count` segments divide the sequence (into whole phase blocks with angle increments).
static bool divides(const m3_scan_args& a, int64_t count) {
  return a.length % (count * (a.phase_mode == M3_PHASE_ANGLES ? 64 : 1)) == 0;
}

static Segments auto_segments(const m3_scan_args& a, int64_t unit, int concurrent) {
  const int64_t tok = sub_chunk_tokens(a), len = a.length;
  const int64_t bh = static_cast<int64_t>(a.batch) * a.heads, bhc = bh * concurrent;
  auto rounds = [&](int64_t n) { return static_cast<double>((bhc * n + 255) / 256); };
  const double walk = a.phase_mode == M3_PHASE_ANGLES ? kWalk * static_cast<double>(len / 64) : 0.0;
  const bool f32 = a.act_dtype == M3_F32;
  const double prologue = a.phase_mode == M3_PHASE_NONE ? 0.8 : 3.0;
  Segments best = cut(len, unit, 1);
  double best_cost = 0.95 * rounds(1) * (prologue + static_cast<double>((len + tok - 1) / tok));
  for (int n = 2; n <= kMaxSegments && bh * n <= INT32_MAX; ++n) {
    const Segments s = cut(len, unit, n);
    const int shortest = f32 ? (n <= 16 ? 2 : 4) : (n <= 8 ? 4 : 8);
    if (s.len < shortest * tok) break;
    if (s.count != n || (concurrent > kOwnCalls && !divides(a, n))) continue;
    const double cost = rounds(n) * (2 * prologue + (1.0 + kStateOnly) * static_cast<double>(s.len / tok)) +
                        kCompose + kPerSeg * n + walk;
    if (cost < best_cost * (1.0 - 1e-9)) {
      best = s;
      best_cost = cost;
    }
  }
  return best;
}

// The shapes the chunked MFMA kernels tile: up to 128 columns, 64 values and 32 angles at ranks 1,
// 2, 4 and 8, with d_state a power of 2; in FP32 also any other, with the MIMO rotation where its
// pairs lie whole 8-column lanes apart (d_state 96, 4 x 1500 tokens, 16 heads: 21.7 ms on the
// recurrent scan, 216 us here); and the 16-wave kernel's calls at every d_state it takes. Others
// take the recurrent scan (rscan.hip), and so does every d_state that is no power of 2 with `rows`
// false (the least workspace), and one token, its whole call one kernel there (31 us with the
// Python host, 36 as prep and scan; 4 tokens 63 and 36).
static bool tiled_shape(const m3_scan_args& a, bool rows = true) {
  const bool fits = a.d_state >= 4 && a.d_state <= kNPad && a.head_dim <= kPPad &&
                    a.num_angles <= kSMax &&
                    (a.rank == 1 || a.rank == 2 || a.rank == 4 || a.rank == 8);
  if (fits && pow2(a.d_state)) return true;
  if (a.length == 1) return false;
  if (fits && rows && a.act_dtype == M3_F32 && a.q.ptr != nullptr &&
      (a.phase_mode == M3_PHASE_NONE || a.mimo_rotation == 0 || a.d_state % 16 == 0)) {
    return true;
  }
  return rows && form16_of(a, true) >= 0;
}

static Segments segments_for(const m3_scan_args& a, int concurrent = 1) {
  const int64_t len = a.length;
  const Segments one{1, static_cast<int>((len > 0 ? len + 63 : 64) / 64 * 64)};
  if (!tiled_shape(a)) return a.segments > 1 ? Segments{-1, 0} : one;
  if (a.segments == 1 || len <= 0 || a.batch <= 0) return one;
  if (a.segments < 0) return Segments{-1, 0};
  const int64_t unit = a.phase_mode == M3_PHASE_ANGLES ? 64 : sub_chunk_tokens(a);
  if (a.segments == 0) return auto_segments(a, unit, concurrent > 1 ? concurrent : 1);
  // an explicit count divides the sequence (its segments are rounded up to whole sub-chunks: of a
  // count above what that leaves, fewer run), or is the library's own choice (m3_scan_segments),
  // whose last segment may be shorter
  if (a.segments <= kMaxSegments && static_cast<int64_t>(a.batch) * a.heads * a.segments <= INT32_MAX) {
    if (divides(a, a.segments)) return cut(len, unit, a.segments);
    for (int c = 1; c <= kOwnCalls; ++c) {
      const Segments s = auto_segments(a, unit, c);
      if (s.count == a.segments) return s;
    }
  }
  return Segments{-1, 0};
}

static m3_tensor contiguous(void* p, int dtype, std::initializer_list<int64_t> dims) {
  m3_tensor t{};
  t.ptr = p;
  t.dtype = dtype;
  int64_t st = 1;
  const int nd = static_cast<int>(dims.size());
  for (int i = nd - 1; i >= 0; --i) {
    t.stride[i] = st;
    st *= dims.begin()[i];
  }
  return t;
}

// Byte offsets of the segment buffers, after the prep region.
struct SegPlan {
  size_t prep_bytes, total_bytes;
  size_t o_state, o_decay, o_blk, o_k, o_in_state, o_in_phase;
};

static SegPlan plan_segments(const m3_scan_args& a, const Segments& s, bool rows) {
  SegPlan sp{};
  ScanGeom g{};
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  sp.prep_bytes = up(ws_layout(a, g, form16_of(a, rows)));
  const size_t es = a.act_dtype == M3_F32 ? 4 : 2;
  const size_t pairs = static_cast<size_t>(a.batch) * a.heads, segs = pairs * s.count;
  size_t off = sp.prep_bytes;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off += up(bytes);
    return o;
  };
  const size_t PN = static_cast<size_t>(a.head_dim) * a.d_state;
  sp.o_state = take(segs * PN * 4);
  sp.o_decay = take(segs * 4);
  sp.o_blk = take(pairs * ((a.length + 63) / 64) * a.num_angles * 4);
  sp.o_k = take(segs * a.rank * a.d_state * es);
  sp.o_in_state = take(segs * PN * 4);
  sp.o_in_phase = take(segs * a.num_angles * 4);
  sp.total_bytes = off;
  return sp;
}

// The segmented scan: pass 1 (prep + scan of every segment from zero), the composition, pass 2
// (scan of every segment from its true start; prep's results are the same and are reused).
template <typename T, int R>
static int launch_segmented(const m3_scan_args& a, const Segments& s, bool rows,
                            hipStream_t stream) {
  const SegPlan sp = plan_segments(a, s, rows);
  if (a.workspace == nullptr || a.workspace_bytes < sp.total_bytes || !aligned16(a.workspace)) {
    return fail(M3_EWORKSPACE, "m3_scan_fwd: needs a 16-byte aligned workspace of %zu bytes",
                sp.total_bytes);
  }
  char* ws = static_cast<char*>(a.workspace);
  const int G = s.count;
  const int64_t B = a.batch, BG = B * G, H = a.heads, P = a.head_dim, N = a.d_state;
  const int64_t S = a.num_angles;
  const bool angles = a.phase_mode == M3_PHASE_ANGLES;
  SegGeom sg{};
  sg.G = G;
  sg.Ls = s.len;
  sg.nblk = (a.length + 63) / 64;
  sg.seg_state = reinterpret_cast<float*>(ws + sp.o_state);
  sg.seg_decay = reinterpret_cast<float*>(ws + sp.o_decay);
  sg.seg_blk = reinterpret_cast<float*>(ws + sp.o_blk);
  sg.seg_k = ws + sp.o_k;
  sg.in_state = reinterpret_cast<float*>(ws + sp.o_in_state);
  sg.in_phase = reinterpret_cast<float*>(ws + sp.o_in_phase);

  m3_scan_args a1 = a;
  a1.workspace_bytes = sp.prep_bytes;
  a1.initial_state = m3_tensor{};
  a1.initial_phase = m3_tensor{};
  a1.initial_k = m3_tensor{};
  a1.initial_value = m3_tensor{};
  a1.final_state = contiguous(sg.seg_state, M3_F32, {BG, H, P, N});
  a1.final_decay = contiguous(sg.seg_decay, M3_F32, {BG, H});
  a1.final_phase = m3_tensor{};
  a1.block_phase = angles ? contiguous(sg.seg_blk, M3_F32, {B, H, sg.nblk, S}) : m3_tensor{};
  a1.final_k = contiguous(sg.seg_k, a.act_dtype, {BG, H, R, N});
  const Split first{G, s.len, 0}, second{G, s.len, 1};
  const int form16 = form16_of(a, rows);
  int rc = launch_pass<T, R>(a1, stream, true, form16, &first, /*state_only=*/true);
  if (rc != M3_OK) return rc;

  // at most kMaxSegments x kSMax + 3 kMaxSegments floats: within the default 64 KiB
  const size_t clds = compose_lds_bytes(G, a.num_angles);
  static_assert(sizeof(float) * (kMaxSegments * kSMax + 3 * kMaxSegments) <= 65536,
                "compose_kernel's LDS fits the default limit");
  const unsigned row_groups = static_cast<unsigned>((P + kCompRows - 1) / kCompRows);
  hipLaunchKernelGGL((compose_kernel<T, R>),
                     dim3(static_cast<unsigned>(a.batch) * a.heads * row_groups),
                     dim3(kCompBlock), clds, stream, a, sg);
  rc = check_launch("m3_scan_fwd (compose)");
  if (rc != M3_OK) return rc;

  m3_scan_args a2 = a;
  a2.workspace_bytes = sp.prep_bytes;
  a2.initial_state = contiguous(sg.in_state, M3_F32, {BG, H, P, N});
  a2.initial_phase = angles ? contiguous(sg.in_phase, M3_F32, {BG, H, S}) : m3_tensor{};
  a2.initial_k = m3_tensor{};  // (in in_state)
  a2.initial_value = m3_tensor{};
  a2.final_decay = m3_tensor{};  // compose_kernel's
  return launch_pass<T, R>(a2, stream, false, form16, &second);
}

template <typename T, int R>
static int launch_scan_r(const m3_scan_args& a, bool rows, hipStream_t stream) {
  const Segments s = segments_for(a);
  if (s.count < 0) {
    return fail(M3_EUNSUPPORTED,
                "m3_scan_fwd: %d segments: a request is 1 < segments <= 256 dividing L (into whole "
                "64-token blocks with angle phases), or a count m3_scan_segments gave",
                a.segments);
  }
  if (s.count > 1) return launch_segmented<T, R>(a, s, rows, stream);
  return launch_pass<T, R>(a, stream, true, form16_of(a, rows));
}

template <typename T>
static int launch_scan(const m3_scan_args& a, bool rows, hipStream_t stream) {
  switch (a.rank) {
    case 1: return launch_scan_r<T, 1>(a, rows, stream);
    case 2: return launch_scan_r<T, 2>(a, rows, stream);
    case 4: return launch_scan_r<T, 4>(a, rows, stream);
    case 8: return launch_scan_r<T, 8>(a, rows, stream);
    default: return fail(M3_EUNSUPPORTED, "m3_scan_fwd: rank %d not in {1, 2, 4, 8}", a.rank);
  }
}

// A per-token tensor may run backwards (stride[1] < 0: token t at ptr + t * stride[1]; the
// reverse direction of a bidirectional layer reads the forward projection this way); the
// other checks see the forward stride.
static int check_token_tensor(const m3_tensor& t, const char* name, int dims, int64_t inner,
                              bool required, int dtype) {
  m3_tensor f = t;
  if (f.stride[1] < 0) f.stride[1] = -f.stride[1];
  return check_tensor(f, name, dims, inner, required, dtype);
}

static int validate_scan(const m3_scan_args& a) {
  if (a.batch < 0 || a.length < 0 || a.heads <= 0 || a.groups <= 0 || a.rank <= 0 ||
      a.d_state <= 0 || a.head_dim <= 0 || a.num_angles < 0) {
    return fail(M3_EINVAL, "m3_scan_fwd: invalid dimensions");
  }
  if (a.heads % a.groups != 0) return fail(M3_EINVAL, "m3_scan_fwd: heads %% groups != 0");
  if (!valid_dtype(a.act_dtype)) return fail(M3_EINVAL, "m3_scan_fwd: invalid act_dtype");
  if (a.d_state < 4) return fail(M3_EUNSUPPORTED, "m3_scan_fwd: d_state %d < 4", a.d_state);
  if (!tiled_shape(a) && !rscan_fits(a)) {
    return fail(M3_EUNSUPPORTED,
                "m3_scan_fwd: rank %d, d_state %d, head_dim %d, %d angles: the recurrent scan's "
                "per-token q / k / value vectors exceed 160 KiB of LDS",
                a.rank, a.d_state, a.head_dim, a.num_angles);
  }
  if (!tiled_shape(a) && a.segments > 1) {
    return fail(M3_EUNSUPPORTED, "m3_scan_fwd: segments > 1 need a shape the MFMA kernel tiles");
  }
  if (a.phase_mode < M3_PHASE_NONE || a.phase_mode > M3_PHASE_ANGLES) {
    return fail(M3_EINVAL, "m3_scan_fwd: invalid phase_mode");
  }
  if (a.phase_mode != M3_PHASE_NONE &&
      (a.mimo_rotation ? 4 * a.num_angles != a.d_state : 2 * a.num_angles > a.d_state)) {
    return fail(M3_EUNSUPPORTED, "m3_scan_fwd: num_angles %d does not fit d_state %d (mimo=%d)",
                a.num_angles, a.d_state, a.mimo_rotation);
  }
  const int act = a.act_dtype, N = a.d_state, P = a.head_dim;
  const bool angles = a.phase_mode == M3_PHASE_ANGLES;
  int rc;
  if ((rc = check_token_tensor(a.q, "q", 5, N, true, act)) ||
      (rc = check_token_tensor(a.k, "k", 5, N, true, act)) ||
      (rc = check_tensor(a.q_norm_w, "q_norm_w", 1, N, false, -1)) ||
      (rc = check_tensor(a.k_norm_w, "k_norm_w", 1, N, a.q_norm_w.ptr != nullptr, -1)) ||
      (rc = check_tensor(a.q_bias, "q_bias", 3, N, false, -1)) ||
      (rc = check_tensor(a.k_bias, "k_bias", 3, N, a.q_bias.ptr != nullptr, -1)) ||
      (rc = check_token_tensor(a.value, "value", 4, P, true, act)) ||
      (rc = check_token_tensor(a.gate, "gate", 4, P, true, act)) ||
      (rc = check_token_tensor(a.dt, "dt", 3, 1, true, -1)) ||
      (rc = check_token_tensor(a.a, "a", 3, 1, true, -1)) ||
      (rc = check_tensor(a.dt_bias, "dt_bias", 1, 1, a.raw_dt != 0, -1)) ||
      (rc = check_token_tensor(a.trap, "trap", 3, 1, true, -1)) ||
      (rc = check_token_tensor(a.phase, "phase", angles ? 3 : 4, 1,
                               a.phase_mode != M3_PHASE_NONE,
                               a.phase_mode == M3_PHASE_GIVEN ? M3_F32 : -1)) ||
      (rc = check_tensor(a.initial_phase, "initial_phase", 3, 1, false, M3_F32)) ||
      (rc = check_tensor(a.D, "D", 1, 1, true, -1)) ||
      (rc = check_tensor(a.mimo_x, "mimo_x", 3, P, a.rank > 1, -1)) ||
      (rc = check_tensor(a.mimo_z, "mimo_z", 3, P, a.rank > 1, -1)) ||
      (rc = check_tensor(a.mimo_out, "mimo_out", 3, P, a.rank > 1, -1)) ||
      (rc = check_tensor(a.initial_state, "initial_state", 4, N, false, M3_F32)) ||
      (rc = check_tensor(a.initial_k, "initial_k", 4, N, false, act)) ||
      (rc = check_tensor(a.initial_value, "initial_value", 3, P, a.initial_k.ptr != nullptr,
                         act)) ||
      (rc = check_token_tensor(a.out, "out", 4, P, true, act)) ||
      (rc = check_tensor(a.final_state, "final_state", 4, N, true, M3_F32)) ||
      (rc = check_tensor(a.final_phase, "final_phase", 3, 1, false, M3_F32)) ||
      (rc = check_tensor(a.final_decay, "final_decay", 2, 1, false, M3_F32)) ||
      (rc = check_tensor(a.block_phase, "block_phase", 4, 1, false, M3_F32)) ||
      (rc = check_tensor(a.final_k, "final_k", 4, N, false, act))) {
    return rc;
  }
  if ((a.q_norm_w.ptr == nullptr) != (a.k_norm_w.ptr == nullptr) ||
      (a.q_bias.ptr == nullptr) != (a.k_bias.ptr == nullptr)) {
    return fail(M3_EINVAL, "m3_scan_fwd: q/k norm weights and biases come in pairs");
  }
  // per-token offsets within one batch row are 32-bit in the kernel
  const int64_t lim = INT32_MAX;
  const m3_tensor* per_token[] = {&a.q, &a.k, &a.value, &a.gate, &a.dt, &a.a, &a.trap, &a.out};
  for (const m3_tensor* t : per_token) {
    if (static_cast<int64_t>(a.length) * (t->stride[1] < 0 ? -t->stride[1] : t->stride[1]) >=
        lim) {
      return fail(M3_EUNSUPPORTED, "m3_scan_fwd: a batch row exceeds 2^31 elements");
    }
  }
  if (a.phase_mode != M3_PHASE_NONE &&
      static_cast<int64_t>(a.length) * (a.phase.stride[1] < 0 ? -a.phase.stride[1]
                                                               : a.phase.stride[1]) >= lim) {
    return fail(M3_EUNSUPPORTED, "m3_scan_fwd: a batch row of phase exceeds 2^31 elements");
  }
  if (a.length > 1) {
    const bool back = a.q.stride[1] < 0;
    const m3_tensor* ts[] = {&a.k, &a.value, &a.gate, &a.dt, &a.a, &a.trap, &a.out};
    bool same = true;
    for (const m3_tensor* t : ts) same = same && ((t->stride[1] < 0) == back);
    if (a.phase_mode != M3_PHASE_NONE) same = same && ((a.phase.stride[1] < 0) == back);
    if (!same) {
      return fail(M3_EINVAL, "m3_scan_fwd: per-token tensors must all run the same way");
    }
  }
  if ((a.final_phase.ptr != nullptr || a.block_phase.ptr != nullptr) && !angles) {
    return fail(M3_EINVAL, "m3_scan_fwd: final_phase / block_phase need phase_mode ANGLES");
  }
  return M3_OK;
}

size_t scan_need(const m3_scan_args& a, bool rows) {
  if (!tiled_shape(a, rows)) return 0;  // the recurrent scan needs no workspace
  const Segments s = segments_for(a);
  if (s.count > 1) return plan_segments(a, s, rows).total_bytes;
  ScanGeom g{};
  return ws_layout(a, g, form16_of(a, rows));
}

int scan_run(const m3_scan_args& a, bool rows, hipStream_t stream) {
  int rc = validate_scan(a);
  if (rc != M3_OK) return rc;
  if (a.batch == 0) return M3_OK;
  if (!tiled_shape(a, rows)) {
    if (!rscan_fits(a)) return fail(M3_EUNSUPPORTED, "m3_scan_fwd: no kernel without a workspace");
    return launch_recurrent_scan(a, stream);
  }
  switch (a.act_dtype) {
    case M3_F32: return launch_scan<float>(a, rows, stream);
    case M3_BF16: return launch_scan<__bf16>(a, rows, stream);
    default: return launch_scan<_Float16>(a, rows, stream);
  }
}

}  // namespace m3

extern "C" int m3_scan_workspace_size(const m3_scan_args* args, size_t* bytes) {
  m3::clear_error();
  if (args == nullptr || bytes == nullptr) {
    return m3::fail(M3_EINVAL, "m3_scan_workspace_size: NULL argument");
  }
  *bytes = m3::scan_need(*args, true);
  return M3_OK;
}

extern "C" int m3_scan_segments(const m3_scan_args* args, int concurrent_calls,
                                int* segments) {
  m3::clear_error();
  if (args == nullptr || segments == nullptr) {
    return m3::fail(M3_EINVAL, "m3_scan_segments: NULL argument");
  }
  if (concurrent_calls < 1) {
    return m3::fail(M3_EINVAL, "m3_scan_segments: concurrent_calls must be at least 1");
  }
  const int G = m3::segments_for(*args, concurrent_calls).count;
  if (G < 0) {
    return m3::fail(M3_EUNSUPPORTED, "m3_scan_segments: the requested %d segments cannot be met",
                    args->segments);
  }
  // an explicit request is answered with itself (it can be passed back as it is)
  *segments = args->segments > 0 ? args->segments : G;
  return M3_OK;
}

extern "C" int m3_scan_fwd(const m3_scan_args* args, hipStream_t stream) {
  m3::clear_error();
  if (args == nullptr) return m3::fail(M3_EINVAL, "m3_scan_fwd: args is NULL");
  const int rc = m3::scan_run(*args, true, stream);
  if (rc != M3_EWORKSPACE) return rc;
  // (nothing was launched) less workspace than the query's answer: the routes that need least, where
  // it covers them
  const size_t least = m3::scan_need(*args, false);
  const bool given = args->workspace != nullptr && m3::aligned16(args->workspace);
  if (least > 0 && (!given || args->workspace_bytes < least)) return rc;
  m3::clear_error();
  return m3::scan_run(*args, false, stream);
}
