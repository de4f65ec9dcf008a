// Device helpers, MFMA policies and launch geometry shared by the chunked scan kernels
// (scan.hip, scan16_kernel.hpp).
#pragma once

#include "m3_common.hpp"
#include "m3_host.hpp"
#include "m3_math.h"

#include <type_traits>

namespace m3 {

constexpr int kThreads = 512;
constexpr int kWaves = 8;
constexpr int kTiles = 4;  // 16x16 state tiles per wave (N_pad * P_pad <= 128 * 64)

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// MFMA policy per activation type: 16-bit types use 16x16x32 (K = 32, 8 elements per lane),
// FP32 uses 16x16x4 (K = 4, one element per lane). ROWS is the sub-chunk height.
template <typename T> struct Mma;
template <> struct Mma<__bf16> {
  static constexpr int ROWS = 64, PAD = 8;
  typedef bf16x8 v8;
  typedef bf16x4 v4;
  typedef bf16x2 v2;
  static __device__ __forceinline__ f4 mma(v8 a, v8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma<_Float16> {
  static constexpr int ROWS = 64, PAD = 8;
  typedef f16x8 v8;
  typedef f16x4 v4;
  typedef f16x2 v2;
  static __device__ __forceinline__ f4 mma(v8 a, v8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma<float> {
  static constexpr int ROWS = 32, PAD = 4;
  typedef float v8;  // unused: FP32 operands are single elements
  typedef f4 v4;
  typedef f32x2 v2;
  static __device__ __forceinline__ f4 mma(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// Compile-time LDS layout. Operand tiles are padded to N = 128 and P = 64 (the largest shapes
// the kernel takes; every Mamba3 configuration has P <= 64), so every offset and loop bound is a
// constant; smaller shapes run on zero padding.
constexpr int kNPad = 128, kPPad = 64, kSMax = 32, kRMax = 8;
constexpr int kNT = kNPad / 16, kPT = kPPad / 16;  // 16-row tiles of N and P

template <typename T> struct Layout {
  static constexpr int ROWS = Mma<T>::ROWS, PAD = Mma<T>::PAD, ES = sizeof(T);
  static constexpr int LQ = kNPad + PAD;   // row stride (elements) of Qs, Ks, Sb
  static constexpr int LR = ROWS + PAD;    // row stride (elements) of KT, VT
  static constexpr int LP = kPPad + PAD;   // row stride (elements) of VR, ZR
  static constexpr int al(int x) { return (x + 15) / 16 * 16; }
  static constexpr int QS = 0;
  static constexpr int KS = al(QS + ROWS * LQ * ES);
  static constexpr int KT = al(KS + ROWS * LQ * ES);
  static constexpr int VT = al(KT + kNPad * LR * ES);
  static constexpr int VR = al(VT + kPPad * LR * ES);
  static constexpr int ZR = al(VR + ROWS * LP * ES);
  static constexpr int SB = al(ZR + ROWS * LP * ES);
  static constexpr int FB = al(SB + kPPad * LQ * ES);
  // float scratch, offsets in floats from FB, sized for TM = ROWS tokens (rank 1): two side
  // blocks alternating (a sub-chunk's scalar block, ScBlk, then the (q, k) RMSNorm factors of
  // its rows), the angle tile, two cos / sin tables ([token][angle][cos, sin], token stride CST
  // for 16-byte aligned rows)
  static constexpr int TM = ROWS;
  static constexpr int SCB = 5 * TM + 8 + 2 * ROWS, SC0 = 0;
  static constexpr int ANG = SC0 + 2 * SCB;  // [TM / 4][kSMax][4]
  static constexpr int CST = 2 * kSMax + 4, CSB = TM * CST;
  static constexpr int CS0 = ANG + TM * kSMax, PBASE = CS0 + 2 * CSB;
  static constexpr int POFF = PBASE + kSMax, MX = POFF + kSMax, MZ = MX + kRMax * kPPad;
  static constexpr int MO = MZ + kRMax * kPPad;
  static constexpr int BYTES = FB + 4 * (MO + kRMax * kPPad);
};

// Per-token scalar block of one sub-chunk of TOK tokens (floats, token-indexed arrays): dt, the
// within-chunk cumsum of adt, the exp-trapezoid scale, gamma, scale * decay to the end of the
// token's 16-row tile; then the cumsum at each tile end, exp of the last cumsum and the last
// cumsum itself. LO (d_state no power of 2): the cumsum counts a step below kDecayLow as that, and
// DEC holds the sum of the steps as they are. The prep pass writes them; the scan copies them to LDS (and takes exp(cum) and
// scale * exp(cum_last - cum) from them itself, an exp per lane).
template <int TOK> struct ScBlk {
  static constexpr int DTV = 0, CUM = TOK, SCL = 2 * TOK, GAM = 3 * TOK, BSC = 4 * TOK;
  static constexpr int CEND = 5 * TOK, ECL = 5 * TOK + 4, CL = 5 * TOK + 5;
  static constexpr int DEC = 5 * TOK + 6;
  static constexpr int SIZE = 5 * TOK + 8;
};

// exp of it is 0 in FP32. A step that resets the state (adt = -inf, or any value far below this)
// makes differences of a plain cumsum NaN, or loses the steps after it to the sum's rounding; the
// recurrent scan, where the LO calls came from, multiplies by exp(adt) and takes it as it is.
constexpr float kDecayLow = -104.f;

// Per-launch values shared by host and device.
struct ScanGeom {
  int xcd_map;           // 1: map blocks so each XCD holds consecutive (b, h)
  int vec_qk, vec_vz;    // 1: q/k rows and v/z rows may be loaded with 16 / 8-byte vectors
  int vec_nw;            // 1: both norm weights unit-stride and 8-byte aligned (4-element loads)
  // prep workspace, float offsets of its regions (-1: absent): RMSNorm factors [B][L][G*R][2]
  // (q, k), pi tanh(angle) [B][L4][S][4] (4 consecutive tokens of one angle together, L4 =
  // ceil(L / 4)), scalar blocks [B*H][nsub][scw] of `tok`-token sub-chunks
  int64_t ws_norm, ws_ang, ws_sc;
  int L4, tok, nsub, scw;
  // the call's split: segments per batch row and tokens per segment (the last may be shorter; a
  // multiple of `tok`, and of 64 with angle increments). One workgroup per (batch, segment,
  // head); the per-token tensors and prep's results stay the whole row's, the initial_* tensors
  // are per segment. last_only: the final_* outputs are per batch row and the last segment's
  // alone (pass 2), else per segment (pass 1).
  int segs, seg_len, last_only;
  int ws_bytes;  // workspace bytes when below 2^31 (the projection form addresses it in 32 bits)
  // the 16-wave kernel (scan16_kernel): its form (Form16, -1: the call takes another kernel),
  // whether the columns are permuted into slots (the MIMO rotation), and the q / k rows [B][L][G][R][2]
  // in slot order, 128 slots in the activation dtype (forms kModel, kCopy) or d_state in FP32 (kRows),
  // after the regions above (byte offset)
  int form16, perm;
  // d_state no power of 2: the kernels that hold no value in fewer bits than the recurrent scan
  int lo;
  int64_t ws_qk;
  // projection form (the full-shape kernel): q, k, value, gate, dt, a, trap are slices of one
  // projection row; byte offsets of each slice from `proj`, the batch / token strides and the
  // group / rank / head strides of the slices, in bytes
  const char* proj;
  int64_t proj_b, out_b;
  int tok_b, o_q, o_k, o_v, o_z, o_dt, o_a, o_tr, qk_g, qk_r, vz_h, sc_h, out_t, out_h;
  // the output's physical start and the offset of logical token 0 from it (non-zero when the
  // call runs backwards: token strides < 0, logical token t at physical token L - 1 - t)
  const char* out_base;
  int out_o0;
};

__device__ __forceinline__ f4 zero4() {
  f4 z;
  z[0] = z[1] = z[2] = z[3] = 0.f;
  return z;
}

template <typename T>
__device__ __forceinline__ T* lds_t(char* base, int off) {
  return reinterpret_cast<T*>(base + off);
}

// ------------------------------------------------------------------ raw register tiles

// Activation elements held as raw bits until they are used: W8 words hold 8 elements,
// W4 words hold 4 (two 16-bit elements per word, or one FP32 element per word).
template <typename T> struct Words {
  static constexpr int W8 = sizeof(T) == 4 ? 8 : 4;
  static constexpr int W4 = sizeof(T) == 4 ? 4 : 2;
};

__device__ __forceinline__ float bits_to_f(uint32_t bits16, __bf16*) {
  return __uint_as_float(bits16 << 16);
}
__device__ __forceinline__ float bits_to_f(uint32_t bits16, _Float16*) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(bits16)));
}

template <typename T, int NW>
__device__ __forceinline__ float raw_get(const uint32_t (&w)[NW], int i) {
  if constexpr (sizeof(T) == 4) {
    return __uint_as_float(w[i]);
  } else {
    const uint32_t x = w[i >> 1];
    return bits_to_f((i & 1) ? (x >> 16) : (x & 0xffffu), static_cast<T*>(nullptr));
  }
}

template <typename T>
__device__ __forceinline__ uint32_t elem_bits(const T* p) {
  if constexpr (sizeof(T) == 4) {
    return __float_as_uint(*p);
  } else {
    return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, *p));
  }
}

// Load up to E elements (n valid, the rest zero) into raw words; one vector load when `vec`
// and all E are valid (16 bytes, or 8 bytes for four 16-bit elements).
template <typename T, int E, int NW>
__device__ __forceinline__ void load_words(uint32_t (&w)[NW], const T* p, int n, bool vec) {
  if (vec && n >= E) {
    if constexpr (NW == 2) {
      const uint2 q = *reinterpret_cast<const uint2*>(p);
      w[0] = q.x; w[1] = q.y;
    } else {
#pragma unroll
      for (int j = 0; j < NW; j += 4) {
        const uint4 q = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint32_t*>(p) + j);
        w[j] = q.x; w[j + 1] = q.y; w[j + 2] = q.z; w[j + 3] = q.w;
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < NW; ++j) w[j] = 0u;
#pragma unroll
  for (int i = 0; i < E; ++i) {
    if (i < n) {
      const uint32_t e = elem_bits(p + i);
      if constexpr (sizeof(T) == 4) {
        w[i] = e;
      } else {
        w[i >> 1] |= e << (16 * (i & 1));
      }
    }
  }
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Two values rounded to a 16-bit type (round to nearest even) and packed into one word, a
// first: one packed convert for bf16.
template <typename T>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  typedef T t2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, t2));
}

// Two adjacent activation values stored with one LDS write.
template <typename T>
__device__ __forceinline__ void st_pair(T* dst, float a, float b) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<f32x2*>(dst) = (f32x2){a, b};
  } else {
    *reinterpret_cast<uint32_t*>(dst) = pack2<T>(a, b);
  }
}

// Four adjacent activation values stored with one LDS write.
template <typename T>
__device__ __forceinline__ void st_quad(T* dst, f4 x) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<f4*>(dst) = x;
  } else {
    *reinterpret_cast<u32x2*>(dst) = (u32x2){pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3])};
  }
}

template <typename T>
__device__ __forceinline__ void st_row8(T* dst, const float* x) {
  if constexpr (sizeof(T) == 4) {
    f4 a, b;
#pragma unroll
    for (int i = 0; i < 4; ++i) { a[i] = x[i]; b[i] = x[4 + i]; }
    reinterpret_cast<f4*>(dst)[0] = a;
    reinterpret_cast<f4*>(dst)[1] = b;
  } else {
    *reinterpret_cast<u32x4*>(dst) = (u32x4){pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3]),
                                             pack2<T>(x[4], x[5]), pack2<T>(x[6], x[7])};
  }
}

// ------------------------------------------------------------------ scan

// Wave-level scans with DPP row shifts (no LDS traffic). row_shr:n = 0x110 + n; lanes whose
// source lies before their 16-lane row read 0.
template <int CTRL>
__device__ __forceinline__ float dpp_shr(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                                               CTRL, 0xf, 0xf, true));
}

// Inclusive scan within aligned segments of SEG lanes (SEG a power of 2, <= 16). For SEG = 16
// the segment is the DPP row, whose shifts already read 0 before the row's first lane (the
// same +0 the masks add), so no mask is applied.
template <int SEG>
__device__ __forceinline__ float seg_incl_scan(float x, int lane) {
  const int j = lane & (SEG - 1);
  constexpr bool ROW = SEG == 16;
  if constexpr (SEG > 1) { const float u = dpp_shr<0x111>(x); x += (ROW || j >= 1) ? u : 0.f; }
  if constexpr (SEG > 2) { const float u = dpp_shr<0x112>(x); x += (ROW || j >= 2) ? u : 0.f; }
  if constexpr (SEG > 4) { const float u = dpp_shr<0x114>(x); x += (ROW || j >= 4) ? u : 0.f; }
  if constexpr (SEG > 8) { const float u = dpp_shr<0x118>(x); x += (ROW || j >= 8) ? u : 0.f; }
  return x;
}

// Sum over each 16-lane row, in every lane of the row: DPP row rotations by 8, 4, 2 and 1.
__device__ __forceinline__ float row16_sum(float x) {
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x128,
                                                             0xf, 0xf, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x124,
                                                             0xf, 0xf, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x122,
                                                             0xf, 0xf, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x121,
                                                             0xf, 0xf, false));
  return x;
}

__device__ __forceinline__ float readlane_f(float x, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));
}

// Inclusive scan over the 64 lanes of a wave.
__device__ __forceinline__ float wave_incl_scan(float x, int lane) {
  x = seg_incl_scan<16>(x, lane);
  const float r0 = readlane_f(x, 15), r1 = readlane_f(x, 31), r2 = readlane_f(x, 47);
  const int row = lane >> 4;
  x += row >= 1 ? r0 : 0.f;
  x += row >= 2 ? r1 : 0.f;
  x += row >= 3 ? r2 : 0.f;
  return x;
}

// Transposed operand tiles ([n or p][row]) XOR-swizzle their 8-row groups by a key taken from
// the tile row (n or p) so that the column-wise stores of the staging spread over the LDS banks;
// every reader applies the same swizzle. Groups of 8 (16-bit: 16 bytes) stay contiguous.
template <int ROWS>
__device__ __forceinline__ int swz(int row, int key) {
  return row ^ (8 * (key & (ROWS / 8 - 1)));
}

// Buffer resource over `bytes` bytes from `base` (raw, stride 0): loads at offsets beyond the
// extent return zero, stores there are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), static_cast<short>(0), bytes,
                                           0x00020000);
}

// NW raw words (NW in {2, 4, 8}) from a buffer at byte offset `off`.
template <int NW>
__device__ __forceinline__ void bload_words(uint32_t (&w)[NW], __amdgpu_buffer_rsrc_t r, int off) {
  if constexpr (NW == 2) {
    const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    w[0] = v[0];
    w[1] = v[1];
  } else {
#pragma unroll
    for (int j = 0; j < NW; j += 4) {
      const u32x4 v =
          __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 4 * j, 0, 0));
      w[j] = v[0];
      w[j + 1] = v[1];
      w[j + 2] = v[2];
      w[j + 3] = v[3];
    }
  }
}

__device__ __forceinline__ float bload_f32(__amdgpu_buffer_rsrc_t r, int off) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// Four consecutive activation values stored as one vector (8 bytes for 16-bit types).
template <typename T>
__device__ __forceinline__ void bstore_quad(f4 x, __amdgpu_buffer_rsrc_t r, int off) {
  if constexpr (sizeof(T) == 4) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), r, off, 0, 0);
  } else {
    typename Mma<T>::v4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = from_f<T>(x[i]);
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, 0);
  }
}

// Column of angle `col` in the cos / sin table row of token tt. SWZ (64-token sub-chunks, 32
// angles): blocks of 4 angles are XOR-swizzled by the token's 16-token block, spreading the
// phase stage's column writes over the LDS banks, and the two angle pairs of a block swap places
// in every other token pair, so the 16-byte reads of two token rows 2 apart (136 floats: the
// same banks shifted by 8) fall into different halves of each 8-float group. A reader takes a
// block as two pairs, each at its own cs_col.
template <bool SWZ>
__device__ __forceinline__ int cs_col(int col, int tt) {
  return SWZ ? col ^ (4 * ((tt >> 4) & 3)) ^ (2 * ((tt >> 1) & 1)) : col;
}

// How a phase becomes cos and sin. kFast: the hardware functions (the phase times 1 / 2 pi in FP32:
// an error of |phase| 2^-24, for phases reduced below a few turns). The calls that came from the
// recurrent scan, which takes any given phase to full precision (LO), keep that: kFull the library's
// functions (FP32), kWide the hardware functions of the turns reduced in 64 bits (16-bit: hook form;
// the phase times 1 / 2 pi as two doubles, its product error folded in: exact to the hardware
// functions' own error below 10^20).
enum Trig { kFast, kFull, kWide };

template <Trig TR>
__device__ __forceinline__ void sincos_of(float x, float* s, float* c) {
  if constexpr (TR == kFast) {
    __sincosf(x, s, c);
  } else if constexpr (TR == kFull) {
    sincosf(x, s, c);
  } else {
    constexpr double kHi = 0x1.45f306dc9c883p-3, kLo = -0x1.6b01ec5417056p-57;  // 1 / 2 pi
    const double xd = x, t = xd * kHi;
    double r = (t - __builtin_rint(t)) + (__builtin_fma(xd, kHi, -t) + xd * kLo);
    r -= __builtin_rint(r);
    *s = __builtin_amdgcn_sinf(static_cast<float>(r));
    *c = __builtin_amdgcn_cosf(static_cast<float>(r));
  }
}

// Bounded phase (model.py:215-256) of tokens TPL pg .. TPL pg + TPL-1 of the sub-chunk at t0 for
// angle ps: fmod-reduced increments summed within 64-token blocks, an fmod-reduced carry between
// blocks, the running block sum and carry in pbase / poff; cos / sin into the table of angle ps.
template <int PG, int TPL, int CST, bool SWZ, bool EXACT, Trig TR>
__device__ __forceinline__ void phase_stage(float* tab, int ps, float* pbase, float* poff,
                                            const float* dtv, int t0, int L, int pg, int lane,
                                            bool angles, const float (&pa)[TPL], float* fph,
                                            float* fblk, int64_t blk_stride) {
  float ph[TPL];
  if (angles) {
    float x[TPL];
    float mx = 0.f;  // largest |increment| of the lane (NaN and inf reduce like any x below)
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
      x[i] = __fmul_rn(pa[i], dtv[TPL * pg + i]);  // dt is 0 past the sub-chunk's last token
      mx = fmaxf(mx, fabsf(x[i]));
    }
    // fmodf(x, 2 pi) is x itself for |x| < 2 pi (dt < 2, the usual case); the reductions are
    // chosen per wave, so no lane branches on its own elements
    float inc[TPL];
    if (__builtin_amdgcn_ballot_w64(!(mx < M3_TWO_PI_F)) == 0) {
#pragma unroll
      for (int i = 0; i < TPL; ++i) inc[i] = x[i];
    } else if (__builtin_amdgcn_ballot_w64(!(mx < 1048576.0f)) == 0) {
#pragma unroll
      for (int i = 0; i < TPL; ++i) inc[i] = m3_fmod_2pi_small(x[i]);
    } else {
#pragma unroll
      for (int i = 0; i < TPL; ++i) inc[i] = m3_fmod_2pi(x[i]);
    }
    float cpre[TPL];
    float run = 0.f;
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
      run = __fadd_rn(run, inc[i]);
      cpre[i] = run;
    }
    const float incl = seg_incl_scan<PG>(run, lane);
    // the previous lane's inclusive sum: sums of earlier tokens only (incl - run would round in
    // the later tokens of this lane's group)
    float excl = dpp_shr<0x111>(incl);
    if (pg == 0) excl = 0.f;
    float base = *pbase, off = *poff;
    if ((t0 & 63) == 0 && t0 > 0) {
      // the block that just ended: its increment sum, when asked for (block_phase)
      if (fblk != nullptr && pg == 0) fblk[((t0 >> 6) - 1) * blk_stride] = base;
      off = m3_fmod_2pi_small(__fadd_rn(off, base));
      base = 0.f;
    }
    // the final phase (token L - 1), when this sub-chunk holds it (wave-uniform test)
    const bool last = fph != nullptr && t0 <= L - 1 && L - 1 - t0 < PG * TPL;
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
      // |base|, |excl + cpre| <= 64 * 2 pi and |off| < 2 pi: within the reduction's range.
      // !EXACT (16-bit activations): sin / cos reduce the phase themselves (below 66 turns, the
      // hardware's range), a difference far below the 16-bit rounding of the rotated values.
      const float raw = __fadd_rn(__fadd_rn(base, __fadd_rn(excl, cpre[i])), off);
      ph[i] = EXACT ? m3_fmod_2pi_small(raw) : raw;
    }
    if (last) {  // one wave-uniform branch instead of a lane test per token
#pragma unroll
      for (int i = 0; i < TPL; ++i) {
        if (t0 + TPL * pg + i == L - 1) *fph = EXACT ? ph[i] : m3_fmod_2pi_small(ph[i]);
      }
    }
    if (pg == PG - 1) {
      *pbase = __fadd_rn(base, incl);
      *poff = off;
    }
  } else {
#pragma unroll
    for (int i = 0; i < TPL; ++i) ph[i] = pa[i];
  }
#pragma unroll
  for (int i = 0; i < TPL; ++i) {
    const int tt = TPL * pg + i;
    float2 v;
    sincos_of<TR>(ph[i], &v.y, &v.x);
    *reinterpret_cast<float2*>(tab + tt * CST + 2 * cs_col<SWZ>(ps, tt)) = v;
  }
}

// Where a 16-wave call's q / k rows come from (scan16_kernel.hpp).
enum Form16 { kModel, kRows, kProj, kCopy, kHook };

// The column of slot `slot`: the identity, or with the MIMO pairs (perm: S angles, columns j and
// 2S + j) their two columns side by side first, then the columns S .. 2S - 1 and 3S ..
__device__ __forceinline__ int slot_col(int slot, int perm, int S) {
  if (!perm) return slot;
  if (slot < 2 * S) return (slot >> 1) + (slot & 1) * 2 * S;
  const int u = slot - 2 * S;
  return u < S ? S + u : 2 * S + u;
}

// The 16-wave scan of a 16-bit call (scan16_kernel.hpp), prep's results in `prep`.
template <typename T>
int launch_scan16(const m3_scan_args& a, const ScanGeom& g, const float* prep, bool state_only,
                  hipStream_t stream);

}  // namespace m3
