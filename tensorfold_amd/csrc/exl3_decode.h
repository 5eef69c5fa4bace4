// EXL3 trellis decode shared by the dense linear and the routed experts: window extraction, codebooks, the
// 128-point Hadamard butterfly, and one wave's decode-and-MFMA walk over a 128-column block.
//
// A tile holds 256 values of k2/2 bits in a circular bitstream (most significant bit of each little-endian 32-bit
// word first); value p is the 16-bit window ending at bit E(p), pushed through a procedural codebook to an fp16
// value, and lands at row 2 (l % 4) + (j & 1) + 8 ((j >> 1) & 1), column l / 4 + 8 (j >> 2) of the 16 x 16 tile
// (l = p / 8, j = p % 8)  (reference: docs/recipes/exl3.md:43-63, cuda/exl3/format.py:31-110).
//
// On a 64-lane wave the B operand of v_mfma_f32_16x16x32_f16 is 32 inputs x 16 columns, 8 values a lane: lane
// (column c, quarter kq) takes, from each of two consecutive k tiles, the four stream-consecutive values
// p0 .. p0 + 3 with p0 = 8 (4 (c % 8) + kq) + 4 (c / 8).  They sit in rows {2 kq, 2 kq + 1, 2 kq + 8, 2 kq + 9} of
// column c, so the A operand reads the rotated activations at the same eight inputs and no value moves across
// lanes.  Rows of the call are MFMA rows: independent by construction.  K is split over waves and blocks as a
// function of the shape only and every sum runs in a fixed order.


#ifndef TF_EXL3_DECODE_H
#define TF_EXL3_DECODE_H

#include <hip/hip_fp16.h>

#include "tf_common.h"

namespace tf {
namespace {

constexpr float HAD_SCALE = 0.08838834764831845f;   // 1 / sqrt(128)

template <int K2>
__host__ __device__ constexpr int tile_words() {
  return 4 * K2;
}

// E(p): one past the last stream bit of value p's window
template <int K2>
__host__ __device__ constexpr int stream_end(int p) {
  return (K2 & 1) ? ((p + 1) * K2 - ((p + 1) & 1)) / 2 : (p + 1) * (K2 / 2);
}

// bit distance from value p0's window to value p0 + j's, p0 a multiple of 4
template <int K2>
__host__ __device__ constexpr int delta(int j) {
  return stream_end<K2>(j) - stream_end<K2>(0);
}

// The stored words lane (L, h) needs of a tile for its four values p0 .. p0 + 3 (p0 = 8 L + 4 h): two, or three when
// the four windows span more than 32 bits.  The first window starts 1 to 32 bits into the first word (not 0 to 31): the
// shift that lines it up is then 31 to 0 and one v_alignbit_b32 does it.  With 0 to 31 the case of no shift needed a
// select, and the compiler made it a branch around the second word's LDS read, one in every column tile: the walk
// waited on two LDS round trips in a row sixteen times a pair (that and the runs' wider loads: 8 rows through 288 experts at 4
// bits 250 -> 234 us, an MLP at 3 bits and one row 63.3 -> 59.4; a pair of k tiles is 225 vector instructions beside 16
// matrix ones at 4 bits of mcg).
template <int K2>
struct Windows {
  static constexpr int TW = tile_words<K2>(), R = 32 * TW;
  static constexpr int NW = delta<K2>(3) > 16 ? 3 : 2;
  int wi, wi1, wi2, sh;                                        // the words and the shift: the same for every tile
  __device__ __forceinline__ Windows(int L, int h) {
    const int p0 = 8 * L + 4 * h;
    // one bit before the first window, E(p0) - 16 - 1; p0 is even, p0 * K2 / 2 whole
    const int before = (stream_end<K2>(0) + p0 * K2 / 2 - 17 + R) % R;
    wi = before >> 5;
    wi1 = (wi + 1) % TW;
    wi2 = (wi + 2) % TW;
    sh = 31 - (before & 31);
  }
  __device__ __forceinline__ void load(const uint32_t* tile, uint32_t (&w)[NW]) const {
    w[0] = tile[wi];
    w[1] = tile[wi1];
    if constexpr (NW == 3) w[2] = tile[wi2];
  }
  // the 16-bit states of the four values
  __device__ __forceinline__ void states(const uint32_t (&w)[NW], uint32_t (&s)[4]) const {
    const uint32_t hi = __builtin_amdgcn_alignbit(w[0], w[1], sh);        // the stream from the first window on, 32 bits
    uint32_t lo = 0;
    if constexpr (NW == 3) lo = __builtin_amdgcn_alignbit(w[1], w[2], sh);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = delta<K2>(j);
      if (d + 16 <= 32) s[j] = (hi >> (16 - d)) & 0xFFFFu;
      else if (d < 32) s[j] = __builtin_amdgcn_alignbit(hi, lo, 48 - d) & 0xFFFFu;
      else s[j] = (lo >> (48 - d)) & 0xFFFFu;
    }
  }
};

// The hashed word of a state of the 3inst and mcg codebooks: the value is the fp16 sum of its two halves.  3inst's multiply
// and add are one v_mad_u64_u32 (2.08 ns a wave and SIMD against 1.75 each for a multiply and an add; the upper half of its
// result is not used, which the compiler must not learn): 227 vector instructions a pair of k tiles instead of 291, an MLP
// 5120 -> 17408 -> 5120 at 3 bits and one row 59.7 -> 55.9 us.
// At 5 bits and more the 64-bit results do not fit beside the windows (8 rows through experts at 6 bits spilled and took 1.4
// times as long): a multiply and an add there.
template <int CB, int K2>
__device__ __forceinline__ uint32_t code_word(uint32_t s) {
  uint32_t x;
  if constexpr (CB == 1) {
    x = s * 0xCBAC1FEDu;
  } else if constexpr (K2 >= 10) {
    x = s * 89226354u + 64248484u;
  } else {
    uint64_t wide = (uint64_t)s * 89226354u + 64248484u;
    asm("" : "+v"(wide));
    x = (uint32_t)wide;
  }
  return (x & 0x8FFF8FFFu) ^ 0x3B603B60u;
}

// (half(xa.lo) + half(xa.hi)) | (half(xb.lo) + half(xb.hi)) << 16.  The second add writes the upper half of the
// register the first one wrote and keeps the lower: two instructions for two values, where the compiler's own
// pairing pads each result and ORs them (a third).  The same IEEE add as __hadd.
__device__ __forceinline__ uint32_t half_sums(uint32_t xa, uint32_t xb) {
  uint32_t r;
  asm("v_add_f16_sdwa %0, %1, %1 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1" : "=v"(r) : "v"(xa));
  asm("v_add_f16_sdwa %0, %1, %1 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 src1_sel:WORD_1"
      : "+v"(r)
      : "v"(xb));
  return r;
}

// The mul1 values of two states, packed.  v_sad_u8 against zero adds a word's four bytes to an accumulator, its _hi
// form to the upper half; the accumulator starts as fp16 1024 in both halves (0x6400 + a sum of at most 1,020 is the fp16
// of 1024 + the sum), and one packed fp16 fma
// scales and shifts both.
__device__ __forceinline__ uint32_t mul1_pair(uint32_t sa, uint32_t sb) {
  uint32_t t = __builtin_amdgcn_sad_u8(sa * 0x83DCD12Du, 0u, 0x64006400u);
  t = __builtin_amdgcn_sad_hi_u8(sb * 0x83DCD12Du, 0u, t);
  typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;
  const f16x2_t r = __builtin_elementwise_fma(__builtin_bit_cast(f16x2_t, t), __builtin_bit_cast(f16x2_t, 0x1EEE1EEEu),
                                              __builtin_bit_cast(f16x2_t, 0xC931C931u));
  return __builtin_bit_cast(uint32_t, r);
}

// the fp16 bits of the lane's four values of one tile, as two packed words
template <int K2, int CB>
__device__ __forceinline__ void decode4(const Windows<K2>& win, const uint32_t (&w)[Windows<K2>::NW], uint32_t& lo,
                                        uint32_t& hi) {
  uint32_t s[4];
  win.states(w, s);
  if constexpr (CB == 2) {
    lo = mul1_pair(s[0], s[1]);
    hi = mul1_pair(s[2], s[3]);
  } else {
    lo = half_sums(code_word<CB, K2>(s[0]), code_word<CB, K2>(s[1]));
    hi = half_sums(code_word<CB, K2>(s[2]), code_word<CB, K2>(s[3]));
  }
}

template <int K2, int CB>
__device__ __forceinline__ void values4(const uint32_t* tile, int L, int h, uint16_t (&v)[4]) {
  const Windows<K2> win(L, h);
  uint32_t w[Windows<K2>::NW], lo, hi;
  win.load(tile, w);
  decode4<K2, CB>(win, w, lo, hi);
  v[0] = (uint16_t)lo;
  v[1] = (uint16_t)(lo >> 16);
  v[2] = (uint16_t)hi;
  v[3] = (uint16_t)(hi >> 16);
}

// The lane's value of another lane of its row of 16: lane ^ M.  gfx9 has quad permutes, a row's halves mirrored (lane ^ 7) and a
// rotation of the row, so 4 is two moves.
template <int M>
__device__ __forceinline__ float row_xor(float v) {
  static_assert(M == 1 || M == 2 || M == 4 || M == 8, "inside a row of 16 lanes");
  int u = __builtin_bit_cast(int, v);
  if constexpr (M == 1) u = __builtin_amdgcn_mov_dpp(u, 0xB1, 0xF, 0xF, true);
  if constexpr (M == 2) u = __builtin_amdgcn_mov_dpp(u, 0x4E, 0xF, 0xF, true);
  if constexpr (M == 4) u = __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(u, 0x141, 0xF, 0xF, true), 0x1B, 0xF, 0xF, true);
  if constexpr (M == 8) u = __builtin_amdgcn_mov_dpp(u, 0x128, 0xF, 0xF, true);
  return __builtin_bit_cast(float, u);
}

// One butterfly step between lane and lane ^ M: the lower lane's sum, the upper lane's (lower - upper) difference, each one
// rounding.  Steps of 16 and 32 lanes are the lane-swap instructions: of two copies of a value one ends with the lower
// lane's in both places, the other with the upper's.  All six steps stay in registers; through LDS (ds_bpermute) a step
// was a round trip of a hundred cycles, and the steps bound the prompt's rotation and the tail of every decode launch.
template <int M>
__device__ __forceinline__ float butterfly(float v, int lane) {
  const float sign = (lane & M) ? -1.f : 1.f;
  if constexpr (M < 16) {
    return fmaf(v, sign, row_xor<M>(v));
  } else {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto t = M == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false) : __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaf(__builtin_bit_cast(float, (uint32_t)t[1]), sign, __builtin_bit_cast(float, (uint32_t)t[0]));
  }
}

// Unscaled Walsh-Hadamard transform of 128 values, two a lane (elements 2 lane, 2 lane + 1), fixed butterfly order.
__device__ __forceinline__ void fwht128(float& a, float& b, int lane) {
  const float s = a + b, d = a - b;
  a = butterfly<1>(s, lane), b = butterfly<1>(d, lane);
  a = butterfly<2>(a, lane), b = butterfly<2>(b, lane);
  a = butterfly<4>(a, lane), b = butterfly<4>(b, lane);
  a = butterfly<8>(a, lane), b = butterfly<8>(b, lane);
  a = butterfly<16>(a, lane), b = butterfly<16>(b, lane);
  a = butterfly<32>(a, lane), b = butterfly<32>(b, lane);
}

// The same transform of four blocks a wave, eight values a lane (elements 8 (lane % 16) on): the same sums in the same
// order, so the same bits; three steps between a lane's own values, four between lanes, for eight values at once.
__device__ __forceinline__ void fwht128x8(float (&v)[8], int lane) {
#pragma unroll
  for (int m = 1; m < 8; m <<= 1)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (!(i & m)) {
        const float s = v[i] + v[i + m], d = v[i] - v[i + m];
        v[i] = s;
        v[i + m] = d;
      }
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = butterfly<1>(v[i], lane);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = butterfly<2>(v[i], lane);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = butterfly<4>(v[i], lane);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = butterfly<8>(v[i], lane);
}

// eight values at element i, a multiple of 8, of a tensor that starts on any 4 bytes
typedef uint32_t __attribute__((ext_vector_type(4), aligned(4))) words4_t;

__device__ __forceinline__ void load8(const void* p, int dtype, size_t i, float (&v)[8]) {
  if (dtype == TF_F32) {
    const words4_t u = *reinterpret_cast<const words4_t*>(static_cast<const float*>(p) + i);
    const words4_t w = *reinterpret_cast<const words4_t*>(static_cast<const float*>(p) + i + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = __builtin_bit_cast(float, (uint32_t)u[j]), v[4 + j] = __builtin_bit_cast(float, (uint32_t)w[j]);
    return;
  }
  const words4_t u = *reinterpret_cast<const words4_t*>(static_cast<const uint16_t*>(p) + i);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (dtype == TF_BF16) {
      v[2 * j] = bf16_lo(u[j]);
      v[2 * j + 1] = bf16_hi(u[j]);
    } else {
      const uint32_t w = u[j];
      const __half2 h = __builtin_bit_cast(__half2, w);
      v[2 * j] = __low2float(h);
      v[2 * j + 1] = __high2float(h);
    }
  }
}

__device__ __forceinline__ void store8(void* p, int dtype, size_t i, const float (&v)[8]) {
  if (dtype == TF_F32) {
    words4_t u, w;
#pragma unroll
    for (int j = 0; j < 4; ++j) u[j] = __builtin_bit_cast(uint32_t, v[j]), w[j] = __builtin_bit_cast(uint32_t, v[4 + j]);
    *reinterpret_cast<words4_t*>(static_cast<float*>(p) + i) = u;
    *reinterpret_cast<words4_t*>(static_cast<float*>(p) + i + 4) = w;
    return;
  }
  words4_t u;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    u[j] = dtype == TF_BF16 ? pack_bf16(v[2 * j], v[2 * j + 1]) : __builtin_bit_cast(uint32_t, __floats2half2_rn(v[2 * j], v[2 * j + 1]));
  *reinterpret_cast<words4_t*>(static_cast<uint16_t*>(p) + i) = u;
}

__device__ __forceinline__ void load2(const void* p, int dtype, size_t i, float& a, float& b) {
  if (dtype == TF_F32) {
    const float2 u = *reinterpret_cast<const float2*>(static_cast<const float*>(p) + i);
    a = u.x;
    b = u.y;
  } else if (dtype == TF_BF16) {
    const uint32_t u = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(p) + i);
    a = bf16_lo(u);
    b = bf16_hi(u);
  } else {
    const __half2 u = *reinterpret_cast<const __half2*>(static_cast<const __half*>(p) + i);
    a = __low2float(u);
    b = __high2float(u);
  }
}

__device__ __forceinline__ void store2(void* p, int dtype, size_t i, float a, float b) {
  if (dtype == TF_F32) {
    *reinterpret_cast<float2*>(static_cast<float*>(p) + i) = make_float2(a, b);
  } else if (dtype == TF_BF16) {
    *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(p) + i) = pack_bf16(a, b);
  } else {
    *reinterpret_cast<__half2*>(static_cast<__half*>(p) + i) = __floats2half2_rn(a, b);
  }
}


// The lane's two columns' output scales and bias of a layer, loaded once for all the rows a wave finishes.
struct OutScale {
  float sa, sb, ba, bb;
  __device__ __forceinline__ OutScale(const uint16_t* svh, const uint16_t* bias, int col) {
    load2(svh, TF_F16, col, sa, sb);
    ba = bb = 0.f;
    has_bias = bias != nullptr;
    if (bias) load2(bias, TF_F16, col, ba, bb);
  }
  bool has_bias;
};

// the finished outputs of one row's 128 columns from their fp32 sums: H / sqrt(128), * svh, + bias
__device__ __forceinline__ void finish_values(float& a, float& b, int lane, const OutScale& s) {
  fwht128(a, b, lane);
  a = a * HAD_SCALE * s.sa;
  b = b * HAD_SCALE * s.sb;
  if (s.has_bias) {
    a += s.ba;
    b += s.bb;
  }
}

__device__ __forceinline__ void finish_row(float a, float b, int lane, const OutScale& s, void* y, int y_dtype,
                                           size_t at) {
  finish_values(a, b, lane, s);
  store2(y, y_dtype, at, a, b);
}

__device__ __forceinline__ void finish_row(float a, float b, int lane, const uint16_t* svh, const uint16_t* bias,
                                           int col, void* y, int y_dtype, size_t at) {
  finish_row(a, b, lane, OutScale(svh, bias, col), y, y_dtype, at);
}

// a value as a store to `dtype` and a load back leave it
__device__ __forceinline__ float rounded(float v, int dtype) {
  if (dtype == TF_F32) return v;
  if (dtype == TF_BF16) return round_bf16(v);
  return __half2float(__float2half_rn(v));
}

// SwiGLU of one row's 128 columns of gate (g) and up (u), two a lane, then the next layer's input rotation with its
// input scales (sa, sb): xh[at ..] = fp16(((act * suh) H) / sqrt(128)).  g and u are rounded to `dtype` first (what a
// y of that type holds), act = rounded(rounded(g / (1 + exp(-g))) * u): the roundings of the two elementwise steps
// on tensors of that type.
__device__ __forceinline__ void swiglu_rot(float g0, float g1, float u0, float u1, int dtype, int lane, float sa,
                                           float sb, uint16_t* xh, size_t at) {
  g0 = rounded(g0, dtype), g1 = rounded(g1, dtype), u0 = rounded(u0, dtype), u1 = rounded(u1, dtype);
  float a = rounded(rounded(g0 / (1.f + expf(-g0)), dtype) * u0, dtype);
  float b = rounded(rounded(g1 / (1.f + expf(-g1)), dtype) * u1, dtype);
  a *= sa;
  b *= sb;
  fwht128(a, b, lane);
  store2(xh, TF_F16, at, a * HAD_SCALE, b * HAD_SCALE);
}

// The first of `pairs` k-tile pairs of slot `slot` out of `nslots` (at most 65,535): floor(slot * pairs / nslots) without
// a 64-bit division.
__device__ __forceinline__ int first_pair(uint32_t slot, uint32_t pairs, uint32_t nslots) {
  const uint32_t q = pairs / nslots, r = pairs - q * nslots;
  return (int)(slot * q + slot * r / nslots);
}

// One wave's sums of up to 16 rows over the k-tile pairs [pr0, pr1) of a 128-column block: acc[j] is the 16 x 16
// tile of column tile j.  xr: the lane's A row (row c of the pass) + 2 kq; stage: this wave's own 16 * 128 words of LDS.
template <int K2, int CB>
__device__ __forceinline__ void wave_block(const uint16_t* xr, const uint32_t* tiles, int64_t stride_k, int pr0, int pr1,
                                           uint32_t* stage, int lane, int L, int h, f32x4_t (&acc)[8]) {
  constexpr int TW = tile_words<K2>();
  // The stored words of a k-tile pair (two runs of 8 tiles) come in with coalesced loads of up to 16 bytes a lane, one
  // pair ahead, and go through the wave's own part of LDS as they lie: each lane then reads the two or three words its
  // windows start in.  (A lane loading its words itself costs sixteen times the load instructions, and the kernel was
  // bound by their issue.)  Each lane keeps its wrapped word numbers, the same in every tile, so no tile needs a copy of
  // its first words at its end; a tile's words are at most 64, one a bank.  The pair's number is a scalar (the same
  // in the whole wave), so a run's address costs no vector instructions.
  constexpr int NW = Windows<K2>::NW;
  constexpr int RUN = 8 * TW, PER = RUN / 64, N4 = PER / 4, REM = PER % 4;      // words a run; whole words a lane
  constexpr bool HALF = RUN % 64 != 0;                                          // an odd K2: 32 words more
  const Windows<K2> win(L, h);
  pr0 = __builtin_amdgcn_readfirstlane(pr0);
  pr1 = __builtin_amdgcn_readfirstlane(pr1);
  const uint32_t* own0 = stage + win.wi;
  const uint32_t* own1 = stage + win.wi1;
  const uint32_t* own2 = stage + win.wi2;
  const int rem_at = 256 * N4 + REM * lane, half_at = 64 * PER + (lane & 31);
  u32x4_t g4[2][N4 + 1];
  uint32_t gr[2][REM + 1], gh[2];
  u32x4_t av, an;
  auto fetch = [&](int pr, u32x4_t& a) {
    const uint32_t* xk = reinterpret_cast<const uint32_t*>(xr + 32 * pr);
    a = (u32x4_t){xk[0], xk[4], xk[8], xk[12]};
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const uint32_t* run = tiles + (2 * (int64_t)pr + r) * stride_k;
#pragma unroll
      for (int i = 0; i < N4; ++i) g4[r][i] = *reinterpret_cast<const words4_t*>(run + 256 * i + 4 * lane);
#pragma unroll
      for (int i = 0; i < REM; ++i) gr[r][i] = run[rem_at + i];
      if constexpr (HALF) gh[r] = run[half_at];
    }
  };
  auto put = [&]() {
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      uint32_t* dst = stage + r * RUN;
#pragma unroll
      for (int i = 0; i < N4; ++i) *reinterpret_cast<u32x4_t*>(dst + 256 * i + 4 * lane) = g4[r][i];
#pragma unroll
      for (int i = 0; i < REM; ++i) dst[rem_at + i] = gr[r][i];
      if constexpr (HALF) dst[half_at] = gh[r];            // both halves of the wave, the same words
    }
  };
  if (pr0 < pr1) fetch(pr0, av);
  for (int pr = pr0; pr < pr1; ++pr) {
    put();
    __builtin_amdgcn_wave_barrier();         // the wave's LDS accesses run in program order: no wait beyond the data's
    fetch(pr + 1 < pr1 ? pr + 1 : pr, an);
    const f16x8_t a = __builtin_bit_cast(f16x8_t, av);
    // 3inst and mcg: a value is the sum of the two fp16 halves of its hashed word.  The matrix unit adds them: the
    // four hashed words of a tile are the B operand as they stand (eight fp16 numbers) against every input twice
    // over, so the add costs no vector instruction.  The products are exact in fp32, so each weight enters as the
    // exact sum of its halves (the stored value is that sum rounded to fp16: at most 2^-12 relative apart).
    f16x8_t a0, a1;
    if constexpr (CB != 2) {
      const u32x4_t lo = {__builtin_amdgcn_perm(av[0], av[0], 0x01000100u), __builtin_amdgcn_perm(av[0], av[0], 0x03020302u),
                          __builtin_amdgcn_perm(av[1], av[1], 0x01000100u), __builtin_amdgcn_perm(av[1], av[1], 0x03020302u)};
      const u32x4_t hi = {__builtin_amdgcn_perm(av[2], av[2], 0x01000100u), __builtin_amdgcn_perm(av[2], av[2], 0x03020302u),
                          __builtin_amdgcn_perm(av[3], av[3], 0x01000100u), __builtin_amdgcn_perm(av[3], av[3], 0x03020302u)};
      a0 = __builtin_bit_cast(f16x8_t, lo);
      a1 = __builtin_bit_cast(f16x8_t, hi);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      // the widths with three words a window: half of the tiles' reads at a time, or they spill
      if (NW == 3 && j == 4) __builtin_amdgcn_sched_barrier(0);
      uint32_t w0[NW], w1[NW];
      w0[0] = own0[j * TW], w1[0] = own0[(8 + j) * TW];
      w0[1] = own1[j * TW], w1[1] = own1[(8 + j) * TW];
      if constexpr (NW == 3) w0[2] = own2[j * TW], w1[2] = own2[(8 + j) * TW];
      if constexpr (CB != 2) {
        uint32_t s0[4], s1[4];
        win.states(w0, s0);
        win.states(w1, s1);
        const u32x4_t x0 = {code_word<CB, K2>(s0[0]), code_word<CB, K2>(s0[1]), code_word<CB, K2>(s0[2]), code_word<CB, K2>(s0[3])};
        const u32x4_t x1 = {code_word<CB, K2>(s1[0]), code_word<CB, K2>(s1[1]), code_word<CB, K2>(s1[2]), code_word<CB, K2>(s1[3])};
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, __builtin_bit_cast(f16x8_t, x0), acc[j], 0, 0, 0);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, __builtin_bit_cast(f16x8_t, x1), acc[j], 0, 0, 0);
      } else {
        uint32_t b0, b1, b2, b3;
        decode4<K2, CB>(win, w0, b0, b1);
        decode4<K2, CB>(win, w1, b2, b3);
        const u32x4_t bw = {b0, b1, b2, b3};
        const f16x8_t b = __builtin_bit_cast(f16x8_t, bw);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc[j], 0, 0, 0);
      }
    }
    __builtin_amdgcn_wave_barrier();
    av = an;
  }
}

// A pass's sums, D[row 4 kq + i][column c] of column tile j, to red[row][16 j + c]: the rows the pass has, no others.  A wave walks
// four to six pairs, so what it does once weighs: with one row a quarter of the stores are left (that MLP 55.9 -> 51.6 us, 8 rows
// through 288 experts 230 -> 223).
__device__ __forceinline__ void store_rows(float* red, const f32x4_t (&acc)[8], int rows, int c, int kq) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i >= rows) break;
    if (4 * kq + i < rows) {
#pragma unroll
      for (int j = 0; j < 8; ++j) red[(4 * kq + i) * 128 + 16 * j + c] = acc[j][i];
    }
  }
}

// every width ExLlamaV3 writes: k2 = 2 * bits; half-integer widths exist with the mul1 codebook only
#define TF_EXL3_WIDTHS(X, CB) X(2, CB) X(4, CB) X(6, CB) X(8, CB) X(10, CB) X(12, CB) X(14, CB) X(16, CB)
#define TF_EXL3_ALL(X) TF_EXL3_WIDTHS(X, 0) TF_EXL3_WIDTHS(X, 1) TF_EXL3_WIDTHS(X, 2) X(3, 2) X(5, 2) X(7, 2)
// every half-bit count from 2 to 16 with every codebook: what the routed experts and the plain decode accept
// (reference: cuda/exl3/experts.py:15-16, experts_grouped.cuh:184-187)
#define TF_EXL3_ODD(X, CB) X(3, CB) X(5, CB) X(7, CB) X(9, CB) X(11, CB) X(13, CB) X(15, CB)
#define TF_EXL3_EVERY(X) \
  TF_EXL3_WIDTHS(X, 0) TF_EXL3_ODD(X, 0) TF_EXL3_WIDTHS(X, 1) TF_EXL3_ODD(X, 1) TF_EXL3_WIDTHS(X, 2) TF_EXL3_ODD(X, 2)

}  // namespace
}  // namespace tf

#endif  // TF_EXL3_DECODE_H
