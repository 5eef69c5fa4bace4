// Decode-form 4-bit matmuls for 1..16 rows an item: the routed-expert GEMV (tf_experts_run) and the dense lane
// matmul (tf_qmm), plus tf_group_sums.  HBM-bound: one pass over the packed weights.
//
// Mapping of the experts' GEMV (the dense matmul's is with it below).  A lane owns one output column and walks K; the 64 lanes of a wave read 1 KB of codes with one
// 16-byte load each (a chunk: 32 inputs x 64 columns).  The activations of the item's rows are the same for every
// lane: each lane loads dword (lane % 16) of the chunk (one coalesced 64-byte read, fetched with the weights,
// DEPTH groups ahead) and v_dot2c_f32_bf16's DPP form broadcasts dword j across each row of 16 lanes inside the
// multiply itself (row_newbcast:j), so there is no cross-lane reduction, no scalar-cache traffic and no LDS
// traffic in the inner loop.
//
// The experts' K is cut into SLICES fixed slices (a function of the shape alone).  A workgroup's waves each walk a run of
// consecutive slices, park each slice's fp32 sum in LDS, and the sums are added in slice order; how many waves
// share the slices (16, 8 or 4, picked from the launch size) therefore never changes a bit, and neither do the
// other rows of the call.
//
// Arithmetic per group, as the reference's decode form (experts.cu:94-106, qmm.cu:66-76):
//   acc = fma(xs, b, fma(P, s, acc)),   P = sum x * q,   xs = sum x
// with q exact.  For the experts a nibble OR-ed into the bf16 pattern of 128 is 128 + q, so the dot product gives
// P + 128 xs and P = fma(-128, xs, that).

#include <algorithm>
#include <cstdlib>
#include <mutex>

#include "gemv.h"
#include "routing.h"

namespace tf {
namespace {

// A workgroup takes (item, pair of 32-column blocks, RBMAX of the item's rows): one pass over its weights, as with
// item descriptors.  (Taking all of an item's up to 16 rows made it stream the same weights up to eight times, and
// a compute unit's workgroups together overflow the L2 between passes.)  blockIdx.y picks the rows; see expert_unit.
template <int GS, int NM, int EPI, int WAVES>
__global__ void __launch_bounds__(WAVES * 64)
    expert_kernel(const uint16_t* __restrict__ X, int64_t x_stride, int slots, const uint32_t* __restrict__ W, int KG,
                  int NB, const int* __restrict__ items, const int* __restrict__ counts,
                  const int* __restrict__ members, void* __restrict__ out, int N, float limit) {
  extern __shared__ float lds[];
  const int NB2 = (NB + 1) >> 1;
  const int it = blockIdx.x / NB2, cb2 = blockIdx.x - it * NB2;
  if (it >= counts[0]) return;
  const int e = items[3 * it], first = items[3 * it + 1], total = items[3 * it + 2];
  NoHook none;
  // rows RBMAX y .. of every 16 (a decode item holds at most 16, so this runs once)
  for (int skip = RBMAX * blockIdx.y; skip < total; skip += RBMAX * gridDim.y) {
    if (skip != RBMAX * (int)blockIdx.y) __syncthreads();
    expert_unit<GS, NM, EPI, WAVES, 0>(X, x_stride, slots, W, KG, NB, e, min(RBMAX, total - skip),
                                       members + first + skip, cb2, out, N, limit, lds, none);
  }
}

// The same unit taken from an item descriptor as tf_moe_route_decode and tf_moe_route_up write them: one read
// instead of the items -> members chain, and items of at most DTILE pairs.
template <int GS, int NM, int EPI, int WAVES>
__global__ void __launch_bounds__(WAVES * 64)
    expert_desc_kernel(const uint16_t* __restrict__ X, int64_t x_stride, int slots, const uint32_t* __restrict__ W,
                       int KG, int NB, const int* __restrict__ desc, const int* __restrict__ counts,
                       void* __restrict__ out, int N, float limit) {
  extern __shared__ float lds[];
  __shared__ int pairs[16];
  const int NB2 = (NB + 1) >> 1;
  const int it = blockIdx.x / NB2, cb2 = blockIdx.x - it * NB2;
  // the descriptor's words are requested with the count, not after it (a row past the count exists and is ignored)
  const int* d = desc + (size_t)(1 + it) * DESC;
  const int n_items = desc[0], e = d[0], cnt = d[1], p0 = d[4], p1 = d[5];
  if (it >= n_items) return;
  if (threadIdx.x < DTILE) pairs[threadIdx.x] = threadIdx.x ? p1 : p0;
  __syncthreads();
  NoHook none;
  expert_unit<GS, NM, EPI, WAVES, 0>(X, x_stride, slots, W, KG, NB, e, cnt, pairs, cb2, out, N, limit, lds, none);
}

// ---- dense lane matmul ---------------------------------------------------------------------------------------------
//
// A wave takes 64 columns and a run of groups; up to 16 RT rows of the call are the rows of v_mfma_f32_16x16x32_bf16, so
// a weight is unpacked once for all of them (rows are independent there: a row's bits do not depend on the others, on
// RT or on the row tile).  Lane L loads column L's four words of a chunk with one 16-byte load and its scale and bias,
// which change lanes by the lane swaps (`across`) to where the matrix instruction wants them.  A nibble in a byte is
// the e4m3 number q * 2^-9, so v_cvt_scalef32_pk_bf16_fp8 with scale 2^9 makes the operand's bf16 pair, exactly q.  The
// first form made vector dot products of 8 rows a pass and was bound by them: 21 rows x 17408 x 5120 72 -> 28 us
// with its reduce, 64 rows 178 -> 50, 8 rows 31 -> 20, one row 16 as before, and eight times closer to 64 bits (8e-7 ->
// 1e-7 relative: the codes no longer ride on 128, whose part was taken off again).

// one packed word -> eight bf16 codes, inputs in the order (0, 4, 1, 5, 2, 6, 3, 7)
__device__ __forceinline__ bf16x8_t codes8(uint32_t w) {
  const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
  const u32x4_t r = {__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.f, false)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.f, true)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.f, false)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.f, true))};
  return __builtin_bit_cast(bf16x8_t, r);
}

// lane I of the reader's row of 16 lanes
template <int I>
__device__ __forceinline__ float row16_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + I, 0xF, 0xF, true));
}

// Workgroups a compute unit that a launch's registers leave room for.  Told of two, the compiler keeps the accumulators among the
// ordinary registers, which is up to 15 % faster (30 rows x 4745 x 1984 8.8 us, 8.2; 7 rows x 1869 x 1728 in groups of 32 7.9, 7.1),
// but for the register walk of 5 to 8 rows of one weight in groups of 64: 6 rows x 644 x 1984 5.1 us, 5.4; 7 rows x 1000 x 5056
// 11.4, 11.8, with its own group sums 11.3, 12.2; 8 rows x 7073 x 3392 10.1, 10.3, 10.0, 10.6.  (Of several weights it is not: 5 rows
// x 7360 + 512 + 512 x 1024 5.4, 5.0.)
constexpr int qmm_groups(int gs, int ni, bool ring) { return gs == 64 && ni == 2 && !ring ? 1 : 2; }

constexpr int QPART = 68;          // floats of a row of a wave's 64 parked sums: padded against bank conflicts

// LDS floats of a workgroup
constexpr size_t qmm_lds_floats(int waves, int rt) { return (size_t)waves * 16 * rt * QPART; }

// A group in registers: the lane's column's codes, scale and bias; of row tile r the lane's eight inputs of each chunk
// (row 16 r + row_of(c), inputs 8 kq ..) and the group sum of row 16 r + kq + 4 (c % NI).
template <int GS, int RT, bool OWN>
struct DenseStage {
  uint4 w[GS / 32], x[RT][GS / 32];
  uint32_t s, b;
  float xs[RT];
};

// The group sums of OWN calls, which no launch has taken ahead: the row tile's inputs (as the matrix instruction multiplies them)
// times a column of ones, 16 at a time, what the instructions give added in fp32.  Result i is the row of result i of every product, so
// it is where the group's fma wants it.  group_sums_kernel takes them the same way, so both forms of a call have the same bits.
// The instruction cuts off what lies under its largest term instead of rounding each addition, so it is kept to 16 terms, where it
// is as close to 64 bits as rounded fp32 additions (a lane's eight in order, then a tree over lanes).  Error over the magnitudes' sum,
// rms, groups of 32 and 64, with 32 terms an instruction, 16, and rounded additions:
//   normal inputs                     3.58e-10 4.21e-10   3.50e-10 4.19e-10   3.52e-10 4.19e-10
//   their magnitudes                  2.07e-9  4.02e-9    2.10e-9  4.00e-9    2.09e-9  4.00e-9
//   max(z, 0)^2                       1.19e-8  1.92e-8    1.20e-8  1.91e-8    1.20e-8  1.91e-8
//   one sign over three decades       1.23e-8  2.21e-8    1.24e-8  2.20e-8    1.24e-8  2.20e-8
//   exp(2 z)                          3.36e-8  3.53e-8    2.70e-8  3.17e-8    2.56e-8  3.02e-8
// Rounded additions in the launch take 1.02 to 1.6 times its time (21 rows x 17408 x 5120 23.7 us), 32 terms an instruction 0.97 to 1
// (20.8 us where it is 21.4).
__device__ __forceinline__ f32x4_t ones_sum(bf16x8_t x) {
  typedef __attribute__((ext_vector_type(4))) short s16x4_t;
  typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;
  const s16x4_t one = {0x3F80, 0x3F80, 0x3F80, 0x3F80};
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const u32x4_t v = __builtin_bit_cast(u32x4_t, x);
  const u32x2_t first = {v[0], v[1]}, second = {v[2], v[3]};
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4_t, first), one, zero, 0, 0, 0) +
         __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4_t, second), one, zero, 0, 0, 0);
}

// A wave's walk over groups [g, g1) of a column tile for rows r0 .. r0 + valid - 1.  `flush(g, acc)` is called after
// group g has been added (wave-uniform); it may park and clear acc.  Result i of acc[r][t]: row 16 r + kq + 4 i, column
// 16 t + c.
// A lane ends with four of the matrix instruction's rows: 4 kq + (0..3).  The call's row p is put into row
// 4 (p % 4) + p / 4, so that up to four rows fill the lanes' first results and up to eight the first two: a call of at
// most 4 NI rows adds NI results up a lane, not four (17408 x 5120, one row: 17.9 us with NI = 4 for every call, 16.3 so).
template <int GS, int RT, int NI, bool OWN, class FLUSH>
__device__ __forceinline__ void qmm_walk(const uint16_t* __restrict__ X, int64_t ldx, const float* __restrict__ XS,
                                         const uint32_t* __restrict__ W, const uint16_t* __restrict__ S,
                                         const uint16_t* __restrict__ B, int64_t sb_stride, int KG, int tile, int r0,
                                         int valid, int g, int g1, float (&acc)[RT][4][NI], const FLUSH& flush) {
  constexpr int CH = GS / 32;
  const int lane = threadIdx.x & 63, c = lane & 15, kq = lane >> 4;
  static_assert(RT == 1 || NI == 4, "more than 16 rows need every result");
  const uint32_t* wt = W + ((size_t)tile * KG) * (size_t)(CH * 256);
  const uint32_t wo = lane * 4, co = tile * 64 + lane;
  const uint16_t* xl[RT];
  const float* xsl[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {          // rows past the last are the last one again, unstored
    xl[r] = X + (size_t)(r0 + min(16 * r + (c >> 2) + 4 * (c & 3), valid - 1)) * ldx + 8 * kq;
    xsl[r] = OWN ? nullptr : XS + (size_t)(r0 + min(16 * r + kq + 4 * (c & (NI - 1)), valid - 1)) * KG;
  }
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < NI; ++i) acc[r][t][i] = 0.f;
  typedef DenseStage<GS, RT, OWN> Stg;
  auto load = [&](Stg& st, int g) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < CH; ++i) st.w[i] = ldg16(wt + ((size_t)g * CH + i) * 256 + wo);
    st.s = (S + (size_t)g * sb_stride)[co];
    st.b = (B + (size_t)g * sb_stride)[co];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
#pragma unroll
      for (int i = 0; i < CH; ++i) st.x[r][i] = *reinterpret_cast<const uint4*>(xl[r] + (size_t)g * GS + 32 * i);
      if constexpr (!OWN) st.xs[r] = xsl[r][g];
    }
    // With one row tile a stage's requests stay apart from the next's: left alone, the compiler merges the stages' group
    // sums into one load, which arrives with the last stage.  (Two row tiles: 30.2 us so where 28.4 without.)
    if constexpr (RT == 1) asm volatile("" ::: "memory");
  };
  auto add = [&](const Stg& st, int at) __attribute__((always_inline)) {
    f32x4_t p[RT][4], own[RT];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      uint32_t w[4] = {st.w[i].x, st.w[i].y, st.w[i].z, st.w[i].w};
      across(w);
      bf16x8_t xa[RT];
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        xa[r] = __builtin_bit_cast(bf16x8_t, stage8_bf16(st.x[r][i]));
        if constexpr (OWN) own[r] = i ? own[r] + ones_sum(xa[r]) : ones_sum(xa[r]);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bf16x8_t q = codes8(w[t]);
#pragma unroll
        for (int r = 0; r < RT; ++r)
          p[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[r], q, i ? p[r][t] : (f32x4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      }
    }
    uint32_t sb[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) sb[t] = (st.s & 0xFFFFu) | (st.b << 16);
    across(sb);
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      float sc[NI];
      if constexpr (OWN) {
#pragma unroll
        for (int i = 0; i < NI; ++i) sc[i] = own[r][i];
      } else if constexpr (NI == 1) {
        sc[0] = st.xs[r];
      }
      if constexpr (!OWN && NI > 1) sc[0] = row16_lane<0>(st.xs[r]), sc[1] = row16_lane<1>(st.xs[r]);
      if constexpr (!OWN && NI > 2) sc[2] = row16_lane<2>(st.xs[r]), sc[3] = row16_lane<3>(st.xs[r]);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < NI; ++i)
          acc[r][t][i] = fmaf(sc[i], bf16_hi(sb[t]), fmaf(p[r][t][i], bf16_lo(sb[t]), acc[r][t][i]));
    }
    flush(at, acc);
  };
  Stg st[DEPTH];
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (g + d < g1) load(st[d], g + d);
  const int n = g1 - g;
  for (; g + 2 * DEPTH <= g1; g += DEPTH) {
    prio_by_progress(g1 - g, n);
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      add(st[d], g + d);
      load(st[d], g + DEPTH + d);
    }
  }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (g + d < g1) {
      add(st[d], g + d);
      if (g + DEPTH + d < g1) load(st[d], g + DEPTH + d);
    }
#pragma unroll
  for (int d = 0; d < DEPTH - 1; ++d)
    if (g + DEPTH + d < g1) add(st[d], g + DEPTH + d);
}

// The walk of a call of 9 rows and more.  There qmm_walk's stages (one or two row tiles' inputs beside the weights) take 112 to 168
// registers, and the compiler requested two of them together after adding both: every pair of groups waited for a whole
// trip.  Here a stage is the wave's own corner of LDS, filled by loads that go straight there: a group's operands are read out, its
// place takes the request for the group RING_STAGES on, and the arithmetic runs under both requests.  A wave waits for its
// own loads by count; nothing crosses waves.  The same operands and the same order of sums as qmm_walk: the same bits.  Up to 8 rows
// qmm_walk is not so held up and keeps more workgroups a compute unit.  What the ring gains depends on where the weights come from.
// 17408 x 5120, reduce included, weights in the last-level cache (four of them, 200 MB): 9 rows 17.6 -> 16.1 us, 12 18.9 -> 16.6, 16
// 20.6 -> 17.2, 21 24.6 -> 20.5, 32 30.4 -> 22.6, 64 46.9 -> 33.2; from HBM (25 of them): 17.7 -> 18.2, 18.8 -> 18.9, 20.5 ->
// 20.0, 24.6 -> 24.4, 30.3 -> 28.0, 46.7 -> 38.0 (4096 x 4096 from HBM: 9 rows 7.5 -> 8.0, 21 10.0 -> 9.7, 64 17.0 -> 15.8).
// Two stages: three (four in groups of 32) take the fourth workgroup's LDS and were slower from either (16 rows 17.8 and 20.4 us).
constexpr int RING_STAGES = 2;

template <int GS, int RT, bool OWN = false>
struct QmmRing {
  static constexpr int CH = GS / 32;
  static constexpr int AT_SB = CH * 1024, AT_X = AT_SB + 256, AT_XS = AT_X + RT * 16 * GS * 2, STAGE = AT_XS + (OWN ? 0 : RT * 64);      // bytes
  static constexpr int LOADS = CH + 1 + RT * CH + (OWN ? 0 : 1);             // load instructions a group
  static constexpr int WAVE = RING_STAGES * STAGE;
};

// Loads into LDS: a lane's 16 or 4 bytes go to `lds` + its share of the wave's run.  Written as instructions because the compiler
// would wait for every load in flight ahead of any LDS read.  m0 is the compiler's as well, so each says that it writes it.
// A vector memory instruction may read a scalar register five wait states after a vector instruction wrote it, which the
// compiler does not see to in here: bases that come out of `settled` have four of them behind them, the move to m0 is the fifth.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"          // "m0 is reserved": no value is kept there, but the compiler writes it too
#define TF_TO_LDS(LOAD, ...) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t" LOAD ::"s"(lds), __VA_ARGS__ : "memory", "m0")
// N loads in one statement, the j-th with 1,024 j added to both its address and its place
__device__ __forceinline__ void to_lds16(const void* base, const uint32_t (&off)[1], uint32_t lds) {
  TF_TO_LDS("global_load_lds_dwordx4 %1, %2", "v"(off[0]), "s"(base));
}
__device__ __forceinline__ void to_lds16(const void* base, const uint32_t (&off)[2], uint32_t lds) {
  TF_TO_LDS("global_load_lds_dwordx4 %1, %3\n\tglobal_load_lds_dwordx4 %2, %3 offset:1024", "v"(off[0]), "v"(off[1]), "s"(base));
}
__device__ __forceinline__ void to_lds16(const void* base, const uint32_t (&off)[4], uint32_t lds) {
  TF_TO_LDS("global_load_lds_dwordx4 %1, %5\n\tglobal_load_lds_dwordx4 %2, %5 offset:1024\n\t"
            "global_load_lds_dwordx4 %3, %5 offset:2048\n\tglobal_load_lds_dwordx4 %4, %5 offset:3072",
            "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(base));
}
__device__ __forceinline__ void to_lds4(const void* base, uint32_t off, uint32_t lds) {
  TF_TO_LDS("global_load_lds_dword %1, %2", "v"(off), "s"(base));
}
__device__ __forceinline__ void lane_to_lds4(const void* p, uint32_t lds) {
  TF_TO_LDS("global_load_lds_dword %1, off", "v"(p));
}
template <class A, class B, class C>
__device__ __forceinline__ void settled(A*& a, B*& b, C*& c) {
  asm volatile("s_nop 3" : "+s"(a), "+s"(b), "+s"(c));
}
#undef TF_TO_LDS
#pragma clang diagnostic pop

template <int GS, int RT, bool OWN>
__device__ __forceinline__ void qmm_ring_walk(const uint16_t* __restrict__ X, int64_t ldx, const float* __restrict__ XS,
                                              const uint32_t* __restrict__ W, const uint16_t* __restrict__ S,
                                              const uint16_t* __restrict__ B, int64_t sb_stride, int KG, int tile, int r0,
                                              int valid, int g0, int g1, float (&acc)[RT][4][4], unsigned char* ring) {
  typedef QmmRing<GS, RT, OWN> R;
  constexpr int CH = R::CH, P = R::LOADS, ROW = GS * 2, PIECES = ROW / 16;       // bytes of a row's group of inputs; 16-byte pieces
  const int lane = threadIdx.x & 63, c = lane & 15, kq = lane >> 4;
  // operand row o of the matrix instruction's 16 RT holds this row of the call (qmm_walk has the reason)
  auto call_row = [&](int o) { return min((o & ~15) + ((o & 15) >> 2) + 4 * (o & 3), valid - 1); };
  // a row's pieces lie turned by its number, so that 16 lanes reading a piece of 16 rows meet different banks
  auto turn = [&](int o) { return PIECES == 8 ? o & 7 : (o >> 1) & 3; };
  // (the j-th load adds 1,024 j to its address, which its offset does without: all of them 4,096 ahead of the row's)
  uint32_t xoff[RT * CH], woff[CH];
#pragma unroll
  for (int j = 0; j < RT * CH; ++j) {
    const int o = (64 / PIECES) * j + lane / PIECES;
    xoff[j] = (uint32_t)call_row(o) * (uint32_t)ldx * 2u + (((lane % PIECES) ^ turn(o)) * 16) + (4096 - 1024 * j);
  }
#pragma unroll
  for (int i = 0; i < CH; ++i) woff[i] = lane * 16;
  const uint32_t xsoff = (uint32_t)call_row(lane & (16 * RT - 1)) * (uint32_t)KG * 4u;
  const uint16_t* sb = (lane < 32 ? S : B) + tile * 64 + 2 * (lane & 31) + (size_t)g0 * sb_stride;
  const uint16_t* xg = X + (size_t)r0 * ldx + (size_t)g0 * GS - 2048;
  const float* xsg = OWN ? nullptr : XS + (size_t)r0 * KG + g0;
  const uint32_t* wg = W + ((size_t)tile * KG + g0) * (CH * 256);
  const uint32_t at = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)ring);
  // group g's operands; the groups are asked for in turn
  auto request = [&](int g) {
    const uint32_t lds = at + (g & (RING_STAGES - 1)) * R::STAGE;
    const uint32_t* w = wg;
    const uint16_t* x = xg;
    const float* xs = xsg;
    settled(w, x, xs);
    to_lds16(w, woff, lds);
    lane_to_lds4(sb, lds + R::AT_SB);
    to_lds16(x, xoff, lds + R::AT_X);
    if constexpr (!OWN) {
      if (lane < 16 * RT) to_lds4(xs, xsoff, lds + R::AT_XS);
      xsg += 1;
    }
    wg += CH * 256;
    xg += GS;
    sb += sb_stride;
  };
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[r][t][i] = 0.f;
  for (int d = 0; d < RING_STAGES; ++d)
    if (g0 + d < g1) request(g0 + d);
  for (int g = g0; g < g1; ++g) {
    static_assert(RING_STAGES == 2, "one group's loads may be on their way past the one waited for");
    if (g + 1 < g1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const unsigned char* stage = ring + (g & (RING_STAGES - 1)) * R::STAGE;
    uint32_t w[CH][4], s[4], b[4];
    uint4 x[RT][CH];
    float4 sums[RT];
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) w[i][t] = *reinterpret_cast<const uint32_t*>(stage + i * 1024 + (16 * t + c) * 16 + kq * 4);
#pragma unroll
    for (int r = 0; r < RT; ++r) {
#pragma unroll
      for (int i = 0; i < CH; ++i)
        x[r][i] = *reinterpret_cast<const uint4*>(stage + R::AT_X + (16 * r + c) * ROW + (((4 * i + kq) ^ turn(c)) * 16));
      if constexpr (!OWN) sums[r] = *reinterpret_cast<const float4*>(stage + R::AT_XS + (16 * r + 4 * kq) * 4);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      s[t] = *reinterpret_cast<const uint16_t*>(stage + R::AT_SB + (16 * t + c) * 2);
      b[t] = *reinterpret_cast<const uint16_t*>(stage + R::AT_SB + 128 + (16 * t + c) * 2);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");          // the stage is read: its place is free
    if (g + RING_STAGES < g1) request(g + RING_STAGES);
    f32x4_t p[RT][4], own[RT];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      bf16x8_t xa[RT];
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        xa[r] = __builtin_bit_cast(bf16x8_t, stage8_bf16(x[r][i]));
        if constexpr (OWN) own[r] = i ? own[r] + ones_sum(xa[r]) : ones_sum(xa[r]);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bf16x8_t q = codes8(w[i][t]);
#pragma unroll
        for (int r = 0; r < RT; ++r)
          p[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[r], q, i ? p[r][t] : (f32x4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      if constexpr (OWN) sums[r] = make_float4(own[r][0], own[r][1], own[r][2], own[r][3]);
      const float sc[4] = {sums[r].x, sums[r].y, sums[r].z, sums[r].w};
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[r][t][i] = fmaf(sc[i], __uint_as_float(b[t] << 16), fmaf(p[r][t][i], __uint_as_float(s[t] << 16), acc[r][t][i]));
    }
  }
}

// grid (column tiles of 64 x row tiles of 16 RT, 1, SK).  Slice z takes groups [z * per, (z + 1) * per), its waves
// split them again (added in wave order); SK > 1 leaves the slice's fp32 sums in part[z].
template <int GS, int WAVES, int RT, int NI, bool COH, bool RING, bool OWN>
__device__ __forceinline__ void qmm_block(const uint16_t* __restrict__ X, int64_t ldx, const float* __restrict__ XS,
                                          const uint32_t* __restrict__ W, const uint16_t* __restrict__ S,
                                          const uint16_t* __restrict__ B, int64_t sb_stride, void* __restrict__ out,
                                          float* __restrict__ part_out, int M, int N, int KG, int SK, int f32, int block,
                                          int slice, float* part) {
  constexpr int ROWS = 16 * RT;
  const int tiles = (N + 63) >> 6, tile = block % tiles, r0 = block / tiles * ROWS, valid = min(ROWS, M - r0);
  const int per = KG / SK, gs0 = slice * per;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float acc[RT][4][NI];
  const int g0 = gs0 + (int)((long long)wave * per / WAVES), g1 = gs0 + (int)((long long)(wave + 1) * per / WAVES);
  if constexpr (RING) {
    qmm_ring_walk<GS, RT, OWN>(X, ldx, XS, W, S, B, sb_stride, KG, tile, r0, valid, g0, g1, acc,
                               reinterpret_cast<unsigned char*>(part) + wave * QmmRing<GS, RT, OWN>::WAVE);
    __syncthreads();                                     // the rings are read: the sums take their place
  } else {
    qmm_walk<GS, RT, NI, OWN>(X, ldx, XS, W, S, B, sb_stride, KG, tile, r0, valid, g0, g1, acc, [](int, float (&)[RT][4][NI]) {});
  }
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < NI; ++i) part[(wave * ROWS + 16 * r + kq + 4 * i) * QPART + 16 * t + c] = acc[r][t][i];
  __syncthreads();
  for (int o = tid; o < valid * 64; o += WAVES * 64) {
    const int r = o >> 6, l = o & 63, cc = tile * 64 + l;
    if (cc >= N) continue;
    float s = part[r * QPART + l];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) s += part[(w * ROWS + r) * QPART + l];
    const size_t at = (size_t)(r0 + r) * N + cc;
    if (SK > 1) {
      // COH: another workgroup adds the slices up in this launch: the store goes through to where it can read it
      if (COH) __hip_atomic_store(part_out + (size_t)slice * M * N + at, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else part_out[(size_t)slice * M * N + at] = s;
    } else if (f32) reinterpret_cast<float*>(out)[at] = s;
    else reinterpret_cast<uint16_t*>(out)[at] = (uint16_t)f32_bf16_bits(s);
  }
}

template <int GS, int WAVES, int RT, int NI, bool RING, bool OWN>
__global__ void __launch_bounds__(WAVES * 64, qmm_groups(GS, NI, RING))
    qmm_kernel(const uint16_t* __restrict__ X, int64_t ldx, const float* __restrict__ XS,
               const uint32_t* __restrict__ W, const uint16_t* __restrict__ S, const uint16_t* __restrict__ B,
               int64_t sb_stride, void* __restrict__ out, float* __restrict__ part_out, int M, int N, int KG, int SK,
               int f32) {
  extern __shared__ float lds[];
  qmm_block<GS, WAVES, RT, NI, false, RING, OWN>(X, ldx, XS, W, S, B, sb_stride, out, part_out, M, N, KG, SK, f32, blockIdx.x,
                                                 blockIdx.z, lds);
}

// The split matmul of a few rows and its reduce in one launch with no traffic between workgroups, for callers without
// arrival counters (whole_takes): a workgroup takes a column tile with all of K.  A second launch costs 1.5 to 2 us:
// one row x 2048 x 512 4.3 us in two launches, 2.7 so; 8192 x 1024 4.8, 3.6; 17408 x 1024 5.8, 4.6.  The 4 SK runs of groups that qmm_kernel's waves
// take (slice z, wave w: run 4 z + w) keep their ends; a wave walks 4 SK / WAVES of them one after the other, parks each
// one's sums in LDS, and the end adds a slice's four and then the slices in order: the bits of qmm_kernel and
// qmm_reduce_kernel.
template <int GS, int WAVES, int NI, bool OWN>
__device__ __forceinline__ void qmm_whole_block(const uint16_t* __restrict__ X, int64_t ldx, const float* __restrict__ XS,
                                                const uint32_t* __restrict__ W, const uint16_t* __restrict__ S,
                                                const uint16_t* __restrict__ B, int64_t sb_stride,
                                                void* __restrict__ out, int M, int N, int KG, int SK, int f32, int tile,
                                                float* part) {
  constexpr int ROWS = 4 * NI;
  const int per = KG / SK, runs = 4 * SK / WAVES;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto begin = [&](int u) { return (u >> 2) * per + (int)((long long)(u & 3) * per / 4); };
  auto park = [&](int u, float (&a)[1][4][NI]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < NI; ++i) part[(u * ROWS + kq + 4 * i) * QPART + 16 * t + c] = a[0][t][i], a[0][t][i] = 0.f;
  };
  float acc[1][4][NI];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[0][t][i] = 0.f;
  const int u0 = wave * runs, u1 = u0 + runs;
  if (per < 4)                              // runs without a group take part in the sums as zeros
    for (int u = u0; u < u1; ++u) park(u, acc);
  int u = u0;
  while (u < u1 && begin(u + 1) == begin(u)) ++u;
  int end = u < u1 ? begin(u + 1) : -1;
  auto flush = [&](int g, float (&a)[1][4][NI]) __attribute__((always_inline)) {
    if (g + 1 != end) return;
    park(u, a);
    ++u;
    while (u < u1 && begin(u + 1) == begin(u)) ++u;
    end = u < u1 ? begin(u + 1) : -1;
  };
  qmm_walk<GS, 1, NI, OWN>(X, ldx, XS, W, S, B, sb_stride, KG, tile, 0, M, begin(u0), begin(u1), acc, flush);
  __syncthreads();
  for (int o = tid; o < M * 64; o += WAVES * 64) {
    const int r = o >> 6, l = o & 63, cc = tile * 64 + l;
    if (cc >= N) continue;
    float total = 0.f;
    for (int z = 0; z < SK; ++z) {
      const float* p = part + (4 * z * ROWS + r) * QPART + l;
      float s = p[0];
#pragma unroll
      for (int w = 1; w < 4; ++w) s += p[w * ROWS * QPART];
      total = z ? total + s : s;
    }
    const size_t at = (size_t)r * N + cc;
    if (f32) reinterpret_cast<float*>(out)[at] = total;
    else reinterpret_cast<uint16_t*>(out)[at] = (uint16_t)f32_bf16_bits(total);
  }
}

// LDS bytes of a workgroup (at most 34 KB: eight slices come with NI = 1 only)
constexpr size_t qmm_whole_lds(int sk, int ni) { return sizeof(float) * 4 * sk * 4 * ni * QPART; }

template <int GS, int WAVES, int NI, bool OWN>
__global__ void __launch_bounds__(WAVES * 64)
    qmm_whole_kernel(const uint16_t* __restrict__ X, int64_t ldx, const float* __restrict__ XS,
                     const uint32_t* __restrict__ W, const uint16_t* __restrict__ S, const uint16_t* __restrict__ B,
                     int64_t sb_stride, void* __restrict__ out, int M, int N, int KG, int SK, int f32) {
  extern __shared__ float lds[];
  qmm_whole_block<GS, WAVES, NI, OWN>(X, ldx, XS, W, S, B, sb_stride, out, M, N, KG, SK, f32, blockIdx.x, lds);
}

// What a slice's workgroup does once its sums are in part[z] (stored through to memory): wait for the stores'
// acknowledgement, count itself in at the tile's counter, and if every other slice is there already add them up.
template <int WAVES>
__device__ __forceinline__ void qmm_arrive_tail(int* __restrict__ counter, const float* __restrict__ part_out,
                                                void* __restrict__ out, int M, int N, int SK, int f32, int tile, int* last) {
  __builtin_amdgcn_s_waitcnt(0);        // this wave's stores are acknowledged ...
  __syncthreads();                      // ... every wave's are ...
  if (threadIdx.x == 0)                 // ... then the workgroup counts itself in
    *last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == SK - 1;
  __syncthreads();
  if (!*last) return;
  const long long total = (long long)M * N;
  for (int o = threadIdx.x; o < M * 64; o += WAVES * 64) {
    const int cc = tile * 64 + (o & 63);
    if (cc >= N) continue;
    const size_t at = (size_t)(o >> 6) * N + cc;
    // eight slices' loads go out together, then the sums in slice order
    float acc = 0.f;
    for (int z0 = 0; z0 < SK; z0 += 8) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[j] = __hip_atomic_load(part_out + (long long)(z0 + j < SK ? z0 + j : SK - 1) * total + at, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (z0 + j < SK) acc = z0 + j ? acc + v[j] : v[j];
    }
    if (f32) reinterpret_cast<float*>(out)[at] = acc;
    else reinterpret_cast<uint16_t*>(out)[at] = (uint16_t)f32_bf16_bits(acc);
  }
  if (threadIdx.x == 0) *counter = 0;   // every slice of the tile has arrived: ready for the next call
}

// The split matmul of up to eight rows with its reduce in the same launch: a slice's workgroup leaves its sums in
// part[z] with stores that go through to memory, waits for them to be acknowledged and counts itself in at the column
// tile's counter; the workgroup that finds the others there adds the slices in slice order (qmm_reduce_kernel's
// arithmetic) and puts the counter back to zero.
template <int GS, int WAVES, int NI, bool OWN>
__global__ void __launch_bounds__(WAVES * 64, qmm_groups(GS, NI, false))
    qmm_arrive_kernel(const uint16_t* __restrict__ X, int64_t ldx, const float* __restrict__ XS,
                      const uint32_t* __restrict__ W, const uint16_t* __restrict__ S, const uint16_t* __restrict__ B,
                      int64_t sb_stride, void* __restrict__ out, float* __restrict__ part_out, int* __restrict__ counters,
                      int M, int N, int KG, int SK, int f32) {
  extern __shared__ float lds[];
  __shared__ int last;
  qmm_block<GS, WAVES, 1, NI, true, false, OWN>(X, ldx, XS, W, S, B, sb_stride, out, part_out, M, N, KG, SK, f32, blockIdx.x,
                                                blockIdx.z, lds);
  qmm_arrive_tail<WAVES>(counters + (size_t)blockIdx.x * TF_QMM_COUNTER_STRIDE, part_out, out, M, N, SK, f32, blockIdx.x,
                         &last);
}

// Up to four weights against one x in one launch (and one reduce launch): workgroups [first[w], first[w + 1]) take
// weight w's (column tile, row tile) pairs; grid.z is the largest slice count and a weight's surplus slices leave.
constexpr int GROUP_MAX = 4;
struct GroupArgs {
  const uint32_t* w[GROUP_MAX];
  const uint16_t* s[GROUP_MAX];
  const uint16_t* b[GROUP_MAX];
  void* out[GROUP_MAX];
  float* part[GROUP_MAX];
  int* counters[GROUP_MAX];      // arrival counters of a weight (the arriving form), else unused
  int64_t sb_stride[GROUP_MAX];
  int n[GROUP_MAX], sk[GROUP_MAX];
  int first[GROUP_MAX + 1];      // workgroups (matmul) or 256-element chunks (reduce) before weight w
  int count;
};

template <int GS, int WAVES, int RT, int NI, bool RING = false>
__global__ void __launch_bounds__(WAVES * 64, 2)
    qmm_group_kernel(const uint16_t* __restrict__ X, int64_t ldx, const float* __restrict__ XS, GroupArgs a, int M,
                     int KG, int f32) {
  extern __shared__ float lds[];
  int w = 0;
#pragma unroll
  for (int i = 1; i < GROUP_MAX; ++i)
    if (i < a.count && (int)blockIdx.x >= a.first[i]) w = i;
  if ((int)blockIdx.z >= a.sk[w]) return;
  qmm_block<GS, WAVES, RT, NI, false, RING, false>(X, ldx, XS, a.w[w], a.s[w], a.b[w], a.sb_stride[w], a.out[w], a.part[w], M, a.n[w], KG,
                               a.sk[w], f32, blockIdx.x - a.first[w], blockIdx.z, lds);
}

// the grouped launch on whole column tiles (qmm_whole_kernel's way) of weights that are all cut into 4 or 8 slices
template <int GS, int NI>
__global__ void __launch_bounds__(1024)
    qmm_group_whole_kernel(const uint16_t* __restrict__ X, int64_t ldx, const float* __restrict__ XS, GroupArgs a, int M,
                           int KG, int f32) {
  extern __shared__ float lds[];
  int w = 0;
#pragma unroll
  for (int i = 1; i < GROUP_MAX; ++i)
    if (i < a.count && (int)blockIdx.x >= a.first[i]) w = i;
  qmm_whole_block<GS, 16, NI, false>(X, ldx, XS, a.w[w], a.s[w], a.b[w], a.sb_stride[w], a.out[w], M, a.n[w], KG, a.sk[w], f32,
                              blockIdx.x - a.first[w], lds);
}

// the grouped launch whose slices are added up by the last workgroup of a tile to finish (qmm_arrive_kernel's way);
// a weight whose K is not split stores its rows itself
template <int GS, int WAVES, int NI>
__global__ void __launch_bounds__(WAVES * 64, 2)
    qmm_group_arrive_kernel(const uint16_t* __restrict__ X, int64_t ldx, const float* __restrict__ XS, GroupArgs a, int M,
                            int KG, int f32) {
  extern __shared__ float lds[];
  __shared__ int last;
  int w = 0;
#pragma unroll
  for (int i = 1; i < GROUP_MAX; ++i)
    if (i < a.count && (int)blockIdx.x >= a.first[i]) w = i;
  if ((int)blockIdx.z >= a.sk[w]) return;
  const int block = blockIdx.x - a.first[w];
  qmm_block<GS, WAVES, 1, NI, true, false, false>(X, ldx, XS, a.w[w], a.s[w], a.b[w], a.sb_stride[w], a.out[w], a.part[w], M, a.n[w], KG,
                                    a.sk[w], f32, block, blockIdx.z, lds);
  if (a.sk[w] > 1)
    qmm_arrive_tail<WAVES>(a.counters[w] + (size_t)block * TF_QMM_COUNTER_STRIDE, a.part[w], a.out[w], M, a.n[w],
                           a.sk[w], f32, block, &last);
}

// p[0] + p[stride] + ... (n terms, in that order); eight loads go out together before they are added
__device__ __forceinline__ float ordered_sum(const float* __restrict__ p, long long stride, int n) {
  float acc = 0.f;
  for (int s0 = 0; s0 < n; s0 += 8) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = p[(long long)(s0 + j < n ? s0 + j : n - 1) * stride];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s0 + j < n) acc = s0 + j ? acc + v[j] : v[j];
  }
  return acc;
}

__global__ void qmm_group_reduce_kernel(GroupArgs a, int M, int f32) {
  int w = 0;
#pragma unroll
  for (int i = 1; i < GROUP_MAX; ++i)
    if (i < a.count && (int)blockIdx.x >= a.first[i]) w = i;
  if (a.sk[w] == 1) return;
  const long long total = (long long)M * a.n[w];
  const long long i = (long long)(blockIdx.x - a.first[w]) * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const float* part = a.part[w];
  const float acc = ordered_sum(part + i, total, a.sk[w]);
  if (f32) reinterpret_cast<float*>(a.out[w])[i] = acc;
  else reinterpret_cast<uint16_t*>(a.out[w])[i] = (uint16_t)f32_bf16_bits(acc);
}

// the K slices' partial sums added in slice order, then rounded once (qmm.cu:222-230)
__global__ void qmm_reduce_kernel(const float* __restrict__ part, void* __restrict__ out, long long total, int SK,
                                  int f32) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const float acc = ordered_sum(part + i, total, SK);
  if (f32) reinterpret_cast<float*>(out)[i] = acc;
  else reinterpret_cast<uint16_t*>(out)[i] = (uint16_t)f32_bf16_bits(acc);
}

// A wave takes 16 rows' sums of 16 groups (`ones_sum`); four waves a workgroup along the groups.
template <int GS>
__global__ void __launch_bounds__(256)
    group_sums_kernel(const uint16_t* __restrict__ X, int64_t ldx, int M, int KG, float* __restrict__ XS) {
  const int lane = threadIdx.x & 63, c = lane & 15, kq = lane >> 4;
  const int runs = (KG - 1) / 64 + 1, rt = blockIdx.x / runs;
  const int r0 = rt * 16, g0 = ((blockIdx.x - rt * runs) * 4 + (threadIdx.x >> 6)) * 16;
  if (g0 >= KG) return;
  const uint16_t* xl = X + (size_t)min(r0 + c, M - 1) * ldx + 8 * kq;
  f32x4_t mine = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int j = 0; j < 16; ++j) {
    const size_t at = (size_t)min(g0 + j, KG - 1) * GS;
    f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < GS / 32; ++i) {
      const uint4 v = *reinterpret_cast<const uint4*>(xl + at + 32 * i);
      const f32x4_t t = ones_sum(__builtin_bit_cast(bf16x8_t, stage8_bf16(v)));
      sum = i ? sum + t : t;
    }
    if (c == j) mine = sum;                       // every column holds the sums: lane c keeps group g0 + c's
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (r0 + 4 * kq + i < M && g0 + c < KG) XS[(size_t)(r0 + 4 * kq + i) * KG + g0 + c] = mine[i];
}

constexpr int QMM_WAVES = 4;
// What the ring walk's loads into LDS take: whole dwords (two columns' scales: an even row length on a 4-byte boundary) and 32-bit offsets from 32
// rows' first.
static bool ring_takes(int64_t ldx, int64_t sb_stride, const void* scales, const void* biases) {
  return sb_stride % 2 == 0 && (((uintptr_t)scales | (uintptr_t)biases) & 3) == 0 && ldx < (1ll << 25);
}
// Whether it is the better walk of a weight in sk slices.  Besides up to 8 rows it is not, wherever the weights come from,
// - up to 16 rows where waves have fewer than two groups and nothing to request ahead, in a grouped launch (`least` = 5 halves) two
//   and a half, its narrow weights' waves having fewer still (1536 x 3072 in groups of 32, 12 rows: 8.4 us, 8.7 as a ring; q, k and
//   v of 4096 + 1024 + 1024 columns x 4096 12.0, 12.4; 2048 + 256 + 256 x 2048 in groups of 32 8.8, 9.2; but 4096 + 512 + 512 x
//   7168, three and a half groups, 14.1, 13.0);
// - at 9 and 10 rows of a long walk along a deep K in groups of 64 (9 rows x 8192 x 8192 from the cache 12.7 us, 12.8 as a
//   ring, from HBM 12.7, 13.3; 4096 x 12288 10.6, 10.5, and 10.4, 11.2; 5120 x 17408 16.1, 15.7, and 15.9, 17.3; but 5120 x 8192, four groups a
//   wave, 12.9, 11.9, and 11.5, 11.9; in groups of 32 5120 x 17408 19.1, 17.1, and 19.3, 20.1).
static bool ring_pays(int m, int gs, int kg, int sk, int least) {
  if (m <= 8 || (m <= 16 && 2 * kg < least * QMM_WAVES * sk)) return false;
  return m > 10 || gs != 64 || kg < 128 || kg < 6 * QMM_WAVES * sk;
}
// LDS of its workgroup: the waves' rings, and later their sums in the same place
template <bool OWN>
static size_t ring_lds(int gs, int rt) {
  const int wave = gs == 64 ? (rt == 1 ? QmmRing<64, 1, OWN>::WAVE : QmmRing<64, 2, OWN>::WAVE)
                            : (rt == 1 ? QmmRing<32, 1, OWN>::WAVE : QmmRing<32, 2, OWN>::WAVE);
  return std::max((size_t)QMM_WAVES * wave, sizeof(float) * qmm_lds_floats(QMM_WAVES, rt));
}
constexpr int ARRIVE_ROWS = 8;        // rows up to which, given arrival counters, the split launch adds its own slices

// Without arrival counters: whether whole column tiles (one launch) are faster than the split launch and its reduce.
// `tiles` column tiles of 64, two a compute unit for SK = 2 (eight waves), else one.  They are while K is short: 0.61 to
// 0.97 of the time up to 1,536 inputs, and up to 3,072 (0.84 to 1.02) where the tiles fill half the chip; beyond, a tile's
// 8 or 16 waves walk too long (8192 x 5120 1.00 to 1.16).  Eight slices are two runs a wave: only up to 1,024
// inputs (0.84 to 0.98; at 1,536 1.02 to 1.11), and a call of more than four rows would not fit LDS.
bool whole_takes(int64_t tiles, int sk, int m, int k) {
  if (m > ARRIVE_ROWS || (sk != 2 && sk != 4 && sk != 8) || (sk > 2 && tiles > 256)) return false;
  if (sk == 8) return m <= 4 && k <= 1024 && tiles >= 16;
  return k <= 1536 || (k <= 3072 && tiles >= 128);
}

// Waves a workgroup of the expert GEMV: few workgroups (a small batch) spread each one's K over 16 waves, many
// workgroups keep 4 longer-running waves each so that more of them are resident.  Scheduling only: bits do not move.
int expert_waves(int64_t grid) { return grid < 384 ? 16 : grid < 768 ? 8 : 4; }

template <int GS, int NM, int EPI>
int launch_experts(const uint16_t* x, int64_t x_stride, int slots, const uint32_t* w, int kg, int nb, const int* items,
                   const int* counts, const int* members, void* out, int n, float limit, int64_t max_units,
                   hipStream_t stream) {
  const int nb2 = (nb + 1) / 2;
  const int64_t max_items = (max_units + nb - 1) / nb;
  const int64_t grid = max_items * nb2;
  if (grid < 1) return 0;
  TF_REQUIRE(grid <= 0x7FFFFFFF, "experts: %lld workgroups exceed the grid limit", (long long)grid);
  const size_t smem = sizeof(float) * expert_lds_floats(NM);
  TF_REQUIRE(smem <= 64 * 1024, "experts: K/gs = %d groups need %zu bytes of LDS (limit 65536)", kg, smem);
  const dim3 g((unsigned)grid, 16 / RBMAX);          // decode items hold at most 16 pairs
#define TF_GO(W_)                                                                                                  \
  expert_kernel<GS, NM, EPI, W_><<<g, W_ * 64, smem, stream>>>(x, x_stride, slots, w, kg, nb, items, counts, members, \
                                                               out, n, limit)
  switch (expert_waves(grid)) {
    case 16: TF_GO(16); break;
    case 8: TF_GO(8); break;
    default: TF_GO(4);
  }
#undef TF_GO
  TF_LAUNCH_OK("tf_experts_run");
  return 0;
}

template <int GS, int NM, int EPI>
int launch_experts_desc(const uint16_t* x, int64_t x_stride, int slots, const uint32_t* w, int kg, int nb,
                        const int* desc, const int* counts, void* out, int n, float limit, int64_t max_items,
                        hipStream_t stream) {
  const int nb2 = (nb + 1) / 2;
  const int64_t grid = max_items * nb2;
  if (grid < 1) return 0;
  TF_REQUIRE(grid <= 0x7FFFFFFF, "experts: %lld workgroups exceed the grid limit", (long long)grid);
  const size_t smem = sizeof(float) * expert_lds_floats(NM);
  const dim3 g((unsigned)grid);
#define TF_GO(W_)                                                                                                 \
  expert_desc_kernel<GS, NM, EPI, W_><<<g, W_ * 64, smem, stream>>>(x, x_stride, slots, w, kg, nb, desc, counts, out, n, \
                                                                    limit)
  switch (expert_waves(grid)) {
    case 16: TF_GO(16); break;
    case 8: TF_GO(8); break;
    default: TF_GO(4);
  }
#undef TF_GO
  TF_LAUNCH_OK("tf_experts_run_desc");
  return 0;
}

}  // namespace
}  // namespace tf

using namespace tf;

extern "C" int tf_experts_run_desc(int gs, int epi, const uint16_t* x, int64_t x_stride, int slots, const uint32_t* w,
                                   int kg, int nb, const int32_t* desc, const int32_t* counts, void* out, int n,
                                   float limit, int64_t max_items, tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(gs == 32 || gs == 64, "experts: groups of 32 or 64 inputs, not %d", gs);
  TF_REQUIRE(x && w && desc && counts && out, "experts: null pointer argument");
  TF_REQUIRE(kg >= 1 && nb >= 1 && n == nb * 32, "experts: n (%d) must be the column blocks (%d) times 32", n, nb);
  TF_REQUIRE(aligned16(x) && x_stride % 8 == 0, "x: rows of K = groups * group size inputs, 16-byte aligned");
  TF_REQUIRE(aligned16(w), "w must be 16-byte aligned");
  TF_REQUIRE(slots >= 0 && max_items >= 0, "experts: negative slots or max_items");
  hipStream_t s = as_stream(stream);
#define TF_RUN(GS_, NM_, EPI_)            \
  if (gs == GS_ && epi == EPI_)           \
    return launch_experts_desc<GS_, NM_, EPI_>(x, x_stride, slots, w, kg, nb, desc, counts, out, n, limit, max_items, s);
  TF_RUN(32, 1, 0) TF_RUN(32, 1, 1) TF_RUN(32, 2, 2) TF_RUN(64, 1, 0) TF_RUN(64, 1, 1) TF_RUN(64, 2, 2)
#undef TF_RUN
  set_error("experts: no kernel for group %d and epilogue %d", gs, epi);
  return 1;
}

extern "C" int tf_experts_run(int gs, int epi, const uint16_t* x, int64_t x_stride, int slots, const uint32_t* w,
                              int kg, int nb, const int32_t* items, const int32_t* counts, const int32_t* members,
                              void* out, int n, float limit, int64_t max_units, tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(gs == 32 || gs == 64, "experts: groups of 32 or 64 inputs, not %d", gs);
  TF_REQUIRE(x && w && items && counts && members && out, "experts: null pointer argument");
  TF_REQUIRE(kg >= 1 && nb >= 1 && n == nb * 32, "experts: n (%d) must be the column blocks (%d) times 32", n, nb);
  TF_REQUIRE(aligned16(x) && x_stride % 8 == 0, "x: rows of K = groups * group size inputs, 16-byte aligned");
  TF_REQUIRE(aligned16(w), "w must be 16-byte aligned");
  TF_REQUIRE(slots >= 0 && max_units >= 0, "experts: negative slots or max_units");
  hipStream_t s = as_stream(stream);
#define TF_RUN(GS_, NM_, EPI_)                                                                                    \
  if (gs == GS_ && epi == EPI_)                                                                                   \
    return launch_experts<GS_, NM_, EPI_>(x, x_stride, slots, w, kg, nb, items, counts, members, out, n, limit, \
                                          max_units, s);
  TF_RUN(32, 1, 0) TF_RUN(32, 1, 1) TF_RUN(32, 2, 2) TF_RUN(64, 1, 0) TF_RUN(64, 1, 1) TF_RUN(64, 2, 2)
#undef TF_RUN
  set_error("experts: no kernel for group %d and epilogue %d", gs, epi);
  return 1;
}

extern "C" int tf_group_sums(const uint16_t* x, int64_t ldx, int m, int k, int gs, float* xs, tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(gs == 32 || gs == 64, "group_sums: groups of 32 or 64 inputs, not %d", gs);
  TF_REQUIRE(x && xs && m >= 1 && k >= gs && k % gs == 0, "group_sums: x must be (M, K), K a multiple of the group");
  TF_REQUIRE(aligned16(x) && (m == 1 || ldx % 8 == 0), "x rows must start on 16-byte boundaries");
  const int kg = k / gs;
  const int64_t blocks = (int64_t)((m - 1) / 16 + 1) * ((kg - 1) / 64 + 1);
  TF_REQUIRE(blocks <= 0x7FFFFFFF, "group_sums: grid too large");
  const unsigned grid = (unsigned)blocks;
  if (gs == 64) group_sums_kernel<64><<<grid, 256, 0, as_stream(stream)>>>(x, ldx, m, kg, xs);
  else group_sums_kernel<32><<<grid, 256, 0, as_stream(stream)>>>(x, ldx, m, kg, xs);
  TF_LAUNCH_OK("tf_group_sums");
  return 0;
}

// tf_qmm, tf_qmm_own_sums (OWN: no xs) and tf_qmm_static: the checks and launches of the decode-form matmul; `part` holds the K slices.
template <bool OWN>
static int qmm_launch(const uint16_t* x, int64_t ldx, const float* xs, const uint32_t* weight, const uint16_t* scales,
                      const uint16_t* biases, int64_t sb_stride, void* out, float* part, int32_t* counters,
                      int n_counters, int m, int n, int k, int sk, int gs, int bm, int f32, int reduce,
                      tf_stream_t stream) {
  TF_REQUIRE(gs == 32 || gs == 64, "groups of 32 or 64");
  TF_REQUIRE(bm == 16 || bm == 32 || bm == 64, "row tile 16, 32 or 64");
  TF_REQUIRE(x && (OWN || xs) && weight && scales && biases && out && m >= 1 && n >= 1, "qmm: null pointer or empty shape");
  TF_REQUIRE(aligned16(x) && (m == 1 || ldx % 8 == 0), "x rows must start on 16-byte boundaries");
  TF_REQUIRE(ldx >= k || m == 1, "x: (M, K) bf16 with contiguous rows");
  const int kg = k / gs, npad = (n + 127) / 128 * 128;
  TF_REQUIRE(k % gs == 0 && sk >= 1 && kg % sk == 0, "K splits into whole groups a slice");
  TF_REQUIRE(sb_stride >= npad, "scales and biases: (K / gs, n padded to 128) bf16, rows may be strided");
  TF_REQUIRE(aligned16(weight), "packed weight must be 16-byte aligned");
  TF_REQUIRE(sk == 1 || part, "part: at least (SK, M, n) fp32 is needed when K is split");
  hipStream_t s = as_stream(stream);
  // up to 16 rows are one row tile of the matrix instruction; past that a workgroup takes two (`bm` is the caller's row
  // tile: accepted, and no longer what decides)
  const int rt = m <= 16 ? 1 : 2, tiles = (n + 63) / 64, rts = (m + 16 * rt - 1) / (16 * rt);
  const bool ring = ring_pays(m, gs, kg, sk, 4) && ring_takes(ldx, sb_stride, scales, biases);
  const size_t smem = ring ? ring_lds<OWN>(gs, rt) : sizeof(float) * qmm_lds_floats(QMM_WAVES, rt);
  TF_REQUIRE((int64_t)tiles * rts <= 0x7FFFFFFF && sk <= 65535, "qmm: grid too large");
  const dim3 grid((unsigned)(tiles * rts), 1, (unsigned)sk);
  if (reduce && sk > 1 && counters && m <= ARRIVE_ROWS && tiles <= n_counters) {
    // few rows and arrival counters: the slices are added up by the last workgroup of a tile to finish
#define TF_GO(GS_, NI_)                                                                                             \
  qmm_arrive_kernel<GS_, QMM_WAVES, NI_, OWN><<<grid, QMM_WAVES * 64, smem, s>>>(x, ldx, xs, weight, scales, biases, sb_stride, \
                                                                            out, part, counters, m, n, kg, sk, f32)
    if (gs == 64) {
      if (m <= 4) TF_GO(64, 1);
      else TF_GO(64, 2);
    } else {
      if (m <= 4) TF_GO(32, 1);
      else TF_GO(32, 2);
    }
#undef TF_GO
    TF_LAUNCH_OK("tf_qmm");
    return 0;
  }
  if (reduce && whole_takes(tiles, sk, m, k)) {
    const size_t whole = qmm_whole_lds(sk, m <= 4 ? 1 : 2);
#define TF_GO(GS_, W_, NI_)                                                                                              \
  qmm_whole_kernel<GS_, W_, NI_, OWN><<<(unsigned)tiles, W_ * 64, whole, s>>>(x, ldx, xs, weight, scales, biases, sb_stride, out, \
                                                                         m, n, kg, sk, f32)
    if (gs == 64) {
      if (sk == 2 && m <= 4) TF_GO(64, 8, 1);
      else if (sk == 2) TF_GO(64, 8, 2);
      else if (m <= 4) TF_GO(64, 16, 1);
      else TF_GO(64, 16, 2);
    } else {
      if (sk == 2 && m <= 4) TF_GO(32, 8, 1);
      else if (sk == 2) TF_GO(32, 8, 2);
      else if (m <= 4) TF_GO(32, 16, 1);
      else TF_GO(32, 16, 2);
    }
#undef TF_GO
    TF_LAUNCH_OK("tf_qmm");
    return 0;
  }
#define TF_GO(GS_, RT_, NI_, RING_)                                                                                      \
  qmm_kernel<GS_, QMM_WAVES, RT_, NI_, RING_, OWN><<<grid, QMM_WAVES * 64, smem, s>>>(x, ldx, xs, weight, scales, biases,     \
                                                                                 sb_stride, out, part, m, n, kg, sk, f32)
  if (gs == 64) {
    if (m <= 4) TF_GO(64, 1, 1, false);
    else if (m <= 8) TF_GO(64, 1, 2, false);
    else if (ring && m <= 16) TF_GO(64, 1, 4, true);
    else if (ring) TF_GO(64, 2, 4, true);
    else if (m <= 16) TF_GO(64, 1, 4, false);
    else TF_GO(64, 2, 4, false);
  } else {
    if (m <= 4) TF_GO(32, 1, 1, false);
    else if (m <= 8) TF_GO(32, 1, 2, false);
    else if (ring && m <= 16) TF_GO(32, 1, 4, true);
    else if (ring) TF_GO(32, 2, 4, true);
    else if (m <= 16) TF_GO(32, 1, 4, false);
    else TF_GO(32, 2, 4, false);
  }
#undef TF_GO
  TF_LAUNCH_OK("tf_qmm");
  if (sk > 1 && reduce) {
    const long long total = (long long)m * n;
    qmm_reduce_kernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(part, out, total, sk, f32);
    TF_LAUNCH_OK("tf_qmm reduce");
  }
  return 0;
}

extern "C" int tf_qmm(const uint16_t* x, int64_t ldx, const float* xs, const uint32_t* weight, const uint16_t* scales,
                      const uint16_t* biases, int64_t sb_stride, void* out, float* part, int32_t* counters,
                      int n_counters, int m, int n, int k, int sk, int gs, int bm, int f32, int reduce,
                      tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(!counters || n_counters >= 0, "qmm: a negative number of counters");
  return qmm_launch<false>(x, ldx, xs, weight, scales, biases, sb_stride, out, part, counters, n_counters, m, n, k, sk, gs, bm,
                    f32, reduce, stream);
}

extern "C" int tf_qmm_own_sums(const uint16_t* x, int64_t ldx, const uint32_t* weight, const uint16_t* scales,
                               const uint16_t* biases, int64_t sb_stride, void* out, float* part, int32_t* counters,
                               int n_counters, int m, int n, int k, int sk, int gs, int bm, int f32, int reduce,
                               tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(!counters || n_counters >= 0, "qmm: a negative number of counters");
  return qmm_launch<true>(x, ldx, nullptr, weight, scales, biases, sb_stride, out, part, counters, n_counters, m, n, k, sk, gs,
                          bm, f32, reduce, stream);
}

// The K slices of tf_qmm_static: one array a GPU, part of the loaded code object, so no call ever allocates it.
// Host code may not use the array's name as an address; it asks the runtime once a device for where that device
// holds its copy and passes that pointer to the kernels like any other buffer.
static __device__ __align__(256) float scratch[TF_QMM_STATIC_FLOATS];
// the arrival counters of the column tiles, zero when the image is loaded and put back to zero by every launch
static __device__ __align__(256) int scratch_counters[TF_QMM_STATIC_COUNTERS * TF_QMM_COUNTER_STRIDE];

// where the current device holds the two arrays (asked once a device)
static bool static_scratch(float** part, int32_t** counters) {
  constexpr int MAX_DEVICES = 64;
  static float* where[MAX_DEVICES];
  static int32_t* where_counters[MAX_DEVICES];
  static std::mutex guard;
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
    set_error("tf_qmm_static: no current HIP device (or its index is %d or more)", MAX_DEVICES);
    return false;
  }
  std::lock_guard<std::mutex> lock(guard);
  if (!where[dev]) {
    void *p = nullptr, *c = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e == hipSuccess) e = hipGetSymbolAddress(&c, HIP_SYMBOL(scratch_counters));
    if (e != hipSuccess || !p || !c) {
      set_error("tf_qmm_static: hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(e));
      return false;
    }
    where[dev] = static_cast<float*>(p);
    where_counters[dev] = static_cast<int32_t*>(c);
  }
  *part = where[dev];
  *counters = where_counters[dev];
  return true;
}

extern "C" int tf_qmm_static(const uint16_t* x, int64_t ldx, const float* xs, const uint32_t* weight,
                             const uint16_t* scales, const uint16_t* biases, int64_t sb_stride, void* out, int m, int n,
                             int k, int sk, int gs, int bm, int f32, tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(m >= 1 && n >= 1 && sk >= 1, "qmm: null pointer or empty shape");
  TF_REQUIRE(sk == 1 || (int64_t)sk * m * n <= (int64_t)TF_QMM_STATIC_FLOATS,
             "tf_qmm_static: %d slices x %d rows x %d columns = %lld fp32 partial sums exceed the built-in %lld; use "
             "tf_qmm with a part buffer", sk, m, n, (long long)sk * m * n, (long long)TF_QMM_STATIC_FLOATS);
  float* part = nullptr;
  int32_t* counters = nullptr;
  if (sk > 1 && !static_scratch(&part, &counters)) return 1;
  return qmm_launch<false>(x, ldx, xs, weight, scales, biases, sb_stride, out, part, counters, TF_QMM_STATIC_COUNTERS, m, n, k,
                    sk, gs, bm, f32, 1, stream);
}

extern "C" int tf_qmm_group(const uint16_t* x, int64_t ldx, const float* xs, int count, const uint32_t* const* weights,
                            const uint16_t* const* scales, const uint16_t* const* biases, const int64_t* sb_strides,
                            void* const* outs, float* const* parts, int32_t* const* counters, const int* n_counters,
                            const int* ns, const int* sks, int m, int k, int gs, int bm, int f32, tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(gs == 32 || gs == 64, "groups of 32 or 64");
  TF_REQUIRE(bm == 16 || bm == 32 || bm == 64, "row tile 16, 32 or 64");
  TF_REQUIRE(count >= 1 && count <= GROUP_MAX, "qmm_group: 1 to %d weights, not %d", GROUP_MAX, count);
  TF_REQUIRE(!counters || n_counters, "qmm_group: counters come with their counts");
  TF_REQUIRE(x && xs && weights && scales && biases && sb_strides && outs && parts && ns && sks && m >= 1,
             "qmm_group: null pointer or empty shape");
  TF_REQUIRE(aligned16(x) && (m == 1 || ldx % 8 == 0), "x rows must start on 16-byte boundaries");
  TF_REQUIRE(ldx >= k || m == 1, "x: (M, K) bf16 with contiguous rows");
  TF_REQUIRE(k % gs == 0, "K splits into whole groups a slice");
  const int kg = k / gs;
  // one pass of rows and every split weight's arrival counters: the arriving form, as tf_qmm
  bool arrive = counters && m <= ARRIVE_ROWS;
  for (int i = 0; i < count && arrive; ++i)
    arrive = sks[i] == 1 || (counters[i] && (ns[i] + 63) / 64 <= n_counters[i]);
  // no counters, and every K split four or eight ways: whole column tiles, as tf_qmm
  bool whole = !arrive;
  int64_t all_tiles = 0;
  int most = 1;
  for (int i = 0; i < count && whole; ++i) {
    whole = sks[i] == 4 || sks[i] == 8;
    all_tiles += ((int64_t)ns[i] + 63) / 64;
    most = std::max(most, sks[i]);
  }
  whole = whole && whole_takes(all_tiles, most, m, k);
  const int rt = m <= 16 ? 1 : 2, rts = (m + 16 * rt - 1) / (16 * rt);
  GroupArgs a{}, r{};
  int max_sk = 1;
  int64_t blocks = 0, chunks = 0;
  bool any_split = false;
  for (int i = 0; i < count; ++i) {
    const int n = ns[i], sk = sks[i], npad = (n + 127) / 128 * 128;
    TF_REQUIRE(weights[i] && scales[i] && biases[i] && outs[i] && n >= 1, "qmm_group: null pointer or empty shape");
    TF_REQUIRE(sk >= 1 && sk <= 65535 && kg % sk == 0, "K splits into whole groups a slice");
    TF_REQUIRE(sb_strides[i] >= npad, "scales and biases: (K / gs, n padded to 128) bf16, rows may be strided");
    TF_REQUIRE(aligned16(weights[i]), "packed weight must be 16-byte aligned");
    TF_REQUIRE(sk == 1 || parts[i], "part: at least (SK, M, n) fp32 is needed when K is split");
    a.w[i] = weights[i];
    a.s[i] = scales[i];
    a.b[i] = biases[i];
    a.out[i] = outs[i];
    a.part[i] = parts[i];
    a.counters[i] = arrive ? counters[i] : nullptr;
    a.sb_stride[i] = sb_strides[i];
    a.n[i] = n;
    a.sk[i] = sk;
    a.first[i] = (int)blocks;
    r.first[i] = (int)chunks;
    blocks += (int64_t)((n + 63) / 64) * rts;
    chunks += ((int64_t)m * n + 255) / 256;
    TF_REQUIRE(blocks <= 0x7FFFFFFF && chunks <= 0x7FFFFFFF, "qmm_group: grid too large");
    max_sk = sk > max_sk ? sk : max_sk;
    any_split = any_split || sk > 1;
  }
  a.count = count;
  a.first[count] = (int)blocks;
  hipStream_t s = as_stream(stream);
  bool ring = false;                          // the weight that gains most decides
  for (int i = 0; i < count; ++i) ring = ring || ring_pays(m, gs, kg, sks[i], 5);
  for (int i = 0; i < count && ring; ++i) ring = ring_takes(ldx, sb_strides[i], scales[i], biases[i]);
  const size_t smem = ring ? ring_lds<false>(gs, rt) : sizeof(float) * qmm_lds_floats(QMM_WAVES, rt);
  const dim3 grid((unsigned)blocks, 1, (unsigned)max_sk);
  if (arrive) {
#define TF_GO(GS_, NI_) \
  qmm_group_arrive_kernel<GS_, QMM_WAVES, NI_><<<grid, QMM_WAVES * 64, smem, s>>>(x, ldx, xs, a, m, kg, f32)
    if (gs == 64) {
      if (m <= 4) TF_GO(64, 1);
      else TF_GO(64, 2);
    } else {
      if (m <= 4) TF_GO(32, 1);
      else TF_GO(32, 2);
    }
#undef TF_GO
    TF_LAUNCH_OK("tf_qmm_group");
    return 0;
  }
  if (whole) {
    const size_t lds = qmm_whole_lds(max_sk, m <= 4 ? 1 : 2);
#define TF_GO(GS_, NI_) qmm_group_whole_kernel<GS_, NI_><<<(unsigned)blocks, 1024, lds, s>>>(x, ldx, xs, a, m, kg, f32)
    if (gs == 64) {
      if (m <= 4) TF_GO(64, 1);
      else TF_GO(64, 2);
    } else {
      if (m <= 4) TF_GO(32, 1);
      else TF_GO(32, 2);
    }
#undef TF_GO
    TF_LAUNCH_OK("tf_qmm_group");
    return 0;
  }
#define TF_GO(GS_, RT_, NI_, RING_) \
  qmm_group_kernel<GS_, QMM_WAVES, RT_, NI_, RING_><<<grid, QMM_WAVES * 64, smem, s>>>(x, ldx, xs, a, m, kg, f32)
  if (gs == 64) {
    if (m <= 4) TF_GO(64, 1, 1, false);
    else if (m <= 8) TF_GO(64, 1, 2, false);
    else if (ring && m <= 16) TF_GO(64, 1, 4, true);
    else if (ring) TF_GO(64, 2, 4, true);
    else if (m <= 16) TF_GO(64, 1, 4, false);
    else TF_GO(64, 2, 4, false);
  } else {
    if (m <= 4) TF_GO(32, 1, 1, false);
    else if (m <= 8) TF_GO(32, 1, 2, false);
    else if (ring && m <= 16) TF_GO(32, 1, 4, true);
    else if (ring) TF_GO(32, 2, 4, true);
    else if (m <= 16) TF_GO(32, 1, 4, false);
    else TF_GO(32, 2, 4, false);
  }
#undef TF_GO
  TF_LAUNCH_OK("tf_qmm_group");
  if (any_split) {
    int first[GROUP_MAX + 1];
    for (int i = 0; i < count; ++i) first[i] = r.first[i];
    r = a;
    for (int i = 0; i < count; ++i) r.first[i] = first[i];
    r.first[count] = (int)chunks;
    qmm_group_reduce_kernel<<<(unsigned)chunks, 256, 0, s>>>(r, m, f32);
    TF_LAUNCH_OK("tf_qmm_group reduce");
  }
  return 0;
}
