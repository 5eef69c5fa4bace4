// MoE glue around the expert kernels: router logits, per-row top-k, the stable grouping of pairs by expert, and the
// weighted combine.  All integer results (ids, members, items) are deterministic and independent of the row count.

#include <type_traits>

#include "routing.h"

namespace tf {
namespace {

// ---- router: logits[m, e] = x[m] . rows[e] on the bf16 matrix cores -----------------------------------------------------
//
// K is cut into ROUTER_SLICES slices of whole 32-input chunks (by the hidden size alone); a slice is one MFMA chain in
// order and the slices' fp32 sums are added in slice order, so a logit's bits depend on its row and expert only.  A
// single chain of 64 to 84 dependent chunks a wave, 8 to 33 waves on the whole chip at decode, was what the first
// form spent its time on (11 us at 1 to 8 rows x 128 experts x 2688, 131 us at 4,096 x 513 x 2048).

constexpr int ROUTER_SLICES = 8;

__device__ __forceinline__ int router_chunk(int s, int chunks) { return s * chunks / ROUTER_SLICES; }

// Few tiles: a workgroup takes 16 RM rows x 16 RN experts, a wave a slice, all of a slice's operands (or UNR chunks
// of them) requested together, the slices added through LDS.  Only chunks that the slice has are requested: asking for
// its last one again up to UNR made hidden sizes up to 896 slower than one chain a wave (32 rows x 128 experts x 512:
// one chain 5.4 us, repeated 6.9, so 5.0) and cost up to a quarter where UNR does not divide a slice (8 x 128 x 4096
// 12.1 -> 9.1 us, x 2688 7.7 -> 7.1; graph replays).
template <int RM, int RN>
using RouterParts = f32x4_t[ROUTER_SLICES][RM * RN][64];

template <int RM, int RN, int UNR>
__device__ __forceinline__ void router_tile(const uint16_t* __restrict__ X, int64_t ldx, const uint16_t* __restrict__ R,
                                            float* __restrict__ out, int M, int D, int NE, int m0, int e0,
                                            RouterParts<RM, RN>& part) {
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint16_t* xa[RM];
  const uint16_t* wb[RN];
#pragma unroll
  for (int i = 0; i < RM; ++i) xa[i] = X + (size_t)min(m0 + 16 * i + r, M - 1) * ldx + kq * 8;
#pragma unroll
  for (int j = 0; j < RN; ++j) wb[j] = R + (size_t)min(e0 + 16 * j + r, NE - 1) * D + kq * 8;
  f32x4_t acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int c0 = router_chunk(wave, D / 32), c1 = router_chunk(wave + 1, D / 32);
  for (int c = c0; c < c1; c += UNR) {
    bf16x8_t a[UNR][RM], b[UNR][RN];
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      if (c + u >= c1) continue;
      const int k0 = 32 * (c + u);
#pragma unroll
      for (int i = 0; i < RM; ++i) a[u][i] = *reinterpret_cast<const bf16x8_t*>(xa[i] + k0);
#pragma unroll
      for (int j = 0; j < RN; ++j) b[u][j] = *reinterpret_cast<const bf16x8_t*>(wb[j] + k0);
    }
#pragma unroll
    for (int u = 0; u < UNR; ++u)
      if (c + u < c1)
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int j = 0; j < RN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][i], b[u][j], acc[i][j], 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) part[wave][i * RN + j][lane] = acc[i][j];
  __syncthreads();
  for (int t = wave; t < RM * RN; t += ROUTER_SLICES) {
    f32x4_t s = part[0][t][lane];
#pragma unroll
    for (int q = 1; q < ROUTER_SLICES; ++q) {
      const f32x4_t v = part[q][t][lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = __fadd_rn(s[i], v[i]);
    }
    const int row = m0 + 16 * (t / RN) + 4 * kq, col = e0 + 16 * (t % RN) + r;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (row + i < M && col < NE) out[(size_t)(row + i) * NE + col] = s[i];
  }
}

template <int RM, int RN, int UNR>
__global__ void __launch_bounds__(64 * ROUTER_SLICES)
    router_kernel(const uint16_t* __restrict__ X, int64_t ldx, const uint16_t* __restrict__ R, float* __restrict__ out,
                  int M, int D, int NE) {
  __shared__ RouterParts<RM, RN> part;
  router_tile<RM, RN, UNR>(X, ldx, R, out, M, D, NE, blockIdx.x * 16 * RM, blockIdx.y * 16 * RN, part);
}

// Many tiles: eight waves on 64 rows x 128 experts, both operands through LDS (whole 128-byte lines from memory, 64 inputs a
// step), a wave on 32 x 32 walking the slices itself.  A step is a chain of LDS trips (the same inputs again and again from
// the cache take as long), so it has as few as it can: both chunks' operands are read together, no condition between them, the
// next step's go to the other stage under the matrix instructions, and two workgroups fit a compute unit.  Up to 16 experts past the last 128
// (a shared expert's gate) are taken by workgroups of their own in router_kernel's way, 64 x 16.
// 4,096 rows x 512 experts x 2048 28.6 us with four waves of 32 x 64, 21.2; x 513 30.4, 23.7.
constexpr int RW_M = 64, RW_N = 128, RW_MORE = 16, RW_STEP = 64, RW_ROW = RW_STEP * 2 + 16;      // bytes of an LDS row, padded
constexpr int RW_THREADS = 512, RW_SETS = 2, RW_LDS = 2 * (RW_M + RW_N) * RW_ROW;
static_assert(RW_THREADS == 64 * ROUTER_SLICES && sizeof(RouterParts<RW_M / 16, 1>) <= RW_LDS, "the narrow tile's workgroup");

__device__ __forceinline__ void router_wide_tile(const uint16_t* __restrict__ X, int64_t ldx, const uint16_t* __restrict__ R,
                                                 float* __restrict__ out, int M, int D, int NE, unsigned char* lds) {
  constexpr int PIECES = (RW_M + RW_N) * 8 / RW_THREADS;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = blockIdx.x * RW_M, e0 = blockIdx.y * RW_N, wm = 32 * (wave & 1), we = 32 * (wave >> 1);
  // this thread's 16-byte pieces of the step's rows
  const uint16_t* src[PIECES];
  int at[PIECES];
#pragma unroll
  for (int j = 0; j < PIECES; ++j) {
    const int row = (tid >> 3) + 64 * j, ch = tid & 7;
    src[j] = (row < RW_M ? X + (size_t)min(m0 + row, M - 1) * ldx : R + (size_t)min(e0 + row - RW_M, NE - 1) * D) + ch * 8;
    at[j] = row * RW_ROW + ch * 16;
  }
  const int chunks = D / 32, steps = (chunks + 1) / 2;
  u32x4_t v[RW_SETS][PIECES];
  // (D in whole chunks of 32: the last step's second half may lie past the row; it is then the first again, and counts as zeros)
  auto load = [&](u32x4_t (&w)[PIECES], int step) __attribute__((always_inline)) {
    const int k0 = min(RW_STEP * step, D - 8 - (tid & 7) * 8);
#pragma unroll
    for (int j = 0; j < PIECES; ++j) w[j] = *reinterpret_cast<const u32x4_t*>(src[j] + k0);
  };
  auto store = [&](int step, int u, u32x4_t (&w)[PIECES]) __attribute__((always_inline)) {
    const bool past = RW_STEP * step + (tid & 7) * 8 >= D;
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
      if (past) w[j] = (u32x4_t){0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4_t*>(lds + u * (RW_LDS / 2) + at[j]) = w[j];
    }
  };
  f32x4_t acc[2][2], sum[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = sum[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  auto join = [](f32x4_t& total, f32x4_t& part) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) total[q] = __fadd_rn(total[q], part[q]);
    part = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  };
  int slice = 0, end = router_chunk(1, chunks);
  while (end == 0) end = router_chunk(++slice + 1, chunks);
  // one step from stage U & 1: set U takes the operands of four steps on, set U + 1 goes to the other stage
  auto walk = [&](int step, auto U) __attribute__((always_inline)) {
    constexpr int u = decltype(U)::value;
    load(v[u], step + RW_SETS);
    // both chunks' operands first, and no condition on the way: a branch between two reads would put a second trip to LDS
    // into every step
    auto operand = [&](int row, int h) {
      return *reinterpret_cast<const bf16x8_t*>(lds + (u & 1) * (RW_LDS / 2) + row * RW_ROW + h * 64 + kq * 16);
    };
    bf16x8_t a[2][2], b[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[h][i] = operand(wm + 16 * i + r, h);
        b[h][i] = operand(RW_M + we + 16 * i + r, h);
      }
    }
    // the other stage was last read before the barrier: its writes land under the matrix instructions
    store(step + 1, 1 - (u & 1), v[(u + 1) % RW_SETS]);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h][i], b[h][j], acc[i][j], 0, 0, 0);
      if (2 * step + h + 1 != end) continue;
      // the slice that ends here joins the sum (slices without a chunk add nothing)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) join(sum[i][j], acc[i][j]);
      do end = router_chunk(++slice + 1, chunks);
      while (slice + 1 < ROUTER_SLICES && end == router_chunk(slice, chunks));
    }
    __syncthreads();
  };
#pragma unroll
  for (int u = 0; u < RW_SETS; ++u) load(v[u], u);
  store(0, 0, v[0]);
  __syncthreads();
  int step = 0;
  static_assert(RW_SETS == 2, "the steps below");
  for (; step + 1 < steps; step += 2) {
    walk(step, std::integral_constant<int, 0>());
    walk(step + 1, std::integral_constant<int, 1>());
  }
  if (step < steps) walk(step, std::integral_constant<int, 0>());
  auto put = [&](int row0, int col, const f32x4_t& s) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (row0 + 4 * kq + q < M && col < NE) out[(size_t)(row0 + 4 * kq + q) * NE + col] = s[q];
  };
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      put(m0 + wm + 16 * i, e0 + we + 16 * j + r, sum[i][j]);
}

__global__ void __launch_bounds__(RW_THREADS, 4)
    router_wide_kernel(const uint16_t* __restrict__ X, int64_t ldx, const uint16_t* __restrict__ R,
                       float* __restrict__ out, int M, int D, int NE) {
  __shared__ __align__(16) unsigned char lds[RW_LDS];
  if (NE - (int)blockIdx.y * RW_N > RW_MORE) router_wide_tile(X, ldx, R, out, M, D, NE, lds);
  else router_tile<RW_M / 16, 1, 4>(X, ldx, R, out, M, D, NE, blockIdx.x * RW_M, blockIdx.y * RW_N,
                                    *reinterpret_cast<RouterParts<RW_M / 16, 1>*>(lds));
}

__global__ void __launch_bounds__(64)
    topk_kernel(const float* __restrict__ L, int64_t ldl, int NE, int TOPK, int shared, int* __restrict__ pick,
                float* __restrict__ wts) {
  const int r = blockIdx.x, slots = TOPK + (shared ? 1 : 0);
  topk_row(L + (size_t)r * ldl, NE, TOPK, shared, threadIdx.x, pick + (size_t)r * slots, wts + (size_t)r * slots);
}

// ---- plan: stable counting sort of pairs by expert -------------------------------------------------------------------

// up to 1024 pairs: one workgroup counts, scans and places; then a wave an expert that has pairs collects them in
// pair order (ballots over the pairs, 64 a step)
__global__ void __launch_bounds__(PLAN_THREADS)
    plan_small_kernel(const int* __restrict__ picks, int P, int E, int T, int* __restrict__ members,
                      int* __restrict__ items, int* __restrict__ counts) {
  __shared__ int pk[PLAN_THREADS];
  __shared__ PlanLds plan;
  plan_small(picks, P, E, T, members, items, counts, pk, plan);
}

// The decode layer's whole routing in one workgroup (rows * slots <= 1024): top-k of every row, the pair sort, one
// descriptor an item for the fused expert kernel {expert, count, first, 0, pairs[16]}, and the zeroing of the fused
// kernel's counters.

__global__ void __launch_bounds__(PLAN_THREADS)
    route_decode_kernel(const float* __restrict__ L, int64_t ldl, int R, int NE, int TOPK, int shared,
                        int* __restrict__ pick, float* __restrict__ wts, int* __restrict__ members,
                        int* __restrict__ items, int* __restrict__ counts, int* __restrict__ desc,
                        int* __restrict__ zero, int n_zero, int have_picks) {
  __shared__ int pk[PLAN_THREADS];
  __shared__ PlanLds plan;
  __shared__ int mem[PLAN_THREADS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int slots = TOPK + (shared ? 1 : 0), P = R * slots, E = NE + (shared ? 1 : 0), T = 16;
  plan.cnt[tid] = 0;
  for (int i = tid; i < n_zero; i += PLAN_THREADS) zero[i] = 0;
  if (!have_picks) {      // else a launch before this one has left the picks and the weights
    for (int r = wave; r < R; r += PLAN_THREADS / 64)
      topk_row(L + (size_t)r * ldl, NE, TOPK, shared, lane, pick + (size_t)r * slots, wts + (size_t)r * slots);
  }
  __threadfence_block();
  __syncthreads();
  int e = tid < P ? pick[tid] : -1;
  if ((unsigned)e >= (unsigned)E) e = -1;
  pk[tid] = e;
  if (e >= 0) atomicAdd(&plan.cnt[e], 1);
  __syncthreads();
  place_items(plan, tid < E ? plan.cnt[tid] : 0, E, T, items, counts);
  for (int x = wave; x < E; x += PLAN_THREADS / 64) {
    const int c = plan.cnt[x], at = plan.first[x];
    if (c)
      expert_pairs(pk, P, x, c, lane, [&](int rank, int p) {
        members[at + rank] = p;
        mem[at + rank] = p;
      });
  }
  __threadfence_block();
  __syncthreads();
  const int* cnt = plan.cnt;
  const int* off = plan.first;
  // the descriptors: the same members cut into items of DTILE, every full item first (they take longest), then the
  // experts' short last items
  const int c = tid < E ? cnt[tid] : 0, f = c / DTILE, r = c - DTILE * f > 0 ? 1 : 0;
  int val[3] = {f, r, 0}, excl[3], tot[3];
  scan3(val, excl, tot);
  if (tid == 0) desc[0] = tot[0] + tot[1];
  for (int j = 0; j < f + r; ++j) {
    int* d = desc + (size_t)(1 + (j < f ? excl[0] + j : tot[0] + excl[1])) * DESC;
    const int first = off[tid] + DTILE * j, n = min(DTILE, c - DTILE * j);
    d[0] = tid;
    d[1] = n;
    d[2] = first;
    d[3] = 0;
    for (int k = 0; k < DTILE; ++k) d[4 + k] = k < n ? mem[first + k] : 0;
  }
}

// wide plans, pass 1: block b ranks its 1024 pairs within each expert (pair order) and leaves its counts in hist[b].
// A pair's rank = the pairs of its expert in earlier waves of the block + those in earlier lanes of its wave: the
// lanes are compared through 64 readlanes, the waves' counts (one writer each: the expert's last lane in the wave)
// are prefixed by a thread an expert.
__global__ void __launch_bounds__(PLAN_THREADS)
    plan_rank_kernel(const int* __restrict__ picks, int P, int E, int* __restrict__ rank, int* __restrict__ hist) {
  constexpr int NW = PLAN_THREADS / 64;
  __shared__ unsigned short wcnt[NW][EMAX];      // pairs of expert e in wave w; then: in the waves before w
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, p = blockIdx.x * PLAN_THREADS + tid;
  for (int i = tid; i < NW * EMAX; i += PLAN_THREADS) (&wcnt[0][0])[i] = 0;
  int e = -1;
  if (p < P) {
    e = picks[p];
    if ((unsigned)e >= (unsigned)E) e = -1;
  }
  int before = 0, later = 0;
  for (int l = 0; l < 64; ++l) {
    const int el = __builtin_amdgcn_readlane(e, l);
    before += (l < lane) & (el == e);
    later |= (l > lane) & (el == e);
  }
  __syncthreads();
  if (e >= 0 && !later) wcnt[wave][e] = (unsigned short)(before + 1);
  __syncthreads();
  if (tid < E) {
    int acc = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const int c = wcnt[w][tid];
      wcnt[w][tid] = (unsigned short)acc;
      acc += c;
    }
    hist[(size_t)blockIdx.x * E + tid] = acc;
  }
  __syncthreads();
  if (e >= 0) rank[p] = wcnt[wave][e] + before;
}

// pass 2 of at most PLACE_BLOCKS blocks, a workgroup each: from the counts of all of them every workgroup works out where its
// own pairs of an expert begin, and puts them there; the first writes items and counts.  What bounds it is the launch and
// three trips to memory in a row (counts, then a place in LDS, then the store); with the offsets a launch of one workgroup and
// the placing a third, both passes of it over the counts were on that chain: the whole sort 12.2 -> 10.5 us at 4,662 pairs x
// 128 experts, 16.9 -> 13.6 at 45,056 x 513, 39.1 -> 25.7 at 262,144 x 513, 46.4 -> 27.5 x 1,024 (graph replays).  Every
// workgroup reads all counts, so the reads grow with the square of the pairs: past 256 blocks (the chip holds them at once; 134 MB
// at 513 experts, 268 MB at 1,024) one workgroup adds the counts up for all of them, as below.
constexpr int PLACE_BLOCKS = 256;
__global__ void __launch_bounds__(PLAN_THREADS)
    plan_place_kernel(const int* __restrict__ picks, int P, int E, int T, const int* __restrict__ rank,
                      const int* __restrict__ hist, int* __restrict__ members, int* __restrict__ items,
                      int* __restrict__ counts) {
  constexpr int CH = 16;             // blocks read together: independent loads, one trip through memory a chunk
  const int tid = threadIdx.x, p = blockIdx.x * PLAN_THREADS + tid, nblk = gridDim.x;
  __shared__ PlanLds plan;
  int e = -1, r = 0;
  if (p < P) {
    e = picks[p];
    r = rank[p];
  }
  int c = 0, before = 0;             // the expert's pairs; those in earlier blocks
  if (tid < E)
    for (int b0 = 0; b0 < nblk; b0 += CH) {
      int v[CH];
#pragma unroll
      for (int i = 0; i < CH; ++i) v[i] = b0 + i < nblk ? hist[(size_t)(b0 + i) * E + tid] : 0;
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        c += v[i];
        before += b0 + i < (int)blockIdx.x ? v[i] : 0;
      }
    }
  place_items(plan, c, E, T, items, counts, blockIdx.x == 0);
  if (blockIdx.x) plan.first[tid] += before;               // (the first block has none, and its items are being read from here)
  __syncthreads();
  if ((unsigned)e < (unsigned)E) members[plan.first[e] + r] = p;
}

// wider: pass 2, one block: hist[b][e] becomes block b's first member of expert e; items and counts are written
__global__ void __launch_bounds__(PLAN_THREADS)
    plan_offsets_kernel(int nblk, int E, int T, int* __restrict__ hist, int* __restrict__ items,
                        int* __restrict__ counts) {
  const int tid = threadIdx.x;
  constexpr int CH = 16;             // blocks read together: independent loads, one trip through memory a chunk
  int c = 0;
  if (tid < E)
    for (int b0 = 0; b0 < nblk; b0 += CH) {
      int v[CH];
#pragma unroll
      for (int i = 0; i < CH; ++i) v[i] = b0 + i < nblk ? hist[(size_t)(b0 + i) * E + tid] : 0;
#pragma unroll
      for (int i = 0; i < CH; ++i) c += v[i];
    }
  __shared__ PlanLds plan;
  place_items(plan, c, E, T, items, counts);
  int run = plan.first[tid];
  if (tid < E)
    for (int b0 = 0; b0 < nblk; b0 += CH) {
      int v[CH];
#pragma unroll
      for (int i = 0; i < CH; ++i) v[i] = b0 + i < nblk ? hist[(size_t)(b0 + i) * E + tid] : 0;
#pragma unroll
      for (int i = 0; i < CH; ++i)
        if (b0 + i < nblk) {
          hist[(size_t)(b0 + i) * E + tid] = run;
          run += v[i];
        }
    }
}

// pass 3: every pair to its place
__global__ void plan_scatter_kernel(const int* __restrict__ picks, int P, int E, const int* __restrict__ rank,
                                    const int* __restrict__ hist, int* __restrict__ members) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  const int e = picks[p];
  if ((unsigned)e < (unsigned)E) members[hist[(size_t)(p / PLAN_THREADS) * E + e] + rank[p]] = p;
}

// ---- combine ---------------------------------------------------------------------------------------------------------

// YKIND: what the pair outputs are stored as: 0 fp32, 1 bf16, 2 fp16
template <int YKIND>
__global__ void __launch_bounds__(256)
    combine_kernel(const void* __restrict__ Y, const float* __restrict__ Wt, uint16_t* __restrict__ out, int S, int D) {
  const int r = blockIdx.x;
  const int d = (blockIdx.y * 256 + threadIdx.x) * 2;
  if (d >= D) return;
  float a0 = 0.f, a1 = 0.f;
  // eight slots' loads go out together, then the sum in slot order
  for (int k0 = 0; k0 < S; k0 += 8) {
    float w[8], v0[8], v1[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = k0 + j < S ? k0 + j : S - 1;
      w[j] = Wt[(size_t)r * S + k];
      const size_t at = ((size_t)r * S + k) * D + d;
      if (YKIND == 1) {
        const uint32_t v = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint16_t*>(Y) + at);
        v0[j] = bf16_lo(v);
        v1[j] = bf16_hi(v);
      } else if (YKIND == 2) {
        typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
        const half2_t v = *reinterpret_cast<const half2_t*>(reinterpret_cast<const _Float16*>(Y) + at);
        v0[j] = (float)v[0];
        v1[j] = (float)v[1];
      } else {
        const float2 v = *reinterpret_cast<const float2*>(reinterpret_cast<const float*>(Y) + at);
        v0[j] = v.x;
        v1[j] = v.y;
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (k0 + j < S) {
        a0 = fmaf(w[j], v0[j], a0);
        a1 = fmaf(w[j], v1[j], a1);
      }
  }
  *reinterpret_cast<uint32_t*>(out + (size_t)r * D + d) = pack_bf16(a0, a1);
}

// 16-bit pair outputs, eight columns a thread (16-byte loads), rows side by side in a workgroup, eight slots a trip to memory and
// then what is left of them: 4,096 rows x 11 x 2048 36.3 us with two columns a thread, 33.0 so (5.7 TB/s); 2,000 x 9 x 1024 10.6, 5.9;
// 777 x 8 x 2688 7.0, 5.2.  A trip's loads are as many as it has slots and none waits for another: with eight in any case, the last slot
// again for those that are not there, the compiler put a slot's loads behind the question whether there is such a slot, and few
// rows were slower than two columns a thread (bf16, 261 x 11 x 1024 4.6 us, 3.2 with two columns, 3.2 so; 456 x 11 x 1216 5.7, 4.9, 3.8).
template <int YKIND>
__global__ void __launch_bounds__(256)
    combine8_kernel(const uint16_t* __restrict__ Y, const float* __restrict__ Wt, uint16_t* __restrict__ out, int rows, int S,
                    int D8) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long r = t / D8;
  if (r >= rows) return;
  const int D = D8 * 8, d = (int)(t - r * D8) * 8;
  const uint16_t* y = Y + (size_t)r * S * D + d;
  float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // N slots from k0 on
  auto take = [&](int k0, auto N) __attribute__((always_inline)) {
    float w[N];
    u32x4_t v[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      w[j] = Wt[(size_t)r * S + k0 + j];
      v[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(y + (size_t)(k0 + j) * D));
    }
    // (nothing is converted before all of them are on their way)
#pragma unroll
    for (int j = 0; j < N; ++j) asm volatile("" : "+v"(w[j]), "+v"(v[j]));
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float lo, hi;
        if (YKIND == 1) {
          lo = bf16_lo(v[j][i]);
          hi = bf16_hi(v[j][i]);
        } else {
          typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
          const uint32_t u = v[j][i];
          const half2_t h = __builtin_bit_cast(half2_t, u);
          lo = (float)h[0];
          hi = (float)h[1];
        }
        a[2 * i] = fmaf(w[j], lo, a[2 * i]);
        a[2 * i + 1] = fmaf(w[j], hi, a[2 * i + 1]);
      }
  };
  int k0 = 0;
  for (; k0 + 8 <= S; k0 += 8) take(k0, std::integral_constant<int, 8>());
  switch (S - k0) {
#define TF_SLOTS(N_) \
  case N_: take(k0, std::integral_constant<int, N_>()); break;
    TF_SLOTS(1) TF_SLOTS(2) TF_SLOTS(3) TF_SLOTS(4) TF_SLOTS(5) TF_SLOTS(6) TF_SLOTS(7)
#undef TF_SLOTS
  }
  *reinterpret_cast<uint4*>(out + (size_t)r * D + d) =
      make_uint4(pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(a[4], a[5]), pack_bf16(a[6], a[7]));
}

// fp32 pair outputs, four columns a thread (16-byte loads): the wide prompt chunks, where the combine is a 370 MB read
__global__ void __launch_bounds__(256)
    combine4_kernel(const float* __restrict__ Y, const float* __restrict__ Wt, uint16_t* __restrict__ out, int S, int D) {
  const int r = blockIdx.x;
  const int d = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (d >= D) return;
  float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
  const float* y = Y + (size_t)r * S * D + d;
  for (int k0 = 0; k0 < S; k0 += 8) {
    float w[8];
    f32x4_t v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = k0 + j < S ? k0 + j : S - 1;
      w[j] = Wt[(size_t)r * S + k];
      v[j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(y + (size_t)k * D));
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (k0 + j < S) {
        a0 = fmaf(w[j], v[j][0], a0);
        a1 = fmaf(w[j], v[j][1], a1);
        a2 = fmaf(w[j], v[j][2], a2);
        a3 = fmaf(w[j], v[j][3], a3);
      }
  }
  *reinterpret_cast<uint2*>(out + (size_t)r * D + d) = make_uint2(pack_bf16(a0, a1), pack_bf16(a2, a3));
}

}  // namespace
}  // namespace tf

using namespace tf;

extern "C" int tf_moe_router(const uint16_t* x, int64_t ldx, const uint16_t* rows, float* logits, int m, int d, int ne,
                             tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(x && rows && logits && m >= 1 && ne >= 1, "router: null pointer or empty shape");
  TF_REQUIRE(d >= 32 && d % 32 == 0, "router: the hidden size (%d) must be a multiple of 32", d);
  TF_REQUIRE(aligned16(x) && aligned16(rows) && ldx % 8 == 0, "router: x and rows must be 16-byte aligned");
  hipStream_t s = as_stream(stream);
  // A compute unit takes 16 to 20 bytes of operands a cycle whatever the tile, so small tiles win while each has a unit
  // to itself and larger ones (operands read fewer times over) once they do not: 392 tiles x 2688 18.3 us as 16 x 16,
  // 13.3 as 32 x 32 (128 tiles 7.4 / 13).  Between the two, 32 x 16 while each has a unit to itself, all of a slice in
  // flight up to 3,072 inputs: 777 rows x 128 x 2688 11.3 us as 32 x 32 (100 units of the 256 at work), 9.6 so; 250 x 512 x 4096
  // 16.8, 13.2; 8,000 x 16 x 512 3.6, 3.5; 1,617 x 2048 14.2 us as 32 x 64, 47 as one wave's 32 x 64.  32 x 64 while each
  // has a unit to itself (4,096 x 128 x 3072 19.3 us, wide 28.1); past that the wide kernel, whose workgroups take 20 us of 2048
  // inputs however few they are (1,500 x 400 x 2048 26.2, 20.3; 2,000 x 512 x 4096 47.9, 36.4), but for a short D, which two rounds of the
  // shorter tiles walk sooner (1,055 x 512 x 288 5.0, 6.5), and where most of the last 64 columns is padding, which costs them little
  // (3,000 x 129 x 1024 9.9, 12.3; 4,100 x 72 x 2048 16.7, 20.1).
  // With up to 32 experts a column tile of 64 or 128 would be mostly padding: 32,768 rows x 8 x 2048 36 us as 32 x 64,
  // 24.7 as 64 x 16 (one wave a tile, the single chain: 27); 16,384 x 32 x 1024 13.1 as 32 x 64, 10.7 as 32 x 32.
  const int64_t tiles = (int64_t)((m + 15) / 16) * ((ne + 15) / 16), narrow = (int64_t)((m + 31) / 32) * ((ne + 63) / 64);
  if (tiles <= 256) {
    const dim3 grid((m + 15) / 16, (ne + 15) / 16);
    if (d <= 32 * 8 * ROUTER_SLICES) router_kernel<1, 1, 8><<<grid, 64 * ROUTER_SLICES, 0, s>>>(x, ldx, rows, logits, m, d, ne);
    else router_kernel<1, 1, 12><<<grid, 64 * ROUTER_SLICES, 0, s>>>(x, ldx, rows, logits, m, d, ne);
  } else if ((int64_t)((m + 31) / 32) * ((ne + 15) / 16) <= 256) {
    const dim3 grid((m + 31) / 32, (ne + 15) / 16);
    if (d <= 32 * 8 * ROUTER_SLICES) router_kernel<2, 1, 8><<<grid, 64 * ROUTER_SLICES, 0, s>>>(x, ldx, rows, logits, m, d, ne);
    else router_kernel<2, 1, 12><<<grid, 64 * ROUTER_SLICES, 0, s>>>(x, ldx, rows, logits, m, d, ne);
  } else if (tiles > 1024 && ne <= 16) {
    router_kernel<4, 1, 4><<<dim3((m + 63) / 64), 64 * ROUTER_SLICES, 0, s>>>(x, ldx, rows, logits, m, d, ne);
  } else if (tiles <= 1024 || ne <= 32) {
    router_kernel<2, 2, 4><<<dim3((m + 31) / 32, (ne + 31) / 32), 64 * ROUTER_SLICES, 0, s>>>(x, ldx, rows, logits, m, d, ne);
  } else if (narrow <= 256 || (narrow <= 512 && (int64_t)((m + 31) / 32) * ((ne + 15) / 16) <= 4 * (d < 512 ? 512 : 240))) {
    router_kernel<2, 4, 4><<<dim3((m + 31) / 32, (ne + 63) / 64), 64 * ROUTER_SLICES, 0, s>>>(x, ldx, rows, logits, m, d, ne);
  } else {
    router_wide_kernel<<<dim3((m + RW_M - 1) / RW_M, (ne + RW_N - 1) / RW_N), RW_THREADS, 0, s>>>(x, ldx, rows, logits, m, d, ne);
  }
  TF_LAUNCH_OK("tf_moe_router");
  return 0;
}

extern "C" int tf_moe_topk(const float* logits, int64_t ldl, int rows, int experts, int top_k, int shared,
                           int32_t* pick, float* wts, tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(logits && pick && wts && rows >= 1, "topk: null pointer or empty shape");
  TF_REQUIRE(experts >= 1 && experts <= 64 * TOPK_VPL, "topk: 1 to %d experts, not %d", 64 * TOPK_VPL, experts);
  TF_REQUIRE(top_k >= 1 && top_k + (shared ? 1 : 0) <= 64 && top_k <= experts, "topk: 1 to 64 slots a row, not %d", top_k);
  TF_REQUIRE(ldl >= experts + (shared ? 1 : 0), "topk: logits rows hold %lld values, %d are read", (long long)ldl,
             experts + (shared ? 1 : 0));
  topk_kernel<<<rows, 64, 0, as_stream(stream)>>>(logits, ldl, experts, top_k, shared, pick, wts);
  TF_LAUNCH_OK("tf_moe_topk");
  return 0;
}

extern "C" int tf_moe_route_decode(const float* logits, int64_t ldl, int rows, int experts, int top_k, int shared,
                                   int32_t* pick, float* wts, int32_t* members, int32_t* items, int32_t* counts,
                                   int32_t* desc, int32_t* zero, int n_zero, tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(logits && pick && wts && members && items && counts && desc, "route: null pointer argument");
  TF_REQUIRE(experts >= 1 && experts + (shared ? 1 : 0) <= EMAX && experts <= 64 * TOPK_VPL,
             "route: at most %d experts", EMAX - 1);
  TF_REQUIRE(top_k >= 1 && top_k + (shared ? 1 : 0) <= 64 && top_k <= experts, "route: 1 to 64 slots a row, not %d", top_k);
  TF_REQUIRE(rows >= 1 && (int64_t)rows * (top_k + (shared ? 1 : 0)) <= PLAN_THREADS,
             "route: the fused decode routing takes at most %d pairs", PLAN_THREADS);
  TF_REQUIRE(ldl >= experts + (shared ? 1 : 0), "route: logits rows are too short");
  TF_REQUIRE(n_zero >= 0 && (n_zero == 0 || zero), "route: bad counter range");
  // more rows than the one workgroup has waves: the top-k runs first, a workgroup a row, spread over the chip
  const int spread = rows > PLAN_THREADS / 64;
  if (spread) topk_kernel<<<rows, 64, 0, as_stream(stream)>>>(logits, ldl, experts, top_k, shared, pick, wts);
  route_decode_kernel<<<1, PLAN_THREADS, 0, as_stream(stream)>>>(logits, ldl, rows, experts, top_k, shared, pick, wts,
                                                                members, items, counts, desc, zero, n_zero, spread);
  TF_LAUNCH_OK("tf_moe_route_decode");
  return 0;
}

extern "C" int tf_experts_plan(const int32_t* picks, int64_t pairs, int experts, int tile, int32_t* members,
                               int32_t* items, int32_t* counts, int32_t* rank, int32_t* hist, tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(picks && members && items && counts, "plan: null pointer argument");
  TF_REQUIRE(experts >= 1 && experts <= EMAX, "experts: at most %d experts", EMAX);
  TF_REQUIRE(tile == 16 || tile == 64 || tile == 128, "items hold 16 pairs (decode) or 64 or 128 (prefill)");
  TF_REQUIRE(pairs >= 0 && pairs <= 0x7FFFFFFF, "plan: pair count out of range");
  hipStream_t s = as_stream(stream);
  const int P = (int)pairs;
  if (P <= PLAN_THREADS) {
    plan_small_kernel<<<1, PLAN_THREADS, 0, s>>>(picks, P, experts, tile, members, items, counts);
    TF_LAUNCH_OK("tf_experts_plan");
    return 0;
  }
  TF_REQUIRE(rank && hist, "experts: plan scratch (rank, hist) is needed past %d pairs", PLAN_THREADS);
  const int nblk = (P + PLAN_THREADS - 1) / PLAN_THREADS;
  plan_rank_kernel<<<nblk, PLAN_THREADS, 0, s>>>(picks, P, experts, rank, hist);
  if (nblk <= PLACE_BLOCKS) {
    plan_place_kernel<<<nblk, PLAN_THREADS, 0, s>>>(picks, P, experts, tile, rank, hist, members, items, counts);
    TF_LAUNCH_OK("tf_experts_plan");
    return 0;
  }
  plan_offsets_kernel<<<1, PLAN_THREADS, 0, s>>>(nblk, experts, tile, hist, items, counts);
  plan_scatter_kernel<<<(P + 255) / 256, 256, 0, s>>>(picks, P, experts, rank, hist, members);
  TF_LAUNCH_OK("tf_experts_plan");
  return 0;
}

extern "C" int tf_moe_combine(const void* y, int y_bf16, const float* wts, uint16_t* out, int rows, int slots, int d,
                              tf_stream_t stream) {
  clear_error();
  TF_REQUIRE(y && wts && out && rows >= 1 && slots >= 1, "combine: null pointer or empty shape");
  TF_REQUIRE(d >= 2 && d % 2 == 0, "combine: the hidden size (%d) must be even", d);
  if (!y_bf16 && d % 4 == 0 && aligned16(y) && rows >= 64) {
    combine4_kernel<<<dim3(rows, (d / 4 + 255) / 256), 256, 0, as_stream(stream)>>>(
        static_cast<const float*>(y), wts, out, slots, d);
    TF_LAUNCH_OK("tf_moe_combine");
    return 0;
  }
  // (a few rows have too few workgroups of eight columns a thread: 100 x 7 x 512 2.8 us, 3.1 so; at 131 of them both take 3.2)
  const int64_t wide = ((int64_t)rows * (d / 8) + 255) / 256;
  if (y_bf16 && d % 8 == 0 && aligned16(y) && aligned16(out) && wide >= 128 && wide <= 0x7FFFFFFF) {
    if (y_bf16 == 1) combine8_kernel<1><<<(unsigned)wide, 256, 0, as_stream(stream)>>>(static_cast<const uint16_t*>(y), wts, out, rows, slots, d / 8);
    else combine8_kernel<2><<<(unsigned)wide, 256, 0, as_stream(stream)>>>(static_cast<const uint16_t*>(y), wts, out, rows, slots, d / 8);
    TF_LAUNCH_OK("tf_moe_combine");
    return 0;
  }
  const dim3 grid(rows, (d / 2 + 255) / 256);
  if (y_bf16 == 1) combine_kernel<1><<<grid, 256, 0, as_stream(stream)>>>(y, wts, out, slots, d);
  else if (y_bf16 == 2) combine_kernel<2><<<grid, 256, 0, as_stream(stream)>>>(y, wts, out, slots, d);
  else combine_kernel<0><<<grid, 256, 0, as_stream(stream)>>>(y, wts, out, slots, d);
  TF_LAUNCH_OK("tf_moe_combine");
  return 0;
}
