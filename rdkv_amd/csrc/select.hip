// Prefill-time selection that feeds the packer: stride-1 score pooling and the row-wise
// Lagrangian knapsack that assigns every token (or channel) a bit width.
//
// The knapsack is a bisection on lambda; one evaluation ("solve") picks, per token, the option
// minimising  score*eps[n] + lambda*bits[n]  and averages the chosen widths over the row.  Widths are
// summed as integers (exact, order-free) and the next lambda is derived redundantly by every thread that
// needs it, so there is no host round trip.  Three forms, the same bits: a workgroup per row (the usual
// one: coalesced, L2-resident after the first pass, no wait between workgroups), few long rows shared by
// several workgroups each, and short rows as a wavefront each with the row in registers.
// All lambda arithmetic is single IEEE operations in the order the reference's tensor
// expressions imply; this file is compiled without floating-point contraction.
#include <algorithm>

#include "rdkv_common.h"

// No fused multiply-adds in this file, whatever the command line says: the reference rounds every
// product and every sum on its own, and HIP's __fmul_rn / __fadd_rn do not stop the compiler from
// contracting them.  (The explicit fmaf calls below stay what they are.)
#pragma clang fp contract(off)

namespace {

constexpr int kMaxOptions = 8;
constexpr int kMaxThreads = 1024;
constexpr int kMaxDoublings = 40;

struct Options {
  int n;
  float bits[kMaxOptions];
  float eps[kMaxOptions];
  int ibits[kMaxOptions];
};

template <typename T, typename Op>
__device__ T block_reduce(T v, Op op, T* lds) {
  // result broadcast to every thread; two barriers; lds holds >= 16 values + is reusable after
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = op(v, __shfl_xor(v, off, 64));
  const int wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[wave] = v;
  __syncthreads();
  T r = lds[0];
  for (int w = 1; w < nw; ++w) r = op(r, lds[w]);
  return r;
}

struct SumI { __device__ int operator()(int a, int b) const { return a + b; } };
struct MaxI { __device__ int operator()(int a, int b) const { return a > b ? a : b; } };
struct MaxF { __device__ float operator()(float a, float b) const { return a > b ? a : b; } };

// Index of the cheapest option for one score; `width` receives its bit width.
template <int N = kMaxOptions>
__device__ __forceinline__ int choose(float s, const Options& o, const float (&lb)[N], int& width) {
  float best = __fadd_rn(__fmul_rn(s, o.eps[0]), lb[0]);
  int idx = 0;
  width = o.ibits[0];
#pragma unroll
  for (int n = 1; n < N; ++n) {
    if (n < o.n) {
      const float c = __fadd_rn(__fmul_rn(s, o.eps[n]), lb[n]);
      if (c < best) { best = c; idx = n; width = o.ibits[n]; }      // strict: the first minimum wins
    }
  }
  return idx;
}

// Row average of the chosen widths at lambda `lam`: fp32 sum (exact, < 2^24) / fp32 length.
__device__ float solve_avg(const float* __restrict__ row, int T, float lam, const Options& o, int* lds) {
  float lb[kMaxOptions];
#pragma unroll
  for (int n = 0; n < kMaxOptions; ++n) lb[n] = n < o.n ? __fmul_rn(lam, o.bits[n]) : 0.f;
  int acc = 0;
  // eight independent loads in flight per thread, then the remainder
  const int step = blockDim.x;
  int t = threadIdx.x;
  for (; t + 7 * step < T; t += 8 * step) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = row[t + u * step];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      int width;
      choose(v[u], o, lb, width);
      acc += width;
    }
  }
  for (; t < T; t += step) {
    int width;
    choose(row[t], o, lb, width);
    acc += width;
  }
  const int total = block_reduce(acc, SumI(), lds);
  return __fdiv_rn((float)total, (float)T);
}

// Writes the allocation at lambda `lam` and (optionally) how many tokens took each option.
__device__ void emit(const float* __restrict__ row, int T, float lam, const Options& o, void* out_row,
                     int out_elem_size, int* counts_row, int* lds) {
  float lb[kMaxOptions];
#pragma unroll
  for (int n = 0; n < kMaxOptions; ++n) lb[n] = n < o.n ? __fmul_rn(lam, o.bits[n]) : 0.f;
  int cnt[kMaxOptions];
#pragma unroll
  for (int n = 0; n < kMaxOptions; ++n) cnt[n] = 0;
  for (int t = threadIdx.x; t < T; t += blockDim.x) {
    int b;
    const int idx = choose(row[t], o, lb, b);
#pragma unroll
    for (int n = 0; n < kMaxOptions; ++n) cnt[n] += (n == idx) ? 1 : 0;
    if (out_elem_size == 1) reinterpret_cast<uint8_t*>(out_row)[t] = (uint8_t)b;
    else reinterpret_cast<int64_t*>(out_row)[t] = (int64_t)b;
  }
  if (counts_row != nullptr) {
#pragma unroll
    for (int n = 0; n < kMaxOptions; ++n) {
      if (n < o.n) {
        const int total = block_reduce(cnt[n], SumI(), lds);
        if (threadIdx.x == 0) counts_row[n] = total;
      }
    }
  }
}

__device__ float row_max(const float* __restrict__ row, int T, float* lds) {
  float m = -__builtin_inff();
  for (int t = threadIdx.x; t < T; t += blockDim.x) m = fmaxf(m, row[t]);
  return block_reduce(m, MaxF(), lds);
}

// The budget of a row (average bits per element): from a tensor, one value for all, or the K budget that the V
// allocation's counts leave a head (k_budget_kernel's expression).  Formed where it is used: the launches that
// filled a tensor with it were 1.3 and 4 us and a gap each of a selected layer's serial chain, and 5 us of host.
struct Budget {
  const float* rows;
  const int32_t* counts;
  int n_options, zero_col, tokens;
  float head_dim, value;
  __device__ __forceinline__ float operator()(int b) const {
    if (counts == nullptr) return rows ? rows[b] : value;
    int kept = tokens - (zero_col >= 0 ? counts[(int64_t)b * n_options + zero_col] : 0);
    if (kept < 1) kept = 1;
    return __fmul_rn(__fdiv_rn(1.0f, __fmul_rn(head_dim, (float)kept)), value);
  }
};

// Phase 1 of the batched form.  Per row: the starting upper bound and how many doublings the row
// asks for on its own (kMaxDoublings if its average never drops to the budget).
__global__ void __launch_bounds__(kMaxThreads)
knapsack_expand_kernel(const float* __restrict__ scores, int64_t stride_b, int T,
                       Budget budget, Options o, float* __restrict__ lam0_out,
                       int* __restrict__ doublings_out) {
  __shared__ int lds[32];
  const int b = blockIdx.x;
  const float* row = scores + (int64_t)b * stride_b;
  const float lam0 = fmaxf(__fmul_rn(row_max(row, T, reinterpret_cast<float*>(lds)), 0.375f), 1e-8f);
  const float bud = budget(b);
  float lam = lam0;
  int d = 0;
  for (; d < kMaxDoublings; ++d) {
    if (!(solve_avg(row, T, lam, o, lds) > bud)) break;
    lam = __fmul_rn(lam, 2.0f);
  }
  if (threadIdx.x == 0) { lam0_out[b] = lam0; doublings_out[b] = d; }
}

// Phase 2: replay the doubling rounds of the whole batch (they stop for every row at once when no
// row asks for more or when every bound has reached 1e12), then bisect this row.
__global__ void __launch_bounds__(kMaxThreads)
knapsack_bisect_kernel(const float* __restrict__ scores, int64_t stride_b, int group_rows, int T,
                       Budget budget, Options o, int max_iters, float tol,
                       const float* __restrict__ lam0_all, const int* __restrict__ doublings_all,
                       void* __restrict__ out, int out_elem_size, int64_t out_stride_b,
                       int* __restrict__ counts) {
  __shared__ int lds[32];
  const int b = blockIdx.x;
  const float* row = scores + (int64_t)b * stride_b;
  // rounds the row's batch executes: min(max_r d_r, 1 + max_r first round after which row r >= 1e12),
  // r over the group_rows consecutive rows that were one call of the reference
  const int r0 = (b / group_rows) * group_rows;
  int dmax = 0, gmax = 0;
  for (int r = r0 + threadIdx.x; r < r0 + group_rows; r += blockDim.x) {
    const int d = doublings_all[r];
    float lam = lam0_all[r];
    int g = kMaxDoublings + 1;                     // never reaches 1e12
    for (int it = 0; it < kMaxDoublings; ++it) {
      if (it < d) lam = __fmul_rn(lam, 2.0f);
      if (lam >= 1e12f) { g = it; break; }
    }
    dmax = max(dmax, d);
    gmax = max(gmax, g);
  }
  dmax = block_reduce(dmax, MaxI(), lds);
  gmax = block_reduce(gmax, MaxI(), lds);
  const int rounds = min(min(dmax, gmax + 1), kMaxDoublings);
  const int mine = min(doublings_all[b], rounds);
  float lam_hi = lam0_all[b];
  for (int i = 0; i < mine; ++i) lam_hi = __fmul_rn(lam_hi, 2.0f);

  const float bud = budget(b);
  float lam_lo = 0.f, lam_final = 0.f;
  if (!(solve_avg(row, T, 0.f, o, lds) <= bud)) {
    const float denom = fmaxf(bud, 1e-8f);
    for (int it = 0; it < max_iters; ++it) {
      const float mid = __fdiv_rn(__fadd_rn(lam_lo, lam_hi), 2.0f);
      const float avg = solve_avg(row, T, mid, o, lds);
      lam_final = mid;
      const float rel = __fdiv_rn(fabsf(__fsub_rn(avg, bud)), denom);
      if (rel < tol) break;
      if (avg > bud) lam_lo = mid; else lam_hi = mid;
    }
  }
  emit(row, T, lam_final, o, reinterpret_cast<uint8_t*>(out) + (int64_t)b * out_stride_b * out_elem_size,
       out_elem_size, counts ? counts + (int64_t)b * o.n : nullptr, lds);
}

// ---------------------------------------------------------------------------------------------
// The same solver with every row shared by several workgroups, for batches too small to fill the
// device with one workgroup per row (one layer's eight heads of 32k tokens kept eight compute units
// busy for ~60 dependent passes).  A row's S workgroups each own a contiguous chunk of it, held in
// registers.  One pass evaluates up to 17 candidate lambdas at once - the next 15 doublings, or
// lambda = 0 and the 15 midpoints four bisection levels can reach (in the first pass together with
// the row's starting lambda, which usually needs no doubling) - as integer width sums of the
// chunk.  The workgroups then exchange their sums: each stores its own as words that carry the
// pass number in their top byte, and reads every workgroup's words until all of them carry it
// (double-buffered by pass parity: a workgroup can be at most one pass ahead of another of its row).
// So a pass costs one store and one load round trip between workgroups, no atomic operation meets
// another on one address, and no ordinary memory changes hands (nothing to write back or
// invalidate).  Every workgroup adds the same integers and takes the same decisions with the
// arithmetic of the one-workgroup kernels.  The launch is sized so that all its workgroups are
// resident together; a wait that does not end within a bound makes the workgroup give up and write
// the invalid width 255 instead of hanging.
// ---------------------------------------------------------------------------------------------
// A workgroup is one, two or four sets of kCoopLanes threads (SETS).  Every set holds the whole chunk and takes its
// share of a pass's candidates: a pass is bound by its chain of vector instructions (3.5 ns each where they depend), and
// one set leaves a SIMD a wavefront or less.  With the midpoints and the way down their tree taken by lanes instead of
// one thread in turn, a call of 8 rows of 4k / 31k scores 34.6 / 43.0 -> 23.6 / 33.4 us (four / two sets).
constexpr int kCoopLanes = 256;
constexpr int kCoopMaxSplit = 64;          // workgroups per row at most
constexpr int kCoopWords = 32;             // words a workgroup can publish per pass (17 are used at most)
constexpr int kCoopMaxIters = 64;          // passes stay below the 255 the tag byte can tell apart
constexpr int kCoopSpinLimit = 1 << 20;
constexpr uint32_t kCoopValueMask = 0xffffffu;
#define RDKV_COOP_SCOPE __HIP_MEMORY_SCOPE_AGENT

// per row: uint32 [2][kCoopMaxSplit][kCoopWords] exchange words, then 4 words for the row's group
constexpr int kCoopRowWords = 2 * kCoopMaxSplit * kCoopWords + 4;

struct CoopCtx {
  int S, sub, t0, t1;
  uint32_t* words;     // the row's exchange words
  int pass;
  int* tot;            // LDS, kCoopWords ints: the totals of the last exchange
  int* failed;         // LDS flag
};

template <int SCOPE>
__device__ __forceinline__ uint32_t coop_poll(const uint32_t* p, uint32_t tag, int* failed) {
  uint32_t w = __hip_atomic_load(p, __ATOMIC_RELAXED, SCOPE);
  int spins = 0;
  while ((w >> 24) != tag) {
    if (*failed || ++spins > kCoopSpinLimit) {
      *failed = 1;
      return 0u;
    }
    __builtin_amdgcn_s_sleep(1);
    w = __hip_atomic_load(p, __ATOMIC_RELAXED, SCOPE);
  }
  return w & kCoopValueMask;
}

// Publishes this workgroup's n values (mine[i] in LDS, each below 2^24) and leaves in c.tot[i] their
// sum over the row's workgroups (MAX: the maximum of the 32-bit numbers mine[0] << 16 | mine[1]
// in c.tot[0]).
template <bool MAX, int SETS>
__device__ void coop_exchange(CoopCtx& c, int n, const int* mine) {
  const uint32_t tag = (uint32_t)(c.pass + 1);
  uint32_t* buf = c.words + (c.pass & 1) * (kCoopMaxSplit * kCoopWords);
  if ((int)threadIdx.x < n)
    __hip_atomic_store(&buf[c.sub * kCoopWords + threadIdx.x], (tag << 24) | ((uint32_t)mine[threadIdx.x] & kCoopValueMask),
                       __ATOMIC_RELAXED, RDKV_COOP_SCOPE);
  if ((int)threadIdx.x < kCoopWords) c.tot[threadIdx.x] = 0;
  __syncthreads();
  if (MAX) {
    for (int wg = threadIdx.x; wg < c.S; wg += blockDim.x) {
      const uint32_t hi = coop_poll<RDKV_COOP_SCOPE>(&buf[wg * kCoopWords], tag, c.failed);
      const uint32_t lo = coop_poll<RDKV_COOP_SCOPE>(&buf[wg * kCoopWords + 1], tag, c.failed);
      atomicMax(reinterpret_cast<unsigned int*>(&c.tot[0]), (hi << 16) | lo);
    }
  } else {
    // a thread's words (word i of every kThreads / kCoopWords-th workgroup) are requested together and
    // asked for again until all carry the tag
    constexpr int kThreads = SETS * kCoopLanes, kPer = kCoopMaxSplit * kCoopWords / kThreads;
    static_assert(kCoopWords == 32 && kThreads % kCoopWords == 0, "the lane pairing below assumes 32 words");
    const int i = threadIdx.x & (kCoopWords - 1);
    uint32_t w[kPer];
    bool want[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      want[k] = i < n && (int)threadIdx.x + k * kThreads < c.S * kCoopWords;
      w[k] = tag << 24;
    }
    int spins = 0;
    for (;;) {
#pragma unroll
      for (int k = 0; k < kPer; ++k)
        if (want[k]) w[k] = __hip_atomic_load(&buf[threadIdx.x + k * kThreads], __ATOMIC_RELAXED, RDKV_COOP_SCOPE);
      bool ok = true;
#pragma unroll
      for (int k = 0; k < kPer; ++k) ok = ok && (w[k] >> 24) == tag;
      if (ok) break;
      if (*c.failed || ++spins > kCoopSpinLimit) {
        *c.failed = 1;
#pragma unroll
        for (int k = 0; k < kPer; ++k) w[k] = 0u;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    int sum = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) sum += want[k] ? (int)(w[k] & kCoopValueMask) : 0;
    // lanes l and l ^ 32 hold the same i
    sum += __shfl_xor(sum, 32, 64);
    if ((threadIdx.x & 63) < kCoopWords && i < n) atomicAdd(&c.tot[i], sum);
  }
  __syncthreads();
  ++c.pass;
}

// Width sums of this workgroup's chunk at n candidate lambdas (lam[0 .. n) in LDS), summed over the
// workgroup into red[0 .. n) (LDS, zero on entry).  se[j][k] = held score j times eps[k], +inf for
// the options past the last (their cost is never the smallest, so all eight are walked without a
// branch); valid[j]: the thread has a j-th score.
template <int HELD, int SETS, int NOPT>
__device__ void coop_chunk_sums(const float* __restrict__ row, const CoopCtx& c, const float (&se)[HELD][NOPT],
                                const bool (&valid)[HELD], const float* lam, int n, const Options& o, int* red) {
  // Two candidates a step (one with more than five options, whose products take too many registers): their sums go
  // through the rows of sixteen lanes as the halves of one integer (16 lanes of up to eight widths of at most 255).
  constexpr int kEach = NOPT <= 5 ? 2 : 1;
  const int set = __builtin_amdgcn_readfirstlane(threadIdx.x / kCoopLanes), lane = threadIdx.x % kCoopLanes;
  for (int i = kEach * set; i < n; i += kEach * SETS) {
    float lb[kEach][NOPT];
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const float at = lam[i + e < n ? i + e : i];
#pragma unroll
      for (int k = 0; k < NOPT; ++k) lb[e][k] = __fmul_rn(at, o.bits[k]);
    }
    int acc = 0;
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      int sum = 0;
#pragma unroll
      for (int j = 0; j < HELD; ++j) {
        float best = __fadd_rn(se[j][0], lb[e][0]);
        int width = o.ibits[0];
#pragma unroll
        for (int k = 1; k < NOPT; ++k) {
          const float cst = __fadd_rn(se[j][k], lb[e][k]);
          const bool lt = cst < best;                                  // strict: the first minimum wins
          best = lt ? cst : best;
          width = lt ? o.ibits[k] : width;
        }
        sum += valid[j] ? width : 0;
      }
      acc |= sum << (16 * e);
    }
    // the wavefront's sum without a trip through LDS per step: within rows of sixteen lanes by
    // lane permutations, then the four row totals
    acc += __builtin_amdgcn_update_dpp(0, acc, 0xB1, 0xF, 0xF, false);     // lane ^ 1
    acc += __builtin_amdgcn_update_dpp(0, acc, 0x4E, 0xF, 0xF, false);     // lane ^ 2
    acc += __builtin_amdgcn_update_dpp(0, acc, 0x141, 0xF, 0xF, false);    // mirror within eight
    acc += __builtin_amdgcn_update_dpp(0, acc, 0x140, 0xF, 0xF, false);    // mirror within sixteen
    int total[kEach];
#pragma unroll
    for (int e = 0; e < kEach; ++e) total[e] = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t v = (uint32_t)__builtin_amdgcn_readlane(acc, 16 * r);
      total[0] += (int)(v & 0xffffu);
      if (kEach == 2) total[kEach - 1] += (int)(v >> 16);
    }
    if (HELD == 8 && c.t1 - c.t0 > HELD * kCoopLanes) {      // (uniform) a chunk beyond what is held
#pragma unroll
      for (int e = 0; e < kEach; ++e) {
        int rest = 0;
        for (int t = c.t0 + lane + HELD * kCoopLanes; t < c.t1; t += kCoopLanes) {
          int width;
          choose(row[t], o, lb[e], width);
          rest += width;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) rest += __shfl_xor(rest, off, 64);
        total[e] += rest;
      }
    }
    if ((threadIdx.x & 63) == 0) {
      atomicAdd(&red[i], total[0]);
      if (kEach == 2 && i + 1 < n) atomicAdd(&red[i + 1], total[kEach - 1]);
    }
  }
  __syncthreads();
}

// The midpoints that four bisection levels over (lo, hi) can reach: node 1 is that of the interval itself, node 2n
// that of the lower half of node n's, node 2n + 1 that of the upper half.  Thread n goes its own way down to node n (one
// thread writing all fifteen in turn, with divisions: 0.7 us of a pass).  (Halving by a product is the same
// correctly rounded number as the reference's division by two.)
__device__ __forceinline__ void coop_midpoints(float lo, float hi, float* cand) {
  const int n = threadIdx.x;
  if (n >= 1 && n < 16) {
    float mid = __fmul_rn(__fadd_rn(lo, hi), 0.5f);
    for (int bit = 30 - __clz(n); bit >= 0; --bit) {
      if ((n >> bit) & 1) lo = mid; else hi = mid;
      mid = __fmul_rn(__fadd_rn(lo, hi), 0.5f);
    }
    cand[n] = mid;
  }
}

__global__ void coop_init_kernel(uint32_t* state, int64_t n_words) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_words) state[i] = 0u;
}

// Wavefronts that a SIMD has room for: with the products of five options at most and up to four scores a thread the
// kernel fits 64 registers (two of one set's, five options, go to scratch; 62 .. 83 with eight products always held), beyond
// that 128.
constexpr int coop_waves(int held, int options) { return held <= 4 && options <= 5 ? 8 : 4; }
// (NOPT: the options are walked to a compile-time count, the usual four or five, or all eight)
template <int HELD, int SETS, int NOPT>
__global__ void __launch_bounds__(SETS * kCoopLanes) __attribute__((amdgpu_waves_per_eu(coop_waves(HELD, NOPT))))
knapsack_coop_kernel(const float* __restrict__ scores, int64_t stride_b, int group_rows, int T, int S,
                     Budget budget, Options o, int max_iters, float tol,
                     uint32_t* __restrict__ state, void* __restrict__ out, int out_elem_size,
                     int64_t out_stride_b, int* __restrict__ counts) {
  __shared__ int lds[64];
  __shared__ int red[kCoopWords];
  __shared__ int tot[kCoopWords];
  __shared__ float cand[kCoopWords + 1];   // the pass's candidate lambdas (and the next doubling base)
  __shared__ int failed;
  const int b = blockIdx.x / S;
  CoopCtx c;
  c.S = S; c.sub = blockIdx.x % S;
  const int chunk = (T + S - 1) / S;
  c.t0 = min(T, c.sub * chunk);
  c.t1 = min(T, c.t0 + chunk);
  c.words = state + (int64_t)b * kCoopRowWords;
  c.pass = 0;
  c.tot = tot;
  c.failed = &failed;
  if (threadIdx.x < kCoopWords) red[threadIdx.x] = 0;
  if (threadIdx.x == 0) failed = 0;
  const float* row = scores + (int64_t)b * stride_b;
  const float bud = budget(b);
  float se[HELD][NOPT];
  bool valid[HELD];
  float m = -__builtin_inff();
#pragma unroll
  for (int j = 0; j < HELD; ++j) {
    const int t = c.t0 + (int)(threadIdx.x % kCoopLanes) + j * kCoopLanes;
    valid[j] = t < c.t1;
    const float v = valid[j] ? row[t] : 0.f;
    if (valid[j]) m = fmaxf(m, v);
#pragma unroll
    for (int k = 0; k < NOPT; ++k) se[j][k] = k < o.n ? __fmul_rn(v, o.eps[k]) : __builtin_inff();
  }
  for (int t = c.t0 + (int)threadIdx.x + HELD * kCoopLanes; t < c.t1; t += SETS * kCoopLanes) m = fmaxf(m, row[t]);
  __syncthreads();

  // ---- the row maximum
  m = block_reduce(m, MaxF(), reinterpret_cast<float*>(lds));
  if (threadIdx.x == 0) {
    const uint32_t bits = rdkv_float_to_ordered(m);
    red[0] = (int)(bits >> 16);
    red[1] = (int)(bits & 0xffffu);
  }
  __syncthreads();
  coop_exchange<true, SETS>(c, 2, red);
  const float lam0 = fmaxf(__fmul_rn(rdkv_ordered_to_float((uint32_t)tot[0]), 0.375f), 1e-8f);
  __syncthreads();
  if (threadIdx.x < 2) red[threadIdx.x] = 0;

  // ---- first pass: lam0 itself (the first candidate of the doubling rounds) together with what the
  // bisection starts with when the row needs no doubling, which is the usual case: lambda = 0 and the
  // 15 midpoints of four bisection levels over (0, lam0).  A row that does need doubling goes through
  // the rounds 15 candidates at a time and bisects from scratch.
  // d: the first k with avg(lam0 * 2^k) <= budget
  int d = -1;
  {
    if (threadIdx.x == 0) {
      cand[0] = lam0;
      cand[1] = 0.f;
    }
    coop_midpoints(0.f, lam0, cand + 1);
    __syncthreads();
    coop_chunk_sums<HELD, SETS, NOPT>(row, c, se, valid, cand, 17, o, red);
    coop_exchange<false, SETS>(c, 17, red);
    if ((int)threadIdx.x < 17) red[threadIdx.x] = 0;
    if (!(__fdiv_rn((float)tot[0], (float)T) > bud)) d = 0;
    __syncthreads();
    float lam = __fmul_rn(lam0, 2.0f);
    for (int base = 1; base < kMaxDoublings && d < 0; base += 15) {
      const int n = min(15, kMaxDoublings - base);
      if (threadIdx.x == 0) {
        for (int i = 0; i < n; ++i) {
          cand[i] = lam;
          lam = __fmul_rn(lam, 2.0f);
        }
        cand[kCoopWords] = lam;
      }
      __syncthreads();
      lam = cand[kCoopWords];
      coop_chunk_sums<HELD, SETS, NOPT>(row, c, se, valid, cand, n, o, red);
      coop_exchange<false, SETS>(c, n, red);
      if ((int)threadIdx.x < n) red[threadIdx.x] = 0;
      for (int i = 0; i < n; ++i) {
        const float avg = __fdiv_rn((float)tot[i], (float)T);
        if (!(avg > bud)) {
          d = base + i;
          break;
        }
      }
      __syncthreads();
    }
    if (d < 0) d = kMaxDoublings;
  }
  // (d == 0: the first pass's sums of lambda = 0 and the 15 midpoints are what the bisection's first pass needs)
  bool have_first = d == 0;
  // ---- the rounds the row's group executes (as in knapsack_bisect_kernel): every row publishes
  // its lam0 and doublings, every workgroup reads those of its group
  const int r0 = (b / group_rows) * group_rows;
  {
    if (c.sub == 0 && threadIdx.x < 3) {
      const uint32_t bits = __float_as_uint(lam0);
      const uint32_t v = threadIdx.x == 0 ? bits >> 16 : (threadIdx.x == 1 ? bits & 0xffffu : (uint32_t)d);
      __hip_atomic_store(&c.words[2 * kCoopMaxSplit * kCoopWords + threadIdx.x], (0xA5u << 24) | v, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);            // (the rows of a group sit on different dies)
    }
    // The group can only lower this row's count when another row's rounds end early, and they
    // end no earlier than this row's own lambda reaches 1e12 (g_own, below): while g_own + 1 >= d
    // the minimum leaves d as it is whatever the other rows say, and nothing is waited for.
    int g_own = kMaxDoublings + 1;
    if (d > 0) {
      float lam = lam0;
      for (int it = 0; it < kMaxDoublings; ++it) {
        if (it < d) lam = __fmul_rn(lam, 2.0f);
        if (lam >= 1e12f) { g_own = it; break; }
      }
    }
    const bool ask_group = g_own + 1 < d;
    int dmax = 0, gmax = 0;
    for (int r = r0 + threadIdx.x; ask_group && r < r0 + group_rows; r += blockDim.x) {
      const uint32_t* gw = state + (int64_t)r * kCoopRowWords + 2 * kCoopMaxSplit * kCoopWords;
      uint32_t w3[3] = {0u, 0u, 0u};
      for (int spins = 0;; ++spins) {                      // the three words together, until all carry the tag
#pragma unroll
        for (int k = 0; k < 3; ++k) w3[k] = __hip_atomic_load(&gw[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((w3[0] >> 24) == 0xA5u && (w3[1] >> 24) == 0xA5u && (w3[2] >> 24) == 0xA5u) break;
        if (failed || spins > kCoopSpinLimit) {
          failed = 1;
          w3[0] = w3[1] = w3[2] = 0u;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      const uint32_t hi = w3[0] & kCoopValueMask, lo = w3[1] & kCoopValueMask;
      const int dr = (int)(w3[2] & kCoopValueMask);
      float lam = __uint_as_float((hi << 16) | lo);
      int g = kMaxDoublings + 1;                     // never reaches 1e12
      for (int it = 0; it < kMaxDoublings; ++it) {
        if (it < dr) lam = __fmul_rn(lam, 2.0f);
        if (lam >= 1e12f) { g = it; break; }
      }
      dmax = max(dmax, dr);
      gmax = max(gmax, g);
    }
    if (ask_group) {                                   // (uniform over the workgroup)
      dmax = block_reduce(dmax, MaxI(), lds);
      gmax = block_reduce(gmax, MaxI(), lds);
      __syncthreads();
      const int rounds = min(min(dmax, gmax + 1), kMaxDoublings);
      d = min(d, rounds);
    }
  }
  float lam_hi = lam0;
  for (int i = 0; i < d; ++i) lam_hi = __fmul_rn(lam_hi, 2.0f);

  // ---- bisection, four levels per pass: node 1 is the midpoint of (lo, hi), node 2n that of the
  // lower half of node n's interval, node 2n + 1 that of the upper half
  float lam_lo = 0.f, lam_final = 0.f;
  {
    const float denom = fmaxf(bud, 1e-8f);
    bool first = true, done = max_iters <= 0;
    int it = 0;
    // (with max_iters = 0 the reference still evaluates lambda = 0, but nothing depends on it)
    while (!done) {
      const int at = have_first ? 1 : 0;   // where lambda = 0 sits in cand / tot; the nodes follow it
      if (!have_first) {
        if (threadIdx.x == 0) cand[0] = 0.f;   // lambda = 0 decides whether to bisect at all (first pass; unused afterwards)
        coop_midpoints(lam_lo, lam_hi, cand);
        __syncthreads();
        coop_chunk_sums<HELD, SETS, NOPT>(row, c, se, valid, cand, 16, o, red);
        coop_exchange<false, SETS>(c, 16, red);
        if (threadIdx.x < kCoopWords) red[threadIdx.x] = 0;
      }
      have_first = false;
      if (first) {
        first = false;
        if (__fdiv_rn((float)tot[at], (float)T) <= bud) done = true;
      }
      // every node's comparisons at once, one in each of sixteen lanes, then the way down over their bits
      const float avg = __fdiv_rn((float)tot[at + (threadIdx.x & 15)], (float)T);
      const uint32_t hit = (uint32_t)__ballot(__fdiv_rn(fabsf(__fsub_rn(avg, bud)), denom) < tol);
      const uint32_t over = (uint32_t)__ballot(avg > bud);
      int node = 1, last = 0, lo_node = 0, hi_node = 0;
      for (int lvl = 0; lvl < 4 && !done; ++lvl) {
        last = node;
        ++it;
        if ((hit >> node) & 1) {
          done = true;
        } else if ((over >> node) & 1) {
          lo_node = node;
          node = 2 * node + 1;
        } else {
          hi_node = node;
          node = 2 * node;
        }
        if (it >= max_iters) done = true;
      }
      if (last) lam_final = cand[at + last];
      if (lo_node) lam_lo = cand[at + lo_node];
      if (hi_node) lam_hi = cand[at + hi_node];
      __syncthreads();                                // everyone has read the totals before the next pass rewrites them
    }
  }

  // ---- the allocation of this workgroup's chunk and the per-option counts of the row
  {
    float lb[NOPT];
#pragma unroll
    for (int n = 0; n < NOPT; ++n) lb[n] = n < o.n ? __fmul_rn(lam_final, o.bits[n]) : 0.f;
    int cnt[NOPT];
#pragma unroll
    for (int n = 0; n < NOPT; ++n) cnt[n] = 0;
    uint8_t* out_row = reinterpret_cast<uint8_t*>(out) + (int64_t)b * out_stride_b * out_elem_size;
    const bool bad = failed != 0;
    for (int t = c.t0 + threadIdx.x; t < c.t1; t += blockDim.x) {
      int w;
      const int idx = choose(row[t], o, lb, w);
      if (bad) w = 255;
#pragma unroll
      for (int n = 0; n < NOPT; ++n) cnt[n] += (n == idx) ? 1 : 0;
      if (out_elem_size == 1) out_row[t] = (uint8_t)w;
      else reinterpret_cast<int64_t*>(out_row)[t] = (int64_t)w;
    }
    if (counts != nullptr) {
#pragma unroll
      for (int n = 0; n < NOPT; ++n) {
        if (n < o.n) {
          int v = cnt[n];
          v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);
          v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);
          v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, false);
          v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, false);
          const int total = __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) +
                            __builtin_amdgcn_readlane(v, 32) + __builtin_amdgcn_readlane(v, 48);
          if ((threadIdx.x & 63) == 0) atomicAdd(&red[n], total);
        }
      }
      __syncthreads();
      coop_exchange<false, SETS>(c, o.n, red);
      if (c.sub == 0 && (int)threadIdx.x < o.n) counts[(int64_t)b * o.n + threadIdx.x] = tot[threadIdx.x];
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The same solver for short rows (a head's channels): a wavefront per row with the row in registers
// and a workgroup per group of rows, so that a pass has no barrier, the rows' doublings meet in LDS,
// and one launch replaces two.  Bound by its chain of dependent passes (a wavefront sum each).
// A call of 8 rows of 128 / 256 scores 18.3 / 19.7 -> 11.3 / 11.6 us (the host side of the call), 256
// rows of 128 19.9 -> 11.2.
// ---------------------------------------------------------------------------------------------
constexpr int kGroupMaxRows = kMaxThreads / 64;
constexpr int kGroupMaxHeld = 4;

// Sum over the wavefront, in every lane.
__device__ __forceinline__ int wave_sum_uniform(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);     // lane ^ 1
  v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);     // lane ^ 2
  v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, false);    // mirror within eight
  v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, false);    // mirror within sixteen
  return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) + __builtin_amdgcn_readlane(v, 32) +
         __builtin_amdgcn_readlane(v, 48);
}

// The rows first .. first + group_rows, by the first group_rows wavefronts of the workgroup (the others meet its one
// barrier).  taken(row, score, width): called by the lane of every score.  Returns the counts of the wavefront's row.
template <int NOPT>
struct GroupCounts {
  int n[NOPT];
};
template <int HELD, int NOPT, typename Taken>
__device__ __forceinline__ GroupCounts<NOPT> knapsack_group_rows(const float* __restrict__ scores, int64_t stride_b, int first,
                                                                 int group_rows, int T, const Budget& budget, const Options& o,
                                                                 int max_iters, float tol, Taken taken) {
  __shared__ float s_lam0[kGroupMaxRows];
  __shared__ int s_d[kGroupMaxRows];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = first + (wave < group_rows ? wave : 0);
  const float* row = scores + (int64_t)b * stride_b;
  const float bud = budget(b);
  float se[HELD][NOPT];       // score times eps (+inf for the options past the last: never the smallest)
  float m = -__builtin_inff();
#pragma unroll
  for (int j = 0; j < HELD; ++j) {
    const int t = lane + 64 * j;
    const float v = t < T ? row[t] : 0.f;
    if (t < T) m = fmaxf(m, v);
#pragma unroll
    for (int k = 0; k < NOPT; ++k) se[j][k] = k < o.n ? __fmul_rn(v, o.eps[k]) : __builtin_inff();
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  // the option of held score j at the lambda whose products are in lb: index and width
  auto pick = [&](int j, const float (&lb)[NOPT], int& width) __attribute__((always_inline)) {
    float best = __fadd_rn(se[j][0], lb[0]);
    int idx = 0;
    width = o.ibits[0];
#pragma unroll
    for (int k = 1; k < NOPT; ++k) {
      const float cst = __fadd_rn(se[j][k], lb[k]);
      const bool lt = cst < best;                                  // strict: the first minimum wins
      best = lt ? cst : best;
      idx = lt ? k : idx;
      width = lt ? o.ibits[k] : width;
    }
    return idx;
  };
  auto solve = [&](float lam) __attribute__((always_inline)) {
    float lb[NOPT];
#pragma unroll
    for (int k = 0; k < NOPT; ++k) lb[k] = __fmul_rn(lam, o.bits[k]);
    int acc = 0;
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
      int width;
      pick(j, lb, width);
      acc += lane + 64 * j < T ? width : 0;
    }
    return __fdiv_rn((float)wave_sum_uniform(acc), (float)T);
  };

  // the doublings the row asks for on its own
  const float lam0 = fmaxf(__fmul_rn(m, 0.375f), 1e-8f);
  int d = 0;
  {
    float lam = lam0;
    for (; d < kMaxDoublings; ++d) {
      if (!(solve(lam) > bud)) break;
      lam = __fmul_rn(lam, 2.0f);
    }
  }
  if (lane == 0 && wave < group_rows) {
    s_lam0[wave] = lam0;
    s_d[wave] = d;
  }
  __syncthreads();
  // the rounds its group executes (as in knapsack_bisect_kernel): lane r replays row r
  int dmax = 0, gmax = 0;
  if (lane < group_rows) {
    float lam = s_lam0[lane];
    dmax = s_d[lane];
    gmax = kMaxDoublings + 1;                      // never reaches 1e12
    for (int it = 0; it < kMaxDoublings; ++it) {
      if (it < dmax) lam = __fmul_rn(lam, 2.0f);
      if (lam >= 1e12f) { gmax = it; break; }
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    dmax = max(dmax, __shfl_xor(dmax, off, 64));
    gmax = max(gmax, __shfl_xor(gmax, off, 64));
  }
  const int mine = min(d, min(min(dmax, gmax + 1), kMaxDoublings));
  float lam_hi = lam0;
  for (int i = 0; i < mine; ++i) lam_hi = __fmul_rn(lam_hi, 2.0f);

  float lam_lo = 0.f, lam_final = 0.f;
  if (!(solve(0.f) <= bud)) {
    const float denom = fmaxf(bud, 1e-8f);
    for (int it = 0; it < max_iters; ++it) {
      const float mid = __fdiv_rn(__fadd_rn(lam_lo, lam_hi), 2.0f);
      const float avg = solve(mid);
      lam_final = mid;
      const float rel = __fdiv_rn(fabsf(__fsub_rn(avg, bud)), denom);
      if (rel < tol) break;
      if (avg > bud) lam_lo = mid; else lam_hi = mid;
    }
  }
  float lb[NOPT];
#pragma unroll
  for (int k = 0; k < NOPT; ++k) lb[k] = __fmul_rn(lam_final, o.bits[k]);
  GroupCounts<NOPT> cnt;
#pragma unroll
  for (int k = 0; k < NOPT; ++k) cnt.n[k] = 0;
#pragma unroll
  for (int j = 0; j < HELD; ++j) {
    const int t = lane + 64 * j;
    int w;
    const int idx = pick(j, lb, w);
    if (t < T) {
#pragma unroll
      for (int k = 0; k < NOPT; ++k) cnt.n[k] += k == idx ? 1 : 0;
      if (wave < group_rows) taken(b, t, w);
    }
  }
  return cnt;
}

template <int HELD, int NOPT>
__global__ void __launch_bounds__(kMaxThreads)
knapsack_group_kernel(const float* __restrict__ scores, int64_t stride_b, int group_rows, int T,
                      Budget budget, Options o, int max_iters, float tol, void* __restrict__ out,
                      int out_elem_size, int64_t out_stride_b, int* __restrict__ counts) {
  const auto cnt = knapsack_group_rows<HELD, NOPT>(
      scores, stride_b, blockIdx.x * group_rows, group_rows, T, budget, o, max_iters, tol, [&](int b, int t, int w) {
        if (out_elem_size == 1) reinterpret_cast<uint8_t*>(out)[(int64_t)b * out_stride_b + t] = (uint8_t)w;
        else reinterpret_cast<int64_t*>(out)[(int64_t)b * out_stride_b + t] = (int64_t)w;
      });
  if (counts != nullptr) {
    const int b = blockIdx.x * group_rows + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int k = 0; k < NOPT; ++k) {
      if (k < o.n) {
        const int total = wave_sum_uniform(cnt.n[k]);
        if ((threadIdx.x & 63) == 0) counts[(int64_t)b * o.n + k] = total;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The K allocation of a layer and the token order of its V allocation in one launch: neither needs the other, and both
// stand between the V allocation and the host, which sizes the packed tensors by what they find.  As launches of
// their own (the K rows 7 us on one compute unit, a histogram of the widths, the order) they followed each other.
//  * Workgroup (0, 0): the K rows, a wavefront each; their class counts.
//  * Workgroups (chunk, 1 + head): 1024 tokens of a head each.  What lies ahead of its tokens a workgroup counts itself,
//    from all of the row's bytes (16 a load; a dword's four widths by one count of set bits per class), instead of reading
//    a histogram that another launch has written; beyond 64k tokens that would be more than the histogram's launch.
// With the exchange words cleared by the pooling launch, three launches instead of nine (two of them conversions of the
// widths to int16) up to the host's read: a selected layer of 8 heads, 4k / 31k tokens 108.0 / 109.8 -> 97.1 / 97.3 us.
// Results and words as plan_hist_kernel and plan_scatter_kernel leave them (pack_plan.hip).
// ---------------------------------------------------------------------------------------------
constexpr int kOrderThreads = 1024;
constexpr int64_t kOrderMaxTokens = 65536;
struct OrderArgs {
  const uint8_t* v_bits;          // rows of v_stride bytes, a multiple of 16
  int64_t v_stride;
  int T, H;
  int32_t *order, *rank3;         // [H, T]
  int32_t *counts4, *info;
  uint32_t* minmax;
  int minmax_per_head, D;
  int16_t *v16, *k16;             // the widths as [H, T] and [H, D], or null
  uint64_t* words;
  uint32_t tag;
};
struct KRows {
  const float* scores;
  int64_t stride_b;
  Options o;
  uint8_t* out;                   // [H, D]
};

__device__ __forceinline__ int width_class(uint32_t w) {
  return w == 2 ? 0 : w == 4 ? 1 : w == 8 ? 2 : w == 16 ? 3 : w == 0 ? 4 : 5;
}

template <int HELD, int NOPT>
__global__ void __launch_bounds__(kOrderThreads)
select_order_kernel(OrderArgs a, KRows k, Budget budget, int max_iters, float tol) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (blockIdx.y == 0) {
    if (blockIdx.x > 0) return;
    int own[4] = {0, 0, 0, 0};    // this lane's channels of 2, 4, 8 or 16 bit, and of another width
    knapsack_group_rows<HELD, NOPT>(k.scores, k.stride_b, 0, a.H, a.D, budget, k.o, max_iters, tol, [&](int b, int t, int w) {
      k.out[(int64_t)b * a.D + t] = (uint8_t)w;
      if (a.k16) a.k16[(int64_t)b * a.D + t] = (int16_t)w;
      own[0] += w == 2 ? 1 : 0;
      own[1] += w == 4 ? 1 : 0;
      own[2] += w == 8 || w == 16 ? 1 : 0;
      own[3] += w != 0 && w != 2 && w != 4 && w != 8 && w != 16 ? 1 : 0;
    });
    if (wave < a.H) {
      const int n2 = wave_sum_uniform(own[0]), n4 = wave_sum_uniform(own[1]), n8 = wave_sum_uniform(own[2]);
      const int bad = wave_sum_uniform(own[3]);
      if (lane < 6) {
        const int v = lane == 0 ? n2 : lane == 1 ? n4 : lane == 2 ? n8 : lane == 3 ? bad : 0;
        a.info[8 * wave + 2 + lane] = v;
        rdkv_host_word(a.words, 12 * (int64_t)wave + 6 + lane, a.tag, v);
      }
    }
    return;
  }
  constexpr int kWaves = kOrderThreads / 64;
  __shared__ int wsum[kWaves][10];             // all of the row's tokens by class 2, 4, 8, 16 bit, other; those ahead
  __shared__ int wcnt[kWaves][6], wpre[kWaves][6], red[12];
  const int h = blockIdx.y - 1, chunk = blockIdx.x, T = a.T;
  const uint8_t* row = a.v_bits + (int64_t)h * a.v_stride;
  const int t = chunk * kOrderThreads + tid;
  const uint32_t width = t < T ? row[t] : 0u;
  int all[5] = {0, 0, 0, 0, 0}, ahead[5] = {0, 0, 0, 0, 0};
  const int vectors = (T + 15) / 16, before = chunk * (kOrderThreads / 16);
  for (int v = tid; v < vectors; v += kOrderThreads) {
    const uint4 q = reinterpret_cast<const uint4*>(row)[v];
    uint32_t w[4] = {q.x, q.y, q.z, q.w};
    int n[5] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int left = T - (16 * v + 4 * e);         // bytes past the row's end hold anything
      if (left < 4) w[e] = left <= 0 ? 0u : w[e] & ((1u << (8 * left)) - 1u);
      const uint32_t one = w[e] & 0x1e1e1e1eu;
      // (more bits in a byte than the widths have, or more than one of them: byte by byte)
      const uint32_t two = one & ((one | 0x80808080u) - 0x01010101u) & 0x1e1e1e1eu;
      if (one != w[e] || two != 0) {
        for (int i = 0; i < 4; ++i) {
          const int c = width_class((w[e] >> (8 * i)) & 255u);
#pragma unroll
          for (int m = 0; m < 4; ++m) n[m] += c == m ? 1 : 0;
          n[4] += c == 5 ? 1 : 0;
        }
      } else {
#pragma unroll
        for (int m = 0; m < 4; ++m) n[m] += __popc(one & (0x02020202u << m));
      }
    }
#pragma unroll
    for (int m = 0; m < 5; ++m) {
      all[m] += n[m];
      ahead[m] += v < before ? n[m] : 0;
    }
  }
#pragma unroll
  for (int m = 0; m < 5; ++m) {
    const int s_all = wave_sum_uniform(all[m]), s_ahead = wave_sum_uniform(ahead[m]);
    if (lane == 0) {
      wsum[wave][m] = s_all;
      wsum[wave][5 + m] = s_ahead;
    }
  }
  const int cls = t < T ? width_class(width) : -1;
  int my_rank = 0;
  uint64_t qmask = 0;
  auto lanes_below = [](uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
  };
#pragma unroll
  for (int m = 0; m < 6; ++m) {
    const uint64_t in = __ballot(cls == m);
    if (m < 3) qmask |= in;
    if (cls == m) my_rank = lanes_below(in);
    if (lane == 0) wcnt[wave][m] = __popcll(in);
  }
  const int my_q = lanes_below(qmask);
  __syncthreads();
  if (tid < 10) {
    int s = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s += wsum[w][tid];
    red[tid < 4 ? tid : tid == 4 ? 5 : tid < 9 ? 1 + tid : 11] = s;      // [0 .. 5] all, [6 .. 11] ahead, by class
  } else if (tid >= 64 && tid < 70) {
    const int m = tid - 64;
    int s = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      wpre[w][m] = s;
      s += wcnt[w][m];
    }
  }
  __syncthreads();
  // (class 4, evicted, is what the others leave)
  const int evicted = T - (red[0] + red[1] + red[2] + red[3] + red[5]);
  const int evicted_ahead = chunk * kOrderThreads - (red[6] + red[7] + red[8] + red[9] + red[11]);
  int pos = 0, before_q = 0, base = 0;
#pragma unroll
  for (int m = 0; m < 6; ++m) {
    const int before_me = (m == 4 ? evicted_ahead : red[6 + m]) + wpre[wave][m];
    if (cls == m) pos = base + before_me + my_rank;
    if (m < 3) before_q += before_me;
    base += m == 4 ? evicted : red[m];
  }
  if (t < T) {
    a.order[(int64_t)h * T + pos] = t;
    a.rank3[(int64_t)h * T + t] = before_q + my_q;
    if (a.v16) a.v16[(int64_t)h * T + t] = (int16_t)width;
  }
  if (chunk == 0) {
    if (tid < 6) {
      const int v = tid == 4 ? evicted : red[tid];
      if (tid < 4) a.counts4[4 * h + tid] = v;
      else a.info[8 * h + tid - 4] = v;
      rdkv_host_word(a.words, 12 * (int64_t)h + tid, a.tag, v);
    }
    for (int i = tid; a.minmax && i < a.minmax_per_head; i += kOrderThreads)
      a.minmax[(int64_t)h * a.minmax_per_head + i] = rdkv_float_to_ordered(((i / a.D) & 1) ? -__builtin_inff() : __builtin_inff());
  }
}

// Independent rows with lambda kept in double (the single-row solver applied to each row).
__global__ void __launch_bounds__(kMaxThreads)
knapsack_rows_kernel(const float* __restrict__ scores, int64_t stride_b, int T,
                     const double* __restrict__ budget, Options o, int max_iters, double tol,
                     void* __restrict__ out, int out_elem_size, int64_t out_stride_b,
                     int* __restrict__ counts) {
  __shared__ int lds[32];
  const int b = blockIdx.x;
  const float* row = scores + (int64_t)b * stride_b;
  const double bud = budget[b];
  double lam_lo = 0.0;
  double lam_hi = (double)row_max(row, T, reinterpret_cast<float*>(lds)) * 0.375;
  double avg = (double)solve_avg(row, T, (float)lam_hi, o, lds);
  for (int rounds = 0; avg > bud && lam_hi < 1e12 && rounds < 2200; ++rounds) {
    lam_hi *= 2.0;
    avg = (double)solve_avg(row, T, (float)lam_hi, o, lds);
  }
  double lam_final = 0.0;
  if (!((double)solve_avg(row, T, 0.f, o, lds) <= bud)) {
    const double denom = bud > 1e-8 ? bud : 1e-8;
    for (int it = 0; it < max_iters; ++it) {
      const double mid = (lam_lo + lam_hi) / 2.0;
      avg = (double)solve_avg(row, T, (float)mid, o, lds);
      lam_final = mid;
      if (fabs(avg - bud) / denom < tol) break;
      if (avg > bud) lam_lo = mid; else lam_hi = mid;
    }
  }
  emit(row, T, (float)lam_final, o, reinterpret_cast<uint8_t*>(out) + (int64_t)b * out_stride_b * out_elem_size,
       out_elem_size, counts ? counts + (int64_t)b * o.n : nullptr, lds);
}

// out[b, l] over the window l-pad .. l-pad+k-1 of row b; left-to-right fp32 sum from 0, one division.
template <bool AVG, bool REFLECT>
__global__ void pool_kernel(const float* __restrict__ in, int64_t in_stride_b, int T, int k, int pad,
                            float* __restrict__ out, int64_t out_stride_b, int L, uint32_t* clear, int clear_words) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  // (the row's exchange words of the allocation that follows, for which they would be a launch ahead of it)
  for (int i = l; i < clear_words; i += gridDim.x * blockDim.x) clear[(int64_t)blockIdx.y * clear_words + i] = 0u;
  if (l >= L) return;
  const float* row = in + (int64_t)blockIdx.y * in_stride_b;
  float acc = AVG ? 0.f : -__builtin_inff();
  for (int j = 0; j < k; ++j) {
    int i = l + j - pad;
    float v;
    if (REFLECT) {
      if (i < 0) i = -i;
      if (i >= T) i = 2 * (T - 1) - i;
      v = row[i];
    } else {
      v = (i >= 0 && i < T) ? row[i] : (AVG ? 0.f : -__builtin_inff());
    }
    acc = AVG ? __fadd_rn(acc, v) : fmaxf(acc, v);
  }
  if (AVG) acc = __fdiv_rn(acc, (float)k);
  out[(int64_t)blockIdx.y * out_stride_b + l] = acc;
}

int fail(const char* msg) {
  rdkv_set_error("%s", msg);
  return RDKV_EINVAL;
}

// Per-head K budget of the joint selection as a launch of its own: k_budget_bits / (head_dim * max(kept, 1)) evaluated
// the way the reference's tensor expression is: fp32 product, fp32 reciprocal, fp32 product.
__global__ void k_budget_kernel(const int32_t* __restrict__ counts, int n_options, int zero_col, int rows,
                                int tokens, float head_dim, float k_budget_bits, float* __restrict__ out) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  out[r] = Budget{nullptr, counts, n_options, zero_col, tokens, head_dim, k_budget_bits}(r);
}

int make_options(const float* bits_host, const float* eps_host, int n, Options* o) {
  if (bits_host == nullptr || eps_host == nullptr || n < 1 || n > kMaxOptions)
    return fail("knapsack: need 1..8 bit options");
  o->n = n;
  for (int i = 0; i < kMaxOptions; ++i) {
    const float b = i < n ? bits_host[i] : 0.f;
    if (!(b >= 0.f && b <= 255.f) || b != (float)(int)b)
      return fail("knapsack: bit options must be integers in 0..255");
    o->bits[i] = b;
    o->ibits[i] = (int)b;
    o->eps[i] = i < n ? eps_host[i] : 0.f;
  }
  return 0;
}

int threads_for(int64_t T) {
  int64_t t = ((T + 63) / 64) * 64;
  return (int)(t < 64 ? 64 : (t > kMaxThreads ? kMaxThreads : t));
}

int check_common(const void* scores, int B, int64_t T, const void* budget, const void* out, int out_elem_size) {
  if (B < 0 || T < 0) return fail("knapsack: negative size");
  if (B > 0 && T == 0) return fail("knapsack: rows are empty (no maximum)");
  if (T > (1 << 20)) return fail("knapsack: rows longer than 2^20 tokens are not supported");
  if (B > 0 && (scores == nullptr || budget == nullptr || out == nullptr)) return fail("knapsack: null pointer");
  if (out_elem_size != 1 && out_elem_size != 8) return fail("knapsack: out_elem_size must be 1 or 8");
  return 0;
}

}  // namespace

// 0 / 1 / 2: the kernel that holds 2 / 4 / 8 scores of a chunk per thread in registers
static int coop_held_index(int64_t chunk) { return chunk <= 2 * kCoopLanes ? 0 : (chunk <= 4 * kCoopLanes ? 1 : 2); }

typedef void (*CoopKernel)(const float*, int64_t, int, int, int, Budget, Options, int, float, uint32_t*, void*, int, int64_t, int*);
// [up to four / five / eight options][sets 1 / 2 / 4][scores held]
#define RDKV_COOP_SETS(SETS, NOPT) {knapsack_coop_kernel<2, SETS, NOPT>, knapsack_coop_kernel<4, SETS, NOPT>, knapsack_coop_kernel<8, SETS, NOPT>}
#define RDKV_COOP(NOPT) {RDKV_COOP_SETS(1, NOPT), RDKV_COOP_SETS(2, NOPT), RDKV_COOP_SETS(4, NOPT)}
static const CoopKernel kCoopKernels[3][3][3] = {RDKV_COOP(4), RDKV_COOP(5), RDKV_COOP(kMaxOptions)};

// Workgroups a row is shared by in the cooperative form (0: one workgroup per row, the two-launch
// form): a power of two, chunks of at least 512 scores, at most 64 per row, at most 3.5 / 2.5 / 2 workgroups per compute
// unit by the scores held, and only when that gives a row at least sixteen (with fewer, one workgroup per row was as fast or
// faster on 64 rows of 32k scores) - or all that its length allows for a row of 1024 .. 8191 in a launch of at
// most kCoopShortGrid workgroups.  A call of 8 rows in two launches / shared: 1024 scores 34.6 / 21.7 us, 2048
// 39.3 / 22.4, 3000 46.8 / 26.6, 4096 41.1 / 23.6; 64 rows of 1024 / 2048 34.6 / 24.7 and 40.9 / 23.5; 256 rows of 4096,
// which would get two each, 52.4 / 58.0; 8 of 512, one each, 27.
// kernel: the workgroups' sets (log2).  One set / the rule's: 8 rows of 4096 / 16k / 31k scores 34.6 / 23.6, 36.3 / 28.8,
// 43.0 / 33.5, 64 rows of 2048 29.0 / 23.5; and a row is shared by half as many where that makes room for a second set and
// a thread still holds its scores (16 rows of 16k 36.0 -> 31.9).
// The workgroups of a launch wait for each other, so launches on streams of their own must find room together, or each
// holds what the others wait for until the bound ends all of them.  Four run side by side on the hardware queues that a
// process has by default.  So a launch takes sets only while it leaves room for three more like it, or, from 4096 scores
// on, for as many as its one-set form did (two or three, for more than about one workgroup per compute unit).  Room is
// counted in eighths of a SIMD's registers, whatever the kernel: one, two or four workgroups' wavefronts of 64 or 128
// registers are powers of two of them, and what is short of room is never kept out by smaller pieces for good.  (Sets taken up
// to half of a kernel's slots: three selections of 8 x 31k side by side had no room, and 2 rows of 128k took four sets,
// 43.2 us against 44.6 now.)
constexpr int64_t kCoopShortGrid = 512;
static int coop_split_rule(int cus, int B, int64_t T, int max_iters, int n_options, int* kernel) {
  if (B <= 0 || T < 1024 || max_iters > kCoopMaxIters) return 0;
  auto held_of = [T](int64_t split) { return coop_held_index((T + split - 1) / split); };
  constexpr int kMost[3] = {7, 5, 4};            // halves of a workgroup per compute unit, by scores held
  int64_t S = T / 512;
  if (S > kCoopMaxSplit) S = kCoopMaxSplit;
  // (a shorter split means longer chunks, which can select the next kernel: settle in at most three steps)
  // (a power of two: chunks of a whole number of scores per thread measured faster than the larger
  // split in between - 16 rows of 32k: 68 us with 32 workgroups per row, 74 us with 40)
  auto pow2_floor = [](int64_t v) { int64_t p = 1; while (2 * p <= v) p *= 2; return v >= 1 ? p : 0; };
  S = pow2_floor(S);
  const int64_t allowed = S;
  for (int step = 0; step < 3 && S >= 1; ++step) {
    const int64_t cap = (int64_t)cus * kMost[held_of(S)] / 2 / B;
    if (S <= cap) break;
    S = pow2_floor(cap);
  }
  if (S < 1 || (int64_t)B * S > (int64_t)cus * kMost[held_of(S)] / 2) return 0;
  if (S < 16 && !(T < 8192 && S == allowed && (int64_t)B * S <= kCoopShortGrid)) return 0;
  const int64_t beside = T < 4096 ? 4 : std::min<int64_t>(4, (int64_t)cus * kMost[held_of(S)] / (B * S));
  auto fits = [&](int64_t split, int e) {
    return ((int64_t)B * split << e) * beside <= (int64_t)cus * coop_waves(2 << held_of(split), n_options);
  };
  auto sets_for = [&](int64_t split) { return fits(split, 2) ? 2 : fits(split, 1) ? 1 : 0; };
  if (T < 4096 && !fits(S, 0)) return 0;
  *kernel = sets_for(S);
  if (*kernel == 0 && S >= 32 && (T + S / 2 - 1) / (S / 2) <= 8 * kCoopLanes && sets_for(S / 2) > 0) {
    S /= 2;
    *kernel = sets_for(S);
  }
  // (a chunk's width sum must fit the 24 value bits of an exchange word)
  return (T + S - 1) / S <= 32768 ? (int)S : 0;
}
static int coop_split(int B, int64_t T, int max_iters, int n_options, int* kernel) {
  if (B <= 0 || T < 1024 || max_iters > kCoopMaxIters) return 0;
  static int cus_of_device[64];            // (0 = not asked yet; a race between first callers writes the same value)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cus_of_device[dev] == 0) {
    int cus = 0;                           // (asked again next time where it fails)
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return 0;
    cus_of_device[dev] = cus;
  }
  return coop_split_rule(cus_of_device[dev], B, T, max_iters, n_options, kernel);
}

RDKV_API int rdkv_knapsack_split(int compute_units, int B, int64_t T, int max_iters, int n_options, int* sets) {
  int kernel = 0;
  const int S = coop_split_rule(compute_units, B, T, max_iters, n_options, &kernel);
  *sets = S ? 1 << kernel : 0;
  return S;
}

RDKV_API int64_t rdkv_knapsack_workspace_bytes(int B) {
  const int64_t b = B > 0 ? B : 0;
  return b * 8 + 256 + b * (int64_t)kCoopRowWords * 4;
}

static uint32_t* coop_state(void* workspace, int B) {
  return reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(workspace) + (((int64_t)B * 8 + 255) / 256) * 256);
}

static int knapsack_batched(const float* scores, int64_t stride_b, int B, int64_t T, const Budget& budget,
                            const void* given, const float* bits_host, const float* eps_host, int n_options, int max_iters, float tol,
                            int group_rows, void* out, int out_elem_size, int64_t out_stride_b, int32_t* counts,
                            void* workspace, int64_t workspace_bytes, void* stream, bool cleared = false) {
  Options o;
  if (int rc = make_options(bits_host, eps_host, n_options, &o)) return rc;
  if (int rc = check_common(scores, B, T, given, out, out_elem_size)) return rc;
  if (B == 0) return 0;
  if (workspace == nullptr || workspace_bytes < rdkv_knapsack_workspace_bytes(B))
  {
    rdkv_set_error("rdkv_knapsack_batched: workspace too small");
    return RDKV_EWORKSPACE;
  }
  if (max_iters < 0) return fail("knapsack: negative max_iters");
  if (group_rows <= 0) group_rows = B;
  if (B % group_rows != 0) return fail("knapsack: the batch is not a whole number of row groups");
  float* lam0 = reinterpret_cast<float*>(workspace);
  int* doublings = reinterpret_cast<int*>(lam0 + B);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  int sets = 0;      // (log2)
  if (const int S = coop_split(B, T, max_iters, o.n, &sets)) {
    // few long rows: every row shared by S workgroups, one launch after clearing its state
    uint32_t* state = coop_state(workspace, B);
    const int64_t n_words = (int64_t)B * kCoopRowWords;
    if (!cleared)
      hipLaunchKernelGGL(coop_init_kernel, dim3((unsigned)rdkv_cdiv(n_words, 256)), dim3(256), 0, s, state, n_words);
    const int64_t chunk = (T + S - 1) / S;
    hipLaunchKernelGGL(kCoopKernels[o.n <= 4 ? 0 : o.n == 5 ? 1 : 2][sets][coop_held_index(chunk)], dim3((unsigned)(B * S)), dim3(kCoopLanes << sets), 0, s,
                       scores, stride_b, group_rows, (int)T, S,
                       budget, o, max_iters, tol, state, out, out_elem_size, out_stride_b, counts);
    RDKV_CHECK_LAUNCH("rdkv_knapsack_batched");
    return RDKV_OK;
  }
  if (T <= 64 * kGroupMaxHeld && group_rows <= kGroupMaxRows) {
    // short rows: a wavefront per row, a workgroup per group (the rows of a group meet in LDS: at most sixteen, the
    // wavefronts of a workgroup; longer rows have no registers left per lane and are the other form's)
#define RDKV_LAUNCH_GROUP(HELD, NOPT)                                                                              \
  hipLaunchKernelGGL((knapsack_group_kernel<HELD, NOPT>), dim3(B / group_rows), dim3(64 * group_rows), 0, s, scores, \
                     stride_b, group_rows, (int)T, budget, o, max_iters, tol, out, out_elem_size, out_stride_b, counts)
    if (T <= 128 && o.n <= 5) RDKV_LAUNCH_GROUP(2, 5);
    else if (o.n <= 5) RDKV_LAUNCH_GROUP(4, 5);
    else RDKV_LAUNCH_GROUP(4, kMaxOptions);
#undef RDKV_LAUNCH_GROUP
    RDKV_CHECK_LAUNCH("rdkv_knapsack_batched");
    return RDKV_OK;
  }
  const int threads = threads_for(T);
  hipLaunchKernelGGL(knapsack_expand_kernel, dim3(B), dim3(threads), 0, s, scores, stride_b, (int)T, budget, o,
                     lam0, doublings);
  hipLaunchKernelGGL(knapsack_bisect_kernel, dim3(B), dim3(threads), 0, s, scores, stride_b, group_rows, (int)T, budget,
                     o, max_iters, tol, lam0, doublings, out, out_elem_size, out_stride_b, counts);
  RDKV_CHECK_LAUNCH("rdkv_knapsack_batched");
  return RDKV_OK;
}

RDKV_API int rdkv_knapsack_batched(const float* scores, int64_t stride_b, int B, int64_t T,
                                   const float* budget, const float* bits_host, const float* eps_host,
                                   int n_options, int max_iters, float tol, int group_rows, void* out,
                                   int out_elem_size, int64_t out_stride_b, int32_t* counts, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  return knapsack_batched(scores, stride_b, B, T, Budget{budget, nullptr, 0, 0, 0, 0.f, 0.f}, budget, bits_host, eps_host,
                          n_options, max_iters, tol, group_rows, out, out_elem_size, out_stride_b, counts, workspace,
                          workspace_bytes, stream);
}

RDKV_API int rdkv_knapsack_batched_value(const float* scores, int64_t stride_b, int B, int64_t T, float value,
                                         const int32_t* kept_counts, int kept_options, int zero_option, int64_t tokens,
                                         int head_dim, const float* bits_host, const float* eps_host, int n_options,
                                         int max_iters, float tol, int group_rows, void* out, int out_elem_size,
                                         int64_t out_stride_b, int32_t* counts, void* workspace, int64_t workspace_bytes,
                                         void* stream) {
  if (kept_counts != nullptr && (kept_options < 1 || kept_options > kMaxOptions || zero_option >= kept_options || tokens < 0 ||
                                 tokens > 0x7fffffffLL || head_dim < 1 || kept_counts == counts))
    return fail("knapsack: bad counts for the budget");
  return knapsack_batched(scores, stride_b, B, T,
                          Budget{nullptr, kept_counts, kept_options, zero_option, (int)tokens, (float)head_dim, value}, scores,
                          bits_host, eps_host, n_options, max_iters, tol, group_rows, out, out_elem_size, out_stride_b, counts,
                          workspace, workspace_bytes, stream);
}

RDKV_API int rdkv_knapsack_rows(const float* scores, int64_t stride_b, int B, int64_t T, const double* budget,
                                const float* bits_host, const float* eps_host, int n_options, int max_iters,
                                double tol, void* out, int out_elem_size, int64_t out_stride_b,
                                int32_t* counts, void* stream) {
  Options o;
  if (int rc = make_options(bits_host, eps_host, n_options, &o)) return rc;
  if (int rc = check_common(scores, B, T, budget, out, out_elem_size)) return rc;
  if (B == 0) return 0;
  if (max_iters < 0) return fail("knapsack: negative max_iters");
  hipLaunchKernelGGL(knapsack_rows_kernel, dim3(B), dim3(threads_for(T)), 0, reinterpret_cast<hipStream_t>(stream),
                     scores, stride_b, (int)T, budget, o, max_iters, tol, out, out_elem_size, out_stride_b, counts);
  RDKV_CHECK_LAUNCH("rdkv_knapsack_rows");
  return RDKV_OK;
}

static int pool_scores(const float* scores, int64_t stride_b, int B, int64_t T, int kernel_size, int is_avg, int reflect,
                       float* out, int64_t out_stride_b, uint32_t* clear, void* stream) {
  if (B < 0 || T < 0 || kernel_size < 1) return fail("pool_scores: bad size");
  if (T > (1 << 30)) return fail("pool_scores: row too long");
  int k = kernel_size;
  if (reflect) {
    if (T <= 0) return fail("pool_scores: cannot reflect-pool an empty score sequence");
    if (k > 2 * T - 1) k = (int)(2 * T - 1);
  }
  const int pad = k / 2;
  const int64_t L = T + 2 * pad - k + 1;
  if (L <= 0) return fail("pool_scores: output would be empty");
  if (B == 0) return 0;
  if (scores == nullptr || out == nullptr) return fail("pool_scores: null pointer");
  if (B > 65535) return fail("pool_scores: more than 65535 rows");
  const dim3 grid((unsigned)((L + 255) / 256), (unsigned)B), block(256);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
#define RDKV_POOL(A, R) \
  hipLaunchKernelGGL((pool_kernel<A, R>), grid, block, 0, s, scores, stride_b, (int)T, k, pad, out, out_stride_b, (int)L, \
                     clear, clear ? kCoopRowWords : 0)
  if (is_avg) { if (reflect) RDKV_POOL(true, true); else RDKV_POOL(true, false); }
  else        { if (reflect) RDKV_POOL(false, true); else RDKV_POOL(false, false); }
#undef RDKV_POOL
  RDKV_CHECK_LAUNCH("rdkv_pool_scores");
  return RDKV_OK;
}

RDKV_API int rdkv_pool_scores(const float* scores, int64_t stride_b, int B, int64_t T, int kernel_size,
                              int is_avg, int reflect, float* out, int64_t out_stride_b, void* stream) {
  return pool_scores(scores, stride_b, B, T, kernel_size, is_avg, reflect, out, out_stride_b, nullptr, stream);
}

// What rdkv_pool_scores, the V and the K allocation and rdkv_pack_layer_plan_start do for a layer, in three launches.
RDKV_API int rdkv_select_layer_start(const float* scores, int64_t stride_b, int H, int64_t T, int kernel_size, int is_avg,
                                     int reflect, float* pooled, float v_budget, const float* v_bits_host,
                                     const float* v_eps_host, int n_v_options, int zero_option, uint8_t* v_bits,
                                     int64_t v_stride, int32_t* v_counts, const float* channels, int64_t channel_stride, int D,
                                     float k_kept_bits, const float* k_bits_host, const float* k_eps_host, int n_k_options,
                                     uint8_t* k_bits, int max_iters, float tol, int32_t* order, int32_t* rank3, int32_t* plan,
                                     float* minmax_ws, int minmax_floats_per_head, int16_t* v_bits16, int16_t* k_bits16,
                                     uint64_t* host_words, uint32_t tag, void* workspace, int64_t workspace_bytes, void* stream) {
  if (H < 1 || H > kGroupMaxRows || T < 1 || T > kOrderMaxTokens || D < 1 || D > 64 * kGroupMaxHeld) {
    rdkv_set_error("rdkv_select_layer_start: %d heads of %lld tokens and %d channels", H, (long long)T, D);
    return RDKV_EUNSUPPORTED;
  }
  if (!v_counts || !channels || !k_bits || !order || !rank3 || !plan || !host_words || v_stride < T || v_stride % 16 != 0 ||
      reinterpret_cast<uintptr_t>(v_bits) % 16 != 0 || zero_option >= n_v_options || channel_stride < D)
    return fail("rdkv_select_layer_start: bad arguments");
  if (kernel_size > 1 && (reflect ? std::min<int64_t>(kernel_size, 2 * T - 1) : kernel_size) % 2 == 0)
    return fail("rdkv_select_layer_start: an even kernel changes the rows' length");
  if (workspace == nullptr || workspace_bytes < rdkv_knapsack_workspace_bytes(H)) {
    rdkv_set_error("rdkv_select_layer_start: workspace too small");
    return RDKV_EWORKSPACE;
  }
  if (max_iters < 0) return fail("knapsack: negative max_iters");
  Options ko;
  if (int rc = make_options(k_bits_host, k_eps_host, n_k_options, &ko)) return rc;
  bool cleared = false;
  const float* rows = scores;
  int64_t row_stride = stride_b;
  if (kernel_size > 1) {
    int sets = 0;
    cleared = coop_split(H, T, max_iters, n_v_options, &sets) > 0;
    if (int rc = pool_scores(scores, stride_b, H, T, kernel_size, is_avg, reflect, pooled, T, cleared ? coop_state(workspace, H) : nullptr,
                             stream))
      return rc;
    rows = pooled;
    row_stride = T;
  }
  if (int rc = knapsack_batched(rows, row_stride, H, T, Budget{nullptr, nullptr, 0, 0, 0, 0.f, v_budget}, rows, v_bits_host, v_eps_host,
                                n_v_options, max_iters, tol, H, v_bits, 1, v_stride, v_counts, workspace, workspace_bytes, stream,
                                cleared))
    return rc;
  OrderArgs a;
  a.v_bits = v_bits; a.v_stride = v_stride; a.T = (int)T; a.H = H; a.order = order; a.rank3 = rank3;
  a.counts4 = plan; a.info = plan + 4 * H; a.minmax = reinterpret_cast<uint32_t*>(minmax_ws);
  a.minmax_per_head = minmax_floats_per_head; a.D = D; a.v16 = v_bits16; a.k16 = k_bits16; a.words = host_words; a.tag = tag;
  const KRows k = {channels, channel_stride, ko, k_bits};
  const Budget kept = {nullptr, v_counts, n_v_options, zero_option, (int)T, (float)D, k_kept_bits};
  const dim3 grid((unsigned)rdkv_cdiv(T, kOrderThreads), (unsigned)(H + 1));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
#define RDKV_LAUNCH_ORDER(HELD, NOPT) \
  hipLaunchKernelGGL((select_order_kernel<HELD, NOPT>), grid, dim3(kOrderThreads), 0, s, a, k, kept, max_iters, tol)
  if (D <= 128 && ko.n <= 5) RDKV_LAUNCH_ORDER(2, 5);
  else if (ko.n <= 5) RDKV_LAUNCH_ORDER(4, 5);
  else RDKV_LAUNCH_ORDER(4, kMaxOptions);
#undef RDKV_LAUNCH_ORDER
  RDKV_CHECK_LAUNCH("rdkv_select_layer_start");
  return RDKV_OK;
}

RDKV_API int rdkv_k_budget_per_head(const int32_t* counts, int n_options, int zero_option, int rows, int64_t T,
                                    int head_dim, float k_budget_bits, float* out, void* stream) {
  if (rows < 0 || n_options < 1 || n_options > kMaxOptions || zero_option >= n_options || T < 0 || head_dim < 1)
    return fail("k_budget_per_head: bad arguments");
  if (rows == 0) return RDKV_OK;
  if (counts == nullptr || out == nullptr) return fail("k_budget_per_head: null pointer");
  hipLaunchKernelGGL(k_budget_kernel, dim3((rows + 255) / 256), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     counts, n_options, zero_option, rows, (int)T, (float)head_dim, k_budget_bits, out);
  RDKV_CHECK_LAUNCH("rdkv_k_budget_per_head");
  return RDKV_OK;
}
