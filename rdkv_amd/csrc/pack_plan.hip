// Device-side planning for the whole-layer packer: everything the reference derives on the host
// from the per-head bit allocations (obkv_accel/packing.py:241-294 channel sort / prune / padding,
// :1417-1431 stable token sort by width, :1245-1260 padding mask, :1262-1316 per-head metadata) is
// computed here so that the host needs one small read (the per-head class sizes, which fix the
// shapes of the packed tensors) and no per-head loop.
#include "pack_tables.h"

namespace {

constexpr int kTokClasses = 6;      // 2, 4, 8, 16 bit, evicted (0), anything else

__device__ __forceinline__ int token_class(int bits) {
  return bits == 2 ? 0 : bits == 4 ? 1 : bits == 8 ? 2 : bits == 16 ? 3 : bits == 0 ? 4 : 5;
}

// Widths of up to eight layers of one shape, H heads each.
constexpr int kPlanLayers = 8;
struct PlanWidths {
  const void *v[kPlanLayers], *k[kPlanLayers];
  int64_t v_stride_h, k_stride_h;
  int v_es, k_es, H, T, D;
};

// Token planning in two launches over a (chunk, head) grid.  A thread takes four tokens of a chunk, 64 apart, a
// wavefront 256 neighbours: 32 heads of 32k tokens are one workgroup a compute unit (with one token a thread two rounds
// of four times the workgroups: 7 + 14 us for the pair, now 7.5 + 8.7).  Bound: the chain of a workgroup - widths, the
// counts of its wavefronts, the head's counts by chunk, the order's stores.
constexpr int kPlanTokens = 4;      // per thread
constexpr int kPlanChunk = kPlanThreads * kPlanTokens, kPlanWaves = kPlanThreads / 64;

// First launch: per-chunk class histogram hist[h][chunk][6]; the chunk-0 block of each head also
// counts the head's channel classes, writes the start values of its share of the K min / max scratch and, where asked
// for, the head's widths as bytes (invalid ones as 255).
__global__ void __launch_bounds__(kPlanThreads)
plan_hist_kernel(PlanWidths w, int32_t *__restrict__ hist, int32_t *__restrict__ info, uint32_t *__restrict__ minmax,
                 int minmax_per_head, uint8_t *__restrict__ k8) {
  __shared__ int wcnt[kPlanWaves][kTokClasses];
  __shared__ int kcnt[4];
  const int h = blockIdx.y, layer = h / w.H, hl = h - layer * w.H, chunk = blockIdx.x, nchunks = gridDim.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid < 4) kcnt[tid] = 0;
  const int t0 = chunk * kPlanChunk + wave * 64 * kPlanTokens + lane;
  int cls[kPlanTokens];
#pragma unroll
  for (int i = 0; i < kPlanTokens; ++i) {
    const int t = t0 + 64 * i;
    cls[i] = t < w.T ? token_class(load_int(w.v[layer], w.v_es, hl * w.v_stride_h + t)) : -1;
  }
#pragma unroll
  for (int k = 0; k < kTokClasses; ++k) {
    int n = 0;
#pragma unroll
    for (int i = 0; i < kPlanTokens; ++i) n += __popcll(__ballot(cls[i] == k));
    if (lane == 0) wcnt[wave][k] = n;
  }
  __syncthreads();
  if (chunk == 0) {
    if (minmax)
      for (int i = tid; i < minmax_per_head; i += kPlanThreads)
        minmax[(int64_t)h * minmax_per_head + i] = rdkv_float_to_ordered(((i / w.D) & 1) ? -INFINITY : INFINITY);
    int bad = 0;
    for (int ch = tid; ch < w.D; ch += kPlanThreads) {
      const int bits = load_int(w.k[layer], w.k_es, hl * w.k_stride_h + ch), kc = channel_class(bits);
      if (kc >= 0) atomicAdd(&kcnt[kc], 1);
      if (kc == -2) bad = 1;
      if (k8) k8[(int64_t)h * w.D + ch] = kc == -2 ? 255 : bits;
    }
    if (bad) atomicAdd(&kcnt[3], 1);
    __syncthreads();
    if (tid < 4) info[8 * h + 2 + tid] = kcnt[tid];
    if (tid >= 4 && tid < 6) info[8 * h + 2 + tid] = 0;
  }
  if (tid < kTokClasses) {
    int n = 0;
#pragma unroll
    for (int i = 0; i < kPlanWaves; ++i) n += wcnt[i][tid];
    hist[((int64_t)h * nchunks + chunk) * kTokClasses + tid] = n;
  }
}

// The sum over the 64 lanes, in every lane.
__device__ __forceinline__ int wave_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, true);       // quad_perm [1,0,3,2]
  v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, true);       // quad_perm [2,3,0,1]
  v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);      // row_half_mirror
  v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true);      // row_mirror
  const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
  v = (int)(r[0] + r[1]);
  const auto t = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
  return (int)(t[0] + t[1]);
}

// Second launch: every block sums the histograms of its head (class totals and what lies before
// its chunk) and scatters its tokens.  order[h, :] = token indices sorted by class, stable (the
// classes in the order 2, 4, 8, 16 bit, evicted, invalid); rank3[h, t] (or null) = number of tokens before
// t that are quantized (2/4/8 bit); counts4[h] = (n2, n4, n8, n16); info[h][0..1] = (evicted,
// invalid widths).
__global__ void __launch_bounds__(kPlanThreads)
plan_scatter_kernel(PlanWidths w, const int32_t *__restrict__ hist, int32_t *__restrict__ order, int64_t order_stride_h,
                    int32_t *__restrict__ rank3, int64_t rank3_stride_h, int32_t *__restrict__ counts4,
                    int32_t *__restrict__ info, uint64_t *__restrict__ host_words, uint32_t tag) {
  __shared__ int total[kTokClasses], before[kTokClasses];       // of the head, of its chunks before this one
  __shared__ int wcnt[kPlanWaves][kTokClasses];
  const int h = blockIdx.y, layer = h / w.H, hl = h - layer * w.H, chunk = blockIdx.x, nchunks = gridDim.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t0 = chunk * kPlanChunk + wave * 64 * kPlanTokens + lane;
  int cls[kPlanTokens];
#pragma unroll
  for (int i = 0; i < kPlanTokens; ++i) {
    const int t = t0 + 64 * i;
    cls[i] = t < w.T ? token_class(load_int(w.v[layer], w.v_es, hl * w.v_stride_h + t)) : -1;
  }
  if (wave < kTokClasses) {            // a class a wavefront
    int all = 0, ahead = 0;
    for (int c = lane; c < nchunks; c += 64) {
      const int v = hist[((int64_t)h * nchunks + c) * kTokClasses + wave];
      all += v;
      ahead += c < chunk ? v : 0;
    }
    all = wave_sum(all);
    ahead = wave_sum(ahead);
    if (lane == 0) {
      total[wave] = all;
      before[wave] = ahead;
    }
  }
  // of the wavefront's 256 tokens: those of a token's class before it, the quantized ones before it
  int rank[kPlanTokens], q_rank[kPlanTokens], run[kTokClasses], q_run = 0;
#pragma unroll
  for (int k = 0; k < kTokClasses; ++k) run[k] = 0;
#pragma unroll
  for (int i = 0; i < kPlanTokens; ++i) {
    uint64_t q = 0;
    rank[i] = 0;
#pragma unroll
    for (int k = 0; k < kTokClasses; ++k) {
      const uint64_t m = __ballot(cls[i] == k);
      if (k < 3) q |= m;
      if (cls[i] == k) rank[i] = run[k] + lanes_below(m);
      run[k] += __popcll(m);
    }
    q_rank[i] = q_run + lanes_below(q);
    q_run += __popcll(q);
  }
#pragma unroll
  for (int k = 0; k < kTokClasses; ++k)
    if (lane == 0) wcnt[wave][k] = run[k];
  __syncthreads();
  int base[kTokClasses], before_q = 0, seg_base = 0;     // where the wavefront's tokens of a class begin
#pragma unroll
  for (int k = 0; k < kTokClasses; ++k) {
    int ahead = before[k];
    // (lane i holds what wavefront i counted)
    ahead += wave_sum(lane < wave ? wcnt[lane & (kPlanWaves - 1)][k] : 0);
    base[k] = seg_base + ahead;
    if (k < 3) before_q += ahead;
    seg_base += total[k];
  }
#pragma unroll
  for (int i = 0; i < kPlanTokens; ++i) {
    const int t = t0 + 64 * i;
    int pos = rank[i];
#pragma unroll
    for (int k = 0; k < kTokClasses; ++k) pos += cls[i] == k ? base[k] : 0;
    if (t < w.T) {
      order[(int64_t)h * order_stride_h + pos] = t;
      if (rank3) rank3[(int64_t)h * rank3_stride_h + t] = before_q + q_rank[i];
    }
  }
  if (chunk == 0) {
    if (tid < 4) counts4[4 * h + tid] = total[tid];
    if (tid == 4) info[8 * h + 0] = total[4];
    if (tid == 5) info[8 * h + 1] = total[5];
    // the head's twelve numbers to the host, each word with the call's tag: whole whenever its tag is there
    if (host_words && tid < 12) {
      const int v = tid < 6 ? total[tid] : info[8 * h + tid - 4];
      rdkv_host_word(host_words, 12 * (int64_t)h + tid, tag, v);
    }
  }
}

__global__ void __launch_bounds__(kPlanThreads) layer_tables_kernel(LayerTables a) { layer_tables_block(a, blockIdx.x); }

__global__ void __launch_bounds__(256) softmax_mask_kernel(LayerMask a) {
  softmax_mask_block(a, blockIdx.x, gridDim.x, blockIdx.y);
}

// Both in one launch (heads of up to 256 channels): blocks [0, H_kv) build the channel tables, the
// nbx * H_q blocks after them write the mask - two launches of a few microseconds each were a
// tenth of a 32k-token layer's packing time.
__global__ void __launch_bounds__(256) layer_tables_mask_kernel(LayerTables t, LayerMask m, int H_kv, int nbx) {
  const int b = blockIdx.x;
  if (b < H_kv) {
    layer_tables_block(t, b);
  } else {
    const int r = b - H_kv;
    softmax_mask_block(m, r % nbx, nbx, r / nbx);
  }
}

bool elem_size_ok(int es) { return es == 1 || es == 2 || es == 4 || es == 8; }

}  // namespace

RDKV_API int64_t rdkv_pack_layer_plan_ints(int H_kv, int64_t T) {
  if (H_kv < 0 || T < 0) return 0;
  return (int64_t)H_kv * (12 + kTokClasses * rdkv_cdiv(T, kPlanThreads));      // (the histograms take a quarter of theirs)
}

// n_layers of a plan from layer `first` on: their rows of order, rank3, counts and info, their part of the histograms
static void launch_plan(const PlanWidths &w, int n_heads, int64_t first_head, int64_t all_heads, int32_t *order,
                        int64_t order_stride_h, int32_t *rank3, int64_t rank3_stride_h, int32_t *plan, float *minmax_ws,
                        int minmax_floats_per_head, uint8_t *k8, uint64_t *host_words, uint32_t tag, hipStream_t s) {
  const int64_t nchunks = rdkv_cdiv(w.T, kPlanChunk), f = first_head;
  int32_t *counts4 = plan + 4 * f, *info = plan + 4 * all_heads + 8 * f, *hist = plan + 12 * all_heads + kTokClasses * nchunks * f;
  const dim3 grid((unsigned)nchunks, n_heads);
  hipLaunchKernelGGL(plan_hist_kernel, grid, dim3(kPlanThreads), 0, s, w, hist, info,
                     minmax_ws ? (uint32_t *)minmax_ws + f * minmax_floats_per_head : nullptr, minmax_floats_per_head,
                     k8 ? k8 + f * w.D : nullptr);
  hipLaunchKernelGGL(plan_scatter_kernel, grid, dim3(kPlanThreads), 0, s, w, hist, order + f * order_stride_h, order_stride_h,
                     rank3 ? rank3 + f * rank3_stride_h : nullptr, rank3_stride_h, counts4, info,
                     host_words ? host_words + 12 * f : nullptr, tag);
}

RDKV_API int rdkv_pack_layer_plan_start(const void *v_bits, int vb_elem_size, int64_t vb_stride_h, const void *k_bits,
                                        int kb_elem_size, int64_t kb_stride_h, int H_kv, int64_t T, int D,
                                        int32_t *order, int64_t order_stride_h, int32_t *rank3,
                                        int64_t rank3_stride_h, int32_t *plan, float *minmax_ws,
                                        int minmax_floats_per_head, uint64_t *host_words, uint32_t tag, void *stream) {
  const char *fn = "rdkv_pack_layer_plan";
  RDKV_REQUIRE(H_kv >= 1 && H_kv <= 65535 && D >= 1 && T >= 1 && T <= (1LL << 30), "%s: bad shape", fn);
  RDKV_REQUIRE(elem_size_ok(vb_elem_size) && elem_size_ok(kb_elem_size), "%s: element sizes must be 1, 2, 4 or 8", fn);
  RDKV_REQUIRE(k_bits && plan && v_bits && order && rank3, "%s: null pointer", fn);
  const PlanWidths w{{v_bits}, {k_bits}, vb_stride_h, kb_stride_h, vb_elem_size, kb_elem_size, H_kv, (int)T, D};
  launch_plan(w, H_kv, 0, H_kv, order, order_stride_h, rank3, rank3_stride_h, plan, minmax_ws, minmax_floats_per_head, nullptr,
              host_words, tag, (hipStream_t)stream);
  RDKV_CHECK_LAUNCH(fn);
  return RDKV_OK;
}

RDKV_API int rdkv_plan_layers(const void *const *v_bits, int vb_elem_size, const void *const *k_bits, int kb_elem_size,
                              int n_layers, int H_kv, int64_t T, int D, int32_t *order, int32_t *plan, float *minmax_ws,
                              int minmax_floats_per_head, uint8_t *k_bits_u8, uint64_t *host_words, uint32_t tag,
                              void *stream) {
  const char *fn = "rdkv_plan_layers";
  RDKV_REQUIRE(n_layers >= 0 && H_kv >= 1 && H_kv <= 65535 / kPlanLayers && D >= 1 && T >= 1 && T <= (1LL << 30), "%s: bad shape",
               fn);
  RDKV_REQUIRE(elem_size_ok(vb_elem_size) && elem_size_ok(kb_elem_size), "%s: element sizes must be 1, 2, 4 or 8", fn);
  RDKV_REQUIRE(n_layers == 0 || (v_bits && k_bits && plan && order), "%s: null pointer", fn);
  for (int l = 0; l < n_layers; ++l) RDKV_REQUIRE(v_bits[l] && k_bits[l], "%s: null pointer", fn);
  for (int first = 0; first < n_layers; first += kPlanLayers) {
    const int n = n_layers - first < kPlanLayers ? n_layers - first : kPlanLayers;
    PlanWidths w{{}, {}, T, D, vb_elem_size, kb_elem_size, H_kv, (int)T, D};
    for (int l = 0; l < n; ++l) w.v[l] = v_bits[first + l], w.k[l] = k_bits[first + l];
    launch_plan(w, n * H_kv, (int64_t)first * H_kv, (int64_t)n_layers * H_kv, order, T, nullptr, 0, plan, minmax_ws,
                minmax_floats_per_head, k_bits_u8, host_words, tag, (hipStream_t)stream);
  }
  RDKV_CHECK_LAUNCH(fn);
  return RDKV_OK;
}

RDKV_API int rdkv_pack_layer_plan(const void *v_bits, int vb_elem_size, int64_t vb_stride_h, const void *k_bits,
                                  int kb_elem_size, int64_t kb_stride_h, int H_kv, int64_t T, int D,
                                  int32_t *order, int64_t order_stride_h, int32_t *rank3,
                                  int64_t rank3_stride_h, int32_t *plan, void *stream) {
  return rdkv_pack_layer_plan_start(v_bits, vb_elem_size, vb_stride_h, k_bits, kb_elem_size, kb_stride_h, H_kv, T, D, order,
                                    order_stride_h, rank3, rank3_stride_h, plan, nullptr, 0, nullptr, 0, stream);
}

RDKV_API int rdkv_pack_layer_tables(const void *k_bits, int kb_elem_size, int64_t kb_stride_h, int H_kv, int D,
                                    int G, const int32_t *counts4, const int32_t *info, int n2p, int n4p, int n8, int kept_max,
                                    int64_t max_tv, int max_n16, const int32_t *order, int64_t order_stride_h,
                                    const int32_t *rank3, int64_t rank3_stride_h, int ref_head, int64_t tv_ref,
                                    int32_t *slot_channel, int64_t *perm, int64_t *perm_for_q, int64_t *sort_ch,
                                    int32_t *seg_ch, int32_t *seg_tok, int32_t *t_eff, int32_t *t_eff_k,
                                    int32_t *n_v16, int64_t *sort_idx, float *softmax_mask, void *stream) {
  const char *fn = "rdkv_pack_layer_tables";
  RDKV_REQUIRE(H_kv >= 1 && H_kv <= 65535 && D >= 1 && D <= kPlanThreads && G >= 1, "%s: bad shape", fn);
  RDKV_REQUIRE(elem_size_ok(kb_elem_size), "%s: element size must be 1, 2, 4 or 8", fn);
  RDKV_REQUIRE(n2p >= 0 && n4p >= 0 && n8 >= 0 && n2p % 4 == 0 && n4p % 2 == 0 && kept_max >= 0 &&
                   kept_max <= n2p + n4p + n8, "%s: bad segment sizes", fn);
  RDKV_REQUIRE(max_tv >= 0 && max_n16 >= 0 && ref_head >= 0 && ref_head < H_kv && tv_ref >= 0 && tv_ref <= max_tv,
               "%s: bad token counts", fn);
  const int Dp = n2p + n4p + n8;
  RDKV_REQUIRE(k_bits && counts4 && info && seg_ch && seg_tok && t_eff && t_eff_k && n_v16, "%s: null pointer", fn);
  RDKV_REQUIRE(Dp == 0 || (slot_channel && perm && perm_for_q), "%s: null channel table", fn);
  RDKV_REQUIRE(kept_max == 0 || sort_ch, "%s: null channel sort table", fn);
  RDKV_REQUIRE(tv_ref == 0 || (sort_idx && order && rank3), "%s: null token tables", fn);
  hipStream_t s = (hipStream_t)stream;
  const int threads = ((D + 63) / 64) * 64;
  LayerTables t;
  t.k_bits = k_bits; t.kb_es = kb_elem_size; t.kb_stride_h = kb_stride_h; t.D = D; t.G = G;
  t.counts4 = counts4; t.info = info; t.n2p = n2p; t.n4p = n4p; t.n8o = n8; t.kept_max = kept_max; t.max_tv = max_tv;
  t.slot_channel = slot_channel; t.perm = perm; t.perm_q = perm_for_q; t.sort_ph = sort_ch;
  t.seg_ph = seg_ch; t.seg_tok = seg_tok; t.t_eff = t_eff; t.t_eff_k = t_eff_k; t.n_v16 = n_v16;
  const int64_t max_tk = max_tv + max_n16;
  if (max_tk > 0) {
    RDKV_REQUIRE(softmax_mask, "%s: null mask", fn);
    int64_t bx = rdkv_cdiv(max_tk, 256 * 4);
    if (bx > 1024) bx = 1024;
    LayerMask m;
    m.counts4 = counts4; m.G = G; m.max_tv = max_tv; m.max_tk = max_tk; m.mask = softmax_mask;
    m.ord_ref = order ? order + (int64_t)ref_head * order_stride_h : nullptr;
    m.rank_ref = rank3 ? rank3 + (int64_t)ref_head * rank3_stride_h : nullptr;
    m.tv_ref = tv_ref; m.sort_idx = sort_idx;
    const int64_t blocks = (int64_t)H_kv + bx * H_kv * G;
    if (threads <= 256 && blocks <= 0x7fffffffLL) {
      hipLaunchKernelGGL(layer_tables_mask_kernel, dim3((unsigned)blocks), dim3(256), 0, s, t, m, H_kv, (int)bx);
    } else {
      hipLaunchKernelGGL(layer_tables_kernel, dim3(H_kv), dim3(threads), 0, s, t);
      hipLaunchKernelGGL(softmax_mask_kernel, dim3((unsigned)bx, (unsigned)(H_kv * G)), dim3(256), 0, s, m);
    }
  } else {
    hipLaunchKernelGGL(layer_tables_kernel, dim3(H_kv), dim3(threads), 0, s, t);
  }
  RDKV_CHECK_LAUNCH(fn);
  return RDKV_OK;
}
