// Channel tables and padding mask of a packed layer, for the launches that write them (pack_plan.hip, quantize.hip).
#pragma once
#include "rdkv_common.h"

namespace {

constexpr int kPlanThreads = 1024;

__device__ __forceinline__ int load_int(const void *p, int elem_size, int64_t i) {
  switch (elem_size) {
    case 1: return reinterpret_cast<const uint8_t *>(p)[i];
    case 2: return reinterpret_cast<const int16_t *>(p)[i];
    case 4: return reinterpret_cast<const int32_t *>(p)[i];
    default: {
      const int64_t v = reinterpret_cast<const int64_t *>(p)[i];
      return (v < -1 || v > 1 << 20) ? -1 : (int)v;
    }
  }
}

// widths above 8 are stored as 8 bit; 0 = pruned (-1); anything else is invalid (-2)
__device__ __forceinline__ int channel_class(int bits) {
  return bits == 2 ? 0 : bits == 4 ? 1 : (bits == 8 || bits == 16) ? 2 : bits == 0 ? -1 : -2;
}

__device__ __forceinline__ int lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
}

// One workgroup per KV head: channel tables with the layer-wide padded segment sizes and the
// per-head scalars.
struct LayerTables {
  const void *k_bits;
  int kb_es;
  int64_t kb_stride_h;
  int D, G;
  const int32_t *counts4, *info;
  int n2p, n4p, n8o, kept_max;
  int64_t max_tv;
  int32_t *slot_channel;              // or null: nobody reads it
  int64_t *perm, *perm_q, *sort_ph;
  int32_t *seg_ph, *seg_tok, *t_eff, *t_eff_k, *n_v16;
};
struct LayerMask {
  const int32_t *counts4;
  int G;
  int64_t max_tv, max_tk;
  float *mask;
  const int32_t *ord_ref, *rank_ref;
  int64_t tv_ref;
  int64_t *sort_idx;
};

__device__ __forceinline__ void layer_tables_block(const LayerTables &a, int h) {
  const void *k_bits = a.k_bits;
  const int kb_es = a.kb_es, D = a.D, G = a.G, n2p = a.n2p, n4p = a.n4p, n8o = a.n8o, kept_max = a.kept_max;
  const int64_t kb_stride_h = a.kb_stride_h;
  const int32_t *counts4 = a.counts4, *info = a.info;
  int32_t *slot_channel = a.slot_channel, *seg_ph = a.seg_ph, *seg_tok = a.seg_tok, *t_eff = a.t_eff,
          *t_eff_k = a.t_eff_k, *n_v16 = a.n_v16;
  int64_t *perm = a.perm, *perm_q = a.perm_q, *sort_ph = a.sort_ph;
  __shared__ int wcnt[kPlanThreads / 64][3];
  __shared__ int wpre[kPlanThreads / 64][3];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = blockDim.x >> 6;
  const int Dp = n2p + n4p + n8o;
  const int n2 = info[8 * h + 2], n4 = info[8 * h + 3];
  for (int j = tid; j < Dp; j += blockDim.x) {
    if (slot_channel) slot_channel[(int64_t)h * Dp + j] = -1;
    perm[(int64_t)h * Dp + j] = 0;
  }
  for (int j = tid; j < kept_max; j += blockDim.x) sort_ph[(int64_t)h * kept_max + j] = 0;
  if (tid < 3) {
    seg_ph[3 * h + tid] = info[8 * h + 2 + tid];
    seg_tok[3 * h + tid] = counts4[4 * h + tid];
  }
  if (tid == 0) {
    const int tv = counts4[4 * h] + counts4[4 * h + 1] + counts4[4 * h + 2], n16 = counts4[4 * h + 3];
    t_eff[h] = tv;
    t_eff_k[h] = tv + n16;
    n_v16[h] = n16;
  }
  const int ch = tid;                                   // D <= blockDim (checked by the host)
  const int cls = ch < D ? channel_class(load_int(k_bits, kb_es, (int64_t)h * kb_stride_h + ch)) : -1;
  int my_rank = 0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const uint64_t m = __ballot(cls == k);
    if (cls == k) my_rank = lanes_below(m);
    if (lane == 0) wcnt[wave][k] = __popcll(m);
  }
  __syncthreads();
  if (tid < 3) {
    int s = 0;
    for (int w = 0; w < nwaves; ++w) { wpre[w][tid] = s; s += wcnt[w][tid]; }
  }
  __syncthreads();                                      // also orders the fills above before the scatter
  if (cls >= 0) {
    const int r = wpre[wave][cls] + my_rank;
    const int slot = (cls == 0 ? 0 : cls == 1 ? n2p : n2p + n4p) + r;
    const int sorted = (cls == 0 ? 0 : cls == 1 ? n2 : n2 + n4) + r;
    if (slot_channel) slot_channel[(int64_t)h * Dp + slot] = ch;
    perm[(int64_t)h * Dp + slot] = ch;
    sort_ph[(int64_t)h * kept_max + sorted] = ch;
  }
  __syncthreads();
  for (int j = tid; j < G * Dp; j += blockDim.x)
    perm_q[((int64_t)h * G + j / Dp) * Dp + j % Dp] = perm[(int64_t)h * Dp + j % Dp];
}

// mask[hq, col] = 0 where the canvas column holds a token of head hq / G, -inf where it is padding;
// the first row of blocks also writes the sort index of head `ref`'s quantized tokens
// (sort_idx[i] = rank among them of the i-th token in sorted order).
__device__ __forceinline__ void softmax_mask_block(const LayerMask &a, int bx, int nbx, int hq) {
  const int h = hq / a.G;
  if (hq == 0) {
    for (int64_t i = (int64_t)bx * blockDim.x + threadIdx.x; i < a.tv_ref; i += (int64_t)nbx * blockDim.x)
      a.sort_idx[i] = a.rank_ref[a.ord_ref[i]];
  }
  const int64_t tv = (int64_t)a.counts4[4 * h] + a.counts4[4 * h + 1] + a.counts4[4 * h + 2], n16 = a.counts4[4 * h + 3];
  for (int64_t col = (int64_t)bx * blockDim.x + threadIdx.x; col < a.max_tk; col += (int64_t)nbx * blockDim.x) {
    const bool valid = col < tv || (col >= a.max_tv && col < a.max_tv + n16);
    a.mask[(int64_t)hq * a.max_tk + col] = valid ? 0.0f : -__builtin_inff();
  }
}

}  // namespace
