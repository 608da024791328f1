// Prefill packer that writes the streaming format (stream_format.h) straight from fp16 K / V:
// what the reference's per-layer composition (obkv_fast.py:1141-1155: per head build_packed_layer,
// packing.py:801-1013, then _pad_and_stack_per_head_layers, packing.py:1019-1317) followed by a
// re-layout would leave in the blob, bit for bit, without the padded intermediate.  Codes, scales
// and zero-points are those of the reference's quantizer (packing.py:141-165): V per token over
// its 128 channels, K per channel over the head's rows of the zero-padded canvas the reference
// re-quantizes K from (packing.py:1186-1215: a head with fewer rows than the layer's maxima has
// zero rows there, so 0 joins its per-channel min / max).
//
// Three launches for up to eight layers: the per-channel K min / max of every head (quantize.hip), one small
// workgroup per head that turns them into the quantizer of every channel and writes the unit's slot table, and
// resident workgroups that walk the heads' 64-token tiles, a quarter of a tile to each wavefront: it reads its tokens'
// K and V rows (gathered through the head's class-sorted token order) with 16-byte loads, quantizes them in
// registers, parks the codes in LDS as bytes, requests the next tile's rows and assembles this one's dwords from LDS
// meanwhile.  Between them the launches write every byte of the blob.
#include "rdkv_common.h"
#include <math.h>
#include <string.h>

#include <algorithm>
#include <cstddef>
#include <vector>

#include "stream_format.h"

#pragma clang fp contract(off)   // the quantizer rounds every product and sum on its own

namespace {

constexpr int kD = 128;
constexpr int kMaxSlots = 4 * RDKV_MAX_STEPS;

__device__ __forceinline__ int load_bits(const void *p, int elem_size, int64_t idx) {
  switch (elem_size) {
    case 1: return (int)reinterpret_cast<const uint8_t *>(p)[idx];
    case 2: return (int)reinterpret_cast<const int16_t *>(p)[idx];
    case 4: return (int)reinterpret_cast<const int32_t *>(p)[idx];
    default: return (int)reinterpret_cast<const int64_t *>(p)[idx];
  }
}

// The K row of a head with c2 / c4 / c8 channels at 2 / 4 / 8 bit.  Slot order: 8-bit channels, 4-bit, 2-bit, each
// padded to whole dwords (4 / 8 / 16 channels).  A narrow code is the same number in a wider field, so the stragglers
// of a narrow class move into the pad slots of the wider ones when that saves a whole dword of the row; a row still
// longer than 32 dwords is stored entirely as 8 bit.
struct RowPlan {
  int c4, c8;
  int m4, t8, t4;         // stragglers: 4-bit channels among the 8-bit slots, 2-bit ones among the 8- and 4-bit slots
  int n8, n4, n2;         // channels in the slots of a class
  int all8;               // 4- and 2-bit slots' channels follow the 8-bit ones
  int d8, d4, d2;
  __host__ __device__ static int pad_to(int n, int a) { return (a - n % a) % a; }
  __host__ __device__ RowPlan(int c2, int c4_, int c8_) : c4(c4_), c8(c8_), m4(0), t8(0), t4(0), all8(0) {
    const int r4 = c4 % 8;
    if (r4 > 0 && r4 <= pad_to(c8, 4)) m4 = r4;
    n8 = c8 + m4;
    n4 = c4 - m4;
    const int r2 = c2 % 16, p8 = pad_to(n8, 4), p4 = pad_to(n4, 8);
    if (r2 > 0 && r2 <= p8 + p4) {
      t8 = r2 < p8 ? r2 : p8;
      t4 = r2 - t8;
    }
    n8 += t8;
    n4 += t4;
    n2 = c2 - t8 - t4;
    all8 = (n8 + 3) / 4 + (n4 + 7) / 8 + (n2 + 15) / 16 > 32;
    d8 = ((all8 ? n8 + n4 + n2 : n8) + 3) / 4;
    d4 = all8 ? 0 : (n4 + 7) / 8;
    d2 = all8 ? 0 : (n2 + 15) / 16;
  }
  __host__ __device__ int slots() const { return 4 * (d8 + 2 * d4 + 4 * d2); }
  // what slot i holds: the position in the layer's padded sorted channel order, or -1
  __host__ __device__ int source(int i, int n2p, int n4p) const {
    int in8 = i, in4 = i - 4 * d8, in2 = in4 - 8 * d4;
    if (all8) in4 = i - n8, in2 = in4 - n4;
    if (in8 < (all8 ? n8 : 4 * d8))
      return in8 < c8 ? n2p + n4p + in8 : in8 < c8 + m4 ? n2p + c4 - m4 + in8 - c8 : in8 < n8 ? n2 + in8 - c8 - m4 : -1;
    if (in4 < (all8 ? n4 : 8 * d4)) return in4 < c4 - m4 ? n2p + in4 : in4 < n4 ? n2 + t8 + in4 - (c4 - m4) : -1;
    return in2 < n2 ? in2 : -1;
  }
};
__host__ __device__ inline int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }
// A unit's sections from `off` on (a multiple of 256); returns where they end.
__host__ __device__ inline int64_t lay_out_unit(const RowPlan &r, const int32_t *n_tok, int64_t off, RdkvUnit &u) {
  int64_t tiles[4], n_q_tiles = 0, n_tiles = 0;
  for (int c = 0; c < 4; ++c) {
    tiles[c] = ((int64_t)n_tok[c] + RDKV_TILE - 1) / RDKV_TILE;
    n_tiles += tiles[c];
    if (c < 3) n_q_tiles += tiles[c];
    u.n_tok[c] = n_tok[c];
  }
  u.d8 = r.d8;
  u.d4 = r.d4;
  u.d2 = r.d2;
  u.k_off = (uint64_t)off;
  off = align256(off + n_tiles * RDKV_TILE * 4 * (r.d8 + r.d4 + r.d2));
  for (int c = 0; c < 4; ++c) {
    u.v_off[c] = (uint64_t)off;
    off = align256(off + tiles[c] * rdkv_v_tile_bytes(c));
  }
  u.sz_off = (uint64_t)off;
  off = align256(off + n_q_tiles * RDKV_TILE * 4);
  u.qtab_off = (uint64_t)off;
  return align256(off + (int64_t)r.slots() * (int64_t)sizeof(RdkvSlot));
}

struct StreamPackArgs {
  const __half *K, *V;
  int64_t stride_h, stride_t;
  const int32_t *order;
  int64_t order_stride_h;
  const void *k_bits;
  int kb_elem_size;
  int64_t kb_stride_h;
  int n2p, n4p;                   // the layer's padded 2-bit / 4-bit channel counts (maxima over heads)
  int64_t max_tv;
  int max_n16;
  uint32_t *mm;                   // per head: 128 minima, 128 maxima (order-preserving integers)
  RdkvUnit *units;                // offsets relative to `blob`; written by the first launch where src_slot is null,
  const int32_t *counts, *info;   // ... from the plan's numbers
  const int16_t *src_slot;
  int n_slots_max, max_tiles;
  uint8_t *blob;
  uint32_t *scale_max;            // [2][H_kv] float bits: largest K channel scale, largest V token scale
  int H_kv;
  int64_t blob_bytes;
};
// The layers of a launch.  Where the host knows the tiles of every head, and the heads are few enough for a lane each,
// the packing workgroups of head r (over all layers) are begin[r] .. begin[r + 1] of a flat grid; otherwise every head
// has as many, and blockIdx is (workgroup, head, layer).
constexpr int kBatchLayers = 8, kTableHeads = 64;
struct StreamPackBatch {
  StreamPackArgs layer[kBatchLayers];
  int32_t begin[kTableHeads + 1];
  int32_t by_table;
};
// where a layer's channel parameters lie in its scratch
__device__ __forceinline__ float4 *chan_params_of(const StreamPackArgs &a) {
  return reinterpret_cast<float4 *>(a.mm + (int64_t)a.H_kv * 2 * kD);
}

// The K quantizer of one channel: scale, zero point, 1 / scale (rdkv_qcode's estimate) and, as bits,
// the channel's stream slot with its width class (slot | class << 8; -1 for a channel that is not
// kept).  slot_params_kernel makes them for every head of a batch's layers, the packing workgroups
// read them.
__device__ __forceinline__ float4 make_chan(float scale, float zp, float inv, int slot_cls) {
  return make_float4(scale, zp, inv, __int_as_float(slot_cls));
}

// One workgroup per head: stream slot -> position in the reference's padded sorted channel order
// (src_slot, or RowPlan where the unit is planned here) -> width class and rank in the class -> the rank-th
// channel of that width in ascending channel order (the stable sort of packing.py:241-294) -> the channel's parameters from its
// min / max.  Writes the per-channel parameters, the unit's slot table in the blob (with the
// alignment gap behind it, and behind the last head the rest of the blob: no byte of the blob is
// left to the caller), and starts the head's two scale maxima.
__global__ void __launch_bounds__(128)
slot_params_kernel(StreamPackBatch batch) {
  const StreamPackArgs &a = batch.layer[blockIdx.z];
  float4 *chan_params = chan_params_of(a);
  __shared__ int ch_of[3 * kD], first_wave_count[3], slot_of_ch[kD];
  __shared__ float4 slot_p[kMaxSlots];
  __shared__ float wave_max[2];
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  // the head's unit: given, or planned here as the host plans it (the heads ahead of it only for where it begins)
  const bool planned = a.src_slot == nullptr;
  const RowPlan row(planned ? a.info[8 * h + 2] : 0, planned ? a.info[8 * h + 3] : 0, planned ? a.info[8 * h + 4] : 0);
  RdkvUnit u;
  if (planned) {
    __shared__ int64_t ahead[2];
    int64_t off = 0;
    for (int i = tid; i < h; i += 128) {
      RdkvUnit other;
      off += lay_out_unit(RowPlan(a.info[8 * i + 2], a.info[8 * i + 3], a.info[8 * i + 4]), a.counts + 4 * i, 0, other);
    }
    for (int o = 1; o < 64; o <<= 1) off += __shfl_xor((long long)off, o, 64);
    if (lane == 0) ahead[tid >> 6] = off;
    __syncthreads();
    lay_out_unit(row, a.counts + 4 * h, ahead[0] + ahead[1], u);
    u.q_row = u.work_begin = u.work_count = 0;      // (the packer's launches do not look at them)
    if (tid == 0) a.units[h] = u;
  } else {
    u = a.units[h];
  }
  const int n_slots = 4 * (u.d8 + 2 * u.d4 + 4 * u.d2);
  // rank of channel c inside its width class = channels below it of the same class: a ballot per
  // class in each of the two wavefronts that hold the 128 channels, plus the first wavefront's count
  int b = load_bits(a.k_bits, a.kb_elem_size, (int64_t)h * a.kb_stride_h + tid);
  b = b > 8 ? 8 : b;                                             // 16 is stored as 8 bit
  const int cls = b == 2 ? 0 : (b == 4 ? 1 : (b == 8 ? 2 : -1));
  int rank = 0;
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    const unsigned long long m = __ballot(cls == x);
    if (cls == x) rank = __popcll(m & ((1ull << lane) - 1ull));
    if (tid == 0) first_wave_count[x] = __popcll(m);
  }
  slot_of_ch[tid] = -1;
  __syncthreads();
  if (cls >= 0) ch_of[cls * kD + rank + (tid >= 64 ? first_wave_count[cls] : 0)] = tid;
  __syncthreads();
  const int tv = u.n_tok[0] + u.n_tok[1] + u.n_tok[2];
  const bool has_pad = tv < a.max_tv || u.n_tok[3] < a.max_n16;   // zero rows of the canvas join the min / max
  const int16_t *slots = a.src_slot + (int64_t)h * a.n_slots_max;
  float smax = 0.0f;
  for (int i = tid; i < n_slots; i += 128) {
    const int r = planned ? row.source(i, a.n2p, a.n4p) : slots[i];
    uint32_t w0 = 0, w1 = 0;
    if (r >= 0) {
      int c, rk;
      if (r < a.n2p) { c = 0; rk = r; }
      else if (r < a.n2p + a.n4p) { c = 1; rk = r - a.n2p; }
      else { c = 2; rk = r - a.n2p - a.n4p; }
      const int ch = ch_of[c * kD + rk];
      const float qmax = c == 0 ? 3.0f : (c == 1 ? 15.0f : 255.0f);
      float mn = rdkv_ordered_to_float(a.mm[(int64_t)h * 2 * kD + ch]);
      float mx = rdkv_ordered_to_float(a.mm[(int64_t)h * 2 * kD + kD + ch]);
      if (has_pad) {
        mn = fminf(mn, 0.0f);
        mx = fmaxf(mx, 0.0f);
      }
      const RdkvQParams q = rdkv_qparams(mn, mx, qmax);
      slot_p[i] = make_chan(q.scale, q.zp, q.inv, i | (c << 8));
      slot_of_ch[ch] = i;
      const uint16_t sc = rdkv_f2h(q.scale);
      w0 = (uint32_t)ch | ((uint32_t)sc << 16);
      w1 = (uint32_t)rdkv_f2h(q.zp);
      smax = fmaxf(smax, rdkv_h2f(sc));
    }
    uint32_t *qt = reinterpret_cast<uint32_t *>(a.blob + u.qtab_off + 8 * (int64_t)i);   // {channel, scale, zp, 0}
    qt[0] = w0;
    qt[1] = w1;
  }
  // the bytes behind the slot table: up to the next 256-byte boundary, or to the end of the blob
  {
    const int64_t from = (int64_t)u.qtab_off + 8 * (int64_t)n_slots;
    const int64_t to = h == a.H_kv - 1 ? a.blob_bytes : (from + 255) / 256 * 256;
    uint32_t *z = reinterpret_cast<uint32_t *>(a.blob + from);
    for (int64_t i = tid; i < (to - from) / 4; i += 128) z[i] = 0u;
  }
  for (int o = 1; o < 64; o <<= 1) smax = fmaxf(smax, __shfl_xor(smax, o, 64));
  if (lane == 0) wave_max[tid >> 6] = smax;
  __syncthreads();
  // the accumulators go back to their start values: the next call finds them ready
  a.mm[(int64_t)h * 2 * kD + tid] = rdkv_float_to_ordered(INFINITY);
  a.mm[(int64_t)h * 2 * kD + kD + tid] = rdkv_float_to_ordered(-INFINITY);
  const int s = slot_of_ch[tid];
  chan_params[(int64_t)h * kD + tid] = s >= 0 ? slot_p[s] : make_chan(0.f, 0.f, 0.f, -1);
  if (tid == 0) {
    // largest K scale (as the fp16 value the decode kernel reads); the tile workgroups raise the V one
    a.scale_max[h] = __float_as_uint(fmaxf(wave_max[0], wave_max[1]));
    a.scale_max[a.H_kv + h] = 0u;
  }
}

// min and max over the sixteen lanes of a row (lane ^ 1, lane ^ 2, mirror of eight, mirror of sixteen)
__device__ __forceinline__ float row16_min(float v) {
  v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false)));
  v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false)));
  v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, false)));
  v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, false)));
  return v;
}
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, false)));
  return v;
}

__device__ __forceinline__ float half_at(const uint4 &v, int e) {      // element e of eight fp16 values
  const uint32_t w = e < 2 ? v.x : (e < 4 ? v.y : (e < 6 ? v.z : v.w));
  return __half2float(__ushort_as_half((uint16_t)((e & 1) ? (w >> 16) : (w & 0xffffu))));
}

// The code estimate of x (rdkv_qcode's x * (1 / scale) + zp, clamped, rounded to the nearest even
// integer by the byte conversion) placed in byte B of `old`, and whether the estimate lies so close
// to a rounding boundary that the exact quotient has to decide.  For estimates inside the clamp's
// range the distance to the boundary is |fract(t) - 1/2|, the same number rdkv_qcode tests; outside
// it the test can only raise the flag needlessly.  Callers collect the flags of several codes and
// branch once (a branch per code cost more than the arithmetic).
template <int B>
__device__ __forceinline__ uint32_t code_byte(float x, const RdkvQParams &q, float qmax, uint32_t old, bool &near) {
  const float t = fmaf(x, q.inv, q.zp);
  near |= fabsf(__builtin_amdgcn_fractf(t) - 0.5f) < 2e-4f;
  return __builtin_amdgcn_cvt_pk_u8_f32(fminf(fmaxf(t, 0.0f), qmax), B, old);
}
__device__ __forceinline__ bool code_is_near(float x, const RdkvQParams &q) {
  return fabsf(__builtin_amdgcn_fractf(fmaf(x, q.inv, q.zp)) - 0.5f) < 2e-4f;
}

// lane N of every row of sixteen lanes to all lanes of the row
template <int N>
__device__ __forceinline__ float row16_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xF, 0xF, false));
}

// The V tile of class CLS from the code bytes of a wavefront's sixteen tokens, the first nv of which are there (fp16 bits
// for the fp16-kept class): lane l assembles the dwords that hold channels l and l + 64 of its quads 4g .. 4g + 3
// (stream_format.h: element k of an operand is token 4 * quad + k; 8-bit dword 2 * quad + j, 4-bit
// dword quad with operand j, 2-bit dword quad >> 1 with operand 2 * (quad & 1) + j; j = channel half).
template <int CLS>
__device__ __forceinline__ void v_tile(const uint8_t (*cv)[kD], const uint16_t (*raw)[kD], int nv, int g, uint32_t *v_out) {
  const int l = threadIdx.x & 63;
  // dword di of lane l sits at v_out[((di >> 2) * 64 + l) * 4 + (di & 3)]: a lane's dwords 4n .. 4n + 3 are 16 contiguous bytes
  uint4 *out4 = reinterpret_cast<uint4 *>(v_out);
  if (CLS == 3) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int quad = 4 * g + q;
      uint32_t w[4] = {0u, 0u, 0u, 0u};             // dwords 4 * quad + 2 * j + {0, 1}
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int t = 4 * q + k;
          const uint32_t bits = t < nv ? (uint32_t)raw[t][l + 64 * j] : 0u;
          w[2 * j + (k >> 1)] |= bits << (16 * (k & 1));
        }
      out4[quad * 64 + l] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    return;
  }
  constexpr int NF = CLS == 2 ? 4 : (CLS == 1 ? 8 : 16);
  constexpr int FW = 32 / NF;
  uint32_t w8[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};   // class 2: dwords 8g .. 8g + 7; class 1: 4g .. 4g + 3; class 0: 2g, 2g + 1
#pragma unroll
  for (int q = 0; q < 4; ++q) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int t = 4 * q + k;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint32_t c = t < nv ? (uint32_t)cv[t][l + 64 * j] : 0u;
        if (CLS == 2) w8[2 * q + j] |= c << (FW * rdkv_field_of(0, k, NF));
        else if (CLS == 1) w8[q] |= c << (FW * rdkv_field_of(j, k, NF));
        else w8[q >> 1] |= c << (FW * rdkv_field_of(2 * (q & 1) + j, k, NF));
      }
    }
  }
  if (CLS == 2) {
    out4[(2 * g) * 64 + l] = make_uint4(w8[0], w8[1], w8[2], w8[3]);
    out4[(2 * g + 1) * 64 + l] = make_uint4(w8[4], w8[5], w8[6], w8[7]);
  } else if (CLS == 1) {
    out4[g * 64 + l] = make_uint4(w8[0], w8[1], w8[2], w8[3]);
  } else {
    *reinterpret_cast<uint2 *>(v_out + ((g >> 1) * 64 + l) * 4 + 2 * (g & 1)) = make_uint2(w8[0], w8[1]);
  }
}

// one K dword of NF fields from the tile's code bytes: field f is element k of operand s
// (stream_format.h), whose slot is 4 * (step0 + s) + k
template <int NF>
__device__ __forceinline__ uint32_t k_dword(const uint8_t *codes_t, int step0) {
  uint32_t w = 0;
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    int s, k;
    rdkv_operand_of(f, NF, &s, &k);
    w |= (uint32_t)codes_t[4 * (step0 + s) + k] << ((32 / NF) * f);
  }
  return w;
}

// Where tile ti of a unit lies: its class, index inside the class, valid tokens and first row in the
// head's sorted token order (quantized classes, then the fp16 zone).  Selects, no indexed arrays.
struct TileInfo {
  int cls, tl, nv;
  int64_t row0;
};
__device__ __forceinline__ TileInfo tile_info(const RdkvUnit &u, int ti) {
  const int t0 = (u.n_tok[0] + RDKV_TILE - 1) / RDKV_TILE, t1 = t0 + (u.n_tok[1] + RDKV_TILE - 1) / RDKV_TILE;
  const int t2 = t1 + (u.n_tok[2] + RDKV_TILE - 1) / RDKV_TILE;
  TileInfo r;
  r.cls = ti < t0 ? 0 : (ti < t1 ? 1 : (ti < t2 ? 2 : 3));
  r.tl = ti - (r.cls == 0 ? 0 : (r.cls == 1 ? t0 : (r.cls == 2 ? t1 : t2)));
  const int n = r.cls == 0 ? u.n_tok[0] : (r.cls == 1 ? u.n_tok[1] : (r.cls == 2 ? u.n_tok[2] : u.n_tok[3]));
  const int64_t c0 = r.cls == 0 ? 0
                                : (r.cls == 1 ? (int64_t)u.n_tok[0]
                                              : (r.cls == 2 ? (int64_t)u.n_tok[0] + u.n_tok[1]
                                                            : (int64_t)u.n_tok[0] + u.n_tok[1] + u.n_tok[2]));
  r.nv = min(RDKV_TILE, n - r.tl * RDKV_TILE);
  r.row0 = c0 + (int64_t)r.tl * RDKV_TILE;
  return r;
}

// Workgroup (x, head) takes the head's 64-token tiles x, x + gridDim.x, ..., a quarter of a tile to each of its four
// wavefronts, which share nothing but the channel table: every quad of tokens and every K row lies within a quarter.
// Lane (p = lane % 16, r = lane / 16) loads 16 bytes (eight channels, 8p .. 8p + 7) of the K and the V row of tokens r,
// r + 4, r + 8, r + 12 of the quarter and turns them into codes in registers: the V parameters of a token come from a
// min / max over the sixteen lanes that hold it.  Codes are parked in LDS as bytes (K at its stream slot, V at its
// channel), from where the dwords of the K rows and of the V tile are assembled and stored coalesced.
// Latency bound (half of a wavefront's cycles were waits, 46 % of the vector issue slots used): the rows of the next tile
// are requested as soon as the codes are parked, into the registers that held this tile's, and come in under the
// assembly; nothing makes a wavefront wait for another.  One layer of 8 x 32k / 128k tokens 54.8 / 170 -> 51.2 / 155 us.
__global__ void __launch_bounds__(256, 3)
stream_pack_kernel(StreamPackBatch batch) {
  int layer = blockIdx.z, h = blockIdx.y, ti = blockIdx.x, stride = gridDim.x;
  const int tid = threadIdx.x, lane = tid & 63;
  if (batch.by_table) {
    const int row = __popcll(__ballot(batch.begin[lane] <= ti)) - 1;      // (a head without tiles begins where the next does)
    stride = batch.begin[row + 1] - batch.begin[row];
    ti -= batch.begin[row];
    layer = row / batch.layer[0].H_kv;
    h = row - layer * batch.layer[0].H_kv;
  }
  const StreamPackArgs a = batch.layer[layer];
  const float4 *chan_params = chan_params_of(a);
  constexpr int kRows = RDKV_TILE / 4;                                          // tokens of a wavefront
  __shared__ __align__(16) uint8_t ck_all[4][kRows][kMaxSlots];                 // K code of (token, stream slot)
  __shared__ __align__(16) uint8_t cv_all[4][kRows * kD * 2];                   // V code of (token, channel); fp16 bits for class 3
  __shared__ float4 chan[kD];                                                   // the head's channel quantizers
  const int g = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint8_t (*ck)[kMaxSlots] = ck_all[g];
  uint8_t (*cv)[kD] = reinterpret_cast<uint8_t (*)[kD]>(cv_all[g]);
  uint16_t (*raw)[kD] = reinterpret_cast<uint16_t (*)[kD]>(cv_all[g]);
  const RdkvUnit u = a.units[h];
  const int R = u.d8 + u.d4 + u.d2;
  const int n_tiles = (u.n_tok[0] + RDKV_TILE - 1) / RDKV_TILE + (u.n_tok[1] + RDKV_TILE - 1) / RDKV_TILE +
                      (u.n_tok[2] + RDKV_TILE - 1) / RDKV_TILE + (u.n_tok[3] + RDKV_TILE - 1) / RDKV_TILE;
  if (ti >= n_tiles) return;
  const int p = lane & 15, r = lane >> 4;
  const int32_t *ord = a.order + (int64_t)h * a.order_stride_h;
  const __half *Kh = a.K + (int64_t)h * a.stride_h, *Vh = a.V + (int64_t)h * a.stride_h;

  // token indices of a tile (tokens past the tile's end repeat its first row; their codes are
  // dropped at assembly) and the rows behind them
  int32_t tok[4];
  auto load_tok = [&](int tile) {
    const TileInfo t = tile_info(u, tile);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = kRows * g + r + 4 * i;
      tok[i] = ord[t.row0 + (at < t.nv ? at : 0)];
    }
  };
  uint4 kraw[4], vraw[4];
  auto load_rows = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      kraw[i] = *(reinterpret_cast<const uint4 *>(Kh + (int64_t)tok[i] * a.stride_t) + p);
      vraw[i] = *(reinterpret_cast<const uint4 *>(Vh + (int64_t)tok[i] * a.stride_t) + p);
    }
  };

  load_tok(ti);
  if (tid < kD) chan[tid] = chan_params[(int64_t)h * kD + tid];
  load_rows();
  if (ti + stride < n_tiles) load_tok(ti + stride);
  // pad slots hold code 0: nothing writes them afterwards
  {
    uint4 *z = reinterpret_cast<uint4 *>(&ck[0][0]);
    for (int i = lane; i < kRows * kMaxSlots / 16; i += 64) z[i] = make_uint4(0u, 0u, 0u, 0u);
  }
  float v_scale_max = 0.0f;          // largest V scale among the tokens whose parameters this lane worked out
  __syncthreads();                   // the channel table

  for (; ti < n_tiles; ti += stride) {
    const TileInfo t = tile_info(u, ti);
    const int cls = t.cls, nv = t.nv - kRows * g;        // valid tokens from this quarter's first on (may be none)

    // ---- V: per-token parameters and codes (quantized classes), or the rows as they are
    if (cls < 3) {
      const float qmax = cls == 0 ? 3.0f : (cls == 1 ? 15.0f : 255.0f);
      float mn[4], mx[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float lo = half_at(vraw[i], 0), hi = lo;
#pragma unroll
        for (int e = 1; e < 8; ++e) {
          lo = fminf(lo, half_at(vraw[i], e));
          hi = fmaxf(hi, half_at(vraw[i], e));
        }
        mn[i] = row16_min(lo);
        mx[i] = row16_max(hi);
      }
      // lane p works out the parameters of token r + 4 * (p % 4) (three divisions), the row shares them
      const int mine = p & 3;
      const RdkvQParams qm = rdkv_qparams(mine == 0 ? mn[0] : (mine == 1 ? mn[1] : (mine == 2 ? mn[2] : mn[3])),
                                          mine == 0 ? mx[0] : (mine == 1 ? mx[1] : (mine == 2 ? mx[2] : mx[3])), qmax);
      if (p < 4) {
        const int tt = r + 4 * p;
        const uint16_t sc = rdkv_f2h(qm.scale);
        *reinterpret_cast<uint32_t *>(a.blob + u.sz_off + 4 * ((int64_t)ti * RDKV_TILE + kRows * g + tt)) =
            tt < nv ? (uint32_t)sc | ((uint32_t)rdkv_f2h(qm.zp) << 16) : 0u;
        if (tt < nv) v_scale_max = fmaxf(v_scale_max, rdkv_h2f(sc));
      }
      RdkvQParams qt[4];
      qt[0].scale = row16_bcast<0>(qm.scale); qt[0].zp = row16_bcast<0>(qm.zp); qt[0].inv = row16_bcast<0>(qm.inv);
      qt[1].scale = row16_bcast<1>(qm.scale); qt[1].zp = row16_bcast<1>(qm.zp); qt[1].inv = row16_bcast<1>(qm.inv);
      qt[2].scale = row16_bcast<2>(qm.scale); qt[2].zp = row16_bcast<2>(qm.zp); qt[2].inv = row16_bcast<2>(qm.inv);
      qt[3].scale = row16_bcast<3>(qm.scale); qt[3].zp = row16_bcast<3>(qm.zp); qt[3].inv = row16_bcast<3>(qm.inv);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const RdkvQParams q = qt[i];
        bool near = false;
        uint32_t w0 = 0, w1 = 0;
        w0 = code_byte<0>(half_at(vraw[i], 0), q, qmax, w0, near);
        w0 = code_byte<1>(half_at(vraw[i], 1), q, qmax, w0, near);
        w0 = code_byte<2>(half_at(vraw[i], 2), q, qmax, w0, near);
        w0 = code_byte<3>(half_at(vraw[i], 3), q, qmax, w0, near);
        w1 = code_byte<0>(half_at(vraw[i], 4), q, qmax, w1, near);
        w1 = code_byte<1>(half_at(vraw[i], 5), q, qmax, w1, near);
        w1 = code_byte<2>(half_at(vraw[i], 6), q, qmax, w1, near);
        w1 = code_byte<3>(half_at(vraw[i], 7), q, qmax, w1, near);
        if (near) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float x = half_at(vraw[i], e);
            if (code_is_near(x, q)) {
              const uint32_t c = rdkv_qcode_exact(x, q, qmax);
              uint32_t &w = e < 4 ? w0 : w1;
              w = (w & ~(0xffu << (8 * (e & 3)))) | (c << (8 * (e & 3)));
            }
          }
        }
        *reinterpret_cast<uint2 *>(&cv[r + 4 * i][8 * p]) = make_uint2(w0, w1);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<uint4 *>(&raw[r + 4 * i][8 * p]) = vraw[i];
    }

    // ---- K codes to their stream slots
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float4 cp = chan[8 * p + e];
      const int slot_cls = __float_as_int(cp.w);
      if (slot_cls >= 0) {
        const int slot = slot_cls & 0xff, c = slot_cls >> 8;
        const float qmax = c == 0 ? 3.0f : (c == 1 ? 15.0f : 255.0f);
        RdkvQParams q;
        q.scale = cp.x; q.zp = cp.y; q.inv = cp.z;
        bool near = false;
        uint32_t c4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) c4[i] = code_byte<0>(half_at(kraw[i], e), q, qmax, 0u, near);
        if (near) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float x = half_at(kraw[i], e);
            if (code_is_near(x, q)) c4[i] = rdkv_qcode_exact(x, q, qmax);
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) ck[r + 4 * i][slot] = (uint8_t)c4[i];
      }
    }
    // the rows of the next tile come in under the assembly
    if (ti + stride < n_tiles) {
      load_rows();
      if (ti + 2 * stride < n_tiles) load_tok(ti + 2 * stride);
    }
    rdkv_wave_order();

    // ---- K tile: rows of R dwords, chunks of up to four dwords per token, the quarter's sixteen tokens of each
    uint32_t *k_out = reinterpret_cast<uint32_t *>(a.blob + u.k_off) + (int64_t)ti * RDKV_TILE * R;
    auto k_row_dword = [&](int tt, int j) -> uint32_t {
      if (tt >= nv) return 0u;
      if (j < u.d8) return k_dword<4>(ck[tt], j);
      if (j < u.d8 + u.d4) return k_dword<8>(ck[tt], u.d8 + 2 * (j - u.d8));
      return k_dword<16>(ck[tt], u.d8 + 2 * u.d4 + 4 * (j - u.d8 - u.d4));
    };
    for (int c = 0; c < R / 4; ++c) k_out[256 * c + 64 * g + lane] = k_row_dword(lane >> 2, 4 * c + (lane & 3));
    const int wc = R & 3;
    if (lane < kRows * wc) {
      const int tt = wc == 1 ? lane : (wc == 2 ? lane >> 1 : lane / 3);
      k_out[256 * (R / 4) + kRows * wc * g + lane] = k_row_dword(tt, 4 * (R / 4) + lane - tt * wc);
    }

    // ---- V tile of the class
    const uint64_t v_base = cls == 0 ? u.v_off[0] : (cls == 1 ? u.v_off[1] : (cls == 2 ? u.v_off[2] : u.v_off[3]));
    uint32_t *v_out = reinterpret_cast<uint32_t *>(a.blob + v_base) + (int64_t)t.tl * (rdkv_v_tile_bytes(cls) / 4);
    if (cls == 0) v_tile<0>(cv, raw, nv, g, v_out);
    else if (cls == 1) v_tile<1>(cv, raw, nv, g, v_out);
    else if (cls == 2) v_tile<2>(cv, raw, nv, g, v_out);
    else v_tile<3>(cv, raw, nv, g, v_out);
    rdkv_wave_order();
  }

  // the head's largest V scale (as the fp16 value the decode kernel will read): one atomic per
  // workgroup at most, none once the stored maximum has reached it (thousands of same-address
  // atomics would otherwise queue up behind each other)
  for (int o = 1; o < 64; o <<= 1) v_scale_max = fmaxf(v_scale_max, __shfl_xor(v_scale_max, o, 64));
  __shared__ float wave_max[4];
  if ((tid & 63) == 0) wave_max[tid >> 6] = v_scale_max;
  __syncthreads();
  if (tid == 0) {
    const float m = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
    uint32_t *dst = &a.scale_max[a.H_kv + h];
    const uint32_t mine = __float_as_uint(m);
    if (mine > __hip_atomic_load(dst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(dst, mine);
  }
}

// The smallest e >= 0 with v * 2^(6 - e) < 2^15, at most 40 and, for what is beyond 2^40, 32; 0 for a NaN.
__device__ __forceinline__ int v_shift_of(float v) {
  if (!(v > 0.0f)) return 0;
  const int ex = (int)((__float_as_uint(v) >> 23) & 255u) - 126;      // v = m * 2^ex, 0.5 <= m < 1 (subnormals: -126)
  return min(max(min(ex, 41) - 9, 0), 40);
}

// A cache's tables from the host memory they were written to (`src`, which the device reads itself) to where they stay,
// the work items among them (from byte `work_at` on) with the scales that launches before this one have left on the
// device, as rdkv_stream_work_scales fills them, and the scales to the host.  A copy queued behind the packer began
// 15 us after its end and this launch behind the copy; with a copy back, a wait for it and the upload behind it, a
// build's last 70 us were the host's alone.
__global__ void __launch_bounds__(256)
stream_tables_kernel(const uint4 *src, uint4 *dst, int pieces, int work_at, int n_work, const float *__restrict__ scales, int H_kv,
                     int n_units, uint64_t *words, uint32_t tag) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  auto scale = [&](int u, int which) { return scales[(int64_t)(u / H_kv) * 2 * H_kv + which * H_kv + u % H_kv]; };
  uint4 v = i < pieces ? src[i] : make_uint4(0u, 0u, 0u, 0u);
  // (an item is eight pieces, its unit the first word of the first, the scale fields the last words of the last)
  static_assert(sizeof(RdkvWork) == 128 && offsetof(RdkvWork, unit) == 0 && offsetof(RdkvWork, k_scale_max) == 120 &&
                    offsetof(RdkvWork, v_shift) == 124, "an item's layout");
  const int unit = __shfl((int)v.x, (threadIdx.x & 63) & ~7);
  const int at = i - work_at;
  if (at >= 0 && at < 8 * n_work && (at & 7) == 7) {
    v.z = __float_as_uint(scale(unit, 0));
    v.w = (uint32_t)v_shift_of(scale(unit, 1));
  }
  if (i < pieces) dst[i] = v;
  if (i < 2 * n_units) rdkv_host_word(words, i, tag, __float_as_int(scale(i >> 1, i & 1)));
}

}  // namespace

RDKV_API int rdkv_stream_tables_device(const void *src, void *dst, int64_t bytes, int64_t work_at, int n_work, const float *scales,
                                       int H_kv, int n_units, uint64_t *host_words, uint32_t tag, void *stream) {
  const char *fn = "rdkv_stream_tables_device";
  RDKV_REQUIRE(bytes >= 0 && bytes % 16 == 0 && bytes < (1LL << 34) && (bytes == 0 || (src && dst)) &&
                   (((uintptr_t)src | (uintptr_t)dst) % 16) == 0, "%s: bad tables", fn);
  // (whole items in whole groups of eight lanes)
  RDKV_REQUIRE(n_work >= 0 && work_at >= 0 && work_at % 128 == 0 && work_at + n_work * (int64_t)sizeof(RdkvWork) <= bytes,
               "%s: work items outside the tables", fn);
  RDKV_REQUIRE(n_units >= 1 && n_units <= (1 << 28) && H_kv >= 1 && n_units % H_kv == 0 && scales && host_words,
               "%s: bad arguments", fn);
  const int64_t n = std::max<int64_t>(bytes / 16, 2 * (int64_t)n_units);
  hipLaunchKernelGGL(stream_tables_kernel, dim3((unsigned)rdkv_cdiv(n, 256)), dim3(256), 0, (hipStream_t)stream, (const uint4 *)src,
                     (uint4 *)dst, (int)(bytes / 16), (int)(work_at / 16), n_work, scales, H_kv, n_units, host_words, tag);
  RDKV_CHECK_LAUNCH(fn);
  return RDKV_OK;
}

RDKV_API int rdkv_pack_layer_stream_ws_init(float *minmax_ws, int H_kv, void *stream) {
  const char *fn = "rdkv_pack_layer_stream_ws_init";
  RDKV_REQUIRE(minmax_ws && H_kv >= 1 && H_kv <= 65535, "%s: bad arguments", fn);
  rdkv_layer_k_minmax_init(minmax_ws, H_kv, kD, (hipStream_t)stream);
  RDKV_CHECK_LAUNCH(fn);
  return RDKV_OK;
}

// As many workgroups as the device holds at once.  With the tiles of every head, the most that any workgroup has is as
// small as that number allows: the heads of a layer keep between half and all of their tokens, and with the longest head's
// share given to every head the launch ran its last quarter on a part of its wavefronts (four layers of 8 x 32k, Dirichlet
// shares, 153 -> 132 us; equal heads the same).  One and a third times as many workgroups 160, twice 139, four times 138.
static int launch_stream_pack(StreamPackBatch &batch, const int32_t *const *head_tiles, int n_layers, int H_kv, hipStream_t s) {
  hipLaunchKernelGGL(slot_params_kernel, dim3(H_kv, 1, n_layers), dim3(128), 0, s, batch);
  int max_tiles = 0;
  for (int l = 0; l < n_layers; ++l) max_tiles = std::max(max_tiles, batch.layer[l].max_tiles);
  if (max_tiles == 0) return RDKV_OK;
  static int resident_of_device[64];     // (0 = not asked yet; a race between first callers writes the same value)
  int resident = 512, dev = 0;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64) {
    if (resident_of_device[dev] == 0) {
      int cus = 0, per_cu = 0;
      const bool ok = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0 &&
                      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, stream_pack_kernel, 256, 0) == hipSuccess &&
                      per_cu > 0;
      if (ok) resident_of_device[dev] = cus * per_cu;   // (otherwise asked again next time)
    }
    if (resident_of_device[dev] > 0) resident = resident_of_device[dev];
  }
  batch.by_table = head_tiles != nullptr && (int64_t)H_kv * n_layers <= std::min(kTableHeads, resident);
  for (int l = 0; l < n_layers && batch.by_table; ++l) batch.by_table = head_tiles[l] != nullptr;
  if (batch.by_table) {
    const int heads = H_kv * n_layers;
    auto tiles = [&](int r) { return (int64_t)head_tiles[r / H_kv][r % H_kv]; };
    int64_t all = 0, n = 0;
    for (int r = 0; r < heads; ++r) all += tiles(r);
    if (all == 0) return RDKV_OK;
    for (int64_t per = (all + resident - 1) / resident;; ++per) {
      n = 0;
      for (int r = 0; r < heads; ++r) {
        batch.begin[r] = (int32_t)n;
        n += (tiles(r) + per - 1) / per;
      }
      if (n <= resident) break;        // (at the latest with a workgroup a head)
    }
    for (int r = heads; r <= kTableHeads; ++r) batch.begin[r] = (int32_t)n;
    hipLaunchKernelGGL(stream_pack_kernel, dim3((unsigned)n), dim3(256), 0, s, batch);
    return RDKV_OK;
  }
  const int rows = H_kv * n_layers, target = std::max(1, (resident + rows - 1) / rows);
  const int per = (max_tiles + target - 1) / target;
  const int gx = (max_tiles + per - 1) / per;
  hipLaunchKernelGGL(stream_pack_kernel, dim3(gx, H_kv, n_layers), dim3(256), 0, s, batch);
  return RDKV_OK;
}

static int fill_stream_args(const char *fn, StreamPackArgs *a, const void *K_f16, const void *V_f16, int64_t stride_h,
                            int64_t stride_t, int H_kv, const int32_t *order, int64_t order_stride_h, const int32_t *counts,
                            const void *k_bits, int kb_elem_size, int64_t kb_stride_h, int n2p, int n4p, int n8,
                            int64_t max_tv, int max_n16, RdkvUnit *units, const int32_t *info, const int16_t *src_slot,
                            int n_slots_max, int max_tiles, uint8_t *blob, int64_t blob_bytes, float *minmax_ws,
                            float *scale_max) {
  // (minmax_ws holds the min / max accumulators, H_kv * 256 floats, then the channel parameters,
  // H_kv * 128 * 4 floats)
  RDKV_REQUIRE(H_kv >= 1 && H_kv <= 65535 && max_tiles >= 0 && max_tv >= 0 && max_n16 >= 0 && blob_bytes >= 0 &&
                   blob_bytes % 4 == 0,
               "%s: bad shape", fn);
  RDKV_REQUIRE(K_f16 && V_f16 && order && counts && k_bits && units && (src_slot || info) && blob && minmax_ws && scale_max,
               "%s: null pointer", fn);
  RDKV_REQUIRE(kb_elem_size == 1 || kb_elem_size == 2 || kb_elem_size == 4 || kb_elem_size == 8,
               "%s: element size of k_bits must be 1, 2, 4 or 8", fn);
  RDKV_REQUIRE(n2p >= 0 && n4p >= 0 && n8 >= 0 && n2p % 4 == 0 && n4p % 2 == 0 && n2p + n4p + n8 <= 3 * kD,
               "%s: bad padded channel counts (%d,%d,%d)", fn, n2p, n4p, n8);
  RDKV_REQUIRE(n_slots_max >= 1 && n_slots_max <= kMaxSlots, "%s: n_slots_max=%d outside 1..%d", fn, n_slots_max,
               kMaxSlots);
  if (stride_t % 8 != 0 || stride_h % 8 != 0 || ((uintptr_t)K_f16 % 16) != 0 || ((uintptr_t)V_f16 % 16) != 0) {
    rdkv_set_error("%s: K and V rows must be 16-byte aligned", fn);
    return RDKV_EUNSUPPORTED;
  }
  a->K = (const __half *)K_f16; a->V = (const __half *)V_f16;
  a->stride_h = stride_h; a->stride_t = stride_t;
  a->order = order; a->order_stride_h = order_stride_h;
  a->k_bits = k_bits; a->kb_elem_size = kb_elem_size; a->kb_stride_h = kb_stride_h;
  a->n2p = n2p; a->n4p = n4p;
  a->max_tv = max_tv; a->max_n16 = max_n16;
  a->mm = reinterpret_cast<uint32_t *>(minmax_ws);
  a->units = units; a->counts = counts; a->info = info; a->src_slot = src_slot; a->n_slots_max = n_slots_max; a->max_tiles = max_tiles;
  a->blob = blob;
  a->scale_max = reinterpret_cast<uint32_t *>(scale_max);
  a->H_kv = H_kv;
  a->blob_bytes = blob_bytes;
  return RDKV_OK;
}

RDKV_API int rdkv_pack_layer_stream(const void *K_f16, const void *V_f16, int64_t stride_h, int64_t stride_t,
                                    int H_kv, const int32_t *order, int64_t order_stride_h,
                                    const int32_t *counts, const void *k_bits, int kb_elem_size,
                                    int64_t kb_stride_h, int n2p, int n4p, int n8, int64_t max_tv, int max_n16,
                                    const RdkvUnit *units, const int16_t *src_slot, int n_slots_max,
                                    int max_tiles, uint8_t *blob, int64_t blob_bytes, float *minmax_ws,
                                    int minmax_ws_ready, float *scale_max, void *stream) {
  const char *fn = "rdkv_pack_layer_stream";
  StreamPackBatch batch;
  const int rc = fill_stream_args(fn, &batch.layer[0], K_f16, V_f16, stride_h, stride_t, H_kv, order, order_stride_h, counts,
                                  k_bits, kb_elem_size, kb_stride_h, n2p, n4p, n8, max_tv, max_n16,
                                  const_cast<RdkvUnit *>(units), nullptr, src_slot, n_slots_max, max_tiles, blob, blob_bytes, minmax_ws, scale_max);
  if (rc != RDKV_OK) return rc;
  hipStream_t s = (hipStream_t)stream;
  // per-channel min / max of every head's kept rows (the K canvas without its zero rows)
  if (minmax_ws_ready != 2) {
    const int mrc = rdkv_layer_k_minmax(fn, K_f16, stride_h, stride_t, H_kv, kD, order, order_stride_h, counts, max_tv + max_n16,
                                        minmax_ws, /*init=*/minmax_ws_ready == 0, s);
    if (mrc != RDKV_OK) return mrc;
  }
  launch_stream_pack(batch, nullptr, 1, H_kv, s);
  RDKV_CHECK_LAUNCH(fn);
  return RDKV_OK;
}

// Layers packed one by one leave the device between them what a launch's first and last tiles take, and the slot
// parameters 4.5 us each: four layers of 8 x 32k tokens 223 us of launches, together 164.
RDKV_API int rdkv_pack_layers_stream(const RdkvStreamLayer *layers, int n_layers, int H_kv, const int32_t *order,
                                     int64_t order_stride_h, const int32_t *counts, const int32_t *info, const void *k_bits,
                                     int kb_elem_size, int64_t kb_stride_h, RdkvUnit *units, float *minmax_ws, float *scale_max, void *stream) {
  const char *fn = "rdkv_pack_layers_stream";
  RDKV_REQUIRE(n_layers >= 0 && (n_layers == 0 || layers), "%s: bad arguments", fn);
  for (int pass = 0; pass < 2; ++pass) {          // (every layer's arguments are looked at before the first launch)
    for (int first = 0; first < n_layers; first += kBatchLayers) {
      const int n = std::min(kBatchLayers, n_layers - first);
      StreamPackBatch batch;
      const int32_t *head_tiles[kBatchLayers];
      for (int i = 0; i < n; ++i) {
        const int64_t l = first + i, row = l * H_kv;
        const RdkvStreamLayer &y = layers[l];
        head_tiles[i] = y.head_tiles;
        for (int h = 0; y.head_tiles && h < H_kv; ++h)
          RDKV_REQUIRE(y.head_tiles[h] >= 0 && y.head_tiles[h] <= y.max_tiles, "%s: head_tiles outside 0..max_tiles", fn);
        const int rc = fill_stream_args(fn, &batch.layer[i], y.K_f16, y.V_f16, y.stride_h, y.stride_t, H_kv,
                                        order ? order + row * order_stride_h : nullptr, order_stride_h,
                                        counts ? counts + 4 * row : nullptr,
                                        k_bits ? (const uint8_t *)k_bits + row * kb_stride_h * kb_elem_size : nullptr, kb_elem_size,
                                        kb_stride_h, y.n2p, y.n4p, y.n8, y.max_tv, y.max_n16, units ? units + row : nullptr,
                                        info ? info + 8 * row : nullptr, nullptr, kMaxSlots, y.max_tiles, y.blob,
                                        y.blob_bytes, minmax_ws ? minmax_ws + row * 768 : nullptr,
                                        scale_max ? scale_max + 2 * row : nullptr);
        if (rc != RDKV_OK) return rc;
      }
      if (pass == 1) launch_stream_pack(batch, head_tiles, n, H_kv, (hipStream_t)stream);
    }
  }
  RDKV_CHECK_LAUNCH(fn);
  return RDKV_OK;
}

// Host side of the streaming format (no GPU work): the unit descriptors of one layer's heads.
RDKV_API int rdkv_stream_plan_layer(const int32_t *tok_counts, int64_t tok_stride, const int32_t *ch_counts,
                                    int64_t ch_stride, int H_kv, int n2p, int n4p, int first_q_row, int G,
                                    RdkvUnit *units, int16_t *src_slot, int n_slots_max, int64_t *sizes) {
  const char *fn = "rdkv_stream_plan_layer";
  RDKV_REQUIRE(tok_counts && ch_counts && units && sizes, "%s: null pointer", fn);
  RDKV_REQUIRE(H_kv >= 1 && G >= 1 && n2p >= 0 && n4p >= 0 && n2p % 4 == 0 && n4p % 2 == 0, "%s: bad shape", fn);
  RDKV_REQUIRE(!src_slot || n_slots_max == kMaxSlots, "%s: n_slots_max must be %d", fn, kMaxSlots);
  int64_t off = 0, stream_bytes = 0, algo_bytes = 0;
  int max_tiles = 0;
  for (int h = 0; h < H_kv; ++h) {
    const int32_t *nt = tok_counts + h * tok_stride, *cc = ch_counts + h * ch_stride;
    const int c2 = cc[0], c4 = cc[1], c8 = cc[2];
    RDKV_REQUIRE(c2 >= 0 && c4 >= 0 && c8 >= 0 && c2 <= n2p && c4 <= n4p && c2 + c4 + c8 <= kD &&
                     nt[0] >= 0 && nt[1] >= 0 && nt[2] >= 0 && nt[3] >= 0,
                 "%s: bad counts of head %d", fn, h);
    const RowPlan row_plan(c2, c4, c8);
    const int n_slots = row_plan.slots(), R = row_plan.d8 + row_plan.d4 + row_plan.d2;
    RDKV_REQUIRE(n_slots <= kMaxSlots, "%s: %d channel steps exceed %d", fn, n_slots / 4, RDKV_MAX_STEPS);
    if (src_slot)
      for (int i = 0; i < n_slots_max; ++i)
        src_slot[(int64_t)h * n_slots_max + i] = i < n_slots ? (int16_t)row_plan.source(i, n2p, n4p) : (int16_t)-1;
    int64_t n_tiles = 0, n_q_tiles = 0, v_bytes = 0;
    for (int c = 0; c < 4; ++c) {
      const int64_t tiles = ((int64_t)nt[c] + RDKV_TILE - 1) / RDKV_TILE;
      n_tiles += tiles;
      if (c < 3) n_q_tiles += tiles;
      v_bytes += tiles * rdkv_v_tile_bytes(c);
    }
    RDKV_REQUIRE(n_tiles <= 0x7fffffff, "%s: too many tiles", fn);
    if (n_tiles > max_tiles) max_tiles = (int)n_tiles;
    RdkvUnit u;
    memset(&u, 0, sizeof(u));
    off = lay_out_unit(row_plan, nt, off, u);
    u.q_row = first_q_row + h * G;
    units[h] = u;
    stream_bytes += n_tiles * RDKV_TILE * 4 * R + v_bytes + n_q_tiles * RDKV_TILE * 4 + (int64_t)n_slots * (int64_t)sizeof(RdkvSlot);
    // the reference's own bytes for the same content: packed K rows and channel parameters, packed
    // V rows, per-token parameters, fp16-kept rows
    const int64_t row = (c2 + 3) / 4 + (c4 + 1) / 2 + c8;
    const int64_t n_all = (int64_t)nt[0] + nt[1] + nt[2] + nt[3];
    algo_bytes += n_all * row + 4 * (4 * ((c2 + 3) / 4) + 2 * ((c4 + 1) / 2) + c8) + 32 * (int64_t)nt[0] +
                  64 * (int64_t)nt[1] + 128 * (int64_t)nt[2] + 4 * ((int64_t)nt[0] + nt[1] + nt[2]) +
                  256 * (int64_t)nt[3];
  }
  sizes[0] = off;
  sizes[1] = max_tiles;
  sizes[2] = stream_bytes;
  sizes[3] = algo_bytes;
  return RDKV_OK;
}

// The unit that merges an output row - the unit itself, or the first source of its row (which then carries
// the row's item count, the others 0) - and its item range and the unit's descriptor in every work item.
static void finish_work(RdkvUnit *units, int U, int multi_source, RdkvWork *work, int nw) {
  std::vector<int32_t> merger((size_t)U);
  if (multi_source) {
    int first = 0;
    for (int u = 0; u < U; ++u) {
      if (u == 0 || units[u].q_row != units[u - 1].q_row) first = u;
      else {
        units[first].work_count += units[u].work_count;
        units[u].work_count = 0;
      }
      merger[u] = first;
    }
  } else {
    for (int u = 0; u < U; ++u) merger[u] = u;
  }
  for (int i = 0; i < nw; ++i) {
    RdkvWork &w = work[i];
    const int m = merger[(size_t)w.unit];
    w.u = units[w.unit];
    w.merge_unit = m;
    w.merge_begin = units[m].work_begin;
    w.merge_count = units[m].work_count;
  }
}

// The other decomposition, for caches of few units: every unit is cut on its own, into runs of equal cost
// (costs as in rdkv_stream_partition, without an item cost), and every run is a work item and a workgroup
// of its own (no group table).  A unit gets as many of the n_items runs as its share of the cost asks for, at
// least one, none more than its tiles or kMaxRuns: the longest run is as short as n_items of them can make it.
// A workgroup that holds the end of one unit and the start of the next works through two items one after the
// other, 4 us more than one of the same number of tiles, and every workgroup waits for the slowest: 8 units of
// 4k / 16k / 32k tokens, a decode step 19.4 / 19.5 / 22.5 us with a boundary inside some workgroups, 15.1 / 16.6 /
// 19.4 without; 256 units of 2k tokens 37.1 / 26.8.
// (The merge takes up to 128 partials of a row in one pass: a row of several sources may have more, each of its units
// up to kMaxRuns; work_count of its first unit says how many, for the caller to decide.)
constexpr int kMaxRuns = 96;
RDKV_API int rdkv_stream_partition_units(RdkvUnit *units, int n_units, int n_items, const double *cost_tile,
                                         double cost_k_dword, int multi_source, RdkvWork *work, int work_capacity,
                                         int *n_work, double *costs) {
  const char *fn = "rdkv_stream_partition_units";
  RDKV_REQUIRE(units && cost_tile && work && n_work && costs && n_units >= 0 && n_items >= 1, "%s: bad arguments", fn);
  RDKV_REQUIRE(work_capacity >= std::max(n_items, n_units), "%s: work table too small", fn);
  const int U = n_units;
  std::vector<double> tile_cost((size_t)U * 4), unit_cost((size_t)U, 0.0);
  std::vector<int64_t> tiles((size_t)U * 4), unit_tiles((size_t)U, 0);
  double all = 0.0;
  for (int u = 0; u < U; ++u) {
    const double k_row = cost_k_dword * (double)((int64_t)units[u].d8 + units[u].d4 + units[u].d2);
    for (int c = 0; c < 4; ++c) {
      RDKV_REQUIRE(units[u].n_tok[c] >= 0, "%s: negative token count", fn);
      tile_cost[4 * u + c] = k_row + cost_tile[c];
      tiles[4 * u + c] = ((int64_t)units[u].n_tok[c] + RDKV_TILE - 1) / RDKV_TILE;
      unit_tiles[u] += tiles[4 * u + c];
      unit_cost[u] += tile_cost[4 * u + c] * (double)tiles[4 * u + c];
    }
    RDKV_REQUIRE(unit_tiles[u] <= 0x7fffffffLL, "%s: too many tiles", fn);
    all += unit_cost[u];
  }
  // the shortest run length that n_items runs can keep to, by bisection above the mean
  auto runs_of = [&](int u, double length) -> int64_t {
    if (unit_tiles[u] == 0 || !(length > 0.0)) return 1;
    const double k = ceil(unit_cost[u] / length), most = (double)std::min<int64_t>(kMaxRuns, unit_tiles[u]);
    return std::max<int64_t>(1, (int64_t)std::min(k, most));
  };
  auto fit = [&](double length) {
    int64_t n = 0;
    for (int u = 0; u < U; ++u) n += runs_of(u, length);
    return n <= n_items;
  };
  double length = all, low = all / n_items;      // (`all` leaves every unit one run)
  if (fit(low)) length = low;
  else
    for (int it = 0; it < 50; ++it) {
      const double mid = 0.5 * (length + low);
      (fit(mid) ? length : low) = mid;
    }
  int nw = 0;
  double longest = 0.0;
  for (int u = 0; u < U; ++u) {
    const int64_t k = runs_of(u, length);
    units[u].work_begin = nw;
    units[u].work_count = (int32_t)k;
    int64_t t = 0, left = tiles[4 * u];      // tiles given out; tiles left of class c
    double acc = 0.0;
    int c = 0;
    for (int64_t i = 0; i < k; ++i) {
      RdkvWork &w = work[nw++];
      memset(&w, 0, sizeof(w));
      w.unit = u;
      w.tile_begin = (int32_t)t;
      // run i goes to the tile boundary nearest (i + 1) / k of the unit's cost, takes one tile at least and
      // leaves one to every later run
      const double from = acc, want = unit_cost[u] * (double)(i + 1) / (double)k;
      const int64_t last = unit_tiles[u] - (k - 1 - i);
      for (bool first = true; t < last; first = false) {
        while (left == 0) left = tiles[4 * u + ++c];
        const double cost = tile_cost[4 * u + c];
        if (!first && i + 1 < k && acc + 0.5 * cost > want) break;
        acc += cost;
        --left;
        ++t;
      }
      w.tile_end = (int32_t)t;
      longest = std::max(longest, acc - from);
    }
  }
  finish_work(units, U, multi_source, work, nw);
  *n_work = nw;
  costs[0] = longest;
  costs[1] = all;
  return RDKV_OK;
}

// Host side of the fused kernel's work decomposition (no GPU work): cut the unit-major, class-minor
// sequence of 64-token tiles into n_groups contiguous runs of equal modelled cost (shares
// proportional to speed[g % n_speed]), one run per workgroup; a run that crosses a unit boundary
// becomes several work items; a unit without tiles gets one empty item.  Every tile costs
// cost_tile[class] + cost_k_dword * (d8 + d4 + d2), the first tile of a unit cost_item more.
// Cumulative costs and shares are summed in order, in double precision.
// units[n_units] (ordered; with multi_source the sources of one output row adjacent): work_begin /
// work_count are written; with multi_source the first unit of a run of equal q_row carries the
// run's item count, the others 0.  work[work_capacity >= n_groups + 2 * n_units]: unit, tile range,
// the unit's descriptor, the merging unit and its item range (k_scale_max / v_shift: see
// rdkv_stream_work_scales).  groups[n_groups + 1]: offsets into work.  Returns the item count in
// *n_work.
RDKV_API int rdkv_stream_partition(RdkvUnit *units, int n_units, int n_groups, const double *cost_tile,
                                   double cost_k_dword, double cost_item, const double *speed, int n_speed,
                                   int multi_source, RdkvWork *work, int work_capacity, int32_t *groups,
                                   int *n_work) {
  const char *fn = "rdkv_stream_partition";
  RDKV_REQUIRE(units && cost_tile && work && groups && n_work && n_units >= 0 && n_groups >= 1, "%s: bad arguments", fn);
  RDKV_REQUIRE(n_speed >= 0 && (n_speed == 0 || speed), "%s: bad speed table", fn);
  RDKV_REQUIRE((int64_t)work_capacity >= (int64_t)n_groups + 2 * (int64_t)n_units, "%s: work table too small", fn);
  const int U = n_units;
  std::vector<int64_t> unit_start((size_t)U + 1, 0);
  for (int u = 0; u < U; ++u) {
    int64_t t = 0;
    for (int c = 0; c < 4; ++c) {
      RDKV_REQUIRE(units[u].n_tok[c] >= 0, "%s: negative token count", fn);
      t += ((int64_t)units[u].n_tok[c] + RDKV_TILE - 1) / RDKV_TILE;
    }
    unit_start[u + 1] = unit_start[u] + t;
  }
  const int64_t total = unit_start[U];
  RDKV_REQUIRE(total <= 0x7fffffffLL, "%s: too many tiles", fn);
  // cumulative cost of every tile
  std::vector<double> cum((size_t)total);
  {
    double acc = 0.0;
    int64_t i = 0;
    for (int u = 0; u < U; ++u) {
      const double R = (double)((int64_t)units[u].d8 + units[u].d4 + units[u].d2);
      bool first = true;
      for (int c = 0; c < 4; ++c) {
        const int64_t nt = ((int64_t)units[u].n_tok[c] + RDKV_TILE - 1) / RDKV_TILE;
        const double seg = cost_k_dword * R + cost_tile[c];
        for (int64_t t = 0; t < nt; ++t) {
          acc += first ? seg + cost_item : seg;
          first = false;
          cum[(size_t)i++] = acc;
        }
      }
    }
  }
  // group boundaries
  std::vector<int64_t> group_cuts((size_t)n_groups + 1, 0);
  group_cuts[n_groups] = total;
  if (total > 0 && n_groups > 1) {
    std::vector<double> share_cum((size_t)n_groups);
    double acc = 0.0;
    for (int g = 0; g < n_groups; ++g) {
      acc += n_speed ? speed[g % n_speed] : 1.0;
      share_cum[g] = acc;
    }
    const double all = cum[(size_t)total - 1];
    for (int g = 0; g + 1 < n_groups; ++g) {
      const double thr = all * (share_cum[g] / share_cum[n_groups - 1]);
      const int64_t idx = std::lower_bound(cum.begin(), cum.end(), thr) - cum.begin();   // first cum >= thr
      group_cuts[g + 1] = std::min(idx + 1, total);
    }
  }
  for (int g = 1; g <= n_groups; ++g) group_cuts[g] = std::max(group_cuts[g], group_cuts[g - 1]);
  // items: walk units and group cuts together
  int nw = 0, g = 0;
  std::vector<int32_t> item_group;
  item_group.reserve((size_t)n_groups + 2 * (size_t)U);
  for (int u = 0; u < U; ++u) {
    const int64_t a = unit_start[u], b = unit_start[u + 1];
    units[u].work_begin = nw;
    if (a == b) {
      // an empty unit: one empty item, in the group of the position it sits at
      while (g + 1 < n_groups && group_cuts[g + 1] <= a) ++g;
      RdkvWork &w = work[nw++];
      memset(&w, 0, sizeof(w));
      w.unit = u;
      item_group.push_back(std::min(g, n_groups - 1));
    } else {
      int64_t s = a;
      while (s < b) {
        while (g + 1 < n_groups && group_cuts[g + 1] <= s) ++g;
        const int64_t next_cut = g + 1 <= n_groups ? group_cuts[g + 1] : total;
        const int64_t e = std::min(b, next_cut > s ? next_cut : b);
        RdkvWork &w = work[nw++];
        memset(&w, 0, sizeof(w));
        w.unit = u;
        w.tile_begin = (int32_t)(s - a);
        w.tile_end = (int32_t)(e - a);
        item_group.push_back(std::min(g, n_groups - 1));
        s = e;
      }
    }
    units[u].work_count = nw - units[u].work_begin;
  }
  // group offsets: first item of every group
  {
    int i = 0;
    for (int gg = 0; gg <= n_groups; ++gg) {
      while (i < nw && item_group[(size_t)i] < gg) ++i;
      groups[gg] = i;
    }
  }
  finish_work(units, U, multi_source, work, nw);
  *n_work = nw;
  return RDKV_OK;
}

// k_scale_max and v_shift of every work item from its unit's largest scales (scale_max[unit][0] = K
// channel scale, [1] = V token scale): v_shift = the smallest e >= 0 with scale * 2^(6 - e) < 2^15,
// at most 40 (0 for a NaN).
RDKV_API int rdkv_stream_work_scales(RdkvWork *work, int n_work, const float *scale_max, int n_units) {
  const char *fn = "rdkv_stream_work_scales";
  RDKV_REQUIRE(n_work >= 0 && (n_work == 0 || (work && scale_max)), "%s: bad arguments", fn);
  for (int i = 0; i < n_work; ++i) {
    const int u = work[i].unit;
    RDKV_REQUIRE(u >= 0 && u < n_units, "%s: item %d names unit %d", fn, i, u);
    work[i].k_scale_max = scale_max[2 * u];
    double v = (double)scale_max[2 * u + 1];
    if (!(v == v)) v = 0.0;
    v = std::min(std::max(v, 0.0), 1099511627776.0);     // 2^40 stands for infinity
    int ex = 0;
    frexp(v, &ex);                                         // v = m * 2^ex, 0.5 <= m < 1
    work[i].v_shift = std::min(std::max(ex - 9, 0), 40);
  }
  return RDKV_OK;
}
