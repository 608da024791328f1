// A packed layer back to dense fp16 K and V: one launch each, every output byte written once.
// The values are the ones rdkv_dequant_f16 gives segment by segment (half((code - zp) * scale),
// obkv_accel/packing.py:581-709, 1427-1444, trizone_decompress.py:91-182); here the channel scatter
// of K, the class walk of V, the zero rows of the stripe and the fp16-kept rows are part of the
// same pass, so nothing is dequantized into a temporary and copied again.
// The per-head counts that the host checks leave the launches as words in host memory when their first workgroup
// starts (rdkv_host_word): two layers of 16k / 31k / 64k tokens 107 / 121 / 261 us a call; with the
// counts joined, copied and the stream waited for 174 / 174 / 313.
#include "rdkv_common.h"

namespace {

constexpr int kChan = 128;        // channels of a workgroup (16 threads x 8), further ones in grid.z
constexpr int kLdsBytes = 48 << 10;
constexpr int kMaxTileRows = 64;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// half((code - zp) * scale).  The product must exist as an fp32 value before it is rounded: merged
// with the conversion it would be a fused multiply-add with +0, and (code - zp) * 0 = -0 would
// come out as +0.
__device__ __forceinline__ uint32_t dequant_bits(uint32_t code, float zp, float scale) {
  float v = __fmul_rn(__fsub_rn((float)code, zp), scale);
  asm volatile("" : "+v"(v));
  return rdkv_f2h(v);
}

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

// Two codes (below 256) in the halves of `codes`, dequantized in packed fp16: 0x6400 | code is the bit
// pattern of 1024 + code, the subtraction of 1024 + zp leaves the exact integer code - zp (zp whole and
// at most 1024 in magnitude), and the fp16 product of two fp16 numbers is the rounding of their exact
// product, which is what the fp32 form rounds too; a zero keeps its sign.
__device__ __forceinline__ bool whole_zp(float zp) { return fabsf(zp) <= 1024.0f && rintf(zp) == zp; }
__device__ __forceinline__ uint32_t dequant_pair(uint32_t codes, uint32_t zp1024, uint32_t scale) {
  half2_t v = __builtin_bit_cast(half2_t, codes | 0x64006400u) - __builtin_bit_cast(half2_t, zp1024);
  return __builtin_bit_cast(uint32_t, v * __builtin_bit_cast(half2_t, scale));
}

// One bit-width segment of the K rows of one head.
struct KSeg {
  const uint8_t *base;      // first row of head 0
  int64_t stride_h, stride_t;
  int sub;                  // bytes of a row
};

// ---------------------------------------------------------------------------
// K.  grid = (workgroups per head, H_kv, channel chunks of 128).  A workgroup walks tiles of
// `rows` tokens: the tile's packed rows are copied to LDS with 16-byte loads (rows stored back to
// back; byte copies otherwise), then sixteen threads share a token, each writing eight
// channels with one 16-byte store.  A thread's channels are the same for every token, so
// where their codes lie in a row, their scales and zero points are worked out once per
// workgroup.  Codes are dequantized as packed fp16 pairs (bit-identical where the zero points are
// whole numbers, which the quantizer's are), two thirds fewer vector instructions than in fp32.
// Bound: the fp16 rows written (256 B a token for ~40 B read).  Nothing reads them soon, so they are
// stored with the nontemporal hint: 19 us instead of 26 for 8 heads of 25 300 rows (52 MB written;
// a plain fill of the same bytes takes 9 us).  What is left above that is the chain tables -> tile
// -> LDS -> rows, twice per workgroup.  The per-head launches of dequantize, concatenate and indexed
// copy that this replaces took 430 us of device time for such a layer, and as much again on the host.
// ---------------------------------------------------------------------------
template <bool DENSE>
__global__ void __launch_bounds__(256)
unpack_k_kernel(KSeg s2, KSeg s4, KSeg s8, const __half *__restrict__ scale, const __half *__restrict__ zp,
                int64_t ks_sh, const int64_t *__restrict__ sort_idx, int64_t sort_sh, int sort_n,
                const int32_t *__restrict__ counts, int c2, int c4, int c8, int64_t T, int D, int rows,
                uint16_t *__restrict__ out, int32_t *__restrict__ check, uint64_t *__restrict__ words, uint32_t tag) {
  extern __shared__ __attribute__((aligned(16))) uint8_t s_rows[];
  // per channel: where its code lies in a row (LDS offset | segment << 16 | shift << 18) and
  // its scale | zero point
  __shared__ uint32_t s_at[kChan], s_sz[kChan];
  const int h = blockIdx.y, ch0 = blockIdx.z * kChan, tid = threadIdx.x;
  if (tid < kChan) {
    s_at[tid] = 3u << 16;               // a pruned channel: code 0, scale 0, zero point 0 -> +0
    s_sz[tid] = 0;
  }
  const int n2p = 4 * s2.sub, n4p = 2 * s4.sub;
  // LDS areas of the three segments; each begins at the misalignment of its tile's first byte
  const int area4 = (rows * s2.sub + 47) & ~15, area8 = area4 + ((rows * s4.sub + 47) & ~15);
  int n2 = c2, n4 = c4, n8 = c8;
  if (counts) {
    n2 = counts[3 * h];
    n4 = counts[3 * h + 1];
    n8 = counts[3 * h + 2];
  }
  // (counts of a tensor that was overwritten must not lead outside the rows; the host reports them)
  const bool reports = (check || words) && blockIdx.x == 0 && blockIdx.z == 0;
  auto report = [&](int i, int v) {
    if (check) check[4 * h + i] = v;
    if (words) rdkv_host_word(words, 4 * (int64_t)h + i, tag, v);
  };
  if (reports && tid == 0) {
    report(0, n2);
    report(1, n4);
    report(2, n8);
  }
  n2 = min(max(n2, 0), n2p);
  n4 = min(max(n4, 0), n4p);
  n8 = min(max(n8, 0), s8.sub);
  const int kept = min(n2 + n4 + n8, sort_n);
  __syncthreads();
  bool whole = true, outside = false;
  for (int i = tid; i < kept; i += 256) {
    const int64_t ch = sort_idx[h * sort_sh + i] - ch0;
    outside = outside || ch + ch0 < 0 || ch + ch0 >= D;
    const int slot = i < n2 ? i : i < n2 + n4 ? n2p + (i - n2) : n2p + n4p + (i - n2 - n4);
    const __half sc = scale[h * ks_sh + slot], zz = zp[h * ks_sh + slot];
    uint32_t at;
    if (i < n2)
      at = (slot % s2.sub) | (2 * (slot / s2.sub)) << 18;
    else if (i < n2 + n4)
      at = (area4 + (slot - n2p) % s4.sub) | 1u << 16 | (4 * ((slot - n2p) / s4.sub)) << 18;
    else
      at = (area8 + slot - n2p - n4p) | 2u << 16;
    if (ch < 0 || ch >= kChan) continue;
    s_at[ch] = at;
    s_sz[ch] = __half_as_ushort(sc) | (uint32_t)__half_as_ushort(zz) << 16;
    whole = whole && whole_zp(__half2float(zz));
  }
  whole = __syncthreads_and(whole);
  if (reports) {
    outside = __syncthreads_or(outside);
    if (tid == 0) report(3, outside ? 1 : 0);
  }
  const int oct = tid & 15, c0 = 8 * oct;
  int at[8], step[8], seg[8], shift[8], width[8];
  uint32_t sz[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t a = s_at[c0 + j];
    sz[j] = s_sz[c0 + j];
    seg[j] = (a >> 16) & 3;
    at[j] = seg[j] == 3 ? 0 : a & 0xffffu;
    shift[j] = a >> 18;
    width[j] = seg[j] == 3 ? 0 : 2 << seg[j];
    step[j] = seg[j] == 0 ? s2.sub : seg[j] == 1 ? s4.sub : seg[j] == 2 ? s8.sub : 0;
  }
  uint32_t sc2[4], zz2[4];              // the pairs' scales, and 1024 + zero point
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sc2[j] = (sz[2 * j] & 0xffffu) | sz[2 * j + 1] << 16;
    zz2[j] = rdkv_f2h(1024.0f + rdkv_h2f(sz[2 * j] >> 16)) | (uint32_t)rdkv_f2h(1024.0f + rdkv_h2f(sz[2 * j + 1] >> 16)) << 16;
  }
  const KSeg segs[3] = {s2, s4, s8};
  const int areas[3] = {0, area4, area8};
  const int64_t n_tiles = (T + rows - 1) / rows;
  for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const int64_t t0 = tile * rows;
    const int n = (int)min((int64_t)rows, T - t0);
    int mis[3] = {0, 0, 0};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if (segs[k].sub == 0) continue;
      const uint8_t *p = segs[k].base + h * segs[k].stride_h + t0 * segs[k].stride_t;
      if (DENSE) {
        // whole aligned 16-byte pieces: the first and the last may begin before and end after the
        // tile's bytes, inside the same 16 bytes as one of them
        mis[k] = (int)(reinterpret_cast<uintptr_t>(p) & 15);
        const int bytes = mis[k] + n * segs[k].sub;
        const u32x4 *src = reinterpret_cast<const u32x4 *>(p - mis[k]);
        u32x4 *dst = reinterpret_cast<u32x4 *>(s_rows + areas[k]);
        for (int i = tid; 16 * i < bytes; i += 256) dst[i] = src[i];
      } else {
        for (int i = tid; i < n * segs[k].sub; i += 256)
          s_rows[areas[k] + i] = p[(i / segs[k].sub) * segs[k].stride_t + i % segs[k].sub];
      }
    }
    __syncthreads();
    int pos[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      pos[j] = at[j] + (seg[j] == 0 ? mis[0] : seg[j] == 1 ? mis[1] : seg[j] == 2 ? mis[2] : 0) + (tid >> 4) * step[j];
    uint16_t *o = out + ((int64_t)h * T + t0 + (tid >> 4)) * D + ch0 + c0;
    for (int r = tid >> 4; r < n; r += 16, o += 16 * (int64_t)D) {
      uint32_t code[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        code[j] = __builtin_amdgcn_ubfe((uint32_t)s_rows[pos[j]], shift[j], width[j]);
        pos[j] += 16 * step[j];
      }
      u32x4 v;
      if (whole) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = dequant_pair(code[2 * j] | code[2 * j + 1] << 16, zz2[j], sc2[j]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t lo = dequant_bits(code[2 * j], rdkv_h2f(sz[2 * j] >> 16), rdkv_h2f(sz[2 * j] & 0xffffu));
          const uint32_t hi = dequant_bits(code[2 * j + 1], rdkv_h2f(sz[2 * j + 1] >> 16), rdkv_h2f(sz[2 * j + 1] & 0xffffu));
          v[j] = lo | hi << 16;
        }
      }
      if ((D & 7) == 0) {
        if (ch0 + c0 < D) __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(o));
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (ch0 + c0 + j < D) o[j] = (uint16_t)(v[j >> 1] >> (16 * (j & 1)));
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// V.  grid = (ceil(T / 64), H_kv, channel chunks of 128), four tokens per thread group of sixteen.
// Rows [0, max_tv): the head's 2-, 4- and 8-bit tokens one class after the other, zeros behind them;
// rows [max_tv, max_tv + n16): the fp16 rows as they are.  Eight channels of a thread lie in one
// quarter (half) of the split layout, so their codes are eight consecutive bytes at one shift.
// Bound: the rows read and written: 77 MB in 14.5 us for 8 heads of 25 300 rows (5.3 TB/s, the rate of
// a large copy; 19 us with plain stores).
// ---------------------------------------------------------------------------
template <bool WIDE>
__global__ void __launch_bounds__(256)
unpack_v_kernel(const uint8_t *__restrict__ V2, int64_t v2_sh, const uint8_t *__restrict__ V4, int64_t v4_sh,
                const uint8_t *__restrict__ V8, int64_t v8_sh, const __half *__restrict__ scale,
                const __half *__restrict__ zp, int64_t s_sh, const int32_t *__restrict__ counts, int m2, int m4, int m8,
                int64_t max_tv, const uint16_t *__restrict__ V16, int64_t v16_sh, int n16, int D,
                uint16_t *__restrict__ out, const int32_t *__restrict__ totals, uint64_t *__restrict__ words, uint32_t tag) {
  constexpr int kTok = 4;
  const int h = blockIdx.y, c0 = blockIdx.z * kChan + 8 * (threadIdx.x & 15);
  const int64_t T = max_tv + n16;
  if (words && blockIdx.x == 0 && blockIdx.z == 0 && threadIdx.x < 4)
    rdkv_host_word(words, 4 * (int64_t)h + threadIdx.x, tag, threadIdx.x < 3 ? counts[3 * h + threadIdx.x] : totals[h]);
  // (clamped as above; a head never has more rows than the stripe)
  const int64_t e2 = min((int64_t)min(max(counts[3 * h], 0), m2), max_tv);
  const int64_t e4 = min(e2 + min(max(counts[3 * h + 1], 0), m4), max_tv);
  const int64_t e8 = min(e4 + min(max(counts[3 * h + 2], 0), m8), max_tv);
  if (c0 >= D) return;
  const int q2 = max(D / 4, 1), q4 = max(D / 2, 1);    // (not used by rows of a width that D cannot have)
  const int off2 = c0 % q2, off4 = c0 % q4, sh2 = 2 * (c0 / q2), sh4 = 4 * (c0 / q4);
  u32x2 codes[kTok];
  __half sc[kTok], zz[kTok];
  int bits[kTok], shift[kTok];
  // every load before the first use, none in a branch of its own: a row without codes reads the start
  // of the output instead
#pragma unroll
  for (int k = 0; k < kTok; ++k) {
    const int64_t t = (int64_t)blockIdx.x * 64 + 16 * k + (threadIdx.x >> 4);
    const bool in2 = t < e2, in4 = t < e4, in8 = t < e8;
    bits[k] = in2 ? 2 : in4 ? 4 : in8 ? 8 : 0;
    shift[k] = in2 ? sh2 : in4 ? sh4 : 0;
    const uint8_t *row = reinterpret_cast<const uint8_t *>(out);
    row = in8 ? V8 + h * v8_sh + (t - e4) * D : row;
    row = in4 ? V4 + h * v4_sh + (t - e2) * q4 : row;
    row = in2 ? V2 + h * v2_sh + t * q2 : row;
    const int64_t m = in8 ? h * s_sh + t : 0;
    sc[k] = scale[m];
    zz[k] = zp[m];
    if (WIDE) {
      codes[k] = *reinterpret_cast<const u32x2 *>(row + (in2 ? off2 : in4 ? off4 : in8 ? c0 : 0));
    } else {
      uint32_t b[2] = {0, 0};
      const int width = in2 ? q2 : in4 ? q4 : D;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int c = c0 + j;
        if (c < D && in8) b[j >> 2] |= ((row[c % width] >> (bits[k] * (c / width))) & 255u) << (8 * (j & 3));
      }
      codes[k] = u32x2{b[0], b[1]};
      shift[k] = 0;
    }
  }
#pragma unroll
  for (int k = 0; k < kTok; ++k) {
    const int64_t t = (int64_t)blockIdx.x * 64 + 16 * k + (threadIdx.x >> 4);
    if (t >= T) continue;
    uint16_t *o = out + ((int64_t)h * T + t) * D + c0;
    const uint16_t *kept = t >= max_tv ? V16 + h * v16_sh + (t - max_tv) * D + c0 : nullptr;
    const uint32_t m = (1u << bits[k]) - 1u, field = m | m << 16;
    const float sf = bits[k] ? __half2float(sc[k]) : 0.0f, zf = bits[k] ? __half2float(zz[k]) : 0.0f;
    u32x4 v;
    if (whole_zp(zf)) {
      const uint32_t s2 = rdkv_f2h(sf) * 0x10001u, z2 = rdkv_f2h(1024.0f + zf) * 0x10001u;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // bytes 2j and 2j+1 of the eight codes, one in each half (bits above a field are cut off after the shift)
        const uint32_t pair = __builtin_amdgcn_perm(0u, codes[k][j >> 1], j & 1 ? 0x0c030c02u : 0x0c010c00u);
        v[j] = dequant_pair((pair >> shift[k]) & field, z2, s2);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t b = codes[k][j >> 1] >> (shift[k] + 16 * (j & 1));
        v[j] = dequant_bits(b & m, zf, sf) | dequant_bits((b >> 8) & m, zf, sf) << 16;
      }
    }
    if (WIDE) {
      if (kept) v = *reinterpret_cast<const u32x4 *>(kept);
      __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(o));
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (c0 + j < D) o[j] = kept ? kept[j] : (uint16_t)(v[j >> 1] >> (16 * (j & 1)));
    }
  }
}

}  // namespace

static int unpack_layer_k(const uint8_t *K2, int64_t k2_stride_h, int64_t k2_stride_t, const uint8_t *K4,
                          int64_t k4_stride_h, int64_t k4_stride_t, const uint8_t *K8, int64_t k8_stride_h,
                          int64_t k8_stride_t, const void *scale_f16, const void *zp_f16, int64_t ks_stride_h,
                          const int64_t *sort_idx, int64_t sort_stride_h, int sort_n, const int32_t *counts, int n2,
                          int n4, int n8, int n2p, int n4p, int n8w, int H_kv, int64_t T, int D, void *out_f16,
                          int32_t *check, uint64_t *words, uint32_t tag, void *stream) {
  RDKV_REQUIRE(H_kv >= 1 && H_kv <= 65535 && T >= 0 && D >= 1 && D <= 65535 * kChan, "rdkv_unpack_layer_k: bad shape");
  RDKV_REQUIRE(n2p >= 0 && n2p % 4 == 0 && n4p >= 0 && n4p % 2 == 0 && n8w >= 0 && sort_n >= 0,
               "rdkv_unpack_layer_k: bad segment widths %d/%d/%d", n2p, n4p, n8w);
  if (T == 0) return RDKV_OK;
  KSeg s2{K2, k2_stride_h, k2_stride_t, K2 ? n2p / 4 : 0}, s4{K4, k4_stride_h, k4_stride_t, K4 ? n4p / 2 : 0},
      s8{K8, k8_stride_h, k8_stride_t, K8 ? n8w : 0};
  RDKV_REQUIRE((K2 || n2p == 0) && (K4 || n4p == 0) && (K8 || n8w == 0), "rdkv_unpack_layer_k: null segment");
  const int row_bytes = s2.sub + s4.sub + s8.sub;
  RDKV_REQUIRE(out_f16 && (row_bytes == 0 || (scale_f16 && zp_f16)) && (sort_n == 0 || sort_idx),
               "rdkv_unpack_layer_k: null pointer");
  RDKV_REQUIRE(D % 8 || ((uintptr_t)out_f16 % 16) == 0, "rdkv_unpack_layer_k: output rows must be 16-byte aligned");
  RDKV_REQUIRE(row_bytes <= kLdsBytes, "rdkv_unpack_layer_k: rows of %d bytes", row_bytes);
  const int rows = row_bytes ? (kLdsBytes / row_bytes < kMaxTileRows ? kLdsBytes / row_bytes : kMaxTileRows) : kMaxTileRows;
  const size_t lds = (size_t)rows * row_bytes + 3 * 48;
  const bool dense = k2_stride_t == s2.sub && k4_stride_t == s4.sub && k8_stride_t == s8.sub;
  const int chunks = (int)rdkv_cdiv(D, kChan);
  // eight workgroups per compute unit keep its wavefront slots full, each pays its channel tables once,
  // and all get the same number of tiles
  const int64_t most = rdkv_cdiv(2048, (int64_t)H_kv * chunks), tiles = rdkv_cdiv(T, rows);
  const int64_t per_head = rdkv_cdiv(tiles, rdkv_cdiv(tiles, most));
  dim3 g((unsigned)per_head, H_kv, chunks);
  hipLaunchKernelGGL(dense ? unpack_k_kernel<true> : unpack_k_kernel<false>, g, dim3(256), lds, (hipStream_t)stream, s2, s4,
                     s8, (const __half *)scale_f16, (const __half *)zp_f16, ks_stride_h, sort_idx, sort_stride_h, sort_n,
                     counts, n2, n4, n8, T, D, rows, (uint16_t *)out_f16, check, words, tag);
  RDKV_CHECK_LAUNCH("rdkv_unpack_layer_k");
  return RDKV_OK;
}

RDKV_API int rdkv_unpack_layer_k(const uint8_t *K2, int64_t k2_stride_h, int64_t k2_stride_t, const uint8_t *K4,
                                 int64_t k4_stride_h, int64_t k4_stride_t, const uint8_t *K8, int64_t k8_stride_h,
                                 int64_t k8_stride_t, const void *scale_f16, const void *zp_f16, int64_t ks_stride_h,
                                 const int64_t *sort_idx, int64_t sort_stride_h, int sort_n, const int32_t *counts,
                                 int n2, int n4, int n8, int n2p, int n4p, int n8w, int H_kv, int64_t T, int D,
                                 void *out_f16, void *stream) {
  return unpack_layer_k(K2, k2_stride_h, k2_stride_t, K4, k4_stride_h, k4_stride_t, K8, k8_stride_h, k8_stride_t, scale_f16,
                        zp_f16, ks_stride_h, sort_idx, sort_stride_h, sort_n, counts, n2, n4, n8, n2p, n4p, n8w, H_kv, T, D,
                        out_f16, nullptr, nullptr, 0, stream);
}

RDKV_API int rdkv_unpack_layer_k_checked(
    const uint8_t *K2, int64_t k2_stride_h, int64_t k2_stride_t, const uint8_t *K4, int64_t k4_stride_h,
    int64_t k4_stride_t, const uint8_t *K8, int64_t k8_stride_h, int64_t k8_stride_t, const void *scale_f16,
    const void *zp_f16, int64_t ks_stride_h, const int64_t *sort_idx, int64_t sort_stride_h, int sort_n,
    const int32_t *counts, int n2, int n4, int n8, int n2p, int n4p, int n8w, int H_kv, int64_t T, int D, void *out_f16,
    int32_t *check, void *stream) {
  RDKV_REQUIRE(check && T > 0, "rdkv_unpack_layer_k_checked: nothing to check into or no rows");
  return unpack_layer_k(K2, k2_stride_h, k2_stride_t, K4, k4_stride_h, k4_stride_t, K8, k8_stride_h, k8_stride_t, scale_f16,
                        zp_f16, ks_stride_h, sort_idx, sort_stride_h, sort_n, counts, n2, n4, n8, n2p, n4p, n8w, H_kv, T, D,
                        out_f16, check, nullptr, 0, stream);
}

RDKV_API int rdkv_unpack_layer_k_words(
    const uint8_t *K2, int64_t k2_stride_h, int64_t k2_stride_t, const uint8_t *K4, int64_t k4_stride_h,
    int64_t k4_stride_t, const uint8_t *K8, int64_t k8_stride_h, int64_t k8_stride_t, const void *scale_f16,
    const void *zp_f16, int64_t ks_stride_h, const int64_t *sort_idx, int64_t sort_stride_h, int sort_n,
    const int32_t *counts, int n2, int n4, int n8, int n2p, int n4p, int n8w, int H_kv, int64_t T, int D, void *out_f16,
    uint64_t *words, uint32_t tag, void *stream) {
  RDKV_REQUIRE(words && T > 0, "rdkv_unpack_layer_k_words: no words or no rows");
  return unpack_layer_k(K2, k2_stride_h, k2_stride_t, K4, k4_stride_h, k4_stride_t, K8, k8_stride_h, k8_stride_t, scale_f16,
                        zp_f16, ks_stride_h, sort_idx, sort_stride_h, sort_n, counts, n2, n4, n8, n2p, n4p, n8w, H_kv, T, D,
                        out_f16, nullptr, words, tag, stream);
}

static int unpack_layer_v(const uint8_t *V2, int64_t v2_stride_h, const uint8_t *V4, int64_t v4_stride_h,
                          const uint8_t *V8, int64_t v8_stride_h, const void *scale_f16, const void *zp_f16,
                          int64_t s_stride_h, const int32_t *counts, int m2, int m4, int m8, int64_t max_tv,
                          const void *V16_f16, int64_t v16_stride_h, int n16, int H_kv, int D, void *out_f16,
                          const int32_t *totals, uint64_t *words, uint32_t tag, void *stream) {
  RDKV_REQUIRE(H_kv >= 1 && H_kv <= 65535 && max_tv >= 0 && n16 >= 0 && D >= 1 && D <= 65535 * kChan,
               "rdkv_unpack_layer_v: bad shape");
  RDKV_REQUIRE((!V2 || m2 <= 0 || D % 4 == 0) && (!V4 || m4 <= 0 || D % 2 == 0),
               "rdkv_unpack_layer_v: rows of %d codes that are no whole bytes", D);
  const int64_t T = max_tv + n16;
  if (T == 0) return RDKV_OK;
  if (!V2) m2 = 0;
  if (!V4) m4 = 0;
  if (!V8) m8 = 0;
  RDKV_REQUIRE(m2 >= 0 && m4 >= 0 && m8 >= 0, "rdkv_unpack_layer_v: negative counts");
  RDKV_REQUIRE(out_f16 && counts && (n16 == 0 || V16_f16) && (m2 + m4 + m8 == 0 || (scale_f16 && zp_f16)),
               "rdkv_unpack_layer_v: null pointer");
  const int64_t blocks = rdkv_cdiv(T, 64);
  RDKV_REQUIRE(blocks <= 0x7fffffffLL, "rdkv_unpack_layer_v: too many rows");
  if (m2 + m4 + m8 == 0) scale_f16 = zp_f16 = out_f16;      // (read, and not used, where no row has codes)
  // eight codes of a thread as one 8-byte load: a quarter row is whole 8-byte pieces, rows aligned
  const bool wide = D % 32 == 0 && (((uintptr_t)V2 | (uintptr_t)V4 | (uintptr_t)V8) % 8) == 0 &&
                    ((v2_stride_h | v4_stride_h | v8_stride_h) % 8) == 0 && ((uintptr_t)out_f16 % 16) == 0 &&
                    ((uintptr_t)V16_f16 % 16) == 0 && v16_stride_h % 8 == 0;
  dim3 g((unsigned)blocks, H_kv, (unsigned)rdkv_cdiv(D, kChan));
  hipLaunchKernelGGL(wide ? unpack_v_kernel<true> : unpack_v_kernel<false>, g, dim3(256), 0, (hipStream_t)stream, V2,
                     v2_stride_h, V4, v4_stride_h, V8, v8_stride_h, (const __half *)scale_f16, (const __half *)zp_f16,
                     s_stride_h, counts, m2, m4, m8, max_tv, (const uint16_t *)V16_f16, v16_stride_h, n16, D,
                     (uint16_t *)out_f16, totals, words, tag);
  RDKV_CHECK_LAUNCH("rdkv_unpack_layer_v");
  return RDKV_OK;
}

RDKV_API int rdkv_unpack_layer_v(const uint8_t *V2, int64_t v2_stride_h, const uint8_t *V4, int64_t v4_stride_h,
                                 const uint8_t *V8, int64_t v8_stride_h, const void *scale_f16, const void *zp_f16,
                                 int64_t s_stride_h, const int32_t *counts, int m2, int m4, int m8, int64_t max_tv,
                                 const void *V16_f16, int64_t v16_stride_h, int n16, int H_kv, int D, void *out_f16,
                                 void *stream) {
  return unpack_layer_v(V2, v2_stride_h, V4, v4_stride_h, V8, v8_stride_h, scale_f16, zp_f16, s_stride_h, counts, m2, m4, m8,
                        max_tv, V16_f16, v16_stride_h, n16, H_kv, D, out_f16, nullptr, nullptr, 0, stream);
}

RDKV_API int rdkv_unpack_layer_v_words(const uint8_t *V2, int64_t v2_stride_h, const uint8_t *V4, int64_t v4_stride_h,
                                       const uint8_t *V8, int64_t v8_stride_h, const void *scale_f16, const void *zp_f16,
                                       int64_t s_stride_h, const int32_t *counts, int m2, int m4, int m8, int64_t max_tv,
                                       const void *V16_f16, int64_t v16_stride_h, int n16, int H_kv, int D, void *out_f16,
                                       const int32_t *totals, uint64_t *words, uint32_t tag, void *stream) {
  RDKV_REQUIRE(words && totals && max_tv + n16 > 0, "rdkv_unpack_layer_v_words: no words, no totals or no rows");
  return unpack_layer_v(V2, v2_stride_h, V4, v4_stride_h, V8, v8_stride_h, scale_f16, zp_f16, s_stride_h, counts, m2, m4, m8,
                        max_tv, V16_f16, v16_stride_h, n16, H_kv, D, out_f16, totals, words, tag, stream);
}
