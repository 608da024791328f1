// A packed layer back to dense fp16 K and V, with its additive padding mask: one launch, every output byte
// written once.
// The values are the ones rdkv_dequant_f16 gives segment by segment (half((code - zp) * scale),
// obkv_accel/packing.py:581-709, 1427-1444, trizone_decompress.py:91-182); here the channel scatter
// of K, the class walk of V, the zero rows of the stripe and the fp16-kept rows are part of the
// same pass, so nothing is dequantized into a temporary and copied again.
// The per-head counts that the host checks leave the launches as words in host memory when their first workgroup
// starts (rdkv_host_word); joined, copied and the stream waited for, they took 67 us more for two layers of 16k tokens.
// Bound: the bytes.  A layer of 8 heads x 25 300 rows (104 MB written, 20 read) takes 25.4 us, 4.9 TB/s; a launch for K
// (18.8 us), one for V (14) and one for the mask (3) took 36, for K's workgroups are bound by the instructions of their
// set-up and the chain tables -> rows, V's by their loads, and side by side each fills the other's waits.  Two layers
// and their masks 103 -> 86 us a call, 48 of them on the device.
#include "rdkv_common.h"

namespace {

constexpr int kChan = 128;        // channels of a workgroup (16 threads x 8), further ones in grid.z
constexpr int kLdsBytes = 48 << 10;
constexpr int kMaxTileRows = 128;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
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

// What a launch does: workgroups of one kind follow those of the other, so that K's (bound by their instructions)
// and V's (bound by their bytes) share a compute unit.
struct KSide {
  KSeg seg[3];
  const __half *scale, *zp;
  int64_t ks_sh;
  const int64_t *sort_idx;
  int64_t sort_sh;
  const int32_t *counts;
  int64_t T;
  uint16_t *out;
  int32_t *check;
  uint64_t *words;
  int sort_n, n[3], rows;
  int blocks;               // workgroups per head (and chunk of channels)
  uint32_t tag;
};
struct VSide {
  const uint8_t *seg[3];
  int64_t sh[3];
  const __half *scale, *zp;
  int64_t s_sh;
  const int32_t *counts, *totals;
  int64_t max_tv;
  const uint16_t *V16;
  int64_t v16_sh;
  uint16_t *out;
  uint64_t *words;
  int m[3], n16;
  int blocks;
  uint32_t tag;
};
// fp32 rows to fp16 rows with zeros behind them (the additive padding mask)
struct MaskSide {
  const float *in;
  uint16_t *out;
  uint32_t n, width, out_width;       // elements written; of a row
  int blocks;
};

// ---------------------------------------------------------------------------
// K.  A workgroup walks tiles of `rows` tokens: the tile's packed rows go to LDS with direct 16-byte loads (rows
// stored back to back; byte copies otherwise), asked for before the channel tables, which hide them; then sixteen
// threads share a token, each writing eight channels with one 16-byte store.  A thread's channels are the same for
// every token, so where their codes lie in a row, their scales and zero points are worked out once per workgroup.
// Codes are dequantized as packed fp16 pairs (bit-identical where the zero points are whole numbers, which the
// quantizer's are), two thirds fewer vector instructions than in fp32.
// Nothing reads the rows soon, so they are stored with the nontemporal hint.
// ---------------------------------------------------------------------------
template <bool DENSE>
__device__ __forceinline__ void unpack_k(const KSide &k, int D, int bx, uint8_t *s_rows, uint32_t *s_at, uint32_t *s_step,
                                         uint32_t *s_sz) {
  const int h = blockIdx.y, ch0 = blockIdx.z * kChan, tid = threadIdx.x, rows = k.rows;
  const int64_t T = k.T, n_tiles = (T + rows - 1) / rows;
  const int sub2 = k.seg[0].sub, sub4 = k.seg[1].sub, sub8 = k.seg[2].sub;
  // LDS areas of the three segments; each begins at the misalignment of its tile's first byte, the same for every
  // tile of a head (rows is a multiple of 16)
  const int area[3] = {0, (rows * sub2 + 47) & ~15, ((rows * sub2 + 47) & ~15) + ((rows * sub4 + 47) & ~15)};
  const uint8_t *base[3];
  int mis[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    base[i] = k.seg[i].base + h * k.seg[i].stride_h;
    mis[i] = DENSE ? (int)(reinterpret_cast<uintptr_t>(base[i]) & 15) : 0;
  }
  auto request = [&](int64_t tile) __attribute__((always_inline)) {
    const int64_t t0 = tile * rows;
    const int n = (int)min((int64_t)rows, T - t0);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int sub = k.seg[i].sub;
      if (sub == 0) continue;
      const uint8_t *p = base[i] + t0 * k.seg[i].stride_t;
      if (DENSE) {
        // whole aligned 16-byte pieces: the first and the last may begin before and end after the
        // tile's bytes, inside the same 16 bytes as one of them
        const int bytes = mis[i] + n * sub;
        const uint8_t *src = p - mis[i] + 16 * tid;
        uint8_t *dst = s_rows + area[i] + 1024 * __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll 1
        for (int at = 0; at < bytes; at += 4096)
          if (at + 16 * tid < bytes)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + at),
                                             (__attribute__((address_space(3))) void *)(dst + at), 16, 0, 0);
      } else {
#pragma unroll 1
        for (int at = tid; at < n * sub; at += 256) s_rows[area[i] + at] = p[(at / sub) * k.seg[i].stride_t + at % sub];
      }
    }
  };
  int64_t tile = bx;
  if (tile < n_tiles) request(tile);
  if (tid < kChan) {
    s_at[tid] = 0;                      // a pruned channel: code 0, scale 0, zero point 0 -> +0
    s_step[tid] = 0;
    s_sz[tid] = 0;
  }
  const int n2p = 4 * sub2, n4p = 2 * sub4;
  int n2 = k.n[0], n4 = k.n[1], n8 = k.n[2];
  if (k.counts) {
    n2 = k.counts[3 * h];
    n4 = k.counts[3 * h + 1];
    n8 = k.counts[3 * h + 2];
  }
  // (counts of a tensor that was overwritten must not lead outside the rows; the host reports them)
  const bool reports = (k.check || k.words) && bx == 0 && blockIdx.z == 0;
  auto report = [&](int i, int v) {
    if (k.check) k.check[4 * h + i] = v;
    if (k.words) rdkv_host_word(k.words, 4 * (int64_t)h + i, k.tag, v);
  };
  if (reports && tid == 0) {
    report(0, n2);
    report(1, n4);
    report(2, n8);
  }
  n2 = min(max(n2, 0), n2p);
  n4 = min(max(n4, 0), n4p);
  n8 = min(max(n8, 0), sub8);
  const int kept = min(n2 + n4 + n8, k.sort_n);
  __syncthreads();
  bool whole = true, outside = false;
#pragma unroll 1
  for (int i = tid; i < kept; i += 256) {
    const int64_t ch = k.sort_idx[h * k.sort_sh + i] - ch0;
    outside = outside || ch + ch0 < 0 || ch + ch0 >= D;
    const bool in2 = i < n2, in4 = !in2 && i < n2 + n4;
    const int of = in2 ? i : in4 ? i - n2 : i - n2 - n4, slot = of + (in2 ? 0 : in4 ? n2p : n2p + n4p);
    const __half sc = k.scale[h * k.ks_sh + slot], zz = k.zp[h * k.ks_sh + slot];
    // (a quarter of the row's 2-bit bytes, or half of its 4-bit ones, per bit position)
    const int part = in2 ? (of >= sub2) + (of >= 2 * sub2) + (of >= 3 * sub2) : in4 ? of >= sub4 : 0;
    const int sub = in2 ? sub2 : in4 ? sub4 : sub8;
    if (ch < 0 || ch >= kChan) continue;
    s_at[ch] = ((in2 ? area[0] + mis[0] : in4 ? area[1] + mis[1] : area[2] + mis[2]) + of - part * sub) |
               (in2 ? 3u << 24 | 2 * part << 16 : in4 ? 15u << 24 | 4 * part << 16 : 255u << 24);
    s_step[ch] = sub;
    s_sz[ch] = __half_as_ushort(sc) | (uint32_t)__half_as_ushort(zz) << 16;
    whole = whole && whole_zp(__half2float(zz));
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0): this wavefront's pieces of the first tile are in LDS
  whole = __syncthreads_and(whole);
  if (reports) {
    outside = __syncthreads_or(outside);
    if (tid == 0) report(3, outside ? 1 : 0);
  }
  const int c0 = 8 * (tid & 15), row0 = tid >> 4;
  int at[8], step[8];
  u16x2 shift[4];                       // of the pairs
  uint32_t mask[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    mask[j] = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t a = s_at[c0 + 2 * j + i], sub = s_step[c0 + 2 * j + i];
      at[2 * j + i] = (a & 0xffffu) + row0 * sub;
      step[2 * j + i] = 16 * sub;
      shift[j][i] = (a >> 16) & 255u;
      mask[j] |= (a >> 24) << (16 * i);
    }
  }
  if (tile >= n_tiles) return;
  const auto *lds = (const __attribute__((address_space(3))) uint8_t *)s_rows;
  uint32_t sc2[4], zz2[4];              // the pairs' scales, and 1024 + zero point
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t lo = s_sz[c0 + 2 * j], hi = s_sz[c0 + 2 * j + 1];
    sc2[j] = (lo & 0xffffu) | hi << 16;
    zz2[j] = rdkv_f2h(1024.0f + rdkv_h2f(lo >> 16)) | (uint32_t)rdkv_f2h(1024.0f + rdkv_h2f(hi >> 16)) << 16;
  }
  const bool fast = whole && (D & 7) == 0, inside = ch0 + c0 < D;
  for (;;) {
    const int64_t t0 = tile * rows;
    const int n = (int)min((int64_t)rows, T - t0);
    const __attribute__((address_space(3))) uint8_t *pos[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) pos[j] = lds + at[j];
    uint16_t *o = k.out + ((int64_t)h * T + t0 + row0) * D + ch0 + c0;
    auto codes = [&](int j) __attribute__((always_inline)) {
      const u16x2 bytes = {*pos[2 * j], *pos[2 * j + 1]};
      pos[2 * j] += step[2 * j];
      pos[2 * j + 1] += step[2 * j + 1];
      return __builtin_bit_cast(uint32_t, bytes >> shift[j]) & mask[j];
    };
    if (fast) {
#pragma unroll 1
      for (int r = row0; r < n; r += 16, o += 16 * (int64_t)D) {
        u32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = dequant_pair(codes(j), zz2[j], sc2[j]);
        if (inside) __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(o));
      }
    } else {
#pragma unroll 1
      for (int r = row0; r < n; r += 16, o += 16 * (int64_t)D)
#pragma unroll 1
        for (int j = 0; j < 8; ++j) {     // (scales and zero points from LDS for each row: the registers are the fast path's)
          const uint32_t a = s_at[c0 + j], sz = s_sz[c0 + j];
          const uint32_t code = (uint32_t)(s_rows[(a & 0xffffu) + r * s_step[c0 + j]] >> (a >> 16 & 255u)) & (a >> 24);
          if (ch0 + c0 + j < D) o[j] = (uint16_t)dequant_bits(code, rdkv_h2f(sz >> 16), rdkv_h2f(sz & 0xffffu));
        }
    }
    tile += k.blocks;
    if (tile >= n_tiles) return;
    __syncthreads();                         // every wavefront has done with the rows
    request(tile);
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// V.  64 tokens a workgroup, four per thread group of sixteen.
// Rows [0, max_tv): the head's 2-, 4- and 8-bit tokens one class after the other, zeros behind them;
// rows [max_tv, max_tv + n16): the fp16 rows as they are.  Eight channels of a thread lie in one
// quarter (half) of the split layout, so their codes are eight consecutive bytes at one shift.
// Bound: the rows read and written: 77 MB in 14.5 us for 8 heads of 25 300 rows (5.3 TB/s, the rate of
// a large copy; 19 us with plain stores).
// ---------------------------------------------------------------------------
template <bool WIDE>
__device__ __forceinline__ void unpack_v(const VSide &v_, int D, int bx) {
  constexpr int kTok = 4;
  const int h = blockIdx.y, c0 = blockIdx.z * kChan + 8 * (threadIdx.x & 15);
  const int32_t *counts = v_.counts;
  const int64_t max_tv = v_.max_tv, T = max_tv + v_.n16, s_sh = v_.s_sh, v16_sh = v_.v16_sh;
  const uint8_t *V2 = v_.seg[0], *V4 = v_.seg[1], *V8 = v_.seg[2];
  const int64_t v2_sh = v_.sh[0], v4_sh = v_.sh[1], v8_sh = v_.sh[2];
  const int m2 = v_.m[0], m4 = v_.m[1], m8 = v_.m[2];
  const __half *scale = v_.scale, *zp = v_.zp;
  const uint16_t *V16 = v_.V16;
  uint16_t *out = v_.out;
  if (v_.words && bx == 0 && blockIdx.z == 0 && threadIdx.x < 4)
    rdkv_host_word(v_.words, 4 * (int64_t)h + threadIdx.x, v_.tag,
                   threadIdx.x < 3 ? counts[3 * h + threadIdx.x] : v_.totals[h]);
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
    const int64_t t = (int64_t)bx * 64 + 16 * k + (threadIdx.x >> 4);
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
    const int64_t t = (int64_t)bx * 64 + 16 * k + (threadIdx.x >> 4);
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

// grid = (workgroups of the three kinds, H_kv, channel chunks of 128)
template <bool DENSE, bool WIDE>
__global__ void __launch_bounds__(256, DENSE ? 8 : 4) unpack_layer_kernel(KSide k, VSide v, MaskSide m, int D) {
  extern __shared__ __attribute__((aligned(16))) uint8_t s_rows[];
  // per channel: where its code lies in a row (LDS byte | shift << 16 | mask << 24), the bytes of a row of its
  // segment, and its scale | zero point
  __shared__ __attribute__((aligned(16))) uint32_t s_at[kChan], s_step[kChan], s_sz[kChan];
  const int x = blockIdx.x, pairs = min(k.blocks, v.blocks);
  const bool of_pair = x < 2 * pairs;
  if (of_pair ? (x & 1) == 0 : x < 2 * pairs + k.blocks - pairs) {
    unpack_k<DENSE>(k, D, of_pair ? x >> 1 : x - pairs, s_rows, s_at, s_step, s_sz);
  } else if (x < k.blocks + v.blocks) {
    unpack_v<WIDE>(v, D, of_pair ? x >> 1 : x - k.blocks);
  } else if (blockIdx.z == 0) {
    const uint32_t first = (((uint32_t)blockIdx.y * m.blocks + x - k.blocks - v.blocks) * 8) * 256 + threadIdx.x;
#pragma unroll 1
    for (uint32_t i = first; i < min(m.n, first + 8 * 256); i += 256) {
      const uint32_t row = i / m.out_width, c = i - row * m.out_width;
      m.out[i] = c < m.width ? rdkv_f2h(m.in[(int64_t)row * m.width + c]) : (uint16_t)0;
    }
  }
}

}  // namespace

static int k_side(KSide &k, bool &dense, size_t &lds, const uint8_t *K2, int64_t k2_stride_h, int64_t k2_stride_t, const uint8_t *K4,
                          int64_t k4_stride_h, int64_t k4_stride_t, const uint8_t *K8, int64_t k8_stride_h,
                          int64_t k8_stride_t, const void *scale_f16, const void *zp_f16, int64_t ks_stride_h,
                          const int64_t *sort_idx, int64_t sort_stride_h, int sort_n, const int32_t *counts, int n2,
                          int n4, int n8, int n2p, int n4p, int n8w, int H_kv, int64_t T, int D, void *out_f16,
                          int32_t *check, uint64_t *words, uint32_t tag) {
  RDKV_REQUIRE(H_kv >= 1 && H_kv <= 65535 && T >= 0 && D >= 1 && D <= 65535 * kChan, "rdkv_unpack_layer_k: bad shape");
  RDKV_REQUIRE(n2p >= 0 && n2p % 4 == 0 && n4p >= 0 && n4p % 2 == 0 && n8w >= 0 && sort_n >= 0,
               "rdkv_unpack_layer_k: bad segment widths %d/%d/%d", n2p, n4p, n8w);
  if (T == 0) return RDKV_OK;      // (no workgroups)
  KSeg s2{K2, k2_stride_h, k2_stride_t, K2 ? n2p / 4 : 0}, s4{K4, k4_stride_h, k4_stride_t, K4 ? n4p / 2 : 0},
      s8{K8, k8_stride_h, k8_stride_t, K8 ? n8w : 0};
  RDKV_REQUIRE((K2 || n2p == 0) && (K4 || n4p == 0) && (K8 || n8w == 0), "rdkv_unpack_layer_k: null segment");
  const int row_bytes = s2.sub + s4.sub + s8.sub;
  RDKV_REQUIRE(out_f16 && (row_bytes == 0 || (scale_f16 && zp_f16)) && (sort_n == 0 || sort_idx),
               "rdkv_unpack_layer_k: null pointer");
  RDKV_REQUIRE(D % 8 || ((uintptr_t)out_f16 % 16) == 0, "rdkv_unpack_layer_k: output rows must be 16-byte aligned");
  RDKV_REQUIRE(row_bytes <= kLdsBytes, "rdkv_unpack_layer_k: rows of %d bytes", row_bytes);
  const int chunks = (int)rdkv_cdiv(D, kChan);
  // a workgroup pays its channel tables once, and a layer needs two workgroups a compute unit (8 heads of 25 300
  // rows 27.0 us with tiles of 64 rows, 25.4 with 128)
  int rows = T * H_kv * chunks >= 512 * kMaxTileRows ? kMaxTileRows : kMaxTileRows / 2;
  if (row_bytes && kLdsBytes / row_bytes < rows) rows = kLdsBytes / row_bytes;
  if (rows > 16) rows &= ~15;      // (whole sixteens: the tiles of a head are aligned alike)
  lds = (size_t)rows * row_bytes + 3 * 48;
  dense = k2_stride_t == s2.sub && k4_stride_t == s4.sub && k8_stride_t == s8.sub && rows % 16 == 0;
  // eight workgroups per compute unit keep its wavefront slots full, each pays its channel tables once,
  // and all get the same number of tiles
  const int64_t most = rdkv_cdiv(2048, (int64_t)H_kv * chunks), tiles = rdkv_cdiv(T, rows);
  k = KSide{{s2, s4, s8}, (const __half *)scale_f16, (const __half *)zp_f16, ks_stride_h, sort_idx, sort_stride_h, counts, T,
            (uint16_t *)out_f16, check, words, sort_n, {n2, n4, n8}, rows, (int)rdkv_cdiv(tiles, rdkv_cdiv(tiles, most)), tag};
  return RDKV_OK;
}

static int v_side(VSide &v, bool &wide, const uint8_t *V2, int64_t v2_stride_h, const uint8_t *V4, int64_t v4_stride_h,
                          const uint8_t *V8, int64_t v8_stride_h, const void *scale_f16, const void *zp_f16,
                          int64_t s_stride_h, const int32_t *counts, int m2, int m4, int m8, int64_t max_tv,
                          const void *V16_f16, int64_t v16_stride_h, int n16, int H_kv, int D, void *out_f16,
                          const int32_t *totals, uint64_t *words, uint32_t tag) {
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
  wide = D % 32 == 0 && (((uintptr_t)V2 | (uintptr_t)V4 | (uintptr_t)V8) % 8) == 0 &&
                    ((v2_stride_h | v4_stride_h | v8_stride_h) % 8) == 0 && ((uintptr_t)out_f16 % 16) == 0 &&
                    ((uintptr_t)V16_f16 % 16) == 0 && v16_stride_h % 8 == 0;
  v = VSide{{V2, V4, V8}, {v2_stride_h, v4_stride_h, v8_stride_h}, (const __half *)scale_f16, (const __half *)zp_f16, s_stride_h,
            counts, totals, max_tv, (const uint16_t *)V16_f16, v16_stride_h, (uint16_t *)out_f16, words, {m2, m4, m8}, n16,
            (int)blocks, tag};
  return RDKV_OK;
}

static int launch_unpack(const KSide &k, const VSide &v, const MaskSide &m, bool dense, bool wide, size_t lds, int H_kv, int D,
                         const char *name, void *stream) {
  const int64_t blocks = (int64_t)k.blocks + v.blocks + m.blocks;
  if (blocks == 0) return RDKV_OK;
  RDKV_REQUIRE(blocks <= 0x7fffffffLL, "%s: too many rows", name);
  auto *kernel = dense ? (wide ? unpack_layer_kernel<true, true> : unpack_layer_kernel<true, false>)
                       : (wide ? unpack_layer_kernel<false, true> : unpack_layer_kernel<false, false>);
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks, H_kv, (unsigned)rdkv_cdiv(D, kChan)), dim3(256), lds, (hipStream_t)stream,
                     k, v, m, D);
  RDKV_CHECK_LAUNCH(name);
  return RDKV_OK;
}

static int unpack_layer_k(const uint8_t *K2, int64_t k2_stride_h, int64_t k2_stride_t, const uint8_t *K4,
                          int64_t k4_stride_h, int64_t k4_stride_t, const uint8_t *K8, int64_t k8_stride_h,
                          int64_t k8_stride_t, const void *scale_f16, const void *zp_f16, int64_t ks_stride_h,
                          const int64_t *sort_idx, int64_t sort_stride_h, int sort_n, const int32_t *counts, int n2,
                          int n4, int n8, int n2p, int n4p, int n8w, int H_kv, int64_t T, int D, void *out_f16,
                          int32_t *check, uint64_t *words, uint32_t tag, void *stream) {
  KSide k{};
  bool dense = false;
  size_t lds = 0;
  const int rc = k_side(k, dense, lds, K2, k2_stride_h, k2_stride_t, K4, k4_stride_h, k4_stride_t, K8, k8_stride_h, k8_stride_t,
                        scale_f16, zp_f16, ks_stride_h, sort_idx, sort_stride_h, sort_n, counts, n2, n4, n8, n2p, n4p, n8w, H_kv,
                        T, D, out_f16, check, words, tag);
  return rc != RDKV_OK ? rc : launch_unpack(k, VSide{}, MaskSide{}, dense, true, lds, H_kv, D, "rdkv_unpack_layer_k", stream);
}

static int unpack_layer_v(const uint8_t *V2, int64_t v2_stride_h, const uint8_t *V4, int64_t v4_stride_h,
                          const uint8_t *V8, int64_t v8_stride_h, const void *scale_f16, const void *zp_f16,
                          int64_t s_stride_h, const int32_t *counts, int m2, int m4, int m8, int64_t max_tv,
                          const void *V16_f16, int64_t v16_stride_h, int n16, int H_kv, int D, void *out_f16,
                          const int32_t *totals, uint64_t *words, uint32_t tag, void *stream) {
  VSide v{};
  bool wide = false;
  const int rc = v_side(v, wide, V2, v2_stride_h, V4, v4_stride_h, V8, v8_stride_h, scale_f16, zp_f16, s_stride_h, counts, m2,
                        m4, m8, max_tv, V16_f16, v16_stride_h, n16, H_kv, D, out_f16, totals, words, tag);
  return rc != RDKV_OK ? rc : launch_unpack(KSide{}, v, MaskSide{}, true, wide, 0, H_kv, D, "rdkv_unpack_layer_v", stream);
}

RDKV_API int rdkv_unpack_layer(const RdkvDenseLayer *y, void *stream) {
  RDKV_REQUIRE(y && y->k_words && y->v_words && y->totals && y->T > 0 && y->max_tv + (int64_t)y->n16 > 0,
               "rdkv_unpack_layer: no words, no totals or no rows");
  RDKV_REQUIRE(y->mask_rows >= 0 && y->mask_width >= 0 && y->mask_extra >= 0, "rdkv_unpack_layer: bad mask shape");
  const int64_t out_width = y->mask_width + y->mask_extra, n = y->mask ? y->mask_rows * out_width : 0;
  RDKV_REQUIRE(!y->mask || (y->mask_out_f16 && y->mask_rows <= 0x7fffffffLL && out_width <= 0x7fffffffLL && n <= 0x7fffffffLL),
               "rdkv_unpack_layer: no mask output or too large a mask");
  KSide k{};
  VSide v{};
  bool dense = false, wide = false;
  size_t lds = 0;
  int rc = k_side(k, dense, lds, y->K[0], y->k_stride_h[0], y->k_stride_t[0], y->K[1], y->k_stride_h[1], y->k_stride_t[1],
                  y->K[2], y->k_stride_h[2], y->k_stride_t[2], y->k_scale_f16, y->k_zp_f16, y->ks_stride_h, y->sort_idx,
                  y->sort_stride_h, y->sort_n, y->k_counts, y->n[0], y->n[1], y->n[2], y->np[0], y->np[1], y->np[2], y->H_kv,
                  y->T, y->D, y->K_out_f16, nullptr, y->k_words, y->tag);
  if (rc == RDKV_OK)
    rc = v_side(v, wide, y->V[0], y->v_stride_h[0], y->V[1], y->v_stride_h[1], y->V[2], y->v_stride_h[2], y->v_scale_f16,
                y->v_zp_f16, y->vs_stride_h, y->v_counts, y->m[0], y->m[1], y->m[2], y->max_tv, y->V16_f16, y->v16_stride_h,
                y->n16, y->H_kv, y->D, y->V_out_f16, y->totals, y->v_words, y->tag);
  if (rc != RDKV_OK) return rc;
  const MaskSide m{y->mask, (uint16_t *)y->mask_out_f16, (uint32_t)n, (uint32_t)y->mask_width, (uint32_t)out_width,
                   (int)rdkv_cdiv(n, 2048 * (int64_t)y->H_kv)};
  return launch_unpack(k, v, m, dense, wide, lds, y->H_kv, y->D, "rdkv_unpack_layer", stream);
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
