// Decode attention over the reference's padded ("shared-max stripe") tensor layout:
// K scores, masked softmax and the V weighted sum as three separate entry points with
// the call shape of obkv_accel/triton_k_kernel.py:1211 and triton_v_kernel.py:1729, and a
// layer's call in which the softmax is part of the other two (rdkv_attn_scores,
// rdkv_v_weighted_sum_scores).  These keep the reference's semantics for callers that overwrite
// packed tensors in place or pass strided score buffers; the streaming fused kernel is the fast path.
// Arithmetic: K scores of rows stored back to back are exact integer products of the codes with
// q * scale in 46 bits, joined in fp32 at the end; everything else - scores of other rows, softmax,
// V sum - is fp32 operands, products and sums.  Fixed summation order (deterministic).
#include "rdkv_common.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr float kInvSqrtD = 0.08838834764831845f;  // 1/sqrt(128), triton_k_kernel.py:280
constexpr int kD = 128;
constexpr int kGB = 4;  // query heads processed together per pass

__device__ __forceinline__ float load_q(const void *q, int dtype, int64_t idx) {
  if (dtype == RDKV_DTYPE_F32) return reinterpret_cast<const float *>(q)[idx];
  if (dtype == RDKV_DTYPE_F16) return __half2float(reinterpret_cast<const __half *>(q)[idx]);
  const uint32_t b = reinterpret_cast<const uint16_t *>(q)[idx];
  return __uint_as_float(b << 16);
}

// ---------------------------------------------------------------------------
// K scores.  grid = (ceil(T/256), H_kv); one thread per token, kGB heads per pass.
// qs[g][c] = q[hq, perm[c]] * scale[c]; bias[g] = sum_c zp[c]*qs[g][c];
// out = (sum_c code*qs - bias) / sqrt(128)      (triton_k_kernel.py:14-17)
// This kernel reads the rows where they lie, a byte at a time, whatever their strides;
// k_qk_dot_mfma_kernel below is the one for densely stored rows.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_qk_dot_strided_kernel(const void *__restrict__ q, int q_dtype, int64_t q_stride_h, int G,
                const uint8_t *__restrict__ K2, int64_t k2_sh, int64_t k2_st,
                const uint8_t *__restrict__ K4, int64_t k4_sh, int64_t k4_st,
                const uint8_t *__restrict__ K8, int64_t k8_sh, int64_t k8_st,
                const __half *__restrict__ scale, const __half *__restrict__ zp, int64_t ks_sh,
                const int64_t *__restrict__ perm, int64_t perm_sh, int n2p, int n4p, int n8,
                int64_t T, float *__restrict__ out, int64_t out_sh) {
  extern __shared__ float smem[];
  const int Dp = n2p + n4p + n8;
  const int hkv = blockIdx.y;
  float *s_qs = smem;               // [kGB][Dp]
  float *s_bias = smem + kGB * Dp;  // [kGB] (+ reduction scratch)
  const int sub2 = n2p >> 2, sub4 = n4p >> 1;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint8_t *r2 = K2 ? K2 + hkv * k2_sh + t * k2_st : nullptr;
  const uint8_t *r4 = K4 ? K4 + hkv * k4_sh + t * k4_st : nullptr;
  const uint8_t *r8 = K8 ? K8 + hkv * k8_sh + t * k8_st : nullptr;

  for (int g0 = 0; g0 < G; g0 += kGB) {
    __syncthreads();
    if (threadIdx.x < kGB) s_bias[threadIdx.x] = 0.0f;
    __syncthreads();
    for (int i = threadIdx.x; i < kGB * Dp; i += blockDim.x) {
      const int g = i / Dp, c = i - g * Dp;
      float v = 0.0f;
      if (g0 + g < G) {
        const int hq = hkv * G + g0 + g;
        const int64_t ch = perm[(perm_sh ? hq : 0) * perm_sh + c];
        v = load_q(q, q_dtype, hq * q_stride_h + ch) * __half2float(scale[hkv * ks_sh + c]);
      }
      s_qs[i] = v;
    }
    __syncthreads();
    // bias: fixed-order sum by one thread per head (Dp <= ~132 terms)
    if (threadIdx.x < kGB) {
      float b = 0.0f;
      for (int c = 0; c < Dp; ++c) b += __half2float(zp[hkv * ks_sh + c]) * s_qs[threadIdx.x * Dp + c];
      s_bias[threadIdx.x] = b;
    }
    __syncthreads();
    if (t < T) {
      float acc[kGB];
#pragma unroll
      for (int g = 0; g < kGB; ++g) acc[g] = 0.0f;
      for (int j = 0; j < sub2; ++j) {
        const uint32_t b = r2[j];
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          const float cv = (float)((b >> (2 * f)) & 3u);
          const int c = j + f * sub2;
#pragma unroll
          for (int g = 0; g < kGB; ++g) acc[g] += cv * s_qs[g * Dp + c];
        }
      }
      for (int j = 0; j < sub4; ++j) {
        const uint32_t b = r4[j];
        const float lo = (float)(b & 15u), hi = (float)(b >> 4);
        const int c = n2p + j;
#pragma unroll
        for (int g = 0; g < kGB; ++g) acc[g] += lo * s_qs[g * Dp + c] + hi * s_qs[g * Dp + c + sub4];
      }
      for (int j = 0; j < n8; ++j) {
        const float cv = (float)r8[j];
        const int c = n2p + n4p + j;
#pragma unroll
        for (int g = 0; g < kGB; ++g) acc[g] += cv * s_qs[g * Dp + c];
      }
#pragma unroll
      for (int g = 0; g < kGB; ++g)
        if (g0 + g < G) out[(int64_t)(hkv * G + g0 + g) * out_sh + t] = (acc[g] - s_bias[g]) * kInvSqrtD;
    }
  }
}

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef floatx4 __attribute__((aligned(4))) floatx4_a4;   // a 16-byte load from any float
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

typedef int intx4 __attribute__((ext_vector_type(4)));

// The power of two on the codes of a width: all are below 2^7 then (8-bit codes less 128), their q * scale
// of one size, and the shift that cuts the codes out puts it there.
__device__ __forceinline__ int k_code_log(int width) { return width == 2 ? 5 : width == 4 ? 3 : 0; }
// The part of a zero point that is taken off the codes exactly: its nearest integer, kept within -64 .. 319
// times the codes' power of two (the digits' sums stay below 2^31).  The quantizer only produces a width's own
// codes, for which nothing is left over; whatever is left of another value enters as a bias term.
__device__ __forceinline__ float zp_whole(float z, int log) {
  return fminf(fmaxf(rintf(z), (float)(-(64 >> log))), (float)(319 >> log));
}

// Maximum over the wavefront, in every lane, in the vector ALU.
__device__ __forceinline__ float wave_max_alu(float v) {
  v = rdkv_row16_max(v);
  auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  v = fmaxf(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
  auto t = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  return fmaxf(__builtin_bit_cast(float, (unsigned)t[0]), __builtin_bit_cast(float, (unsigned)t[1]));
}

// Sum over the 16 lanes of a row, in every lane.
__device__ __forceinline__ float row16_sum(float v) {
  v += rdkv_dpp_mov<0x128>(v);
  v += rdkv_dpp_mov<0x124>(v);
  v += rdkv_dpp_mov<0x122>(v);
  return v + rdkv_dpp_mov<0x121>(v);
}

// Softmax of a row in pieces: a piece's maximum m and its sum l of exp(x - m).  Where all of a piece is -inf,
// exp(x - 0) keeps the sum at 0 (NaN: NaN); the weights themselves are exp(x - m) / l with the row's own m.
__device__ __forceinline__ float softmax_at(float m) { return m == -INFINITY ? 0.0f : m; }
__device__ __forceinline__ void softmax_rebase(float m, float &l, float to) { l *= __expf(m - softmax_at(to)); }

// A barrier for what went through LDS, without waiting for loads in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Sixteen bytes of LDS as words.  (Read as a vector, which may be anything, the compiler waits for every load into LDS
// that is in flight, which the next tile's rows are: a call of 8 KV heads x 128k, low-bit 53.8 us, now 53.1.)
__device__ __forceinline__ intx4 lds_row(const int8_t *p) {
  const uint32_t *w = reinterpret_cast<const uint32_t *>(p);
  return intx4{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
}

// Blocks of the int8 products: 64 channels each, at most two per width (2 | 4 | 8 bit: blocks 0, 1 | 2, 3 | 4, 5).
constexpr int kKBlocks = 6;

// Where channel j of a row of `sub` bytes and plane p (bit field p of its byte) enters: block, byte of the
// block's 64.  A lane group (lane / 16) of a block holds sixteen codes a token: one dword of four 2-bit
// planes, two dwords of two 4-bit planes or four dwords, plane by plane.
__device__ __forceinline__ int k_slot(int width, int p, int j) {
  const int dj = j >> 2, b = j & 3;
  if (width == 2) return (dj >> 2) * 64 + (dj & 3) * 16 + 4 * p + b;
  if (width == 4) return (2 + (dj >> 3)) * 64 + ((dj >> 1) & 3) * 16 + 4 * ((dj & 1) * 2 + p) + b;
  return (4 + (dj >> 4)) * 64 + ((dj >> 2) & 3) * 16 + 4 * (dj & 3) + b;
}

// K scores for rows stored back to back (token stride = row bytes), query heads g0 .. g0 + 4 NG of every
// KV head.  A workgroup walks 256-token tiles of one KV head (tile = blockIdx.x, + gridDim.x, ...).  The rows
// of a tile are one contiguous run per width, copied to LDS in aligned 16-byte pieces by loads that go there
// directly, the next tile's under the current one's arithmetic.  The products run on
// v_mfma_i32_16x16x64_i8 and are exact: the columns are sixteen tokens, whose bytes are cut from LDS, shifted
// and masked, nothing more (8-bit codes less 128); the rows are the four upper base-256 digits of q * scale of
// four query heads, as integers of 30 bits after a power of two per head that brings its largest just under
// 2^30, and a second product's rows are the two digits below those (heads of both groups in one): 46 bits, so a
// channel keeps all 24 of its fp32 product down to 2^-22 of the head's largest.  (One extreme token widens its
// channel's scale; all others lie at that channel's zero, and their scores come from channels 2^-10 of it and
// less.  64 channels of 8 bit, one with a token 512 / 4096 / 30000 times as large and a query 8 times: error of
// the others' scores 4.3e-8 / 4.7e-8 / 4.9e-8; with 30 bits alone 1.4e-7 / 1.4e-6 / 1.0e-5, with fp16 pairs in
// fp32 sums 6.9e-8 / 7.0e-8 / 9.3e-8.  The second product is always formed: a test of how many channels need it
// has heads on its wrong side, 47 of 64 extreme ones for instance.)
// The codes of the narrow widths enter times 2^5 and 2^3, so that every width's q * scale has a like part of
// those bits.  The sums start from minus the zero points' part, formed by the same
// products, so they are sums of the signed values themselves; a lane ends up with the six digits' sums of one
// token and head and joins them in fp32, one rounding and one of the factor 1 / sqrt(128).  Error against 64
// bits: 4.0e-8 of the scores in the 2-norm (fp16 pairs in fp32 sums: 4.1e-8 .. 5.2e-8).
// What bounds it: the chain of the set-up (tables and query, digits, first tile) and the padded rows' loads; at 128k
// the vector instructions (nine tenths of the cycles).  With v_mfma_f32_4x4x4_16b_f16 over code - zp as fp16 (7 vector
// instructions and three table reads from LDS per four codes, here 2 and none, and rows through registers, with 40
// scalar instructions and 5 branches a piece) the scores alone of 8 KV heads x 1.5k / 32k / 128k (low-bit) took 8.8 /
// 18.6 / 32.5 us, now 7.3 / 13.4 / 17.9 (with 30 bits 6.9 / 12.5 / 16.7); eight query heads per KV head, 32k 21.9, now
// 17.3 (15.8), 100k 44.5, now 30.7 (28.9).
// The reference layout pads every head's segments to the widest head's: channels whose stored scale is zero
// contribute exactly nothing, blocks past a head's last such channel are skipped.
// CPT = channels per thread (Dp <= 256 CPT).
// STATS: the launch also forms the scores of the appended keys (its first st.new_groups workgroups of a KV head),
// adds the mask, and every workgroup leaves its part of a row's softmax, maximum and sum, as a pair, so no
// launch reads the rows again for them (13.1 us at 32k, two launches of 11.7 at 128k).  With it this launch takes 8.1
// us at 1.5k, 15.5 at 32k, 20.6 at 128k, with eight query heads per KV head 20.9 at 32k and 41.8 at 100k (same run as
// above).  Error of the weights against 64 bits 5.1e-8 .. 6.4e-8 in the 2-norm (a launch of their own: 6.4e-8 .. 1.2e-7).
// Dynamic LDS: KSetup, then one or two tiles of 16-byte pieces, each with 128 bytes that reads past the
// last row may touch.
template <int NG>
struct KSetup {
  alignas(16) int8_t digit[kKBlocks][NG][16][64];   // [block][head group][head, digit][code]
  alignas(16) int8_t low[kKBlocks][4][2 * NG][64];  // [block][head][head group, lower digit][code]
  alignas(16) int8_t zero[kKBlocks][2][64];         // zero points: low and high digit of base 128
  float q[4 * NG][kD];
  float big[4][4 * NG], rest[4][4 * NG];            // by wavefront: largest |q * scale| of a head, its bias
  float last[4][4];                                 // by wavefront: last channel of a width that counts
};

// What a STATS launch takes besides: the additive mask (or null), the appended keys, fp32 rows of 16-byte
// alignment, `per_group` of them a workgroup, and where the pairs go, [H_q][gridDim.x].
struct KStats {
  const float *mask;
  int64_t mask_sh;
  const float *k_new;
  int64_t kn_sh, kn_st, n_new;
  int new_groups, per_group;
  float2 *pairs;
};

constexpr int kKNewKeys = 64;      // appended keys of a pass of a workgroup: two for each eight lanes
constexpr int kKNewGroups = 128;   // workgroups of a KV head that take appended keys, at most
constexpr int kKMaxPairs = 1024 + kKNewGroups;   // what a row's softmax comes in, at most
constexpr int kKMaxSub2 = 32, kKMaxSub4 = 64, kKMaxSub8 = 128;   // bytes of a row by width: two blocks each

constexpr int kKMaxLds = 160 * 1024;   // LDS of a compute unit, and of a workgroup at most
// Workgroups per compute unit (wavefronts per SIMD) the kernel is compiled for.  Eight heads' digits take 72
// registers; with four wavefronts they are read from LDS for every tile: 8 KV heads x 100k 42.3 us, now 31.6 (with the
// softmax 50.3 / 42.4), 128k of 128 4-bit channels 40.2 / 30.2.
constexpr int k_resident(int ng) { return ng == 1 ? 4 : 3; }

// 16-byte pieces of a tile of 256 rows of `sub` bytes that may start and end anywhere in a piece.
constexpr int k_tile_pieces(int sub) { return sub ? (256 * sub + 30) / 16 : 0; }
constexpr int k_tile_lds(int sub2, int sub4, int sub8) {
  return 16 * (k_tile_pieces(sub2) + k_tile_pieces(sub4) + k_tile_pieces(sub8)) + 128;
}
static_assert(sizeof(KSetup<2>) + 2 * k_tile_lds(kKMaxSub2, kKMaxSub4, kKMaxSub8) <= kKMaxLds, "two tiles of any row fit");

// One pair per query head of a workgroup from its wavefronts' (su.big: maxima, su.rest: sums).
template <int NG>
__device__ __forceinline__ void k_write_pairs(const KSetup<NG> &su, int tl, int heads, int64_t first, const KStats &st) {
  lds_barrier();
  if (tl < heads) {
    const float m = fmaxf(fmaxf(su.big[0][tl], su.big[1][tl]), fmaxf(su.big[2][tl], su.big[3][tl]));
    float l = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      float lw = su.rest[w][tl];
      softmax_rebase(su.big[w][tl], lw, m);
      l += lw;
    }
    st.pairs[(first + tl) * gridDim.x + blockIdx.x] = make_float2(m, l);
  }
}

// scores[t] = sum_d (q[d] / sqrt(128)) k[t][d] for the workgroup's appended keys and NHD query heads: eight
// lanes per key (sixteen channels each, 16-byte loads), two keys per lane group in flight; lane kc of the
// eight keeps head kc.  The same products and sums as new_zone_scores below.
template <int NG>
__device__ __forceinline__ void k_new_keys(KSetup<NG> &su, const float (&qrow)[2 * NG], int G, int g0, int64_t T,
                                           float *__restrict__ out, int64_t out_sh, const KStats &st) {
  constexpr int NHD = 4 * NG;
  const int tl = threadIdx.x, lane = tl & 63, wave = tl >> 6, tg = lane >> 3, kc = lane & 7, hkv = blockIdx.y;
#pragma unroll
  for (int u = 0; u < 2 * NG; ++u) (&su.q[0][0])[tl + 256 * u] = qrow[u] * kInvSqrtD;
  lds_barrier();
  const float *kh = st.k_new + hkv * st.kn_sh;
  const int64_t a = (int64_t)blockIdx.x * st.per_group, b = min(a + st.per_group, st.n_new);
  const bool mine = kc < NHD && g0 + kc < G;
  float *dst = out + (int64_t)(hkv * G + g0 + kc) * out_sh + T;
  float m = -INFINITY, l = 0.0f;
  for (int64_t t0 = a + wave * 8 + tg; t0 < b; t0 += kKNewKeys) {
    floatx4 kr[2][4];
    const bool two = t0 + 32 < b;
    const int64_t t1 = two ? t0 + 32 : t0;
#pragma unroll
    for (int j = 0; j < 4; ++j) kr[0][j] = reinterpret_cast<const floatx4 *>(kh + t0 * st.kn_st)[8 * j + kc];
#pragma unroll
    for (int j = 0; j < 4; ++j) kr[1][j] = reinterpret_cast<const floatx4 *>(kh + t1 * st.kn_st)[8 * j + kc];
    float own[2] = {0.0f, 0.0f};
#pragma unroll 1
    for (int g = 0; g < NHD; ++g) {
      floatx4 qv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) qv[j] = *reinterpret_cast<const floatx4 *>(&su.q[g][32 * j + 4 * kc]);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          p[j] = fmaf(kr[u][j].w, qv[j].w, fmaf(kr[u][j].z, qv[j].z, fmaf(kr[u][j].y, qv[j].y, kr[u][j].x * qv[j].x)));
        float v = (p[0] + p[1]) + (p[2] + p[3]);
        v += rdkv_dpp_mov<0xB1>(v);          // quad_perm [1,0,3,2]
        v += rdkv_dpp_mov<0x4E>(v);          // quad_perm [2,3,0,1]
        v += rdkv_dpp_mov<0x141>(v);         // row_half_mirror: the other quad of the eight lanes
        own[u] = kc == g ? v : own[u];
      }
    }
    if (!two) own[1] = -INFINITY;
    const float to = fmaxf(m, fmaxf(own[0], own[1]));
    softmax_rebase(m, l, to);
    m = to;
    l += __expf(own[0] - softmax_at(m)) + (two ? __expf(own[1] - softmax_at(m)) : 0.0f);
    if (mine) {
      dst[t0] = own[0];
      if (two) dst[t1] = own[1];
    }
  }
  // the lanes of a head: kc + 8 k
  float M = fmaxf(m, rdkv_dpp_mov<0x128>(m));
  M = fmaxf(M, __shfl_xor(M, 16, 64));
  M = fmaxf(M, __shfl_xor(M, 32, 64));
  softmax_rebase(m, l, M);
  l += rdkv_dpp_mov<0x128>(l);
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (lane < NHD) {
    su.big[wave][lane] = M;
    su.rest[wave][lane] = l;
  }
  k_write_pairs<NG>(su, tl, min(NHD, G - g0), (int64_t)hkv * G + g0, st);
}

template <int NG, int CPT, bool STATS>
__global__ void __launch_bounds__(256, k_resident(NG))
k_qk_dot_mfma_kernel(const void *__restrict__ q, int q_dtype, int64_t q_stride_h, int G, int g0,
                     const uint8_t *__restrict__ K2, int64_t k2_sh, const uint8_t *__restrict__ K4,
                     int64_t k4_sh, const uint8_t *__restrict__ K8, int64_t k8_sh,
                     const __half *__restrict__ scale, const __half *__restrict__ zp, int64_t ks_sh,
                     const int64_t *__restrict__ perm, int64_t perm_sh, int n2p, int n4p, int n8,
                     int64_t T, float *__restrict__ out, int64_t out_sh, int tile_lds, KStats st) {
  extern __shared__ __align__(16) float smem[];
  constexpr int NHD = 4 * NG;
  constexpr bool kMaskAhead = NG == 1;
  const int Dp = n2p + n4p + n8;
  const int hkv = blockIdx.y;
  const int sub2 = n2p >> 2, sub4 = n4p >> 1;
  KSetup<NG> &su = *reinterpret_cast<KSetup<NG> *>(smem);
  constexpr int rows_off = (int)sizeof(KSetup<NG>);
  uint8_t *rows = reinterpret_cast<uint8_t *>(smem) + rows_off;
  const int tl = threadIdx.x, lane = tl & 63, wave = __builtin_amdgcn_readfirstlane(tl >> 6);
  const __half *sc_h = scale + hkv * ks_sh, *zp_h = zp + hkv * ks_sh;
  const int ntiles = (int)((T + 255) >> 8);
  const int rowb[3] = {sub2, sub4, n8};
  const uint32_t *lds32 = reinterpret_cast<const uint32_t *>(smem);

  // The three row runs of a tile as 16-byte pieces, one run behind the other in LDS: address of a run's first
  // piece, where its rows start in it, pieces.  (An aligned piece that holds a byte of a row is mapped.)
  struct Run { uint64_t at; int skew, n; };
  auto run_of = [&](int tile, int sgm) __attribute__((always_inline)) {
    const int64_t t0 = (int64_t)tile * 256;
    const int ntok = T - t0 < 256 ? (int)(T - t0) : 256;
    const uint8_t *base = sgm == 0 ? K2 + hkv * k2_sh : sgm == 1 ? K4 + hkv * k4_sh : K8 + hkv * k8_sh;
    const uint64_t g = (uint64_t)(uintptr_t)(base + t0 * rowb[sgm]);
    Run r;
    r.skew = (int)(g & 15);
    r.at = g - r.skew;
    r.n = rowb[sgm] ? (r.skew + ntok * rowb[sgm] + 15) >> 4 : 0;
    return r;
  };
  auto issue_rows = [&](int tile, int buffer) __attribute__((always_inline)) {
    const Run r0 = run_of(tile, 0), r1 = run_of(tile, 1), r2 = run_of(tile, 2);
    const int f1 = r0.n, f2 = f1 + r1.n, all = f2 + r2.n;
    const uint64_t b1 = r1.at - 16 * (int64_t)f1, b2 = r2.at - 16 * (int64_t)f2;
    uint8_t *to = rows + buffer * tile_lds + wave * 1024;
    for (int k = 0; k < all; k += 256) {
      const int piece = k + tl;
      const uint64_t from = (piece < f1 ? r0.at : piece < f2 ? b1 : b2) + 16 * (uint64_t)(uint32_t)piece;
      if (piece < all)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)from,
                                         (__attribute__((address_space(3))) void *)(to + 16 * k), 16, 0, 0);
    }
  };

  // ---- set-up: channel tables and query rows (no load waits for another), then the first tile's rows ---------
  const int walkers = STATS ? gridDim.x - st.new_groups : gridDim.x;    // workgroups that walk the tiles
  int tile = STATS ? (int)blockIdx.x - st.new_groups : blockIdx.x;
  int ch[CPT][NHD];
  float scv[CPT], zpv[CPT], qrow[2 * NG];
  floatx4 mask_next[NG];
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    const int c = min(tl + 256 * u, Dp - 1);
    scv[u] = __half2float(sc_h[c]);
    zpv[u] = __half2float(zp_h[c]);
#pragma unroll
    for (int g = 0; g < NHD; ++g) {
      const int hq = hkv * G + min(g0 + g, G - 1);
      ch[u][g] = (int)perm[(perm_sh ? hq : 0) * perm_sh + c] & (kD - 1);
    }
  }
  auto q_loads = [&](auto elem) __attribute__((always_inline)) {   // one straight run of loads per query type
#pragma unroll
    for (int u = 0; u < 2 * NG; ++u) {
      const int i = tl + 256 * u;
      qrow[u] = elem((int64_t)(hkv * G + min(g0 + (i >> 7), G - 1)) * q_stride_h + (i & 127));
    }
  };
  if (q_dtype == RDKV_DTYPE_F32)
    q_loads([&](int64_t i) { return reinterpret_cast<const float *>(q)[i]; });
  else if (q_dtype == RDKV_DTYPE_F16)
    q_loads([&](int64_t i) { return __half2float(reinterpret_cast<const __half *>(q)[i]); });
  else
    q_loads([&](int64_t i) { return __uint_as_float((uint32_t)reinterpret_cast<const uint16_t *>(q)[i] << 16); });
  if (STATS && (int)blockIdx.x < st.new_groups) {
    k_new_keys<NG>(su, qrow, G, g0, T, out, out_sh, st);
    return;
  }
  const int r = lane & 15, grp = lane >> 4;
  // the mask values of a lane's four tokens and NG heads
  auto load_mask = [&](int tile) __attribute__((always_inline)) {
    const int64_t t = (int64_t)tile * 256 + wave * 64 + r;
#pragma unroll
    for (int hg = 0; hg < NG; ++hg) mask_next[hg] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (!st.mask) return;
#pragma unroll
    for (int hg = 0; hg < NG; ++hg) {
      const float *row = st.mask + (int64_t)(hkv * G + min(g0 + 4 * hg + grp, G - 1)) * st.mask_sh;
#pragma unroll
      for (int i = 0; i < 4; ++i) mask_next[hg][i] = row[min(t + 16 * i, T - 1)];
    }
  };
  float m_run[NG], l_run[NG];
#pragma unroll
  for (int hg = 0; hg < NG; ++hg) {
    m_run[hg] = -INFINITY;
    l_run[hg] = 0.0f;
  }
  for (int i = tl; i < (int)(sizeof(su.digit) + sizeof(su.low) + sizeof(su.zero)) / 16; i += 256)
    reinterpret_cast<u32x4 *>(smem)[i] = u32x4{0, 0, 0, 0};
#pragma unroll
  for (int u = 0; u < 2 * NG; ++u) (&su.q[0][0])[tl + 256 * u] = qrow[u];
  // (behind the wait for the small loads: loads return in order, and theirs would wait for the rows)
  if (STATS && kMaskAhead) load_mask(tile);
  issue_rows(tile, 0);
  lds_barrier();
  float qv[CPT][NHD];
#pragma unroll
  for (int u = 0; u < CPT; ++u)
#pragma unroll
    for (int g = 0; g < NHD; ++g) qv[u][g] = su.q[g][ch[u][g]];
  float mloc[NHD], bias[NHD];
  float last[3] = {0.0f, 0.0f, 0.0f};   // channels of a segment up to the last one with a nonzero scale
  bool rest = false;
#pragma unroll
  for (int g = 0; g < NHD; ++g) mloc[g] = bias[g] = 0.0f;
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    const int c = tl + 256 * u;
    const bool counts = c < Dp && scv[u] != 0.0f;
    const int log = k_code_log(c < n2p ? 2 : c < n2p + n4p ? 4 : 8);
    const float left = counts ? zpv[u] - zp_whole(zpv[u], log) : 0.0f;
    rest |= left != 0.0f;
#pragma unroll
    for (int g = 0; g < NHD; ++g) {
      qv[u][g] = counts && g0 + g < G ? qv[u][g] * scv[u] : 0.0f;
      mloc[g] = fmaxf(mloc[g], fabsf(qv[u][g]) <= 3.0e38f ? ldexpf(fabsf(qv[u][g]), -log) : INFINITY);   // (NaN too)
      bias[g] += left * qv[u][g];
    }
    if (counts) {
      if (c < n2p) last[0] = fmaxf(last[0], (float)(c + 1));
      else if (c < n2p + n4p) last[1] = fmaxf(last[1], (float)(c - n2p + 1));
      else last[2] = fmaxf(last[2], (float)(c - n2p - n4p + 1));
    }
  }
#pragma unroll
  for (int g = 0; g < NHD; ++g) mloc[g] = wave_max_alu(mloc[g]);
#pragma unroll
  for (int i = 0; i < 3; ++i) last[i] = wave_max_alu(last[i]);
  if (__builtin_amdgcn_ballot_w64(rest) != 0) {   // (normally nothing is left of the zero points)
#pragma unroll
    for (int g = 0; g < NHD; ++g) bias[g] = rdkv_wave_sum(bias[g]);
  }
  if (lane == 0) {
#pragma unroll
    for (int g = 0; g < NHD; ++g) {
      su.big[wave][g] = mloc[g];
      su.rest[wave][g] = bias[g];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) su.last[wave][i] = last[i];
  }
  lds_barrier();
  // the digits of q * scale, and of the zero points (8-bit codes come less 128, so theirs do too)
  int ex[NHD];   // big = m * 2^x with 0.5 <= m < 1  ->  30 - x
#pragma unroll
  for (int g = 0; g < NHD; ++g) {
    const float big = fmaxf(fmaxf(su.big[0][g], su.big[1][g]), fmaxf(su.big[2][g], su.big[3][g]));
    ex[g] = 30 - ((int)(__float_as_uint(big) >> 23) - 126);
  }
#pragma unroll
  for (int u = 0; u < CPT; ++u) {
    const int c = tl + 256 * u;
    if (c < Dp) {
      const int width = c < n2p ? 2 : c < n2p + n4p ? 4 : 8, sub = width == 2 ? sub2 : width == 4 ? sub4 : n8;
      const int cc = c - (width == 2 ? 0 : width == 4 ? n2p : n2p + n4p);
      const int p = cc / sub, slot = k_slot(width, p, cc - p * sub), blk = slot >> 6, at = slot & 63;
      const int log = k_code_log(width), z = (int)zp_whole(zpv[u], log) * (1 << log) - (width == 8 ? 128 : 0), zlo = ((z + 64) & 127) - 64;
      su.zero[blk][0][at] = (int8_t)zlo;
      su.zero[blk][1][at] = (int8_t)((z - zlo) >> 7);
#pragma unroll
      for (int g = 0; g < NHD; ++g) {
        // the nearest integer and sixteen bits of what it leaves (exact), within what two digits reach
        const float v = ldexpf(qv[u][g], ex[g] - log), whole = rintf(v);
        const int rest16 = (int)rintf((v - whole) * 65536.0f), carry = rest16 > 0x7f7f ? 1 : 0;
        const int x = ((int)whole + carry + 0x00808080) ^ 0x00808080, y = (rest16 - (carry << 16) + 0x80) ^ 0x80;
#pragma unroll
        for (int l = 0; l < 4; ++l) su.digit[blk][g >> 2][4 * (g & 3) + l][at] = (int8_t)(x >> (8 * l));
#pragma unroll
        for (int l = 0; l < 2; ++l) su.low[blk][g & 3][2 * (g >> 2) + l][at] = (int8_t)(y >> (8 * l));
      }
    }
  }
  // blocks that any channel of this head needs
  float ext[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) ext[i] = fmaxf(fmaxf(su.last[0][i], su.last[1][i]), fmaxf(su.last[2][i], su.last[3][i]));
  const int e2 = __builtin_amdgcn_readfirstlane((int)ext[0]), e4 = __builtin_amdgcn_readfirstlane((int)ext[1]),
            e8 = __builtin_amdgcn_readfirstlane((int)ext[2]);
  const int blocks[3] = {(min(e2, sub2) + 15) >> 4, (min(e4, sub4) + 31) >> 5, (e8 + 63) >> 6};
  lds_barrier();
  constexpr bool kLowHeld = !STATS;      // (no registers for them beside the softmax: from LDS for every tile)
  intx4 dig[kKBlocks][NG], low[kLowHeld ? kKBlocks : 1], start[NG], start_low{0, 0, 0, 0};
  auto low_from_lds = [&](int b) __attribute__((always_inline)) {
    return lds_row(&su.low[b][r >> 2][r & (2 * NG - 1)][16 * grp]);
  };
#pragma unroll
  for (int hg = 0; hg < NG; ++hg) start[hg] = intx4{0, 0, 0, 0};
#pragma unroll
  for (int b = 0; b < kKBlocks; ++b) {
    if ((b & 1) < blocks[b >> 1]) {
      intx4 z = lds_row(&su.zero[b][r & 1][16 * grp]);
      if (r > 1) z = intx4{0, 0, 0, 0};
      const intx4 lower = low_from_lds(b);
      if (kLowHeld) low[kLowHeld ? b : 0] = lower;
      start_low = __builtin_amdgcn_mfma_i32_16x16x64_i8(lower, z, start_low, 0, 0, 0);
#pragma unroll
      for (int hg = 0; hg < NG; ++hg) {
        dig[b][hg] = lds_row(&su.digit[b][hg][r][16 * grp]);
        start[hg] = __builtin_amdgcn_mfma_i32_16x16x64_i8(dig[b][hg], z, start[hg], 0, 0, 0);
      }
    }
  }
  // minus the zero points' part, from its two digits' columns
  auto minus_zero = [&](intx4 v) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = -(__shfl(v[i], 16 * grp, 64) + 128 * __shfl(v[i], 16 * grp + 1, 64));
    return v;
  };
  start_low = minus_zero(start_low);
  float half_up[NG], factor[NG], offset[NG];    // of this lane's head, lane / 16 of the group: 2^-e in two parts
  constexpr bool kParked = STATS && NG > 1;     // (eight heads and their softmax: no registers for these)
  floatx4 *parked = reinterpret_cast<floatx4 *>(su.q);   // (the query is done with) by head: the sums' start, then these
  if (kParked && wave == 0 && r == 0) reinterpret_cast<intx4 *>(parked)[8 * NG + grp] = start_low;
#pragma unroll
  for (int hg = 0; hg < NG; ++hg) {
    start[hg] = minus_zero(start[hg]);
    const int g = 4 * hg + grp;
    const float big = fmaxf(fmaxf(su.big[0][g], su.big[1][g]), fmaxf(su.big[2][g], su.big[3][g]));
    const int e = 30 - ((int)(__float_as_uint(big) >> 23) - 126);
    half_up[hg] = ldexpf(1.0f, -(e >> 1));
    factor[hg] = big <= 3.0e38f ? ldexpf(kInvSqrtD, (e >> 1) - e) : __builtin_nanf("");
    offset[hg] = -((su.rest[0][g] + su.rest[1][g]) + (su.rest[2][g] + su.rest[3][g])) * kInvSqrtD;
    if (kParked && wave == 0 && r == 0) {
      reinterpret_cast<intx4 *>(parked)[8 * hg + grp] = start[hg];
      parked[8 * hg + 4 + grp] = floatx4{half_up[hg], factor[hg], offset[hg], 0.f};
    }
  }

  // ---- tiles: a wavefront's 64 tokens are four products of sixteen, lane r of product j token r + 16 j ------
  // (Sixteen lanes then read rows that lie one row apart.  Four apart, with one 16-byte store a lane for its four
  // tokens, rows of whole 32 or 64 bytes put them on two or four LDS banks: the scores of 8 KV heads x 128k, 96
  // 8-bit channels, 48.6 us, now 26.3; 64 of 8 and 64 of 4 bit 40.4 / 28.0; 128 of 4 bit 36.8 / 26.1.)
  for (int buffer = 0;; buffer ^= 1) {
    __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0): this wavefront's pieces are in LDS
    __syncthreads();                         // all are; and every wavefront has done with the other buffer
    const int next = tile + walkers;
    const bool more = next < ntiles;
    floatx4 mask[NG];
    if (STATS) {      // (ahead of the next rows: loads return in order; a tile ahead where there are registers)
      if (!kMaskAhead) load_mask(tile);
#pragma unroll
      for (int hg = 0; hg < NG; ++hg) mask[hg] = mask_next[hg];
      if (kMaskAhead && more) load_mask(next);
    }
    if (more) issue_rows(next, buffer ^ 1);
    const int64_t t0 = (int64_t)tile * 256;
    const int ntok = T - t0 < 256 ? (int)(T - t0) : 256;
    const int tok = wave * 64 + r;
    intx4 acc[4][NG], acc_low[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc_low[j] = kParked ? reinterpret_cast<const intx4 *>(parked)[8 * NG + grp] : start_low;
#pragma unroll
      for (int hg = 0; hg < NG; ++hg) acc[j][hg] = kParked ? reinterpret_cast<const intx4 *>(parked)[8 * hg + grp] : start[hg];
    }
    {
      const Run r0 = run_of(tile, 0), r1 = run_of(tile, 1), r2 = run_of(tile, 2);
      const int begin = rows_off + buffer * tile_lds;
      const int base[3] = {begin + r0.skew + tok * sub2 + 4 * grp, begin + 16 * r0.n + r1.skew + tok * sub4 + 8 * grp,
                           begin + 16 * (r0.n + r1.n) + r2.skew + tok * n8 + 16 * grp};
#pragma unroll
      for (int b = 0; b < kKBlocks; ++b) {
        if ((b & 1) < blocks[b >> 1]) {
          const int w = b >> 1, nd = 1 << w;       // dwords a lane takes of a row
          const intx4 lower = kLowHeld ? low[kLowHeld ? b : 0] : low_from_lds(b);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int off = base[w] + 16 * j * rowb[w] + (b & 1) * 16 * nd;
            const uint32_t *W = lds32 + (off >> 2);
            const uint32_t sh = (uint32_t)off & 3u;
            uint32_t raw[5], d[4];
#pragma unroll
            for (int i = 0; i <= nd; ++i) raw[i] = W[i];
#pragma unroll
            for (int i = 0; i < nd; ++i) d[i] = __builtin_amdgcn_alignbyte(raw[i + 1], raw[i], sh);
            intx4 codes;
            if (w == 0)
              codes = intx4{(int)((d[0] << 5) & 0x60606060u), (int)((d[0] << 3) & 0x60606060u),
                            (int)((d[0] << 1) & 0x60606060u), (int)((d[0] >> 1) & 0x60606060u)};
            else if (w == 1)
              codes = intx4{(int)((d[0] << 3) & 0x78787878u), (int)((d[0] >> 1) & 0x78787878u),
                            (int)((d[1] << 3) & 0x78787878u), (int)((d[1] >> 1) & 0x78787878u)};
            else
              codes = intx4{(int)(d[0] ^ 0x80808080u), (int)(d[1] ^ 0x80808080u), (int)(d[2] ^ 0x80808080u),
                            (int)(d[3] ^ 0x80808080u)};
#pragma unroll
            for (int hg = 0; hg < NG; ++hg)
              acc[j][hg] = __builtin_amdgcn_mfma_i32_16x16x64_i8(dig[b][hg], codes, acc[j][hg], 0, 0, 0);
            acc_low[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(lower, codes, acc_low[j], 0, 0, 0);
          }
        }
      }
    }
#pragma unroll
    for (int hg = 0; hg < NG; ++hg) {
      const int g = g0 + 4 * hg + grp;
      if (g < G && tok < ntok) {
        floatx4 v, join{half_up[hg], factor[hg], offset[hg], 0.f};
        if (kParked) join = parked[8 * hg + 4 + grp];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const intx4 x = acc[j][hg];
          // (the upper two digits' sum as an fp32 number and what it leaves: one rounding that counts)
          const float x3 = (float)x[3], x2 = (float)x[2], head = fmaf(x3, 256.0f, x2), left = fmaf(x3, 256.0f, -head) + x2;
          const float tail = fmaf((float)acc_low[j][2 * hg + 1], 256.0f, (float)acc_low[j][2 * hg]);
          const float sum = fmaf(head, 65536.0f, fmaf(left, 65536.0f, fmaf((float)x[1], 256.0f, fmaf(tail, 0x1p-16f, (float)x[0]))));
          v[j] = fmaf(sum * join[0], join[1], join[2]);
          if (STATS) v[j] += mask[hg][j];
        }
        if (STATS) {
          float to = m_run[hg];
#pragma unroll
          for (int j = 0; j < 4; ++j) to = tok + 16 * j < ntok ? fmaxf(to, v[j]) : to;
          softmax_rebase(m_run[hg], l_run[hg], to);
          m_run[hg] = to;
#pragma unroll
          for (int j = 0; j < 4; ++j) l_run[hg] += tok + 16 * j < ntok ? __expf(v[j] - softmax_at(to)) : 0.0f;
        }
        float *dst = out + (int64_t)(hkv * G + g) * out_sh + t0 + tok;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (tok + 16 * i < ntok) dst[16 * i] = v[i];
      }
    }
    if (!more) break;
    tile = next;
  }
  if (STATS) {
#pragma unroll
    for (int hg = 0; hg < NG; ++hg) {
      const float m = rdkv_row16_max(m_run[hg]);
      softmax_rebase(m_run[hg], l_run[hg], m);
      const float l = row16_sum(l_run[hg]);
      if (r == 0) {
        su.big[wave][4 * hg + grp] = m;
        su.rest[wave][4 * hg + grp] = l;
      }
    }
    k_write_pairs<NG>(su, tl, min(NHD, G - g0), (int64_t)hkv * G + g0, st);
  }
}

// Compute units of the current device, asked once per device (0 = not asked yet; a race between
// two first calls stores the same number twice).
int compute_units() {
  static int cu_of_device[64];
  int dev = 0, n_cu = 256;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64) {
    if (cu_of_device[dev] == 0) {
      int v = 0;
      if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
        cu_of_device[dev] = v;
    }
    if (cu_of_device[dev] > 0) n_cu = cu_of_device[dev];
  }
  return n_cu;
}

__global__ void zero_rows_kernel(float *out, int64_t out_sh, int64_t T) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < T) out[blockIdx.y * out_sh + t] = 0.0f;
}

// ---------------------------------------------------------------------------
// softmax over [scores_old + mask | scores_new], one block per query head.
// ---------------------------------------------------------------------------
// Keys of the new zone, for a launch that forms their scores itself (k == nullptr: the scores are
// given): k fp32 [H_kv, n_new, 128], rows 16-byte aligned; q as rdkv_k_qk_dot takes it.
struct NewKeys {
  const void *q;
  int64_t q_sh;
  int q_dtype, G;
  const float *k;
  int64_t k_sh, k_st;
};

// scores[t] = sum_d (q[d] / sqrt(128)) k[t][d] for the keys a .. b of query head h, by the whole workgroup:
// eight lanes per key (sixteen channels each, 16-byte loads), two keys per lane group in flight.
// The caller's barrier makes them visible.  (As launches of their own - the scaled query, a library
// product, the copy into the score rows - these few hundred dot products and the weighted values took
// 24 us of a 76 us layer and four of its ten launches; 32k layer 102 -> 51 us, 128k 115.5 -> 97.)
__device__ __forceinline__ void new_zone_scores(const NewKeys &nk, int h, int64_t a, int64_t b, float *scores) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int tg = lane >> 3, kc = lane & 7;
  const float *kh = nk.k + (int64_t)(h / nk.G) * nk.k_sh;
  if (a + wave * 8 >= b) return;
  float qv[16];
  auto q_loads = [&](auto elem) __attribute__((always_inline)) {   // one straight run of loads per query type
#pragma unroll
    for (int i = 0; i < 16; ++i) qv[i] = elem(h * nk.q_sh + 32 * (i >> 2) + 4 * kc + (i & 3)) * kInvSqrtD;
  };
  if (nk.q_dtype == RDKV_DTYPE_F32)
    q_loads([&](int64_t i) { return reinterpret_cast<const float *>(nk.q)[i]; });
  else if (nk.q_dtype == RDKV_DTYPE_F16)
    q_loads([&](int64_t i) { return __half2float(reinterpret_cast<const __half *>(nk.q)[i]); });
  else
    q_loads([&](int64_t i) { return __uint_as_float((uint32_t)reinterpret_cast<const uint16_t *>(nk.q)[i] << 16); });
  for (int64_t t0 = a + wave * 8 + tg; t0 < b; t0 += 16 * nw) {
    floatx4 kr[2][4];
    const int64_t t1 = t0 + 8 * nw < b ? t0 + 8 * nw : t0;
#pragma unroll
    for (int j = 0; j < 4; ++j) kr[0][j] = reinterpret_cast<const floatx4 *>(kh + t0 * nk.k_st)[8 * j + kc];
#pragma unroll
    for (int j = 0; j < 4; ++j) kr[1][j] = reinterpret_cast<const floatx4 *>(kh + t1 * nk.k_st)[8 * j + kc];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float p[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        p[j] = fmaf(kr[u][j].w, qv[4 * j + 3], fmaf(kr[u][j].z, qv[4 * j + 2], fmaf(kr[u][j].y, qv[4 * j + 1], kr[u][j].x * qv[4 * j])));
      float v = (p[0] + p[1]) + (p[2] + p[3]);
      v += rdkv_dpp_mov<0xB1>(v);          // quad_perm [1,0,3,2]
      v += rdkv_dpp_mov<0x4E>(v);          // quad_perm [2,3,0,1]
      v += rdkv_dpp_mov<0x141>(v);         // row_half_mirror: the other quad of the eight lanes
      if (kc == 0) scores[u ? t1 : t0] = v;   // (t1 == t0 writes its score again)
    }
  }
}

// The same as a launch of its own, kNewPerBlock keys of a head per workgroup (a pass of its wavefronts).
// grid = (8, G, H_kv * eighths of the pieces): the G heads that read a piece are eight apart in launch order,
// on one die, whose L2 serves the repeats.
constexpr int kNewPerBlock = 256;
constexpr int64_t kNewOwnLaunch = 1024;
__global__ void __launch_bounds__(1024)
new_zone_scores_kernel(NewKeys nk, int64_t n_new, int eighths, float *__restrict__ scores, int64_t stride_h) {
  const int kv = blockIdx.z / eighths, h = kv * nk.G + blockIdx.y;
  const int64_t a = ((int64_t)(blockIdx.z - kv * eighths) * 8 + blockIdx.x) * kNewPerBlock;
  const int64_t b = a + kNewPerBlock < n_new ? a + kNewPerBlock : n_new;
  new_zone_scores(nk, h, a, b, scores + h * stride_h);
}

__device__ float block_reduce(float v, bool is_max, float *scratch) {
  v = is_max ? rdkv_wave_max(v) : rdkv_wave_sum(v);
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) scratch[w] = v;
  __syncthreads();
  float r = scratch[0];
  for (int i = 1; i < nw; ++i) r = is_max ? fmaxf(r, scratch[i]) : r + scratch[i];
  return r;
}

__global__ void __launch_bounds__(1024)
softmax_rows_kernel(const float *__restrict__ so, int64_t so_sh, const float *__restrict__ mask,
                    int64_t mask_sh, int64_t T_old, const float *sn, int64_t sn_sh,
                    int64_t n_new, float *__restrict__ wo, int64_t wo_sh, float *wn,
                    int64_t wn_sh, NewKeys nk) {
  __shared__ float scratch[16];
  const int h = blockIdx.x;
  const float *a = so ? so + h * so_sh : nullptr;
  const float *m = mask ? mask + h * mask_sh : nullptr;
  const float *b = sn ? sn + h * sn_sh : nullptr;
  if (nk.k) {
    new_zone_scores(nk, h, 0, n_new, wn + h * wn_sh);
    __syncthreads();
  }
  float mx = -INFINITY;
  for (int64_t t = threadIdx.x; t < T_old; t += blockDim.x) mx = fmaxf(mx, a[t] + (m ? m[t] : 0.0f));
  for (int64_t t = threadIdx.x; t < n_new; t += blockDim.x) mx = fmaxf(mx, b[t]);
  mx = block_reduce(mx, true, scratch);
  float sum = 0.0f;
  for (int64_t t = threadIdx.x; t < T_old; t += blockDim.x) sum += __expf(a[t] + (m ? m[t] : 0.0f) - mx);
  for (int64_t t = threadIdx.x; t < n_new; t += blockDim.x) sum += __expf(b[t] - mx);
  sum = block_reduce(sum, false, scratch);
  const float inv = 1.0f / sum;
  for (int64_t t = threadIdx.x; t < T_old; t += blockDim.x)
    wo[h * wo_sh + t] = __expf(a[t] + (m ? m[t] : 0.0f) - mx) * inv;
  for (int64_t t = threadIdx.x; t < n_new; t += blockDim.x) wn[h * wn_sh + t] = __expf(b[t] - mx) * inv;
}

// The same softmax for rows whose zone A+B part can be read and written 16 bytes at a time (bases
// and row strides 16-byte aligned): a thread keeps its share of the row in registers (NV float4:
// rows of up to 4096 * NV scores are read once and written once; mask added on the way in), or
// (NV = 0, longer rows) streams the row three times with 16-byte accesses.  In place is fine: a
// thread only ever rewrites elements it has read itself.  The mask rows are as long as the layer has
// keys, any number, so they start at any float; they too are read 16 bytes at a time (the load only
// needs dword alignment; a variant per alignment took the same time).
template <int NV>
__global__ void __launch_bounds__(1024)
softmax_rows_vec_kernel(const float *__restrict__ so, int64_t so_sh, const float *__restrict__ mask,
                        int64_t mask_sh, int64_t T_old, const float *sn, int64_t sn_sh,
                        int64_t n_new, float *wo, int64_t wo_sh, float *wn, int64_t wn_sh, NewKeys nk) {
  __shared__ float scratch[16];
  const int h = blockIdx.x, tid = threadIdx.x;
  const float *a = so + h * so_sh;
  const float *m = mask ? mask + h * mask_sh : nullptr;
  const float *b = sn ? sn + h * sn_sh : nullptr;
  const float4 *a4 = reinterpret_cast<const float4 *>(a);
  const floatx4_a4 *m4 = reinterpret_cast<const floatx4_a4 *>(m);
  float4 *w4 = reinterpret_cast<float4 *>(wo + h * wo_sh);
  const int64_t n4 = T_old >> 2;
  constexpr int kKeep = NV > 0 ? NV : 1;
  float4 x[kKeep];
  auto load4 = [&](int64_t i) {
    float4 v = a4[i];
    if (m) {
      const floatx4 k = m4[i];
      v.x += k.x; v.y += k.y; v.z += k.z; v.w += k.w;
    }
    return v;
  };
  float mx = -INFINITY;
  if (NV > 8 && nk.k) new_zone_scores(nk, h, 0, n_new, wn + h * wn_sh);   // (no registers for both)
  if (NV > 0) {
#pragma unroll
    for (int k = 0; k < kKeep; ++k) {
      const int64_t i = tid + (int64_t)k * 1024;
      x[k] = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
      if (i < n4) x[k] = a4[i];
    }
    if (NV <= 8 && nk.k) new_zone_scores(nk, h, 0, n_new, wn + h * wn_sh);   // (behind the row's requests)
    if (m && n4 > 0) {
      // The mask values of eight float4s are requested together and none of the loads is conditional
      // (a slot past the row reads the row's first float4 and drops it): with the load inside the
      // range check the compiler waits for each one before it issues the next, sixteen round trips
      // one after the other, which was most of this kernel's time.
      constexpr int kB = kKeep < 8 ? kKeep : 8;
#pragma unroll
      for (int k0 = 0; k0 < kKeep; k0 += kB) {
        floatx4 mk[kB];
#pragma unroll
        for (int j = 0; j < kB; ++j) {
          const int64_t i = tid + (int64_t)(k0 + j) * 1024;
          mk[j] = m4[i < n4 ? i : 0];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kB; ++j) {
          const int64_t i = tid + (int64_t)(k0 + j) * 1024;
          if (i < n4) {
            x[k0 + j].x += mk[j].x; x[k0 + j].y += mk[j].y; x[k0 + j].z += mk[j].z; x[k0 + j].w += mk[j].w;
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kKeep; ++k) mx = fmaxf(fmaxf(mx, fmaxf(x[k].x, x[k].y)), fmaxf(x[k].z, x[k].w));
  } else {
    if (nk.k) new_zone_scores(nk, h, 0, n_new, wn + h * wn_sh);
    for (int64_t i = tid; i < n4; i += 1024) {
      const float4 v = load4(i);
      mx = fmaxf(fmaxf(mx, fmaxf(v.x, v.y)), fmaxf(v.z, v.w));
    }
  }
  if (nk.k) __syncthreads();
  // the last T_old % 4 scores and the new zone, element by element
  for (int64_t t = 4 * n4 + tid; t < T_old; t += 1024) mx = fmaxf(mx, a[t] + (m ? m[t] : 0.0f));
  for (int64_t t = tid; t < n_new; t += 1024) mx = fmaxf(mx, b[t]);
  mx = block_reduce(mx, true, scratch);
  float sum = 0.0f;
  if (NV > 0) {
#pragma unroll
    for (int k = 0; k < kKeep; ++k) {   // (slots past the row hold -inf: their weight is 0)
      x[k].x = __expf(x[k].x - mx); x[k].y = __expf(x[k].y - mx);
      x[k].z = __expf(x[k].z - mx); x[k].w = __expf(x[k].w - mx);
      sum += (x[k].x + x[k].y) + (x[k].z + x[k].w);
    }
  } else {
    for (int64_t i = tid; i < n4; i += 1024) {
      const float4 v = load4(i);
      sum += (__expf(v.x - mx) + __expf(v.y - mx)) + (__expf(v.z - mx) + __expf(v.w - mx));
    }
  }
  for (int64_t t = 4 * n4 + tid; t < T_old; t += 1024) sum += __expf(a[t] + (m ? m[t] : 0.0f) - mx);
  for (int64_t t = tid; t < n_new; t += 1024) sum += __expf(b[t] - mx);
  sum = block_reduce(sum, false, scratch);
  const float inv = 1.0f / sum;
  // tail first: in place, its inputs must be read before anything of the row is rewritten by
  // this thread (other threads never touch these elements)
  for (int64_t t = 4 * n4 + tid; t < T_old; t += 1024)
    wo[h * wo_sh + t] = __expf(a[t] + (m ? m[t] : 0.0f) - mx) * inv;
  if (NV > 0) {
#pragma unroll
    for (int k = 0; k < kKeep; ++k) {
      const int64_t i = tid + (int64_t)k * 1024;
      if (i < n4) w4[i] = make_float4(x[k].x * inv, x[k].y * inv, x[k].z * inv, x[k].w * inv);
    }
  } else {
    for (int64_t i = tid; i < n4; i += 1024) {
      const float4 v = load4(i);
      w4[i] = make_float4(__expf(v.x - mx) * inv, __expf(v.y - mx) * inv, __expf(v.z - mx) * inv,
                          __expf(v.w - mx) * inv);
    }
  }
  for (int64_t t = tid; t < n_new; t += 1024) wn[h * wn_sh + t] = __expf(b[t] - mx) * inv;
}

// The same softmax with a row cut into S pieces of whole float4s, one workgroup each, for long rows
// of few heads (one workgroup per head leaves most compute units idle): the first launch leaves
// every piece's maximum and its sum of exp(x - maximum) in the workspace, the second combines
// the S pairs of its row in index order (every workgroup the same arithmetic) and writes the
// weights of its piece.  A piece is at most 4096 float4s, held in registers within a launch, and its
// share of the new zone; the last piece also takes the last T_old % 4 scores.  Same alignment conditions as
// softmax_rows_vec_kernel; in place is fine for the same reason.
constexpr int kSoftmaxMaxSplit = 32;
constexpr int kSoftmaxPieceVec = 4;      // float4s per thread and piece
constexpr int64_t kSoftmaxSplitMinRow = 65537;   // up to 64k scores a row is read once by one workgroup: 12.4 us at 38k against 14.7 split

template <bool WRITE>
__global__ void __launch_bounds__(1024)
softmax_rows_split_kernel(const float *__restrict__ so, int64_t so_sh, const float *__restrict__ mask,
                          int64_t mask_sh, int64_t T_old, const float *sn, int64_t sn_sh,
                          int64_t n_new, float *wo, int64_t wo_sh, float *wn, int64_t wn_sh, float *ws, NewKeys nk) {
  __shared__ float scratch[16];
  const int h = blockIdx.y, c = blockIdx.x, S = gridDim.x, tid = threadIdx.x;
  const float *a = so + h * so_sh;
  const float *m = mask ? mask + h * mask_sh : nullptr;
  const float *b = sn ? sn + h * sn_sh : nullptr;
  const float4 *a4 = reinterpret_cast<const float4 *>(a);
  const floatx4_a4 *m4 = reinterpret_cast<const floatx4_a4 *>(m);
  const int64_t n4 = T_old >> 2, per = (n4 + S - 1) / S;
  const int64_t lo = c * per, hi = lo + per < n4 ? lo + per : n4;
  const bool last = c == S - 1;
  const int64_t n_per = (n_new + S - 1) / S, n_lo = c * n_per < n_new ? c * n_per : n_new,
                n_hi = n_lo + n_per < n_new ? n_lo + n_per : n_new;
  float4 x[kSoftmaxPieceVec];
#pragma unroll
  for (int k = 0; k < kSoftmaxPieceVec; ++k) {
    const int64_t i = lo + tid + (int64_t)k * 1024;
    x[k] = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
    if (i < hi) x[k] = a4[i];
  }
  if (!WRITE && nk.k) {
    new_zone_scores(nk, h, n_lo, n_hi, wn + h * wn_sh);
    __syncthreads();
  }
  if (m && lo < hi) {
    // (all mask loads of the piece requested together, none conditional: see softmax_rows_vec_kernel)
    floatx4 mk[kSoftmaxPieceVec];
#pragma unroll
    for (int k = 0; k < kSoftmaxPieceVec; ++k) {
      const int64_t i = lo + tid + (int64_t)k * 1024;
      const int64_t ic = i < hi ? i : lo;
      mk[k] = m4[ic];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < kSoftmaxPieceVec; ++k) {
      const int64_t i = lo + tid + (int64_t)k * 1024;
      if (i < hi) {
        x[k].x += mk[k].x; x[k].y += mk[k].y; x[k].z += mk[k].z; x[k].w += mk[k].w;
      }
    }
  }
  float *pair = ws + ((int64_t)h * S) * 2;
  if (!WRITE) {
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < kSoftmaxPieceVec; ++k) mx = fmaxf(fmaxf(mx, fmaxf(x[k].x, x[k].y)), fmaxf(x[k].z, x[k].w));
    if (last)
      for (int64_t t = 4 * n4 + tid; t < T_old; t += 1024) mx = fmaxf(mx, a[t] + (m ? m[t] : 0.0f));
    for (int64_t t = n_lo + tid; t < n_hi; t += 1024) mx = fmaxf(mx, b[t]);
    mx = block_reduce(mx, true, scratch);
    float sum = 0.0f;
    if (mx > -INFINITY) {        // (a piece that is masked out entirely adds nothing)
#pragma unroll
      for (int k = 0; k < kSoftmaxPieceVec; ++k)
        sum += (__expf(x[k].x - mx) + __expf(x[k].y - mx)) + (__expf(x[k].z - mx) + __expf(x[k].w - mx));
      if (last)
        for (int64_t t = 4 * n4 + tid; t < T_old; t += 1024) sum += __expf(a[t] + (m ? m[t] : 0.0f) - mx);
      for (int64_t t = n_lo + tid; t < n_hi; t += 1024) sum += __expf(b[t] - mx);
    }
    sum = block_reduce(sum, false, scratch);
    if (tid == 0) {
      pair[2 * c] = mx;
      pair[2 * c + 1] = sum;
    }
  } else {
    float mx = -INFINITY;
    for (int i = 0; i < S; ++i) mx = fmaxf(mx, pair[2 * i]);
    float sum = 0.0f;
    for (int i = 0; i < S; ++i) {
      const float mi = pair[2 * i];
      if (mi > -INFINITY) sum += pair[2 * i + 1] * __expf(mi - mx);
    }
    const float inv = 1.0f / sum;
    if (last) {   // tail first: read before this thread rewrites anything of the row
      for (int64_t t = 4 * n4 + tid; t < T_old; t += 1024)
        wo[h * wo_sh + t] = __expf(a[t] + (m ? m[t] : 0.0f) - mx) * inv;
    }
    float4 *w4 = reinterpret_cast<float4 *>(wo + h * wo_sh);
#pragma unroll
    for (int k = 0; k < kSoftmaxPieceVec; ++k) {
      const int64_t i = lo + tid + (int64_t)k * 1024;
      if (i < hi)
        w4[i] = make_float4(__expf(x[k].x - mx) * inv, __expf(x[k].y - mx) * inv, __expf(x[k].z - mx) * inv,
                            __expf(x[k].w - mx) * inv);
    }
    for (int64_t t = n_lo + tid; t < n_hi; t += 1024) wn[h * wn_sh + t] = __expf(b[t] - mx) * inv;
  }
}

// ---------------------------------------------------------------------------
// V weighted sum.  grid = (kVChunks, H_kv, quads of query heads), block = 4 wavefronts.
// A step is 64 consecutive tokens of a quantized class of the head (2 | 4 | 8 bit) or 32 of the fp16 zone B;
// the wavefronts of a head take its steps in turn, the next step's loads in flight under a step's arithmetic.
// Eight lanes share four tokens: lane li owns channels 16 li .. + 15 in every class (in a 2- or 4-bit row
// these are one field of sixteen bytes), 16 bytes of each token per load (fp16: two).
// The sums run on v_mfma_f32_4x4x1_16b_f32 (16 blocks of 4 heads x 1 token x 4 channels), which rounds as a
// multiply-add does: the weight (times the token's scale) is the fp32 number itself, a value the code less the
// middle of its width's range (exact; smaller sums that cancel), the zero point's part of it a sum beside; fp16
// rows as they are.
// (Weights as an fp16 pair on v_mfma_f32_4x4x4_16b_f16, four tokens an instruction, are 22 or 23 bits and nothing
// below 2^-36 of the largest: an fp16 row with a weight near 1 and values near 0 - an attention sink - left the others
// 2.7e-7, here 1.1e-7.  With a third term, 24 bits, the error still grows with the number of tokens: that
// instruction cuts off, towards minus infinity, whatever lies below 24 bits of its largest product, 5e-7 over 16000
// 2-bit tokens of like weight, here 1.4e-7.)
// Error against 64 bits over random layers of 1k .. 128k tokens: a layer's call 2.2e-7 .. 5.9e-7 of the result in the
// 2-norm, the sum alone 0.9e-7 .. 2.0e-7; with fp16 pairs 2.1e-7 .. 6.1e-7 and 1.0e-7 .. 2.7e-7, on the vector ALU with
// uncentred codes 2.4e-7 .. 9.5e-7 and 0.9e-7 .. 1.6e-6.
// What bounds it: set-up and the latency of a few steps per wavefront at 32k, at 128k the vector instructions (63 % of
// the cycles) and the products (24 %), which overlap only between the two wavefronts of a SIMD.  Us with its
// reduction of 8 KV heads x 1.5k / 32k / 128k (low-bit): on the vector ALU (a conversion and a multiply-add per head and
// code) 12.9 / 22.5 / 39.7, with fp16 pairs 11.9 / 19.7 / 29.9, now 13.9 / 20.1 / 34.3; eight query heads per KV head, 32k
// 28.6 / 29.5 / 30.4 (two workgroups of four heads, eight apart in the launch, so that a die's L2 serves the second; one
// workgroup for all eight had no registers for a step in flight).
// Weights and values that are not finite stay in their head and channel, as in plain arithmetic.
// ---------------------------------------------------------------------------
constexpr int kVChunks = 64;
constexpr int kVWaves = 4;
constexpr int kVParts = kVChunks * kVWaves;   // wavefronts that share a head's steps
constexpr int kVNew = 8;                      // appended tokens a wavefront takes at a time
constexpr int v_step_tokens(int cls) { return cls == 3 ? 32 : 64; }   // tokens of a step: 128 bytes of codes a lane

typedef floatx4 __attribute__((aligned(4))) floatx4_w;
typedef unsigned long long __attribute__((aligned(2))) u64_a2;   // four fp16 values from any element

// What a lane holds of a step: quantized rows raw[4 a + k] of tokens t0 + 32 a + 4 sub + k, fp16 rows
// raw[2 k], raw[2 k + 1] of tokens t0 + 4 sub + k; weights of head lane % 4, scales, zero points.
// Where the four tokens of an a pass the end of the class, w, s and z start up to three columns early (v_tail).
struct VTile {
  uint4 raw[8];
  floatx4 w[2];
  unsigned long long s[2], z[2];
};

// A class of the head's tokens: its rows, how many, the column of the first in the weight (and scale) rows.
struct VClass {
  const uint8_t *codes;
  int n;
  int64_t col;
};

__device__ __forceinline__ int v_lane_offset(int cls, int li) { return cls == 3 ? 32 * li : 16 * (li & ((2 << cls) - 1)); }

// The loads of a step of any class, without a branch on the class or on the end of its tokens (a load in
// a branch of its own is waited for there): rows past the end are the last row again, columns are held
// back to the last four (the first four of the row, if these are not there; the caller sees to it that they are).
__device__ __forceinline__ void v_load(int cls, const VClass c, const uint16_t *sc, const uint16_t *zz, int t0,
                                       const float *wrow, int sub, int li, VTile &L) {
  // Bases are the wavefront's, offsets from them 32 bits a lane: 64-bit addresses by lane were 31 of the step's 480
  // vector instructions.  (The sum at 128k low-bit, with 85 % of its cycles in vector instructions: 25.9 -> 25.0 us.)
  const int row_log = 5 + cls, last = c.n - 1 - t0;
  const bool wide = cls == 3;
  const uint8_t *base = c.codes + ((int64_t)t0 << row_log);
  const uint32_t lane_off = (uint32_t)v_lane_offset(cls, li), lane_odd = lane_off + (wide ? 16 : 0);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int row = min(4 * sub + (wide ? j >> 1 : 32 * (j >> 2) + (j & 3)), last);
    const uint32_t at = ((uint32_t)row << row_log) + (wide && (j & 1) ? lane_odd : lane_off);
    L.raw[j] = *reinterpret_cast<const uint4 *>(base + at);
  }
  const int lo = c.col < 4 ? (int)c.col : 4;       // (columns may be held back to before the class's first)
  const float *wb = wrow + (c.col - lo);
  // (fp16 rows have no scales: bytes of the rows themselves, not looked at)
  const uint16_t *sb = wide ? reinterpret_cast<const uint16_t *>(c.codes) : sc + (c.col - lo);
  const uint16_t *zb = wide ? reinterpret_cast<const uint16_t *>(c.codes) : zz + (c.col - lo);
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const uint32_t rel = (uint32_t)max(min(t0 + 4 * sub + 32 * a + lo, c.n - 4 + lo), 0);
    L.w[a] = *reinterpret_cast<const floatx4_w *>(wb + rel);
    L.s[a] = *reinterpret_cast<const u64_a2 *>(sb + rel);
    L.z[a] = *reinterpret_cast<const u64_a2 *>(zb + rel);
  }
}

// The last step of a class: what was read early moves to its place, weights (fp16 rows: values too) past the end become 0.
template <bool WIDE>
__device__ __forceinline__ void v_tail(const VClass c, int t0, int sub, VTile &L) {
#pragma unroll
  for (int a = 0; a < (WIDE ? 1 : 2); ++a) {
    const int t = t0 + 4 * sub + 32 * a;
    int64_t col = c.col + (t < c.n - 4 ? t : c.n - 4);
    col = col > 0 ? col : 0;
    const int64_t early = c.col + t - col;
    const int d = early < 4 ? (int)early : 4;
    if (!WIDE) {
      L.s[a] = d < 4 ? L.s[a] >> (16 * d) : 0;
      L.z[a] = d < 4 ? L.z[a] >> (16 * d) : 0;
    }
    floatx4 w = L.w[a];
#pragma unroll
    for (int r = 1; r <= 3; ++r)
      if (d >= r) w = floatx4{w[1], w[2], w[3], w[3]};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      L.w[a][k] = t + k < c.n ? w[k] : 0.0f;
      if (WIDE && t + k >= c.n) L.raw[2 * k] = L.raw[2 * k + 1] = make_uint4(0u, 0u, 0u, 0u);   // (0 times infinity is not 0)
    }
  }
}

// Sums of a wavefront: acc[c][i] is channel 16 li + c of head i over the lane's tokens; zacc, of the lane's own head
// lane % 4, the sum of weight * scale * (zero point - middle code).
struct VSums {
  floatx4 acc[16];
  float zacc;
};

// A step's products, token t of `tokens` by `convert(t, weight, values)`: a token's values are formed under the products
// of the token before, eight vector instructions to four products (a value that a product waits for costs it two idle
// cycles and more, at two wavefronts per SIMD; 2, 4, 16 and 30 instructions at a time, or left to the compiler, the sum
// of 8 KV heads x 128k low-bit takes 0.6 .. 3.8 us more).
template <int TOKENS, class Convert>
__device__ __forceinline__ void v_products(VSums &S, Convert convert) {
  float ws[2], v[2][16];
  convert(0, ws[0], v[0]);
#pragma unroll
  for (int t = 0; t < TOKENS; ++t) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 16; ++c) S.acc[c] = __builtin_amdgcn_mfma_f32_4x4x1f32(ws[t & 1], v[t & 1][c], S.acc[c], 0, 0, 0);
    if (t + 1 < TOKENS) {
      convert(t + 1, ws[(t + 1) & 1], v[(t + 1) & 1]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);      // vector instructions
        __builtin_amdgcn_sched_group_barrier(0x8, 4, 0);      // matrix instructions
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
}

template <int I>
__device__ __forceinline__ float v_quad_lane(float v) { return rdkv_dpp_mov<0x55 * I>(v); }
__device__ __forceinline__ float v_quad_value(float v, int i) {   // (i is a constant after unrolling)
  return i == 0 ? v_quad_lane<0>(v) : i == 1 ? v_quad_lane<1>(v) : i == 2 ? v_quad_lane<2>(v) : v_quad_lane<3>(v);
}

// The widths share one body (shift and mask at run time): a body each made a small call wait for their
// instructions (1.5k tokens: 11.9 us of V, not 9.5).
__device__ __forceinline__ void v_step(const VTile &L, int cls, int li, VSums &S) {
  // a code's field goes to the top of its byte, top bit flipped, and half of the field's unit under it: as a signed
  // byte the code less the middle of its range, times 2^6, 2^4 or 1, which the weights carry the other way
  const int shift = cls == 0 ? 6 - 2 * (li >> 1) : cls == 1 ? 4 - 4 * (li >> 2) : 0;
  const uint32_t mask = cls == 0 ? 0xC0C0C0C0u : cls == 1 ? 0xF0F0F0F0u : 0xFFFFFFFFu;
  const uint32_t flip = cls == 0 ? 0xA0A0A0A0u : cls == 1 ? 0x88888888u : 0x80808080u;
  const float mid = cls == 0 ? 1.5f : cls == 1 ? 7.5f : 128.0f, down = cls == 0 ? 0x1p-6f : cls == 1 ? 0x1p-4f : 1.0f;
  v_products<8>(S, [&](int t, float &ws, float (&v)[16]) __attribute__((always_inline)) {
    const uint4 r = L.raw[t];
    const int a = t >> 2, k = t & 3;
    ws = L.w[a][k] * rdkv_h2f((uint16_t)(L.s[a] >> (16 * k)));
    S.zacc = fmaf(ws, rdkv_h2f((uint16_t)(L.z[a] >> (16 * k))) - mid, S.zacc);
    ws *= down;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t f = (((q == 0 ? r.x : q == 1 ? r.y : q == 2 ? r.z : r.w) << shift) & mask) ^ flip;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * q + j] = (float)(int8_t)(f >> (8 * j));
    }
  });
}

// A step of fp16 rows.
__device__ __forceinline__ void v_step_wide(const VTile &L, VSums &S) {
  v_products<4>(S, [&](int t, float &ws, float (&v)[16]) __attribute__((always_inline)) {
    ws = L.w[0][t];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const uint4 r = L.raw[2 * t + (q >> 2)];
      const uint32_t d = (q & 3) == 0 ? r.x : (q & 3) == 1 ? r.y : (q & 3) == 2 ? r.z : r.w;
      v[2 * q] = rdkv_h2f((uint16_t)d);
      v[2 * q + 1] = rdkv_h2f((uint16_t)(d >> 16));
    }
  });
}

// The weight of a score; weights that are given are {0, 1, false}.
struct VWeights {
  float m, inv;
  bool scores;
  __device__ __forceinline__ float operator()(float s) const { return scores ? __expf(s - m) * inv : s; }
};

// What a launch over scores takes: their softmax in pairs, [H_q][n_pairs] (k_qk_dot_mfma_kernel), and where
// a head's {maximum, 1 / sum} goes for the launch that turns the scores themselves into weights.
struct VScores {
  const float2 *pairs;
  int n_pairs;
  float2 *rows;
};

// {maximum, 1 / sum} of query head lane % 4 of the workgroup's four, by the whole workgroup: a head's pairs on
// 64 lanes, up to four of them requested at once.
__device__ __forceinline__ VWeights v_row_softmax(const VScores vs, int first, int ng, float2 (&scratch)[kVWaves][4]) {
  const int tl = threadIdx.x, h = tl & 3, lane = tl & 63;
  const float2 *p = vs.pairs + (int64_t)(first + min(h, ng - 1)) * vs.n_pairs;
  float m = -INFINITY, l = 0.0f;
  for (int i0 = tl >> 2; i0 < vs.n_pairs; i0 += 256) {
    float2 x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = p[min(i0 + 64 * u, vs.n_pairs - 1)];
#pragma unroll
    for (int u = 1; u < 4; ++u)
      if (i0 + 64 * u >= vs.n_pairs) x[u] = make_float2(-INFINITY, 0.0f);
    const float to = fmaxf(fmaxf(fmaxf(x[0].x, x[1].x), fmaxf(x[2].x, x[3].x)), m);
    softmax_rebase(m, l, to);
    m = to;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      softmax_rebase(x[u].x, x[u].y, to);
      l += x[u].y;
    }
  }
  float M = fmaxf(m, rdkv_dpp_mov<0x124>(m));      // the lanes of a head: h + 4 k
  M = fmaxf(M, rdkv_dpp_mov<0x128>(M));
  M = fmaxf(M, __shfl_xor(M, 16, 64));
  M = fmaxf(M, __shfl_xor(M, 32, 64));
  softmax_rebase(m, l, M);
  l += rdkv_dpp_mov<0x124>(l);
  l += rdkv_dpp_mov<0x128>(l);
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (lane < 4) scratch[tl >> 6][lane] = make_float2(M, l);
  lds_barrier();
  float2 y[kVWaves];
#pragma unroll
  for (int w = 0; w < kVWaves; ++w) y[w] = scratch[w][h];
  m = fmaxf(fmaxf(y[0].x, y[1].x), fmaxf(y[2].x, y[3].x));
  l = 0.0f;
#pragma unroll
  for (int w = 0; w < kVWaves; ++w) {
    softmax_rebase(y[w].x, y[w].y, m);
    l += y[w].y;
  }
  return VWeights{m, 1.0f / l, true};
}

// The steps part, part + kVParts, ... of a class and one query head (its weight row w) in plain fp32
// arithmetic: a token a lane group.
__device__ __forceinline__ void v_plain_class(int cls, const VClass c, const uint16_t *sc, const uint16_t *zz, const float *w,
                                              int before, int part, int sub, int li, float (&acc)[16], float &zacc,
                                              const VWeights of) {
  const int shift = cls == 0 ? 2 * (li >> 1) : cls == 1 ? 4 * (li >> 2) : 0, ntok = v_step_tokens(cls);
  const uint32_t mask = cls == 0 ? 3u : cls == 1 ? 15u : 255u;
#pragma unroll 1
  for (int s = (part - before % kVParts + kVParts) % kVParts; (int64_t)s * ntok < c.n; s += kVParts)
#pragma unroll 1
    for (int t = s * ntok + sub; t < min(s * ntok + ntok, c.n); t += 8) {
      const uint8_t *p = c.codes + v_lane_offset(cls, li) + ((int64_t)t << (5 + cls));
      float ws = of(w[c.col + t]);
      if (cls != 3) {
        ws *= rdkv_h2f(sc[c.col + t]);
        zacc += ws * rdkv_h2f(zz[c.col + t]);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float v = cls == 3 ? rdkv_h2f(reinterpret_cast<const uint16_t *>(p)[i]) : (float)((p[i] >> shift) & mask);
        acc[i] += ws * v;
      }
    }
}

// The fp32 value rows of the new zone (v == nullptr: none) and their weights.
struct NewValues {
  const float *v, *w;
  int64_t v_sh, v_st, w_sh;
  int64_t n;
};

// The two values a lane keeps of two sums over lanes l and l ^ 32 (l ^ 16): lanes of the lower half (of even
// rows) the first, the others the second, in the vector ALU.
__device__ __forceinline__ float fold32(float a, float b) {
  auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
__device__ __forceinline__ float fold16(float a, float b) {
  auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}

template <bool SCORES>
__global__ void __launch_bounds__(64 * kVWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
v_weighted_sum_kernel(const float *__restrict__ w, int64_t w_sh, int G,
                      const uint8_t *__restrict__ V2, int64_t v2_sh, const uint8_t *__restrict__ V4,
                      int64_t v4_sh, const uint8_t *__restrict__ V8, int64_t v8_sh,
                      const uint16_t *__restrict__ scale, const uint16_t *__restrict__ zp, int64_t vs_sh,
                      const int32_t *__restrict__ seg_bounds, int N2h, int N4h, int N8h,
                      const uint8_t *__restrict__ V16, int64_t v16_sh, const int32_t *__restrict__ n_v16,
                      int64_t max_T_v, NewValues nv, float *__restrict__ partial, int H_q, VScores vs) {
  const int hkv = blockIdx.y, chunk = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = lane >> 3, li = lane & 7;
  int N2 = N2h, N4 = N4h, N8 = N8h;
  if (seg_bounds) {
    N2 = seg_bounds[hkv * 3 + 0];
    N4 = seg_bounds[hkv * 3 + 1];
    N8 = seg_bounds[hkv * 3 + 2];
  }
  const int N16 = (V16 && n_v16) ? n_v16[hkv] : 0;
  const uint16_t *sc = scale + hkv * vs_sh, *zz = zp + hkv * vs_sh;
  const VClass c0{V2 + hkv * v2_sh, V2 ? max(N2, 0) : 0, 0}, c1{V4 + hkv * v4_sh, V4 ? max(N4, 0) : 0, N2},
      c2{V8 + hkv * v8_sh, V8 ? max(N8, 0) : 0, (int64_t)N2 + N4}, c3{V16 + 2 * hkv * v16_sh, max(N16, 0), max_T_v};
  // steps of a class and those before it
  const int e0 = (c0.n + 63) / 64, e1 = e0 + (c1.n + 63) / 64, e2 = e1 + (c2.n + 63) / 64, e3 = e2 + (c3.n + 31) / 32;
  const int part = chunk * kVWaves + wave, g0 = 4 * blockIdx.z, ng = min(G - g0, 4);
  const bool live = (lane & 3) < ng;
  const float *w0 = w + (int64_t)(hkv * G + g0) * w_sh, *wrow = w0 + (live ? lane & 3 : 0) * w_sh;
  __shared__ float s_acc[kVWaves][4][kD];
  VSums S;
  S.zacc = 0.0f;
#pragma unroll
  for (int c = 0; c < 16; ++c) S.acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
  // (weight or scale rows of fewer than four columns: the plain sums below)
  const bool narrow = (e2 > 0 && (int64_t)N2 + N4 + N8 < 4) || (N16 > 0 && max_T_v + N16 < 4);
  const int todo = narrow ? 0 : e3;
  // (assignments: a conditional of two variables is an address the compiler keeps in scratch memory)
  auto class_of = [&](int s, VClass &c, int &before) __attribute__((always_inline)) {
    int cls = 3;
    c = c3;
    before = e2;
    if (s < e2) { c = c2; cls = 2; before = e1; }
    if (s < e1) { c = c1; cls = 1; before = e0; }
    if (s < e0) { c = c0; cls = 0; before = 0; }
    return cls;
  };
  auto load = [&](int s, VTile &L) __attribute__((always_inline)) {
    VClass c;
    int before;
    const int cls = class_of(s, c, before);
    v_load(cls, c, sc, zz, v_step_tokens(cls) * (s - before), wrow, sub, li, L);
  };
  VTile cur, nxt;
  int s = part;
  if (s < todo) load(s, cur);
  VWeights weight{0.0f, 1.0f, false};       // of the lane's own head
  if (SCORES) {
    __shared__ float2 s_row[kVWaves][4];
    weight = v_row_softmax(vs, hkv * G + g0, ng, s_row);
    if (chunk == 0 && (int)threadIdx.x < ng) vs.rows[hkv * G + g0 + threadIdx.x] = make_float2(weight.m, weight.inv);
  }
  auto run = [&](auto wide_c, int end) __attribute__((always_inline)) {
    constexpr bool WIDE = decltype(wide_c)::value;
    while (s < min(todo, end)) {
      load(s + kVParts < todo ? s + kVParts : s, nxt);      // (nothing left: the same step again, from the cache)
      int before;
      VClass c;
      const int cls = class_of(s, c, before), t0 = v_step_tokens(cls) * (s - before);
      if (SCORES) {
#pragma unroll
        for (int a = 0; a < (WIDE ? 1 : 2); ++a)
#pragma unroll
          for (int k = 0; k < 4; ++k) cur.w[a][k] = weight(cur.w[a][k]);
      }
      if (t0 + v_step_tokens(cls) > c.n) v_tail<WIDE>(c, t0, sub, cur);
      if (WIDE) v_step_wide(cur, S);
      else v_step(cur, cls, li, S);
      cur = nxt;
      s += kVParts;
    }
  };
  run(std::false_type{}, e2);
  // (an infinite weight makes NaN of the codes' and the zero points' part together, whatever the middle code is)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float zi = v_quad_value(fmaf(S.zacc, 0.0f, S.zacc), i);
#pragma unroll
    for (int c = 0; c < 16; ++c) S.acc[c][i] -= zi;
  }
  run(std::true_type{}, e3);
  // the new zone, fp32: eight tokens at a time, the last wavefronts first (they have the fewest steps)
  if (nv.v) {
    const float *vh = nv.v + hkv * nv.v_sh + 16 * li, *wh = nv.w + (int64_t)(hkv * G + g0 + (live ? lane & 3 : 0)) * nv.w_sh;
    for (int64_t t0 = (int64_t)kVNew * (kVParts - 1 - part); t0 < nv.n; t0 += (int64_t)kVNew * kVParts) {
      const bool in = t0 + sub < nv.n;
      const int64_t t = in ? t0 + sub : t0;
      floatx4 r[4];
      float wn = weight(wh[t]);
#pragma unroll
      for (int j = 0; j < 4; ++j) r[j] = reinterpret_cast<const floatx4 *>(vh + t * nv.v_st)[j];
      if (!in) {
        wn = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int c = 0; c < 16; ++c) S.acc[c] = __builtin_amdgcn_mfma_f32_4x4x1f32(wn, r[c >> 2][c & 3], S.acc[c], 0, 0, 0);
    }
  }
  // Fold the eight token lanes of the wavefront, halving the channels a lane keeps with every exchange:
  // in the end lane (b5, b4, b3, li) has channels 16 li + 8 b5 + 4 b4 + 2 b3 and the next.  (Folding all
  // sixteen on every lane takes 320 instructions instead of 112.)  Then the wavefronts, in a fixed order.
  const bool b3 = lane & 8;
  const int ch = 16 * li + 8 * (lane >> 5) + 4 * ((lane >> 4) & 1) + 2 * ((lane >> 3) & 1);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a[8], b[4], r[2];
#pragma unroll
    for (int c = 0; c < 8; ++c) a[c] = fold32(S.acc[c][i], S.acc[c + 8][i]);
#pragma unroll
    for (int c = 0; c < 4; ++c) b[c] = fold16(a[c], a[c + 4]);
#pragma unroll
    for (int c = 0; c < 2; ++c) r[c] = (b3 ? b[c + 2] : b[c]) + rdkv_dpp_mov<0x128>(b3 ? b[c] : b[c + 2]);
    *reinterpret_cast<float2 *>(&s_acc[wave][i][ch]) = make_float2(r[0], r[1]);
  }
  if (narrow) {
#pragma unroll 1
    for (int g = 0; g < ng; ++g) {
      float acc[16], zacc = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll 1
      for (int cls = 0; cls < 4; ++cls) {
        const int first = cls == 0 ? 0 : cls == 1 ? e0 : cls == 2 ? e1 : e2, last = cls == 0 ? e0 : cls == 1 ? e1 : cls == 2 ? e2 : e3;
        int before;
        VClass c;
        class_of(first, c, before);
        const VWeights of{__shfl(weight.m, g, 64), __shfl(weight.inv, g, 64), SCORES};
        if (first < last) v_plain_class(cls, c, sc, zz, w0 + g * w_sh, first, part, sub, li, acc, zacc, of);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float v = acc[i] - zacc;
        for (int o = 8; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
        if (sub == 0) s_acc[wave][g][16 * li + i] += v;      // (behind the new zone's sums, same wavefront)
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < ng * kD; i += blockDim.x) {
    const int g = i / kD, d = i % kD;
    float v = s_acc[0][g][d];
#pragma unroll
    for (int wv = 1; wv < kVWaves; ++wv) v += s_acc[wv][g][d];
    partial[((int64_t)chunk * H_q + hkv * G + g0 + g) * kD + d] = v;
  }
}

// Rows of scores that become weights in place, n of them each (s == nullptr: none).
struct ScoreRows {
  float *s;
  int64_t sh, n;
  const float2 *rows;      // {maximum, 1 / sum} by head
};
constexpr int kRowPiece = 8192;      // scores a workgroup turns

// out[hq, d] = sum over chunks in chunk order: eight groups of chunks in parallel, then the groups.  The
// workgroups behind the first H_q turn a piece of a score row each, beside the sums (32 rows of 24k scores: 4.8 us, the sums alone 3.9).
__global__ void __launch_bounds__(1024)
v_reduce_kernel(const float *__restrict__ partial, int H_q, float *__restrict__ out, int64_t out_sh, ScoreRows sr) {
  __shared__ float s_part[8][kD];
  if ((int)blockIdx.x >= H_q) {
    const int h = (blockIdx.x - H_q) % H_q;
    const int64_t a = (int64_t)((blockIdx.x - H_q) / H_q) * kRowPiece, left = sr.n - a;
    float *x = sr.s + h * sr.sh + a;
    const float2 row = sr.rows[h];
    const VWeights weight{row.x, row.y, true};
    if (left >= kRowPiece) {
      floatx4_a4 *x4 = reinterpret_cast<floatx4_a4 *>(x) + threadIdx.x;
      floatx4 v[2] = {x4[0], x4[1024]};
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) v[i][k] = weight(v[i][k]);
      x4[0] = v[0];
      x4[1024] = v[1];
    } else {
      for (int t = threadIdx.x; t < (int)left; t += 1024) x[t] = weight(x[t]);
    }
    return;
  }
  const int hq = blockIdx.x, d = threadIdx.x & 127, grp = threadIdx.x >> 7;
  constexpr int per = kVChunks / 8;
  float s = 0.0f;
#pragma unroll 4
  for (int c = grp * per; c < (grp + 1) * per; ++c) s += partial[((int64_t)c * H_q + hq) * kD + d];
  s_part[grp][d] = s;
  __syncthreads();
  if (grp == 0) {
    float t = s_part[0][d];
#pragma unroll
    for (int g = 1; g < 8; ++g) t += s_part[g][d];
    out[hq * out_sh + d] = t;
  }
}

}  // namespace

// stats (or null): mask and appended keys of a launch that leaves the rows' softmax in pairs; *n_pairs of them a
// row, 0 where the rows are not for the int8 products and the scores of the packed keys are all that was formed.
static int k_scores(const void *q, int q_dtype, int64_t q_stride_h, int H_q, int H_kv, const uint8_t *K2,
                    int64_t k2_stride_h, int64_t k2_stride_t, const uint8_t *K4, int64_t k4_stride_h, int64_t k4_stride_t,
                    const uint8_t *K8, int64_t k8_stride_h, int64_t k8_stride_t, const void *scale_f16, const void *zp_f16,
                    int64_t ks_stride_h, const int64_t *perm, int64_t perm_stride_h, int n2p, int n4p, int n8,
                    int64_t T_eff, float *out, int64_t out_stride_h, KStats *stats, int *n_pairs, void *stream) {
  *n_pairs = 0;
  RDKV_REQUIRE(H_q > 0 && H_kv > 0 && H_q % H_kv == 0, "rdkv_k_qk_dot: H_q=%d not a multiple of H_kv=%d", H_q,
               H_kv);
  RDKV_REQUIRE(H_kv <= 65535, "rdkv_k_qk_dot: H_kv=%d exceeds the launch grid", H_kv);
  RDKV_REQUIRE(q_dtype >= 0 && q_dtype <= 2, "rdkv_k_qk_dot: unknown q dtype %d", q_dtype);
  RDKV_REQUIRE(n2p >= 0 && n4p >= 0 && n8 >= 0 && n2p % 4 == 0 && n4p % 2 == 0,
               "rdkv_k_qk_dot: bad segment sizes (%d,%d,%d)", n2p, n4p, n8);
  RDKV_REQUIRE(T_eff >= 0, "rdkv_k_qk_dot: negative T_eff");
  if (T_eff == 0) return RDKV_OK;
  RDKV_REQUIRE(out, "rdkv_k_qk_dot: null out");
  hipStream_t s = (hipStream_t)stream;
  const int Dp = n2p + n4p + n8;
  const int64_t tblocks = rdkv_cdiv(T_eff, 256);
  RDKV_REQUIRE(tblocks <= 0x7fffffffLL, "rdkv_k_qk_dot: T_eff too large");
  if (Dp == 0) {  // no kept channels: scores are zero (triton_k_kernel.py:1265-1268)
    hipLaunchKernelGGL(zero_rows_kernel, dim3((unsigned)tblocks, H_q), dim3(256), 0, s, out, out_stride_h, T_eff);
    RDKV_CHECK_LAUNCH("rdkv_k_qk_dot(zero)");
    return RDKV_OK;
  }
  RDKV_REQUIRE(q && scale_f16 && zp_f16 && perm, "rdkv_k_qk_dot: null pointer");
  RDKV_REQUIRE((n2p == 0 || K2) && (n4p == 0 || K4) && (n8 == 0 || K8), "rdkv_k_qk_dot: missing K segment");
  RDKV_REQUIRE(Dp <= 1024, "rdkv_k_qk_dot: %d padded channels unsupported", Dp);
  const size_t shmem = (size_t)(kGB * Dp + 2 * kGB) * sizeof(float);
  const int sub2 = n2p / 4, sub4 = n4p / 2;
  const bool dense = (n2p == 0 || k2_stride_t == sub2) && (n4p == 0 || k4_stride_t == sub4) &&
                     (n8 == 0 || k8_stride_t == n8);
  const int G = H_q / H_kv;
  const int ng = G > 4 ? 2 : 1;
  const size_t setup = ng == 2 ? sizeof(KSetup<2>) : sizeof(KSetup<1>);
  const int tile_lds = k_tile_lds(sub2, sub4, n8);
  if (dense && sub2 <= kKMaxSub2 && sub4 <= kKMaxSub4 && n8 <= kKMaxSub8) {
    // Workgroups per KV head: a tile each where all are resident at once, else an even share of the tiles, the next
    // one's rows loaded under the current one.  (Also where two tiles leave room for two workgroups a compute unit
    // only: 8 KV heads x 128k, 128 channels of 8 bit 48.9 us, with a tile and its set-up a workgroup, three
    // resident, 62.7; 64 of each width 31.6 and 62.4; 64 + 80 + 120 58.3 and 72.9.)
    const int64_t cus = compute_units();
    if (stats && stats->n_new > 0) {
      const int64_t passes = rdkv_cdiv(stats->n_new, kKNewKeys), per = rdkv_cdiv(passes, kKNewGroups);
      stats->per_group = (int)std::min<int64_t>(per * kKNewKeys, 0x7fffffc0);
      stats->new_groups = (int)rdkv_cdiv(passes, per);
    }
    // (the workgroups of the appended keys come first; what walks the tiles fills the rest of the device, as far as
    // there are pairs for it: all of it up to 256 compute units)
    const int64_t beside = stats ? stats->new_groups : 0;
    auto resident = [&](size_t lds) {
      const int64_t all = std::max<int64_t>(1, std::min<int64_t>(k_resident(ng), kKMaxLds / (int64_t)(lds + 512)) * cus / H_kv);
      const int64_t walkers = std::max(all - beside, (all + 1) / 2);
      return stats ? std::min<int64_t>(walkers, kKMaxPairs - beside) : walkers;
    };
    size_t staged = setup + tile_lds;
    int64_t wph = tblocks;
    if (tblocks > resident(staged)) {
      staged += tile_lds;
      wph = rdkv_cdiv(tblocks, rdkv_cdiv(tblocks, resident(staged)));
    }
    wph += beside;
    if (stats) *n_pairs = (int)wph;
#define RDKV_LAUNCH_K_MFMA(NG_, CPT_, STATS_)                                                                      \
  do {                                                                                                             \
    if (staged > 64 * 1024)                                                                                        \
      RDKV_REQUIRE(hipFuncSetAttribute(reinterpret_cast<const void *>(k_qk_dot_mfma_kernel<NG_, CPT_, STATS_>),    \
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kKMaxLds) == hipSuccess,        \
                   "rdkv_k_qk_dot: the device refuses %d bytes of LDS per workgroup", (int)staged);                \
    for (int g0 = 0; g0 < G; g0 += 4 * NG_)                                                                          \
      hipLaunchKernelGGL((k_qk_dot_mfma_kernel<NG_, CPT_, STATS_>), dim3((unsigned)wph, H_kv), dim3(256), staged, s,   \
                     q, q_dtype, q_stride_h, G, g0, K2, k2_stride_h, K4, k4_stride_h, K8, k8_stride_h,             \
                     (const __half *)scale_f16, (const __half *)zp_f16, ks_stride_h, perm, perm_stride_h, n2p,     \
                     n4p, n8, T_eff, out, out_stride_h, tile_lds, stats ? *stats : KStats{});                      \
  } while (0)
#define RDKV_LAUNCH_K_MFMA_S(NG_, CPT_)                                                                            \
  do {                                                                                                             \
    if (stats) RDKV_LAUNCH_K_MFMA(NG_, CPT_, true);                                                                \
    else RDKV_LAUNCH_K_MFMA(NG_, CPT_, false);                                                                     \
  } while (0)
    if (ng == 1 && Dp <= 256) RDKV_LAUNCH_K_MFMA_S(1, 1);
    else if (ng == 1) RDKV_LAUNCH_K_MFMA_S(1, 2);
    else if (Dp <= 256) RDKV_LAUNCH_K_MFMA_S(2, 1);
    else RDKV_LAUNCH_K_MFMA_S(2, 2);
#undef RDKV_LAUNCH_K_MFMA_S
#undef RDKV_LAUNCH_K_MFMA
  } else {
    hipLaunchKernelGGL(k_qk_dot_strided_kernel, dim3((unsigned)tblocks, H_kv), dim3(256), shmem, s, q, q_dtype,
                       q_stride_h, G, K2, k2_stride_h, k2_stride_t, K4, k4_stride_h, k4_stride_t, K8,
                       k8_stride_h, k8_stride_t, (const __half *)scale_f16, (const __half *)zp_f16, ks_stride_h,
                       perm, perm_stride_h, n2p, n4p, n8, T_eff, out, out_stride_h);
  }
  RDKV_CHECK_LAUNCH("rdkv_k_qk_dot");
  return RDKV_OK;
}

RDKV_API int rdkv_k_qk_dot(const void *q, int q_dtype, int64_t q_stride_h, int H_q, int H_kv,
                           const uint8_t *K2, int64_t k2_stride_h, int64_t k2_stride_t, const uint8_t *K4,
                           int64_t k4_stride_h, int64_t k4_stride_t, const uint8_t *K8, int64_t k8_stride_h,
                           int64_t k8_stride_t, const void *scale_f16, const void *zp_f16,
                           int64_t ks_stride_h, const int64_t *perm, int64_t perm_stride_h, int n2p, int n4p,
                           int n8, int64_t T_eff, float *out, int64_t out_stride_h, void *stream) {
  int n_pairs;
  return k_scores(q, q_dtype, q_stride_h, H_q, H_kv, K2, k2_stride_h, k2_stride_t, K4, k4_stride_h, k4_stride_t, K8,
                  k8_stride_h, k8_stride_t, scale_f16, zp_f16, ks_stride_h, perm, perm_stride_h, n2p, n4p, n8, T_eff, out,
                  out_stride_h, nullptr, &n_pairs, stream);
}

RDKV_API int64_t rdkv_softmax_rows_workspace_bytes(int H_q) {
  return (int64_t)(H_q > 0 ? H_q : 0) * kSoftmaxMaxSplit * 2 * (int64_t)sizeof(float);
}

static int softmax_rows(const float *scores_old, int64_t so_stride_h, const float *mask, int64_t mask_stride_h,
                        int64_t T_old, const float *scores_new, int64_t sn_stride_h, int64_t n_new, float *w_old,
                        int64_t wo_stride_h, float *w_new, int64_t wn_stride_h, NewKeys nk, int H_q,
                        void *workspace, int64_t workspace_bytes, void *stream) {
  RDKV_REQUIRE(H_q > 0 && H_q <= 65535 && T_old >= 0 && n_new >= 0, "rdkv_softmax_rows: bad sizes");
  RDKV_REQUIRE(T_old + n_new > 0, "rdkv_softmax_rows: empty rows");
  RDKV_REQUIRE(T_old == 0 || (scores_old && w_old), "rdkv_softmax_rows: null old-zone pointer");
  RDKV_REQUIRE(n_new == 0 || (scores_new && w_new), "rdkv_softmax_rows: null new-zone pointer");
  // 16-byte accesses need aligned rows; views that are not go element by element
  const bool vec = T_old >= 4 && ((uintptr_t)scores_old % 16) == 0 && so_stride_h % 4 == 0 &&
                   ((uintptr_t)w_old % 16) == 0 && wo_stride_h % 4 == 0;
  // Pieces per row: enough workgroups for two per compute unit, pieces of at most 4096 float4s;
  // rows that one workgroup holds in registers (64k scores), or heads enough to fill the device, stay with one.
  if (vec && workspace && T_old >= kSoftmaxSplitMinRow) {
    const int64_t n4 = T_old >> 2;
    int64_t S = std::min<int64_t>(kSoftmaxMaxSplit, (2 * (int64_t)compute_units()) / H_q);
    S = std::max(S, rdkv_cdiv(n4, 1024 * kSoftmaxPieceVec));
    if (S >= 2 && S <= kSoftmaxMaxSplit && workspace_bytes >= rdkv_softmax_rows_workspace_bytes(H_q)) {
#define RDKV_LAUNCH_SPLIT(WR)                                                                                     \
  hipLaunchKernelGGL((softmax_rows_split_kernel<WR>), dim3((unsigned)S, H_q), dim3(1024), 0,                  \
                     (hipStream_t)stream, scores_old, so_stride_h, mask, mask_stride_h, T_old, scores_new,        \
                     sn_stride_h, n_new, w_old, wo_stride_h, w_new, wn_stride_h, (float *)workspace, nk)
      RDKV_LAUNCH_SPLIT(false);
      RDKV_LAUNCH_SPLIT(true);
#undef RDKV_LAUNCH_SPLIT
      RDKV_CHECK_LAUNCH("rdkv_softmax_rows");
      return RDKV_OK;
    }
  }
  // One workgroup per head reads that head's keys on its own: from 1024 appended tokens on their scores are a
  // launch of their own, over the whole device.  8 KV heads, G = 4, 40k-token layer, us a call with / without
  // it: 512 tokens 49.2 / 49.4, 1024 49.8 / 52.6, 4096 54 / 72, 16384 78 / 151; without packed tokens 512
  // 16.9 / 17.0, 1024 17.7 / 18.8, 4096 23.5 / 41.8, 16384 49 / 122.  (The split form above deals the keys to
  // its pieces: 131k layer, 4096 tokens 103.5 / 101.9, 16384 138.4 / 138.1.)
  const int64_t eighths = rdkv_cdiv(n_new, 8 * kNewPerBlock);
  if (nk.k && n_new >= kNewOwnLaunch && nk.G <= 65535 && eighths * (H_q / nk.G) <= 65535) {
    hipLaunchKernelGGL(new_zone_scores_kernel, dim3(8, nk.G, (unsigned)(eighths * (H_q / nk.G))), dim3(1024), 0,
                       (hipStream_t)stream, nk, n_new, (int)eighths, w_new, wn_stride_h);
    nk.k = nullptr;
  }
#define RDKV_LAUNCH_SOFTMAX(KERNEL)                                                                             \
  hipLaunchKernelGGL(KERNEL, dim3(H_q), dim3(1024), 0, (hipStream_t)stream, scores_old, so_stride_h, mask,      \
                     mask_stride_h, T_old, scores_new, sn_stride_h, n_new, w_old, wo_stride_h, w_new, wn_stride_h, nk)
#define RDKV_LAUNCH_SOFTMAX_NV(NV) RDKV_LAUNCH_SOFTMAX((softmax_rows_vec_kernel<NV>))
  if (!vec) RDKV_LAUNCH_SOFTMAX(softmax_rows_kernel);
  else if (T_old <= 4096 * 2) RDKV_LAUNCH_SOFTMAX_NV(2);
  else if (T_old <= 4096 * 8) RDKV_LAUNCH_SOFTMAX_NV(8);
  else if (T_old <= 4096 * 16) RDKV_LAUNCH_SOFTMAX_NV(16);
  else RDKV_LAUNCH_SOFTMAX_NV(0);
#undef RDKV_LAUNCH_SOFTMAX_NV
#undef RDKV_LAUNCH_SOFTMAX
  RDKV_CHECK_LAUNCH("rdkv_softmax_rows");
  return RDKV_OK;
}

RDKV_API int rdkv_softmax_rows_ws(const float *scores_old, int64_t so_stride_h, const float *mask,
                                  int64_t mask_stride_h, int64_t T_old, const float *scores_new,
                                  int64_t sn_stride_h, int64_t n_new, float *w_old, int64_t wo_stride_h,
                                  float *w_new, int64_t wn_stride_h, int H_q, void *workspace,
                                  int64_t workspace_bytes, void *stream) {
  return softmax_rows(scores_old, so_stride_h, mask, mask_stride_h, T_old, scores_new, sn_stride_h, n_new, w_old,
                      wo_stride_h, w_new, wn_stride_h, NewKeys{nullptr, 0, 0, 1, nullptr, 0, 0}, H_q, workspace,
                      workspace_bytes, stream);
}

RDKV_API int rdkv_softmax_rows_new_keys(const float *scores_old, int64_t so_stride_h, const float *mask,
                                        int64_t mask_stride_h, int64_t T_old, const void *q, int q_dtype,
                                        int64_t q_stride_h, const float *k_new, int64_t kn_stride_h,
                                        int64_t kn_stride_t, int64_t n_new, float *w_old, int64_t wo_stride_h,
                                        float *w_new, int64_t wn_stride_h, int H_q, int H_kv, void *workspace,
                                        int64_t workspace_bytes, void *stream) {
  const char *fn = "rdkv_softmax_rows_new_keys";
  RDKV_REQUIRE(H_q > 0 && H_kv > 0 && H_q % H_kv == 0, "%s: H_q=%d not a multiple of H_kv=%d", fn, H_q, H_kv);
  RDKV_REQUIRE(q_dtype >= 0 && q_dtype <= 2, "%s: unknown q dtype %d", fn, q_dtype);
  RDKV_REQUIRE(n_new == 0 || (q && k_new), "%s: null pointer", fn);
  RDKV_REQUIRE(n_new <= 1 || kn_stride_t >= kD, "%s: key rows overlap", fn);
  RDKV_REQUIRE(((uintptr_t)k_new % 16) == 0 && kn_stride_h % 4 == 0 && kn_stride_t % 4 == 0,
               "%s: key rows must be 16-byte aligned", fn);
  return softmax_rows(scores_old, so_stride_h, mask, mask_stride_h, T_old, w_new, wn_stride_h, n_new, w_old,
                      wo_stride_h, w_new, wn_stride_h,
                      NewKeys{q, q_stride_h, q_dtype, H_q / H_kv, n_new > 0 ? k_new : nullptr, kn_stride_h, kn_stride_t},
                      H_q, workspace, workspace_bytes, stream);
}

RDKV_API int64_t rdkv_attn_scores_workspace_bytes(int H_q) {
  return (int64_t)(H_q > 0 ? H_q : 0) * (1 + kKMaxPairs) * (int64_t)sizeof(float2);
}

RDKV_API int rdkv_attn_scores(const void *q, int q_dtype, int64_t q_stride_h, int H_q, int H_kv, const uint8_t *K2,
                              int64_t k2_stride_h, int64_t k2_stride_t, const uint8_t *K4, int64_t k4_stride_h,
                              int64_t k4_stride_t, const uint8_t *K8, int64_t k8_stride_h, int64_t k8_stride_t,
                              const void *scale_f16, const void *zp_f16, int64_t ks_stride_h, const int64_t *perm,
                              int64_t perm_stride_h, int n2p, int n4p, int n8, int64_t T_old, const float *mask,
                              int64_t mask_stride_h, const float *k_new, int64_t kn_stride_h, int64_t kn_stride_t,
                              int64_t n_new, float *scores, int64_t stride_h, void *workspace, int64_t workspace_bytes,
                              int *n_pairs, void *stream) {
  const char *fn = "rdkv_attn_scores";
  RDKV_REQUIRE(n_pairs && scores && T_old > 0 && n_new >= 0, "%s: bad arguments", fn);
  RDKV_REQUIRE(n_new == 0 || (q && k_new), "%s: null pointer", fn);
  RDKV_REQUIRE(n_new <= 1 || kn_stride_t >= kD, "%s: key rows overlap", fn);
  RDKV_REQUIRE(((uintptr_t)k_new % 16) == 0 && kn_stride_h % 4 == 0 && kn_stride_t % 4 == 0,
               "%s: key rows must be 16-byte aligned", fn);
  RDKV_REQUIRE(H_q > 0 && H_q <= 65535, "%s: H_q=%d", fn, H_q);
  if (!workspace || workspace_bytes < rdkv_attn_scores_workspace_bytes(H_q)) {
    rdkv_set_error("rdkv_attn_scores: workspace of %lld bytes required", (long long)rdkv_attn_scores_workspace_bytes(H_q));
    return RDKV_EWORKSPACE;
  }
  KStats stats{mask, mask_stride_h, k_new, kn_stride_h, kn_stride_t, n_new, 0, 0, (float2 *)workspace + H_q};
  const int rc = k_scores(q, q_dtype, q_stride_h, H_q, H_kv, K2, k2_stride_h, k2_stride_t, K4, k4_stride_h, k4_stride_t, K8,
                          k8_stride_h, k8_stride_t, scale_f16, zp_f16, ks_stride_h, perm, perm_stride_h, n2p, n4p, n8, T_old,
                          scores, stride_h, &stats, n_pairs, stream);
  if (rc != RDKV_OK || *n_pairs > 0) return rc;
  return rdkv_softmax_rows_new_keys(scores, stride_h, mask, mask_stride_h, T_old, q, q_dtype, q_stride_h, k_new, kn_stride_h,
                                    kn_stride_t, n_new, scores, stride_h, scores + T_old, stride_h, H_q, H_kv, workspace,
                                    workspace_bytes, stream);
}

RDKV_API int rdkv_softmax_rows(const float *scores_old, int64_t so_stride_h, const float *mask,
                               int64_t mask_stride_h, int64_t T_old, const float *scores_new,
                               int64_t sn_stride_h, int64_t n_new, float *w_old, int64_t wo_stride_h,
                               float *w_new, int64_t wn_stride_h, int H_q, void *stream) {
  return rdkv_softmax_rows_ws(scores_old, so_stride_h, mask, mask_stride_h, T_old, scores_new, sn_stride_h, n_new,
                              w_old, wo_stride_h, w_new, wn_stride_h, H_q, nullptr, 0, stream);
}

RDKV_API int64_t rdkv_v_weighted_sum_workspace_bytes(int H_q) {
  return (int64_t)kVChunks * (H_q > 0 ? H_q : 0) * kD * (int64_t)sizeof(float);
}

static int v_weighted_sum(const float *w, int64_t w_stride_h, int H_q, int H_kv, const uint8_t *V2, int64_t v2_stride_h,
                          const uint8_t *V4, int64_t v4_stride_h, const uint8_t *V8, int64_t v8_stride_h,
                          const void *scale_f16, const void *zp_f16, int64_t vs_stride_h,
                          const int32_t *seg_bounds_dev, int N2, int N4, int N8, const void *V16_f16,
                          int64_t v16_stride_h, const int32_t *n_v16_dev, int64_t max_T_v, const NewValues &nv,
                          const VScores &vs, const ScoreRows &sr, float *out, int64_t out_stride_h, void *workspace,
                          int64_t workspace_bytes, void *stream) {
  RDKV_REQUIRE(H_q > 0 && H_kv > 0 && H_q % H_kv == 0, "rdkv_v_weighted_sum: H_q=%d not a multiple of H_kv=%d",
               H_q, H_kv);
  RDKV_REQUIRE(w && out, "rdkv_v_weighted_sum: null pointer");
  RDKV_REQUIRE(N2 >= 0 && N4 >= 0 && N8 >= 0 && max_T_v >= 0, "rdkv_v_weighted_sum: negative count");
  if (!workspace || workspace_bytes < rdkv_v_weighted_sum_workspace_bytes(H_q)) {
    rdkv_set_error("rdkv_v_weighted_sum: workspace of %lld bytes required",
                   (long long)rdkv_v_weighted_sum_workspace_bytes(H_q));
    return RDKV_EWORKSPACE;
  }
  if (!seg_bounds_dev) {
    RDKV_REQUIRE((N2 == 0 || V2) && (N4 == 0 || V4) && (N8 == 0 || V8), "rdkv_v_weighted_sum: missing V segment");
  }
  RDKV_REQUIRE((int64_t)N2 + N4 + N8 == 0 || (scale_f16 && zp_f16) || seg_bounds_dev,
               "rdkv_v_weighted_sum: missing scale/zp");
  hipStream_t s = (hipStream_t)stream;
  // wide loads: the packed rows are 32 / 64 / 128 / 256 bytes long, so 16-byte aligned bases suffice
  RDKV_REQUIRE(((uintptr_t)V2 % 16) == 0 && ((uintptr_t)V4 % 16) == 0 && ((uintptr_t)V8 % 16) == 0 &&
                   ((uintptr_t)V16_f16 % 16) == 0 && v2_stride_h % 16 == 0 && v4_stride_h % 16 == 0 &&
                   v8_stride_h % 16 == 0 && v16_stride_h % 8 == 0,
               "rdkv_v_weighted_sum: V segments must be 16-byte aligned");
  const int G = H_q / H_kv;
  const int64_t quads = rdkv_cdiv(G, 4);
  RDKV_REQUIRE(H_kv <= 65535 && quads <= 65535, "rdkv_v_weighted_sum: too many heads");
  const int64_t pieces = sr.s ? rdkv_cdiv(sr.n, kRowPiece) : 0;
  RDKV_REQUIRE((1 + pieces) * H_q <= 0x7fffffffLL, "rdkv_v_weighted_sum: rows too long");
#define RDKV_LAUNCH_V(SCORES_)                                                                                        \
  hipLaunchKernelGGL(v_weighted_sum_kernel<SCORES_>, dim3(kVChunks, H_kv, (unsigned)quads), dim3(64 * kVWaves), 0, s, \
                     w, w_stride_h, G, V2, v2_stride_h, V4, v4_stride_h, V8, v8_stride_h, (const uint16_t *)scale_f16, \
                     (const uint16_t *)zp_f16, vs_stride_h, seg_bounds_dev, N2, N4, N8, (const uint8_t *)V16_f16,     \
                     v16_stride_h, n_v16_dev, max_T_v, nv, (float *)workspace, H_q, vs)
  if (vs.pairs) RDKV_LAUNCH_V(true);
  else RDKV_LAUNCH_V(false);
#undef RDKV_LAUNCH_V
  hipLaunchKernelGGL(v_reduce_kernel, dim3((unsigned)((1 + pieces) * H_q)), dim3(8 * kD), 0, s, (const float *)workspace, H_q,
                     out, out_stride_h, sr);
  RDKV_CHECK_LAUNCH("rdkv_v_weighted_sum");
  return RDKV_OK;
}

RDKV_API int rdkv_v_weighted_sum(const float *w, int64_t w_stride_h, int H_q, int H_kv, const uint8_t *V2,
                                 int64_t v2_stride_h, const uint8_t *V4, int64_t v4_stride_h, const uint8_t *V8,
                                 int64_t v8_stride_h, const void *scale_f16, const void *zp_f16,
                                 int64_t vs_stride_h, const int32_t *seg_bounds_dev, int N2, int N4, int N8,
                                 const void *V16_f16, int64_t v16_stride_h, const int32_t *n_v16_dev,
                                 int64_t max_T_v, float *out, int64_t out_stride_h, void *workspace,
                                 int64_t workspace_bytes, void *stream) {
  return v_weighted_sum(w, w_stride_h, H_q, H_kv, V2, v2_stride_h, V4, v4_stride_h, V8, v8_stride_h, scale_f16, zp_f16,
                        vs_stride_h, seg_bounds_dev, N2, N4, N8, V16_f16, v16_stride_h, n_v16_dev, max_T_v, NewValues{}, VScores{},
                        ScoreRows{}, out, out_stride_h, workspace, workspace_bytes, stream);
}

RDKV_API int rdkv_v_weighted_sum_new_values(
    const float *w, int64_t w_stride_h, int H_q, int H_kv, const uint8_t *V2, int64_t v2_stride_h, const uint8_t *V4,
    int64_t v4_stride_h, const uint8_t *V8, int64_t v8_stride_h, const void *scale_f16, const void *zp_f16,
    int64_t vs_stride_h, const int32_t *seg_bounds_dev, int N2, int N4, int N8, const void *V16_f16,
    int64_t v16_stride_h, const int32_t *n_v16_dev, int64_t max_T_v, const float *w_new, int64_t wn_stride_h,
    const float *v_new, int64_t vn_stride_h, int64_t vn_stride_t, int64_t n_new, float *out, int64_t out_stride_h,
    void *workspace, int64_t workspace_bytes, void *stream) {
  const char *fn = "rdkv_v_weighted_sum_new_values";
  RDKV_REQUIRE(n_new >= 0 && (n_new == 0 || (w_new && v_new)), "%s: bad new zone", fn);
  RDKV_REQUIRE(((uintptr_t)v_new % 16) == 0 && vn_stride_h % 4 == 0 && vn_stride_t % 4 == 0,
               "%s: value rows must be 16-byte aligned", fn);
  return v_weighted_sum(w, w_stride_h, H_q, H_kv, V2, v2_stride_h, V4, v4_stride_h, V8, v8_stride_h, scale_f16, zp_f16,
                        vs_stride_h, seg_bounds_dev, N2, N4, N8, V16_f16, v16_stride_h, n_v16_dev, max_T_v,
                        NewValues{n_new > 0 ? v_new : nullptr, w_new, vn_stride_h, vn_stride_t, wn_stride_h, n_new},
                        VScores{}, ScoreRows{}, out, out_stride_h, workspace, workspace_bytes, stream);
}

RDKV_API int rdkv_v_weighted_sum_scores(
    float *scores, int64_t stride_h, int H_q, int H_kv, const uint8_t *V2, int64_t v2_stride_h, const uint8_t *V4,
    int64_t v4_stride_h, const uint8_t *V8, int64_t v8_stride_h, const void *scale_f16, const void *zp_f16,
    int64_t vs_stride_h, const int32_t *seg_bounds_dev, int N2, int N4, int N8, const void *V16_f16,
    int64_t v16_stride_h, const int32_t *n_v16_dev, int64_t max_T_v, int64_t T_old, const float *v_new,
    int64_t vn_stride_h, int64_t vn_stride_t, int64_t n_new, void *softmax_ws, int n_pairs, int keep_weights, float *out,
    int64_t out_stride_h, void *workspace, int64_t workspace_bytes, void *stream) {
  const char *fn = "rdkv_v_weighted_sum_scores";
  RDKV_REQUIRE(scores && softmax_ws && T_old >= 0 && n_new >= 0 && (n_new == 0 || v_new), "%s: bad arguments", fn);
  RDKV_REQUIRE(n_pairs >= 0 && n_pairs <= kKMaxPairs, "%s: %d pairs", fn, n_pairs);
  RDKV_REQUIRE(((uintptr_t)v_new % 16) == 0 && vn_stride_h % 4 == 0 && vn_stride_t % 4 == 0,
               "%s: value rows must be 16-byte aligned", fn);
  float2 *rows = (float2 *)softmax_ws;
  const VScores vs = n_pairs > 0 ? VScores{rows + H_q, n_pairs, rows} : VScores{};
  const ScoreRows sr = n_pairs > 0 && keep_weights ? ScoreRows{scores, stride_h, T_old + n_new, rows} : ScoreRows{};
  return v_weighted_sum(scores, stride_h, H_q, H_kv, V2, v2_stride_h, V4, v4_stride_h, V8, v8_stride_h, scale_f16, zp_f16,
                        vs_stride_h, seg_bounds_dev, N2, N4, N8, V16_f16, v16_stride_h, n_v16_dev, max_T_v,
                        NewValues{n_new > 0 ? v_new : nullptr, scores + T_old, vn_stride_h, vn_stride_t, stride_h, n_new}, vs,
                        sr, out, out_stride_h, workspace, workspace_bytes, stream);
}
