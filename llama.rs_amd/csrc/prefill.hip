// Multi-token prefill kernels: the prompt goes through each layer as a
// T-row batch (CausalModel::prefill, src/architecture.rs:60-77, computed the
// way Qwen2Model::forward_impl, src/model.rs:135-271, computes one token).
//
// The weight matrices run as MFMA dequant-GEMMs: a workgroup owns a 64- or
// 128-token x 128-row output tile (of one K range when K is split).  It
// dequantizes its 128 weight rows 64 columns at a time from the native GGUF
// blocks (value_at, src/quant.rs:349-456) into LDS, stages the matching
// activation tile, and accumulates v_mfma_f32_16x16x32_f16 products in f32.
// Eight waves share a tile (prefill_gemm8_kernel; the four-wave form is kept
// for comparison): four stage the weights, four the activations, and each
// multiplies BM/2 tokens x 32 rows.  The raw
// weight blocks and activations of the next 64 columns are loaded into
// registers before the current ones are multiplied, so the loads' latency
// hides behind the MFMAs.  Causal attention runs on f32 MFMA
// (attention_tile_kernel).
//
// Precision: f32 operands are carried as f16 pairs, v = hi + lo with hi =
// f16(v) and lo = f16(v - hi) (22 significant bits), and each product is
// hi*hi + hi*lo + lo*hi (the lo*lo term is below f32 rounding of the sum), so
// the GEMM is close to an f32 GEMM rather than an f16 one.  Most products of
// the types in prefill_reg.hip take its kernels instead.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <cstring>

#include "common.h"
#include "wave_dev.h"
#include "prefill.h"
#include "quant_dev.h"

namespace llrs {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int BN = 128, KC = 64, LS = KC + 8;
// Weight-row tiles from which 128-token tiles are used (at 256+ tokens);
// split K makes up the workgroups the larger tiles leave out.
constexpr int kTile128Rows = 16;  // weight rows per tile; LS: LDS row stride in halves

// The 32 values of `row` at columns [k0, k0 + 32) (k0 a multiple of 32), as
// value_at computes them, in two stages: load() issues the loads of the raw
// block bytes, decode() turns them into values once they have arrived.
template <uint32_t TY> struct Deq {
  struct Raw { const uint8_t *row; uint32_t ty; };
  static __device__ __forceinline__ void load(const uint8_t *row, uint32_t ty, int, Raw &r) {
    r.row = row;
    r.ty = ty;
  }
  static __device__ __forceinline__ void decode(const Raw &r, int k0, float (&v)[32]) {
#pragma unroll
    for (int j = 0; j < 32; j++) v[j] = value_dev(r.row, r.ty, (uint32_t)(k0 + j));
  }
};

// Byte i of the little-endian words w.
__device__ __forceinline__ int byte_of(const uint32_t *w, int i) { return (int)((w[i >> 2] >> (8 * (i & 3))) & 0xff); }

template <> struct Deq<LLRS_Q4_K> {
  struct Raw { uint4 hdr, q0, q1; };  // d, dmin, 12 scale bytes; the sub-block's 32 quant bytes
  static __device__ __forceinline__ void load(const uint8_t *row, uint32_t, int k0, Raw &r) {
    const uint8_t *b = row + (size_t)(k0 >> 8) * 144;
    const int g = (k0 & 255) >> 5;
    r.hdr = *reinterpret_cast<const uint4 *>(b);
    r.q0 = *reinterpret_cast<const uint4 *>(b + 16 + (g >> 1) * 32);
    r.q1 = *reinterpret_cast<const uint4 *>(b + 32 + (g >> 1) * 32);
  }
  static __device__ __forceinline__ void decode(const Raw &r, int k0, float (&v)[32]) {
#pragma clang fp contract(off)
    const int g = (k0 & 255) >> 5;
    const uint32_t s[3] = {r.hdr.y, r.hdr.z, r.hdr.w};
    int sc, mn;  // scale_min_k4 (src/quant.rs:338-347) on the scale bytes in registers
    if (g < 4) {
      sc = byte_of(s, g) & 63;
      mn = byte_of(s, g + 4) & 63;
    } else {
      sc = (byte_of(s, g + 4) & 0x0f) | ((byte_of(s, g - 4) >> 6) << 4);
      mn = (byte_of(s, g + 4) >> 4) | ((byte_of(s, g) >> 6) << 4);
    }
    const float ds = f16_bits_to_f32((uint16_t)(r.hdr.x & 0xffff)) * (float)sc;
    const float dm = f16_bits_to_f32((uint16_t)(r.hdr.x >> 16)) * (float)mn;
    const uint32_t w[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
    const int shift = (g & 1) * 4;
#pragma unroll
    for (int j = 0; j < 32; j++) {
      const int q = (int)((w[j >> 2] >> (8 * (j & 3) + shift)) & 15);
      v[j] = ds * (float)q - dm;
    }
  }
};

template <> struct Deq<LLRS_Q6_K> {
  struct Raw { uint32_t ql[9], qh[9], shl, shh; uint16_t s2, d; };
  static __device__ __forceinline__ void load(const uint8_t *row, uint32_t, int k0, Raw &r) {
    const uint8_t *b = row + (size_t)(k0 >> 8) * 210;
    const int j0 = k0 & 255, half = j0 >> 7, quarter = (j0 >> 5) & 3;
    load9(b + half * 64 + (quarter & 1) * 32, r.ql, r.shl);
    load9(b + 128 + half * 32, r.qh, r.shh);
    r.s2 = ld_u16(b + 192 + half * 8 + quarter * 2);
    r.d = ld_u16(b + 208);
  }
  static __device__ __forceinline__ void decode(const Raw &r, int k0, float (&v)[32]) {
#pragma clang fp contract(off)
    const int quarter = (k0 >> 5) & 3;
    const float d = f16_bits_to_f32(r.d);
    const float sc0 = d * (float)(int8_t)(r.s2 & 0xff), sc1 = d * (float)(int8_t)(r.s2 >> 8);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const uint32_t l = realign(r.ql, k, r.shl), h = realign(r.qh, k, r.shh);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int lb = (int)((l >> (8 * e)) & 0xff);
        const int lo = quarter < 2 ? (lb & 15) : (lb >> 4);
        const int hi = (int)((h >> (8 * e + 2 * quarter)) & 3);
        const int j = 4 * k + e;
        v[j] = (j < 16 ? sc0 : sc1) * (float)((lo | (hi << 4)) - 32);
      }
    }
  }
};

template <> struct Deq<LLRS_Q8_0> {
  struct Raw { uint32_t q[9], sh; uint16_t d; };
  static __device__ __forceinline__ void load(const uint8_t *row, uint32_t, int k0, Raw &r) {
    const uint8_t *b = row + (size_t)(k0 >> 5) * 34;
    load9(b + 2, r.q, r.sh);
    r.d = ld_u16(b);
  }
  static __device__ __forceinline__ void decode(const Raw &r, int, float (&v)[32]) {
    const float d = f16_bits_to_f32(r.d);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const uint32_t w = realign(r.q, k, r.sh);
#pragma unroll
      for (int e = 0; e < 4; e++) v[4 * k + e] = d * (float)(int8_t)((w >> (8 * e)) & 0xff);
    }
  }
};

template <> struct Deq<LLRS_Q5_0> {
  struct Raw { uint32_t r[9], sh; uint16_t d; };  // qh (4 bytes) then 16 bytes of nibbles
  static __device__ __forceinline__ void load(const uint8_t *row, uint32_t, int k0, Raw &r) {
    const uint8_t *b = row + (size_t)(k0 >> 5) * 22;
    load9(b + 2, r.r, r.sh);
    r.d = ld_u16(b);
  }
  static __device__ __forceinline__ void decode(const Raw &r, int, float (&v)[32]) {
#pragma clang fp contract(off)
    const uint32_t qh = realign(r.r, 0, r.sh);
    const float d = f16_bits_to_f32(r.d);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t w = realign(r.r, k + 1, r.sh);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int j = 4 * k + e;
        const int lo = (int)((w >> (8 * e)) & 15), hi = (int)((w >> (8 * e + 4)) & 15);
        v[j] = d * ((float)(lo | (int)(((qh >> j) & 1) << 4)) - 16.0f);
        v[j + 16] = d * ((float)(hi | (int)(((qh >> (j + 16)) & 1) << 4)) - 16.0f);
      }
    }
  }
};

// F16 and BF16 rows (16-bit values, four 16-byte loads) and F32 rows (eight):
// rows of a multiple of 32 columns, so every load is 16-byte aligned.  The
// element-wise decode of the general case (2-byte loads, a type switch per
// element) bound such products; 301 tokens through four 0.5B-shape BF16
// layers: 2,518 us with it, 736 us with these loads and one weight plane.
template <uint32_t TY> struct DeqFloat {
  static constexpr int kLoads = TY == LLRS_F32 ? 8 : 4;
  struct Raw { uint4 q[kLoads]; };
  static __device__ __forceinline__ void load(const uint8_t *row, uint32_t, int k0, Raw &r) {
    const uint4 *p = reinterpret_cast<const uint4 *>(row + (size_t)k0 * (TY == LLRS_F32 ? 4 : 2));
#pragma unroll
    for (int i = 0; i < kLoads; i++) r.q[i] = p[i];
  }
  static __device__ __forceinline__ void decode(const Raw &r, int, float (&v)[32]) {
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
      const uint32_t w[4] = {r.q[i].x, r.q[i].y, r.q[i].z, r.q[i].w};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if constexpr (TY == LLRS_F32) {
          v[4 * i + e] = __uint_as_float(w[e]);
        } else if constexpr (TY == LLRS_F16) {
          v[8 * i + 2 * e] = f16_bits_to_f32((uint16_t)(w[e] & 0xffff));
          v[8 * i + 2 * e + 1] = f16_bits_to_f32((uint16_t)(w[e] >> 16));
        } else {
          v[8 * i + 2 * e] = __uint_as_float(w[e] << 16);
          v[8 * i + 2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
        }
      }
    }
  }
};
template <> struct Deq<LLRS_F16> : DeqFloat<LLRS_F16> {};
template <> struct Deq<LLRS_BF16> : DeqFloat<LLRS_BF16> {};
template <> struct Deq<LLRS_F32> : DeqFloat<LLRS_F32> {};

// Whether a type's weights need one f16 plane only.  An F16 weight is its own
// hi; a BF16 weight (8 significant bits) is exact in f16 from 2^-17 up, and
// below that hi is its rounding to f16's 2^-24 grid, which leaves lo = 0 too.
template <uint32_t TY> constexpr bool kOnePlane = TY == LLRS_F16 || TY == LLRS_BF16;

__device__ __forceinline__ void split_f16(float v, f16 &hi, f16 &lo) {
  hi = (f16)v;
  lo = (f16)(v - (float)hi);
}

// A wave's MI x NJ accumulator blocks of 16 x 16 (tokens tb + 16 i + ..., rows
// nb + 16 j + ...; D layout: lane holds row (lane & 15) and tokens
// 4 * (lane >> 4) + e) into C: C (=|+=) acc (+ bias), or with K split the
// split's partial tile into `part` (split_reduce_kernel adds them up).
template <int MI, int NJ>
__device__ __forceinline__ void store_tile(const PrefillGemmArgs &g, const f32x4 (&acc)[MI][NJ], int nb, int tb,
                                           int lane) {
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      const int n = nb + 16 * j + (lane & 15);
      if (n >= g.n) continue;
      const float bias = (!g.accumulate && g.bias) ? g.bias[n] : 0.f;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int t = tb + 16 * i + 4 * (lane >> 4) + e;
        if (t >= g.t) continue;
        if (g.ksplit > 1) {
          g.part[((size_t)blockIdx.z * g.t + t) * g.n + n] = acc[i][j][e];
        } else {
          float *c = g.c + (size_t)t * g.ldc + n;
          *c = g.accumulate ? *c + acc[i][j][e] : acc[i][j][e] + bias;
        }
      }
    }
}

// BM tokens x BN weight rows per workgroup (BM = 64 or 128).
template <uint32_t TY, int BM>
__global__ __launch_bounds__(256) void prefill_gemm_kernel(PrefillGemmArgs g) {
  constexpr int MI = BM / 32;    // 16-token MFMA blocks per wave
  constexpr int APT = BM / 4;    // activation halves per thread and plane
  constexpr int TPR = 64 / APT;  // threads per activation row
  extern __shared__ __align__(16) f16 lds[];
  f16 *As = lds, *Al = As + BM * LS, *Ws = Al + BM * LS, *Wl = Ws + BN * LS;
  const int n0 = blockIdx.x * BN, t0 = blockIdx.y * BM;
  // This workgroup's K range (split K: whole KC chunks per split).
  const int per = ((g.k + KC - 1) / KC + g.ksplit - 1) / g.ksplit * KC;
  const int kb = blockIdx.z * per, ke = min(g.k, kb + per);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;  // the wave's (BM/2)-token x 64-row quarter
  f32x4 acc[MI][4];
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Staging roles: activations BM rows x TPR runs of APT halves, weights 128
  // rows x 2 runs of 32 values.  Rows past the tile's end read row 0 and are
  // zeroed on their way into LDS.
  const int ar = tid / TPR, ac = (tid % TPR) * APT;
  const int wr = tid >> 1, wc = (tid & 1) * 32;
  const bool a_ok = t0 + ar < g.t, w_ok = n0 + wr < g.n;
  const size_t aoff = (size_t)(a_ok ? t0 + ar : 0) * g.lda + ac;
  const uint8_t *wrow = g.w + (size_t)(w_ok ? n0 + wr : 0) * g.row_bytes;
  half8 ah[APT / 8], alo[APT / 8];
  typename Deq<TY>::Raw raw;
  auto load_chunk = [&](int k0) {
    const int kk = min(k0 + ac, ke - APT);  // columns past the range: a valid read, zeroed below
#pragma unroll
    for (int h = 0; h < APT / 8; h++) {
      ah[h] = *reinterpret_cast<const half8 *>(g.a + aoff - ac + kk + 8 * h);
      alo[h] = *reinterpret_cast<const half8 *>(g.a_lo + aoff - ac + kk + 8 * h);
    }
    Deq<TY>::load(wrow, g.type, min(k0 + wc, ke - 32), raw);
  };
  // A split whose range is empty (rounding of the per-split chunk count)
  // loads nothing and writes zero partials.
  if (kb < ke) load_chunk(kb);
  for (int k0 = kb; k0 < ke; k0 += KC) {
    const int kc = min(KC, ke - k0);  // 32 or 64
    __syncthreads();  // the previous chunk's MFMAs have read LDS
    {
      const bool in = a_ok && ac < kc;
      const half8 z = half8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int h = 0; h < APT / 8; h++) {
        *reinterpret_cast<half8 *>(As + ar * LS + ac + 8 * h) = in ? ah[h] : z;
        *reinterpret_cast<half8 *>(Al + ar * LS + ac + 8 * h) = in ? alo[h] : z;
      }
    }
    {
      float v[32];
      Deq<TY>::decode(raw, min(k0 + wc, ke - 32), v);  // the columns load_chunk read
      const bool in = w_ok && wc < kc;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        half8 h, l;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          f16 a, b;
          split_f16(in ? v[8 * q + e] : 0.f, a, b);
          h[e] = a;
          l[e] = b;
        }
        *reinterpret_cast<half8 *>(Ws + wr * LS + wc + 8 * q) = h;
        *reinterpret_cast<half8 *>(Wl + wr * LS + wc + 8 * q) = l;
      }
    }
    __syncthreads();
    if (k0 + KC < ke) load_chunk(k0 + KC);  // in flight during the MFMAs below
    for (int ks = 0; ks < kc; ks += 32) {
      half8 af[MI], al[MI], bf[4], bl[4];
#pragma unroll
      for (int i = 0; i < MI; i++) {
        const int o = (wm * (BM / 2) + 16 * i + (lane & 15)) * LS + ks + 8 * (lane >> 4);
        af[i] = *reinterpret_cast<const half8 *>(As + o);
        al[i] = *reinterpret_cast<const half8 *>(Al + o);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int o = (wn * 64 + 16 * j + (lane & 15)) * LS + ks + 8 * (lane >> 4);
        bf[j] = *reinterpret_cast<const half8 *>(Ws + o);
        bl[j] = *reinterpret_cast<const half8 *>(Wl + o);
      }
#pragma unroll
      for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], bf[j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bl[j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
    }
  }
  store_tile<MI, 4>(g, acc, n0 + wn * 64, t0 + wm * (BM / 2), lane);
}

// The same tile, products and LDS layout with eight waves, so that two
// workgroups per CU put four waves on each SIMD (the four-wave kernel's two
// leave the matrix cores waiting on the staging chain's latency).  Waves 0-3
// dequantize the weight tile (32 values per thread, as above) while waves
// 4-7 stage the activation tile, so each SIMD holds one wave of each kind;
// all eight run MFMAs, each on BM/2 tokens x 32 rows of the tile.  A thread
// keeps only its role's next-chunk registers (a union), which holds a wave
// to 128 registers.  Each output is the same sequence of MFMAs as in the
// four-wave kernel.  Measured 4-5% faster per product (7B shape, 512
// tokens); LLRS_PREFILL_GEMM=4 selects the four-wave kernel.
template <uint32_t TY, int BM>
__global__ __launch_bounds__(512) void prefill_gemm8_kernel(PrefillGemmArgs g) {
  constexpr int MI = BM / 32;    // 16-token MFMA blocks per wave (BM/2 tokens)
  constexpr int NJ = 2;          // 16-row MFMA blocks per wave (32 rows)
  constexpr int APT = BM / 4;    // activation halves per staging thread and plane
  constexpr int TPR = 64 / APT;  // staging threads per activation row
  extern __shared__ __align__(16) f16 lds[];
  f16 *As = lds, *Al = As + BM * LS, *Ws = Al + BM * LS, *Wl = Ws + BN * LS;
  const int n0 = blockIdx.x * BN, t0 = blockIdx.y * BM;
  const int per = ((g.k + KC - 1) / KC + g.ksplit - 1) / g.ksplit * KC;
  const int kb = blockIdx.z * per, ke = min(g.k, kb + per);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;  // BM/2 tokens x 32 rows
  const bool wstage = wave < 4;             // weight staging (else activation staging)
  const int st = tid & 255;                 // thread index within the staging group
  f32x4 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int ar = st / TPR, ac = (st % TPR) * APT;
  const int wr = st >> 1, wc = (st & 1) * 32;
  const bool a_ok = t0 + ar < g.t, w_ok = n0 + wr < g.n;
  const size_t aoff = (size_t)(a_ok ? t0 + ar : 0) * g.lda + ac;
  const uint8_t *wrow = g.w + (size_t)(w_ok ? n0 + wr : 0) * g.row_bytes;
  union Pre {
    struct { half8 ah[APT / 8], al[APT / 8]; } a;
    typename Deq<TY>::Raw raw;
  } pre;
  auto load_chunk = [&](int k0) {
    if (wstage) {
      Deq<TY>::load(wrow, g.type, min(k0 + wc, ke - 32), pre.raw);
    } else {
      const int kk = min(k0 + ac, ke - APT);  // columns past the range: a valid read, zeroed below
#pragma unroll
      for (int h = 0; h < APT / 8; h++) {
        pre.a.ah[h] = *reinterpret_cast<const half8 *>(g.a + aoff - ac + kk + 8 * h);
        pre.a.al[h] = *reinterpret_cast<const half8 *>(g.a_lo + aoff - ac + kk + 8 * h);
      }
    }
  };
  if (kb < ke) load_chunk(kb);
  for (int k0 = kb; k0 < ke; k0 += KC) {
    const int kc = min(KC, ke - k0);  // 32 or 64
    __syncthreads();  // the previous chunk's MFMAs have read LDS
    if (wstage) {
      float v[32];
      Deq<TY>::decode(pre.raw, min(k0 + wc, ke - 32), v);  // the columns load_chunk read
      const bool in = w_ok && wc < kc;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        half8 h, l;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          f16 a, b;
          split_f16(in ? v[8 * q + e] : 0.f, a, b);
          h[e] = a;
          l[e] = b;
        }
        *reinterpret_cast<half8 *>(Ws + wr * LS + wc + 8 * q) = h;
        if constexpr (!kOnePlane<TY>) *reinterpret_cast<half8 *>(Wl + wr * LS + wc + 8 * q) = l;
      }
    } else {
      const bool in = a_ok && ac < kc;
      const half8 z = half8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int h = 0; h < APT / 8; h++) {
        *reinterpret_cast<half8 *>(As + ar * LS + ac + 8 * h) = in ? pre.a.ah[h] : z;
        *reinterpret_cast<half8 *>(Al + ar * LS + ac + 8 * h) = in ? pre.a.al[h] : z;
      }
    }
    __syncthreads();
    if (k0 + KC < ke) load_chunk(k0 + KC);  // in flight during the MFMAs below
    for (int ks = 0; ks < kc; ks += 32) {
      half8 af[MI], al[MI], bf[NJ], bl[NJ];
#pragma unroll
      for (int i = 0; i < MI; i++) {
        const int o = (wm * (BM / 2) + 16 * i + (lane & 15)) * LS + ks + 8 * (lane >> 4);
        af[i] = *reinterpret_cast<const half8 *>(As + o);
        al[i] = *reinterpret_cast<const half8 *>(Al + o);
      }
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        const int o = (wn * 32 + 16 * j + (lane & 15)) * LS + ks + 8 * (lane >> 4);
        bf[j] = *reinterpret_cast<const half8 *>(Ws + o);
        if constexpr (!kOnePlane<TY>) bl[j] = *reinterpret_cast<const half8 *>(Wl + o);
      }
#pragma unroll
      for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[i], bf[j], acc[i][j], 0, 0, 0);
          if constexpr (!kOnePlane<TY>)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bl[j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
    }
  }
  store_tile<MI, NJ>(g, acc, n0 + wn * 32, t0 + wm * (BM / 2), lane);
}


// xs + xs_lo [t][s] = the sum over j < 32 of a[t][32 s + j] + a_lo[t][32 s + j]
// (in that order, in f32), as an f16 pair, for s < nsub.
__global__ void xsum_f16_kernel(const f16 *__restrict__ a, const f16 *__restrict__ a_lo, int lda,
                                int nsub, f16 *__restrict__ xs, f16 *__restrict__ xs_lo, int ldxs) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y;
  if (s >= nsub) return;
  const half8 *p = reinterpret_cast<const half8 *>(a + (size_t)t * lda + 32 * s);
  const half8 *q = reinterpret_cast<const half8 *>(a_lo + (size_t)t * lda + 32 * s);
  float sum = 0.f;
#pragma unroll
  for (int h = 0; h < 4; h++) {
    const half8 x = p[h], y = q[h];
#pragma unroll
    for (int e = 0; e < 8; e++) sum += (float)x[e] + (float)y[e];
  }
  split_f16(sum, xs[(size_t)t * ldxs + s], xs_lo[(size_t)t * ldxs + s]);
}

__global__ void embed_rows_kernel(const uint8_t *__restrict__ emb, uint32_t ty, size_t row_bytes,
                                  int H, uint32_t vocab, const uint32_t *__restrict__ tok, int T,
                                  float *__restrict__ x) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y;
  if (c >= H || t >= T) return;
  uint32_t id = tok[t];
  if (id >= vocab) id = vocab - 1;  // validated on the host; never read past the table
  x[(size_t)t * H + c] = value_dev(emb + (size_t)id * row_bytes, ty, (uint32_t)c);
}

// RMSNorm::forward (src/model.rs:65-73) per token row, rounded to f16.
// With xs set (H a multiple of 32), also the activation sums of the output
// that Q4_K products read: xs + xs_lo [row][s] = the sum of (hi + lo) over
// columns 32 s ... 32 s + 31 (a 32-lane half-wave of one pass), as f16 pairs.
__device__ __forceinline__ void half_wave_xsum(float v, int col, f16 *xs, f16 *xs_lo) {
#pragma unroll
  for (int b = 1; b < 32; b <<= 1) v += lane_partner(v, b);
  if ((threadIdx.x & 31) == 0) split_f16(v, xs[col >> 5], xs_lo[col >> 5]);
}

// A thread holds eight consecutive columns (two 16-byte loads of x and of w, all
// issued before the row's sum; one 16-byte store a plane), and four lanes a
// 32-column sum.  One column a thread and pass chained the sums' exchanges 14
// times over 3,584 columns: 10.0 us for 24 such rows, 6.0 this way.
__global__ __launch_bounds__(1024) void rmsnorm_rows_f16_kernel(const float *__restrict__ x,
                                                                const float *__restrict__ w,
                                                                f16 *__restrict__ out,
                                                                f16 *__restrict__ out_lo, int H,
                                                                float eps, f16 *__restrict__ xs,
                                                                f16 *__restrict__ xs_lo, int ldxs) {
#pragma clang fp contract(off)
  __shared__ float red[16];
  const float4 *xr = reinterpret_cast<const float4 *>(x + (size_t)blockIdx.x * H), *wr = reinterpret_cast<const float4 *>(w);
  const int G = H / 8, tid = threadIdx.x, nt = blockDim.x;
  const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
  // The first group stays in registers (the whole row up to 8,192 columns).
  const bool own = tid < G;
  const float4 x0 = own ? xr[2 * tid] : z, x1 = own ? xr[2 * tid + 1] : z;
  const float4 w0 = own ? wr[2 * tid] : z, w1 = own ? wr[2 * tid + 1] : z;
  auto square = [](float4 a, float4 b) {
    return a.x * a.x + a.y * a.y + a.z * a.z + a.w * a.w + b.x * b.x + b.y * b.y + b.z * b.z + b.w * b.w;
  };
  float s = square(x0, x1);
  for (int g = tid + nt; g < G; g += nt) s += square(xr[2 * g], xr[2 * g + 1]);
  s = wave_total(s);
  if ((tid & 63) == 0) red[tid >> 6] = s;
  __syncthreads();
  float tot = 0.f;
  for (int i = 0; i < nt >> 6; i++) tot += red[i];
  const float inv = 1.0f / sqrtf(tot / (float)H + eps);
  auto emit = [&](int g, float4 a, float4 b, float4 u, float4 v) {  // every lane of a group of four takes part
    const float xv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}, wv[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
    half8 h, l;
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      f16 hi, lo;
      split_f16(xv[e] * (inv * wv[e]), hi, lo);
      h[e] = hi;
      l[e] = lo;
      sum += (float)hi + (float)lo;
    }
    if (g < G) {
      *reinterpret_cast<half8 *>(out + (size_t)blockIdx.x * H + 8 * g) = h;
      *reinterpret_cast<half8 *>(out_lo + (size_t)blockIdx.x * H + 8 * g) = l;
    }
    if (xs) {
      sum += lane_partner(sum, 1);
      sum += lane_partner(sum, 2);
      if ((g & 3) == 0 && g < G)
        split_f16(sum, xs[(size_t)blockIdx.x * ldxs + (g >> 2)], xs_lo[(size_t)blockIdx.x * ldxs + (g >> 2)]);
    }
  };
  emit(tid, x0, x1, w0, w1);
  for (int g0 = nt; g0 < G; g0 += nt) {
    const int g = g0 + tid;
    const bool in = g < G;
    emit(g, in ? xr[2 * g] : z, in ? xr[2 * g + 1] : z, in ? wr[2 * g] : z, in ? wr[2 * g + 1] : z);
  }
}

// Causal GQA attention (src/model.rs:206-231, softmax_inplace 298-313) for a
// tile of 16 query rows of one head, on f32 matrix cores: fp32 products and
// sums as the scalar loop has them, in another order.  The four waves take
// every fourth 16-key block of the causal range and keep a running max;
// their partial states are merged through LDS at the end.
//
// Both products keep the query index in lane % 16, so neither the scores nor
// the weights move between lanes:
//   S^T (keys x queries) = K Q^T     A = K rows, B = Q rows, contraction over
//                                    the head dims (lane group g holds dims
//                                    g*HD/4 ... g*HD/4 + HD/4 - 1)
//   O^T (dims x queries) = V^T P^T   A = V, B = the lane's own weights (the
//                                    score registers r = key 4g + r)
// and O^T's rows come out as dims (4g + r) * HD/16 + t for tile t: each lane
// ends with HD/4 consecutive dims of its query.  Keys past a query's position
// weigh 0 and their V rows are clamped to rows the tile may read.  The
// uniform fallback applies when no finite positive total remains.
template <int HD>
__global__ __launch_bounds__(256, 3) void attention_tile_kernel(const float *__restrict__ q,
                                                             const float *__restrict__ k_cache,
                                                             const float *__restrict__ v_cache,
                                                             int T, int start, int nh, int nkv,
                                                             float scale, f16 *__restrict__ out,
                                                             f16 *__restrict__ out_lo) {
  constexpr int DPL = HD / 4;  // head dims per lane in S (32 contraction steps at 128)
  constexpr int NT = HD / 16;  // 16-dim output tiles of O^T
  __shared__ float so[4][16][HD + 4];
  __shared__ float sm[4][16], sl[4][16];
  const int q0 = (gridDim.x - 1 - blockIdx.x) * 16;  // the longest tiles start first
  const int h = blockIdx.y, kvh = h / (nh / nkv), kvw = nkv * HD;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int pmax = start + min(q0 + 15, T - 1);
  const int pq = start + min(q0 + i, T - 1);  // rows past T mask as the last row
  float qv[DPL];
  {
    const float *qp = q + (size_t)min(q0 + i, T - 1) * nh * HD + h * HD + g * DPL;
#pragma unroll
    for (int d = 0; d < DPL; d += 4) *reinterpret_cast<float4 *>(qv + d) = *reinterpret_cast<const float4 *>(qp + d);
  }
  const float *kc = k_cache + (size_t)kvh * HD + g * DPL;
  const float *vc = v_cache + (size_t)kvh * HD + i * NT;
  f32x4 o[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float M = -INFINITY, L = 0.f;
  const int nb = pmax / 16 + 1;
  // The K rows of a block are loaded as soon as the previous block's scores
  // are computed and its V rows once its output products are issued, so each
  // load's latency overlaps the other half of an iteration.
  float kk[DPL], vv[4][NT];
  auto load_k = [&](int key0) {
    const float *kp = kc + (size_t)min(key0 + i, pmax) * kvw;
#pragma unroll
    for (int d = 0; d < DPL; d += 4) *reinterpret_cast<float4 *>(kk + d) = *reinterpret_cast<const float4 *>(kp + d);
  };
  auto load_v = [&](int key0) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const float *vp = vc + (size_t)min(key0 + 4 * g + s, pmax) * kvw;
#pragma unroll
      for (int t = 0; t < NT; t += (NT >= 4 ? 4 : NT)) {
        if constexpr (NT >= 4)
          *reinterpret_cast<float4 *>(&vv[s][t]) = *reinterpret_cast<const float4 *>(vp + t);
        else if constexpr (NT == 2)
          *reinterpret_cast<float2 *>(&vv[s][t]) = *reinterpret_cast<const float2 *>(vp + t);
        else
          vv[s][t] = vp[t];
      }
    }
  };
  if (wave < nb) {
    load_k(wave * 16);
    load_v(wave * 16);
  }
  for (int b = wave; b < nb; b += 4) {
    const int key0 = b * 16;
    // Two independent chains over the head dims (d mod 2), summed at the end.
    f32x4 sp[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int d = 0; d < DPL; d++) sp[d & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[d], qv[d], sp[d & 1], 0, 0, 0);
    const f32x4 st = sp[0] + sp[1];
    if (b + 4 < nb) load_k(key0 + 64);
    float sc[4], mc = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      sc[r] = key0 + 4 * g + r <= pq ? st[r] * scale : -INFINITY;
      mc = fmaxf(mc, sc[r]);
    }
    mc = fmaxf(mc, lane_partner(mc, 16));
    mc = fmaxf(mc, lane_partner(mc, 32));
    const float Mn = fmaxf(M, mc);
    const bool live = Mn != -INFINITY;
    const float alpha = live ? expf(M - Mn) : 1.f;
    float pw[4], ls = 0.f;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      pw[r] = live ? expf(sc[r] - Mn) : 0.f;
      ls += pw[r];
    }
    L = L * alpha + ls;
    M = Mn;
#pragma unroll
    for (int t = 0; t < NT; t++) {
      o[t] *= alpha;
#pragma unroll
      for (int s = 0; s < 4; s++) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[s][t], pw[s], o[t], 0, 0, 0);
    }
    if (b + 4 < nb) load_v(key0 + 64);
  }
  L += lane_partner(L, 16);
  L += lane_partner(L, 32);
  if (g == 0) {
    sm[wave][i] = M;
    sl[wave][i] = L;
  }
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) so[wave][i][(4 * g + r) * NT + t] = o[t][r];
  __syncthreads();
  // Merge: thread -> query qi, dims c*NT ... c*NT + NT - 1.
  const int qi = threadIdx.x >> 4, c = threadIdx.x & 15;
  if (q0 + qi >= T) return;
  float Mt = -INFINITY;
#pragma unroll
  for (int w = 0; w < 4; w++) Mt = fmaxf(Mt, sm[w][qi]);
  float Lt = 0.f, acc[NT];
#pragma unroll
  for (int e = 0; e < NT; e++) acc[e] = 0.f;
#pragma unroll
  for (int w = 0; w < 4; w++) {
    const float mw = sm[w][qi];
    const float f = mw == -INFINITY ? 0.f : expf(mw - Mt);
    Lt += sl[w][qi] * f;
#pragma unroll
    for (int e = 0; e < NT; e++) acc[e] += so[w][qi][c * NT + e] * f;
  }
  const int p = start + q0 + qi;
  const size_t at = (size_t)(q0 + qi) * nh * HD + h * HD + c * NT;
  if (isfinite(Lt) && Lt > 0.f) {
#pragma unroll
    for (int e = 0; e < NT; e++) split_f16(acc[e] / Lt, out[at + e], out_lo[at + e]);
  } else {
    const float *vp = v_cache + (size_t)kvh * HD + c * NT;
    for (int e = 0; e < NT; e++) {
      float vs = 0.f;
      for (int j = 0; j <= p; j++) vs += vp[(size_t)j * kvw + e];
      split_f16(vs / (float)(p + 1), out[at + e], out_lo[at + e]);
    }
  }
}

typedef _Float16 half4v __attribute__((ext_vector_type(4)));

// One layer's cache rows of positions [0, P) as f16 hi/lo planes for
// attention_f16_kernel, in blocks of 16 positions (16 * kvw halves a block
// and plane) laid out so that each MFMA operand load of a 16-key block reads
// one contiguous run:
//   K: [block][dim / 32][position % 16][dim % 32]
//   V: [block][dim][position % 16]      (V transposed within the block)
// Positions P .. P16 - 1 (P16 = P rounded up to 16) are zeros, so every block
// a query tile reads holds finite values.  kvw is a multiple of 32.  A
// workgroup moves one block of 16 positions x 64 dims, V through LDS.
__device__ __forceinline__ size_t kblk_index(int pos, int dim, int kvw) {
  return (size_t)(pos >> 4) * 16 * kvw + (size_t)(dim >> 5) * 512 + (pos & 15) * 32 + (dim & 31);
}
__device__ __forceinline__ size_t vblk_index(int pos, int dim, int kvw) {
  return (size_t)(pos >> 4) * 16 * kvw + (size_t)dim * 16 + (pos & 15);
}

__global__ __launch_bounds__(256) void kv_split_f16_kernel(const float *__restrict__ k,
                                                           const float *__restrict__ v, int kvw, int P,
                                                           f16 *__restrict__ kh, f16 *__restrict__ kl,
                                                           f16 *__restrict__ vh, f16 *__restrict__ vl) {
  __shared__ float tile[16][65];
  const int p0 = blockIdx.x * 16, d0 = blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int pl = ty * 4 + r, pos = p0 + pl, dim = d0 + tx;
    float kx = 0.f, vx = 0.f;
    if (pos < P && dim < kvw) {
      kx = k[(size_t)pos * kvw + dim];
      vx = v[(size_t)pos * kvw + dim];
    }
    if (dim < kvw) {
      const size_t o = kblk_index(pos, dim, kvw);
      split_f16(kx, kh[o], kl[o]);
    }
    tile[pl][tx] = vx;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; r++) {  // 16 consecutive positions of 16 consecutive dims: 512 contiguous bytes
    const int pl = threadIdx.x & 15, dl = r * 16 + (threadIdx.x >> 4), dim = d0 + dl;
    if (dim < kvw) {
      const size_t o = vblk_index(p0 + pl, dim, kvw);
      split_f16(tile[pl][dl], vh[o], vl[o]);
    }
  }
}

// Split-half RoPE (src/model.rs:87-95) of 16 positions' rows of one head, by
// absolute position: blockIdx.y a query head (in place), a key head (into the
// cache, KVCache::update, src/cache.rs:38-53) or a value head (copied to the
// cache).  With kh set, the new rows also go to the f16 planes that
// kv_split_f16_kernel describes (earlier rows are its job), with zeros after the
// last one in its block.  Sixteen lanes a position.  Bound by a launch's own
// time: 5.1 us for 24 tokens of 28 + 4 heads of 128, where a workgroup a token
// and a kv_split_f16_kernel over all rows after it took 5.4 + 4.4.
template <int HD>
__global__ __launch_bounds__(256) void rope_append_kernel(float *__restrict__ q, const float *__restrict__ k,
                                                          const float *__restrict__ v,
                                                          const float *__restrict__ rope, int T, int start, int nh,
                                                          int nkv, float *__restrict__ k_cache,
                                                          float *__restrict__ v_cache, f16 *__restrict__ kh,
                                                          f16 *__restrict__ kl, f16 *__restrict__ vh,
                                                          f16 *__restrict__ vl) {
  constexpr int half = HD / 2, P = HD >= 32 ? HD / 32 : 1;  // pairs a lane
  __shared__ float tile[16][HD + 1];
  const int kvw = nkv * HD, y = blockIdx.y, c = threadIdx.x & 15, tl = threadIdx.x >> 4;
  const int p0 = (start & ~15) + 16 * blockIdx.x, pos = p0 + tl, t = pos - start;
  const bool in = t >= 0 && t < T;
  if (y < nh + nkv) {
    const bool is_q = y < nh;
    const int d0 = (is_q ? y : y - nh) * HD;  // the head's first column
    const float *src = is_q ? q + (size_t)t * nh * HD + d0 : k + (size_t)t * kvw + d0;
    const float *cs = rope + (size_t)pos * HD, *sn = cs + half;
#pragma unroll
    for (int e = 0; e < P; e++) {
      const int j = c * P + e;
      if (HD == 16 && j >= half) continue;
      float a = 0.f, b = 0.f;
      if (in) {
        const float re = src[j], im = src[j + half];
        a = re * cs[j] - im * sn[j];
        b = re * sn[j] + im * cs[j];
        float *dst = is_q ? q + (size_t)t * nh * HD + d0 : k_cache + (size_t)pos * kvw + d0;
        dst[j] = a;
        dst[j + half] = b;
      }
      if (kh && !is_q && t >= 0) {
        const size_t o = kblk_index(pos, d0 + j, kvw), o2 = kblk_index(pos, d0 + j + half, kvw);
        split_f16(a, kh[o], kl[o]);
        split_f16(b, kh[o2], kl[o2]);
      }
    }
    return;
  }
  const int d0 = (y - nh - nkv) * HD;
#pragma unroll
  for (int e = 0; e < HD / 16; e++) {
    const int d = c + 16 * e;
    const float x = in ? v[(size_t)t * kvw + d0 + d] : 0.f;
    if (in) v_cache[(size_t)pos * kvw + d0 + d] = x;
    if (kh) tile[tl][d] = x;
  }
  if (!kh) return;
  __syncthreads();
  for (int i = threadIdx.x; i < 2 * HD; i += 256) {  // a dim's 16 positions in one plane: 32 contiguous bytes
    const int d = i % HD;
    f16 *plane = i < HD ? vh : vl;
    half8 w[2];
#pragma unroll
    for (int r = 0; r < 16; r++) {
      f16 hi, lo;
      split_f16(tile[r][d], hi, lo);
      w[r >> 3][r & 7] = i < HD ? hi : lo;
    }
    f16 *dst = plane + vblk_index(p0, d0 + d, kvw);
    if (p0 >= start) {
      reinterpret_cast<half8 *>(dst)[0] = w[0];
      reinterpret_cast<half8 *>(dst)[1] = w[1];
    } else {
#pragma unroll
      for (int r = 0; r < 16; r++)
        if (p0 + r >= start) dst[r] = w[r >> 3][r & 7];
    }
  }
}

// attention_tile_kernel's tiles, order, online softmax and merge with f16
// matrix products: q, K, V and the softmax weights as hi + lo pairs and three
// MFMAs per product (hi*hi, hi*lo, lo*hi), accumulated in f32.  Scores: S^T =
// K Q^T in v_mfma_f32_16x16x32_f16 steps of 32 head dims (K rows from kh/kl);
// output: O^T = V^T P^T in v_mfma_f32_16x16x16_f16 steps of 16 keys (V^T rows
// from vth/vtl, 16 output dims a tile).  One score step covers 32 dims where
// the f32 kernel's covers 4, which moves the kernel off the matrix cores'
// f32 rate.  HD >= 32.
// QT tiles of 16 query rows a workgroup share the K and V loads, which bound the
// kernel (16 KB from L2 per tile and 16 keys: 13 TB/s with one tile).
template <int HD, int QT>
__global__ __launch_bounds__(256, QT == 1 ? 3 : 2) void attention_f16_kernel(const float *__restrict__ q,
                                                            const f16 *__restrict__ kh,
                                                            const f16 *__restrict__ kl,
                                                            const f16 *__restrict__ vh,
                                                            const f16 *__restrict__ vl,
                                                            const float *__restrict__ v_cache, int T,
                                                            int start, int nh, int nkv, float scale,
                                                            f16 *__restrict__ out, f16 *__restrict__ out_lo,
                                                            f16 *__restrict__ xs, f16 *__restrict__ xs_lo, int ldxs) {
  constexpr int NC = HD / 32;  // 32-dim score steps
  constexpr int NT = HD / 16;  // 16-dim output tiles
  __shared__ float so[4][16][HD + 4];
  __shared__ float sm[4][16], sl[4][16];
  const int q0 = (gridDim.x - 1 - blockIdx.x) * 16 * QT;  // the longest tiles start first
  const int h = blockIdx.y, kvh = h / (nh / nkv), kvw = nkv * HD;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int pmax = start + min(q0 + 16 * QT - 1, T - 1);
  int pq[QT];  // rows past T mask as the last row
  half8 qh[QT][NC], ql[QT][NC];
#pragma unroll
  for (int u = 0; u < QT; u++) {
    const int row = min(q0 + 16 * u + i, T - 1);
    pq[u] = start + row;
    const float *qp = q + (size_t)row * nh * HD + h * HD + 8 * g;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const float4 a = *reinterpret_cast<const float4 *>(qp + 32 * c);
      const float4 b = *reinterpret_cast<const float4 *>(qp + 32 * c + 4);
      const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int e = 0; e < 8; e++) {
        f16 hi, lo;
        split_f16(x[e], hi, lo);
        qh[u][c][e] = hi;
        ql[u][c][e] = lo;
      }
    }
  }
  // Lane (i, g): K of key 16 b + i, dims 32 c + 8 g ...; V^T row (dim) 16 t + i,
  // keys 16 b + 4 g ... (kv_split_f16_kernel's block layout; 16 * kvw halves a block).
  const size_t ko = (size_t)kvh * (HD / 32) * 512 + i * 32 + 8 * g;
  const size_t vo = (size_t)(kvh * HD + i) * 16 + 4 * g;
  f32x4 o[QT][NT];
  float M[QT], L[QT];
#pragma unroll
  for (int u = 0; u < QT; u++) {
    M[u] = -INFINITY;
    L[u] = 0.f;
#pragma unroll
    for (int t = 0; t < NT; t++) o[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int nb = pmax / 16 + 1;
  half8 kah[NC], kal[NC];
  half4v vah[NT], val[NT];
  auto load_k = [&](int key0) {
    const size_t r = (size_t)key0 * kvw + ko;  // key0 / 16 blocks of 16 * kvw
#pragma unroll
    for (int c = 0; c < NC; c++) {
      kah[c] = *reinterpret_cast<const half8 *>(kh + r + 512 * c);
      kal[c] = *reinterpret_cast<const half8 *>(kl + r + 512 * c);
    }
  };
  auto load_v = [&](int key0) {
    const size_t r = (size_t)key0 * kvw + vo;
#pragma unroll
    for (int t = 0; t < NT; t++) {
      vah[t] = *reinterpret_cast<const half4v *>(vh + r + 256 * t);
      val[t] = *reinterpret_cast<const half4v *>(vl + r + 256 * t);
    }
  };
  if (wave < nb) {
    load_k(wave * 16);
    load_v(wave * 16);
  }
  for (int b = wave; b < nb; b += 4) {
    const int key0 = b * 16;
    f32x4 st[QT];
#pragma unroll
    for (int u = 0; u < QT; u++) {
      f32x4 s0 = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
      for (int c = 0; c < NC; c++) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kal[c], qh[u][c], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kah[c], ql[u][c], s1, 0, 0, 0);
        s0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(kah[c], qh[u][c], s0, 0, 0, 0);
      }
      st[u] = s0 + s1;
    }
    if (b + 4 < nb) load_k(key0 + 64);
#pragma unroll
    for (int u = 0; u < QT; u++) {
      float sc[4], mc = -INFINITY;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        sc[r] = key0 + 4 * g + r <= pq[u] ? st[u][r] * scale : -INFINITY;
        mc = fmaxf(mc, sc[r]);
      }
      mc = fmaxf(mc, lane_partner(mc, 16));
      mc = fmaxf(mc, lane_partner(mc, 32));
      const float Mn = fmaxf(M[u], mc);
      const bool live = Mn != -INFINITY;
      const float alpha = live ? expf(M[u] - Mn) : 1.f;
      float ls = 0.f;
      half4v ph, pl;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float pw = live ? expf(sc[r] - Mn) : 0.f;
        ls += pw;
        f16 hi, lo;
        split_f16(pw, hi, lo);
        ph[r] = hi;
        pl[r] = lo;
      }
      L[u] = L[u] * alpha + ls;
      M[u] = Mn;
#pragma unroll
      for (int t = 0; t < NT; t++) {
        o[u][t] *= alpha;
        o[u][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(val[t], ph, o[u][t], 0, 0, 0);
        o[u][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(vah[t], pl, o[u][t], 0, 0, 0);
        o[u][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(vah[t], ph, o[u][t], 0, 0, 0);
      }
    }
    if (b + 4 < nb) load_v(key0 + 64);
  }
#pragma unroll
  for (int u = 0; u < QT; u++) {
    if (u) __syncthreads();  // the tile before has been merged
    L[u] += lane_partner(L[u], 16);
    L[u] += lane_partner(L[u], 32);
    if (g == 0) {
      sm[wave][i] = M[u];
      sl[wave][i] = L[u];
    }
    // D layout of O^T: lane (i, g) holds query i, dims 16 t + 4 g + r.
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) so[wave][i][16 * t + 4 * g + r] = o[u][t][r];
    __syncthreads();
    // Merge: thread -> query qi, dims c*NT ... c*NT + NT - 1.
    const int qi = threadIdx.x >> 4, c = threadIdx.x & 15;
    if (q0 + 16 * u + qi >= T) continue;
    float Mt = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; w++) Mt = fmaxf(Mt, sm[w][qi]);
    float Lt = 0.f, acc[NT];
#pragma unroll
    for (int e = 0; e < NT; e++) acc[e] = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const float mw = sm[w][qi];
      const float f = mw == -INFINITY ? 0.f : expf(mw - Mt);
      Lt += sl[w][qi] * f;
#pragma unroll
      for (int e = 0; e < NT; e++) acc[e] += so[w][qi][c * NT + e] * f;
    }
    const int p = start + q0 + 16 * u + qi;
    const size_t at = (size_t)(q0 + 16 * u + qi) * nh * HD + h * HD + c * NT;
    float sum = 0.f;
    auto emit = [&](int e, float v) {
      f16 hi, lo;
      split_f16(v, hi, lo);
      out[at + e] = hi;
      out_lo[at + e] = lo;
      sum += (float)hi + (float)lo;
    };
    if (isfinite(Lt) && Lt > 0.f) {
#pragma unroll
      for (int e = 0; e < NT; e++) emit(e, acc[e] / Lt);
    } else {
      const float *vp = v_cache + (size_t)kvh * HD + c * NT;
      for (int e = 0; e < NT; e++) {
        float vs = 0.f;
        for (int j = 0; j <= p; j++) vs += vp[(size_t)j * kvw + e];
        emit(e, vs / (float)(p + 1));
      }
    }
    // The output's 32-column sums, 32 / NT lanes of the query's 16: in a pass of
    // their own (xsum_f16_kernel) they took 4.4 us for 24 tokens; nothing here.
    if (xs) {
#pragma unroll
      for (int b = 1; b < 32 / NT; b <<= 1) sum += lane_partner(sum, b);
      if (c % (32 / NT) == 0) {
        const size_t o = (size_t)(q0 + 16 * u + qi) * ldxs + (h * HD + c * NT) / 32;
        split_f16(sum, xs[o], xs_lo[o]);
      }
    }
  }
}

// With xs set (cols, the row length, a multiple of 32): the activation sums
// of the output as rmsnorm_rows_f16_kernel writes them.
__global__ __launch_bounds__(256) void swiglu_f16_kernel(const float *__restrict__ g, const float *__restrict__ u,
                                                         f16 *__restrict__ out, f16 *__restrict__ out_lo,
                                                         size_t n, int cols, f16 *__restrict__ xs,
                                                         f16 *__restrict__ xs_lo, int ldxs) {
#pragma clang fp contract(off)
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  float v = 0.f;
  if (i < n) {
    const float x = g[i];
    f16 h, l;
    split_f16((x / (1.0f + expf(-x))) * u[i], h, l);
    out[i] = h;
    out_lo[i] = l;
    v = (float)h + (float)l;
  }
  const size_t i32 = i & ~(size_t)31;  // the half-wave's first element: n is a multiple of 32 with xs
  if (xs && i32 < n) {
    const size_t row = i32 / (size_t)cols;
    half_wave_xsum(v, (int)(i32 - row * cols), xs + row * ldxs, xs_lo + row * ldxs);
  }
}



// C[t][j] = (C[t][j] when accumulating, else bias[j] or 0) + the split-K
// partials of splits 0, 1, ..., ksplit - 1, added in that order.
__global__ void split_reduce_kernel(float *__restrict__ c, int ldc, const float *__restrict__ bias,
                                    const float *__restrict__ part, int n, int t, int ksplit,
                                    int accumulate) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (j >= n || r >= t) return;
  float *cp = c + (size_t)r * ldc + j;
  float v = accumulate ? *cp : (bias ? bias[j] : 0.f);
  for (int z = 0; z < ksplit; z++) v += part[((size_t)z * t + r) * n + j];
  *cp = v;
}

// split_reduce_kernel for a dual gate/up product: row f of gate is virtual
// column (f / 64) * 128 + f % 64, of up that + 64; h + hl [t][f] = silu(g) * u
// of the partial sums (split order), as the dual products write it, and with xso
// the 32-column sums (half_wave_xsum).
__global__ __launch_bounds__(256) void split_reduce_swiglu_kernel(const float *__restrict__ part, int nv, int t_rows,
                                                                  int ksplit, int rows, f16 *__restrict__ h,
                                                                  f16 *__restrict__ hl, int ldh,
                                                                  f16 *__restrict__ xso, f16 *__restrict__ xso_lo,
                                                                  int ldxso) {
#pragma clang fp contract(off)
  const int f = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y;
  float v = 0.f;
  if (f < rows) {
    const size_t vg = (size_t)(f >> 6) * 128 + (f & 63), zs = (size_t)t_rows * nv;
    const float *p = part + (size_t)t * nv;
    float x = 0.f, u = 0.f;
    for (int z = 0; z < ksplit; z++) {
      x += p[z * zs + vg];
      u += p[z * zs + vg + 64];
    }
    f16 hi, lo;
    split_f16((x / (1.0f + expf(-x))) * u, hi, lo);
    h[(size_t)t * ldh + f] = hi;
    hl[(size_t)t * ldh + f] = lo;
    v = (float)hi + (float)lo;
  }
  const int f32 = f & ~31;
  if (xso && f32 < rows) half_wave_xsum(v, f32, xso + (size_t)t * ldxso, xso_lo + (size_t)t * ldxso);
}

// split_reduce_kernel for a segmented product: column j of the partials
// belongs to segment i (seg_base[i] <= j < seg_base[i + 1]) and goes to
// seg_c[i] + r * seg_ldc[i] + (j - seg_base[i]), from its bias or 0 (or C
// when accumulating) plus the partials in split order.
struct SegOut {
  float *c[3];
  int ldc[3];
  const float *bias[3];
  int base[4];
  int nseg;
};
__global__ void split_reduce_seg_kernel(SegOut o, const float *__restrict__ part, int n, int t, int ksplit,
                                        int accumulate) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (j >= n || r >= t) return;
  const int s = (o.nseg > 1 && j >= o.base[1]) + (o.nseg > 2 && j >= o.base[2]);
  const int jl = j - o.base[s];
  float *cp = o.c[s] + (size_t)r * o.ldc[s] + jl;
  float v = accumulate ? *cp : (o.bias[s] ? o.bias[s][jl] : 0.f);
  for (int z = 0; z < ksplit; z++) v += part[((size_t)z * t + r) * n + j];
  *cp = v;
}

}  // namespace

namespace {

// Workgroup slots of the device for the GEMM: two workgroups per CU (their
// LDS, 55-74 KB each, allows two).
int gemm_slots() {
  static int slots = 0;
  if (!slots) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
    slots = 2 * cus;
  }
  return slots;
}

// The eight-wave kernel unless LLRS_PREFILL_GEMM=4 asks for the four-wave one
// (for comparisons; read at every launch, so a test can switch it).
bool eight_waves() {
  const char *e = getenv("LLRS_PREFILL_GEMM");
  return !(e && strcmp(e, "4") == 0);
}

void launch_tiles(const PrefillGemmArgs &a, int bm, hipStream_t s) {
  const dim3 grid((unsigned)((a.n + BN - 1) / BN), (unsigned)((a.t + bm - 1) / bm), (unsigned)a.ksplit);
  const size_t lds = (size_t)2 * (bm + BN) * LS * sizeof(f16);
  const bool w8 = eight_waves();
#define GEMM8(T)                                                                           \
  if (bm == 128)                                                                           \
    hipLaunchKernelGGL((prefill_gemm8_kernel<T, 128>), grid, dim3(512), lds, s, a); \
  else                                                                                     \
    hipLaunchKernelGGL((prefill_gemm8_kernel<T, 64>), grid, dim3(512), lds, s, a);
#define GEMM4(T)                                                                       \
  if (bm == 128)                                                                       \
    hipLaunchKernelGGL((prefill_gemm_kernel<T, 128>), grid, dim3(256), lds, s, a);     \
  else                                                                                 \
    hipLaunchKernelGGL((prefill_gemm_kernel<T, 64>), grid, dim3(256), lds, s, a);
  if (w8) {
    switch (a.type) {
      case LLRS_Q4_K: GEMM8(LLRS_Q4_K) break;
      case LLRS_Q6_K: GEMM8(LLRS_Q6_K) break;
      case LLRS_Q8_0: GEMM8(LLRS_Q8_0) break;
      case LLRS_Q5_0: GEMM8(LLRS_Q5_0) break;
      case LLRS_F16: GEMM8(LLRS_F16) break;
      case LLRS_BF16: GEMM8(LLRS_BF16) break;
      case LLRS_F32: GEMM8(LLRS_F32) break;
      default: GEMM8(0xffffffffu) break;
    }
    return;
  }
  switch (a.type) {
    case LLRS_Q4_K: GEMM4(LLRS_Q4_K) break;
    case LLRS_Q6_K: GEMM4(LLRS_Q6_K) break;
    case LLRS_Q8_0: GEMM4(LLRS_Q8_0) break;
    case LLRS_Q5_0: GEMM4(LLRS_Q5_0) break;
    default: GEMM4(0xffffffffu) break;
  }
#undef GEMM4
#undef GEMM8
}

// The tiles of `a` (bm tokens each; -r: register-decoded, r row waves a group) with K
// split over `ksplit` workgroups, then the fixed-order reduction of their
// partials into C.
int launch_split(PrefillGemmArgs a, int bm, int ksplit, hipStream_t s) {
  a.ksplit = ksplit;
  if (ksplit > 1) {
    if (!a.part || (size_t)ksplit * a.t * a.n > a.part_cap)
      return set_error(LLRS_E_INVALID, "prefill GEMM: split-K scratch of %zu floats is too small (%d x %d x %d)",
                       a.part_cap, ksplit, a.t, a.n);
  }
  if (bm > 0)
    launch_tiles(a, bm, s);
  else
    launch_prefill_reg(a, -bm, s);
  if (ksplit > 1 && a.w2)
    hipLaunchKernelGGL(split_reduce_swiglu_kernel, dim3((unsigned)((a.dual_rows + 255) / 256), (unsigned)a.t),
                       dim3(256), 0, s, a.part, a.n, a.t, ksplit, a.dual_rows, a.h, a.hl, a.ldh, a.xso, a.xso_lo,
                       a.ldxso);
  else if (ksplit > 1 && a.nseg > 0) {
    SegOut o{};
    o.nseg = a.nseg;
    for (int i = 0; i < a.nseg; i++) {
      o.c[i] = a.seg_c[i];
      o.ldc[i] = a.seg_ldc[i];
      o.bias[i] = a.seg_bias[i];
    }
    for (int i = 0; i <= a.nseg; i++) o.base[i] = a.seg_base[i];
    hipLaunchKernelGGL(split_reduce_seg_kernel, dim3((unsigned)((a.n + 255) / 256), (unsigned)a.t), dim3(256), 0,
                       s, o, a.part, a.n, a.t, ksplit, a.accumulate);
  } else if (ksplit > 1)
    hipLaunchKernelGGL(split_reduce_kernel, dim3((unsigned)((a.n + 255) / 256), (unsigned)a.t), dim3(256), 0,
                       s, a.c, a.ldc, a.bias, a.part, a.n, a.t, ksplit, a.accumulate);
  return LLRS_OK;
}

}  // namespace

size_t prefill_split_scratch_floats() { return (size_t)gemm_slots() * BN * 128; }

bool prefill_codes_enabled() {
  const char *e = getenv("LLRS_PREFILL_CODES");
  return eight_waves() && !(e && strcmp(e, "f32") == 0);
}

int launch_xsum_f16(const f16 *a, const f16 *a_lo, int lda, int k, int T, f16 *xs, f16 *xs_lo, int ldxs,
                    hipStream_t s) {
  if (k % 32 || lda % 8 || T <= 0 || ldxs < k / 32)
    return set_error(LLRS_E_UNSUPPORTED, "activation sums over %d columns (lda %d, ldxs %d)", k, lda, ldxs);
  const int nsub = k / 32;
  hipLaunchKernelGGL(xsum_f16_kernel, dim3((unsigned)((nsub + 63) / 64), (unsigned)T), dim3(64), 0, s, a,
                     a_lo, lda, nsub, xs, xs_lo, ldxs);
  LLRS_HIP(hipGetLastError());
  return LLRS_OK;
}

// Whether a product of 16-bit weights (nothing to decode) is better off with the
// LDS-staged kernel's 128-token tiles: from 16 of a row wave's tiles (32 rows x up
// to 64 tokens) a CU (four layers of the 7B shape in BF16, 900 tokens: 6,145
// against 7,326 us; of 1.5B in F16, 900: 2,574 against 2,045).
static bool many_half_tiles(uint32_t type, int rows, int t) {
  if (type != LLRS_F16 && type != LLRS_BF16) return false;
  const int tt = prefill_reg_token_tile(type, t);
  return (long)((rows + 31) / 32) * ((t + tt - 1) / tt) >= 8L * gemm_slots();
}

bool prefill_fuses(uint32_t type, size_t row_bytes, int rows, int t) {
  if (!prefill_codes_enabled() || !prefill_reg_supports(type)) return false;
  if ((uint64_t)row_bytes * (uint64_t)rows >= 1ull << 32) return false;  // its rows' offsets are 32-bit words
  return !many_half_tiles(type, rows, t);
}

// The rows of `g` from `from` on (a multiple of 64 of a dual product's gate
// rows), `rows` of them (of each matrix).
static PrefillGemmArgs rows_of(const PrefillGemmArgs &g, int from, int rows) {
  PrefillGemmArgs r = g;
  r.w = g.w + (size_t)from * (size_t)g.row_bytes;
  if (g.w2) {
    r.w2 = g.w2 + (size_t)from * (size_t)g.row_bytes;
    r.dual_rows = rows;
    r.n = 2 * rows;
    r.h = g.h + from;
    r.hl = g.hl + from;
    if (g.xso) {
      r.xso = g.xso + from / 32;
      r.xso_lo = g.xso_lo + from / 32;
    }
  } else {
    r.n = rows;
    r.c = g.c + from;
    r.bias = g.bias ? g.bias + from : nullptr;
  }
  return r;
}

// Whether the many-token kernel takes a register-decoded product: past one
// 64-token tile, unless its tiles neither fill three quarters of the slots nor
// leave room to split K (measured with workgroups of half the waves: 7B gate/up
// over 128 tokens, 296 tiles for 512 slots, 137 us against 112; over 256, 187
// against 214).  Q6_K ffn_down of 7B over 128
// tokens: 78 us against 96, q and k over 256: 31 against 35, over 128 equal.
static bool takes_big(const PrefillGemmArgs &g) {
  if (g.t <= 64 || g.type == LLRS_F16 || g.type == LLRS_BF16) return false;
  const int tile = prefill_reg_big_row_tile(g.type, g.w2 != nullptr), rows = g.w2 ? g.dual_rows : g.n;
  const long tiles = (long)((rows + tile - 1) / tile) * ((g.t + 63) / 64), slots = gemm_slots() / 2;
  return 2 * tiles <= slots || 4 * tiles >= 3 * slots;
}

// Register-decoded products over many tokens, one workgroup a CU: whole rounds
// of tiles run as they are; a last round that would fill at most half the
// slots (or a product with fewer tiles than slots) splits K over them.
static int launch_reg_big(const PrefillGemmArgs &g, hipStream_t s) {
  const int slots = gemm_slots() / 2, nb = (g.k + 255) / 256;
  const int tile = prefill_reg_big_row_tile(g.type, g.w2 != nullptr), rows = g.w2 ? g.dual_rows : g.n;
  const int nt = (rows + tile - 1) / tile, mt = (g.t + 63) / 64;
  auto splits = [&](int tiles, int n) {
    const int ks = std::max(1, std::min({slots / tiles, nb, (int)(g.part_cap / ((size_t)g.t * n))}));
    const int per = (nb + ks - 1) / ks;
    return (nb + per - 1) / per;
  };
  const int per_round = slots / mt;  // row tiles per round of slots
  const int full = per_round > 0 && g.nseg == 0 ? nt / per_round * per_round : 0, rem = nt - full;
  if (full > 0 && rem > 0 && rem * mt * 2 <= slots) {
    PrefillGemmArgs m = rows_of(g, 0, full * tile);
    m.ksplit = 1;
    launch_prefill_reg(m, 0, s);
    const PrefillGemmArgs r = rows_of(g, full * tile, rows - full * tile);
    return launch_split(r, 0, splits(rem * mt, r.n), s);
  }
  return launch_split(g, 0, nt * mt < slots ? splits(nt * mt, g.n) : 1, s);
}

// The register-decoded products, one workgroup a CU.  Its row waves (1 to 5 a
// group) and the K ranges (whole rounds of 512 columns) are those for which
// the CUs' passes x (rounds x waves per SIMD + a start of two) come out least.
static int launch_reg(const PrefillGemmArgs &g, hipStream_t s) {
  const int cus = gemm_slots() / 2, nu = (g.k + 511) / 512;
  const int tile = prefill_reg_row_tile(g.w2 != nullptr), tt = prefill_reg_token_tile(g.type, g.t);
  const int rows = g.w2 ? g.dual_rows : g.n, mt = (g.t + tt - 1) / tt;
  int best = INT_MAX, row_waves = 1, per = nu;
  for (int rw = prefill_reg_max_row_waves(); rw >= 1; rw--) {
    if (g.w2 && g.xso && rw % 2) continue;  // sums of 32 columns: pairs of waves
    const int wgs = (rows + tile * rw - 1) / (tile * rw) * mt;
    const int ks = std::max(1, std::min({cus / wgs, nu, (int)(g.part_cap / ((size_t)g.t * g.n))}));
    const int rounds = (nu + ks - 1) / ks, passes = (wgs * ((nu + rounds - 1) / rounds) + cus - 1) / cus;
    const int cost = passes * (rounds * ((rw + 2) / 2) + 2);
    if (cost < best) {
      best = cost;
      row_waves = rw;
      per = rounds;
    }
  }
  // The kernel cuts ceil(blocks / ksplit) 256-column blocks a range; 2 per of
  // them leave its last range short, never empty.
  const int nb = (g.k + 255) / 256;
  return launch_split(g, -row_waves, (nb + 2 * per - 1) / (2 * per), s);
}

int launch_prefill_gemm(const PrefillGemmArgs &g, hipStream_t s) {
  if (g.k % 32 || g.lda % 8 || g.n <= 0 || g.k <= 0 || g.t <= 0)
    return set_error(LLRS_E_UNSUPPORTED, "prefill GEMM shape %d x %d (lda %d) is not supported", g.n,
                     g.k, g.lda);
  if (g.xs && (g.type != LLRS_Q4_K || g.k % 256 || g.ldxs % 8 || g.ldxs < g.k / 32))
    return set_error(LLRS_E_UNSUPPORTED, "prefill GEMM: activation sums (ldxs %d) for a type %u product of %d columns",
                     g.ldxs, g.type, g.k);
  const bool reg = prefill_fuses(g.type, (size_t)g.row_bytes, g.n, g.t) && (g.type != LLRS_Q4_K || g.xs);
  if (g.w2 && (!reg || g.dual_rows <= 0 || g.dual_rows % 64 || g.n != 2 * g.dual_rows || !g.h || !g.hl ||
               (g.xso && g.ldxso < g.dual_rows / 32)))
    return set_error(LLRS_E_UNSUPPORTED, "prefill GEMM: dual gate/up product of %d rows is not supported", g.dual_rows);
  if (g.nseg > 0 && (!reg || g.nseg > 3 || g.seg_base[0] != 0 || g.seg_base[g.nseg] != g.n))
    return set_error(LLRS_E_UNSUPPORTED, "prefill GEMM: segmented product of %d segments is not supported", g.nseg);
  for (int i = 1; i < g.nseg; i++)
    if (g.seg_base[i] % BN || g.seg_base[i] <= g.seg_base[i - 1])
      return set_error(LLRS_E_UNSUPPORTED, "prefill GEMM: segment boundary %d is not a multiple of %d", g.seg_base[i], BN);
  if (reg) {
    LLRS_TRY(takes_big(g) ? launch_reg_big(g, s) : launch_reg(g, s));
    LLRS_HIP(hipGetLastError());
    return LLRS_OK;
  }
  // 128-token tiles when there are enough of them (the dequantized weight
  // tile then serves twice the tokens), else 64.  Products with fewer tiles
  // than half the slots split K over up to 8 workgroups (at least 6 K chunks
  // each).  Otherwise whole rounds of tiles run as they are, and a last
  // round that would fill at most half the slots runs as its own launch with
  // K split over the slots.  Split partials are reduced in split order, so C
  // is the same bit for bit on every run.
  const int slots = gemm_slots();
  const int ntiles = (g.n + BN - 1) / BN;
  const int bm = (g.t >= 256 && ntiles >= kTile128Rows) ? 128 : 64;
  const int mt = (g.t + bm - 1) / bm, chunks = (g.k + KC - 1) / KC;
  int ks = 1;
  while (ks < 8 && ntiles * mt * ks * 2 <= slots && chunks / (ks * 2) >= 6) ks *= 2;
  const int per_round = slots / mt;  // row tiles per round of slots
  const int full = (ks == 1 && per_round > 0) ? ntiles / per_round * per_round : 0;
  const int rem = ntiles - full;
  if (full > 0 && rem > 0 && rem * mt * 2 <= slots) {
    PrefillGemmArgs m = rows_of(g, 0, full * BN);
    m.ksplit = 1;
    launch_tiles(m, bm, s);
    LLRS_TRY(launch_split(rows_of(g, full * BN, g.n - full * BN), bm,
                          std::max(1, std::min({8, slots / (rem * mt), chunks / 6})), s));
  } else {
    LLRS_TRY(launch_split(g, bm, ks, s));
  }
  LLRS_HIP(hipGetLastError());
  return LLRS_OK;
}

int launch_embed_rows(const llrs_tensor *emb, const uint32_t *tok, int T, float *x, hipStream_t s) {
  const int H = (int)emb->cols;
  hipLaunchKernelGGL(embed_rows_kernel, dim3((H + 255) / 256, T), dim3(256), 0, s, emb->dev,
                     emb->type, emb->row_bytes, H, (uint32_t)emb->rows, tok, T, x);
  LLRS_HIP(hipGetLastError());
  return LLRS_OK;
}

int launch_rmsnorm_rows_f16(const float *x, const float *w, f16 *out, f16 *out_lo, int T, int H,
                            float eps, hipStream_t s, f16 *xs, f16 *xs_lo, int ldxs) {
  if (xs && (H % 32 || ldxs < H / 32))
    return set_error(LLRS_E_UNSUPPORTED, "activation sums over %d columns (ldxs %d)", H, ldxs);
  if (H % 8) return set_error(LLRS_E_UNSUPPORTED, "prefill RMSNorm over %d columns", H);
  const int threads = std::min(1024, (H / 8 + 63) / 64 * 64);
  hipLaunchKernelGGL(rmsnorm_rows_f16_kernel, dim3(T), dim3(threads), 0, s, x, w, out, out_lo, H, eps, xs, xs_lo,
                     ldxs);
  LLRS_HIP(hipGetLastError());
  return LLRS_OK;
}

bool prefill_attention_f16() {
  const char *e = getenv("LLRS_PREFILL_ATTN");
  return !(e && strcmp(e, "f32") == 0);
}

static bool use_f16_planes(const PrefillKvF16 *kvf, int hd) { return kvf && hd >= 32 && prefill_attention_f16(); }

int launch_rope_append(float *q, const float *k, const float *v, const float *rope, int T, int start,
                       int nh, int nkv, int hd, float *k_cache, float *v_cache, hipStream_t s,
                       const PrefillKvF16 *kvf) {
  PrefillKvF16 f{};
  if (use_f16_planes(kvf, hd)) {
    f = *kvf;
    const int kvw = nkv * hd, P = start + T;
    if (((P + 15) & ~15) > f.positions || f.kvw != kvw || kvw % 32)
      return set_error(LLRS_E_INVALID, "prefill attention: f16 K/V scratch of %d positions x %d for %d x %d",
                       f.positions, f.kvw, P, kvw);
    if (start > 0)  // the rows of earlier calls and chunks (the planes serve every layer in turn)
      hipLaunchKernelGGL(kv_split_f16_kernel, dim3((unsigned)((start + 15) / 16), (unsigned)((kvw + 63) / 64)),
                         dim3(256), 0, s, k_cache, v_cache, kvw, start, f.kh, f.kl, f.vh, f.vl);
  }
  const dim3 grid((unsigned)((start + T + 15) / 16 - start / 16), (unsigned)(nh + 2 * nkv));
#define ROPE(D)                                                                                                  \
  hipLaunchKernelGGL(rope_append_kernel<D>, grid, dim3(256), 0, s, q, k, v, rope, T, start, nh, nkv, k_cache, \
                     v_cache, f.kh, f.kl, f.vh, f.vl)
  switch (hd) {
    case 16: ROPE(16); break;
    case 32: ROPE(32); break;
    case 64: ROPE(64); break;
    case 128: ROPE(128); break;
    default: return set_error(LLRS_E_UNSUPPORTED, "attention head_dim %d is not supported", hd);
  }
#undef ROPE
  LLRS_HIP(hipGetLastError());
  return LLRS_OK;
}

int launch_attention_rows(const float *q, const float *k_cache, const float *v_cache, int T,
                          int start, int nh, int nkv, int hd, float scale, f16 *out, f16 *out_lo,
                          hipStream_t s, const PrefillKvF16 *kvf, f16 *xs, f16 *xs_lo, int ldxs) {
  if (T <= 0 || nkv <= 0 || nh % nkv)
    return set_error(LLRS_E_UNSUPPORTED, "attention over %d rows with %d/%d heads", T, nh, nkv);
  const dim3 grid((unsigned)((T + 15) / 16), (unsigned)nh);
  if (use_f16_planes(kvf, hd)) {
    const dim3 grid2((unsigned)((T + 31) / 32), (unsigned)nh);
    // Two tiles of query rows a workgroup while every CU still gets one (fewer
    // would leave CUs idle behind workgroups of twice the length): 2,000 rows of 12
    // heads 169 us against 231 with one, 512 rows of 28 heads 28 against 39.
    const bool two = (long)grid2.x * nh >= gemm_slots() / 2;
#define ATT16(D)                                                                                            \
  if (two)                                                                                                  \
    hipLaunchKernelGGL((attention_f16_kernel<D, 2>), grid2, dim3(256), 0, s, q, kvf->kh, kvf->kl, kvf->vh,  \
                       kvf->vl, v_cache, T, start, nh, nkv, scale, out, out_lo, xs, xs_lo, ldxs);           \
  else                                                                                                      \
    hipLaunchKernelGGL((attention_f16_kernel<D, 1>), grid, dim3(256), 0, s, q, kvf->kh, kvf->kl, kvf->vh,   \
                       kvf->vl, v_cache, T, start, nh, nkv, scale, out, out_lo, xs, xs_lo, ldxs)
    switch (hd) {
      case 32: ATT16(32); break;
      case 64: ATT16(64); break;
      case 128: ATT16(128); break;
      default: return set_error(LLRS_E_UNSUPPORTED, "attention head_dim %d is not supported", hd);
    }
#undef ATT16
    LLRS_HIP(hipGetLastError());
    return LLRS_OK;
  }
#define ATT(D)                                                                                   \
  hipLaunchKernelGGL(attention_tile_kernel<D>, grid, dim3(256), 0, s, q, k_cache, v_cache, T, start, \
                     nh, nkv, scale, out, out_lo)
  switch (hd) {
    case 16: ATT(16); break;
    case 32: ATT(32); break;
    case 64: ATT(64); break;
    case 128: ATT(128); break;
    default: return set_error(LLRS_E_UNSUPPORTED, "attention head_dim %d is not supported", hd);
  }
#undef ATT
  LLRS_HIP(hipGetLastError());
  if (xs) return launch_xsum_f16(out, out_lo, nh * hd, nh * hd, T, xs, xs_lo, ldxs, s);
  return LLRS_OK;
}

int launch_swiglu_f16(const float *g, const float *u, f16 *out, f16 *out_lo, size_t n, int cols, hipStream_t s,
                      f16 *xs, f16 *xs_lo, int ldxs) {
  if (xs && (cols <= 0 || cols % 32 || n % (size_t)cols || ldxs < cols / 32))
    return set_error(LLRS_E_UNSUPPORTED, "activation sums over rows of %d columns (ldxs %d)", cols, ldxs);
  hipLaunchKernelGGL(swiglu_f16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g, u, out,
                     out_lo, n, cols, xs, xs_lo, ldxs);
  LLRS_HIP(hipGetLastError());
  return LLRS_OK;
}


}  // namespace llrs
