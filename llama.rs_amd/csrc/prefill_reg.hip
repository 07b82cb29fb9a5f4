// The batched prefill's matrix products with the weights decoded in registers.
//
// C[t][n] = sum_k A[t][k] W[n][k] (CausalModel::prefill's products,
// src/architecture.rs:60-77; value_at, src/quant.rs:349-456), activations as
// f16 hi + lo pairs, on v_mfma_f32_16x16x32_f16 with f32 sums.
//
// A wave owns a few tiles of 16 weight rows.  It copies their native GGUF
// blocks, 256 columns at a time, through its own part of LDS (no barrier);
// lane (n = lane & 15, kg = lane >> 4) then reads row n's codes of columns 8 kg
// .. 8 kg + 7 of every 32-column step and turns them into the MFMA's operand
// in registers.  The tokens' activations are shared by the waves through LDS
// in fragment order, a few steps at a time, double-buffered; the next weights
// and activations are in flight while the current ones are multiplied.
//
// prefill_reg_kernel (tiles of 16, 32 or 64 tokens): one workgroup a CU, two
// groups of one to five row waves on alternate units of columns, summed
// through LDS at the end, and a staging wave each.  Short prompts are the
// weights' stream plus its decoding: the LDS-staged kernel (prefill.hip) computes
// 64 tokens for any prompt up to 64 and decodes on half its waves behind two
// barriers per 64 columns.  7B shape, 24 tokens, per launch: gate/up 96 -> 39
// us, ffn_down (Q6_K) 84 -> 36, q and k 15.4 -> 10.8, V (Q8_0) 17 -> 6.7.
// What bounds it: the decoding (~14 VALU operations per 16 x 32 weights and
// lane, Q6_K ~30) and the MFMAs, on 2.3 to 3 waves a SIMD.
//
// prefill_reg_big_kernel (64-token tiles of many): see there.
//
// Per type (the operand is always exact in f16):
//   Q4_K  sc * q per column in units of the block's d; dmin * m through the
//         activations' 32-column sums
//   Q6_K  sc * (q - 32) as f16 hi + lo (|.| <= 4,096: three MFMAs), units of d
//   Q8_0, Q5_0  the integer code; each step's sum is scaled by the block's d
//   F16, BF16   the value itself (a BF16 value, 8 significant bits, is exact in
//         f16 from 2^-17 up and rounded to its 2^-24 grid below)
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "prefill.h"
#include "quant_dev.h"
#include "wave_dev.h"

namespace llrs {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#define INLINE __attribute__((always_inline))

__device__ __forceinline__ void split_f16(float v, f16 &hi, f16 &lo) {
  hi = (f16)v;
  lo = (f16)(v - (float)hi);
}

// Four codes (a byte each) as 1024 + code in f16: the bit pattern 0x6400 | code.
__device__ __forceinline__ void biased(uint32_t v, half2v &a, half2v &b) {
  a = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u));
  b = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u));
}
__device__ __forceinline__ half8 join(half2v a, half2v b, half2v c, half2v d) {
  return half8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}
// Byte i of v as 1024 + byte, in both halves.
__device__ __forceinline__ half2v twice(uint32_t v, int i) {
  return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, v, 0x04000400u + (uint32_t)i * 0x00010001u));
}
// Eight codes (v0, v1) minus an integer offset, exact.
__device__ __forceinline__ half8 offset_codes(uint32_t v0, uint32_t v1, float off) {
  const half2v o = {(f16)(-1024.f - off), (f16)(-1024.f - off)};
  half2v a, b, c, d;
  biased(v0, a, b);
  biased(v1, c, d);
  return join(a + o, b + o, c + o, d + o);
}
// Bits 0..3 of t -> bit 4 of bytes 0..3.
__device__ __forceinline__ uint32_t spread4(uint32_t t) { return ((t & 15u) * 0x00204081u & 0x01010101u) << 4; }

// Eight bytes at an even LDS address: three aligned words, realigned.
struct Bytes8 {
  uint32_t w[3], sh;
  __device__ __forceinline__ Bytes8(const uint8_t *p) {
    const uint32_t o = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 3);
    const uint32_t *a = reinterpret_cast<const uint32_t *>(p - o);
    w[0] = a[0];
    w[1] = a[1];
    w[2] = a[2];
    sh = o;
  }
  __device__ __forceinline__ uint32_t lo() const { return __builtin_amdgcn_alignbyte(w[1], w[0], sh); }
  __device__ __forceinline__ uint32_t hi() const { return __builtin_amdgcn_alignbyte(w[2], w[1], sh); }
};

// How a type's products are scaled.
enum Unit { kNone, kBlock, kStep };  // the value itself; d per 256 columns; d per 32 columns

// Row<TY>: one weight row's unit (kCols columns, kBytes) in LDS, for the lane's
// kg.  A row is copied there in kSpan aligned 16-byte pieces (enough for any
// even start, and such that 16 rows kSpan + kPad pieces apart start in distinct
// bank quads).  weight() gives the operand of step s of the unit (and its low
// part).
template <uint32_t TY> struct Row;

// Members that not every type has a use for.
struct RowBase {
  static constexpr int kPlanes = 1, kPad = 0;
  __device__ __forceinline__ float d() const { return 1.f; }
  __device__ __forceinline__ float step_d(int) const { return 1.f; }
  __device__ __forceinline__ float dmin() const { return 0.f; }
  __device__ __forceinline__ uint32_t mins(bool) const { return 0; }
};

template <> struct Row<LLRS_Q4_K> : RowBase {
  static constexpr Unit kUnit = kBlock;
  static constexpr int kCols = 256, kBytes = 144, kSpan = 9;
  const uint8_t *p;
  uint4 hdr;
  __device__ __forceinline__ void open(const uint8_t *row) {
    p = row;
    hdr = *reinterpret_cast<const uint4 *>(row);
  }
  __device__ __forceinline__ float d() const { return f16_bits_to_f32((uint16_t)(hdr.x & 0xffff)); }
  __device__ __forceinline__ float dmin() const { return f16_bits_to_f32((uint16_t)(hdr.x >> 16)); }
  // scale_min_k4 (src/quant.rs:338-347) of sub-blocks 0-3 or 4-7, a byte each.
  __device__ __forceinline__ uint32_t scales(bool upper) const {
    return upper ? (hdr.w & 0x0f0f0f0fu) | ((hdr.y >> 2) & 0x30303030u) : hdr.y & 0x3f3f3f3fu;
  }
  __device__ __forceinline__ uint32_t mins(bool upper) const {
    return upper ? ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u) : hdr.z & 0x3f3f3f3fu;
  }
  // sc * q: (1024 + q) * sc - 1024 * sc in one exact fma.
  __device__ __forceinline__ void weight(int s, int kg, half8 &h, half8 &) const {
    const uint2 q = *reinterpret_cast<const uint2 *>(p + 16 + (s >> 1) * 32 + 8 * kg);
    const half2v f = twice(scales(s >= 4), s & 3) + half2v{(f16)-1024.f, (f16)-1024.f};
    const half2v c = f * half2v{(f16)-1024.f, (f16)-1024.f};
    const int sh = 4 * (s & 1);
    half2v a, b, e, g;
    biased((q.x >> sh) & 0x0f0f0f0fu, a, b);
    biased((q.y >> sh) & 0x0f0f0f0fu, e, g);
    h = join(__builtin_elementwise_fma(a, f, c), __builtin_elementwise_fma(b, f, c),
             __builtin_elementwise_fma(e, f, c), __builtin_elementwise_fma(g, f, c));
  }
};

// Steps 4 h + 0 .. 3 are the quarters of half h; quarters j and j + 2 share 32
// ql bytes (low and high nibbles), all four the half's 32 qh bytes.
template <> struct Row<LLRS_Q6_K> : RowBase {
  static constexpr Unit kUnit = kBlock;
  static constexpr int kPlanes = 2;
  static constexpr int kCols = 256, kBytes = 210, kSpan = 15;
  const uint8_t *p;
  uint16_t db;
  __device__ __forceinline__ void open(const uint8_t *row) {
    p = row;
    db = ld_u16(row + 208);
  }
  __device__ __forceinline__ float d() const { return f16_bits_to_f32(db); }
  // hi = the f16 rounding of sc * (q - 32), lo = the exact remainder.
  __device__ __forceinline__ void weight(int s, int kg, half8 &h, half8 &l) const {
#pragma clang fp contract(off)
    const int hf = s >> 2, qt = s & 3;
    const Bytes8 ql(p + hf * 64 + (qt & 1) * 32 + 8 * kg), qh(p + 128 + hf * 32 + 8 * kg);
    // The int8 scale as 1024 + (scale + 128), less 1,152.
    const half2v f = twice(p[192 + hf * 8 + qt * 2 + (kg >> 1)] ^ 0x80u, 0) + half2v{(f16)-1152.f, (f16)-1152.f};
    const half2v off = {(f16)-1056.f, (f16)-1056.f};
    half2v x[4];
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const uint32_t lw = k ? ql.hi() : ql.lo(), hw = k ? qh.hi() : qh.lo();
      const uint32_t q = ((qt < 2 ? lw : lw >> 4) & 0x0f0f0f0fu) | (((hw >> (2 * qt)) & 0x03030303u) << 4);
      biased(q, x[2 * k], x[2 * k + 1]);
    }
    half2v hi[4], lo[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const half2v v = x[k] + off;
      hi[k] = v * f;
      lo[k] = __builtin_elementwise_fma(v, f, -hi[k]);
    }
    h = join(hi[0], hi[1], hi[2], hi[3]);
    l = join(lo[0], lo[1], lo[2], lo[3]);
  }
};

template <> struct Row<LLRS_Q8_0> : RowBase {
  static constexpr Unit kUnit = kStep;
  static constexpr int kCols = 256, kBytes = 272, kSpan = 19;
  const uint8_t *p;
  __device__ __forceinline__ void open(const uint8_t *row) { p = row; }
  __device__ __forceinline__ float step_d(int s) const { return f16_bits_to_f32(ld_u16(p + 34 * s)); }
  __device__ __forceinline__ void weight(int s, int kg, half8 &h, half8 &) const {
    const Bytes8 q(p + 34 * s + 2 + 8 * kg);
    h = offset_codes(q.lo() ^ 0x80808080u, q.hi() ^ 0x80808080u, 128.f);
  }
};

template <> struct Row<LLRS_Q5_0> : RowBase {
  static constexpr Unit kUnit = kStep;
  static constexpr int kCols = 256, kBytes = 176, kSpan = 13;
  const uint8_t *p;
  __device__ __forceinline__ void open(const uint8_t *row) { p = row; }
  __device__ __forceinline__ float step_d(int s) const { return f16_bits_to_f32(ld_u16(p + 22 * s)); }
  __device__ __forceinline__ void weight(int s, int kg, half8 &h, half8 &) const {
    const Bytes8 q(p + 22 * s + 6 + 8 * (kg & 1));  // columns 0-15: low nibbles, 16-31: high
    const uint32_t b = p[22 * s + 2 + kg], n = 4u * (kg >> 1);
    h = offset_codes(((q.lo() >> n) & 0x0f0f0f0fu) | spread4(b), ((q.hi() >> n) & 0x0f0f0f0fu) | spread4(b >> 4), 16.f);
  }
};

template <uint32_t TY> struct RowHalf : RowBase {
  static constexpr Unit kUnit = kNone;
  static constexpr int kCols = 128, kBytes = 256, kSpan = 16, kPad = 1;
  const uint8_t *p;
  __device__ __forceinline__ void open(const uint8_t *row) { p = row; }
  __device__ __forceinline__ void weight(int s, int kg, half8 &h, half8 &) const {
    const uint4 q = *reinterpret_cast<const uint4 *>(p + 64 * s + 16 * kg);
    if constexpr (TY == LLRS_F16) {
      h = __builtin_bit_cast(half8, q);
    } else {
      const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        h[2 * e] = (f16)__uint_as_float(w[e] << 16);
        h[2 * e + 1] = (f16)__uint_as_float(w[e] & 0xffff0000u);
      }
    }
  }
};
template <> struct Row<LLRS_F16> : RowHalf<LLRS_F16> {};
template <> struct Row<LLRS_BF16> : RowHalf<LLRS_BF16> {};

__device__ __forceinline__ f32x4 mfma(half8 a, half8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Buffer b (SA steps) of the unit at column k0: the products of a wave's RT row
// tiles w with the TT token tiles at frag (the lane's slot of the first
// fragment), into blk for a block type, acc otherwise.
template <uint32_t TY, int TT, int RT, int SA, class B>
__device__ __forceinline__ void multiply(f32x4 (&acc)[TT][RT], B &blk, const Row<TY> (&w)[RT], const uint8_t *frag, int b,
                                         int k0, int ke, int kg) {
  using R = Row<TY>;
#pragma unroll
  for (int s = 0; s < SA; s++) {
    // All ones inside the range (opaque: as a condition the compiler branches
    // on it around every sum and spills).
    uint32_t in = k0 + 32 * (b * SA + s) < ke ? ~0u : 0u;
    if constexpr (R::kUnit != kBlock) asm("" : "+v"(in));
    half8 wh[RT], wl[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
      w[r].weight(b * SA + s, kg, wh[r], wl[r]);
      if constexpr (R::kUnit == kNone)
        wh[r] = __builtin_bit_cast(half8, __builtin_bit_cast(u32x4, wh[r]) & u32x4{in, in, in, in});
    }
#pragma unroll
    for (int i = 0; i < TT; i++) {
      const half8 ah = *reinterpret_cast<const half8 *>(frag + (s * TT + i) * 1024);
      const half8 al = *reinterpret_cast<const half8 *>(frag + ((SA + s) * TT + i) * 1024);
      if constexpr (R::kUnit == kStep) {
        f32x4 c[RT];
#pragma unroll
        for (int r = 0; r < RT; r++) c[r] = mfma(al, wh[r], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int r = 0; r < RT; r++) c[r] = mfma(ah, wh[r], c[r]);
#pragma unroll
        for (int r = 0; r < RT; r++) acc[i][r] += __uint_as_float(__float_as_uint(w[r].step_d(b * SA + s)) & in) * c[r];
      } else {
        auto &dst = [&]() -> f32x4(&)[RT] {
          if constexpr (R::kUnit == kBlock) return blk[i];
          else return acc[i];
        }();
#pragma unroll
        for (int r = 0; r < RT; r++) dst[r] = mfma(al, wh[r], dst[r]);
        if constexpr (R::kPlanes == 2) {
#pragma unroll
          for (int r = 0; r < RT; r++) dst[r] = mfma(ah, wl[r], dst[r]);
        }
#pragma unroll
        for (int r = 0; r < RT; r++) dst[r] = mfma(ah, wh[r], dst[r]);
      }
    }
  }
}

// Step s of a buffer with its operands wh decoded, while those of the step after it
// are decoded (ahead) in the MFMAs' shadow: two VALU operations after each, the
// fragments one token tile early.
template <uint32_t TY, int TT, int RT, int SA>
__device__ __forceinline__ void multiply_ahead(f32x4 (&acc)[TT][RT], const Row<TY> (&w)[RT], half8 (&wh)[RT],
                                               const uint8_t *frag, int step, bool ahead, int kg) {
  half8 nh[RT], none;
  if (ahead) {
#pragma unroll
    for (int r = 0; r < RT; r++) w[r].weight(step + 1, kg, nh[r], none);
  }
  const int s = step % SA;
#pragma unroll
  for (int i = 0; i < TT; i++) {
    const half8 ah = *reinterpret_cast<const half8 *>(frag + (s * TT + i) * 1024);
    const half8 al = *reinterpret_cast<const half8 *>(frag + ((SA + s) * TT + i) * 1024);
#pragma unroll
    for (int r = 0; r < RT; r++) acc[i][r] = mfma(al, wh[r], acc[i][r]);
#pragma unroll
    for (int r = 0; r < RT; r++) acc[i][r] = mfma(ah, wh[r], acc[i][r]);
  }
  __builtin_amdgcn_sched_group_barrier(0x100, 2 + RT, 0);  // LDS reads
#pragma unroll
  for (int i = 0; i < TT; i++) {
    if (i + 1 < TT) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
    for (int m = 0; m < 2 * RT; m++) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // an MFMA
      __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);  // VALU
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  if (ahead) {
#pragma unroll
    for (int r = 0; r < RT; r++) wh[r] = nh[r];
  }
}

// A block type's unit in absolute terms: d times its sums (a block with d = 0
// has finite sums and adds its dmin term only), and for Q4_K - dmin * sum_s m_s
// xsum_s over the block's eight sub-blocks: lane group kg contributes
// sub-blocks 2 kg and 2 kg + 1, exact integers.  sums: [plane][token] 16 bytes.
template <uint32_t TY, int TT, int RT, class B>
__device__ __forceinline__ void finish(f32x4 (&acc)[TT][RT], const B &blk, const Row<TY> (&w)[RT], const uint8_t *sums,
                                       int n, int kg) {
#pragma unroll
  for (int r = 0; r < RT; r++) {
    const float d = w[r].d();
#pragma unroll
    for (int i = 0; i < TT; i++) acc[i][r] += d * blk[i][r];
    if constexpr (TY == LLRS_Q4_K) {
      const uint32_t m2 = (w[r].mins(kg >= 2) >> (16 * (kg & 1))) & 0xffffu;
      const half4v m = {(f16)(float)(m2 & 0xff), (f16)(float)(m2 >> 8), (f16)0.f, (f16)0.f};
      const float dm = w[r].dmin();
#pragma unroll
      for (int i = 0; i < TT; i++) {
        const half2v xh = *reinterpret_cast<const half2v *>(sums + (16 * i + n) * 16 + 4 * kg);
        const half2v xl = *reinterpret_cast<const half2v *>(sums + (16 * (TT + i) + n) * 16 + 4 * kg);
        const half4v ah = {xh[0], xh[1], (f16)0.f, (f16)0.f}, al = {xl[0], xl[1], (f16)0.f, (f16)0.f};
        f32x4 c = __builtin_amdgcn_mfma_f32_16x16x16f16(al, m, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x16f16(ah, m, c, 0, 0, 0);
        acc[i][r] -= dm * c;
      }
    }
  }
}

// A wave's RT * 16 weight rows on their way to its part of LDS.  Consecutive
// lanes copy consecutive 16-byte pieces of a row: loads of one row per lane (the
// operands' own layout) touch a cache line per lane and ran at a fraction of
// this rate.  A piece's place is kept as one word, row start + 16 * piece:
// adding the unit's offset and clearing the low bits aligns it.
template <uint32_t TY, int RT, bool DUAL> struct Rows {
  using R = Row<TY>;
  static constexpr int NP = RT * 16 * R::kSpan, NW = (NP + 63) / 64;  // pieces, and per lane
  static constexpr int GR = DUAL ? RT * 8 : RT * 16;                  // rows in one matrix
  const uint8_t *w0, *w1;
  uint32_t piece[NW], from[RT], last;  // from: where the lane's operand rows start
  u32x4 reg[NW];
  int units;
  // i0: the wave's first row in its matrix (rows past its `rows` read the last
  // one); ke: the end of the K range (units past it read the last one).
  __device__ __forceinline__ Rows(const PrefillGemmArgs &g, int seg, int i0, int rows, int ke) {
    const int lane = threadIdx.x & 63;
    w0 = g.nseg > 0 ? g.seg_w[seg] : g.w;
    w1 = DUAL ? g.w2 : w0;
    auto row_at = [&](int i) { return (uint32_t)min(i0 + (DUAL ? i % GR : i), rows - 1) * (uint32_t)g.row_bytes; };
#pragma unroll
    for (int j = 0; j < NW; j++) {
      const int v = min(lane + 64 * j, NP - 1);
      piece[j] = row_at(v / R::kSpan) + 16 * (v % R::kSpan);
    }
#pragma unroll
    for (int r = 0; r < RT; r++) from[r] = row_at(16 * r + (lane & 15));
    last = ((uint32_t)rows * (uint32_t)g.row_bytes + (uint32_t)kTensorTailPad - 16) & ~15u;
    units = (ke - 1) / R::kCols;
  }
  __device__ __forceinline__ uint32_t offset(int k0) const { return (uint32_t)min(k0 / R::kCols, units) * R::kBytes; }
  __device__ __forceinline__ void load(int k0) {
    const uint32_t o = offset(k0);
#pragma unroll
    for (int j = 0; j < NW; j++) {
      // A dual wave's second half of rows is in the other matrix.
      const uint8_t *const m0 = w0, *const m1 = w1;
      const uint8_t *m = DUAL && (int)(threadIdx.x & 63) + 64 * j >= GR * R::kSpan ? m1 : m0;
      reg[j] = *reinterpret_cast<const u32x4 *>(m + min((piece[j] + o) & ~15u, last));
    }
  }
  __device__ __forceinline__ void store(uint8_t *to) const {
#pragma unroll
    for (int j = 0; j < NW; j++) {
      const int v = (int)(threadIdx.x & 63) + 64 * j;
      if (NP % 64 == 0 || j + 1 < NW || v < NP) *reinterpret_cast<u32x4 *>(to + 16 * (v + R::kPad * (v / R::kSpan))) = reg[j];
    }
  }
  __device__ __forceinline__ void open(Row<TY> (&w)[RT], const uint8_t *at, int k0) const {
#pragma unroll
    for (int r = 0; r < RT; r++)
      w[r].open(at + (16 * r + (int)(threadIdx.x & 15)) * (R::kSpan + R::kPad) * 16 + ((from[r] + offset(k0)) & 15));
  }
};

// Outputs of a workgroup's waves: lane (n, kg) holds row n of each tile and
// tokens 4 kg + e.  mine: whether this wave has any; lds: free for the dual
// product's 32-column sums of a wave's 16-row tile pairs.
template <int TT, int RT, bool DUAL>
__device__ __forceinline__ void store_outputs(const PrefillGemmArgs &g, const f32x4 (&acc)[TT][RT], float *lds, int seg,
                                              int sbase, int srows, int r0, int t0, int nrw, int wave, bool mine) {
  constexpr int GT = DUAL ? RT / 2 : RT;
  const int lane = threadIdx.x & 63, n = lane & 15, kg = lane >> 4, T = g.t;
  if (DUAL && g.ksplit == 1) {
#pragma clang fp contract(off)
    // [wave][16 TT tokens]: the sums over the wave's 16 GT columns (at most 32).
    if (mine) {
#pragma unroll
      for (int i = 0; i < TT; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int t = t0 + 16 * i + 4 * kg + e;
          float v = 0.f;
#pragma unroll
          for (int r = 0; r < GT; r++) {
            const int f = r0 + 16 * r + n;
            const float x = acc[i][r][e], up = acc[i][r + GT][e];
            f16 hi = 0, lo = 0;
            if (f < g.dual_rows && t < T) {
              split_f16((x / (1.0f + expf(-x))) * up, hi, lo);
              g.h[(size_t)t * g.ldh + f] = hi;
              g.hl[(size_t)t * g.ldh + f] = lo;
            }
            v += (float)hi + (float)lo;
          }
          if (g.xso) {
#pragma unroll
            for (int b = 1; b < 16; b <<= 1) v += lane_partner(v, b);
            if (GT == 2) {
              if (n == 0 && t < T && r0 < g.dual_rows)
                split_f16(v, g.xso[(size_t)t * g.ldxso + (r0 >> 5)], g.xso_lo[(size_t)t * g.ldxso + (r0 >> 5)]);
            } else if (n == 0) {
              lds[wave * 16 * TT + 16 * i + 4 * kg + e] = v;
            }
          }
        }
    }
    if (GT == 2 || !g.xso) return;
    __syncthreads();
    // Two neighbouring waves' rows are one 32-column sub-block of the next
    // product (dual workgroups with sums have an even number of row waves).
    const int i = threadIdx.x % (16 * TT), t = t0 + i;
    for (int p = threadIdx.x / (16 * TT); p < nrw / 2; p += blockDim.x / (16 * TT)) {
      const int q = blockIdx.x * (nrw / 2) + p;
      if (t < T && 32 * q < g.dual_rows)
        split_f16(lds[2 * p * 16 * TT + i] + lds[(2 * p + 1) * 16 * TT + i], g.xso[(size_t)t * g.ldxso + q],
                  g.xso_lo[(size_t)t * g.ldxso + q]);
    }
    return;
  }
  if (!mine) return;
#pragma unroll
  for (int i = 0; i < TT; i++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int t = t0 + 16 * i + 4 * kg + e;
      if (t >= T) continue;
      if (g.ksplit > 1) {
        float *p = g.part + ((size_t)blockIdx.z * T + t) * g.n;
#pragma unroll
        for (int r = 0; r < RT; r++) {
          const int f = r0 + 16 * (r % GT) + n;
          if (f - sbase >= srows) continue;
          // A dual product's virtual column: 64 gate rows, then the same 64 up rows.
          p[DUAL ? (f >> 6) * 128 + (f & 63) + (r >= GT ? 64 : 0) : f] = acc[i][r][e];
        }
      } else if constexpr (!DUAL) {
        float *c = g.nseg > 0 ? g.seg_c[seg] + (size_t)t * g.seg_ldc[seg] : g.c + (size_t)t * g.ldc;
        const float *bias = g.nseg > 0 ? g.seg_bias[seg] : g.bias;
#pragma unroll
        for (int r = 0; r < RT; r++) {
          const int f = r0 - sbase + 16 * r + n;
          if (f >= srows) continue;
          c[f] = g.accumulate ? c[f] + acc[i][r][e] : acc[i][r][e] + (bias ? bias[f] : 0.f);
        }
      }
    }
}

// A workgroup is KW = 2 groups of up to kMaxRowWaves row waves and one staging
// wave.  Its LDS, in bytes: the groups' activations (two buffers of SA steps)
// and sums of the unit's sub-blocks (Q4_K), the row waves' rows.
constexpr int KW = 2, kMaxRowWaves = 5;
constexpr int kSmallRT = 2;  // row tiles of a row wave
constexpr int steps_per_buffer(int TT) { return TT == 1 ? 4 : 2; }
constexpr size_t acts_bytes(int TT) { return (size_t)KW * 2 * 2 * steps_per_buffer(TT) * TT * 1024; }
template <uint32_t TY> constexpr size_t sums_bytes(int TT) { return TY == LLRS_Q4_K ? (size_t)KW * 2 * 16 * TT * 16 : 0; }
template <uint32_t TY, int RT> constexpr size_t wave_bytes() { return (size_t)RT * 16 * (Row<TY>::kSpan + Row<TY>::kPad) * 16; }
template <uint32_t TY> constexpr size_t lds_bytes(int TT, int row_waves) {
  return acts_bytes(TT) + sums_bytes<TY>(TT) + KW * row_waves * wave_bytes<TY, kSmallRT>();
}

// 16 TT tokens x 32 weight rows a row wave (the two groups share the rows and
// take alternate units of columns), one K range.  DUAL: a wave's tiles are 16
// gate rows and the same 16 up rows.
template <uint32_t TY, int TT, bool DUAL>
__global__ __launch_bounds__(64 * (kMaxRowWaves + 1) * KW, 3) void prefill_reg_kernel(PrefillGemmArgs g) {
  using R = Row<TY>;
  constexpr int RT = kSmallRT;
  constexpr bool kUnits = R::kUnit == kBlock, kMins = TY == LLRS_Q4_K;
  constexpr int SA = steps_per_buffer(TT), NB = R::kCols / (32 * SA);  // steps of a buffer, buffers of a unit
  constexpr int NF = 2 * SA * TT;                    // activation fragments of a buffer
  constexpr int GT = DUAL ? RT / 2 : RT;             // row tiles of the wave in one matrix
  constexpr int UK = R::kCols * KW;                  // columns of a round
  static_assert(NB % 2 == 0, "a unit is an even number of buffers");
  extern __shared__ __align__(16) uint8_t lds[];
  const int nrw = blockDim.x / (64 * KW) - 1;        // row waves of a group
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kq = wv > nrw ? 1 : 0, wave = wv - kq * (nrw + 1), n = lane & 15, kg = lane >> 4;
  const int t0 = blockIdx.y * 16 * TT, T = g.t, K = g.k;
  const int nb = (K + 255) >> 8, per = (nb + g.ksplit - 1) / g.ksplit;
  const int kb = blockIdx.z * per * 256, ke = min(K, kb + per * 256);
  const int k1 = kb + R::kCols * kq;                             // the group's first column
  const int rounds = kb < ke ? (ke - kb + UK - 1) / UK : 0;      // the same in every wave
  uint8_t *const acts = lds + (size_t)kq * 2 * NF * 1024;
  uint8_t *const sums = lds + acts_bytes(TT) + (size_t)kq * 2 * 16 * TT * 16;
  // Rows: the wave's segment (boundaries are multiples of 128 rows); rows past
  // the end read the last one and are not stored.
  const int r0 = (blockIdx.x * nrw + wave) * 16 * GT;
  const int seg = g.nseg > 1 ? (r0 >= g.seg_base[1]) + (g.nseg > 2 && r0 >= g.seg_base[2]) : 0;
  const int sbase = g.nseg > 0 ? g.seg_base[seg] : 0;
  const int srows = DUAL ? g.dual_rows : g.nseg > 0 ? g.seg_base[seg + 1] - sbase : g.n;

  f32x4 acc[TT][RT];
#pragma unroll
  for (int i = 0; i < TT; i++)
#pragma unroll
    for (int r = 0; r < RT; r++) acc[i][r] = f32x4{0.f, 0.f, 0.f, 0.f};

  if (wave == nrw) {
    // ---- Staging: buffer m + 1 is written while m is read, m + 2 is in flight ----
    // Fragment f: plane f / (SA TT), step f / TT % SA, token tile f % TT; lane =
    // (token, piece) = (lane / 4, lane % 4), a cache line's half per four lanes.
    // Token t's piece kg lies in slot 16 kg + (t ^ 4 kg) of the fragment, so that
    // neither these stores nor the operand reads meet in a bank.  Columns past
    // the range become zeros.  A wave of its own: a wave's loads return in order,
    // so behind row loads the activations would wait for HBM.
    const int at = lane >> 2, ap = lane & 3, slot = 16 * (16 * ap + (at ^ (4 * ap)));
    const f16 *const ahi = g.a, *const alo = g.a_lo;
    uint32_t arow[TT];
#pragma unroll
    for (int i = 0; i < TT; i++) arow[i] = (uint32_t)min(t0 + 16 * i + at, T - 1) * (uint32_t)g.lda + 8 * ap;
    half8 st[NF];
    const int M = rounds * NB;
    auto column = [&](int m) { return k1 + m / NB * UK + m % NB * 32 * SA; };
    auto load = [&](int m) INLINE {
      const int k0 = column(m);
#pragma unroll
      for (int f = 0; f < NF; f++) {
        const int c = min(k0 + 32 * (f / TT % SA), ke - 32);
        st[f] = *reinterpret_cast<const half8 *>((f < SA * TT ? ahi : alo) + c + arow[f % TT]);
      }
    };
    auto store = [&](int m) INLINE {
      const int k0 = column(m);
#pragma unroll
      for (int f = 0; f < NF; f++) {
        uint32_t in = k0 + 32 * (f / TT % SA) < ke ? ~0u : 0u;
        u32x4 v = __builtin_bit_cast(u32x4, st[f]);
        if constexpr (!kUnits) v &= u32x4{in, in, in, in};  // a block type's units are whole, or not added
        *reinterpret_cast<u32x4 *>(acts + ((m & 1) * NF + f) * 1024 + slot) = v;
      }
    };
    // Q4_K: the sums of the unit's eight sub-blocks, per plane and token.
    constexpr int NX = kMins ? (2 * 16 * TT + 63) / 64 : 1;
    half8 xreg[NX];
    const f16 *xsrc[NX];
#pragma unroll
    for (int j = 0; j < NX; j++) {
      const int i = min(lane + 64 * j, 2 * 16 * TT - 1);
      xsrc[j] = (i < 16 * TT ? g.xs : g.xs_lo) + (size_t)min(t0 + i % (16 * TT), T - 1) * g.ldxs;
    }
    auto load_sums = [&](int k0) INLINE {
      if constexpr (kMins)
#pragma unroll
        for (int j = 0; j < NX; j++) xreg[j] = *reinterpret_cast<const half8 *>(xsrc[j] + (min(k0, ke - 256) >> 5));
    };
    if (M > 0) {
      load(0);
      load_sums(k1);
      store(0);
      load(1);  // NB >= 2
    }
    __syncthreads();
    for (int m = 0; m < M; m++) {
      if (kMins && m % NB == 0) {
#pragma unroll
        for (int j = 0; j < NX; j++)
          if (lane + 64 * j < 2 * 16 * TT) *reinterpret_cast<half8 *>(sums + (lane + 64 * j) * 16) = xreg[j];
        load_sums(column(m + NB));
      }
      if (m + 1 < M) store(m + 1);
      if (m + 2 < M) load(m + 2);
      __syncthreads();
    }
  } else {
    Rows<TY, RT, DUAL> src(g, seg, r0 - sbase, srows, ke);
    uint8_t *const rows = lds + acts_bytes(TT) + sums_bytes<TY>(TT) + (kq * nrw + wave) * wave_bytes<TY, RT>();
    const uint8_t *const frag0 = acts + 16 * (16 * kg + (n ^ (4 * kg)));
    f32x4 blk[kUnits ? TT : 1][kUnits ? RT : 1];

    // One unit: its rows go from the registers to LDS (the wave's own: no
    // barrier), the next unit's are loaded.
    auto round = [&](int k0, auto more) INLINE {
      src.store(rows);
      if constexpr (decltype(more)::value) src.load(k0 + UK);
      __builtin_amdgcn_sched_barrier(0);  // the scheduler would sink the loads to their uses
      R w[RT];
      src.open(w, rows, k0);
      if constexpr (kUnits) {
#pragma unroll
        for (int i = 0; i < TT; i++)
#pragma unroll
          for (int r = 0; r < RT; r++) blk[i][r] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int b = 0; b < NB; b++) {
        multiply<TY, TT, RT, SA>(acc, blk, w, frag0 + (b & 1) * NF * 1024, b, k0, ke, kg);
        if (kUnits && b + 1 == NB && k0 < ke) finish<TY, TT, RT>(acc, blk, w, sums, n, kg);
        __syncthreads();
      }
    };
    if (rounds) src.load(k1);
    __syncthreads();
    if (rounds) {
      int k0 = k1;
      for (int i = 1; i < rounds; i++, k0 += UK) round(k0, std::true_type{});
      round(k0, std::false_type{});
    }
  }

  // The second group's sums join the first's.
  {
    float *sum = reinterpret_cast<float *>(lds) + (size_t)wave * (TT * RT * 4 * 64) + lane;
    if (kq == 1 && wave < nrw) {
#pragma unroll
      for (int i = 0; i < TT; i++)
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
          for (int e = 0; e < 4; e++) sum[((i * RT + r) * 4 + e) * 64] = acc[i][r][e];
    }
    __syncthreads();
    if (kq == 0 && wave < nrw) {
#pragma unroll
      for (int i = 0; i < TT; i++)
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[i][r][e] += sum[((i * RT + r) * 4 + e) * 64];
    }
    __syncthreads();
  }

  store_outputs<TT, RT, DUAL>(g, acc, reinterpret_cast<float *>(lds), seg, sbase, srows, r0, t0, nrw, wave,
                              kq == 0 && wave < nrw);
}

// The same products over many tokens: 64 tokens x eight waves of 16 RT rows, one
// workgroup a CU, whole K ranges; the row waves stage the activations themselves
// (their loads go out before the next unit's rows, and each has a buffer's
// products to land).  RT = 4 reads 8 fragments of LDS per 32 MFMAs, half of LDS's
// rate at the full MFMA rate.  What bounds it is spread out: matrix cores busy
// 45% at the ~1.9 GHz the card then holds, and a half of the MFMAs, all memory
// latency or half of the decoding taken out win 8% each.  7B shape, 512 tokens, per
// layer: gate/up 332 us, ffn_down 251; two workgroups of four waves a CU, which
// load the activations twice and meet twice as often, 340 and 280 (with Q6_K's
// decoding ahead of the products, as Q4_K's, 300); the LDS-staged kernel with
// decoded weights in LDS 361 and 295.
// Four row tiles leave registers for one set of accumulators only, so Q4_K's are
// kept in units of the row's current d, rescaled by d_prev / d at each block (a
// block with d = 0 keeps the unit and multiplies zeros), and its dmin * m term
// is a second, 1/32 as long product at the end: - (dmin m)_s (hi + lo) with
// xsum_s (hi + lo).
constexpr int kBigTT = 4, kBigWaves = 8, kBigSA = 4;
constexpr size_t big_acts_bytes() { return (size_t)2 * 2 * kBigSA * kBigTT * 1024; }
template <uint32_t TY, int RT> constexpr size_t big_lds_bytes() {
  return big_acts_bytes() + kBigWaves * wave_bytes<TY, RT>();
}
template <uint32_t TY, int RT, bool DUAL>
__global__ __launch_bounds__(64 * kBigWaves, 2) void prefill_reg_big_kernel(PrefillGemmArgs g) {
  using R = Row<TY>;
  constexpr bool kRatio = TY == LLRS_Q4_K, kUnits = R::kUnit == kBlock && !kRatio;
  constexpr int TT = kBigTT, SA = kBigSA, NB = R::kCols / (32 * SA), NF = 2 * SA * TT, NL = NF / kBigWaves;
  constexpr int GT = DUAL ? RT / 2 : RT;
  static_assert(kBigWaves == 2 * TT, "waves w and w + TT stage token tile w, half of the steps each");
  extern __shared__ __align__(16) uint8_t lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, kg = lane >> 4;
  const int t0 = blockIdx.y * 16 * TT, T = g.t, K = g.k;
  const int nb = (K + 255) >> 8, per = (nb + g.ksplit - 1) / g.ksplit;
  const int kb = blockIdx.z * per * 256, ke = min(K, kb + per * 256);
  const int r0 = (blockIdx.x * kBigWaves + wave) * 16 * GT;
  const int seg = g.nseg > 1 ? (r0 >= g.seg_base[1]) + (g.nseg > 2 && r0 >= g.seg_base[2]) : 0;
  const int sbase = g.nseg > 0 ? g.seg_base[seg] : 0;
  const int srows = DUAL ? g.dual_rows : g.nseg > 0 ? g.seg_base[seg + 1] - sbase : g.n;
  uint8_t *const rows = lds + big_acts_bytes() + wave * wave_bytes<TY, RT>();
  const uint8_t *const frag0 = lds + 16 * (16 * kg + (n ^ (4 * kg)));

  // This wave's fragments: token tile `wave`, every step, both planes (lane =
  // (token, piece), slots as in prefill_reg_kernel).
  const int at = lane >> 2, ap = lane & 3, slot = 16 * (16 * ap + (at ^ (4 * ap)));
  const int tile = wave % TT, half = wave / TT * (SA / 2);
  const uint32_t arow = (uint32_t)min(t0 + 16 * tile + at, T - 1) * (uint32_t)g.lda + 8 * ap;
  const f16 *const ahi = g.a, *const alo = g.a_lo;
  half8 st[NL];
  auto load_acts = [&](int k0) INLINE {
#pragma unroll
    for (int j = 0; j < NL; j++)
      st[j] = *reinterpret_cast<const half8 *>((j < SA / 2 ? ahi : alo) + min(k0 + 32 * (half + j % (SA / 2)), ke - 32) + arow);
  };
  auto store_acts = [&](int k0, int b) INLINE {
#pragma unroll
    for (int j = 0; j < NL; j++) {
      const int f = j / (SA / 2) * SA + half + j % (SA / 2);
      uint32_t in = k0 + 32 * (f % SA) < ke ? ~0u : 0u;
      u32x4 v = __builtin_bit_cast(u32x4, st[j]);
      if constexpr (R::kUnit != kBlock) v &= u32x4{in, in, in, in};
      *reinterpret_cast<u32x4 *>(lds + (b * NF + f * TT + tile) * 1024 + slot) = v;
    }
  };
  f32x4 acc[TT][RT], blk[kUnits ? TT : 1][kUnits ? RT : 1];
#pragma unroll
  for (int i = 0; i < TT; i++)
#pragma unroll
    for (int r = 0; r < RT; r++) acc[i][r] = f32x4{0.f, 0.f, 0.f, 0.f};
  float u[RT];  // kRatio: the rows' current units
#pragma unroll
  for (int r = 0; r < RT; r++) u[r] = 1.f;
  Rows<TY, RT, DUAL> src(g, seg, r0 - sbase, srows, ke);
  auto round = [&](int k0, auto more) INLINE {
    constexpr bool kMore = decltype(more)::value;
    src.store(rows);
    R w[RT];
    src.open(w, rows, k0);
    if constexpr (kRatio) {
#pragma unroll
      for (int r = 0; r < RT; r++) {
        const float d = w[r].d();
        const bool live = d != 0.f;  // NaN d is live and makes the row NaN, as in f32
        const float ratio = live ? u[r] / d : 1.f;
        u[r] = live ? d : u[r];
        w[r].hdr.y = live ? w[r].hdr.y : 0u;
        w[r].hdr.w = live ? w[r].hdr.w : 0u;
#pragma unroll
        for (int i = 0; i < TT; i++) acc[i][r] *= ratio;
      }
    }
    if constexpr (kUnits) {
#pragma unroll
      for (int i = 0; i < TT; i++)
#pragma unroll
        for (int r = 0; r < RT; r++) blk[i][r] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    half8 wh[RT], none;
    if constexpr (kRatio) {
#pragma unroll
      for (int r = 0; r < RT; r++) w[r].weight(0, kg, wh[r], none);
    }
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const int kn = k0 + 32 * SA * (b + 1);  // the next buffer's columns
      const bool next = b + 1 < NB || kMore;
      if (next) load_acts(kn);
      if (kMore && b == 0) src.load(k0 + R::kCols);
      __builtin_amdgcn_sched_barrier(0);  // the scheduler would sink the loads to their uses
      const uint8_t *const frag = frag0 + (b & 1) * NF * 1024;
      if constexpr (kRatio) {
#pragma unroll
        for (int step = b * SA; step < (b + 1) * SA; step++)
          multiply_ahead<TY, TT, RT, SA>(acc, w, wh, frag, step, step + 1 < R::kCols / 32, kg);
      } else {
        multiply<TY, TT, RT, SA>(acc, blk, w, frag, b, k0, ke, kg);
      }
      if constexpr (kUnits)
        if (b + 1 == NB) finish<TY, TT, RT>(acc, blk, w, nullptr, n, kg);
      if (next) store_acts(kn, (b + 1) & 1);
      __syncthreads();
    }
  };
  if (kb < ke) {
    int k0 = kb;
    load_acts(k0);
    src.load(k0);
    store_acts(k0, 0);
    __syncthreads();
    for (; k0 + R::kCols < ke; k0 += R::kCols) round(k0, std::true_type{});
    round(k0, std::false_type{});
  }
  if constexpr (kRatio) {
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int i = 0; i < TT; i++) acc[i][r] *= u[r];
    // 32 sub-blocks a step: lane group kg takes the eight of block m0 / 8 + kg.
    const int me = ke >> 5;
    for (int m0 = kb >> 5; m0 < me; m0 += 32) {
      const bool in = m0 + 8 * kg < me;
      half8 wh[RT], wl[RT];
#pragma unroll
      for (int r = 0; r < RT; r++) {
        R h;
        const uint8_t *m = src.w0;
        if (r >= GT) m = src.w1;
        h.hdr = *reinterpret_cast<const uint4 *>(m + src.from[r] + (size_t)(in ? (m0 >> 3) + kg : kb >> 8) * R::kBytes);
        const float dm = in ? h.dmin() : 0.f;
        const uint32_t ml = h.mins(false), mu = h.mins(true);
#pragma unroll
        for (int e = 0; e < 8; e++) {
          f16 a, b;
          split_f16(-(dm * (float)(((e < 4 ? ml : mu) >> (8 * (e & 3))) & 0xff)), a, b);
          wh[r][e] = a;
          wl[r][e] = b;
        }
      }
#pragma unroll
      for (int i = 0; i < TT; i++) {
        const size_t o = (size_t)min(t0 + 16 * i + n, T - 1) * g.ldxs + (in ? m0 + 8 * kg : kb >> 5);
        const half8 ah = *reinterpret_cast<const half8 *>(g.xs + o);
        const half8 al = *reinterpret_cast<const half8 *>(g.xs_lo + o);
#pragma unroll
        for (int r = 0; r < RT; r++) {
          acc[i][r] = mfma(al, wh[r], acc[i][r]);
          acc[i][r] = mfma(ah, wl[r], acc[i][r]);
          acc[i][r] = mfma(ah, wh[r], acc[i][r]);
        }
      }
    }
  }
  store_outputs<TT, RT, DUAL>(g, acc, reinterpret_cast<float *>(lds), seg, sbase, srows, r0, t0, kBigWaves, wave, true);
}

// Row tiles of a wave over many tokens: four for Q4_K; Q6_K's three MFMAs a
// product leave LDS at two thirds of its rate with two, and the others' rows
// leave no registers for four (256 a lane).
constexpr int big_row_tiles(uint32_t type) { return type == LLRS_Q4_K ? 4 : 2; }

template <uint32_t TY> void launch_big(const PrefillGemmArgs &a, hipStream_t s) {
  constexpr int RT = big_row_tiles(TY);
  const int rows = a.w2 ? a.dual_rows : a.n, tile = kBigWaves * 16 * (a.w2 ? RT / 2 : RT);
  const dim3 grid((unsigned)((rows + tile - 1) / tile), (unsigned)((a.t + 16 * kBigTT - 1) / (16 * kBigTT)), (unsigned)a.ksplit);
  if (a.w2)
    hipLaunchKernelGGL((prefill_reg_big_kernel<TY, RT, true>), grid, dim3(64 * kBigWaves), (big_lds_bytes<TY, RT>()), s, a);
  else
    hipLaunchKernelGGL((prefill_reg_big_kernel<TY, RT, false>), grid, dim3(64 * kBigWaves), (big_lds_bytes<TY, RT>()), s, a);
}

template <uint32_t TY, int TT> void launch_shape(const PrefillGemmArgs &a, int row_waves, hipStream_t s) {
  const size_t lds = lds_bytes<TY>(TT, row_waves);
  const int rows = a.w2 ? a.dual_rows : a.n, tile = prefill_reg_row_tile(a.w2 != nullptr) * row_waves;
  const dim3 grid((unsigned)((rows + tile - 1) / tile), (unsigned)((a.t + 16 * TT - 1) / (16 * TT)), (unsigned)a.ksplit);
  const dim3 block(64 * (row_waves + 1) * KW);
  if (a.w2)
    hipLaunchKernelGGL((prefill_reg_kernel<TY, TT, true>), grid, block, lds, s, a);
  else
    hipLaunchKernelGGL((prefill_reg_kernel<TY, TT, false>), grid, block, lds, s, a);
}

// F16 and BF16 rows come in units of 128 columns, too few for a 16-token
// tile's two buffers of four steps.
int token_tiles(uint32_t type, int t) {
  return t > 32 ? 4 : t > 16 || type == LLRS_F16 || type == LLRS_BF16 ? 2 : 1;
}

}  // namespace

bool prefill_reg_supports(uint32_t type) {
  return type == LLRS_Q4_K || type == LLRS_Q6_K || type == LLRS_Q8_0 || type == LLRS_Q5_0 || type == LLRS_F16 ||
         type == LLRS_BF16;
}

int prefill_reg_max_row_waves() { return kMaxRowWaves; }
int prefill_reg_row_tile(bool dual) { return 16 * (dual ? kSmallRT / 2 : kSmallRT); }
int prefill_reg_big_row_tile(uint32_t type, bool dual) {
  return kBigWaves * 16 * (dual ? big_row_tiles(type) / 2 : big_row_tiles(type));
}
int prefill_reg_token_tile(uint32_t type, int t) { return 16 * token_tiles(type, t); }

void launch_prefill_reg(const PrefillGemmArgs &a, int row_waves, hipStream_t s) {
  const int tt = token_tiles(a.type, a.t);
#define REG(T)                                      \
  case T:                                           \
    if (row_waves == 0) {                           \
      if constexpr (Row<T>::kUnit != kNone) launch_big<T>(a, s); \
    } else if (tt == 1) {                                  \
      if constexpr (Row<T>::kCols == 256) launch_shape<T, 1>(a, row_waves, s); \
    } else if (tt == 2) {                           \
      launch_shape<T, 2>(a, row_waves, s);          \
    } else {                                        \
      launch_shape<T, 4>(a, row_waves, s);          \
    }                                               \
    break;
  switch (a.type) {
    REG(LLRS_Q4_K) REG(LLRS_Q6_K) REG(LLRS_Q8_0) REG(LLRS_Q5_0) REG(LLRS_F16) REG(LLRS_BF16)
    default: break;
  }
#undef REG
}

}  // namespace llrs
