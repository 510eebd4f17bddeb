// lmx_digit.hpp -- device-side building blocks of the digit kernels
// (included by the .hip sources only): weight planes to signed bytes,
// activations to signed-byte digits, and the 8-bit matrix-core step.
//
// A digit kernel computes sum_k W[r,k] x[k] of one 128-chunk in whole
// numbers.  The chunk's activations become 31-bit fixed point relative to a
// power of two at or above their largest magnitude, each split into four
// signed bytes ("digits", v = d0 + 2^8 d1 + 2^16 d2 + 2^24 d3); the weight
// codes become signed bytes; v_mfma_i32_16x16x64_i8 sums their products
// exactly.  Only the fixed point (2^-31 of that power of two) and the joins and
// fp32 sums over chunks round.  A chunk whose values lie too far apart for a
// fixed point (wide_chunks) is multiplied in fp32 instead: its activations are
// kept as they are in the place of their digits, its multiplier is 0, and
// raw_sum adds their products.
//
// Matrix-core layout (A 16 x 64 = digits, B 64 x 16 = weights, C 16 x 16):
//   A: lane (i = lane % 16, kq = lane / 16) holds row i's bytes of k-slot kq
//   B: lane (j, kq) holds weight row j's bytes of k-slot kq
//   C: lane (j, g) item d = row 4 g + d, column j
// Row i = 4 n + d is digit d of vector n of a "quad" of 4 vectors, so lane
// (j, g) ends with the four digit sums of weight row j and vector g.
// A 128-chunk takes two steps m = 0, 1; k-slot kq is the 32-bit plane word kq
// of the chunk, and its byte B of dword u in step m is k = 32 kq + 8 B + 7 - t
// with t = 4 m + u: the bit of weight k = 8 B + 7 - t is bit t of byte B of a
// plane word (MSB-first planes), so dword t of an unpacked word holds the
// four weights at bit t of its four bytes, whatever the format.
#ifndef LMX_DIGIT_HPP
#define LMX_DIGIT_HPP

#include <hip/hip_runtime.h>

#include "lmx_device.hpp"

namespace lmx {

typedef int v4i __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t bit_select(uint32_t mask, uint32_t a, uint32_t b) {
  return (a & mask) | (b & ~mask);   // v_bfi_b32
}

// Bits 4i + {0,1} / 4i + {2,3} of four planes' words -> nibbles: n[t] nibble
// i holds the four plane bits at word bit 4 i + t.
__device__ __forceinline__ void nibbles(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, uint32_t (&n)[4]) {
  const uint32_t a = bit_select(0x55555555u, w0, w1 << 1), b = bit_select(0x55555555u, w0 >> 1, w1);
  const uint32_t c = bit_select(0x55555555u, w2, w3 << 1), d = bit_select(0x55555555u, w2 >> 1, w3);
  n[0] = bit_select(0x33333333u, a, c << 2);
  n[2] = bit_select(0x33333333u, a >> 2, c);
  n[1] = bit_select(0x33333333u, b, d << 2);
  n[3] = bit_select(0x33333333u, b >> 2, d);
}

// Passes over the planes (one product per scale stage), and the factor 2^-SH
// the bytes carry too much.
template <int FMT> struct Code { static constexpr int SH = 4; };                 // int4: 16 (q - 8)
template <> struct Code<LMX_FMT_INT3> { static constexpr int SH = 5; };          // 32 (q - 4)
template <> struct Code<LMX_FMT_TERNARY> { static constexpr int SH = 6; };
template <> struct Code<LMX_FMT_BINARY> { static constexpr int SH = 6; };
template <> struct Code<LMX_FMT_RRQ2> { static constexpr int SH = 6; };
template <> struct Code<LMX_FMT_RRQ3> { static constexpr int SH = 6; };
template <> struct Code<LMX_FMT_INT8> { static constexpr int SH = 0; };

// Two-bit two's complement values (lo, hi) -> bytes 64 * value.
__device__ __forceinline__ void pair_bytes(uint32_t lo, uint32_t hi, uint32_t (&out)[8]) {
  const uint32_t a = bit_select(0x55555555u, lo, hi << 1), b = bit_select(0x55555555u, lo >> 1, hi);
#pragma unroll
  for (int t = 0; t < 8; t += 2) {
    out[t] = (a << (6 - t)) & 0xC0C0C0C0u;
    out[t + 1] = (b << (6 - t)) & 0xC0C0C0C0u;
  }
}

// The plane words w[P] of 32 weights -> their signed bytes of scale stage s,
// dword t = the weights at bit t of the word's four bytes.
template <int FMT>
__device__ __forceinline__ void code_bytes(const uint32_t *w, int s, uint32_t (&out)[8]) {
  if constexpr (FMT == LMX_FMT_TERNARY) {
    pair_bytes(~w[1], w[0] & ~w[1], out);             // +1 = 01, -1 = 11, 0 = 00
  } else if constexpr (FMT == LMX_FMT_BINARY || FMT == LMX_FMT_RRQ2 || FMT == LMX_FMT_RRQ3) {
    pair_bytes(0xFFFFFFFFu, ~w[s], out);              // bit 1: +1 = 01, bit 0: -1 = 11
  } else if constexpr (FMT == LMX_FMT_INT8) {
    uint32_t lo[4], hi[4];
    nibbles(w[0], w[1], w[2], w[3], lo);
    nibbles(w[4], w[5], w[6], w[7], hi);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      out[t] = bit_select(0x0F0F0F0Fu, lo[t], hi[t] << 4);
      out[t + 4] = bit_select(0x0F0F0F0Fu, lo[t] >> 4, hi[t]);
    }
  } else {
    // offset binary with the top plane inverted = two's complement, in the
    // byte's high nibble (int3: one place up, the low plane 0)
    uint32_t n[4];
    if constexpr (FMT == LMX_FMT_INT3) nibbles(0u, w[0], w[1], ~w[2], n);
    else nibbles(w[0], w[1], w[2], ~w[3], n);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      out[t] = (n[t] << 4) & 0xF0F0F0F0u;
      out[t + 4] = n[t] & 0xF0F0F0F0u;
    }
  }
}

// Where a kernel reads weight codes from: the handle's code copy (4-bit: the
// four nibble words of a plane word, one load and 12 operations per 32
// weights instead of 4 loads and 28; 8-bit: the bytes themselves) or the
// plane tiles.  CW: 32-bit words per plane word of a row.
template <int FMT, bool COPY> struct Source { static constexpr int CW = Fmt<FMT>::P; };
template <> struct Source<LMX_FMT_INT4, true> { static constexpr int CW = 4; };
template <> struct Source<LMX_FMT_INT8, true> { static constexpr int CW = 8; };
template <int FMT> constexpr bool has_copy() { return FMT == LMX_FMT_INT4 || FMT == LMX_FMT_INT8; }

// The code words of plane word kq of weight rows row0 + li in 128-chunk ch;
// ch and row0 are wave-uniform, so a lane's part of the address is 32 bits.
template <int FMT, bool COPY, bool STREAM>
__device__ __forceinline__ void load_codes(const GemvArgs &a, uint32_t ch, uint32_t row0, uint32_t li, uint32_t kq,
                                           uint32_t (&w)[Source<FMT, COPY>::CW]) {
  constexpr int CW = Source<FMT, COPY>::CW;
  const size_t Npad = size_t(uint32_t(a.Npad));
  if constexpr (COPY) {
    const u32x4 *p = static_cast<const u32x4 *>(a.codes) + (ch * Npad + row0) * CW + (li * 4 + kq) * (CW / 4);
#pragma unroll
    for (int i = 0; i < CW / 4; ++i) {
      const u32x4 v = STREAM ? __builtin_nontemporal_load(p + i) : p[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[4 * i + j] = v[j];
    }
  } else if constexpr (CW % 4 == 0) {
    // a whole row of plane 4 i + kq (four words, dealt out by plane_words): a
    // quarter of the loads that single words take (us, words / rows: 4-bit 256 x
    // 2048 3.64 / 3.22, 8192 x 8192 11.8 / 9.7, 8-bit 2048 x 8192 10.4 / 7.2)
    const u32x4 *p = static_cast<const u32x4 *>(a.planes) + ch * CW * Npad + row0;
#pragma unroll
    for (int i = 0; i < CW / 4; ++i) {
      const u32x4 *q = p + (4 * i + kq) * Npad + li;
      const u32x4 v = STREAM ? __builtin_nontemporal_load(q) : *q;
#pragma unroll
      for (int j = 0; j < 4; ++j) w[4 * i + j] = v[j];
    }
  } else {
    const uint32_t *p = static_cast<const uint32_t *>(a.planes) + (ch * CW * Npad + row0) * 4;
#pragma unroll
    for (int i = 0; i < CW; ++i) {
      const uint32_t *q = p + i * Npad * 4 + (li * 4 + kq);
      w[i] = STREAM ? __builtin_nontemporal_load(q) : *q;
    }
  }
}

// Four planes loaded a row per lane (lane group g: word j of plane g in w[j]) ->
// word g of plane j in w[j]: the groups' two bits change places with j's.
__device__ __forceinline__ void plane_words(uint32_t (&w)[4]) {
  const auto swap16 = [&](int i, int j) {
    const auto r = __builtin_amdgcn_permlane16_swap(w[i], w[j], false, false);
    w[i] = r[0], w[j] = r[1];
  };
  const auto swap32 = [&](int i, int j) {
    const auto r = __builtin_amdgcn_permlane32_swap(w[i], w[j], false, false);
    w[i] = r[0], w[j] = r[1];
  };
  swap16(0, 1);
  swap16(2, 3);
  swap32(0, 2);
  swap32(1, 3);
}

// Code words -> signed bytes (code_bytes).
template <int FMT, bool COPY>
__device__ __forceinline__ void source_bytes(const uint32_t *w, int s, uint32_t (&out)[8]) {
  if constexpr (COPY && FMT == LMX_FMT_INT8) {
#pragma unroll
    for (int t = 0; t < 8; ++t) out[t] = w[t];
  } else if constexpr (COPY) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      out[t] = (w[t] << 4) & 0xF0F0F0F0u;
      out[t + 4] = w[t] & 0xF0F0F0F0u;
    }
  } else if constexpr (Source<FMT, COPY>::CW % 4 == 0) {
    constexpr int CW = Source<FMT, COPY>::CW;
    uint32_t p[CW];
#pragma unroll
    for (int i = 0; i < CW; i += 4) {
      uint32_t q[4] = {w[i], w[i + 1], w[i + 2], w[i + 3]};
      plane_words(q);
#pragma unroll
      for (int j = 0; j < 4; ++j) p[i + j] = q[j];
    }
    code_bytes<FMT>(p, s, out);
  } else {
    code_bytes<FMT>(w, s, out);
  }
}

// Largest-magnitude bits of a 31-bit split: the biased exponent field e such
// that every |x| < 2^(e - 126), from the largest |x|'s bits.  At least 29, so
// that 2^(156 - e) and 2^(e - 156) are floats (smaller values are multiplied in
// fp32, see wide_chunks).
__device__ __forceinline__ int split_exponent(uint32_t max_bits) { return max(int(max_bits >> 23), 29); }
constexpr uint32_t kNotFinite = 0x7F800000u;   // bits of |x| at or above: infinite or NaN

// The factor of the fixed point, a power of two (a product, where ldexp takes
// 1.7 times its issue time).
__device__ __forceinline__ float fixed_factor(int e) { return __uint_as_float(uint32_t(283 - e) << 23); }

__device__ __forceinline__ int round_int(float v) {   // floor(v + 0.5) in one operation, exact
  int r;
  asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

// Four activations (x[B], B = 0..3) at 2^(156 - e) fixed point, rounded ->
// dg[d] = their digits d, byte B from x[B].
__device__ __forceinline__ void digits4(const float (&x)[4], int e, uint32_t (&dg)[4]) {
  const float f = fixed_factor(e);
  uint32_t u[4];   // digits 0..2 each 128 up
#pragma unroll
  for (int b = 0; b < 4; ++b) u[b] = uint32_t(round_int(x[b] * f)) + 0x00808080u;
  const uint32_t a = __builtin_amdgcn_perm(u[1], u[0], 0x05010400u), b = __builtin_amdgcn_perm(u[1], u[0], 0x07030602u);
  const uint32_t c = __builtin_amdgcn_perm(u[3], u[2], 0x05010400u), d = __builtin_amdgcn_perm(u[3], u[2], 0x07030602u);
  dg[0] = __builtin_amdgcn_perm(c, a, 0x05040100u) ^ 0x80808080u;
  dg[1] = __builtin_amdgcn_perm(c, a, 0x07060302u) ^ 0x80808080u;
  dg[2] = __builtin_amdgcn_perm(d, b, 0x05040100u) ^ 0x80808080u;
  dg[3] = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

// The digit sums start from the bits of 1.5 * 2^23: |sum| <= 128 * 128 * 128 =
// 2^21, so the bits of start + sum are the float 1.5 * 2^23 + sum.  One
// register quad per kernel; the asm keeps it from being made again per use.
constexpr float kSumStart = 12582912.0f;
__device__ __forceinline__ v4i sum_start() {
  const int m = __float_as_int(kSumStart);
  v4i z = {m, m, m, m};
  asm volatile("" : "+v"(z));
  return z;
}

// The digit sums of one output -> the fixed-point product sum as a float:
// 256 d - kSumStart is exact, so each pair of digits rounds once, as a 32-bit
// integer of the pair would.  Additions and multiply-adds only: integer shifts
// and conversions take 1.6 times their issue time (1.95 against 1.2 ns per
// SIMD; with 384 vectors, us: 8192 x 2048 39.7 to 38.6, RRQ-3 17920 x 1536 127
// to 122).
__device__ __forceinline__ float join_digits(const v4i d) {
  const float lo = fmaf(__int_as_float(d[1]), 256.0f, -257.0f * kSumStart) + __int_as_float(d[0]);
  const float hi = fmaf(__int_as_float(d[3]), 256.0f, -257.0f * kSumStart) + __int_as_float(d[2]);
  return fmaf(hi, 65536.0f, lo);
}

// The same from sums that start at 0, for kernels without registers for the
// start: pairs of digits join exactly in 32 bits.
__device__ __forceinline__ float join_digits_int(const v4i d) {
  const int lo = (d[1] << 8) + d[0], hi = (d[3] << 8) + d[2];
  return fmaf(float(hi), 65536.0f, float(lo));
}

// One 128-chunk of 16 weight rows against a quad: acc (the start) + the
// digit sums of scale stage s (f0, f1: the quad's digit fragments of steps 0 and 1).
__device__ __forceinline__ v4i chunk_product(const uint32_t (&wb)[8], const v4i f0, const v4i f1, v4i acc) {
  const v4i b0 = {int(wb[0]), int(wb[1]), int(wb[2]), int(wb[3])};
  const v4i b1 = {int(wb[4]), int(wb[5]), int(wb[6]), int(wb[7])};
  acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(f0, b0, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(f1, b1, acc, 0, 0, 0);
}

// The products of a chunk that is kept as it is: the sum over the 32 weights of
// plane word kq in wb against their activations, 16 floats from `lo` (step 0)
// and 16 from `hi` (step 1): x[B] of the lane whose k is bit t of the bytes is
// float 4 (t % 4) + B of step t / 4.  Seldom run: it takes as few registers as it
// can, so that the kernels keep the waves they have without it.
__device__ __forceinline__ float raw_sum(const uint32_t (&wb)[8], const char *lo, const char *hi) {
  float s0 = 0.0f, s1 = 0.0f;   // two sums of 16: half the rounding of one of 32
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const float4 x = *reinterpret_cast<const float4 *>((t < 4 ? lo : hi) + (t & 3) * 16);
    s0 = fmaf(float(int(wb[t] << 24) >> 24), x.x, s0);
    s1 = fmaf(float(int(wb[t] << 16) >> 24), x.y, s1);
    s0 = fmaf(float(int(wb[t] << 8) >> 24), x.z, s0);
    s1 = fmaf(float(int(wb[t]) >> 24), x.w, s1);
    __builtin_amdgcn_sched_barrier(0);
  }
  return s0 + s1;
}

// Lane roles while digits are made, a 256-chunk per wave: lane = chunk c (1
// bit), plane word kq (2), k within the byte kl (3); item B is k =
// 128 c + 32 kq + 8 B + kl, bit t = 7 - kl of byte B.
struct DigitLane {
  int c, kq, kl;
  __device__ __forceinline__ explicit DigitLane(int lane) : c(lane >> 5), kq((lane >> 3) & 3), kl(lane & 7) {}
  __device__ __forceinline__ int k(int b) const { return 128 * c + 32 * kq + 8 * b + kl; }
};

// Largest over the 16 lanes of a row (every lane gets it).
__device__ __forceinline__ uint32_t row_max(uint32_t m) {
  m = max(m, dpp_u32<0xB1>(m));    // lane ^ 1
  m = max(m, dpp_u32<0x4E>(m));    // lane ^ 2
  m = max(m, dpp_u32<0x141>(m));   // lane ^ 7: the other four of eight
  return max(m, dpp_u32<0x140>(m));   // lane ^ 15: the other eight of sixteen
}

// |x| bits of a lane's four activations, the largest; and over the 32 lanes of a chunk.
__device__ __forceinline__ uint32_t lane_max_bits(const float (&x)[4]) {
  uint32_t b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = __float_as_uint(x[i]) & 0x7FFFFFFFu;
  return max(max(b[0], b[1]), max(b[2], b[3]));
}
__device__ __forceinline__ uint32_t chunk_max_bits(uint32_t lane_max) {
  const uint32_t m = row_max(lane_max);
  const auto r = __builtin_amdgcn_permlane16_swap(m, m, false, false);
  return max(uint32_t(r[0]), uint32_t(r[1]));
}

// Which of a wave's two 128-chunks are wide (bits 0 and 1): more than half of the
// lanes with a nonzero value have their largest of four below 2^-8 of the power
// of two that the fixed point is relative to (exponent e).  Rounding leaves each
// value off by about 2^-32 of that power; up to there (84 % of Gaussian values
// below it) that is at most 2^-23.5 of a typical value, what fp32 sums of the
// values round off too (1.0e-7 to 1.3e-7 of an output), even for a row without
// weight for the largest.  Wave-uniform, as is maybe_wide: whether one
// may be, the last `zeros` lanes being known to be zero, without a branch.
__device__ __forceinline__ uint64_t small_lanes(uint32_t lane_max, int e) {
  return __builtin_amdgcn_ballot_w64(lane_max < uint32_t(e - 7) << 23);
}
__device__ __forceinline__ bool maybe_wide(uint32_t lane_max, int e, int zeros) {
  const int lanes = kWave - zeros;   // in the chunk that has fewer of them
  return 2 * (__builtin_popcountll(small_lanes(lane_max, e)) - zeros) > (lanes > 32 ? lanes - 32 : lanes);
}
__device__ __forceinline__ unsigned wide_chunks(uint32_t lane_max, int e) {
  const uint64_t nonzero = __builtin_amdgcn_ballot_w64(lane_max != 0), small = small_lanes(lane_max, e) & nonzero;
  const bool lo = 2 * __builtin_popcount(uint32_t(small)) > __builtin_popcount(uint32_t(nonzero));
  const bool hi = 2 * __builtin_popcount(uint32_t(small >> 32)) > __builtin_popcount(uint32_t(nonzero >> 32));
  return unsigned(lo) | unsigned(hi) << 1;
}

// Whether one of the two is wide at the exponent of the whole vector, where a
// chunk with few values may have them all far below a largest that lies elsewhere
// and is no outlier: more than 16 of its lanes, or all that are not zero, or wide
// by itself.
__device__ __forceinline__ bool far_chunks(uint32_t lane_max, int e) {
  const uint64_t nonzero = __builtin_amdgcn_ballot_w64(lane_max != 0), small = small_lanes(lane_max, e) & nonzero;
  const uint32_t z0 = uint32_t(nonzero), z1 = uint32_t(nonzero >> 32), s0 = uint32_t(small), s1 = uint32_t(small >> 32);
  if (__builtin_popcount(s0) > 16 || __builtin_popcount(s1) > 16 || (z0 && s0 == z0) || (z1 && s1 == z1)) return true;
  return nonzero != ~uint64_t(0) && wide_chunks(lane_max, split_exponent(chunk_max_bits(lane_max)));
}

// The multiplier of a chunk's digits.
__device__ __forceinline__ float chunk_mult(uint32_t max_bits, int e, bool wide) {
  if (max_bits >= kNotFinite) return __builtin_nanf("");
  return wide ? 0.0f : __builtin_amdgcn_ldexpf(1.0f, e - 156);
}

}  // namespace lmx

#endif  // LMX_DIGIT_HPP
