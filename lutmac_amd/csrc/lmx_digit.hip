// lmx_digit.hip -- activations split into digits once for many vectors, and
// the dispatch of the digit kernels over the weight formats.
#include "lmx_digit_kernels.hpp"

namespace lmx {

// lmx_digit_fmt.hip, one translation unit per format
template <int FMT> int digit_gemv_fmt(const GemvArgs &a, int nv, void *stream);
template <int FMT> int digit_gemm_fmt(const GemvArgs &a, const DigitVectors &d, void *stream);
template <int FMT> int code_copy_fmt(const void *planes, size_t Npad, size_t Kp, void *codes, void *stream);

namespace {

// A lane's four activations of vector n of a quad's chunk qc: their digits, or
// the activations themselves (16 bytes where the digits have 4 rows of 4).
__device__ __forceinline__ void store_digits(const DigitVectors &d, size_t qc, int n, const DigitLane &dl,
                                             const float (&o)[4], int e, bool wide) {
  const int t = 7 - dl.kl;
  char *dst = d.digits + qc * kQuadChunk + (t >> 2) * 1024 + (dl.kq * 16 + n * 4) * 16;
  if (wide) {
    *reinterpret_cast<float4 *>(dst + (t & 3) * 16) = make_float4(o[0], o[1], o[2], o[3]);
    return;
  }
  uint32_t dg[4];
  digits4(o, e, dg);
#pragma unroll
  for (int q = 0; q < 4; ++q) *reinterpret_cast<uint32_t *>(dst + q * 16 + (t & 3) * 4) = dg[q];
}

// ---------------------------------------------------------------------------
// Digits of many vectors, one workgroup per vector (tile form):
// dig[quad][chunk][step][lane][16 B].  Relative to the vector's largest, which
// saves the products a multiplier per chunk, unless its values lie too far apart
// (far_chunks); then (d.exp kFarVector) relative to each chunk's.  Bound by the
// latency of the row's read and its maximum; up to K = 8192 the row stays in
// registers between the passes (512 vectors of 2048: 4.4 us, once a call, where
// every row block of the products would make them again).
template <bool ROT, int XM>
__global__ __launch_bounds__(512) void digit_split_kernel(const float *__restrict__ x, int cols, int Kp,
                                                          const float *__restrict__ xw, float eps, float factor,
                                                          DigitVectors d) {
  constexpr int NW = 8;
  __shared__ uint32_t mx[NW], wd[NW];
  __shared__ float ssw[NW];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int v = blockIdx.x;
  const DigitLane dl(lane);
  const int pairs = Kp / kRotChunk;
  x += size_t(v) * cols;
  float ss = 0.0f;
  const auto values = [&](int c2, float (&o)[4]) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int k = c2 * kRotChunk + dl.k(b), kc = min(k, cols - 1);
      float t = x[kc];
      if constexpr (XM == kXModeRmsNorm) {
        t = k < cols ? t : 0.0f;
        ss = fmaf(t, t, ss);
        t *= xw[kc];
      }
      o[b] = k < cols ? t : 0.0f;
    }
    if constexpr (ROT) fwht256_regs_x16(o[0], o[1], o[2], o[3], lane);
  };
  constexpr int KEEP = 4;   // 256-chunks of a wave kept between the passes (K <= 8192)
  float keep[KEEP][4];
  uint32_t m = 0;
#pragma unroll
  for (int j = 0; j < KEEP; ++j) {
    if (wave + j * NW < pairs) {
      values(wave + j * NW, keep[j]);
      m = max(m, lane_max_bits(keep[j]));
    }
  }
  for (int c2 = wave + KEEP * NW; c2 < pairs; c2 += NW) {
    float o[4];
    values(c2, o);
    m = max(m, lane_max_bits(o));
  }
  m = row_max(m);
  m = max(m, lane_xor_u32<16>(m, lane));
  m = max(m, lane_xor_u32<32>(m, lane));
  if constexpr (XM == kXModeRmsNorm) ss = lane_sum<32>(ss, lane);
  if (lane == 0) {
    mx[wave] = m;
    ssw[wave] = ss;
  }
  __syncthreads();
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    m = max(m, mx[i]);
    sum += ssw[i];
  }
  const int ev = split_exponent(m);
  bool far = false;
#pragma unroll
  for (int j = 0; j < KEEP; ++j)
    if (wave + j * NW < pairs) far |= far_chunks(lane_max_bits(keep[j]), ev);
  for (int c2 = wave + KEEP * NW; c2 < pairs; c2 += NW) {
    float o[4];
    values(c2, o);
    far |= far_chunks(lane_max_bits(o), ev);
  }
  if (lane == 0) wd[wave] = far;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NW; ++i) far |= wd[i] != 0;
  if (m >= kNotFinite) far = false;
  if (threadIdx.x == 0) {
    float f = factor;
    if constexpr (XM == kXModeRmsNorm) f *= 1.0f / sqrtf(sum / float(cols) + eps);
    d.fac[v] = m >= kNotFinite ? __builtin_nanf("") : f;
    d.exp[v] = far ? kFarVector : ev - 156;
  }
  const size_t first = size_t(v >> 2) * size_t(Kp / kChunk);
  const auto emit = [&](int c2, const float (&o)[4]) {
    const size_t qc = first + size_t(2 * c2 + dl.c);
    int e = ev;
    bool wide = false;
    if (far) {
      const uint32_t lm = lane_max_bits(o), mb = chunk_max_bits(lm);
      e = split_exponent(mb);
      wide = (wide_chunks(lm, e) >> dl.c) & 1;
      if ((lane & 31) == 0) d.mult[qc * 4 + (v & 3)] = chunk_mult(mb, e, wide);
    }
    store_digits(d, qc, v & 3, dl, o, e, wide);
  };
#pragma unroll
  for (int j = 0; j < KEEP; ++j)
    if (wave + j * NW < pairs) emit(wave + j * NW, keep[j]);
  for (int c2 = wave + KEEP * NW; c2 < pairs; c2 += NW) {
    float o[4];
    values(c2, o);
    emit(c2, o);
  }
}

// Digits relative to each 128-chunk (rows form): one wave per vector and
// 256-chunk, so that a few long vectors spread over the chip (16 vectors of
// 8960: 3.9 us).  RMSNorm: the first workgroup of a
// vector sums its squares over the whole row.
template <int XM>
__global__ __launch_bounds__(256) void digit_split_chunks_kernel(const float *__restrict__ x, int cols, int Kp,
                                                                 const float *__restrict__ xw, float eps, float factor,
                                                                 unsigned rotate, DigitVectors d) {
  constexpr int NW = 4;
  __shared__ float ssw[NW];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
  const int v = int(blockIdx.y), c2 = int(blockIdx.x) * NW + wave;
  const DigitLane dl(lane);
  x += size_t(v) * cols;
  float o[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int k = c2 * kRotChunk + dl.k(b);
    const uint32_t kc = uint32_t(min(k, cols - 1));
    float t = x[kc];
    if constexpr (XM == kXModeRmsNorm) t *= xw[kc];
    o[b] = k < cols ? t : 0.0f;
  }
  if (blockIdx.x == 0) {   // the vector's factor
    float f = factor;
    if constexpr (XM == kXModeRmsNorm) {
      float ss = 0.0f;
      for (int k = threadIdx.x; k < cols; k += 256) ss = fmaf(x[k], x[k], ss);
      ss = lane_sum<32>(ss, lane);
      if (lane == 0) ssw[wave] = ss;
      __syncthreads();
      f *= 1.0f / sqrtf(((ssw[0] + ssw[1]) + (ssw[2] + ssw[3])) / float(cols) + eps);
    }
    if (threadIdx.x == 0) d.fac[v] = f;
  }
  if (c2 * kRotChunk >= Kp) return;   // wave-uniform; no barrier follows
  if (rotate == LMX_ROTATE_FWHT256) fwht256_regs_x16(o[0], o[1], o[2], o[3], lane);
  const uint32_t lm = lane_max_bits(o), mb = chunk_max_bits(lm);
  const int e = split_exponent(mb);
  const bool wide = (wide_chunks(lm, e) >> dl.c) & 1;
  const size_t qc = size_t(v >> 2) * size_t(Kp / kChunk) + size_t(2 * c2 + dl.c);
  store_digits(d, qc, v & 3, dl, o, e, wide);
  if ((lane & 31) == 0) {
    d.mult[qc * 4 + (v & 3)] = chunk_mult(mb, e, wide);
    if (v == d.count - 1)   // the last quad's other vectors, so that theirs are no 0
      for (int n = (v & 3) + 1; n < 4; ++n) d.mult[qc * 4 + n] = 1.0f;
  }
}

}  // namespace

// Two row tiles per workgroup once that leaves a workgroup per CU: each makes
// the digits of the whole K (4-bit, us, one tile against two: 2048 x 2048
// 3.18 / 3.44, 3072 x 2048 3.35 / 3.56, 17920 x 1536 5.54 / 5.27, 8192 x 8192
// 12.0 / 8.0).  A workgroup has a wave per 256-chunk and a thread per output
// of its 4 vectors, so a K of one 256-chunk keeps to one tile.
int digit_gemv_tiles(const GemvArgs &a) {
  return a.epi == kEpiSiluPair || (a.Npad / kTile >= 512 && a.Kp > kRotChunk) ? 2 : 1;
}

size_t digit_argmax_slots(const GemvArgs &a) { return size_t(a.Npad) / (kTile * digit_gemv_tiles(a)); }

// The epilogues and transforms every digit kernel serves: a SiLU pair has
// whole 16-row tiles in each half.
static int check_digit_args(const GemvArgs &a, bool norm_pairs) {
  const bool pair = a.epi == kEpiSiluPair;
  if (pair && a.rows % (2 * kTile))
    return fail(LMX_ERR_INVALID_ARGUMENT, "a SiLU pair of %d rows has no whole row tiles", a.rows);
  if ((a.xmode != kXModeNone && a.xmode != kXModeRmsNorm) || (pair && norm_pairs && a.xmode != kXModeRmsNorm))
    return fail(LMX_ERR_INVALID_ARGUMENT, "the digit kernels do not serve transform %d with epilogue %d", a.xmode, a.epi);
  return LMX_OK;
}

int launch_digit_gemv(int fmt, const GemvArgs &a, int nv, void *stream) {
  if (const int st = check_digit_args(a, true)) return st;
  switch (fmt) {
  case LMX_FMT_TERNARY: return digit_gemv_fmt<LMX_FMT_TERNARY>(a, nv, stream);
  case LMX_FMT_BINARY: return digit_gemv_fmt<LMX_FMT_BINARY>(a, nv, stream);
  case LMX_FMT_RRQ2: return digit_gemv_fmt<LMX_FMT_RRQ2>(a, nv, stream);
  case LMX_FMT_RRQ3: return digit_gemv_fmt<LMX_FMT_RRQ3>(a, nv, stream);
  case LMX_FMT_INT3: return digit_gemv_fmt<LMX_FMT_INT3>(a, nv, stream);
  case LMX_FMT_INT4: return digit_gemv_fmt<LMX_FMT_INT4>(a, nv, stream);
  case LMX_FMT_INT8: return digit_gemv_fmt<LMX_FMT_INT8>(a, nv, stream);
  }
  return fail(LMX_ERR_UNSUPPORTED_FORMAT, "unknown format %d", fmt);
}

static float code_factor(int fmt, unsigned rotate) {
  int sh = 6;
  if (fmt == LMX_FMT_INT4) sh = 4;
  if (fmt == LMX_FMT_INT3) sh = 5;
  if (fmt == LMX_FMT_INT8) sh = 0;
  return (rotate == LMX_ROTATE_FWHT256 ? 0.0625f : 1.0f) / float(1 << sh);
}

// digits, mult, fac and exp of `vectors` vectors
size_t digit_bytes(size_t Kp, size_t vectors) {
  const size_t quads = (vectors + 3) / 4;
  return quads * (Kp / kChunk) * (kQuadChunk + 16) + quads * 32;
}

size_t digit_capacity(size_t Kp, size_t bytes) {
  return bytes > kDigitPartials ? (bytes - kDigitPartials) / digit_bytes(Kp, 4) * 4 : 0;
}

DigitVectors digit_vectors(const lmx_weight *w, void *scratch, unsigned *tickets, size_t count) {
  DigitVectors d{};
  d.tickets = tickets;
  const size_t quads = (count + 3) / 4, chunks = w->Kp / kChunk;
  d.digits = static_cast<char *>(scratch);
  d.mult = reinterpret_cast<float *>(d.digits + quads * chunks * kQuadChunk);
  d.fac = d.mult + quads * chunks * 4;
  d.exp = reinterpret_cast<int *>(d.fac + quads * 4);
  d.partials = reinterpret_cast<float *>(d.exp + quads * 4);
  d.count = int(count);
  // The tile kernel from a workgroup of 8 row tiles x 4 quads for every other
  // CU (us, tile / rows form: 8192 x 2048 x 32 vectors 11.9 / 10.8, 17920 x
  // 1536 x 16 10.8 / 12.7, 3001 x 1400 x 128 11.1 / 13.3); with fewer than 4
  // quads from as many products (17920 x 1536 x 8 11.7 / 9.7, 128256 x 2048 x
  // 8 33 / 48).
  d.tile = (w->Npad / kTile + 7) / 8 * quads > 512;
  return d;
}

int launch_digit_split(int fmt, const GemvArgs &a, const DigitVectors &d, void *stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  const float f = code_factor(fmt, a.rotate);
  const bool rot = a.rotate == LMX_ROTATE_FWHT256;
  if (!d.tile) {
    const dim3 grid{unsigned((a.Kp / kRotChunk + 3) / 4), unsigned(d.count)};
    if (a.xmode == kXModeRmsNorm)
      digit_split_chunks_kernel<kXModeRmsNorm><<<grid, dim3(256), 0, st>>>(a.x, a.cols, a.Kp, a.xw, a.eps, f, a.rotate, d);
    else
      digit_split_chunks_kernel<kXModeNone><<<grid, dim3(256), 0, st>>>(a.x, a.cols, a.Kp, a.xw, a.eps, f, a.rotate, d);
    return launched("digit_split_chunks");
  }
#define LMX_SP(R, XM) \
  digit_split_kernel<R, XM><<<dim3(unsigned(d.count)), dim3(512), 0, st>>>(a.x, a.cols, a.Kp, a.xw, a.eps, f, d)
  if (a.xmode == kXModeRmsNorm) {
    if (rot) LMX_SP(true, kXModeRmsNorm); else LMX_SP(false, kXModeRmsNorm);
  } else {
    if (rot) LMX_SP(true, kXModeNone); else LMX_SP(false, kXModeNone);
  }
#undef LMX_SP
  return launched("digit_split");
}

int launch_digit_gemm(int fmt, const GemvArgs &a, const DigitVectors &d, void *stream) {
  if (const int st = check_digit_args(a, false)) return st;
  if (code_copy_bytes(fmt, 1, kRotChunk) && !a.codes)
    return fail(LMX_ERR_INVALID_ARGUMENT, "the split digit kernels need the code copy of format %d", fmt);
  switch (fmt) {
  case LMX_FMT_TERNARY: return digit_gemm_fmt<LMX_FMT_TERNARY>(a, d, stream);
  case LMX_FMT_BINARY: return digit_gemm_fmt<LMX_FMT_BINARY>(a, d, stream);
  case LMX_FMT_RRQ2: return digit_gemm_fmt<LMX_FMT_RRQ2>(a, d, stream);
  case LMX_FMT_RRQ3: return digit_gemm_fmt<LMX_FMT_RRQ3>(a, d, stream);
  case LMX_FMT_INT3: return digit_gemm_fmt<LMX_FMT_INT3>(a, d, stream);
  case LMX_FMT_INT4: return digit_gemm_fmt<LMX_FMT_INT4>(a, d, stream);
  case LMX_FMT_INT8: return digit_gemm_fmt<LMX_FMT_INT8>(a, d, stream);
  }
  return fail(LMX_ERR_UNSUPPORTED_FORMAT, "unknown format %d", fmt);
}

size_t code_copy_bytes(int fmt, size_t Npad, size_t Kp) {
  return fmt == LMX_FMT_INT4 ? Npad * Kp / 2 : fmt == LMX_FMT_INT8 ? Npad * Kp : 0;
}

int launch_code_copy(int fmt, const void *planes, size_t Npad, size_t Kp, void *codes, void *stream) {
  if (fmt == LMX_FMT_INT4) return code_copy_fmt<LMX_FMT_INT4>(planes, Npad, Kp, codes, stream);
  if (fmt == LMX_FMT_INT8) return code_copy_fmt<LMX_FMT_INT8>(planes, Npad, Kp, codes, stream);
  return LMX_OK;
}

}  // namespace lmx
