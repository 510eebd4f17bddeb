// lmx_digit_kernels.hpp -- GEMV and GEMM kernels on the 8-bit matrix cores
// with exact products (lmx_digit.hpp: the digit split, layouts, identities),
// included by the .hip sources only.
//
//   digit_gemv_kernel   1..4 vectors in one launch: every wave makes the
//                       digits of its own 256-chunks in LDS and multiplies
//                       them with its rows
//   digit_rows_kernel   few split vectors or few rows: k over the waves of a
//                       workgroup, fragments straight from the caches
//   digit_tile_kernel   many split vectors and rows: fragments staged in LDS
#ifndef LMX_DIGIT_KERNELS_HPP
#define LMX_DIGIT_KERNELS_HPP

#include <hip/hip_runtime.h>

#include <cstdlib>

#include "lmx_digit.hpp"

namespace lmx {
namespace {

constexpr int kTile = 16;          // weight rows per matrix-core tile
constexpr uint32_t kQuadChunk = 2048;   // digit bytes of a quad's 128-chunk

__device__ __forceinline__ int scale_group(const GemvArgs &a, int ch) {
  return a.gshift >= 0 ? ch >> a.gshift : ch / a.group_chunks;
}

// The lane once more, for loops that seldom run: what they derive from it then
// takes no register through the loops before them.
__device__ __forceinline__ int lane_again() {
  int lane = int(threadIdx.x) & (kWave - 1);
  asm volatile("" : "+v"(lane));
  return lane;
}

// ---------------------------------------------------------------------------
// 1..4 vectors, one launch: RT row tiles per workgroup, the whole K over its
// waves (wave w takes the 256-chunks w, w + W, ... , PPW of them a round).
// NV = 1: the fragment rows of the other three vectors of a quad hold other
// 128-chunks' digits instead (chunk q of a group of four in rows 4 q .. 4 q +
// 3, zeros elsewhere), so four chunks' digit sums land in four lane groups of
// one accumulator and are joined and scaled once.
// NV = 4: one accumulator per chunk, its four lane groups the four vectors.
// From about 20 MB of codes bound by HBM (4-bit 8192 x 8192 7.5 us, 4.8 TB/s,
// 8.0 on the lookup tables; 8-bit 15.2 us, 4.6 TB/s, 16.5), below that by one
// chain of launch, activations, digits, products and the waves' sum: so every
// load of a round is requested at the start, activations first, and 16 waves
// share the K.  Four vectors cost 4-bit 17920 x 1536 6.9 us where the bf16
// matrix cores and their reduction took 10.8.
template <int FMT, bool COPY, int NV, int RT, int PPW, int XM, int EPI>
__global__ __launch_bounds__(1024) void digit_gemv_kernel(GemvArgs a, int nv) {
  constexpr int CW = Source<FMT, COPY>::CW, S = Fmt<FMT>::S;
  constexpr int ROWS = 4 * NV;                     // fragment rows kept
  // a fragment, 16 bytes longer: the digit writes of the steps and chunks of
  // a 256-chunk (4 lanes each of 16 bytes in 64) start in different banks
  constexpr uint32_t FRAG = 4 * ROWS * 16 + (NV == 1 ? 16 : 0);
  constexpr bool PAIR = EPI == kEpiSiluPair;
  constexpr bool NORM = XM == kXModeRmsNorm;
  constexpr int CH = 2 * PPW;                      // 128-chunks of a wave's round
  constexpr int G = NV == 1 ? 4 : 1;               // chunks per accumulator
  constexpr int NG = (CH + G - 1) / G;
  constexpr int OUT = PAIR ? RT / 2 * kTile : RT * kTile;   // outputs per vector
  __shared__ __attribute__((aligned(16))) char frags[16][CH][2][FRAG];   // [wave][chunk][step]
  __shared__ __attribute__((aligned(16))) uint32_t zeros[4];
  __shared__ float mults[16][CH][NV];
  __shared__ float red[16][RT * kTile * NV];
  __shared__ float ssq[16][NV];

  const int lane = threadIdx.x & (kWave - 1), W = blockDim.x / kWave;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
  const int li = lane & 15, kq = lane >> 4;
  const int pairs = a.Kp / kRotChunk;
  const bool rot = a.rotate == LMX_ROTATE_FWHT256;
  const DigitLane dl(lane);
  const v4i start = sum_start();

  // first row of each tile; PAIR: RT/2 tiles of gate rows, then the matching up rows
  uint32_t row0[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    if constexpr (PAIR)
      row0[t] = uint32_t((t < RT / 2 ? 0 : a.rows / 2) + (int(blockIdx.x) * (RT / 2) + t % (RT / 2)) * kTile);
    else
      row0[t] = uint32_t((int(blockIdx.x) * RT + t) * kTile);
  }
  if (NV == 1 && threadIdx.x < 4) zeros[threadIdx.x] = 0u;

  bool any_wide = false;   // of the wave's chunks, perhaps
  float acc[RT], ss[NV];
#pragma unroll
  for (int t = 0; t < RT; ++t) acc[t] = 0.0f;
#pragma unroll
  for (int n = 0; n < NV; ++n) ss[n] = 0.0f;
  float eb0 = 0.0f, eb1 = 0.0f;   // the epilogue thread's bias and residual terms, requested early
  const int on = int(threadIdx.x) / OUT, orow = int(blockIdx.x) * OUT + int(threadIdx.x) % OUT;
  const bool stores = on < nv && on < NV && orow < (PAIR ? a.rows / 2 : a.rows);

  for (int p0 = wave; p0 < pairs; p0 += PPW * W) {
    // ---- the round's activations, then its weights and scales (indices clamped, masked below) ----
    float xr[PPW][NV][4], xw[PPW][4];
#pragma unroll
    for (int p = 0; p < PPW; ++p) {
      const int c2 = min(p0 + p * W, pairs - 1);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const uint32_t k = uint32_t(min(c2 * kRotChunk + dl.k(b), a.cols - 1));
#pragma unroll
        for (int n = 0; n < NV; ++n) xr[p][n][b] = (a.x + size_t(min(n, nv - 1)) * a.cols)[k];
        if constexpr (NORM) xw[p][b] = a.xw[k];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // every wave's activation requests ahead of the weight stream (and the
    // zeros written): the barrier waits for no load
    if (p0 == wave) {
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
    }
    __builtin_amdgcn_sched_barrier(0);
    uint32_t w[PPW][2][RT][CW];
    float sc[G == 4 ? NG : CH][RT][S];
    const auto load_w = [&](int p) {
      const int c2 = min(p0 + p * W, pairs - 1);
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int t = 0; t < RT; ++t)
          load_codes<FMT, COPY, true>(a, uint32_t(2 * c2 + c), row0[t], uint32_t(li), uint32_t(kq), w[p][c][t]);
    };
    const auto load_s = [&](int i) {
      // G = 4: lane group kq takes chunk 4 i + kq of the round; else chunk i
      const int q = G == 4 ? 4 * i + kq : i;
      const int c2 = min(p0 + (q >> 1) * W, pairs - 1);
      const uint32_t g = uint32_t(scale_group(a, 2 * c2 + (q & 1)));
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int s = 0; s < S; ++s) sc[i][t][s] = (a.scales + row0[t])[uint32_t(s * a.n_groups + g) * uint32_t(a.Npad) + uint32_t(li)];
    };
#pragma unroll
    for (int p = 0; p < PPW; ++p) {
      load_w(p);
      if constexpr (G == 4) {
        if (p % 2 == 0) load_s(p / 2);
      } else {
        load_s(2 * p);
        load_s(2 * p + 1);
      }
    }
    if (p0 == wave && stores) {
      if (a.bias) {
        eb0 = a.bias[orow];
        if constexpr (PAIR) eb1 = a.bias[a.rows / 2 + orow];
      }
      if constexpr (!PAIR)
        if (a.resid) eb1 = a.resid[size_t(on) * a.rows + orow];   // read before this thread stores y (resid may be y)
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- digits of the wave's 256-chunks ----
#pragma unroll
    for (int p = 0; p < PPW; ++p) {
      const int c2 = p0 + p * W;
      const bool live = c2 < pairs;   // else zeros: the chunk adds nothing
      const bool full = c2 * kRotChunk + kRotChunk <= a.cols;
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        float x[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          x[b] = xr[p][n][b];
          if (!full) x[b] = live && c2 * kRotChunk + dl.k(b) < a.cols ? x[b] : 0.0f;   // wave-uniform branch
          if constexpr (NORM) {
            ss[n] = fmaf(x[b], x[b], ss[n]);
            x[b] *= xw[p][b];
          }
        }
        if (rot) fwht256_regs_x16(x[0], x[1], x[2], x[3], lane);
        const uint32_t lm = lane_max_bits(x), mb = chunk_max_bits(lm);
        const int e = split_exponent(mb);
        any_wide |= maybe_wide(lm, e, full || rot ? 0 : ((c2 + 1) * kRotChunk - max(a.cols, c2 * kRotChunk)) / 32 * 8);
        uint32_t dg[4];
        digits4(x, e, dg);
        const int t = 7 - dl.kl;
        char *dst = frags[wave][2 * p + dl.c][t >> 2] + (dl.kq * ROWS + 4 * n) * 16 + (t & 3) * 4;
#pragma unroll
        for (int q = 0; q < 4; ++q) *reinterpret_cast<uint32_t *>(dst + q * 16) = dg[q];
        if ((lane & 31) == 0) mults[wave][2 * p + dl.c][n] = chunk_mult(mb, e, false);
      }
    }
    // a wave reads only the digits it wrote; its LDS operations complete in order
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();

    // ---- products ----
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      v4i sum[RT][S];
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int s = 0; s < S; ++s) sum[t][s] = start;
#pragma unroll
      for (int q = 0; q < G; ++q) {
        const int ch = G * i + q;
        if (ch >= CH) break;
        v4i f[2];
        if constexpr (G == 4) {
          const char *src = frags[wave][ch][0] + (kq * ROWS + (li & 3)) * 16;
          const bool mine = (li >> 2) == q;
#pragma unroll
          for (int m = 0; m < 2; ++m)
            f[m] = *reinterpret_cast<const v4i *>(mine ? src + m * FRAG : reinterpret_cast<const char *>(zeros));
        } else {
#pragma unroll
          for (int m = 0; m < 2; ++m)
            f[m] = *reinterpret_cast<const v4i *>(frags[wave][ch][m] + (kq * ROWS + li) * 16);
        }
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
          for (int s = 0; s < S; ++s) {
            uint32_t wb[8];
            source_bytes<FMT, COPY>(w[ch >> 1][ch & 1][t], s, wb);
            sum[t][s] = chunk_product(wb, f[0], f[1], sum[t][s]);
          }
      }
      // lane group kq: chunk 4 i + kq (G = 4) or vector kq of chunk i; a chunk past the round's adds 0
      const float mult = G == 4 ? (4 * i + kq < CH ? mults[wave][min(4 * i + kq, CH - 1)][0] : 0.0f) : mults[wave][i][kq & (NV - 1)];
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int s = 0; s < S; ++s) acc[t] = fmaf(join_digits(sum[t][s]) * mult, sc[i][t][s], acc[t]);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }

  // ---- wide chunks: the wave goes through its own once more and adds, in fp32,
  // what the fixed point left of their activations (exact: their low bits) ----
  if (any_wide) {
    char *raw = frags[wave][0][0];   // [chunk][vector][step][plane word][64 B]
#pragma unroll 1
    for (int c2 = wave; c2 < pairs; c2 += W) {
      const int lane = lane_again(), li = lane & 15, kq = lane >> 4;
      const DigitLane dl(lane);
      unsigned vecs[2] = {0, 0};   // the vectors whose first and second chunk are wide
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        float x[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int k = c2 * kRotChunk + dl.k(b);
          const uint32_t kc = uint32_t(min(k, a.cols - 1));
          const float v = (a.x + size_t(min(n, nv - 1)) * a.cols)[kc];
          x[b] = k < a.cols ? v : 0.0f;
          if constexpr (NORM) x[b] *= a.xw[kc];
        }
        if (rot) fwht256_regs_x16(x[0], x[1], x[2], x[3], lane);
        const uint32_t lm = lane_max_bits(x);
        const int e = split_exponent(chunk_max_bits(lm)), t = 7 - dl.kl;
        const unsigned wide = wide_chunks(lm, e);
        if (!wide) continue;
        vecs[0] |= (wide & 1) << n;
        vecs[1] |= (wide >> 1) << n;
        const float f = fixed_factor(e), back = __builtin_amdgcn_ldexpf(1.0f, e - 156);
#pragma unroll
        for (int b = 0; b < 4; ++b) x[b] = fmaf(float(round_int(x[b] * f)), -back, x[b]);
        *reinterpret_cast<float4 *>(raw + (dl.c * NV + n) * 512 + (t >> 2) * 256 + dl.kq * 64 + (t & 3) * 16) =
            make_float4(x[0], x[1], x[2], x[3]);
      }
      if (!(vecs[0] | vecs[1])) continue;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll 1
      for (int c = 0; c < 2; ++c) {
        const unsigned mine = c ? vecs[1] : vecs[0];
        if (!mine) continue;
        const uint32_t g = uint32_t(scale_group(a, 2 * c2 + c));
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          uint32_t w[CW], wb[8];
          __builtin_amdgcn_sched_barrier(0);   // registers before latency
          load_codes<FMT, COPY, false>(a, uint32_t(2 * c2 + c), row0[t], uint32_t(li), uint32_t(kq), w);
#pragma unroll
          for (int s = 0; s < S; ++s) {
            const float scale = (a.scales + row0[t])[uint32_t(s * a.n_groups + g) * uint32_t(a.Npad) + uint32_t(li)];
            source_bytes<FMT, COPY>(w, s, wb);
#pragma unroll 1
            for (int n = 0; n < NV; ++n) {
              if (!((mine >> n) & 1)) continue;
              const char *src = raw + (c * NV + n) * 512 + kq * 64;
              float v = raw_sum(wb, src, src + 256);
              if constexpr (NV > 1) {   // lane group n holds vector n
                v += lane_xor<16>(v, lane);
                v += lane_xor<32>(v, lane);
                v = kq == n ? v : 0.0f;
              }
              acc[t] = fmaf(v, scale, acc[t]);
            }
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }

  // ---- the lane groups of a wave (NV = 1), then the waves in order ----
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const float v = NV == 1 ? strided_sum<kTile>(acc[t], lane) : acc[t];
    if (kq < NV) red[wave][kq * RT * kTile + t * kTile + li] = v;
  }
  if constexpr (NORM) {
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const float s = lane_sum<32>(ss[n], lane);
      if (lane == 0) ssq[wave][n] = s;
    }
  }
  __syncthreads();
  float v = 0.0f;
  if (stores) {
    const int r = int(threadIdx.x) % OUT;
    float scale = (rot ? 0.0625f : 1.0f) / float(1 << Code<FMT>::SH);
    if constexpr (NORM) {
      float s = 0.0f;
      for (int k = 0; k < W; ++k) s += ssq[k][on];
      scale *= 1.0f / sqrtf(s / float(a.cols) + a.eps);
    }
    const float *rd = red[0] + on * RT * kTile + r;
    if constexpr (PAIR) {
      float u = 0.0f;
      for (int k = 0; k < W; ++k) {
        v += rd[k * RT * kTile * NV];
        u += rd[k * RT * kTile * NV + OUT];
      }
      a.y[size_t(on) * (a.rows / 2) + orow] = silu(fmaf(v, scale, eb0)) * fmaf(u, scale, eb1);
    } else {
      for (int k = 0; k < W; ++k) v += rd[k * RT * kTile * NV];
      v *= scale;
      if (a.bias) v += eb0;
      if (a.resid) v += eb1;
      a.y[size_t(on) * a.rows + orow] = v;
    }
  }
  if constexpr (!PAIR) {
    if (a.amax && threadIdx.x < kWave)   // one vector, at most 64 rows per workgroup
      wave_argmax(a.amax, blockIdx.x, argmax_value(a, v, orow, stores), orow, stores);
  }
}

// y = sum (times the vector's factor and exponent) (+ bias) (+ resid), or the
// SiLU pair's product, of one output.
__device__ __forceinline__ float vector_scale(float sum, float fac, int ex) {
  return __builtin_amdgcn_ldexpf(sum * fac, ex);
}

// The vectors of a split quad (index `quad`, its chunk qc) that keep the chunk as
// it is: bit 16 n for vector n (and 15 more above it).
__device__ __forceinline__ uint64_t raw_vectors(const DigitVectors &d, int quad, size_t qc, int kq) {
  return __builtin_amdgcn_ballot_w64(4 * quad + kq < d.count && d.mult[qc * 4 + kq] == 0.0f);
}

// Their products with the weights wb of a row tile: lane group n that of vector
// n, 0 for the others.
__device__ __forceinline__ float raw_quad(const uint32_t (&wb)[8], const char *chunk, uint64_t mask, int lane) {
  const int kq = lane >> 4;
  float r = 0.0f;
#pragma unroll 1
  for (int n = 0; n < 4; ++n) {
    if (!((mask >> (16 * n)) & 1)) continue;
    const char *src = chunk + (kq * 16 + n * 4) * 16;
    float v = raw_sum(wb, src, src + 1024);
    v += lane_xor<16>(v, lane);
    v += lane_xor<32>(v, lane);
    r = kq == n ? v : r;
  }
  return r;
}

// ---------------------------------------------------------------------------
// NQ quads of vectors against RT row tiles: a workgroup takes one of gridDim.z
// slices of the chunks, spread over its waves, fragments straight from memory
// (each vector's digits are relative to its chunk: d.mult).  With more than
// one slice the workgroups of a row block leave their sums in d.partials and
// the last one to finish (a ticket) adds them in slice order: agent-scope
// relaxed stores and loads, which need no write-back of the XCDs' L2s.
// Bound by the latency of a wave's one or two chunks (codes, digits, scales in
// one round trip, the second chunk's requested before the first is used):
// hence small tiles, k over 16 waves and slices up to a workgroup per CU.  us,
// with the split, before on the bf16 matrix cores or lookup tables: 4-bit 1536
// x 8960 x 16 vectors 10.9 to 9.0, 3001 x 1400 x 13 17.7 to 8.3, ternary 2048 x
// 2048 x 64 34.3 to 8.6.
template <int FMT, bool COPY, int NQ, int RT, int EPI>
__global__ __launch_bounds__(1024) void digit_rows_kernel(GemvArgs a, DigitVectors d) {
  constexpr int CW = Source<FMT, COPY>::CW, S = Fmt<FMT>::S;
  constexpr bool PAIR = EPI == kEpiSiluPair;
  constexpr int SUMS = RT * NQ * kWave;
  __shared__ float red[16][SUMS];
  __shared__ unsigned ticket;
  const int lane = threadIdx.x & (kWave - 1), W = blockDim.x / kWave;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
  const int li = lane & 15, kq = lane >> 4;
  const int Kc = a.Kp / kChunk;
  constexpr bool TIGHT = NQ * RT > 4;   // of 128 registers a wave
  v4i start = {0, 0, 0, 0};
  if constexpr (!TIGHT) start = sum_start();
  const uint32_t Npad = uint32_t(a.Npad);
  const int quads = (d.count + 3) / 4, q0 = int(blockIdx.y) * NQ;
  const int slices = int(gridDim.z), slice = int(blockIdx.z);
  const int ch0 = Kc * slice / slices, ch1 = Kc * (slice + 1) / slices;
  uint32_t row0[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    if constexpr (PAIR)
      row0[t] = uint32_t((t < RT / 2 ? 0 : a.rows / 2) + (int(blockIdx.x) * (RT / 2) + t % (RT / 2)) * kTile);
    else
      row0[t] = uint32_t((int(blockIdx.x) * RT + t) * kTile);
  }
  const size_t qbytes = size_t(Kc) * kQuadChunk;
  uint32_t w[2][RT][CW];
  float sc[2][RT][S], mu[2][NQ];
  v4i f[2][NQ][2];
  const auto load = [&](int b, int ch) {
    const uint32_t g = uint32_t(scale_group(a, ch));
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      load_codes<FMT, COPY, false>(a, uint32_t(ch), row0[t], uint32_t(li), uint32_t(kq), w[b][t]);
#pragma unroll
      for (int s = 0; s < S; ++s)
        sc[b][t][s] = (a.scales + size_t(s * a.n_groups + g) * Npad + row0[t])[uint32_t(li)];
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int qq = min(q0 + q, quads - 1);
      mu[b][q] = (d.mult + (size_t(qq) * Kc + ch) * 4)[uint32_t(kq)];
#pragma unroll
      for (int m = 0; m < 2; ++m)
        f[b][q][m] = reinterpret_cast<const v4i *>(d.digits + size_t(qq) * qbytes + size_t(ch) * kQuadChunk + m * 1024)[lane];
    }
  };
  uint64_t any_wide = 0;   // lanes with a multiplier of 0 among the wave's chunks (in scalar registers)
  float acc[RT][NQ];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[t][q] = 0.0f;
  const auto work = [&](int b) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) any_wide |= __builtin_amdgcn_ballot_w64(mu[b][q] == 0.0f);
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int s = 0; s < S; ++s) {
        uint32_t wb[8];
        source_bytes<FMT, COPY>(w[b][t], s, wb);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const v4i sum = chunk_product(wb, f[b][q][0], f[b][q][1], start);
          acc[t][q] = fmaf((TIGHT ? join_digits_int(sum) : join_digits(sum)) * mu[b][q], sc[b][t][s], acc[t][q]);
        }
      }
  };
  if (ch0 + wave < ch1) load(0, ch0 + wave);
  for (int ch = ch0 + wave; ch < ch1; ch += 2 * W) {
    if (ch + W < ch1) load(1, ch + W);
    work(0);
    if (ch + W >= ch1) break;
    if (ch + 2 * W < ch1) load(0, ch + 2 * W);
    work(1);
  }
  if (any_wide) {   // chunks kept as they are: the wave goes through its own once more
#pragma unroll 1
    for (int ch = ch0 + wave; ch < ch1; ch += W) {
      const int lane = lane_again(), li = lane & 15, kq = lane >> 4;
      const uint32_t g = uint32_t(scale_group(a, ch));
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const size_t qc = size_t(min(q0 + q, quads - 1)) * Kc + ch;
        const uint64_t mask = raw_vectors(d, q0 + q, qc, kq);
        if (!mask) continue;
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          uint32_t cw[CW], wb[8];
          load_codes<FMT, COPY, false>(a, uint32_t(ch), row0[t], uint32_t(li), uint32_t(kq), cw);
#pragma unroll
          for (int s = 0; s < S; ++s) {
            const float scale = (a.scales + size_t(s * a.n_groups + g) * Npad + row0[t])[uint32_t(li)];
            source_bytes<FMT, COPY>(cw, s, wb);
            acc[t][q] = fmaf(raw_quad(wb, d.digits + qc * kQuadChunk, mask, lane), scale, acc[t][q]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int q = 0; q < NQ; ++q) red[wave][(t * NQ + q) * kWave + lane] = acc[t][q];
  __syncthreads();
  const auto wg_sum = [&](int o) {
    float v = 0.0f;
    for (int k = 0; k < W; ++k) v += red[k][o];
    return v;
  };
  const size_t blocks = size_t(gridDim.x) * gridDim.y, block = size_t(blockIdx.y) * gridDim.x + blockIdx.x;
  if (slices > 1) {
    float *part = d.partials + (size_t(slice) * blocks + block) * SUMS;
    for (int o = threadIdx.x; o < SUMS; o += blockDim.x)
      __hip_atomic_store(part + o, wg_sum(o), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0)
      ticket = __hip_atomic_fetch_add(d.tickets + block, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (ticket != unsigned(slices - 1)) return;   // uniform over the workgroup
    if (threadIdx.x == 0) __hip_atomic_store(d.tickets + block, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const auto total = [&](int o) {
    if (slices == 1) return wg_sum(o);
    float v = 0.0f;
    const float *part = d.partials + block * SUMS + o;
    for (int s0 = 0; s0 < slices; s0 += 8) {   // 8 loads in flight, summed in order
      float t[8];
#pragma unroll
      for (int s = 0; s < 8; ++s)
        t[s] = s0 + s < slices ? __hip_atomic_load(part + size_t(s0 + s) * blocks * SUMS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0f;
#pragma unroll
      for (int s = 0; s < 8; ++s) v += t[s];
    }
    return v;
  };
  // output o: (tile, quad, lane) -> row tile * 16 + lane % 16, vector 4 quad + lane / 16
  constexpr int OUT = (PAIR ? RT / 2 : RT) * NQ * kWave;
  for (int o = threadIdx.x; o < OUT; o += blockDim.x) {
    const int l = o & (kWave - 1), q = (o / kWave) % NQ, t = o / (kWave * NQ);
    const int vec = 4 * (q0 + q) + (l >> 4);
    if (vec >= d.count) continue;
    const float fac = d.fac[vec];
    float v = total(o) * fac;
    if constexpr (PAIR) {
      const int h = a.rows / 2, row = (int(blockIdx.x) * (RT / 2) + t) * kTile + (l & 15);
      float u = total(OUT + o) * fac;
      if (a.bias) v += a.bias[row], u += a.bias[h + row];
      a.y[size_t(vec) * h + row] = silu(v) * u;
    } else {
      const int row = (int(blockIdx.x) * RT + t) * kTile + (l & 15);
      if (row < a.rows) {
        if (a.bias) v += a.bias[row];
        if (a.resid) v += a.resid[size_t(vec) * a.rows + row];
        a.y[size_t(vec) * a.rows + row] = v;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Many vectors: 4 waves of RT row tiles x the same NQ quads, the quads'
// fragments of a chunk staged in LDS (two chunks deep); with KS = 2 a second
// set of 4 waves takes every other pair of chunks and the two sums are added
// at the end (half the serial chain where few workgroups are in flight).
// Bound by instruction issue: per 64 products 192 float operations join the
// sums and 64 unpack codes and address; products alone take 32 ns of the 73 ns
// that 4 products and their share take a SIMD (8192 x 2048 x 512 vectors: 46 us
// for 14 us of products).  So 4 waves per SIMD (128 registers) come first: 8
// quads request fragments one chunk ahead, not two.  Halving the LDS reads (2 x
// 2 waves of 4 row tiles) was 20 % slower for its extra unpacking.
template <int FMT, bool COPY, int NQ> constexpr int tile_waves() {
  return NQ == 8 && (Source<FMT, COPY>::CW > 4 || Fmt<FMT>::S > 1) ? 3 : 4;
}

template <int FMT, bool COPY, int NQ, int RT, int KS, int EPI>
__global__ __launch_bounds__(256 * KS, (tile_waves<FMT, COPY, NQ>())) void digit_tile_kernel(GemvArgs a, DigitVectors d) {
  constexpr int CW = Source<FMT, COPY>::CW, S = Fmt<FMT>::S;
  constexpr bool PAIR = EPI == kEpiSiluPair;
  constexpr int WAVES = 4;
  __shared__ __attribute__((aligned(16))) char frags_all[KS][2][NQ * kQuadChunk];
  const int lane = threadIdx.x & (kWave - 1), tid = int(threadIdx.x) % 256;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int kg = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(int(threadIdx.x) / 256);   // the wave's part of k
  auto &frags = frags_all[kg];
  const int li = lane & 15, kq = lane >> 4;
  const int Kc = a.Kp / kChunk;
  const v4i start = sum_start();
  const uint32_t Npad = uint32_t(a.Npad);
  const int quads = (d.count + 3) / 4, q0 = int(blockIdx.y) * NQ;
  const int wg = int(blockIdx.x) * WAVES + wave;   // the wave's group of RT tiles
  const int half_rows = a.rows / 2;
  uint32_t row0[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    if constexpr (PAIR)   // groups past the last redo it and are not stored
      row0[t] = uint32_t((t < RT / 2 ? 0 : half_rows) +
                         min((wg * (RT / 2) + t % (RT / 2)) * kTile, half_rows - kTile));
    else
      row0[t] = uint32_t(min((wg * RT + t) * kTile, a.Npad - kTile));
  }
  const size_t qbytes = size_t(Kc) * kQuadChunk;
  constexpr int LD = NQ * int(kQuadChunk) / (256 * 16);   // 16-byte pieces per thread and chunk
  static_assert(LD * 256 * 16 == NQ * int(kQuadChunk), "whole pieces");
  // A chunk's codes (and fragments: FD) are requested two chunks ahead: they
  // come from the MALL where another XCD wrote or read them first.  Past the
  // last chunk the last one is requested again.
  uint32_t w[2][RT][CW];
  float sc[2][RT][S];
  constexpr int FD = NQ == 8 ? 1 : 2;   // chunks the fragments are requested ahead
  v4i st[FD][LD];
  const char *fsrc[LD];   // wave-uniform: a wave's piece i is half of quad 2 i + wave / 2
#pragma unroll
  for (int i = 0; i < LD; ++i) fsrc[i] = d.digits + size_t(min(q0 + 2 * i + wave / 2, quads - 1)) * qbytes;
  const uint32_t foff = uint32_t(tid % 128) * 16;
  // exponents of the workgroup's vectors, in every wave: lane 4 q + n that of vector n of quad q
  const int ex_lane = d.exp[min(4 * q0 + lane % (4 * NQ), d.count - 1)];
  const auto load_f = [&](int b, int ch) {
    const size_t c = size_t(min(ch, Kc - 1)) * kQuadChunk;
#pragma unroll
    for (int i = 0; i < LD; ++i) st[b % FD][i] = *reinterpret_cast<const v4i *>(fsrc[i] + c + foff);
  };
  const auto store_f = [&](int b) {
#pragma unroll
    for (int i = 0; i < LD; ++i) *reinterpret_cast<v4i *>(frags[b] + (tid + 256 * i) * 16) = st[b % FD][i];
  };
  const auto load_w = [&](int b, int ch) {
    ch = min(ch, Kc - 1);
    const uint32_t g = uint32_t(scale_group(a, ch));
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      load_codes<FMT, COPY, false>(a, uint32_t(ch), row0[t], uint32_t(li), uint32_t(kq), w[b][t]);
#pragma unroll
      for (int s = 0; s < S; ++s)
        sc[b][t][s] = (a.scales + size_t(s * a.n_groups + g) * Npad + row0[t])[uint32_t(li)];
    }
  };
  float acc[RT][NQ];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[t][q] = 0.0f;
  const auto chunk = [&](int ch, const int b) {   // b = ch % 2
    if constexpr (FD == 2) load_f(b, ch + 2 * KS);
    else load_f(b ^ 1, b == 0 ? ch + 1 : ch - 1 + 2 * KS);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      uint32_t wb[RT][8];
      float cs[RT];
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        source_bytes<FMT, COPY>(w[b][t], s, wb[t]);
        cs[t] = KS == 1 || ch < Kc ? sc[b][t][s] : 0.0f;   // past the last chunk: adds nothing
      }
      if (s == S - 1) load_w(b, ch + 2 * KS);   // the words are bytes now
      // The products of quad q run while quad q - 1's sums are joined and quad
      // q + 1's fragments arrive; the barriers keep the compiler from issuing
      // every quad's reads and products first (registers).
      v4i f[2][2], sum[2][RT];
      const auto read = [&](int q) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
          f[q & 1][m] = *reinterpret_cast<const v4i *>(frags[b] + q * kQuadChunk + m * 1024 + lane * 16);
      };
      read(0);
#pragma unroll
      for (int q = 0; q <= NQ; ++q) {
        __builtin_amdgcn_sched_barrier(0);
        if (q + 1 < NQ) read(q + 1);
        if (q < NQ) {
#pragma unroll
          for (int t = 0; t < RT; ++t) sum[q & 1][t] = chunk_product(wb[t], f[q & 1][0], f[q & 1][1], start);
        }
        if (q > 0) {
#pragma unroll
          for (int t = 0; t < RT; ++t) {
            acc[t][q - 1] = fmaf(join_digits(sum[(q - 1) & 1][t]), cs[t], acc[t][q - 1]);
            asm volatile("" : "+v"(acc[t][q - 1]));   // else every join sinks to the chunk's end
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    store_f(b ^ 1);
    __syncthreads();
  };
  load_f(0, 2 * kg);
  load_w(0, 2 * kg);
  if constexpr (FD == 2) load_f(1, 2 * kg + 1);
  load_w(1, 2 * kg + 1);
  store_f(0);
  __syncthreads();
#pragma unroll 1
  for (int c0 = 0; c0 < Kc; c0 += 2 * KS) {   // Kc is even; every part makes the same rounds
    chunk(c0 + 2 * kg, 0);
    chunk(c0 + 2 * kg + 1, 1);
  }
  // Far vectors (rare): their sums start again, chunk by chunk with the chunk's
  // multiplier, a quad at a time straight from memory; the others add 0.
  const uint64_t far = __builtin_amdgcn_ballot_w64(ex_lane == kFarVector);   // bit 4 q + n: vector n of quad q
  if (far) {
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int t = 0; t < RT; ++t) acc[t][q] = (far >> (4 * q + kq)) & 1 ? 0.0f : acc[t][q];
#pragma unroll 1
    for (int ch = kg; ch < Kc; ch += KS) {
      load_w(0, ch);
#pragma unroll
      for (int s = 0; s < S; ++s) {
        uint32_t wb[RT][8];
#pragma unroll
        for (int t = 0; t < RT; ++t) source_bytes<FMT, COPY>(w[0][t], s, wb[t]);
#pragma unroll
        for (int q1 = 0; q1 < NQ; q1 += 2) {   // two quads' loads at a time
          if (!((far >> (4 * q1)) & 255)) continue;   // wave-uniform
          __builtin_amdgcn_sched_barrier(0);
          const int lane = lane_again(), kq = lane >> 4;
          v4i f[2][2];
          float mu[2];
          const char *chunk[2];
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const size_t qc = size_t(min(q0 + q1 + i, quads - 1)) * Kc + ch;
            chunk[i] = d.digits + qc * kQuadChunk;
            const v4i *src = reinterpret_cast<const v4i *>(chunk[i]) + lane;
            f[i][0] = src[0], f[i][1] = src[64];
            mu[i] = d.mult[qc * 4 + kq];
          }
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int q = q1 + i;
            const bool mine = (far >> (4 * q + kq)) & 1;
            const uint64_t raw = __builtin_amdgcn_ballot_w64(mine && mu[i] == 0.0f);
#pragma unroll
            for (int t = 0; t < RT; ++t) {
              const float j = join_digits(chunk_product(wb[t], f[i][0], f[i][1], start));
              acc[t][q] = fmaf(mine ? j * mu[i] : 0.0f, sc[0][t][s], acc[t][q]);
            }
            if (raw) {
#pragma unroll
              for (int t = 0; t < RT; ++t) acc[t][q] = fmaf(raw_quad(wb[t], chunk[i], raw, lane), sc[0][t][s], acc[t][q]);
            }
          }
        }
      }
    }
  }
  if constexpr (KS > 1) {   // the parts of k, in order
    float *red = reinterpret_cast<float *>(frags_all[0][0]);
    constexpr int SUMS = RT * NQ * 256;
    static_assert((KS - 1) * SUMS * sizeof(float) <= sizeof(frags_all), "sums in place of the fragments");
    if (kg > 0) {
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int q = 0; q < NQ; ++q) red[(kg - 1) * SUMS + (t * NQ + q) * 256 + tid] = acc[t][q];
    }
    __syncthreads();
    if (kg > 0) return;   // wave-uniform; no barrier follows
#pragma unroll
    for (int p = 0; p < KS - 1; ++p)
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int q = 0; q < NQ; ++q) acc[t][q] += red[p * SUMS + (t * NQ + q) * 256 + tid];
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int vec = 4 * (q0 + q) + kq;
    if (vec >= d.count) continue;
    const float fac = d.fac[vec];
    const int ev = d.exp[vec], ex = ev == kFarVector ? 0 : ev;
#pragma unroll
    for (int t = 0; t < (PAIR ? RT / 2 : RT); ++t) {
      float v = vector_scale(acc[t][q], fac, ex);
      if constexpr (PAIR) {
        const int row = (wg * (RT / 2) + t) * kTile + li;
        if (row >= half_rows) continue;
        float u = vector_scale(acc[RT / 2 + t][q], fac, ex);
        if (a.bias) v += a.bias[row], u += a.bias[half_rows + row];
        a.y[size_t(vec) * half_rows + row] = silu(v) * u;
      } else {
        const int row = (wg * RT + t) * kTile + li;
        if (row >= a.rows) continue;
        if (a.bias) v += a.bias[row];
        if (a.resid) v += a.resid[size_t(vec) * a.rows + row];
        a.y[size_t(vec) * a.rows + row] = v;
      }
    }
  }
}

int launched(const char *what) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? LMX_OK : fail(LMX_ERR_LAUNCH_FAILED, "%s launch: %s", what, hipGetErrorString(e));
}

// Batches come with a handle, so with its code copy where the format has one.
template <int FMT, int NQ, int RT>
int launch_rows(const GemvArgs &a, const DigitVectors &d, hipStream_t st) {
  constexpr bool COPY = has_copy<FMT>();
  const bool pair = a.epi == kEpiSiluPair;
  const int Kc = a.Kp / kChunk, W = Kc >= 16 ? 16 : Kc;
  const unsigned gx = pair ? a.rows / 2 / (RT / 2 > 0 ? RT / 2 : 1) / kTile : a.Npad / RT / kTile;
  const unsigned gy = ((d.count + 3) / 4 + NQ - 1) / NQ;
  // slices of the chunks where the row blocks alone leave most CUs idle, each
  // wave keeping at least a chunk
  // (at most 256 workgroups then: their tickets and sums fit the scratch)
  int slices = 1;
  while (gx * gy * (slices + 1) <= 256 && Kc / (slices + 1) >= W) ++slices;
  const dim3 grid{gx, gy, unsigned(slices)}, block{unsigned(W * kWave)};
  if (pair) {
    if constexpr (RT >= 2) digit_rows_kernel<FMT, COPY, NQ, RT, kEpiSiluPair><<<grid, block, 0, st>>>(a, d);
  } else {
    digit_rows_kernel<FMT, COPY, NQ, RT, kEpiStore><<<grid, block, 0, st>>>(a, d);
  }
  return launched("digit_rows");
}

template <int FMT, int NQ, int RT, int KS>
int launch_tile(const GemvArgs &a, const DigitVectors &d, hipStream_t st) {
  constexpr bool COPY = has_copy<FMT>();
  const int quads = (d.count + 3) / 4;
  const int groups = a.epi == kEpiSiluPair ? (a.rows / 2 / kTile + RT / 2 - 1) / (RT / 2) : (a.Npad / kTile + RT - 1) / RT;
  const dim3 grid{unsigned((groups + 3) / 4), unsigned((quads + NQ - 1) / NQ)};
  if (a.epi == kEpiSiluPair) digit_tile_kernel<FMT, COPY, NQ, RT, KS, kEpiSiluPair><<<grid, dim3(256 * KS), 0, st>>>(a, d);
  else digit_tile_kernel<FMT, COPY, NQ, RT, KS, kEpiStore><<<grid, dim3(256 * KS), 0, st>>>(a, d);
  return launched("digit_tile");
}

template <int FMT>
int launch_gemm_fmt(const GemvArgs &a, const DigitVectors &d, hipStream_t st) {
  const int quads = (d.count + 3) / 4, tiles = a.Npad / kTile;
  if (d.tile) {
    // 8 quads a workgroup where that leaves two of them per CU and no more
    // padding than 4 quads would (us: 16384 x 2048 x 256 vectors 47 / 51,
    // 8192 x 2048 x 256 30.4 / 29.9, x 128 21.3 / 18.7; 16 vectors 52 / 35 of
    // 128256 rows).  Up to two workgroups per CU, two of their halves of k
    // each (2048 x 8192 x 512 57.4 against 60.8, 8192 x 2048 x 64 12.7 / 14.9,
    // 17920 x 1536 x 64, with 560 workgroups, 20.9 / 18.8).
    const int q4 = (quads + 3) / 4, q8 = (quads + 7) / 8, blocks = (tiles + 7) / 8;
    if (blocks * q8 >= 512 && 10 * 2 * q8 < 11 * q4) return launch_tile<FMT, 8, 2, 1>(a, d, st);
    if (blocks * q4 > 512) return launch_tile<FMT, 4, 2, 1>(a, d, st);
    return launch_tile<FMT, 4, 2, 2>(a, d, st);
  }
  // The smallest tile that one workgroup per CU covers the call with: then the
  // reads of one workgroup, a chunk or two per wave, are what takes the time
  // (us, 4 quads x 2 row tiles / chosen: 2048 x 2048 x 16 vectors 6.9 / 5.8,
  // 1536 x 8960 x 16 9.7 / 8.9, x 8 9.4 / 7.5); beyond that the largest, which
  // reads the codes least often (17920 x 1536 x 16 12.8, 2 quads 13.4).
  const auto fits = [&](int nq, int rt) { return tiles / rt * ((quads + nq - 1) / nq) <= 256; };
  const bool one = a.epi != kEpiSiluPair;
  if (one && fits(1, 1)) return launch_rows<FMT, 1, 1>(a, d, st);
  if (one && quads > 1 && fits(2, 1)) return launch_rows<FMT, 2, 1>(a, d, st);
  if (quads == 1 || fits(1, 2)) return launch_rows<FMT, 1, 2>(a, d, st);
  if (quads == 2 || fits(2, 2)) return launch_rows<FMT, 2, 2>(a, d, st);
  return launch_rows<FMT, 4, 2>(a, d, st);
}

template <int FMT, bool COPY, int NV, int RT, int PPW>
int launch_digit_gemv_cfg(const GemvArgs &a, int nv, int W, hipStream_t st) {
  const dim3 block{unsigned(W * kWave)};
  const bool pair = a.epi == kEpiSiluPair;
  const dim3 grid{unsigned(pair ? a.rows / 2 / (kTile * RT / 2) : a.Npad / (kTile * RT))};
  if (pair) {
    if constexpr (RT == 2)
      digit_gemv_kernel<FMT, COPY, NV, RT, PPW, kXModeRmsNorm, kEpiSiluPair><<<grid, block, 0, st>>>(a, nv);
  } else if (a.xmode == kXModeRmsNorm) {
    digit_gemv_kernel<FMT, COPY, NV, RT, PPW, kXModeRmsNorm, kEpiStore><<<grid, block, 0, st>>>(a, nv);
  } else {
    digit_gemv_kernel<FMT, COPY, NV, RT, PPW, kXModeNone, kEpiStore><<<grid, block, 0, st>>>(a, nv);
  }
  return launched("digit_gemv");
}

template <int FMT, bool COPY, int NV, int RT>
int launch_digit_gemv_rt(const GemvArgs &a, int nv, hipStream_t st) {
  // as few rounds of 256-chunks per wave as 16 waves allow, spread evenly
  const int pairs = a.Kp / kRotChunk;
  const int per = (pairs + 15) / 16;
  const int W = (pairs + per - 1) / per;
  if constexpr (NV == 1) {
    // two 256-chunks per wave and round; in the last of several rounds few waves
    // have a second one, so all 16 share them (us, W even over single chunks / 16:
    // 256 x 8960 5.49 / 4.92, from planes 7.20 / 6.06)
    if (per >= 2) return launch_digit_gemv_cfg<FMT, COPY, NV, RT, 2>(a, nv, per == 2 ? W : 16, st);
  }
  return launch_digit_gemv_cfg<FMT, COPY, NV, RT, 1>(a, nv, W, st);
}

template <int FMT, bool COPY>
int launch_digit_gemv_src(const GemvArgs &a, int nv, hipStream_t st) {
  const bool two = digit_gemv_tiles(a) == 2;
  if (nv == 1) {
    // 8-bit codes of one vector from the planes: their loads are whole 16-byte
    // rows side by side, the copy's alternate 16 of a row's 32 bytes (us, copy /
    // planes: 512 x 2048 3.89 / 3.48, 8192 x 8192 16.4 / 14.5, 512 x 8960 10.2 /
    // 8.5; four vectors, whose codes come once for four products, 3.07 / 3.25 at
    // 512 x 640, 6.16 / 6.35 at 8192 x 2048, 11.4 / 10.4 at 512 x 8960)
    constexpr bool C = COPY && FMT != LMX_FMT_INT8;
    return two ? launch_digit_gemv_rt<FMT, C, 1, 2>(a, nv, st) : launch_digit_gemv_rt<FMT, C, 1, 1>(a, nv, st);
  }
  // Four row tiles share one making of four vectors' digits (us, two tiles /
  // four: 4-bit 10240 x 2048 5.76 / 5.26, 16384 x 4096 11.4 / 8.3, ternary
  // 32768 x 2048 14.1 / 12.1; 8192 x 2048 4.34 / 5.18, 17920 x 1536 7.3 / 8.3).
  // (Not the 8-bit and three-stage formats, whose codes and scales of four
  // tiles spill.)
  if constexpr (FMT != LMX_FMT_INT8 && FMT != LMX_FMT_RRQ3) {
    if (a.epi != kEpiSiluPair && a.Npad / kTile >= 640 && a.Kp >= 2048)
      return launch_digit_gemv_rt<FMT, COPY, 4, 4>(a, nv, st);
  }
  return two ? launch_digit_gemv_rt<FMT, COPY, 4, 2>(a, nv, st) : launch_digit_gemv_rt<FMT, COPY, 4, 1>(a, nv, st);
}

template <int FMT>
int launch_digit_gemv_fmt(const GemvArgs &a, int nv, hipStream_t st) {
  if constexpr (has_copy<FMT>()) {
    if (a.codes) return launch_digit_gemv_src<FMT, true>(a, nv, st);
  }
  return launch_digit_gemv_src<FMT, false>(a, nv, st);
}

// The code copy of 4- and 8-bit planes: one thread per plane word of a row.
// HBM-bound (128256 x 2048 of 4 bits: 42 us); made here and not on the host,
// creating a 17920 x 1536 handle takes 2 ms where it took 13.
template <int FMT>
__global__ __launch_bounds__(256) void code_copy_kernel(const uint32_t *__restrict__ planes, uint32_t Npad, size_t n,
                                                        uint32_t *__restrict__ codes) {
  constexpr int P = Fmt<FMT>::P;
  const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;   // (chunk * Npad + row) * 4 + kq
  if (i >= n) return;
  const size_t rk = i % (size_t(Npad) * 4), ch = i / (size_t(Npad) * 4);
  uint32_t w[P];
#pragma unroll
  for (int p = 0; p < P; ++p) w[p] = planes[(ch * P + p) * Npad * 4 + rk];
  if constexpr (FMT == LMX_FMT_INT4) {
    uint32_t nib[4];
    nibbles(w[0], w[1], w[2], ~w[3], nib);
#pragma unroll
    for (int j = 0; j < 4; ++j) codes[i * 4 + j] = nib[j];
  } else {
    uint32_t out[8];
    code_bytes<FMT>(w, 0, out);
#pragma unroll
    for (int j = 0; j < 8; ++j) codes[i * 8 + j] = out[j];
  }
}

template <int FMT>
int launch_code_copy_fmt(const void *planes, size_t Npad, size_t Kp, void *codes, hipStream_t st) {
  if constexpr (has_copy<FMT>()) {
    const size_t n = Kp / kChunk * Npad * 4;
    code_copy_kernel<FMT><<<dim3(unsigned((n + 255) / 256)), dim3(256), 0, st>>>(
        static_cast<const uint32_t *>(planes), uint32_t(Npad), n, static_cast<uint32_t *>(codes));
    return launched("code_copy");
  }
  return LMX_OK;
}

}  // namespace
}  // namespace lmx

#endif  // LMX_DIGIT_KERNELS_HPP
