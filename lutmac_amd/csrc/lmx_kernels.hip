// lmx_kernels.hip -- gfx950 kernels of the bit-serial LUT-GEMV path.
//
// One GEMV is one launch of a full-K kernel where its tables fit, or
// lut_gemv_kernel (split-K, last-workgroup reduction) elsewhere.  Full-K
// launches with plain activations run lut_gemv_ipl_kernel (interleaved table
// build and lookups) or lut_gemv_plain_kernel (lean front end); fused
// transforms and the argmax epilogue run lut_gemv_fullk_kernel.  All share:
//   * a fused prologue: each wavefront takes 256-chunks of x, rotates them
//     with an in-register FWHT-256 (cross-lane butterflies via shuffles)
//     when asked, and writes the 16-entry partial-sum table of every group
//     of 4 activations straight into LDS (lane l owns group l of a chunk);
//   * the lookup loop: every lane streams one row's bit-planes (one 16-byte
//     non-temporal load per plane per 128-k chunk, 1 KiB contiguous per
//     wavefront), turns each plane nibble into an LDS address with one
//     v_perm and accumulates the looked-up partial sums in fp32.  All 64
//     lanes read the same 16-entry table at a time, so a lookup touches 16
//     consecutive dwords: no bank conflicts;
//   * deterministic reductions (fixed slice order, no float atomics).
// Full-K: a workgroup owns 64/H rows and the whole K (tables of the whole K
// in LDS), k-slices spread over its lanes, slice partials summed in LDS (a
// lane butterfly inside each wave, then the waves in order).
// Split-K: a workgroup owns 64*WAVES rows x one k-slice and writes one
// partial per row; a second kernel (or the last workgroup) sums them.
//
// Per-format identities (T = group table, m_p = plane-p nibble, ~ = 4-bit
// complement, xs = sum of the chunk's activations):
//   ternary  T[~s&~z] - T[s&~z]                    (lut_gemm.hpp:79-99)
//   binary   2*T[m] - T[15]
//   RRQ-k    sum_i s_i * (2*T[m_i] - T[15])        (Int2Block::get generalised)
//   int3     T[m0] + 2T[m1] - 4T[~m2]              ((q-4) with q = 4b2+2b1+b0)
//   int4     T[m0] + 2T[m1] + 4T[m2] - 8T[~m3]     ((q-8))
//   int8     sum_{b<7} 2^b T[m_b] - 128 T[m7]      (two's complement)
#include <hip/hip_runtime.h>

#include <cstdlib>

#include "lmx_device.hpp"

namespace lmx {

// ---------------------------------------------------------------------------
template <int FMT, int CHUNKS, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void lut_gemv_kernel(GemvArgs a, int row_blocks, int splits) {
  constexpr int P = Fmt<FMT>::P, NA = Fmt<FMT>::NA, S = Fmt<FMT>::S;
  constexpr int KS = CHUNKS * kChunk;
  constexpr int ROWS = WAVES * kWave;
  constexpr int C2 = KS / kRotChunk;  // 256-chunks of the slice
  __shared__ __attribute__((aligned(16))) float tables[KS / 4 * 16];
  __shared__ float xsum[CHUNKS];
  __shared__ float xred[WAVES];
  __shared__ unsigned ticket;

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int rb = blockIdx.x % row_blocks;
  const int split = blockIdx.x / row_blocks;
  const int k0 = split * KS;
  const int row = rb * ROWS + wave * kWave + lane;
  const bool active = rb * ROWS + wave * kWave < a.Npad;  // whole wavefronts

  // ---- loads: this wave's activations first, then the lane's plane and
  // scale words, so the table build below only waits for x while the weight
  // stream is still in flight (vector loads retire in issue order).  Loads
  // are unconditional (indices clamped in bounds) so no branch splits them.
  constexpr int XJ = (C2 + WAVES - 1) / WAVES;
  float xv[XJ][4], aux[XJ][4];
#pragma unroll
  for (int j = 0; j < XJ; ++j) {
    const int c2 = min(wave + j * WAVES, C2 - 1);
    load_x4(a.x, k0 + c2 * kRotChunk, a.cols, lane, xv[j][0], xv[j][1], xv[j][2], xv[j][3]);
  }
  if (a.xmode == kXModeRmsNorm || a.xmode == kXModeSiluMul) {
#pragma unroll
    for (int j = 0; j < XJ; ++j) load_aux4(a, k0 + min(wave + j * WAVES, C2 - 1) * kRotChunk, lane, aux[j]);
  }
  __builtin_amdgcn_sched_barrier(0);  // keep the x loads ahead of the weight stream
  u32x4 w[CHUNKS][P];
  float sc[CHUNKS][S];
  {
    const u32x4 *__restrict__ pl = reinterpret_cast<const u32x4 *>(a.planes);
    const size_t Npad = size_t(a.Npad);
    const int c0 = k0 / kChunk;
    const int lr = min(row, a.Npad - 1);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
#pragma unroll
      for (int p = 0; p < P; ++p)
        w[c][p] = __builtin_nontemporal_load(pl + (size_t(c0 + c) * P + p) * Npad + lr);
      const int g = (c0 + c) / a.group_chunks;
#pragma unroll
      for (int s = 0; s < S; ++s) sc[c][s] = a.scales[(size_t(s) * a.n_groups + g) * Npad + lr];
    }
  }

  // ---- prologue: (transform) -> (FWHT-256) -> 16-entry group tables ------
  // Lane l of the wave owning a 256-chunk holds activations 4l..4l+3 = group
  // l of the chunk and writes that group's table.
  const float inv_rms = a.xmode == kXModeRmsNorm ? wg_inv_rms<ROWS>(a.x, a.cols, a.eps, xred) : 1.0f;
#pragma unroll
  for (int j = 0; j < XJ; ++j) {
    const int c2 = wave + j * WAVES;
    if (c2 >= C2) break;   // wave-uniform
    float x0 = xv[j][0], x1 = xv[j][1], x2 = xv[j][2], x3 = xv[j][3];
    xform4(a.xmode, inv_rms, aux[j], x0, x1, x2, x3);
    if (a.rotate == LMX_ROTATE_FWHT256) fwht256_regs(x0, x1, x2, x3, lane);
    float t[16];
    group_table(x0, x1, x2, x3, t);
    float4 *dst = reinterpret_cast<float4 *>(tables + (c2 * 64 + lane) * 16);
    dst[0] = make_float4(t[0], t[1], t[2], t[3]);
    dst[1] = make_float4(t[4], t[5], t[6], t[7]);
    dst[2] = make_float4(t[8], t[9], t[10], t[11]);
    dst[3] = make_float4(t[12], t[13], t[14], t[15]);
    if constexpr (Fmt<FMT>::XS) {
      float s = t[15];
      s = lane_sum<16>(s, lane);
      if ((lane & 31) == 0) xsum[c2 * 2 + (lane >> 5)] = s;
    }
  }
  __syncthreads();

  // ---- lookups: one row per lane ------------------------------------------
  // All 64 lanes read the same 16-entry table at a time: 16 consecutive
  // dwords, no bank conflicts.  v_perm turns a byte of the pre-shifted plane
  // word into the table offset 4*nibble; the group's table offset is an
  // immediate of the ds_read.
  float acc = 0.0f;
  if (active) {
    const uint32_t tbase = lds_addr(tables);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      float A[NA];
#pragma unroll
      for (int i = 0; i < NA; ++i) A[i] = 0.0f;
      chunk_lookups<FMT>(w[c], tbase + c * (32 * 64), 0u, A);
      float xs = 0.0f;
      if constexpr (Fmt<FMT>::XS) xs = xsum[c];
      acc = finish_chunk<FMT>(A, xs, sc[c], acc);
    }
  }

  // ---- split-K reduction --------------------------------------------------
  if (splits == 1) {
    const float out = a.bias && active && row < a.rows ? acc + a.bias[row] : acc;
    if (active && row < a.rows) a.y[row] = out;
    if (a.amax)
      wave_argmax(a.amax, blockIdx.x * WAVES + wave, argmax_value(a, out, row, active && row < a.rows), row,
                  active && row < a.rows);
    return;
  }
  float *part = a.partials + size_t(split) * a.Npad;
  if (a.reduce == kReduceTwoPass) {
    if (active) part[row] = acc;
    return;
  }
  if (a.reduce == kReduceFenceAll) {
    if (active) part[row] = acc;
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) ticket = atomicAdd(a.counters + rb, 1u);
    __syncthreads();
    if (ticket != unsigned(splits - 1)) return;
    __threadfence();
  } else {
    // Partials travel as agent-scope (device-coherent) relaxed atomic stores
    // and loads, which bypass the non-coherent per-XCD L2 state, so no L2
    // writeback or invalidate is needed.  Each thread waits for its store to
    // complete before the barrier; the ticket is taken after the barrier, so
    // the workgroup that draws the last ticket sees every partial.
    if (active) __hip_atomic_store(part + row, acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0)
      ticket = __hip_atomic_fetch_add(a.counters + rb, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (ticket != unsigned(splits - 1)) return;
  }
  const int r = rb * ROWS + threadIdx.x;
  float out = 0.0f;
  if (r < a.rows) {
    // Sum the partials in split order; loads go out 48 at a time so their
    // latencies overlap (one round trip up to 48 splits, K = 12288 at
    // 256-wide slices).
    constexpr int RL = 48;
    float s = 0.0f;
    const float *pr = a.partials + r;
    for (int k0s = 0; k0s < splits; k0s += RL) {
      float v[RL];
#pragma unroll
      for (int j = 0; j < RL; ++j)
        v[j] = k0s + j < splits
                   ? __hip_atomic_load(pr + size_t(k0s + j) * a.Npad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                   : 0.0f;
#pragma unroll
      for (int j = 0; j < RL; ++j) s += v[j];
    }
    out = a.bias ? s + a.bias[r] : s;
    a.y[r] = out;
  }
  if (a.amax) wave_argmax(a.amax, rb * WAVES + wave, argmax_value(a, out, r, r < a.rows), r, r < a.rows);
  if (threadIdx.x == 0) __hip_atomic_store(a.counters + rb, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Second pass of the two-pass split-K reduction: y[r] = sum_s partials[s][r]
// (+ bias).  A workgroup covers 64 rows; its 4 wavefronts each sum a quarter
// of the splits with independent loads, then wave 0 adds the four quarters
// in a fixed order.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float *__restrict__ partials, int splits, int Npad,
                                                            int rows, const float *__restrict__ bias,
                                                            float *__restrict__ y, unsigned long long *amax,
                                                            const unsigned *__restrict__ pcount, float penalty) {
  __shared__ float q[4][kWave];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int r = blockIdx.x * kWave + lane;
  float s = 0.0f;
  if (r < Npad)
    for (int k = wave; k < splits; k += 4) s += partials[size_t(k) * Npad + r];
  q[wave][lane] = s;
  __syncthreads();
  if (wave == 0) {
    float t = (q[0][lane] + q[1][lane]) + (q[2][lane] + q[3][lane]);
    if (r < rows) {
      t = bias ? t + bias[r] : t;
      y[r] = t;
    }
    if (amax)
      wave_argmax(amax, blockIdx.x, pcount && r < rows ? penalised_logit(t, pcount[r], penalty) : t, r, r < rows);
  }
}

// ---------------------------------------------------------------------------
// Full-K variant: a workgroup owns RW = 64/H output rows and the whole
// padded K, so no partial sums leave the workgroup.  The WAVES*H k-slices of
// CPS chunks each are spread over the lanes: lane l of wave w serves row
// l % RW of the workgroup and k-slice w*H + l/RW.  The tables of the whole K
// sit in LDS (16 B per activation); each 256-chunk is rotated by one wave.
// Slice s keeps its tables at s*(CPS*2048 + 256) bytes; with H = 4, two
// quarter-wave slices share an LDS pass, so odd slices are shifted by 64 B
// into other banks (the shift rides in bits 6-7 of the nibble byte); with
// H = 8 four slices share a pass and the same shift halves their overlap.  At the
// end the NS = WAVES*H slice partials of each row are summed in slice order.
template <int WAVES, int H, int CPS>
constexpr uint32_t fullk_prefix_bytes() {
  return (uint32_t(WAVES * H * CPS + WAVES * kWave) * 4 + 255) / 256 * 256;
}

// The lean kernel's prefix: as fullk_prefix_bytes, or with a plane split
// only the WAVES x (rows per workgroup) slice sums it writes (the layered
// plan's 70 chunk blocks leave 2.5 KB of the 160 KB)
template <int WAVES, int H, int CPS, bool PS>
constexpr uint32_t plain_prefix_bytes() {
  if constexpr (PS) return (uint32_t(WAVES * H * CPS + WAVES * (kWave / H / 2)) * 4 + 255) / 256 * 256;
  return fullk_prefix_bytes<WAVES, H, CPS>();
}

template <int H>
__device__ __forceinline__ uint32_t slice_shift(int s) {
  return ((H == 4 || H == 8) && (s & 1)) ? 64u : 0u;
}

template <int FMT, int WAVES, int H, int CPS, bool STAGED>
__global__ __launch_bounds__(WAVES * kWave) void lut_gemv_fullk_kernel(GemvArgs a) {
  constexpr int P = Fmt<FMT>::P, NA = Fmt<FMT>::NA, S = Fmt<FMT>::S;
  constexpr int RW = kWave / H;
  constexpr int NS = WAVES * H;
  constexpr uint32_t SSTRIDE = CPS * 32 * 64 + 256;
  // Wave w owns the 128-chunks of its k-slices, [w*H*CPS, (w+1)*H*CPS), and
  // builds exactly their tables (XJ 256-chunks), so no other wave waits on it.
  constexpr int XJ = H * CPS >= 2 ? H * CPS / 2 : 1;
  constexpr uint32_t PREFIX = fullk_prefix_bytes<WAVES, H, CPS>();
  extern __shared__ __attribute__((aligned(256))) float lds[];
  const int Kc = a.Kp / kChunk;
  const int used = (Kc + CPS - 1) / CPS;                      // slices holding chunks
  float *xsum = lds;                                          // [NS*CPS]
  float *red = lds + NS * CPS;                                // [NS][RW]
  char *tables = reinterpret_cast<char *>(lds) + PREFIX;      // slice s at s*SSTRIDE

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int sub = lane / RW;
  const int s = wave * H + sub;
  const int rl = lane % RW;
  const int row = blockIdx.x * RW + rl;
  const int lr = min(row, a.Npad - 1);

  // ---- loads: activations for this wave's 256-chunks, then the weights ----
  const int C2n = a.Kp / kRotChunk;
  const int own0 = wave * H * CPS, own1 = own0 + H * CPS;   // owned 128-chunks [own0, own1)
  const int c2base = own0 / 2;
  float4 xr[XJ];
  float aux[XJ][4];
#pragma unroll
  for (int j = 0; j < XJ; ++j) {
    const int c2 = min(c2base + j, C2n - 1);
    xr[j] = load_x4_raw(a.x, c2 * kRotChunk, a.cols, lane);
    load_aux4(a, c2 * kRotChunk, lane, aux[j]);
  }
  __builtin_amdgcn_sched_barrier(0);
  // A CU returns vector loads roughly in issue order, so every wave's x
  // requests go out before any wave's weight requests (the barrier does not
  // wait for the loads): no wave's tables wait behind the weight stream.
  __builtin_amdgcn_s_barrier();
  // Weight loads.  STAGED (CPS > 1 only) issues chunk 0 before the table
  // prologue and the later chunks after it, so that HBM serves chunk 0 of
  // every wave first and chunk 1 streams in while chunk 0 is looked up.
  u32x4 w[CPS][P];
  float sc[CPS][S];
  const u32x4 *__restrict__ pl = reinterpret_cast<const u32x4 *>(a.planes);
  const size_t Npad = size_t(a.Npad);
  auto load_planes = [&](int c) {
    const int ch = min(s * CPS + c, Kc - 1);                   // clamped; masked below
#pragma unroll
    for (int p = 0; p < P; ++p) w[c][p] = __builtin_nontemporal_load(pl + (size_t(ch) * P + p) * Npad + lr);
  };
#pragma unroll
  for (int c = 0; c < CPS; ++c) {
    const int ch = min(s * CPS + c, Kc - 1);
    const int g = ch / a.group_chunks;
    if (!STAGED || c == 0) load_planes(c);
#pragma unroll
    for (int t = 0; t < S; ++t) sc[c][t] = a.scales[(size_t(t) * a.n_groups + g) * Npad + lr];
  }
  if constexpr (STAGED) __builtin_amdgcn_sched_barrier(0);

  // ---- prologue: (transform) -> (FWHT-256) -> this wave's group tables ---
  // Lanes 0-31 / 32-63 hold the first / second 128-chunk of a 256-chunk; a
  // lane's values count (norm, tables) only where the wave owns that chunk,
  // which partitions x exactly, so the norm needs no second read of x.
  float inv_rms = 1.0f;
  if (a.xmode == kXModeRmsNorm) {
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < XJ; ++j) {
      const int ch = (c2base + j) * 2 + (lane >> 5);
      float x0, x1, x2, x3;
      mask_x4(xr[j], (c2base + j) * kRotChunk, a.cols, lane, x0, x1, x2, x3);
      if (ch >= own0 && ch < own1 && c2base + j < C2n) ss += (x0 * x0 + x1 * x1) + (x2 * x2 + x3 * x3);
    }
    inv_rms = wg_inv_rms_from<WAVES * kWave>(ss, a.cols, a.eps, red);
  }
#pragma unroll
  for (int j = 0; j < XJ; ++j) {
    const int c2 = c2base + j;
    if (c2 >= C2n) break;   // wave-uniform
    float x0, x1, x2, x3;
    mask_x4(xr[j], c2 * kRotChunk, a.cols, lane, x0, x1, x2, x3);
    xform4(a.xmode, inv_rms, aux[j], x0, x1, x2, x3);
    if (a.rotate == LMX_ROTATE_FWHT256) fwht256_regs(x0, x1, x2, x3, lane);
    float t[16];
    group_table(x0, x1, x2, x3, t);
    const int ch = c2 * 2 + (lane >> 5);                      // 128-chunk of this group
    const bool mine = ch >= own0 && ch < own1;
    const int ts = ch / CPS;                                  // its k-slice
    float4 *dst = reinterpret_cast<float4 *>(tables + ts * SSTRIDE + slice_shift<H>(ts) + (ch % CPS) * 2048 +
                                             (lane & 31) * 64);
    if (mine) {
      dst[0] = make_float4(t[0], t[1], t[2], t[3]);
      dst[1] = make_float4(t[4], t[5], t[6], t[7]);
      dst[2] = make_float4(t[8], t[9], t[10], t[11]);
      dst[3] = make_float4(t[12], t[13], t[14], t[15]);
    }
    if constexpr (Fmt<FMT>::XS) {
      float xs = t[15];
      xs = lane_sum<16>(xs, lane);
      if ((lane & 31) == 0 && mine) xsum[ch] = xs;
    }
  }
  if constexpr (STAGED) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 1; c < CPS; ++c) load_planes(c);
  }
  // Each wave reads only the tables it wrote: a wave-scope fence (LDS
  // operations of a wave complete in order) instead of a workgroup barrier,
  // so every wave starts its lookups as soon as its own data is in.
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();

  // ---- lookups over this lane's k-slice -----------------------------------
  float acc = 0.0f;
  {
    // Lanes whose slice lies past K read slice used-1 (in bounds, possibly
    // another wave's, possibly mid-write) and discard the result.
    const uint32_t tbase = lds_addr(lds) + PREFIX + min(s, used - 1) * SSTRIDE;   // 256-byte aligned
    const uint32_t shift = slice_shift<H>(s) * 0x01010101u;   // bits 6-7 of each byte
#pragma unroll
    for (int c = 0; c < CPS; ++c) {
      float A[NA];
#pragma unroll
      for (int i = 0; i < NA; ++i) A[i] = 0.0f;
      chunk_lookups<FMT>(w[c], tbase + c * 2048, shift, A);
      const int ch = s * CPS + c;
      float xs = 0.0f;
      if constexpr (Fmt<FMT>::XS) xs = xsum[min(ch, Kc - 1)];
      const float nacc = finish_chunk<FMT>(A, xs, sc[c], acc);
      acc = ch < Kc ? nacc : acc;
    }
  }

  // ---- in-workgroup reduction over the k-slices, fixed order --------------
  red[s * RW + rl] = acc;
  __syncthreads();
  const int r = blockIdx.x * RW + threadIdx.x;
  float t = 0.0f;
  if (threadIdx.x < RW) {
#pragma unroll 8
    for (int k = 0; k < NS; ++k) t += red[k * RW + threadIdx.x];
    if (r < a.rows) {
      t = a.bias ? t + a.bias[r] : t;
      a.y[r] = t;
    }
  }
  if (a.amax && threadIdx.x < kWave)
    wave_argmax(a.amax, blockIdx.x, argmax_value(a, t, r, threadIdx.x < RW && r < a.rows), r,
                threadIdx.x < RW && r < a.rows);
}

// Full-K kernel with a lean front end: the same geometry, lookups and
// slice reduction as lut_gemv_fullk_kernel, staggered tables, weight and
// scale addresses in 32-bit offsets with a shift for the scale group, x
// rotated (ROT) without its final 1/16 (folded into the scales), every wave
// building the tables of its own 256-chunks only, and the activation
// transform XM (kXMode*) and the epilogue EPI (kEpi*) fixed at compile
// time.  Needs H*CPS even (each wave owns whole 256-chunks).  No argmax
// epilogue.
// LAY (layered): slice s owns chunks s, s + NS, s + 2 NS, ... (not CPS
// consecutive ones), and chunk ch keeps its tables at ch * kIplChunkBytes,
// back to back: the last layer may be ragged (K = 8960 = 70 chunks on 64
// slices: 6 slices do two chunks), and 70 chunks' tables fit the LDS.
template <int FMT, bool ROT, int WAVES, int H, int CPS, int XM, int EPI = kEpiStore, bool LAY = false, bool PS = false>
__global__ __launch_bounds__(WAVES * kWave) void lut_gemv_plain_kernel(GemvArgs a) {
  constexpr int P = Fmt<FMT>::P, NA = Fmt<FMT>::NA, S = Fmt<FMT>::S;
  // PS (4-bit): the four planes of a row's chunk split over two lanes, planes
  // 0-1 and 2-3 (half the lookups per lane, half the rows per workgroup)
  static_assert(!PS || (FMT == LMX_FMT_INT4 && EPI == kEpiStore), "plane split: 4-bit, plain store");
  constexpr int RW = kWave / H / (PS ? 2 : 1);
  constexpr bool PAIR = EPI == kEpiSiluPair;
  constexpr int HR = RW / 2;   // PAIR: gate rows (then as many up rows) per workgroup
  constexpr int NS = WAVES * H;
  constexpr uint32_t SSTRIDE = stag_slice_bytes(CPS);
  constexpr int XJ = H * CPS / 2;
  static_assert(!LAY || H % 2 == 0, "layered: whole 256-chunks per wave and layer");
  static_assert(H * CPS % 2 == 0, "whole 256-chunks per wave");
  constexpr uint32_t PREFIX = plain_prefix_bytes<WAVES, H, CPS, PS>();
  extern __shared__ __attribute__((aligned(256))) float lds[];
  const int Kc = a.Kp / kChunk;
  const int used = (Kc + CPS - 1) / CPS;
  float *xsum = lds;
  float *red = lds + NS * CPS;
  char *tables = reinterpret_cast<char *>(lds) + PREFIX;

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int s = wave * H + (PS ? (lane / RW) >> 1 : lane / RW);
  const int part = PS ? (lane / RW) & 1 : 0;   // PS: planes 2*part, 2*part + 1
  const int rl = lane % RW;
  // PAIR: the workgroup's rows are gate rows blockIdx.x*HR + [0, HR) and the
  // up rows rows/2 + blockIdx.x*HR + [0, HR) (the host checks rows/2 % HR == 0)
  const int row = PAIR ? (rl < HR ? 0 : a.rows / 2 - HR) + blockIdx.x * HR + rl : blockIdx.x * RW + rl;
  const int lr = min(row, a.Npad - 1);

  // ---- x of this wave's 256-chunks (clamped in bounds, masked below) ----
  const int C2n = a.Kp / kRotChunk;
  const int c2base = wave * XJ;
  // the wave's j-th 256-chunk (increasing in j)
  const auto c2_of = [&](int j) { return LAY ? (j / (H / 2)) * (NS / 2) + wave * (H / 2) + j % (H / 2) : c2base + j; };
  // the chunk that slice s looks up at its step c
  const auto chunk_of = [&](int c) { return LAY ? c * NS + s : s * CPS + c; };
  constexpr bool AUX = XM == kXModeRmsNorm || XM == kXModeSiluMul;
  float4 xr[XJ], xa[XJ];
#pragma unroll
  for (int j = 0; j < XJ; ++j) {
    const int k = min(min(c2_of(j), C2n - 1) * kRotChunk + 4 * lane, a.cols - 4);
    xr[j] = *reinterpret_cast<const float4 *>(a.x + k);
    // norm weight, or the up half of a gate|up vector
    if constexpr (AUX) xa[j] = *reinterpret_cast<const float4 *>((XM == kXModeRmsNorm ? a.xw : a.x + a.cols) + k);
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();   // every wave's x requests ahead of the weight stream

  // ---- weights (chunk 0 now, the rest after the prologue) and scales ----
  constexpr int PL = PS ? 2 : P;   // planes a lane loads
  u32x4 w[CPS][PL];
  float sc[CPS][S];
  const u32x4 *__restrict__ pl = reinterpret_cast<const u32x4 *>(a.planes);
  const uint32_t Npad = uint32_t(a.Npad);
  auto load_planes = [&](int c) {
    const uint32_t ch = uint32_t(min(chunk_of(c), Kc - 1));
#pragma unroll
    for (int p = 0; p < PL; ++p)
      w[c][p] = __builtin_nontemporal_load(pl + ((ch * P + uint32_t(PS ? 2 * part + p : p)) * Npad + uint32_t(lr)));
  };
  load_planes(0);
#pragma unroll
  for (int c = 0; c < CPS; ++c) {
    const int ch = min(chunk_of(c), Kc - 1);
    const int g = a.gshift >= 0 ? ch >> a.gshift : ch / a.group_chunks;
#pragma unroll
    for (int t = 0; t < S; ++t) sc[c][t] = a.scales[(uint32_t(t * a.n_groups + g)) * Npad + uint32_t(lr)];
  }
  // the epilogue thread's bias term (the decoder's residual rides there),
  // requested with the weights so that its round trip overlaps the lookups
  // (not for the SiLU pair, whose gate|up carries no residual: two live
  // registers there cost a workgroup per CU)
  float eb0 = 0.0f;
  if constexpr (!PAIR) {
    if (threadIdx.x < RW && a.bias) {
      const int r = blockIdx.x * RW + threadIdx.x;
      if (r < a.rows) eb0 = a.bias[r];
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  // RMSNorm: the waves' 256-chunks partition x, so the sum of squares over
  // them (zero past cols) is the norm's, summed in the same order in every
  // workgroup (norm.cpp:18-34).
  float inv_rms = 1.0f;
  if constexpr (XM == kXModeRmsNorm) {
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < XJ; ++j) {
      float x0, x1, x2, x3;
      mask_x4(xr[j], c2_of(j) * kRotChunk, a.cols, lane, x0, x1, x2, x3);
      if (c2_of(j) < C2n) ss += (x0 * x0 + x1 * x1) + (x2 * x2 + x3 * x3);
    }
    inv_rms = wg_inv_rms_from<WAVES * kWave>(ss, a.cols, a.eps, red);
  }

  // ---- prologue: (transform) -> (FWHT-256 x16) -> group tables of this wave's chunks ----
  const uint32_t goff = group_offset<true>(lane & 31);
#pragma unroll
  for (int j = 0; j < XJ; ++j) {
    const int c2 = c2_of(j);
    if (c2 >= C2n) break;   // wave-uniform
    float x0, x1, x2, x3;
    mask_x4(xr[j], c2 * kRotChunk, a.cols, lane, x0, x1, x2, x3);
    if constexpr (AUX) {
      const float aux[4] = {xa[j].x, xa[j].y, xa[j].z, xa[j].w};
      xform4(XM, inv_rms, aux, x0, x1, x2, x3);
    }
    if constexpr (ROT) fwht256_regs_x16(x0, x1, x2, x3, lane);
    float t[16];
    group_table(x0, x1, x2, x3, t);
    const int ch = c2 * 2 + (lane >> 5);
    const int ts = LAY ? ch % NS : ch / CPS;   // the slice that looks it up
    float4 *dst = reinterpret_cast<float4 *>(
        tables + (LAY ? ch * kIplChunkBytes : ts * SSTRIDE + (ch % CPS) * kStagChunkBytes) + slice_shift<H>(ts) + goff);
    dst[0] = make_float4(t[0], t[1], t[2], t[3]);
    dst[1] = make_float4(t[4], t[5], t[6], t[7]);
    dst[2] = make_float4(t[8], t[9], t[10], t[11]);
    dst[3] = make_float4(t[12], t[13], t[14], t[15]);
    if constexpr (Fmt<FMT>::XS) {
      float xs = t[15];
      xs = lane_sum<16>(xs, lane);
      if ((lane & 31) == 0) xsum[ch] = xs;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 1; c < CPS; ++c) load_planes(c);
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();

  // ---- lookups over this lane's k-slice ----------------------------------
  constexpr float kScale = ROT ? 0.0625f : 1.0f;   // the FWHT's 1/16, exact
  float acc = 0.0f;
  {
    const uint32_t tbase = lds_addr(lds) + PREFIX + (LAY ? 0u : min(s, used - 1) * SSTRIDE);
    const uint32_t shift = slice_shift<H>(s) * 0x01010101u;
#pragma unroll
    for (int c = 0; c < CPS; ++c) {
      const int ch = chunk_of(c);
      float scl[S];
#pragma unroll
      for (int t = 0; t < S; ++t) scl[t] = sc[c][t] * kScale;
      if constexpr (PS) {
        // two planes as a 2-plane format; the third plane of the 4-bit
        // identity enters inverted, and the part's terms of
        // ((A0 + 2 A1) + 4 A2) - 8 A3 weight its two sums
        u32x4 wl[2] = {w[c][0], w[c][1]};
        const uint32_t inv = part ? 0xFFFFFFFFu : 0u;
        wl[1].x ^= inv;
        wl[1].y ^= inv;
        wl[1].z ^= inv;
        wl[1].w ^= inv;
        float A2[2] = {0.0f, 0.0f};
        if constexpr (LAY)
          chunk_lookups<LMX_FMT_RRQ2, true>(wl, tbase + uint32_t(min(chunk_of(c), Kc - 1)) * kIplChunkBytes, shift, A2);
        else
          chunk_lookups<LMX_FMT_RRQ2, true>(wl, tbase, shift, A2, c * kStagChunkBytes);
        const float c0 = part ? 4.0f : 1.0f, c1 = part ? -8.0f : 2.0f;
        const float nacc = fmaf(scl[0], c0 * A2[0] + c1 * A2[1], acc);
        acc = ch < Kc ? nacc : acc;
      } else {
        float A[NA];
#pragma unroll
        for (int i = 0; i < NA; ++i) A[i] = 0.0f;
        if constexpr (LAY)
          chunk_lookups<FMT, true>(w[c], tbase + uint32_t(min(chunk_of(c), Kc - 1)) * kIplChunkBytes, shift, A);
        else
          chunk_lookups<FMT, true>(w[c], tbase, shift, A, c * kStagChunkBytes);
        float xs = 0.0f;
        if constexpr (Fmt<FMT>::XS) xs = xsum[min(ch, Kc - 1)];
        const float nacc = finish_chunk<FMT>(A, xs, scl, acc);
        acc = ch < Kc ? nacc : acc;
      }
    }
  }

  // ---- in-workgroup reduction: a wave's H slices of a row by a lane
  // butterfly, then the waves in order (fixed, so deterministic) -----------
  {
    const float wsum = strided_sum<RW>(acc, lane);
    if (lane < RW) red[wave * RW + rl] = wsum;
  }
  __syncthreads();
  if constexpr (PAIR) {
    if (threadIdx.x < HR) {
      const int j = blockIdx.x * HR + threadIdx.x;
      float g = 0.0f, u = 0.0f;
#pragma unroll 8
      for (int k = 0; k < WAVES; ++k) {
        g += red[k * RW + threadIdx.x];
        u += red[k * RW + HR + threadIdx.x];
      }
      if (a.bias) g += a.bias[j], u += a.bias[a.rows / 2 + j];
      a.y[j] = silu(g) * u;
    }
  } else if (threadIdx.x < RW) {
    const int r = blockIdx.x * RW + threadIdx.x;
    float t = 0.0f;
#pragma unroll 8
    for (int k = 0; k < WAVES; ++k) t += red[k * RW + threadIdx.x];
    if (r < a.rows) a.y[r] = a.bias ? t + eb0 : t;
  }
}

// Interleaved variant of the plain kernel (two k-slices per wave, H = 2):
// wave w owns the 256-chunks c2 = w*CPS + c, c < CPS, and at step c its
// lower / upper half-wave looks up 128-chunk 2*c2 / 2*c2 + 1, exactly the two
// halves of the 256-chunk it has just rotated.  So every step is "build the
// tables of one 256-chunk, then look them up", and the VALU-heavy table
// build of one wave overlaps the LDS-heavy lookups of the others.  Chunk ch
// keeps its (staggered) tables at ch * kIplChunkBytes, a 256-byte multiple.

template <int WAVES, int CPS>
constexpr uint32_t ipl_prefix_bytes() {
  return (uint32_t(2 * WAVES * CPS + 2 * WAVES * (kWave / 2)) * 4 + 255) / 256 * 256;
}

template <int FMT, bool ROT, int WAVES, int CPS>
__global__ __launch_bounds__(WAVES * kWave) void lut_gemv_ipl_kernel(GemvArgs a) {
  constexpr int P = Fmt<FMT>::P, NA = Fmt<FMT>::NA, S = Fmt<FMT>::S;
  constexpr int RW = kWave / 2;
  constexpr uint32_t PREFIX = ipl_prefix_bytes<WAVES, CPS>();
  extern __shared__ __attribute__((aligned(256))) float lds[];
  const int Kc = a.Kp / kChunk;
  float *xsum = lds;                 // [2*WAVES*CPS]
  float *red = lds + 2 * WAVES * CPS;   // [NS][RW]
  char *tables = reinterpret_cast<char *>(lds) + PREFIX;

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int h = lane >> 5;
  const int rl = lane & (RW - 1);
  const int row = blockIdx.x * RW + rl;
  const int lr = min(row, a.Npad - 1);

  const int C2n = a.Kp / kRotChunk;
  const int c2base = wave * CPS;
  // A wave still on its first step outranks the waves past it (priority 1,
  // dropped once its later steps' loads are out).  The SIMD otherwise serves
  // its oldest waves first, so the youngest wave of each SIMD looked up its
  // first step last and only then requested the rest: its late loads and a
  // tail of lookups alone on the SIMD ended the kernel (measured: int4 8192^2
  // -4.5 %, ternary -8.7 %, binary -5 %, same bits).
  // AGE: past the first step the younger waves outrank the older ones
  // (priority wave / 4, the first step at 3), so the wave whose weights
  // came last is not also served last; measured int4 -1.1 %, int8 -1.6 %,
  // RRQ-2 -1.9 %, RRQ-3 -2.5 %, but ternary +1.3 % and binary +2.2 %.
  constexpr bool AGE = FMT != LMX_FMT_TERNARY && FMT != LMX_FMT_BINARY;
  if constexpr (AGE)
    __builtin_amdgcn_s_setprio(3);
  else
    __builtin_amdgcn_s_setprio(1);
  const int wave_s = __builtin_amdgcn_readfirstlane(wave);
  float4 xr[CPS];
#pragma unroll
  for (int c = 0; c < CPS; ++c) xr[c] = load_x4_raw(a.x, min(c2base + c, C2n - 1) * kRotChunk, a.cols, lane);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();   // every wave's x requests ahead of the weight stream

  u32x4 w[CPS][P];
  float sc[CPS][S];
  const u32x4 *__restrict__ pl = reinterpret_cast<const u32x4 *>(a.planes);
  const uint32_t Npad = uint32_t(a.Npad);
  auto chunk_of = [&](int c) { return min(2 * (c2base + c) + h, Kc - 1); };   // clamped; masked below
  auto load_planes = [&](int c) {
    const uint32_t ch = uint32_t(chunk_of(c));
#pragma unroll
    for (int p = 0; p < P; ++p) w[c][p] = __builtin_nontemporal_load(pl + ((ch * P + p) * Npad + uint32_t(lr)));
  };
  load_planes(0);
#pragma unroll
  for (int c = 0; c < CPS; ++c) {
    const int ch = chunk_of(c);
    const int g = a.gshift >= 0 ? ch >> a.gshift : ch / a.group_chunks;
#pragma unroll
    for (int t = 0; t < S; ++t) sc[c][t] = a.scales[(uint32_t(t * a.n_groups + g)) * Npad + uint32_t(lr)];
  }
  __builtin_amdgcn_sched_barrier(0);

  constexpr float kScale = ROT ? 0.0625f : 1.0f;   // the FWHT's 1/16, exact
  const uint32_t goff = group_offset<true>(lane & 31);
  const uint32_t tb = lds_addr(lds) + PREFIX;
  float acc = 0.0f;
#pragma unroll
  for (int c = 0; c < CPS; ++c) {
    const int c2 = c2base + c;
    if (c2 >= C2n) break;   // wave-uniform: no chunk of this step holds data
    // ---- tables of 256-chunk c2 (128-chunks 2*c2 and 2*c2 + 1) ----
    {
      float x0 = xr[c].x, x1 = xr[c].y, x2 = xr[c].z, x3 = xr[c].w;
      if (c2 * kRotChunk + kRotChunk > a.cols)   // wave-uniform: only the chunk holding the end of x
        mask_x4(xr[c], c2 * kRotChunk, a.cols, lane, x0, x1, x2, x3);
      if constexpr (ROT) fwht256_regs_x16(x0, x1, x2, x3, lane);
      float t[16];
      group_table(x0, x1, x2, x3, t);
      float4 *dst = reinterpret_cast<float4 *>(tables + (2 * c2 + h) * kIplChunkBytes + goff);
      dst[0] = make_float4(t[0], t[1], t[2], t[3]);
      dst[1] = make_float4(t[4], t[5], t[6], t[7]);
      dst[2] = make_float4(t[8], t[9], t[10], t[11]);
      dst[3] = make_float4(t[12], t[13], t[14], t[15]);
      if constexpr (Fmt<FMT>::XS) {
        float xs = t[15];
        xs = lane_sum<16>(xs, lane);
        if ((lane & 31) == 0) xsum[2 * c2 + h] = xs;
      }
    }
    // A wave reads only the tables it wrote; its LDS operations complete in order.
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // ---- lookups of 128-chunk 2*c2 + h ----
    const int ch = 2 * c2 + h;
    float A[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) A[i] = 0.0f;
    chunk_lookups<FMT, true>(w[c], tb + uint32_t(ch) * kIplChunkBytes, 0u, A);
    if (c == 0) {
      // The later chunks' loads go out only now: a wave whose load issue
      // stalls on a full memory queue cannot run its lookups, so issuing them
      // before this chunk's lookups held those lookups back until the HBM
      // stream drained (measured: int4 8192^2 -0.5 us, ternary -0.35 us).
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int cc = 1; cc < CPS; ++cc) load_planes(cc);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (AGE) {
        // priority wave / 4, in one asm block: a branch on the wave index
        // here splits the unrolled step loop and the compiler spills
        asm volatile(
            "s_setprio 0\n"
            "s_cmp_ge_u32 %0, 4\n"
            "s_cbranch_scc0 1f\n"
            "s_setprio 1\n"
            "s_cmp_ge_u32 %0, 8\n"
            "s_cbranch_scc0 1f\n"
            "s_setprio 2\n"
            "s_cmp_ge_u32 %0, 12\n"
            "s_cbranch_scc0 1f\n"
            "s_setprio 3\n"
            "1:" ::"s"(wave_s)
            : "scc");
      } else {
        __builtin_amdgcn_s_setprio(0);
      }
    }
    float xs = 0.0f;
    if constexpr (Fmt<FMT>::XS) xs = xsum[min(ch, Kc - 1)];
    float scl[S];
#pragma unroll
    for (int t = 0; t < S; ++t) scl[t] = sc[c][t] * kScale;
    const float nacc = finish_chunk<FMT>(A, xs, scl, acc);
    acc = ch < Kc ? nacc : acc;
  }

  // ---- in-workgroup reduction: the two half-wave slices of a row by a
  // lane swap, then the waves in order (fixed, so deterministic) ----------
  {
    const float wsum = strided_sum<RW>(acc, lane);
    if (h == 0) red[wave * RW + rl] = wsum;
  }
  __syncthreads();
  if (threadIdx.x < RW) {
    const int r = blockIdx.x * RW + threadIdx.x;
    float t = 0.0f;
#pragma unroll 8
    for (int k = 0; k < WAVES; ++k) t += red[k * RW + threadIdx.x];
    if (r < a.rows) a.y[r] = a.bias ? t + a.bias[r] : t;
  }
}

template <int WAVES, int H, int CPS, bool LAY = false, bool PS = false>
constexpr size_t plain_lds_bytes(size_t Kc) {
  return plain_prefix_bytes<WAVES, H, CPS, PS>() +
         (LAY ? Kc * kIplChunkBytes : (Kc + CPS - 1) / CPS * stag_slice_bytes(CPS));
}

template <int FMT, bool ROT, int WAVES, int H, int CPS, int XM, int EPI = kEpiStore, bool LAY = false, bool PS = false>
static int launch_plain_kernel(const GemvArgs &a, hipStream_t st) {
  const size_t lds = plain_lds_bytes<WAVES, H, CPS, LAY, PS>(size_t(a.Kp / kChunk));
  if (lds > kMaxLdsBytes) return 1;   // staggered tables do not fit: the generic kernel serves it
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void *>(&lut_gemv_plain_kernel<FMT, ROT, WAVES, H, CPS, XM, EPI, LAY, PS>),
      hipFuncAttributeMaxDynamicSharedMemorySize, int(kMaxLdsBytes));
  if (attr != hipSuccess) return fail(LMX_ERR_LAUNCH_FAILED, "hipFuncSetAttribute: %s", hipGetErrorString(attr));
  constexpr int RW = kWave / H / (PS ? 2 : 1);
  const int blocks = EPI == kEpiSiluPair ? a.rows / RW : (a.Npad + RW - 1) / RW;
  lut_gemv_plain_kernel<FMT, ROT, WAVES, H, CPS, XM, EPI, LAY, PS><<<dim3(blocks), dim3(WAVES * kWave), lds, st>>>(a);
  return LMX_OK;
}

// Unrotated 4-bit launches of the 4 x 4 x 1 and 16 x 4 x 1 plans split each
// chunk's planes over two lanes (plane_split_level(): 1, the default; 2 the
// 4 x 4 x 1 plan only; 0 neither).  Splitting the 8 x 8 x 1 plan as well
// (4 rows per workgroup, each building the whole K's tables) measured 9 %
// slower in Llama decode, so the plan chooser takes 16 x 4 x 1 with 8 rows
// per workgroup there instead (choose_fullk).
template <int WAVES, int H, int CPS, bool LAY>
static bool plane_split_plan() {
  if constexpr (LAY || CPS != 1) return false;
  if constexpr (WAVES == 4 && H == 4) return plane_split_level() >= 1;
  if constexpr (WAVES == 16 && H == 4) return plane_split_level() == 1;
  return false;
}

template <int FMT, bool ROT, int WAVES, int CPS>
static int launch_ipl_kernel(const GemvArgs &a, hipStream_t st) {
  const size_t lds = ipl_prefix_bytes<WAVES, CPS>() + size_t(a.Kp / kRotChunk) * 2 * kIplChunkBytes;
  if (lds > kMaxLdsBytes) return 1;
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void *>(&lut_gemv_ipl_kernel<FMT, ROT, WAVES, CPS>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, int(kMaxLdsBytes));
  if (attr != hipSuccess) return fail(LMX_ERR_LAUNCH_FAILED, "hipFuncSetAttribute: %s", hipGetErrorString(attr));
  lut_gemv_ipl_kernel<FMT, ROT, WAVES, CPS><<<dim3((a.Npad + 31) / 32), dim3(WAVES * kWave), lds, st>>>(a);
  return LMX_OK;
}

template <int FMT, int WAVES, int H, int CPS, bool LAY = false>
static int launch_plain_cfg(const GemvArgs &a, hipStream_t st) {
  // Interleaved where it measured faster: two k-slices per wave and at least
  // two steps per wave (one step has nothing to interleave; 17920 x 1536
  // ran 40% slower that way).  RRQ-3 too since the first-step priority
  // (8192^2 -1.6 %; it had been 4 % slower).
  if (a.epi == kEpiSiluPair) {
    // gate|up of the decode step: RMSNorm in, SiLU(gate)*up out (4-bit, unrotated)
    if constexpr (FMT == LMX_FMT_INT4)
      if (a.rotate == LMX_ROTATE_NONE && a.xmode == kXModeRmsNorm && a.rows % (kWave / H) == 0)
        return launch_plain_kernel<FMT, false, WAVES, H, CPS, kXModeRmsNorm, kEpiSiluPair, LAY>(a, st);
    return 1;
  }
  if (a.xmode != kXModeNone) {
    // Fused transforms on the lean kernel: the decode step's linears (4-bit,
    // unrotated); other formats take the generic kernel.
    if constexpr (FMT == LMX_FMT_INT4) {
      if (a.rotate == LMX_ROTATE_NONE) {
        if constexpr (!LAY && CPS == 1)
          if (a.xmode == kXModeRmsNorm && plane_split_plan<WAVES, H, CPS, LAY>())
            return launch_plain_kernel<FMT, false, WAVES, H, CPS, kXModeRmsNorm, kEpiStore, LAY, true>(a, st);
        switch (a.xmode) {
        case kXModeRmsNorm: return launch_plain_kernel<FMT, false, WAVES, H, CPS, kXModeRmsNorm, kEpiStore, LAY>(a, st);
        case kXModeSiluMul: return launch_plain_kernel<FMT, false, WAVES, H, CPS, kXModeSiluMul, kEpiStore, LAY>(a, st);
        }
      }
    }
    return 1;
  }
  if constexpr (!LAY && H == 2 && CPS >= 2) {
    if (a.kfamily != kKernelLean) {
      const int r = a.rotate == LMX_ROTATE_FWHT256 ? launch_ipl_kernel<FMT, true, WAVES, CPS>(a, st)
                                                   : launch_ipl_kernel<FMT, false, WAVES, CPS>(a, st);
      if (r != 1) return r;
    }
  }
  if (a.rotate == LMX_ROTATE_FWHT256) return launch_plain_kernel<FMT, true, WAVES, H, CPS, kXModeNone, kEpiStore, LAY>(a, st);
  if constexpr (FMT == LMX_FMT_INT4 && !LAY && CPS == 1)
    if (plane_split_plan<WAVES, H, CPS, LAY>())
      return launch_plain_kernel<FMT, false, WAVES, H, CPS, kXModeNone, kEpiStore, LAY, true>(a, st);
  return launch_plain_kernel<FMT, false, WAVES, H, CPS, kXModeNone, kEpiStore, LAY>(a, st);
}

// The plain kernel serves full-K launches without a fused transform or an
// argmax epilogue; returns 1 when the configuration is not covered.
template <int FMT>
static int launch_plain(const GemvArgs &a, hipStream_t st) {
  switch (a.fullk) {
  case kFullK_16x2x2: return launch_plain_cfg<FMT, 16, 2, 2>(a, st);
  case kFullK_16x2x3: return launch_plain_cfg<FMT, 16, 2, 3>(a, st);
  case kFullK_8x2x1: return launch_plain_cfg<FMT, 8, 2, 1>(a, st);
  case kFullK_16x4x1: return launch_plain_cfg<FMT, 16, 4, 1>(a, st);
  case kFullK_4x4x1: return launch_plain_cfg<FMT, 4, 4, 1>(a, st);
  case kFullK_8x8x1: return launch_plain_cfg<FMT, 8, 8, 1>(a, st);
  case kFullK_8x8x2L:
    if constexpr (FMT == LMX_FMT_INT4) {
      // unrotated, plain store: 16 waves x 4 slices x 2 layered chunks with
      // the planes split over two lanes (the same 8 rows per workgroup and
      // chunk tables; four waves per SIMD, half the lookups per lane)
      if (a.rotate == LMX_ROTATE_NONE && a.epi == kEpiStore && plane_split_level() == 1) {
        switch (a.xmode) {
        case kXModeNone: return launch_plain_kernel<FMT, false, 16, 4, 2, kXModeNone, kEpiStore, true, true>(a, st);
        case kXModeRmsNorm: return launch_plain_kernel<FMT, false, 16, 4, 2, kXModeRmsNorm, kEpiStore, true, true>(a, st);
        case kXModeSiluMul: return launch_plain_kernel<FMT, false, 16, 4, 2, kXModeSiluMul, kEpiStore, true, true>(a, st);
        }
      }
      return launch_plain_cfg<FMT, 8, 8, 2, true>(a, st);
    }
    return 1;
  }
  return 1;
}

template <int FMT, int WAVES, int H, int CPS, bool STAGED>
static int launch_fullk_kernel(const GemvArgs &a, hipStream_t st) {
  const size_t lds = fullk_lds_bytes(WAVES, H, CPS, a.Kp / kChunk);
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void *>(&lut_gemv_fullk_kernel<FMT, WAVES, H, CPS, STAGED>),
      hipFuncAttributeMaxDynamicSharedMemorySize, int(kMaxLdsBytes));
  if (attr != hipSuccess) return fail(LMX_ERR_LAUNCH_FAILED, "hipFuncSetAttribute: %s", hipGetErrorString(attr));
  if (lds > kMaxLdsBytes) return fail(LMX_ERR_INVALID_ARGUMENT, "full-K tables need %zu B of LDS", lds);
  constexpr int RW = kWave / H;
  lut_gemv_fullk_kernel<FMT, WAVES, H, CPS, STAGED>
      <<<dim3((a.Npad + RW - 1) / RW), dim3(WAVES * kWave), lds, st>>>(a);
  return LMX_OK;
}

template <int FMT, int WAVES, int H, int CPS>
static int launch_fullk_cfg(const GemvArgs &a, hipStream_t st) {
  if constexpr (CPS > 1)
    if (a.staged) return launch_fullk_kernel<FMT, WAVES, H, CPS, true>(a, st);
  return launch_fullk_kernel<FMT, WAVES, H, CPS, false>(a, st);
}

template <int FMT, int WAVES>
static void launch_waves(const GemvArgs &a, hipStream_t st) {
  const int row_blocks = (a.Npad + WAVES * kWave - 1) / (WAVES * kWave);
  const int splits = a.Kp / a.kslice;
  dim3 grid(row_blocks * splits), block(WAVES * kWave);
  if (a.kslice == 512)
    lut_gemv_kernel<FMT, 4, WAVES><<<grid, block, 0, st>>>(a, row_blocks, splits);
  else
    lut_gemv_kernel<FMT, 2, WAVES><<<grid, block, 0, st>>>(a, row_blocks, splits);
}

template <int FMT>
static int launch_fullk(const GemvArgs &a, hipStream_t st) {
  switch (a.fullk) {
  case kFullK_16x2x2: return launch_fullk_cfg<FMT, 16, 2, 2>(a, st);
  case kFullK_16x2x3: return launch_fullk_cfg<FMT, 16, 2, 3>(a, st);
  case kFullK_8x2x1: return launch_fullk_cfg<FMT, 8, 2, 1>(a, st);
  case kFullK_16x1x1: return launch_fullk_cfg<FMT, 16, 1, 1>(a, st);
  case kFullK_16x4x1: return launch_fullk_cfg<FMT, 16, 4, 1>(a, st);
  case kFullK_4x4x1: return launch_fullk_cfg<FMT, 4, 4, 1>(a, st);
  case kFullK_8x8x1: return launch_fullk_cfg<FMT, 8, 8, 1>(a, st);
  case kFullK_8x8x2L:
    return fail(LMX_ERR_INVALID_ARGUMENT, "the layered 8 x 8 x 2 plan has no form for this format and transform");
  }
  return fail(LMX_ERR_INVALID_ARGUMENT, "unknown full-K configuration %d", a.fullk);
}

template <int FMT>
static int launch_fmt(const GemvArgs &a, hipStream_t st) {
  if (a.epi != kEpiStore && silu_pair_rows(FMT, a) == 0)
    return fail(LMX_ERR_INVALID_ARGUMENT, "the SiLU-pair epilogue is not served for this weight and transform");
  if (a.fullk) {
    int r = 1;
    if (!a.amax && a.kfamily != kKernelGeneric) r = launch_plain<FMT>(a, st);
    if (r == 1 && a.fullk == kFullK_8x8x2L) {
      // the layered plan has no generic form (argmax epilogue, a transform
      // with rotation): the split-K kernel, whose scratch every handle holds
      GemvArgs b = a;
      b.fullk = kFullK_None;
      return launch_fmt<FMT>(b, st);
    }
    if (r == 1) r = launch_fullk<FMT>(a, st);
    if (r) return r;
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(LMX_ERR_LAUNCH_FAILED, "lut_gemv_fullk launch: %s", hipGetErrorString(e));
    return LMX_OK;
  }
  if (a.kslice != 256 && a.kslice != 512)
    return fail(LMX_ERR_INVALID_ARGUMENT, "unsupported k-slice %d", a.kslice);
  switch (a.waves) {
  case 1: launch_waves<FMT, 1>(a, st); break;
  case 2: launch_waves<FMT, 2>(a, st); break;
  case 4: launch_waves<FMT, 4>(a, st); break;
  default: return fail(LMX_ERR_INVALID_ARGUMENT, "unsupported waves per workgroup %d", a.waves);
  }
  const int splits = a.Kp / a.kslice;
  if (splits > 1 && a.reduce == kReduceTwoPass)
    splitk_reduce_kernel<<<dim3((a.rows + kWave - 1) / kWave), dim3(256), 0, st>>>(a.partials, splits, a.Npad,
                                                                                  a.rows, a.bias, a.y, a.amax,
                                                                                  a.pcount, a.penalty);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(LMX_ERR_LAUNCH_FAILED, "lut_gemv launch: %s", hipGetErrorString(e));
  return LMX_OK;
}

int silu_pair_rows(int fmt, const GemvArgs &a) {
  if (fmt != LMX_FMT_INT4 || a.rotate != LMX_ROTATE_NONE || a.xmode != kXModeRmsNorm || a.amax ||
      a.kfamily == kKernelGeneric)
    return 0;
  const size_t Kc = size_t(a.Kp / kChunk);
  size_t lds = 0;
  switch (a.fullk) {
  case kFullK_16x2x2: lds = plain_lds_bytes<16, 2, 2>(Kc); break;
  case kFullK_16x2x3: lds = plain_lds_bytes<16, 2, 3>(Kc); break;
  case kFullK_8x2x1: lds = plain_lds_bytes<8, 2, 1>(Kc); break;
  case kFullK_16x4x1: lds = plain_lds_bytes<16, 4, 1>(Kc); break;
  case kFullK_4x4x1: lds = plain_lds_bytes<4, 4, 1>(Kc); break;
  case kFullK_8x8x1: lds = plain_lds_bytes<8, 8, 1>(Kc); break;
  case kFullK_8x8x2L: lds = plain_lds_bytes<8, 8, 2, true>(Kc); break;
  default: return 0;   // split-K, or a configuration only the generic kernel serves
  }
  const int rw = kWave / fullk_shape(a.fullk).h;
  return lds <= kMaxLdsBytes && a.rows % rw == 0 ? rw / 2 : 0;
}

size_t gemv_argmax_slots(const GemvArgs &a) {
  if (a.fullk) return size_t((a.Npad + kWave / fullk_shape(a.fullk).h - 1) / (kWave / fullk_shape(a.fullk).h));
  const int splits = a.Kp / a.kslice;
  if (splits == 1) return size_t((a.Npad + a.waves * kWave - 1) / (a.waves * kWave)) * size_t(a.waves);
  if (a.reduce == kReduceTwoPass) return size_t((a.rows + kWave - 1) / kWave);
  return size_t((a.Npad + a.waves * kWave - 1) / (a.waves * kWave)) * size_t(a.waves);
}

int launch_gemv(int fmt, const GemvArgs &a, void *stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (fmt) {
  case LMX_FMT_TERNARY: return launch_fmt<LMX_FMT_TERNARY>(a, st);
  case LMX_FMT_BINARY: return launch_fmt<LMX_FMT_BINARY>(a, st);
  case LMX_FMT_RRQ2: return launch_fmt<LMX_FMT_RRQ2>(a, st);
  case LMX_FMT_RRQ3: return launch_fmt<LMX_FMT_RRQ3>(a, st);
  case LMX_FMT_INT3: return launch_fmt<LMX_FMT_INT3>(a, st);
  case LMX_FMT_INT4: return launch_fmt<LMX_FMT_INT4>(a, st);
  case LMX_FMT_INT8: return launch_fmt<LMX_FMT_INT8>(a, st);
  }
  return fail(LMX_ERR_UNSUPPORTED_FORMAT, "unknown format %d", fmt);
}

// ---------------------------------------------------------------------------
// Copies x[n] into an aligned buffer zero-padded to n_pad (used when the
// caller's x is not 16-byte aligned or n % 4 != 0).
__global__ __launch_bounds__(256) void stage_x_kernel(const float *__restrict__ x, size_t n, float *__restrict__ out,
                                                      size_t n_pad) {
  const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
  if (i < n_pad) out[i] = i < n ? x[i] : 0.0f;
}

int launch_stage_x(const float *x, size_t n, float *out, size_t n_pad, void *stream) {
  stage_x_kernel<<<dim3((n_pad + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(x, n, out, n_pad);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(LMX_ERR_LAUNCH_FAILED, "stage_x launch: %s", hipGetErrorString(e));
  return LMX_OK;
}

// ---------------------------------------------------------------------------
// Standalone FWHT-256 (apply_hadamard_rotation): one wavefront per chunk.
__global__ __launch_bounds__(256) void fwht256_kernel(float *x, size_t n_chunks) {
  const size_t c = size_t(blockIdx.x) * 4 + threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  if (c >= n_chunks) return;
  float4 *p = reinterpret_cast<float4 *>(x + c * kRotChunk) + lane;
  float4 v = *p;
  fwht256_regs(v.x, v.y, v.z, v.w, lane);
  *p = v;
}

int launch_fwht256(float *x, size_t n, void *stream) {
  const size_t chunks = n / kRotChunk;
  if (chunks == 0) return LMX_OK;
  fwht256_kernel<<<dim3((chunks + 3) / 4), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(x, chunks);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(LMX_ERR_LAUNCH_FAILED, "fwht256 launch: %s", hipGetErrorString(e));
  return LMX_OK;
}

// Length-n orthonormal FWHT (n a power of two, 256 <= n <= 16384) in one
// workgroup through LDS: out = H_n x / sqrt(n).
__global__ __launch_bounds__(1024) void fwht_full_kernel(const float *x, float *out, int n, float scale) {
  __shared__ float buf[16384];
  for (int i = threadIdx.x; i < n; i += blockDim.x) buf[i] = x[i];
  __syncthreads();
  for (int h = 1; h < n; h <<= 1) {
    for (int t = threadIdx.x; t < n / 2; t += blockDim.x) {
      const int j = (t / h) * 2 * h + (t % h);
      const float u = buf[j], v = buf[j + h];
      buf[j] = u + v;
      buf[j + h] = u - v;
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < n; i += blockDim.x) out[i] = buf[i] * scale;
}

int launch_fwht_full(const float *x, float *out, size_t n, void *stream) {
  fwht_full_kernel<<<dim3(1), dim3(1024), 0, static_cast<hipStream_t>(stream)>>>(
      x, out, int(n), float(1.0 / __builtin_sqrt(double(n))));
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(LMX_ERR_LAUNCH_FAILED, "fwht_full launch: %s", hipGetErrorString(e));
  return LMX_OK;
}

// ---------------------------------------------------------------------------
// precompute_luts on the device with the GEMV's own table code.
__global__ __launch_bounds__(256) void luts_kernel(const float *x, size_t n, unsigned rotate, float *luts) {
  const size_t c = size_t(blockIdx.x) * 4 + threadIdx.x / kWave;  // 256-chunk
  const int lane = threadIdx.x & (kWave - 1);
  if (c * kRotChunk >= n) return;
  float x0, x1, x2, x3;
  const size_t k = c * kRotChunk + 4 * lane;
  if (rotate == LMX_ROTATE_FWHT256) {  // n % 256 == 0 and x aligned (checked by the host)
    load_x4(x, int(c * kRotChunk), int(n), lane, x0, x1, x2, x3);
    fwht256_regs(x0, x1, x2, x3, lane);
  } else {
    if (k + 3 >= n) return;  // whole groups only, as precompute_luts
    x0 = x[k]; x1 = x[k + 1]; x2 = x[k + 2]; x3 = x[k + 3];
  }
  float t[16];
  group_table(x0, x1, x2, x3, t);
  float *dst = luts + (k / 4) * 16;
#pragma unroll
  for (int m = 0; m < 16; ++m) dst[m] = t[m];
}

int launch_precompute_luts(const float *x, size_t n, unsigned flags, float *luts, void *stream) {
  const size_t chunks = (n + kRotChunk - 1) / kRotChunk;
  if (chunks == 0) return LMX_OK;
  luts_kernel<<<dim3((chunks + 3) / 4), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(x, n, flags, luts);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(LMX_ERR_LAUNCH_FAILED, "precompute_luts launch: %s", hipGetErrorString(e));
  return LMX_OK;
}

// ---------------------------------------------------------------------------
// extract_indices on the device, with the same lookup-word and nibble
// arithmetic the ternary GEMV uses (32-bit little-endian words of canonical
// plane bytes; group 2j in the high nibble of byte j).
__global__ __launch_bounds__(256) void indices_kernel(const uint8_t *s, const uint8_t *z, size_t n_groups,
                                                      uint8_t *pos, uint8_t *neg) {
  const size_t g = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (g >= n_groups) return;
  const uint32_t w[2] = {uint32_t(s[g / 2]), uint32_t(z[g / 2])};
  uint32_t v[2];
  lookup_words<LMX_FMT_TERNARY>(w, v);
  const uint32_t sh = (g & 1) ? 0u : 4u;
  pos[g] = uint8_t((v[0] >> sh) & 15u);
  neg[g] = uint8_t((v[1] >> sh) & 15u);
}

int launch_extract_indices(const uint8_t *s, const uint8_t *z, size_t n_groups, uint8_t *pos, uint8_t *neg,
                           void *stream) {
  if (n_groups == 0) return LMX_OK;
  indices_kernel<<<dim3((n_groups + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
      s, z, n_groups, pos, neg);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(LMX_ERR_LAUNCH_FAILED, "extract_indices launch: %s", hipGetErrorString(e));
  return LMX_OK;
}

}  // namespace lmx
