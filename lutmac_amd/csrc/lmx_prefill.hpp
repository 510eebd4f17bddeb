// lmx_prefill.hpp -- kernels that take many positions of a prompt at once
// (included by lmx_decode.hip only): embedding rows, RoPE with the KV-cache
// append, and causal attention over the cache in fp32 on the matrix cores.
// Row m = b * T + t of a pass is position p0 + t of sequence b.
#ifndef LMX_PREFILL_HPP
#define LMX_PREFILL_HPP

#include "lmx_device.hpp"
#include "lmx_lanes.hpp"

namespace lmx {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

// RoPE of the pass's q (in place) and k, k and v appended to the cache: the
// decode attention's rotation (pairs (d, d + HD/2), each product rounded).
// One thread per pair; blockIdx.y = row.  Latency-bound: 5 us for 383 rows of
// 3072 (4.7 MB read, 6.3 MB written).
template <int HD>
__global__ __launch_bounds__(256) void prefill_rope_kernel(float *__restrict__ qkv, const float2 *__restrict__ rope,
                                                           float *__restrict__ kc, float *__restrict__ vc, int n_heads,
                                                           int n_kv, int T, int p0, size_t kv_stride) {
#pragma clang fp contract(off)
  constexpr int HALF = HD / 2;
  const int i = int(blockIdx.x) * 256 + int(threadIdx.x);
  const int head = i / HALF, d = i % HALF;
  if (head >= n_heads + 2 * n_kv) return;
  const int b = int(blockIdx.y) / T, pos = p0 + int(blockIdx.y) % T;
  float *row = qkv + size_t(blockIdx.y) * size_t(n_heads + 2 * n_kv) * HD + size_t(head) * HD;
  const size_t at = size_t(b) * kv_stride + size_t(pos) * size_t(n_kv) * HD;
  const float x = row[d], y = row[d + HALF];
  if (head >= n_heads + n_kv) {
    float *v = vc + at + size_t(head - n_heads - n_kv) * HD;
    v[d] = x;
    v[d + HALF] = y;
    return;
  }
  const float2 r = rope[size_t(pos) * HALF + d];
  const float u = x * r.x - y * r.y, v = x * r.y + y * r.x;
  if (head < n_heads) {
    row[d] = u;
    row[d + HALF] = v;
  } else {
    float *k = kc + at + size_t(head - n_heads) * HD;
    k[d] = u;
    k[d + HALF] = v;
  }
}

// Causal attention of a pass over the cache (its own positions appended
// before).  A workgroup takes 16 query rows of one KV head -- row i is query
// head i % group of position i / group -- and its 4 waves the 16-key tiles w,
// w + 4, ... of the keys up to the rows' last position, each with a running
// softmax; the waves' (m, l, o) merge in LDS.  fp32 throughout
// (v_mfma_f32_16x16x4_f32):
//   S^T = K Q^T: A lane (key j, kd) holds K[j][kd*HD/4 + i], B lane (row r, kd)
//     Q[r][kd*HD/4 + i], step i (any order of the dimensions is the same sum);
//     C lane (r, g) item v = key 4 g + v of the tile;
//   O^T = V^T P^T: step v takes key 4 kk + v from lane group kk, which is where
//     S^T left it, so P needs no transpose; A lane (dim, kk) = V[4 kk + v][dim].
// Bound by the serial chain over the last rows' key tiles: 32 heads of 64, 383
// positions 18 us, where one position's step takes 5.6 us in attention.  The 4
// waves share the keys, not the rows, to shorten that chain.
template <int HD>
__global__ __launch_bounds__(256) void prefill_attention_kernel(const float *__restrict__ qkv,
                                                                const float *__restrict__ kc,
                                                                const float *__restrict__ vc, int n_heads, int n_kv,
                                                                int T, int p0, float scale, size_t kv_stride,
                                                                float *__restrict__ out) {
  constexpr int Q = HD / 4, DT = HD / 16, W = 4;
  __shared__ float ms[W][16], ls[W][16];
  __shared__ float os[W][DT * 4][kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
  const int r = lane & 15, g = lane >> 4;
  const int group = n_heads / n_kv, rows = T * group;
  const int kvh = int(blockIdx.y), b = int(blockIdx.z);
  const int i = min(int(blockIdx.x) * 16 + r, rows - 1);   // rows past the last repeat it and are not stored
  const int t = i / group, head = kvh * group + i % group;
  const int pos = p0 + t;
  const int last = p0 + min(int(blockIdx.x) * 16 + 15, rows - 1) / group;   // the tile's last position
  const size_t krow = size_t(n_kv) * HD;
  kc += size_t(b) * kv_stride + size_t(kvh) * HD;
  vc += size_t(b) * kv_stride + size_t(kvh) * HD;

  float q[Q];
  {
    const float *src = qkv + (size_t(b) * T + t) * size_t(n_heads + 2 * n_kv) * HD + size_t(head) * HD + g * Q;
#pragma unroll
    for (int c = 0; c < Q; c += 4) {
      const float4 f = *reinterpret_cast<const float4 *>(src + c);
      q[c] = f.x, q[c + 1] = f.y, q[c + 2] = f.z, q[c + 3] = f.w;
    }
  }
  v4f o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  float m = -INFINITY, l = 0.0f;
  for (int j0 = wave * 16; j0 <= last; j0 += W * 16) {
    // keys past the tile's last position are masked; their rows lie inside the
    // cache, which holds whole 64-position chunks
    float k[Q];
    const float *ks = kc + size_t(j0 + r) * krow + g * Q;
#pragma unroll
    for (int c = 0; c < Q; c += 4) {
      const float4 f = *reinterpret_cast<const float4 *>(ks + c);
      k[c] = f.x, k[c + 1] = f.y, k[c + 2] = f.z, k[c + 3] = f.w;
    }
    float vv[DT][4];
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int v = 0; v < 4; ++v) vv[d][v] = vc[size_t(j0 + 4 * g + v) * krow + d * 16 + r];
    v4f s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = s0;   // two chains
#pragma unroll
    for (int c = 0; c < Q; c += 2) {
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[c], q[c], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[c + 1], q[c + 1], s1, 0, 0, 0);
    }
    float s[4], mt = -INFINITY;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      s[v] = j0 + 4 * g + v <= pos ? (s0[v] + s1[v]) * scale : -INFINITY;
      mt = fmaxf(mt, s[v]);
    }
    mt = fmaxf(mt, lane_xor<16>(mt, lane));
    mt = fmaxf(mt, lane_xor<32>(mt, lane));
    const float mn = fmaxf(m, mt);
    // a tile wholly past a row's position leaves its maximum at -inf
    const float keep = mn == -INFINITY ? 1.0f : expf(m - mn);
    float p[4], ps = 0.0f;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      p[v] = mn == -INFINITY ? 0.0f : expf(s[v] - mn);
      ps += p[v];
    }
    l = l * keep + ps;
    m = mn;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
#pragma unroll
      for (int v = 0; v < 4; ++v) o[d][v] *= keep;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        // a key past the tile's last position may lie past the written cache
        const float val = j0 + 4 * g + v > last ? 0.0f : vv[d][v];
        o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(val, p[v], o[d], 0, 0, 0);
      }
    }
  }
  l += lane_xor<16>(l, lane);   // each lane group summed its own keys
  l += lane_xor<32>(l, lane);
  if (g == 0) {
    ms[wave][r] = m;
    ls[wave][r] = l;
  }
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int v = 0; v < 4; ++v) os[wave][d * 4 + v][lane] = o[d][v];
  __syncthreads();
  // merge: wave w writes dimension tiles w, w + 4, ...
  float M = ms[0][r];
#pragma unroll
  for (int w = 1; w < W; ++w) M = fmaxf(M, ms[w][r]);
  float f[W], L = 0.0f;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    f[w] = expf(ms[w][r] - M);   // 0 for a wave without keys of this row
    L += f[w] * ls[w][r];
  }
  const float inv = 1.0f / L;
  if (int(blockIdx.x) * 16 + r >= rows) return;
  float *dst = out + (size_t(b) * T + t) * size_t(n_heads) * HD + size_t(head) * HD;
  for (int d = wave; d < DT; d += W) {
    float x[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      x[v] = 0.0f;
#pragma unroll
      for (int w = 0; w < W; ++w) x[v] += f[w] * os[w][d * 4 + v][lane];
      x[v] *= inv;
    }
    *reinterpret_cast<float4 *>(dst + d * 16 + 4 * g) = make_float4(x[0], x[1], x[2], x[3]);
  }
}

}  // namespace
}  // namespace lmx

#endif  // LMX_PREFILL_HPP
