// lmx_internal.hpp -- shared definitions of the LUT-GEMV library (not part
// of the C ABI).
#pragma once

#include <cstddef>
#include <cstdint>
#include <string>

#include "lutmac_hip.h"

struct lmx_weight;

namespace lmx {

constexpr int kChunk = 128;        // k per chunk: one uint4 per plane per row
constexpr int kRotChunk = 256;     // FWHT-256 block and device K padding
constexpr int kWave = 64;          // lanes per wavefront (one row per lane)

inline size_t round_up(size_t v, size_t m) { return (v + m - 1) / m * m; }

struct FormatInfo {
  int planes;
  int stages;
  size_t block_bytes;  // reference AoS block size; 0 = no reference block
};

bool format_info(int fmt, FormatInfo *fi);

// Sets the thread-local error message and returns `status`.
int fail(int status, const char *fmt, ...);
void clear_error();

// ---- host repack (lmx_repack.cpp) ----------------------------------------
int blocks_to_planes(int fmt, const uint8_t *blocks, size_t rows, size_t cols,
                     uint8_t *planes, float *scales);
int planes_to_blocks(int fmt, const uint8_t *planes, const float *scales,
                     size_t rows, size_t cols, uint8_t *blocks);
// planes: [P][rows][row_bytes]; tiles: [Kp/128][P][Npad][16].  Columns past
// row_bytes*8 get the format's pad code (pad_byte), rows past `rows` zero.
uint8_t pad_byte(int fmt, int plane);
void tile_planes(int fmt, const uint8_t *planes, size_t rows, size_t row_bytes,
                 size_t Npad, size_t Kp, uint8_t *tiles);
void untile_planes(int fmt, const uint8_t *tiles, size_t rows, size_t row_bytes,
                   size_t Npad, size_t Kp, uint8_t *planes);

// ---- device launches (lmx_kernels.hip) -----------------------------------
struct GemvArgs {
  const void *planes;      // tiled planes
  const void *codes;       // digit kernels: 4- and 8-bit code copy (code_copy_bytes), or null
  const float *scales;     // [S][n_groups][Npad]
  const float *x;          // [cols]
  float *y;                // [rows]
  const float *bias;       // [rows] or null
  const float *resid;      // digit kernels: [batch][rows] added to y (may alias y), or null
  float *partials;         // [splits][Npad]
  unsigned *counters;      // [row_blocks]
  int rows, Npad, cols, Kp;
  int group_chunks;        // chunks per scale group
  int gshift;              // log2(group_chunks) when it is a power of two, else -1
  int n_groups;
  int kslice;              // k per workgroup (multiple of 256, divides Kp)
  unsigned rotate;         // LMX_ROTATE_NONE / LMX_ROTATE_FWHT256
  int reduce;              // split-K reduction strategy (kReduce*)
  int waves;               // wavefronts (64-row slabs) per workgroup: 1, 2 or 4
  int fullk;               // 0: split-K kernel; else a kFullK_* configuration
  int kfamily;             // full-K kernel family for plain activations (kKernel*)
  int staged;              // full-K: issue part of the weight loads after the table prologue
  int xmode;               // activation transform fused into the table prologue (kXMode*)
  const float *xw;         // kXModeRmsNorm: norm weight [cols]
  float eps;               // kXModeRmsNorm: epsilon
  unsigned long long *amax;  // when set: per-wave argmax keys of y (gemv_argmax_slots of them)
  const unsigned *pcount;  // with amax, or null: occurrences of each row's token in the history; the
                           // argmax keys then rank repetition-penalised values (penalised_logit)
  float penalty;           // repetition penalty applied pcount[row] times
  int epi;                 // output epilogue (kEpi*)
};

// Output epilogues of the full-K kernels:
//   kEpiStore:     y[r] = (W x')[r] (+ bias[r])
//   kEpiSiluPair:  rows = 2h (a fused gate|up weight): y[j] = silu(g_j) * u_j for
//                  j < h, g_j = row j, u_j = row h + j (each + bias); a
//                  workgroup computes gate rows and the matching up rows
//                  (model.cpp:36,413-416), so the activation of the down
//                  projection leaves the gate|up launch already formed
constexpr int kEpiStore = 0;
constexpr int kEpiSiluPair = 1;

// Activation transforms applied while the tables are built:
//   kXModeRmsNorm:  x'[k] = x[k] * inv_rms * xw[k], inv_rms = 1/sqrt(sum x^2 / cols + eps)
//                   (norm.cpp:18-34), the sum taken over x[0..cols) by every workgroup
//   kXModeSiluMul:  x'[k] = silu(x[k]) * x[cols + k]  (model.cpp:36,413-416: gate and
//                   up halves of one fused gate|up output)
// (both applied by xform4 after the load)
constexpr int kXModeNone = 0;
constexpr int kXModeRmsNorm = 1;
constexpr int kXModeSiluMul = 2;
constexpr int kAttnChunk = 64;

// Full-K kernel configurations (waves x k-slices per wave x chunks per slice):
// the workgroup holds the tables of the whole K and reduces in LDS.
enum {
  kFullK_None = 0,
  kFullK_16x2x2 = 1,  // 32 rows, 32 slices of 256: K <= 8192
  kFullK_16x2x3 = 2,  // 32 rows, 32 slices of 384: K <= 12288 (LDS-bound ~9472)
  kFullK_8x2x1 = 3,   // 32 rows, 16 slices of 128: K <= 2048
  kFullK_16x1x1 = 4,  // 64 rows, 16 slices of 128: K <= 2048
  kFullK_16x4x1 = 5,  // 16 rows, 64 slices of 128: K <= 8192
  kFullK_4x4x1 = 6,   // 16 rows, 16 slices of 128: K <= 2048
  kFullK_8x8x1 = 7,   // 8 rows, 64 slices of 128: K <= 8192
  kFullK_8x8x2L = 8   // 8 rows, 64 slices x 2 layered chunks (slice s: chunks s, s + 64): 4-bit,
                      // the lean kernel only, K <= 8960 (tables of 70 chunks back to back)
};

constexpr size_t kMaxLdsBytes = 160 * 1024;  // LDS per workgroup on gfx950

// LDS of a full-K launch: x sums + slice partials (rounded to 256 B), then
// one table region of cps*2048 + 256 B per slice that holds chunks.
// A staggered chunk block rounded up to 256 B (v_perm keeps only bytes 1-2
// of a table base), the stride of chunks whose tables sit back to back.
constexpr uint32_t kIplChunkBytes = 2304;

// LDS of a layered launch (kFullK_8x8x2L): the prefix, then Kc chunk blocks.
inline size_t layered_lds_bytes(int waves, int h, int cps, size_t Kc) {
  return (size_t(waves * h * cps + waves * kWave) * 4 + 255) / 256 * 256 + Kc * kIplChunkBytes;
}

inline size_t fullk_lds_bytes(int waves, int h, int cps, size_t Kc) {
  const size_t prefix = (size_t(waves * h * cps + waves * kWave) * 4 + 255) / 256 * 256;
  const size_t used = (Kc + cps - 1) / cps;
  return prefix + used * (size_t(cps) * 2048 + 256);
}

struct FullKShape { int waves, h, cps; };
inline FullKShape fullk_shape(int cfg) {
  switch (cfg) {
  case kFullK_16x2x2: return {16, 2, 2};
  case kFullK_16x2x3: return {16, 2, 3};
  case kFullK_8x2x1: return {8, 2, 1};
  case kFullK_16x1x1: return {16, 1, 1};
  case kFullK_16x4x1: return {16, 4, 1};
  case kFullK_4x4x1: return {4, 4, 1};
  case kFullK_8x8x1: return {8, 8, 1};
  case kFullK_8x8x2L: return {8, 8, 2};
  }
  return {0, 0, 0};
}

// Full-K kernel families for plain activations (no fused transform, no
// argmax): the interleaved table-build/lookup kernel where it applies and
// measured faster (two k-slices and at least two steps per wave, its tables
// fit, not RRQ-3), else the lean kernel, else the generic one (which also
// serves every fused transform).  LMX_KERNEL forces one for tests:
// 1 generic, 2 lean.
constexpr int kKernelAuto = 0;
constexpr int kKernelGeneric = 1;
constexpr int kKernelLean = 2;

// Split-K reduction strategies.
constexpr int kReduceTicket = 0;    // last workgroup of a row block sums (one release per group)
constexpr int kReduceFenceAll = 1;  // same, with a device fence in every thread
constexpr int kReduceTwoPass = 2;   // partials, then a separate reduce kernel

int launch_gemv(int fmt, const GemvArgs &a, void *stream);
// Plane split of unrotated 4-bit lean launches (LMX_PS, read per call): 1
// the 4 x 4 x 1 and 16 x 4 x 1 plans (default), 2 the 4 x 4 x 1 plan only,
// 0 neither.
int plane_split_level();
// Rows of one output half a workgroup covers with kEpiSiluPair for these
// arguments (format, plan, transform), 0 when that epilogue is not served.
int silu_pair_rows(int fmt, const GemvArgs &a);
// ---- digit kernels (lmx_digit.hip): exact products on the 8-bit matrix cores ----
// Vectors split into signed-byte digits by launch_digit_split.
struct DigitVectors {
  char *digits;       // [quads of 4 vectors][Kp/128][2 KiB]
  float *fac;         // [count] factor of a vector's sums (norm, rotation, code scale; NaN: not finite)
  int *exp;           // tile form: [count] the power of two of a vector's digits, or kFarVector
  float *mult;        // rows form and far vectors: [quads][Kp/128][4] that of each vector's chunk (0: the
                      // chunk holds the activations themselves)
  float *partials;    // rows form: sums of k-slices (kDigitPartials bytes)
  unsigned *tickets;  // rows form: [kDigitTickets], zero between launches
  int count;
  int tile;           // for the tile kernel (many vectors and rows), else the rows kernel
};
constexpr int kFarVector = 0x7FFFFFFF;    // a vector whose chunks' digits each have their own power of two (d.mult)
constexpr unsigned kDigitTickets = 256;   // row blocks of a sliced rows launch, at most
// Bytes of slice sums: up to 256 workgroups of 2 row tiles x 4 quads x 64 sums.
constexpr size_t kDigitPartials = 256 * 512 * sizeof(float);
constexpr size_t kDigitTicketBytes = kDigitTickets * sizeof(unsigned);
size_t digit_bytes(size_t Kp, size_t vectors);
size_t digit_capacity(size_t Kp, size_t bytes);   // vectors (a multiple of 4) that fit in bytes
DigitVectors digit_vectors(const lmx_weight *w, void *scratch, unsigned *tickets, size_t count);
// a.x [count][cols], transform a.xmode (a.xw, a.eps), a.rotate -> d
int launch_digit_split(int fmt, const GemvArgs &a, const DigitVectors &d, void *stream);
// y = W x of the split vectors (+ a.bias per row) (+ a.resid per vector row), or the SiLU pair (a.epi)
int launch_digit_gemm(int fmt, const GemvArgs &a, const DigitVectors &d, void *stream);
// 1..4 vectors in one launch, with transform a.xmode and epilogue a.epi
// (argmax keys, one slot per workgroup, for one vector)
int launch_digit_gemv(int fmt, const GemvArgs &a, int nv, void *stream);
size_t digit_argmax_slots(const GemvArgs &a);   // argmax key slots of that launch
int digit_gemv_tiles(const GemvArgs &a);   // 16-row tiles per workgroup of that launch
// 4- and 8-bit codes laid out for the matrix-core operands, made from the
// plane tiles on the device: [Kp/128][Npad][4 plane words][4 or 8 words];
// 0 bytes for the other formats, which the kernels read from the planes.
size_t code_copy_bytes(int fmt, size_t Npad, size_t Kp);
int launch_code_copy(int fmt, const void *planes, size_t Npad, size_t Kp, void *codes, void *stream);

// Number of argmax key slots a launch with these arguments writes.
size_t gemv_argmax_slots(const GemvArgs &a);
int launch_fwht256(float *x, size_t n, void *stream);
int launch_stage_x(const float *x, size_t n, float *out, size_t n_pad, void *stream);
int launch_fwht_full(const float *x, float *out, size_t n, void *stream);
int launch_precompute_luts(const float *x, size_t n, unsigned flags,
                           float *luts, void *stream);
int launch_extract_indices(const uint8_t *s, const uint8_t *z, size_t n_groups,
                           uint8_t *pos, uint8_t *neg, void *stream);

}  // namespace lmx

// Device weight handle (opaque to C callers).
struct lmx_weight {
  int format = 0;
  int device = 0;
  size_t rows = 0, cols = 0;
  size_t Npad = 0, Kp = 0;
  size_t group = 0;        // scale group in k on the device (multiple of 128)
  size_t n_groups = 0;     // Kp / group
  size_t tile_bytes = 0;
  size_t scale_bytes = 0;
  int kslice = 0;          // chosen k-slice per workgroup
  int reduce = 0;          // split-K reduction strategy
  int waves = 4;           // wavefronts per workgroup
  int fullk = 0;           // full-K kernel configuration (kFullK_*), 0 = split-K
  int kfamily = 0;         // full-K kernel family for plain activations (kKernel*)
  int staged = 1;          // full-K: later chunks' weight loads after the prologue
  void *d_weight = nullptr;      // allocation of the planes, codes and scales
  void *d_scratch = nullptr;     // allocation of the counters, staging and partials
  void *d_planes = nullptr;
  float *d_scales = nullptr;
  float *d_partials = nullptr;
  unsigned *d_counters = nullptr;
  float *d_xrot = nullptr;  // staging for LMX_ROTATE_FWHT_FULL (cols floats)
  bool digit = true;             // one vector of 4 or 8 bits on the digit kernels (LMX_DIGIT=0, or a
                                 // lookup-table plan asked for: not)
  void *d_codes = nullptr;       // digit kernels: 4- and 8-bit code copy
  void *d_digits = nullptr;      // scratch of the digit kernels: the memory of d_partials, or the caller's
  size_t digit_cap = 0;          // its bytes
};

namespace lmx {
// Fills a handle's shape, layout sizes and kernel plan for (fmt, rows, cols,
// group) as lmx_weight_create does; allocates nothing, sets no pointers.
void plan_weight(lmx_weight *w, int fmt, size_t rows, size_t cols, size_t group);
// lmx_gemv after its handle check: y = W x for `batch` vectors with the
// handle's pointers (planes, scales, partials, counters, staging).
int gemv_impl(const lmx_weight *w, const float *x, float *y, size_t batch, unsigned flags, void *stream);
// Kernel arguments of a handle (x, y, bias, rotation and transform unset).
GemvArgs weight_args(const lmx_weight *w);
// y = W x of `batch` vectors on the digit kernels (a.bias, a.resid, a.rotate, a.xmode none or RMSNorm,
// a.epi store or SiLU pair; x of any alignment); *done = the vectors covered, the rest (one by one on
// the lookup tables) left to the caller unless `all`; scratch: kDigitTicketBytes of tickets (zero) and
// room for the split digits, else the handle's
int digit_linear(const lmx_weight *w, GemvArgs a, const float *x, float *y, size_t batch, void *stream, size_t *done,
                 bool all, void *scratch = nullptr, size_t scratch_bytes = 0);
}  // namespace lmx
