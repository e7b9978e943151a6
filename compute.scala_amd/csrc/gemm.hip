// Matrix multiplication C = A . B (row-major FP32 in and out) on gfx950 MFMA.
//
// The reference has no GEMM kernel: matrixMultiply is a user idiom of split, broadcast,
// product and join that unrolls into one elementwise kernel (README.md:301-362,
// TensorsSpec.scala:468-528), so every output is a sequential FP32 dot product. Here:
//
//   CS_GEMM_FP32    FP32 operands: on the FP32 MFMA where the product is small, and from three BF16
//                   parts of each operand, exact together, where it is large (gemm_split_kernel)
//   CS_GEMM_BF16    operands rounded to BF16, v_mfma_f32_32x32x16_bf16, FP32 accumulate
//   CS_GEMM_BF16X3  split-BF16x3 (Henry, Tang & Heinecke 2019): A = Ah + Al, B = Bh + Bl
//                   with Ah = bf16(A), Al = bf16(A - Ah); C = Al.Bh + Ah.Bl + Ah.Bh, all
//                   three products on the BF16 MFMA into one FP32 accumulator
//   CS_GEMM_FP8     OCP e4m3 operands with one power-of-two scale per 128-wide K block of
//                   each row of A and each column of B (amax / 448 rounded up to 2^e),
//                   applied by v_mfma_scale_f32_32x32x64_f8f6f4, FP32 accumulate
//
// Small products run on gemm_direct_kernel, straight from A and B (choose_path, below). For the
// others a pre-pass converts A to a K-contiguous operand X[Mp][.] and B to its transpose Y[Np][.]
// (zero padded to the tile sizes; split, interleaved or quantised as the variant needs) in
// the stream's scratch; the main kernel computes C[m][n] = sum_k X[m][k] Y[n][k] with 256
// threads (4 wave64s in 2x2) per output tile: 256x256, each wave owning 128x128 as 4x4 MFMA
// tiles of 32x32 (256 FP32 accumulators per lane), or, where such tiles leave CUs idle, 128x128
// (2048^3 in BF16: 64 tiles 61 us, 256 tiles 37 us).
//
// All variants share one pipeline there. A K stage is 128 bytes of every operand row (32 FP32
// values, 64 BF16 values, 32 hi/lo pairs or 128 e4m3 values); two stages live in LDS (128 or 64 KiB),
// or four of a 128x128 tile. The next stages stream global -> LDS directly (buffer_load ... lds, no registers) while
// the MFMAs of the current one run; inside a stage the fragments of the next MFMA step are
// read from LDS while the current step's MFMAs issue. Each 128-byte LDS row R stores its
// 16-byte piece p at slot p ^ ((R >> 1) & 7), so the fragment reads of 16 consecutive rows
// (the lanes the LDS serves in one cycle) hit 16 different bank groups.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "internal.h"

namespace csmi {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
// Loads of four and two consecutive values at any 4-byte boundary.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

enum Kind { kF32 = 0, kBF16 = 1, kBF16X3 = 2, kFP8 = 3 };

constexpr int kThreads = 256;  // 4 waves, in 2x2
// W x W MFMA tiles of 32x32 per wave make an output tile of tile_edge(W) rows and columns.
constexpr int tile_edge(int W) { return 64 * W; }

// Blocks are dispatched round-robin over the 8 XCDs, each with its own L2. The tile of
// block b: the XCDs get contiguous ranges of tiles, walked in groups of 4 tile rows (column
// by column inside a group), so one XCD's blocks share 4 A panels and a run of B panels.
__device__ __forceinline__ void tile_coords(int b, int tiles_m, int tiles_n, int &tm, int &tn) {
  const int total = tiles_m * tiles_n;
  int t = b;
  if (total % 8 == 0) t = (b % 8) * (total / 8) + b / 8;
  constexpr int G = 4;
  const int per_group = G * tiles_n;
  const int g = t / per_group, local = t % per_group;
  const int rows = min(G, tiles_m - g * G);
  tm = g * G + local % rows;
  tn = local / rows;
}

// ---------------------------------------------------------------------------- pre-pass
// Reads are 16 bytes at any 4-byte boundary, whatever the leading dimension: 4095^3 in BF16 took 169 us
// where rows off the 16-byte grid were read value by value, and takes 153 (4096^3: 148).

// FP32 operands for the FP32 kernel, zero padded to [rows_p][kp]. A (K contiguous): one
// thread per 4 consecutive K values of a row, 16-byte loads and stores.
__device__ __forceinline__ void pack_rows_f32(unsigned bx, const float *__restrict__ src, int rows, int cols, int ld,
                                              int rows_p, int kp, float *__restrict__ out) {
  const int chunks = kp / 4;
  const int64_t idx = int64_t(bx) * 256 + threadIdx.x;
  if (idx >= int64_t(rows_p) * chunks) return;
  const int r = static_cast<int>(idx / chunks), k = static_cast<int>(idx % chunks) * 4;
  const float *p = src + int64_t(r) * ld + k;
  float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (r < rows && k + 4 <= cols) {
    const f4u a = *reinterpret_cast<const f4u *>(p);
    v = make_float4(a[0], a[1], a[2], a[3]);
  } else if (r < rows) {
    v.x = k < cols ? p[0] : 0.0f;
    v.y = k + 1 < cols ? p[1] : 0.0f;
    v.z = k + 2 < cols ? p[2] : 0.0f;
    v.w = k + 3 < cols ? p[3] : 0.0f;
  }
  *reinterpret_cast<float4 *>(out + int64_t(r) * kp + k) = v;
}

// A TK x TN tile of B (K x N, N contiguous): rows k0.., columns n0.., zero outside the source.
// TN / 4 threads per row, one 16-byte load each, so a row's 4 TN bytes are read
// contiguously. Column n of row k sits at (n + k) mod TN: the reads of one column down K
// (lane l at row 4l + j or 8l + e) then spread over the 64 banks without padding.
constexpr int kPackTN = 64;  // B-tile width of the FP32 and BF16 packs
template <int TN>
__device__ __forceinline__ int tile_col(int k, int n) { return (n + k) & (TN - 1); }

// Four consecutive columns of row k of B from column n on.
__device__ __forceinline__ f4u load_b4(const float *__restrict__ src, int n_src, int k_src, int ld, int n, int k) {
  f4u a = {0.0f, 0.0f, 0.0f, 0.0f};
  if (k < k_src && n < n_src) {
    const float *p = src + int64_t(k) * ld + n;
    if (n + 4 <= n_src) {
      a = *reinterpret_cast<const f4u *>(p);
    } else {
      a[0] = p[0];
      if (n + 1 < n_src) a[1] = p[1];
      if (n + 2 < n_src) a[2] = p[2];
    }
  }
  return a;
}

template <int TK, int TN, int kThreadsT>
__device__ __forceinline__ void load_b_tile(float (*tile)[TN], const float *__restrict__ src, int n_src, int k_src,
                                            int ld, int n0, int k0) {
  constexpr int kRowsPerPass = kThreadsT / (TN / 4), kPasses = TK / kRowsPerPass;
  const int t = threadIdx.x, n = (t % (TN / 4)) * 4;
  // all loads in flight before the first LDS write
  f4u a[kPasses];
  if (n0 + TN <= n_src && k0 + TK <= k_src) {
#pragma unroll
    for (int i = 0; i < kPasses; ++i)
      a[i] = *reinterpret_cast<const f4u *>(src + int64_t(k0 + t / (TN / 4) + kRowsPerPass * i) * ld + (n0 + n));
  } else {
#pragma unroll
    for (int i = 0; i < kPasses; ++i)
      a[i] = load_b4(src, n_src, k_src, ld, n0 + n, k0 + t / (TN / 4) + kRowsPerPass * i);
  }
#pragma unroll
  for (int i = 0; i < kPasses; ++i) {
    const int k = t / (TN / 4) + kRowsPerPass * i;
#pragma unroll
    for (int e = 0; e < 4; ++e) tile[k][tile_col<TN>(k, n + e)] = a[i][e];
  }
}

// B (K x N, N contiguous) -> Y[rows_p][kp], row n = column n of B: 64 K x TN N tiles through
// LDS, 16-byte stores along K (each row of Y gets 256 contiguous bytes per tile).
template <int TN>
__device__ __forceinline__ void pack_cols_f32(unsigned bx, unsigned by, const float *__restrict__ src, int n_src,
                                              int k_src, int ld, int rows_p, int kp,
                                              float *__restrict__ out) {
  __shared__ float tile[64][TN];  // [k][rotated n]
  const int n0 = int(bx) * TN, k0 = int(by) * 64, t = threadIdx.x;
  load_b_tile<64, TN, 256>(tile, src, n_src, k_src, ld, n0, k0);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TN / 16; ++i) {
    const int n = t / 16 + 16 * i, c = t % 16, k = k0 + 4 * c;
    if (n0 + n >= rows_p || k >= kp) continue;
    const float4 v =
        make_float4(tile[4 * c][tile_col<TN>(4 * c, n)], tile[4 * c + 1][tile_col<TN>(4 * c + 1, n)],
                    tile[4 * c + 2][tile_col<TN>(4 * c + 2, n)], tile[4 * c + 3][tile_col<TN>(4 * c + 3, n)]);
    *reinterpret_cast<float4 *>(out + int64_t(n0 + n) * kp + k) = v;
  }
}

// Operand rows for the LDS pipeline. BF16: Kp values per row. Split (BF16X3): per 32-wide K
// block, 32 BF16 high parts then 32 BF16 low parts (128 bytes), so that one K stage of a row
// is 128 contiguous bytes in every variant.
// Two floats rounded to BF16 (nearest even) by v_cvt_pk_bf16_f32: a in the low half.
__device__ __forceinline__ uint32_t bf16x2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2_t));
}

__device__ __forceinline__ void store_bf16x8(const float (&v)[8], char *row, int k, bool split) {
  i32x4 hi, lo;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t h = bf16x2(v[2 * e], v[2 * e + 1]);
    hi[e] = int(h);
    // the low parts: each value minus its high part (exact), rounded once more
    lo[e] = int(bf16x2(v[2 * e] - __uint_as_float(h << 16), v[2 * e + 1] - __uint_as_float(h & 0xffff0000u)));
  }
  if (split) {
    char *p = row + (k / 32) * 128 + (k % 32) * 2;
    *reinterpret_cast<i32x4 *>(p) = hi;
    *reinterpret_cast<i32x4 *>(p + 64) = lo;
  } else {
    *reinterpret_cast<i32x4 *>(row + int64_t(k) * 2) = hi;
  }
}

// A (rows x cols, K contiguous) -> X: one thread per 8 consecutive K values of a row, two
// 16-byte loads and one (split: two) 16-byte stores. Rows and K values beyond the source are zero.
template <bool kSplit>
__device__ __forceinline__ void pack_rows_bf16(unsigned bx, const float *__restrict__ src, int rows, int cols, int ld,
                                               int rows_p, int kp, char *__restrict__ out) {
  const int chunks = kp / 8;
  const int64_t idx = int64_t(bx) * 256 + threadIdx.x;
  if (idx >= int64_t(rows_p) * chunks) return;
  const int r = static_cast<int>(idx / chunks), k = static_cast<int>(idx % chunks) * 8;
  float v[8];
  const float *p = src + int64_t(r) * ld + k;
  if (r < rows && k + 8 <= cols) {
    const f4u a = *reinterpret_cast<const f4u *>(p), b = *reinterpret_cast<const f4u *>(p + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = a[e], v[4 + e] = b[e];
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (r < rows && k + e < cols) ? p[e] : 0.0f;
  }
  store_bf16x8(v, out + int64_t(r) * (int64_t(kp) * (kSplit ? 4 : 2)), k, kSplit);
}

// B (K x N, N contiguous) -> Y (row n holds column n of B along K): 64 K x TN N tiles
// through LDS; stores are 16 bytes along K (split: 16 high and 16 low bytes).
template <bool kSplit, int TN>
__device__ __forceinline__ void pack_cols_bf16(unsigned bx, unsigned by, const float *__restrict__ src, int n_src,
                                               int k_src, int ld, int rows_p, int kp,
                                               char *__restrict__ out) {
  __shared__ float tile[64][TN];  // [k][rotated n]
  const int n0 = int(bx) * TN, k0 = int(by) * 64, t = threadIdx.x;
  load_b_tile<64, TN, 256>(tile, src, n_src, k_src, ld, n0, k0);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TN / 32; ++i) {
    const int n = t / 8 + 32 * i, c = t % 8, k = k0 + 8 * c;
    if (n0 + n >= rows_p || k >= kp) continue;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = tile[8 * c + e][tile_col<TN>(8 * c + e, n)];
    store_bf16x8(v, out + int64_t(n0 + n) * (int64_t(kp) * (kSplit ? 4 : 2)), k, kSplit);
  }
}

// FP8 quantisation of 128 values: the scale is 2^e with e the smallest integer such that
// 448 * 2^e >= amax (|x| / 2^e <= 448, the e4m3 maximum); amax = 0 gives e = 0. Returns the
// E8M0 scale byte e + 127.
__device__ __forceinline__ int fp8_scale_exponent(float amax) {
  int e = 0;
  if (amax > 0.0f) {
    int ex;
    frexpf(amax / 448.0f, &ex);  // amax/448 = f * 2^ex, f in [0.5, 1)
    e = ex;
    if (ldexpf(1.0f, e - 1) >= amax / 448.0f) e -= 1;
  }
  return e < -127 ? -127 : (e > 127 ? 127 : e);
}

// Four e4m3 bytes of x[0..3] * inv, packed into one word (byte i = value i).
__device__ __forceinline__ uint32_t fp8x4(float x0, float x1, float x2, float x3, float inv) {
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(x0 * inv, x1 * inv, 0, false);
  w = __builtin_amdgcn_cvt_pk_fp8_f32(x2 * inv, x3 * inv, w, true);
  return static_cast<uint32_t>(w);
}

// A (rows x cols, K contiguous) -> X[rows_p][kp] e4m3 plus scales[kb * rows_p + r]: 16 lanes
// per 128-wide block of a row, 8 consecutive values per lane (two 16-byte loads), one 8-byte
// store per lane.
__device__ __forceinline__ void quantize_rows_fp8(unsigned bx, const float *__restrict__ src, int rows, int cols,
                                                  int ld, int rows_p, int kp, uint8_t *__restrict__ q,
                                                  uint8_t *__restrict__ scales) {
  const int64_t group = (int64_t(bx) * 256 + threadIdx.x) / 16;
  const int l16 = threadIdx.x % 16;
  const int blocks = kp / 128;
  if (group >= int64_t(rows_p) * blocks) return;  // whole groups of 16 lanes leave together
  const int r = static_cast<int>(group / blocks), kb = static_cast<int>(group % blocks);
  const int k = kb * 128 + 8 * l16;
  const float *p = src + int64_t(r) * ld + k;
  float v[8];
  if (r < rows && k + 8 <= cols) {
    const f4u a = *reinterpret_cast<const f4u *>(p), b = *reinterpret_cast<const f4u *>(p + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = a[e], v[4 + e] = b[e];
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (r < rows && k + e < cols) ? p[e] : 0.0f;
  }
  float m = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(v[e]));
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 16));
  const int e = fp8_scale_exponent(m);
  const float inv = ldexpf(1.0f, -e);
  const uint2 w = make_uint2(fp8x4(v[0], v[1], v[2], v[3], inv), fp8x4(v[4], v[5], v[6], v[7], inv));
  *reinterpret_cast<uint2 *>(q + int64_t(r) * kp + k) = w;
  if (l16 == 0) scales[int64_t(kb) * rows_p + r] = static_cast<uint8_t>(e + 127);
}

// B (K x N, N contiguous) -> Y[rows_p][kp] e4m3 (row n = column n of B) plus
// scales[kb * rows_p + n]: a block stages 128 K x 64 N in LDS (16-byte loads along N, all
// in flight together), then 4 lanes quantise one
// column's 128-wide block, 32 consecutive K values per lane and two 16-byte stores each (the
// column's 128 bytes are contiguous in Y).
__device__ __forceinline__ void quantize_cols_fp8(unsigned bx, unsigned by, const float *__restrict__ src, int n_src,
                                                  int k_src, int ld, int rows_p, int kp,
                                                  uint8_t *__restrict__ q_out, uint8_t *__restrict__ scales) {
  __shared__ float tile[128][65];  // [k][n]; row stride 65 words: read j of lane (n, q) hits bank 32q + j + n
  const int n0 = int(bx) * 64, kb = int(by), k0 = kb * 128, t = threadIdx.x;
  const int c4 = (t % 16) * 4;  // first of the four columns this thread loads
  f4u a[8];
  if (n0 + 64 <= n_src && k0 + 128 <= k_src) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      a[i] = *reinterpret_cast<const f4u *>(src + int64_t(k0 + t / 16 + 16 * i) * ld + (n0 + c4));
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = load_b4(src, n_src, k_src, ld, n0 + c4, k0 + t / 16 + 16 * i);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) tile[t / 16 + 16 * i][c4 + e] = a[i][e];
  __syncthreads();
  // 4 lanes per column, 32 consecutive K values each: lane q of column n quantises K rows
  // 32q..32q+31 of the tile and stores them as 32 contiguous bytes of Y's row n.
  const int n = t / 4, q = t % 4;
  if (n0 + n < rows_p) {  // the 4 lanes of a column agree
    float x[32];
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      x[j] = tile[32 * q + j][n];
      m = fmaxf(m, fabsf(x[j]));
    }
    m = fmaxf(m, __shfl_xor(m, 1, 4));
    m = fmaxf(m, __shfl_xor(m, 2, 4));
    const int e = fp8_scale_exponent(m);
    const float inv = ldexpf(1.0f, -e);
    uint32_t w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = fp8x4(x[4 * j], x[4 * j + 1], x[4 * j + 2], x[4 * j + 3], inv);
    uint4 *dst = reinterpret_cast<uint4 *>(q_out + int64_t(n0 + n) * kp + k0 + 32 * q);
    dst[0] = make_uint4(w[0], w[1], w[2], w[3]);
    dst[1] = make_uint4(w[4], w[5], w[6], w[7]);
    if (q == 0) scales[int64_t(kb) * rows_p + n0 + n] = static_cast<uint8_t>(e + 127);
  }
}

// Both operands in one launch: workgroups [0, row_blocks) pack A's rows, the rest B's 64-column
// tiles (N fastest), so the tail of one operand's pass overlaps the start of the other's and
// the call pays one dispatch instead of two.
struct PackArgs {
  const float *a;
  int m, k, lda, mp, kp;
  void *x;
  unsigned row_blocks;
  const float *b;
  int n, ldb, np;
  void *y;
  unsigned cols_gx;
  uint8_t *sx, *sy;  // FP8: the scales of A's rows and B's columns
};

template <int KIND>
__global__ __launch_bounds__(256) void pack_operands_kernel(PackArgs p) {
  const unsigned b = blockIdx.x;
  if (b < p.row_blocks) {
    if constexpr (KIND == kFP8)
      quantize_rows_fp8(b, p.a, p.m, p.k, p.lda, p.mp, p.kp, static_cast<uint8_t *>(p.x), p.sx);
    else if constexpr (KIND == kF32)
      pack_rows_f32(b, p.a, p.m, p.k, p.lda, p.mp, p.kp, static_cast<float *>(p.x));
    else
      pack_rows_bf16<KIND == kBF16X3>(b, p.a, p.m, p.k, p.lda, p.mp, p.kp, static_cast<char *>(p.x));
    return;
  }
  const unsigned c = b - p.row_blocks;
  if constexpr (KIND == kFP8)
    quantize_cols_fp8(c % p.cols_gx, c / p.cols_gx, p.b, p.n, p.k, p.ldb, p.np, p.kp,
                      static_cast<uint8_t *>(p.y), p.sy);
  else if constexpr (KIND == kF32)
    pack_cols_f32<kPackTN>(c % p.cols_gx, c / p.cols_gx, p.b, p.n, p.k, p.ldb, p.np, p.kp,
                           static_cast<float *>(p.y));
  else
    pack_cols_bf16<KIND == kBF16X3, kPackTN>(c % p.cols_gx, c / p.cols_gx, p.b, p.n, p.k, p.ldb, p.np, p.kp,
                                              static_cast<char *>(p.y));
}

// ------------------------------------------------------------------------ main kernel
constexpr int kRowB = 128;                          // bytes of one operand row per K stage
// One operand's rows of a stage (W = 4: 32 KiB, W = 2: 16 KiB), and the stages held of both.
constexpr int panel_bytes(int W) { return tile_edge(W) * kRowB; }
constexpr size_t lds_bytes(int W, int bufs) { return size_t(2) * bufs * panel_bytes(W); }

template <int KIND>
struct Pipe;
template <>
struct Pipe<kF32> {
  // 4 fragment steps of 8 K values; each fragment (4 FP32 values per lane) feeds 4 MFMAs of K 2
  static constexpr int kBytesPerK = 4, kK = 32, kSteps = 4;
  typedef i32x4 Frag;
};
template <>
struct Pipe<kBF16> {
  static constexpr int kBytesPerK = 2, kK = 64, kSteps = 4;  // 4 MFMA K steps of 16
  typedef bf16x8 Frag;
};
template <>
struct Pipe<kBF16X3> {
  static constexpr int kBytesPerK = 4, kK = 32, kSteps = 2;  // hi and lo per K value
  typedef bf16x8 Frag;
};
template <>
struct Pipe<kFP8> {
  static constexpr int kBytesPerK = 1, kK = 128, kSteps = 2;  // 2 MFMA K steps of 64
  typedef i32x8 Frag;
};

#define CSMI_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

template <int KIND>
__device__ __forceinline__ void mma(const typename Pipe<KIND>::Frag &a, const typename Pipe<KIND>::Frag &b,
                                    f32x16 &c, int sa, int sb) {
  if constexpr (KIND == kFP8) {
    // cbsz = blgp = 0: both operands OCP e4m3; one E8M0 scale per lane (byte 0)
    c = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, sa, 0, sb);
  } else {
    (void)sa;
    (void)sb;
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
}

// Waits until at most kLeft of this wave's memory instructions are in flight and its LDS accesses are
// done, then for the other waves. (__syncthreads would wait for every DMA.)
template <int kLeft>
__device__ __forceinline__ void publish_stage() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kLeft) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Runs stage(ks, fill, more) for ks = 0 .. stages - 1. Compile-time constants: fill, stage ks + kAhead
// exists, to be fetched meanwhile; more, stage ks + 1 exists.
template <int kAhead, class Stage>
__device__ __forceinline__ void run_stages(int stages, Stage &stage) {
  int ks = 0;
  for (; ks + kAhead < stages; ++ks) stage(ks, std::true_type(), std::true_type());
  if constexpr (kAhead > 1)
    for (; ks + 1 < stages; ++ks) stage(ks, std::false_type(), std::true_type());
  stage(ks, std::false_type(), std::false_type());
}

// The first of slice i's stages, of n stages cut into `slices` runs.
__device__ __forceinline__ int slice_begin(int n, unsigned i, int slices) {
  return slices == 1 ? int(i) * n : int(int64_t(n) * i / slices);
}

// Slice blockIdx.y of K; several slices write partial results C[slice][M][ldc].
// X: [Mp] rows of Kp * kBytesPerK bytes, Y: [Np] rows likewise. sx / sy: FP8 scales
// [Kp/128][Mp] and [Kp/128][Np]. Host guarantees 256 * row bytes < 2^31.
template <int KIND, int W, int kBufs>
__global__ __launch_bounds__(kThreads, W * kBufs == 4 ? 2 : 1) void gemm_lds_kernel(
    int M, int N, int Kp, int Mp, int Np, const char *__restrict__ X, const char *__restrict__ Y,
    const uint8_t *__restrict__ sx, const uint8_t *__restrict__ sy, float *__restrict__ C, int ldc, int slices) {
  using P = Pipe<KIND>;
  using F = typename P::Frag;
  constexpr int kTile = tile_edge(W), kWaveRows = 32 * W, kPanelB = panel_bytes(W), kStageB = 2 * kPanelB;
  constexpr int kAhead = kBufs - 1;  // stages fetched ahead of the one in use
  constexpr int kDmas = 4 * W;                                 // of a wave, per stage
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1, half = lane >> 5, l32 = lane & 31;
  int tm, tn;
  tile_coords(blockIdx.x, Mp / kTile, Np / kTile, tm, tn);
  const int m0 = tm * kTile, n0 = tn * kTile;
  const int rowb = Kp * P::kBytesPerK;
  const int first = slice_begin(Kp / P::kK, blockIdx.y, slices);
  const int stages = slice_begin(Kp / P::kK, blockIdx.y + 1, slices) - first;
  C += int64_t(blockIdx.y) * M * ldc;

  // Global -> LDS. One DMA instruction of a wave fills a 1 KiB chunk = 8 rows of a panel,
  // lane l writing LDS bytes 16 l .. 16 l + 15: slot l & 7 of row l >> 3 of the chunk. Row R
  // of a panel stores its piece p at slot p ^ ((R >> 1) & 7). DMA d (0..4W - 1) of a stage:
  // operand d & 1, chunk c = 4 (d >> 1) + wave, i.e. rows R = 8 c + (l >> 3), whose key
  // (R >> 1) & 7 = 4 (wave & 1) + (l >> 4) is the same for all DMAs of a lane.
  const int drow = lane >> 3;
  const int dkey = 4 * (wave & 1) + (drow >> 1);
  const unsigned voff = unsigned((drow + 8 * wave) * rowb + (((lane & 7) ^ dkey) << 4));
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(X) + int64_t(m0) * rowb, 0, kTile * rowb, 0x00020000);
  const __amdgpu_buffer_rsrc_t ry =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(Y) + int64_t(n0) * rowb, 0, kTile * rowb, 0x00020000);
  auto dma = [&](int d, int ks, int buf) {
    const int j = d >> 1;
    const unsigned soff = unsigned(32 * j * rowb + (first + ks) * kRowB);
    char *l = lds + buf * kStageB + (d & 1) * kPanelB + (4 * j + wave) * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds((d & 1) ? ry : rx, (lds_void *)(l), 16, voff, soff, 0, 0);
  };

  // Fragment reads: lane (half, l32) of tile i reads row R = wm*32W + 32 i + l32 (A) or
  // wn*32W + 32 i + l32 (B); piece p sits at slot p ^ ((R >> 1) & 7) = p ^ ((l32 >> 1) & 7).
  // The LDS serves 16 lanes per cycle over 64 banks (two 128-byte rows): lanes l32 .. l32 + 15
  // have 16 different (R & 1, (R >> 1) & 7), so they hit 16 different bank groups.
  const int sw = (l32 >> 1) & 7;
  const int arow = (wm * kWaveRows + l32) * kRowB, brow = kPanelB + (wn * kWaveRows + l32) * kRowB;
  auto piece = [&](int buf, int row, int p) -> i32x4 {
    return *reinterpret_cast<const i32x4 *>(lds + buf * kStageB + row + ((p ^ sw) << 4));
  };
  // BF16 step s uses piece 2 s + half (K 16 s + 8 half .. + 7, the MFMA's own K order);
  // BF16X3 step s: high part piece 2 s + half, low part 4 + 2 s + half; FP8 step s: pieces
  // 4 s + 2 half and 4 s + 2 half + 1 (K 64 s + 32 half .. + 31). FP32 step s: piece
  // 2 s + half, K 8 s + 4 half + t for t = 0 .. 3; MFMA t of the step takes value t, so it
  // sums K 8 s + t and 8 s + 4 + t (a K order that A and B share: the sum is unchanged).
  auto frag = [&](int buf, int row, int s, int part) -> F {
    if constexpr (KIND == kFP8) {
      const int p0 = 4 * s + 2 * half;
      const i32x4 x = piece(buf, row, p0), y = piece(buf, row, p0 + 1);
      return i32x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
    } else if constexpr (KIND == kF32) {
      return piece(buf, row, 2 * s + half);
    } else {
      return __builtin_bit_cast(bf16x8, piece(buf, row, 4 * part + 2 * s + half));
    }
  };

  f32x16 acc[W][W];
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  // FP8 scales of the current stage (set 0) and of the next kScales (set i moves to set i - 1 at the
  // stage boundary). They are loaded before the DMAs of stages that may still be in flight when they
  // are needed, since loads return in order.
  constexpr int kScales = kAhead > 1 ? kAhead - 1 : 1;
  int sa[kScales + 1][W], sb[kScales + 1][W];
  auto scales = [&](int ks, int set) {
#pragma unroll
    for (int i = 0; i < W; ++i) {
      if constexpr (KIND == kFP8) {
        sa[set][i] = sx[int64_t(first + ks) * Mp + m0 + wm * kWaveRows + i * 32 + l32];
        sb[set][i] = sy[int64_t(first + ks) * Np + n0 + wn * kWaveRows + i * 32 + l32];
      } else {
        sa[set][i] = sb[set][i] = 0;
      }
    }
  };
  // DMAs of the next stage ride in the first MFMA groups of a stage so that they have most of
  // the stage to land: 4 per group in 4 groups, or 8 per group in 2 for FP8, whose MFMAs take
  // twice the cycles (a group of 4 spans 256 of the stage's 2048).
  auto dma_slot = [&](int group, int ks_next, int buf) {
    constexpr int kPer = KIND == kFP8 ? 8 : 4;
    if (group < 4 * W / kPer) {
#pragma unroll
      for (int e = 0; e < kPer; ++e) dma(kPer * group + e, ks_next, buf);
    }
  };

  // Stage 0 and its scales have landed once at most those of the stages after it are in flight.
#pragma unroll
  for (int i = 0; i < kScales; ++i) scales(min(i, stages - 1), i);
#pragma unroll
  for (int i = 0; i < kAhead; ++i)
    if (i < stages) {
#pragma unroll
      for (int d = 0; d < kDmas; ++d) dma(d, i, i);
    }
  if (stages >= kAhead)
    publish_stage<(kAhead - 1) * kDmas>();
  else
    publish_stage<0>();

  if constexpr (KIND == kBF16X3) {
    // Fragments: al, ah, bl single; bh double (it is used by the first and the last MFMA
    // group of a step). Order per step: A = Al.Bh, B = Ah.Bl, C = Ah.Bh. Ah, Bl of step s
    // are read at its start (used from group B on); Al, Bh of step s + 1 right after group A.
    F al[W], ah[W], bl[W], bh[2][W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
      al[i] = frag(0, arow + i * 32 * kRowB, 0, 1);
      bh[0][i] = frag(0, brow + i * 32 * kRowB, 0, 0);
    }
    auto stage = [&](int ks, auto fill_tag, auto more_tag) {
      constexpr bool kFill = decltype(fill_tag)::value, kMore = decltype(more_tag)::value;
      const int buf = ks & (kBufs - 1), next = (ks + 1) & (kBufs - 1);
#pragma unroll
      for (int s = 0; s < P::kSteps; ++s) {
#pragma unroll
        for (int i = 0; i < W; ++i) {
          ah[i] = frag(buf, arow + i * 32 * kRowB, s, 0);
          bl[i] = frag(buf, brow + i * 32 * kRowB, s, 1);
        }
        CSMI_SCHED_FENCE();
#pragma unroll
        for (int g = 0; g < W; ++g) {
#pragma unroll
          for (int j = 0; j < W; ++j) mma<KIND>(al[g], bh[s & 1][j], acc[g][j], 0, 0);
          if (kFill && s == 0) dma_slot(g, ks + kAhead, (ks + kAhead) & (kBufs - 1));
          CSMI_SCHED_FENCE();
        }
        if (s + 1 < P::kSteps) {
#pragma unroll
          for (int i = 0; i < W; ++i) {
            al[i] = frag(buf, arow + i * 32 * kRowB, s + 1, 1);
            bh[(s + 1) & 1][i] = frag(buf, brow + i * 32 * kRowB, s + 1, 0);
          }
        } else {
          // Every read of this stage's buffer has been issued (Ah, Bl above): publish the next
          // stage (own DMAs landed, then the barrier) and read its first fragments while the
          // remaining two groups run.
          publish_stage<kFill ? (kAhead - 1) * kDmas : 0>();
          if (kMore) {
#pragma unroll
            for (int i = 0; i < W; ++i) {
              al[i] = frag(next, arow + i * 32 * kRowB, 0, 1);
              bh[0][i] = frag(next, brow + i * 32 * kRowB, 0, 0);
            }
          }
        }
        CSMI_SCHED_FENCE();
#pragma unroll
        for (int g = 0; g < W; ++g) {
#pragma unroll
          for (int j = 0; j < W; ++j) mma<KIND>(ah[g], bl[j], acc[g][j], 0, 0);
          CSMI_SCHED_FENCE();
        }
#pragma unroll
        for (int g = 0; g < W; ++g) {
#pragma unroll
          for (int j = 0; j < W; ++j) mma<KIND>(ah[g], bh[s & 1][j], acc[g][j], 0, 0);
          CSMI_SCHED_FENCE();
        }
      }
    };
    run_stages<kAhead>(stages, stage);
  } else {
    // Fragments double-buffered across the K steps of a stage (kSteps is even, so step 0
    // of every stage uses set 0).
    F fa[2][W], fb[2][W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
      fa[0][i] = frag(0, arow + i * 32 * kRowB, 0, 0);
      fb[0][i] = frag(0, brow + i * 32 * kRowB, 0, 0);
    }
    auto stage = [&](int ks, auto fill_tag, auto more_tag) {
      constexpr bool kFill = decltype(fill_tag)::value, kMore = decltype(more_tag)::value;
      const int buf = ks & (kBufs - 1), next = (ks + 1) & (kBufs - 1);
      if (kMore) scales(min(ks + kScales, stages - 1), kScales);
#pragma unroll
      for (int s = 0; s < P::kSteps; ++s) {
        if (s + 1 < P::kSteps) {
#pragma unroll
          for (int i = 0; i < W; ++i) {
            fa[(s + 1) & 1][i] = frag(buf, arow + i * 32 * kRowB, s + 1, 0);
            fb[(s + 1) & 1][i] = frag(buf, brow + i * 32 * kRowB, s + 1, 0);
          }
        } else {
          // The last step's fragments were read during the previous step, so this stage's
          // buffer is no longer read: publish the next stage (own DMAs and scale loads landed,
          // then the barrier) and read its first fragments while this step's MFMAs run.
          publish_stage<kFill ? (kAhead - 1) * kDmas : 0>();
          if (kMore) {
#pragma unroll
            for (int i = 0; i < W; ++i) {
              fa[0][i] = frag(next, arow + i * 32 * kRowB, 0, 0);
              fb[0][i] = frag(next, brow + i * 32 * kRowB, 0, 0);
            }
          }
        }
        CSMI_SCHED_FENCE();
        if constexpr (KIND == kF32) {
          // 4 MFMAs per tile, value t of every fragment in round t: 16 independent
          // accumulators between two uses of one. (__int_as_float, not __builtin_bit_cast: the
          // latter applied to a vector element reads element 0 with this compiler.)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int g = 0; g < W; ++g) {
#pragma unroll
              for (int j = 0; j < W; ++j)
                acc[g][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__int_as_float(fa[s & 1][g][t]),
                                                                 __int_as_float(fb[s & 1][j][t]),
                                                                 acc[g][j], 0, 0, 0);
              if (kFill && t == 0) dma_slot(s * W + g, ks + kAhead, (ks + kAhead) & (kBufs - 1));
              CSMI_SCHED_FENCE();
            }
          }
        } else {
#pragma unroll
          for (int g = 0; g < W; ++g) {
#pragma unroll
            for (int j = 0; j < W; ++j)
              mma<KIND>(fa[s & 1][g], fb[s & 1][j], acc[g][j], sa[0][g], sb[0][j]);
            if (kFill) dma_slot(s * W + g, ks + kAhead, (ks + kAhead) & (kBufs - 1));
            CSMI_SCHED_FENCE();
          }
        }
      }
      if (kMore) {
#pragma unroll
        for (int set = 0; set < kScales; ++set)
#pragma unroll
          for (int i = 0; i < W; ++i) {
            sa[set][i] = sa[set + 1][i];
            sb[set][i] = sb[set + 1][i];
          }
      }
    };
    run_stages<kAhead>(stages, stage);
  }

  // acc[i][j][e]: row = 8*(e/4) + 4*half + e%4, col = l32 of the 32x32 tile (i, j)
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = m0 + wm * kWaveRows + i * 32 + 8 * (e / 4) + 4 * half + (e % 4);
        const int c = n0 + wn * kWaveRows + j * 32 + l32;
        if (r < M && c < N) C[int64_t(r) * ldc + c] = acc[i][j][e];
      }
}

// ------------------------------------------------------------------------ direct kernel
// Products too small to fill the chip with 256 x 256 tiles. A wave owns a (16 T) x (16 T) tile of
// C and reads its operands from A and B as they lie, without a pre-pass and without LDS: per K
// step a lane holds kVals consecutive K values of one row of each 16-row tile of A (16-byte loads
// along K) and, for each of those K, T consecutive columns of B (one load of 4 T bytes along N).
// MFMA tile j takes the columns n0 + T c + j, c = 0..15, so a lane's T columns are the T tiles of
// its 16 x 16 column c, and its results are T consecutive columns too. kWK waves of a workgroup
// take every kWK-th K step of the same tile and add their sums through LDS, in wave order; with
// kWK = 1 the four waves take four tiles below one another instead. The operands of the next step
// load while the current one's MFMAs run.
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int KIND>
constexpr int kDirectVals = KIND == kF32 ? 4 : KIND == kFP8 ? 32 : 8;

template <int KIND, int T>
struct DirectFrags {
  float a[T][kDirectVals<KIND>], b[T][kDirectVals<KIND>];
};

__device__ __forceinline__ bf16x8 to_bf16x8(const float (&v)[8]) {
  i32x4 h;
#pragma unroll
  for (int e = 0; e < 4; ++e) h[e] = int(bf16x2(v[2 * e], v[2 * e + 1]));
  return __builtin_bit_cast(bf16x8, h);
}

__device__ __forceinline__ void split_bf16x8(const float (&v)[8], bf16x8 &hi, bf16x8 &lo) {
  i32x4 h, l;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t w = bf16x2(v[2 * e], v[2 * e + 1]);
    h[e] = int(w);
    l[e] = int(bf16x2(v[2 * e] - __uint_as_float(w << 16), v[2 * e + 1] - __uint_as_float(w & 0xffff0000u)));
  }
  hi = __builtin_bit_cast(bf16x8, h);
  lo = __builtin_bit_cast(bf16x8, l);
}

// 32 values of a 128-wide K block whose other 96 are in lanes 16, 32 and 48 away: quantised with
// the block's scale, as the pre-pass does.
__device__ __forceinline__ i32x8 to_fp8x32(const float (&v)[32], int &scale) {
  float m = 0.0f;
#pragma unroll
  for (int e = 0; e < 32; ++e) m = fmaxf(m, fabsf(v[e]));
  m = fmaxf(m, __shfl_xor(m, 16, 64));
  m = fmaxf(m, __shfl_xor(m, 32, 64));
  const int e = fp8_scale_exponent(m);
  const float inv = ldexpf(1.0f, -e);
  i32x8 w;
#pragma unroll
  for (int j = 0; j < 8; ++j) w[j] = int(fp8x4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3], inv));
  scale = e + 127;
  return w;
}

template <int KIND, int T>
__device__ __forceinline__ void direct_mma(const DirectFrags<KIND, T> &f, f32x4 (&acc)[T][T]) {
  if constexpr (KIND == kF32) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.a[i][t], f.b[j][t], acc[i][j], 0, 0, 0);
  } else if constexpr (KIND == kBF16) {
    bf16x8 a[T], b[T];
#pragma unroll
    for (int i = 0; i < T; ++i) a[i] = to_bf16x8(f.a[i]), b[i] = to_bf16x8(f.b[i]);
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
      for (int j = 0; j < T; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
  } else if constexpr (KIND == kBF16X3) {
    bf16x8 ah[T], al[T], bh[T], bl[T];
#pragma unroll
    for (int i = 0; i < T; ++i) split_bf16x8(f.a[i], ah[i], al[i]), split_bf16x8(f.b[i], bh[i], bl[i]);
#pragma unroll
    for (int part = 0; part < 3; ++part)
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part == 0 ? al[i] : ah[i], part == 1 ? bl[j] : bh[j],
                                                              acc[i][j], 0, 0, 0);
  } else {
    i32x8 a[T], b[T];
    int sa[T], sb[T];
#pragma unroll
    for (int i = 0; i < T; ++i) a[i] = to_fp8x32(f.a[i], sa[i]), b[i] = to_fp8x32(f.b[i], sb[i]);
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
      for (int j = 0; j < T; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[i], b[j], acc[i][j], 0, 0, 0, sa[i], 0, sb[j]);
  }
}

// The sums of K steps first, first + stride, ... of the tile at (m0, n0).
template <int KIND, int T>
__device__ __forceinline__ void direct_tile(int M, int N, int K, const float *__restrict__ A, int lda,
                                            const float *__restrict__ B, int ldb, int m0, int n0, int lane, int first,
                                            int stride, f32x4 (&acc)[T][T]) {
  constexpr int kVals = kDirectVals<KIND>, kStep = 4 * kVals;
  const int l16 = lane & 15, quad = lane >> 4;
  const int nb = n0 + T * l16;  // this lane's T columns
  const bool inside = nb + T <= N;
  const float *arow[T];  // rows past the end repeat the last one: their results are not stored
#pragma unroll
  for (int i = 0; i < T; ++i) arow[i] = A + int64_t(min(m0 + 16 * i + l16, M - 1)) * lda + quad * kVals;
  int ncol[T];
#pragma unroll
  for (int j = 0; j < T; ++j) ncol[j] = min(nb + j, N - 1);

  auto load = [&](int step, DirectFrags<KIND, T> &f) {
    const int k0 = step * kStep, k = k0 + quad * kVals;  // this lane's K values: k .. k + kVals - 1
    const float *brow = B + int64_t(k) * ldb;
    if (k + kVals <= K) {
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int t = 0; t < kVals; t += 4) {
          const f4u v = *reinterpret_cast<const f4u *>(arow[i] + k0 + t);
          f.a[i][t] = v.x, f.a[i][t + 1] = v.y, f.a[i][t + 2] = v.z, f.a[i][t + 3] = v.w;
        }
      if (inside) {
#pragma unroll
        for (int t = 0; t < kVals; ++t) {
          const float *q = brow + int64_t(t) * ldb + nb;
          if constexpr (T == 4) {
            const f4u v = *reinterpret_cast<const f4u *>(q);
            f.b[0][t] = v.x, f.b[1][t] = v.y, f.b[2][t] = v.z, f.b[3][t] = v.w;
          } else if constexpr (T == 2) {
            const f2u v = *reinterpret_cast<const f2u *>(q);
            f.b[0][t] = v.x, f.b[1][t] = v.y;
          } else {
            f.b[0][t] = *q;
          }
        }
      } else {
#pragma unroll
        for (int t = 0; t < kVals; ++t)
#pragma unroll
          for (int j = 0; j < T; ++j) f.b[j][t] = brow[int64_t(t) * ldb + ncol[j]];
      }
    } else {
      // past the end of K: zeros in both operands
#pragma unroll
      for (int t = 0; t < kVals; ++t) {
#pragma unroll
        for (int i = 0; i < T; ++i) f.a[i][t] = k + t < K ? arow[i][k0 + t] : 0.0f;
#pragma unroll
        for (int j = 0; j < T; ++j) f.b[j][t] = k + t < K ? brow[int64_t(t) * ldb + ncol[j]] : 0.0f;
      }
    }
    CSMI_SCHED_FENCE();  // the loads go out before the MFMAs of the step before
  };

#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int steps = (K + kStep - 1) / kStep;
  int step = first;
  if (step < steps) {
    DirectFrags<KIND, T> f[2];
    load(step, f[0]);
    for (;;) {
      if (step + stride >= steps) {
        direct_mma<KIND, T>(f[0], acc);
        break;
      }
      load(step + stride, f[1]);
      direct_mma<KIND, T>(f[0], acc);
      step += stride;
      if (step + stride >= steps) {
        direct_mma<KIND, T>(f[1], acc);
        break;
      }
      load(step + stride, f[0]);
      direct_mma<KIND, T>(f[1], acc);
      step += stride;
    }
  }

}

// acc[i][j][e] of a direct tile is row m0 + 16 i + 4 quad + e, column n0 + T l16 + j.
template <int T>
__device__ __forceinline__ void store_run(int M, int N, float *__restrict__ C, int ldc, int row, int col,
                                          const float (&v)[T]) {
  if (row >= M) return;
  float *c = C + int64_t(row) * ldc + col;
  if (T == 4 && col + 4 <= N) {
    *reinterpret_cast<f4u *>(c) = f4u{v[0], v[1 % T], v[2 % T], v[3 % T]};
    return;
  }
#pragma unroll
  for (int j = 0; j < T; ++j)
    if (col + j < N) c[j] = v[j];
}

template <int T>
__device__ __forceinline__ void store_tile(int M, int N, float *__restrict__ C, int ldc, int m0, int n0, int lane,
                                           const f32x4 (&acc)[T][T]) {
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v[T];
#pragma unroll
      for (int j = 0; j < T; ++j) v[j] = acc[i][j][e];
      store_run<T>(M, N, C, ldc, m0 + 16 * i + 4 * (lane >> 4) + e, n0 + T * (lane & 15), v);
    }
}

template <int KIND, int T, int kWK>
__global__ __launch_bounds__(kWK == 1 ? 256 : 64 * kWK) void gemm_direct_kernel(
    int M, int N, int K, const float *__restrict__ A, int lda, const float *__restrict__ B, int ldb,
    float *__restrict__ C, int ldc, int tiles_m, int slices) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int tm = int(blockIdx.x) % tiles_m, tn = int(blockIdx.x) / tiles_m;
  const int m0 = (kWK == 1 ? tm * 4 + wave : tm) * 16 * T, n0 = tn * 16 * T;
  f32x4 acc[T][T];
  direct_tile<KIND, T>(M, N, K, A, lda, B, ldb, m0, n0, lane, int(blockIdx.y) * kWK + (kWK == 1 ? 0 : wave),
                       kWK * slices, acc);
  C += int64_t(blockIdx.y) * M * ldc;
  if constexpr (kWK == 1) {
    store_tile<T>(M, N, C, ldc, m0, n0, lane, acc);
  } else {
    // part[wave][(i, e, j)][lane]
    extern __shared__ float part[];
    constexpr int kRuns = 4 * T;  // runs of T columns per lane
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < T; ++j) part[((wave * kRuns + 4 * i + e) * T + j) * 64 + lane] = acc[i][j][e];
    __syncthreads();
    for (int run = wave; run < kRuns; run += kWK) {
      float v[T];
#pragma unroll
      for (int j = 0; j < T; ++j) v[j] = part[(run * T + j) * 64 + lane];
      for (int w = 1; w < kWK; ++w)
#pragma unroll
        for (int j = 0; j < T; ++j) v[j] += part[((w * kRuns + run) * T + j) * 64 + lane];
      store_run<T>(M, N, C, ldc, m0 + 16 * (run / 4) + 4 * (lane >> 4) + run % 4, n0 + T * (lane & 15), v);
    }
  }
}

// ------------------------------------------------------------------------ FP32 from three parts
// Large FP32 products on the BF16 matrix cores, which do 16 times the FP32 ones' work per cycle. A
// 24-bit significand is exactly three 8-bit ones, x = h + m + l (each the BF16 nearest to what is
// left; Henry, Tang & Heinecke 2019), and of the nine products the six of hh, hm, mh, mm, hl and lh
// are summed in FP32: what the others would add is below 2^-24 of |a||b|, one unit roundoff, and all but
// that for a = b = 1 + 2^-8 - 2^-17, say. Products that FP32 holds exactly lose nothing. The error against
// FP64 of arbitrary values is that of the FP32 matrix cores or less, since 16 products meet in one rounding
// instead of two: relative to |C|, U(-1,1), K = 16 3.2e-8 / 7.4e-8, 256 2.3e-7 / 2.9e-7, 1024 4.8e-7 /
// 5.7e-7, 4096 1.0e-6 / 1.1e-6. Where all values are that one, FP32 sums round alike (5.9e-8 at K = 4096), and
// the parts' sums do not (3.8e-6).
// The split is exact, and the products' sums are FP32's, only in a range: not for infinities and
// NaN, values that round to an infinite BF16, parts below BF16's normal range, products near FP32's
// least and sums near its greatest (h may be above x, and hh overflow where ab does not). The pre-pass
// keeps the least and the greatest exponent of each of its pieces of A and B (0 as the least for values
// out of range), and a tile of C adds the chunks of 64 K where its rows or columns leave the range from A
// and B on the FP32 matrix cores, whose accumulators lie as the BF16 ones' do.
// A chunk costs about 2.7 times its split form there: 2048^3 with one value out of range 97 us against 95,
// with one in every chunk 166 (180 both when such tiles left the split whole); 4096^3 611 (1345) and
// 1059 (1258; 983 to 1020 in a kernel of FP32 MFMAs alone).
constexpr int kSplitK = 16;  // K values of a stage
// One part of an operand's stage (W = 4: 8 KiB); h, m and l of both operands are a stage (48 KiB), and
// three stages are in LDS (144 KiB).
constexpr int part_bytes(int W) { return tile_edge(W) * kSplitK * 2; }
// The chunks of K whose values are out of range follow, a bit each (check_depth bounds K).
constexpr int kMaxChunks = 1 << 15;
constexpr size_t split_lds_bytes(int W) { return size_t(18) * part_bytes(W) + kMaxChunks / 8; }
// Exponents (biased) of the operands, and of a product of both, that stay on the BF16 path: 2^21 products
// at most (check_depth) of less than 2^(76 + 2) stay far below an overflow.
constexpr unsigned kMinExponent = 24, kMinProduct = 254 - 110, kMaxProduct = 254 + 76;
// The exponents of a piece of an operand: 255 less the least (0 for zeros alone, 255 where a value is out
// of range), and the greatest. Those of several pieces together are the maxima.
typedef uint16_t Exponents __attribute__((ext_vector_type(2)));

struct SplitArgs {
  const float *a, *b;
  int m, n, k, lda, ldb, mp, np, kp;
  char *x, *y;         // [kp / 16][3][2][mp or np][8] BF16
  Exponents *ea, *eb;  // [mp / 64][chunks] and [np / 64][chunks], chunks of 64 K
  unsigned row_blocks;
};

__device__ __forceinline__ bool in_split_range(Exponents a, Exponents b) {
  return 255u - a[0] >= kMinExponent && 255u - b[0] >= kMinExponent && 510u - a[0] - b[0] >= kMinProduct &&
         unsigned(a[1]) + b[1] <= kMaxProduct;
}

// Splits 16 consecutive K values of one row of an operand, stores them and returns their exponents.
__device__ __forceinline__ Exponents split_store(const float (&v)[16], char *dst, int64_t part_stride) {
  unsigned least = 255, greatest = 0;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const uint32_t bits = __float_as_uint(v[e]) & 0x7fffffffu;
    const unsigned x = bits >= 0x7f7f8000u ? 0u : bits == 0 ? 255u : bits >> 23;
    least = min(least, x);
    greatest = max(greatest, bits);
  }
  float r[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) r[e] = v[e];
#pragma unroll
  for (int part = 0; part < 3; ++part) {
    i32x4 w[2];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t h = bf16x2(r[2 * e], r[2 * e + 1]);
      w[e / 4][e % 4] = int(h);
      r[2 * e] -= __uint_as_float(h << 16);
      r[2 * e + 1] -= __uint_as_float(h & 0xffff0000u);
    }
    *reinterpret_cast<i32x4 *>(dst + part * part_stride) = w[0];
    *reinterpret_cast<i32x4 *>(dst + part * part_stride + part_stride / 2) = w[1];
  }
  return Exponents{uint16_t(255 - least), uint16_t(greatest >> 23)};
}

// Workgroups [0, row_blocks) split 64 rows x 64 K of A (a thread per 16 K of a row), the others 64
// columns x 64 K of B (a thread per 16 K of a column: each load of a wave is 256 contiguous bytes).
// Rows, columns and K values past the source are zeros.
__global__ __launch_bounds__(256) void split_operands_kernel(SplitArgs p) {
  __shared__ Exponents waves[4];
  const int t = threadIdx.x;
  Exponents exponents = {0, 0};
  const unsigned chunks = unsigned(p.kp + 63) / 64;
  const bool is_a = blockIdx.x < p.row_blocks;
  const unsigned block = is_a ? blockIdx.x : blockIdx.x - p.row_blocks;
  const unsigned strip = is_a ? block / chunks : block % unsigned(p.np / 64);
  const unsigned chunk = is_a ? block % chunks : block / unsigned(p.np / 64);
  const int row = int(strip) * 64 + (is_a ? t / 4 : t % 64), k = int(chunk) * 64 + 16 * (is_a ? t % 4 : t / 64);
  if (k < p.kp) {
    float v[16];
    if (is_a) {
      const float *src = p.a + int64_t(row) * p.lda + k;
      if (row < p.m && k + 16 <= p.k) {
#pragma unroll
        for (int e = 0; e < 16; e += 4) {
          const f4u x = *reinterpret_cast<const f4u *>(src + e);
          v[e] = x[0], v[e + 1] = x[1], v[e + 2] = x[2], v[e + 3] = x[3];
        }
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = row < p.m && k + e < p.k ? src[e] : 0.0f;
      }
    } else {
      const float *src = p.b + int64_t(k) * p.ldb + row;
      if (row < p.n && k + 16 <= p.k) {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = src[int64_t(e) * p.ldb];
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = row < p.n && k + e < p.k ? src[int64_t(e) * p.ldb] : 0.0f;
      }
    }
    const int64_t part_stride = int64_t(is_a ? p.mp : p.np) * 32;
    char *dst = (is_a ? p.x : p.y) + int64_t(k / 16) * 3 * part_stride + int64_t(row) * 16;
    exponents = split_store(v, dst, part_stride);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1)
    exponents = __builtin_elementwise_max(
        exponents, __builtin_bit_cast(Exponents, __shfl_xor(__builtin_bit_cast(int, exponents), off, 64)));
  if (t % 64 == 0) waves[t / 64] = exponents;
  __syncthreads();
  if (t == 0)
    (is_a ? p.ea : p.eb)[int64_t(strip) * chunks + chunk] = __builtin_elementwise_max(
        __builtin_elementwise_max(waves[0], waves[1]), __builtin_elementwise_max(waves[2], waves[3]));
}

// 4 waves in 2x2 per output tile, W x W MFMA tiles each, as in gemm_lds_kernel. A stage is 16 K
// values: (W = 4) 96 MFMAs per wave, in six groups of 16 that use every accumulator once. Three stages
// live in LDS: while stage s computes, the fragments of s + 1 replace those of s as their last group
// has issued, and stage s + 2 streams into the buffer of s - 1 (six stages of W = 2 gain nothing:
// 2048^3 101.9 us against 103.5). The operands are packed so that each half (eight K values) of each
// part of a stage is contiguous: DMA and fragment reads are linear in LDS, without bank conflicts (with
// whole rows of 16 K contiguous a read met two rows in a bank: 2048^3 103.6 us, 102.0 without).
template <int W>
__global__ __launch_bounds__(kThreads, W == 4 ? 1 : 2) void gemm_split_kernel(
    int M, int N, int K, int Kp, int Mp, int Np, const char *__restrict__ X, const char *__restrict__ Y,
    const Exponents *__restrict__ ea, const Exponents *__restrict__ eb, const float *__restrict__ A, int lda,
    const float *__restrict__ B, int ldb, float *__restrict__ C, int ldc, int slices) {
  constexpr int kTile = tile_edge(W), kWaveRows = 32 * W, kPartB = part_bytes(W), kSplitPanelB = 3 * kPartB,
                kSplitStageB = 2 * kSplitPanelB;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1, half = lane >> 5, l32 = lane & 31;
  int tm, tn;
  tile_coords(blockIdx.x, Mp / kTile, Np / kTile, tm, tn);
  const int m0 = tm * kTile, n0 = tn * kTile;

  C += int64_t(blockIdx.y) * M * ldc;

  const int chunks = (Kp + 63) / 64;
  uint64_t *const out_of_range = reinterpret_cast<uint64_t *>(lds + 3 * kSplitStageB);
  for (int c = threadIdx.x; c - lane < chunks; c += kThreads) {
    Exponents a = {0, 0}, b = {0, 0};
    if (c < chunks) {
#pragma unroll
      for (int i = 0; i < W; ++i) {  // strips of 64 rows, and of 64 columns
        a = __builtin_elementwise_max(a, ea[int64_t(tm * W + i) * chunks + c]);
        b = __builtin_elementwise_max(b, eb[int64_t(tn * W + i) * chunks + c]);
      }
    }
    const uint64_t bits = __ballot(!in_split_range(a, b));
    if (lane == 0) out_of_range[c / 64] = bits;
  }
  __syncthreads();
  // The first chunk from c on that is out of range (out) or in it, at most `chunks`.
  auto next_chunk = [&](int c, bool out) {
    while (c < chunks) {
      const uint64_t bits = out_of_range[c / 64] ^ (out ? 0 : ~uint64_t(0));
      const int at = __ffsll(static_cast<unsigned long long>(bits >> (c % 64)));
      if (at) return __builtin_amdgcn_readfirstlane(min(c + at - 1, chunks));
      c = c / 64 * 64 + 64;
    }
    return chunks;
  };

  // Waves 0 and 1 stream A's panel, 2 and 3 B's: 3W chunks of 1 KiB each per stage.
  const int rows_p = wave < 2 ? Mp : Np;
  const char *const from = wave < 2 ? X + int64_t(m0) * 16 : Y + int64_t(n0) * 16;
  const int part_stride = rows_p * 32;
  const unsigned voff = unsigned(lane) * 16;
  auto dma = [&](int ks, int buf) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char *>(from) + int64_t(ks) * 3 * part_stride, 0,
        5 * (part_stride / 2) + kPartB / 2, 0x00020000);
    char *const l = lds + buf + (wave >> 1) * kSplitPanelB;
#pragma unroll
    for (int i = 0; i < 3 * W; ++i) {
      const int q = (wave & 1) * 3 * W + i;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)(l + q * 1024), 16, voff,
                                               unsigned(q / W * (part_stride / 2) + q % W * 1024), 0, 0);
    }
  };
  const int arow = (wm * kWaveRows + l32) * 16 + half * (kPartB / 2);
  const int brow = kSplitPanelB + (wn * kWaveRows + l32) * 16 + half * (kPartB / 2);
  auto frags = [&](bf16x8 (&f)[W], int buf, int row, int part) {
#pragma unroll
    for (int i = 0; i < W; ++i)
      f[i] = *reinterpret_cast<const bf16x8 *>(lds + buf + part * kPartB + row + i * 512);
  };

  f32x16 acc[W][W];
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  auto group = [&](const bf16x8 (&a)[W], const bf16x8 (&b)[W]) {
    CSMI_SCHED_FENCE();
#pragma unroll
    for (int i = 0; i < W; ++i)
#pragma unroll
      for (int j = 0; j < W; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    CSMI_SCHED_FENCE();
  };

  int cur = 0, nxt = kSplitStageB, nn = 2 * kSplitStageB;  // buffers of stages s, s + 1, s + 2
  bf16x8 ah[W], am[W], al[W], bm[W], bl[W], bh[2][W];
  // Stages [begin, end).
  auto split_stages = [&](int begin, int end) {
    dma(begin, cur);
    if (begin + 1 < end) dma(begin + 1, nxt);
    publish_stage<0>();
    frags(al, cur, arow, 2);
    frags(bh[0], cur, brow, 0);
    frags(bl, cur, brow, 2);
    frags(am, cur, arow, 1);
    frags(bm, cur, brow, 1);
    auto stage = [&](int ks, auto parity) {
      constexpr int P = decltype(parity)::value;
      frags(ah, cur, arow, 0);
      if (ks + 2 < end) dma(ks + 2, nn);
      // past the last stage the reads below fetch what no MFMA uses
      group(al, bh[P]);
      frags(al, nxt, arow, 2);
      group(ah, bl);
      frags(bl, nxt, brow, 2);
      group(am, bm);
      frags(bh[P ^ 1], nxt, brow, 0);
      group(am, bh[P]);
      frags(am, nxt, arow, 1);
      group(ah, bm);
      frags(bm, nxt, brow, 1);
      group(ah, bh[P]);
      // stage s + 2 has landed (own DMAs, then everybody's), and nobody reads stage s any more
      publish_stage<0>();
      const int free = cur;
      cur = nxt, nxt = nn, nn = free;
    };
    int ks = begin;
    for (; ks + 1 < end; ks += 2) {
      stage(ks, std::integral_constant<int, 0>());
      stage(ks + 1, std::integral_constant<int, 1>());
    }
    if (ks < end) stage(ks, std::integral_constant<int, 0>());
  };
  // K values [begin, end), from a multiple of 16 on, on the FP32 matrix cores: per step of 8 a lane holds four
  // consecutive K values of one row and of one column of each MFMA tile, straight from A and B, and MFMA t
  // takes value t of both halves. Rows and columns past the end repeat the
  // last one (their results are not stored); K values past the end are zeros.
  auto fp32_values = [&](int begin, int end) {
    const float *ap[W], *bp[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
      ap[i] = A + int64_t(min(m0 + wm * kWaveRows + 32 * i + l32, M - 1)) * lda + 4 * half;
      bp[i] = B + int64_t(4 * half) * ldb + min(n0 + wn * kWaveRows + 32 * i + l32, N - 1);
    }
    struct Step {
      f4u a[W], b[W];
    };
    // The loads that go out behind the MFMAs of tile row i and value t: all in the first quarter of a step of
    // W = 4, whose one wave per SIMD has nothing else to cover them (4096^3, all out of range, 1080 us, spread
    // over the step 1121), and spread over one of W = 2, where two waves would wait for the same burst
    // (5000^3 2590 us, in the first quarter 4290).
    auto load = [&](int k, int t, int i, Step &f) {
      if (t == 0) f.a[i] = *reinterpret_cast<const f4u *>(ap[i] + k);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (W == 4 ? t == 0 : t == u) f.b[i][u] = bp[i][int64_t(k + u) * ldb];
      CSMI_SCHED_FENCE();
    };
    // Multiplies f and loads `next` from k on.
    auto step = [&](const Step &f, int k, Step &next) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < W; ++i) {
#pragma unroll
          for (int j = 0; j < W; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[i][t], f.b[j][t], acc[i][j], 0, 0, 0);
          load(k, t, i, next);
        }
    };
    const int stop = min(end, K), full = begin + (stop - begin) / 16 * 16;
    if (begin < full) {
      Step f[2];
#pragma unroll
      for (int t = 0; t < 4; ++t)  // in the loop's order, whose waits would be for the last of them otherwise
#pragma unroll
        for (int i = 0; i < W; ++i) load(begin, t, i, f[0]);
#pragma unroll 1
      for (int k = begin; k < full; k += 16) {
        step(f[0], k + 8, f[1]);
        step(f[1], min(k + 16, full - 8), f[0]);  // the last values are not used
      }
    }
#pragma unroll 1
    for (int k = full; k < stop; k += 8) {
      Step f;
#pragma unroll
      for (int i = 0; i < W; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int at = min(k + t, K - 1 - 4 * half);  // negative in the upper half where K < 5: in bounds all the same
          const bool inside = k + t + 4 * half < K;
          const float x = ap[i][at], y = bp[i][int64_t(at) * ldb];
          f.a[i][t] = inside ? x : 0.0f;
          f.b[i][t] = inside ? y : 0.0f;
        }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < W; ++i)
#pragma unroll
          for (int j = 0; j < W; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[i][t], f.b[j][t], acc[i][j], 0, 0, 0);
    }
  };
  constexpr int kPerChunk = 64 / kSplitK;  // stages
  const int last = slice_begin(Kp / kSplitK, blockIdx.y + 1, slices);
#pragma unroll 1
  for (int s = slice_begin(Kp / kSplitK, blockIdx.y, slices); s < last;) {
    const int out = min(next_chunk(s / kPerChunk, true) * kPerChunk, last);
    if (s < out) split_stages(s, out);
    s = max(s, out);
    const int in = min(next_chunk(s / kPerChunk, false) * kPerChunk, last);
    if (s < in) {
      fp32_values(s * kSplitK, in * kSplitK);
      s = in;
    }
  }

  // acc[i][j][e]: row = 8*(e/4) + 4*half + e%4, col = l32 of the 32x32 tile (i, j)
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = m0 + wm * kWaveRows + i * 32 + 8 * (e / 4) + 4 * half + (e % 4);
        const int c = n0 + wn * kWaveRows + j * 32 + l32;
        if (r < M && c < N) C[int64_t(r) * ldc + c] = acc[i][j][e];
      }
}

int64_t round_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

__global__ __launch_bounds__(256) void zero_matrix_kernel(float *__restrict__ C, int M, int N, int ldc) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= int64_t(M) * N) return;
  C[(i / N) * ldc + i % N] = 0.0f;
}

// C = the sum of `slices` partial results [M][N] in their order, four values per thread. Bound by its launch
// (64 x 64 of 16 slices) or its reads (1024 x 1024 of 4: 16 MiB).
__global__ __launch_bounds__(256) void sum_slices_kernel(const float *__restrict__ part, int64_t n, int slices,
                                                         int N, float *__restrict__ C, int ldc) {
  const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  const float *p = part + i;
  if (i + 4 <= n) {
    f4u v = *reinterpret_cast<const f4u *>(p);
#pragma unroll 4
    for (int s = 1; s < slices; ++s) v += *reinterpret_cast<const f4u *>(p + int64_t(s) * n);
    const int64_t r = i / N, c = i % N;
    if (ldc == N || c + 4 <= N) {
      *reinterpret_cast<f4u *>(C + r * ldc + c) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) C[(i + e) / N * ldc + (i + e) % N] = v[e];
    }
  } else {
    for (int e = 0; i + e < n; ++e) {
      float v = p[e];
      for (int s = 1; s < slices; ++s) v += p[int64_t(s) * n + e];
      C[(i + e) / N * ldc + (i + e) % N] = v;
    }
  }
}

// Where the workgroups of a product write: C, or partial results in the stream's scratch behind `used`
// bytes of operands. Without room for them in a captured stream's scratch, K stays whole.
struct Target {
  char *scratch;
  float *out;
  int ld, slices;

  // `reserve`: what the scratch is sized to besides, where it can be: for calls of up to this size under
  // capture, whatever their path.
  Target(cs_stream *stream, int64_t used, int64_t reserve, int M, int N, float *C, int ldc, int wanted)
      : slices(wanted) {
    used = round_up(used, 256);
    int64_t total = used;
    if (slices > 1) total += int64_t(slices) * M * N * 4;
    if (slices > 1 && !scratch_fits(stream, size_t(total))) slices = 1, total = used;
    reserve_scratch(stream, size_t(std::max(total, reserve)));
    scratch = total ? static_cast<char *>(stream_scratch(stream, size_t(total))) : nullptr;
    out = slices > 1 ? reinterpret_cast<float *>(scratch + used) : C;
    ld = slices > 1 ? N : ldc;
  }
  void combine(cs_stream *stream, int M, int N, float *C, int ldc) const {
    const int64_t n = int64_t(M) * N;
    if (slices > 1)
      hipLaunchKernelGGL(sum_slices_kernel, dim3(unsigned((n + 1023) / 1024)), dim3(256), 0, stream->stream, out, n,
                         slices, N, C, ldc);
    CS_HIP(hipGetLastError());
  }
};

// The packed kernel's row offsets are 32 bits wide; K is held to that on every path.
template <int KIND>
void check_depth(int K) {
  using P = Pipe<KIND>;
  if (round_up(K, P::kK) * P::kBytesPerK * tile_edge(4) >= (int64_t(1) << 31))
    fail(CS_INVALID_VALUE, "K = " + std::to_string(K) + " is too large for this GEMM variant (K * bytes per "
                           "value must stay below 8 MiB)");
}

// Scratch of the operands of run_lds.
template <int KIND, int W>
int64_t packed_bytes(int M, int N, int K) {
  using P = Pipe<KIND>;
  const int64_t rows = round_up(M, tile_edge(W)) + round_up(N, tile_edge(W)), Kp = round_up(K, P::kK);
  return rows * Kp * P::kBytesPerK + 4096 + (KIND == kFP8 ? rows * (Kp / 128) + 4096 : 0);
}

template <int KIND, int W, int kBufs>
void run_lds(cs_stream *stream, int M, int N, int K, const float *A, int lda, const float *B, int ldb, float *C,
             int ldc, int slices) {
  using P = Pipe<KIND>;
  constexpr int kTile = tile_edge(W);
  const int64_t Mp = round_up(M, kTile), Np = round_up(N, kTile), Kp = round_up(K, P::kK);
  const int64_t rowb = Kp * P::kBytesPerK;
  const int64_t xbytes = Mp * rowb, ybytes = Np * rowb;
  const Target to(stream, packed_bytes<KIND, W>(M, N, K), packed_bytes<KIND, 4>(M, N, K), M, N, C, ldc, slices);
  char *const base = to.scratch, *x = base, *y = base + xbytes;
  uint8_t *sx = nullptr, *sy = nullptr;
  hipStream_t s = stream->stream;
  if constexpr (KIND == kFP8) {
    sx = reinterpret_cast<uint8_t *>(base + xbytes + ybytes);
    sy = sx + Mp * (Kp / 128);
  }
  {
    PackArgs pa;
    pa.a = A, pa.m = M, pa.k = K, pa.lda = lda, pa.mp = int(Mp), pa.kp = int(Kp), pa.x = x;
    pa.b = B, pa.n = N, pa.ldb = ldb, pa.np = int(Np), pa.y = y;
    pa.sx = sx, pa.sy = sy;
    int64_t col_tiles_k;
    if constexpr (KIND == kFP8) {  // 16 lanes per 128-wide block of a row; 128 K x 64 N column tiles
      pa.row_blocks = unsigned((Mp * (Kp / 128) * 16 + 255) / 256);
      pa.cols_gx = unsigned(Np / 64);
      col_tiles_k = Kp / 128;
    } else {  // one thread per 4 (FP32) or 8 K values of a row; 64 K x kPackTN N column tiles
      pa.row_blocks = unsigned((Mp * (Kp / (KIND == kF32 ? 4 : 8)) + 255) / 256);
      pa.cols_gx = unsigned(Np / kPackTN);
      col_tiles_k = (Kp + 63) / 64;
    }
    const int64_t blocks = int64_t(pa.row_blocks) + int64_t(pa.cols_gx) * col_tiles_k;
    hipLaunchKernelGGL(pack_operands_kernel<KIND>, dim3(unsigned(blocks)), dim3(256), 0, s, pa);
  }
  static std::atomic<uint64_t> allowed{0};
  allow_lds(allowed, stream->device->ordinal, reinterpret_cast<const void *>(&gemm_lds_kernel<KIND, W, kBufs>),
            lds_bytes(W, kBufs));
  const dim3 grid(static_cast<unsigned>((Mp / kTile) * (Np / kTile)), unsigned(to.slices));
  hipLaunchKernelGGL((gemm_lds_kernel<KIND, W, kBufs>), grid, dim3(kThreads), lds_bytes(W, kBufs), s, M, N, int(Kp),
                     int(Mp), int(Np), x, y, sx, sy, to.out, to.ld, to.slices);
  to.combine(stream, M, N, C, ldc);
}

// FP32 from three BF16 parts. False when the operands are too tall for its 32-bit offsets or, in a
// captured stream, too large for its scratch (three parts are 6 bytes of a value, the FP32 kernel's 4).
template <int W>
bool run_split(cs_stream *stream, int M, int N, int K, const float *A, int lda, const float *B, int ldb, float *C,
               int ldc, int slices) {
  constexpr int kTile = tile_edge(W);
  const int64_t Mp = round_up(M, kTile), Np = round_up(N, kTile), Kp = round_up(K, kSplitK);
  if (std::max(Mp, Np) * 96 >= (int64_t(1) << 31)) return false;
  const int64_t xbytes = Mp * Kp * 6, ybytes = Np * Kp * 6, chunks = (Kp + 63) / 64;
  const int64_t ebytes = (Mp + Np) / 64 * chunks * int64_t(sizeof(Exponents));
  const int64_t total = xbytes + ybytes + ebytes + 4096;
  if (!scratch_fits(stream, size_t(total))) return false;
  const Target to(stream, total, packed_bytes<kF32, 4>(M, N, K), M, N, C, ldc, slices);
  char *const base = to.scratch;
  SplitArgs p;
  p.a = A, p.b = B, p.m = M, p.n = N, p.k = K, p.lda = lda, p.ldb = ldb, p.mp = int(Mp), p.np = int(Np), p.kp = int(Kp);
  p.x = base, p.y = base + xbytes;
  p.ea = reinterpret_cast<Exponents *>(base + xbytes + ybytes), p.eb = p.ea + Mp / 64 * chunks;
  p.row_blocks = unsigned(Mp / 64 * chunks);
  const int64_t blocks = int64_t(p.row_blocks) + Np / 64 * chunks;
  hipLaunchKernelGGL(split_operands_kernel, dim3(unsigned(blocks)), dim3(256), 0, stream->stream, p);
  static std::atomic<uint64_t> allowed{0};
  allow_lds(allowed, stream->device->ordinal, reinterpret_cast<const void *>(&gemm_split_kernel<W>),
            split_lds_bytes(W));
  const dim3 grid(unsigned((Mp / kTile) * (Np / kTile)), unsigned(to.slices));
  hipLaunchKernelGGL(gemm_split_kernel<W>, grid, dim3(kThreads), split_lds_bytes(W), stream->stream, M, N, K, int(Kp),
                     int(Mp), int(Np), p.x, p.y, p.ea, p.eb, A, lda, B, ldb, to.out, to.ld, to.slices);
  to.combine(stream, M, N, C, ldc);
  return true;
}

template <int KIND, int T, int kWK>
void run_direct(cs_stream *stream, int M, int N, int K, const float *A, int lda, const float *B, int ldb, float *C,
                int ldc, int slices) {
  const int64_t rows = 16 * T * (kWK == 1 ? 4 : 1);  // of C per workgroup
  const int64_t tiles_m = (M + rows - 1) / rows, tiles_n = (N + 16 * T - 1) / (16 * T);
  const size_t lds = kWK == 1 ? 0 : size_t(kWK) * 256 * T * T * sizeof(float);
  const Target to(stream, 0, packed_bytes<KIND, 4>(M, N, K), M, N, C, ldc, slices);
  hipLaunchKernelGGL((gemm_direct_kernel<KIND, T, kWK>), dim3(unsigned(tiles_m * tiles_n), unsigned(to.slices)),
                     dim3(kWK == 1 ? 256 : 64 * kWK), lds, stream->stream, M, N, K, A, lda, B, ldb, to.out, to.ld,
                     int(tiles_m), to.slices);
  to.combine(stream, M, N, C, ldc);
}

// The direct kernel's launch shape. Where the lines lie (FP32 calls, in us, "T.kWK"):
//   * the largest T that still gives a tile per CU: 300x200x1000 (247 tiles of T = 1) 1.16 5.8,
//     2.8 10.7, 4.4 28.2; 512^3 (256 of T = 2) 2.8 5.8, 1.4 7.1, 4.4 13.1; 1000^3 (256 of T = 4)
//     4.4 29.1, 2.4 33.0, 1.4 51.4. T stays where a larger one would pad the result by more than
//     a third (65536x8x8: 1.1 4.2, 4.1 5.6).
//   * waves per tile as long as they are needed to fill the SIMDs and have a K step each:
//     300x200x1000 1.16 5.8, 1.4 7.2, 1.1 22.2; 2000x64x500 (500 tiles) 1.4 5.4, 1.16 6.5;
//     2048^3 (1024 tiles of T = 4) 4.1 155.9, 4.4 164.5; 65536x8x8 1.1 4.2, 1.4 5.0.
// FP8 holds 32 K values of every row and column per lane: more than T = 2 or than 4 waves per
// tile spills (300x200x1000: 1.4 10.8, 1.16 22.2, 4.4 71.1).
struct DirectPlan {
  int t = 1, wk = 1;
};

DirectPlan plan_direct(int kind, int64_t cus, int64_t M, int64_t N, int64_t K) {
  auto up = [](int64_t v, int64_t a) { return (v + a - 1) / a; };
  DirectPlan p;
  for (int t = kind == kFP8 ? 2 : 4; t > 1; t /= 2) {
    const int64_t e = 16 * t, area = up(M, e) * up(N, e) * e * e;
    if (up(M, e) * up(N, e) >= cus && area * 3 <= up(M, 16) * up(N, 16) * 256 * 4) {
      p.t = t;
      break;
    }
  }
  const int64_t tiles = up(M, 16 * p.t) * up(N, 16 * p.t);
  const int64_t steps = up(K, kind == kF32 ? 16 : kind == kFP8 ? 128 : 32);
  if (steps < 3 || tiles > (p.t == 4 ? 3 : 4) * cus) return p;
  p.wk = 4;
  if (kind != kFP8 && p.t < 4 && tiles <= cus && steps > 4) p.wk = p.t == 1 ? 16 : 8;
  return p;
}

// Whether two ranges of device memory meet.
bool overlap(const float *a, int64_t rows_a, int64_t cols_a, int lda, const float *c, int64_t rows_c, int64_t cols_c,
             int ldc) {
  const float *a1 = a + (rows_a - 1) * lda + cols_a, *c1 = c + (rows_c - 1) * ldc + cols_c;
  return a < c1 && c < a1;
}

// How a product runs: straight from A and B, or packed with 256 x 256 tiles (two stages of them in
// LDS), 128 x 128 tiles (two stages, two workgroups on a CU) or 128 x 128 tiles with four stages, one
// workgroup on a CU.
enum Path { kDirect, kTiles256, kTiles128, kDeep128 };
struct Plan {
  Path path;
  int slices;  // of K, each with workgroups of its own, added by a launch after them
};

// Each path's time is estimated from what it was measured to take (us): the direct kernel's from the
// flops of its padded tiles at the rate of its tile size, with the CUs its last round leaves idle; the
// packed kernels' from two launches, the pre-pass and one round of tiles over K for every 256
// workgroups begun. Over 64 shapes from 512^3 to 4096^3 the choice was within
// 3% of the fastest in 61 and within 7% in the others.
// Measured direct / 128 / deep 128 / 256:
//   FP32    300x200x1000 5.8 / - / - / 140, 1000^3 28 / 53 / - / 130, 2048^3 160 / 104 / - / 242,
//           4096^3 1269 / 620 / - / 594
//   BF16    1000^3 20 / 22 / 19 / 38, 2048^3 122 / 37 / 30 / 61, 2500^3 262 / 53 / 57 / 82, 4096^3
//           982 / 151 / 165 / 144
//   BF16x3  1000^3 20 / 38 / 32 / 74, 2048^3 83 / 65 / 56 / 130, 2500^3 244 / 105 / 112 / 164, 4096^3
//           655 / 356 / 377 / 326
//   FP8     512^3 6.5 / 10.2 / 9.8 / 20, 2048^3 259 / 28 / 24 / 46, 2500^3 522 / 40 / 46 / 61, 4096^3
//           2024 / 99 / 110 / 95
// Where a path starts too few workgroups for the CUs, K is cut into slices with workgroups of their own,
// counted at 3 us of launches and 8 bytes of traffic per partial result, and taken where that gains 5%
// (1 / chosen slices): FP32 64x64x4096 11.2 / 7.1 (16 of the direct kernel), 632x1305x3146 103 / 59 (128
// tiles, 4), BF16 128x1024x4096 27 / 20 (8), 1024x1024x4096 40 / 29 (3), FP8 64x64x4096 16.2 / 6.8.
// With 128 tiles on 64 of the CUs (1024x1024x4096, unsliced) a stage of two waits for the DMA of the next: BF16
// 55 us, with four 40; FP8 38 / 29.
template <int KIND>
Plan choose_path(double cus, double M, double N, double K, const DirectPlan &p) {
  struct Rates {
    double direct[3];   // TFLOP/s of T = 1, 2, 4
    double base;        // of a packed call, and what 256 x 256 tiles add
    double base_256;
    double pack;        // of a value of A or B
    // of one K of a round: 256 x 256 tiles on all CUs, on at most three quarters (a higher clock);
    // 128 x 128 tiles, one on a CU, two together; the same with four stages
    double t256, t256_few, t128, t128_pair, deep;
  };
  constexpr Rates r = KIND == kF32    ? Rates{{45, 80, 110}, 13, -2, 1.8e-6, 0.126, 0.107, 0.036, 0.066, 1e9}
                      : KIND == kBF16 ? Rates{{50, 85, 140}, 7, 0.5, 0.9e-6, 0.0245, 0.0245, 0.0107, 0.0145, 0.0071}
                      : KIND == kBF16X3
                          ? Rates{{50, 90, 190}, 7, 1.5, 1.35e-6, 0.0645, 0.058, 0.0228, 0.0365, 0.0180}
                          : Rates{{25, 60, 60}, 7, 1.5, 0.85e-6, 0.0130, 0.0130, 0.0066, 0.0078, 0.0043};
  auto tiles = [&](double edge) { return std::ceil(M / edge) * std::ceil(N / edge); };
  auto rounds = [&](double n) { return std::ceil(n / cus); };
  const double e = 16.0 * p.t, blocks = p.wk == 1 ? std::ceil(std::ceil(M / e) / 4) * std::ceil(N / e) : tiles(e);
  const double packed = r.base + r.pack * (M + N) * K + 0.5e-6 * M * N;
  const double t256 = tiles(256), r128 = rounds(tiles(128)), pairs = std::floor(r128 / 2);
  const double steps = std::ceil(K / (KIND == kF32 ? 16 : KIND == kFP8 ? 128 : 32));  // of the direct kernel
  // where a workgroup has idle waves nothing hides the padding of FP8's K steps of 128 (1x100000x64: 44 us,
  // packed 19; 3547x68x20, whose four waves have tiles, 5.9 / 8.3)
  const double deep = KIND == kFP8 && p.wk == 1 && M <= 3 * e ? 128 * steps : K;
  const double flops = 2e-6 * tiles(e) * e * e * deep / r.direct[p.t / 2];
  const double out = (KIND == kF32 ? 0.5e-6 : 1.2e-6) * M * N;
  auto direct = [&](double slices) { return 4 + flops * rounds(blocks * slices) * cus / (blocks * slices) + out; };
  const double time[] = {
      direct(1),
      packed + r.base_256 + K * rounds(t256) * (t256 <= 0.75 * cus ? r.t256_few : r.t256),
      packed + K * (pairs * r.t128_pair + (r128 - 2 * pairs) * r.t128),
      r128 == 1 ? packed + K * r.deep : 1e30,  // in several rounds nothing hides their ends
  };
  const int path = int(std::min_element(time, time + 4) - time);
  Plan best = {Path(path), 1};
  double least = time[path];
  auto consider = [&](Path candidate, int slices, double t) {
    t += 3 + 1.2e-6 * slices * M * N;
    if (t < 0.95 * least) best = {candidate, slices}, least = t;
  };
  for (int s = 2; s <= 16 && blocks * s <= cus && p.wk * s <= steps; s *= 2) consider(kDirect, s, direct(s));
  for (int s = 2; s <= 8 && tiles(128) * s <= cus && 128 * s <= K; ++s)
    consider(KIND == kF32 ? kTiles128 : kDeep128, s, packed + K / s * (KIND == kF32 ? r.t128 : r.deep));
  return best;
}

// False where a captured stream's scratch has no room for the operands (but for a C that needs the copies).
template <int KIND, int W, int kBufs>
bool run_packed(cs_stream *stream, int M, int N, int K, const float *A, int lda, const float *B, int ldb, float *C,
                int ldc, bool over, int slices) {
  if constexpr (KIND == kF32)
    if (!over && run_split<W>(stream, M, N, K, A, lda, B, ldb, C, ldc, slices)) return true;
  if (!over && !scratch_fits(stream, size_t(packed_bytes<KIND, W>(M, N, K)))) return false;
  run_lds<KIND, W, kBufs>(stream, M, N, K, A, lda, B, ldb, C, ldc, slices);
  return true;
}

// Rows and columns of C computed together.
constexpr int64_t kMaxEdge = int64_t(1) << 26;

template <int KIND>
void run(cs_stream *stream, int M, int N, int K, const float *A, int lda, const float *B, int ldb, float *C, int ldc) {
  check_depth<KIND>(K);
  const int64_t cus = stream->device->props.multiProcessorCount;
  // A C that overlaps A or B is written only from copies of both.
  const bool over = overlap(A, M, K, lda, C, M, N, ldc) || overlap(B, K, N, ldb, C, M, N, ldc);
  // A launch holds fewer than 2^32 threads, of which a narrow product takes one per value.
  if (!over && std::max(M, N) > kMaxEdge) {
    for (int64_t m = 0; m < M; m += kMaxEdge)
      for (int64_t n = 0; n < N; n += kMaxEdge)
        run<KIND>(stream, int(std::min<int64_t>(M - m, kMaxEdge)), int(std::min<int64_t>(N - n, kMaxEdge)), K,
                  A + m * lda, lda, B + n, ldb, C + m * ldc + n, ldc);
    return;
  }
  const DirectPlan p = plan_direct(KIND, cus, M, N, K);
  Plan plan = choose_path<KIND>(double(cus), M, N, K, p);
  if (over && plan.path == kDirect) plan = {kTiles128, 1};
  int z = plan.slices;
  if (plan.path != kDirect) {
    bool done = false;
    if (plan.path == kTiles256) done = run_packed<KIND, 4, 2>(stream, M, N, K, A, lda, B, ldb, C, ldc, over, z);
    if (plan.path == kTiles128) done = run_packed<KIND, 2, 2>(stream, M, N, K, A, lda, B, ldb, C, ldc, over, z);
    if constexpr (KIND != kF32)
      if (plan.path == kDeep128) done = run_packed<KIND, 2, 4>(stream, M, N, K, A, lda, B, ldb, C, ldc, over, z);
    if (done) return;
    z = 1;
  }
  switch (p.t * 100 + p.wk) {
    case 101: return run_direct<KIND, 1, 1>(stream, M, N, K, A, lda, B, ldb, C, ldc, z);
    case 104: return run_direct<KIND, 1, 4>(stream, M, N, K, A, lda, B, ldb, C, ldc, z);
    case 201: return run_direct<KIND, 2, 1>(stream, M, N, K, A, lda, B, ldb, C, ldc, z);
    case 204: return run_direct<KIND, 2, 4>(stream, M, N, K, A, lda, B, ldb, C, ldc, z);
  }
  if constexpr (KIND != kFP8) {
    switch (p.t * 100 + p.wk) {
      case 116: return run_direct<KIND, 1, 16>(stream, M, N, K, A, lda, B, ldb, C, ldc, z);
      case 208: return run_direct<KIND, 2, 8>(stream, M, N, K, A, lda, B, ldb, C, ldc, z);
      case 401: return run_direct<KIND, 4, 1>(stream, M, N, K, A, lda, B, ldb, C, ldc, z);
      case 404: return run_direct<KIND, 4, 4>(stream, M, N, K, A, lda, B, ldb, C, ldc, z);
    }
  }
  fail(CS_INVALID_OPERATION, "no direct GEMM kernel for this plan");
}

}  // namespace
}  // namespace csmi

using namespace csmi;

extern "C" cs_status cs_gemm(cs_stream *stream, int variant, int M, int N, int K, const float *A, int lda,
                             const float *B, int ldb, float *C, int ldc) {
  return guard([&] {
    if (!stream) fail(CS_INVALID_VALUE, "stream is null");
    if (M < 0 || N < 0 || K < 0) fail(CS_INVALID_VALUE, "negative dimension");
    if (lda < K || ldb < N || ldc < N) fail(CS_INVALID_VALUE, "leading dimension too small");
    if (variant < CS_GEMM_FP32 || variant > CS_GEMM_FP8)
      fail(CS_INVALID_VALUE, "unknown GEMM variant " + std::to_string(variant));
    if (M == 0 || N == 0) return;
    if (!C) fail(CS_INVALID_VALUE, "null matrix pointer");
    set_device(stream->device);
    if (K == 0) {  // empty sums: C = 0, and A and B are not read
      const int64_t n = int64_t(M) * N;
      hipLaunchKernelGGL(zero_matrix_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, stream->stream, C, M, N,
                         ldc);
      CS_HIP(hipGetLastError());
      return;
    }
    if (!A || !B) fail(CS_INVALID_VALUE, "null matrix pointer");
    if (int64_t(M) * K >= (int64_t(1) << 31) || int64_t(N) * K >= (int64_t(1) << 31))
      fail(CS_INVALID_VALUE, "operands are limited to 2^31 elements");
    switch (variant) {
      case CS_GEMM_FP32: run<kF32>(stream, M, N, K, A, lda, B, ldb, C, ldc); break;
      case CS_GEMM_BF16: run<kBF16>(stream, M, N, K, A, lda, B, ldb, C, ldc); break;
      case CS_GEMM_BF16X3: run<kBF16X3>(stream, M, N, K, A, lda, B, ldb, C, ldc); break;
      case CS_GEMM_FP8: run<kFP8>(stream, M, N, K, A, lda, B, ldb, C, ldc); break;
    }
  });
}
