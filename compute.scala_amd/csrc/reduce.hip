// Reductions for gfx950: full sum and max, row-wise sum/max/total in one pass, column sums.
//
// Replaces the reference's `sum` programs (Tensors.scala:308-393, 673-771). Layout and
// arithmetic:
//   * 256-thread workgroups (4 wave64s); each thread reads 16-byte vectors, several in
//     flight, so a row of 4096 floats is 4 loads per thread;
//   * per-thread sums are FP32 with a TwoSum compensation term, combined across the wave
//     with xor shuffles and across the 4 waves through LDS, still as (sum, compensation)
//     pairs, so the in-block result is accurate to about one FP32 rounding;
//   * block results are combined in FP64: every block writes an FP64 partial and a second,
//     one-workgroup kernel adds the partials in a fixed order, so results are deterministic
//     run to run. A last-workgroup ticket in the first kernel was built and measured slower:
//     each workgroup's write-through of its partial, the wait for it and the atomic on one
//     shared counter cost more than the second launch (C3 49.7 us against 44.0, a 16 MiB sum
//     15.9 us against 5.8). One wave per row with eight rows per workgroup (so one partial
//     per eight rows) made the combine 0.45 us shorter and the row pass 0.8 us longer;
//   * max uses fmaxf, which returns the non-NaN operand (OpenCLKernelBuilder.scala:279-285).
// The reference's parallel program loses elements when the local size is not a power of
// two (Tensors.scala:375-387); these kernels sum every element.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "internal.h"

#pragma clang fp contract(off)

namespace csmi {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void two_sum(float a, float b, float &s, float &e) {
  s = a + b;
  float bp = s - a;
  e = (a - (s - bp)) + (b - bp);
}

// Once the running sum s is infinite or NaN it stays so (inf + finite = inf, inf - inf and
// NaN + x = NaN), and only then can a TwoSum error term be NaN. So c is used only while s is
// finite: the result is s itself otherwise, as a plain FP32 sum of the same values gives
// (inf for [1, inf, 2] or [3e38, 3e38], NaN for [inf, -inf]).
struct Acc {
  float s = 0.0f, c = 0.0f;
  __device__ __forceinline__ float result() const { return __builtin_isfinite(s) ? s + c : s; }
  __device__ __forceinline__ double result64() const {
    return __builtin_isfinite(s) ? double(s) + double(c) : double(s);
  }
  __device__ __forceinline__ void add(float x) {
    float t, e;
    two_sum(s, x, t, e);
    s = t;
    c += e;
  }
  __device__ __forceinline__ void merge(float s2, float c2) {
    float t, e;
    two_sum(s, s2, t, e);
    s = t;
    c += c2 + e;
  }
};

__device__ __forceinline__ float nanmax(float a, float b) { return fmaxf(a, b); }

// Sum pair and max across the 64 lanes of a wave.
__device__ __forceinline__ void wave_reduce(Acc &a, float &m) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    float s2 = __shfl_xor(a.s, off, 64);
    float c2 = __shfl_xor(a.c, off, 64);
    float m2 = __shfl_xor(m, off, 64);
    a.merge(s2, c2);
    m = nanmax(m, m2);
  }
}

// Reduces (a, m) over a block of kW waves; the result is valid in thread 0.
template <int kW = kWaves>
__device__ __forceinline__ void block_reduce(Acc &a, float &m) {
  __shared__ float ls[kW], lc[kW], lm[kW];
  wave_reduce(a, m);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    ls[wave] = a.s;
    lc[wave] = a.c;
    lm[wave] = m;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    Acc t;
    t.s = ls[0];
    t.c = lc[0];
    float mm = lm[0];
#pragma unroll
    for (int w = 1; w < kW; ++w) {
      t.merge(ls[w], lc[w]);
      mm = nanmax(mm, lm[w]);
    }
    a = t;
    m = mm;
  }
}

// One workgroup of kFinish threads adds partials[0..n) in FP64 in a fixed order: thread t
// adds pairs 2t, 2t + 2 kFinish, ... (16-byte loads, eight in flight), then a fixed xor-shuffle
// tree inside each wave and the 16 waves in order.
constexpr int kFinish = 1024;
typedef double d2 __attribute__((ext_vector_type(2)));
__global__ __launch_bounds__(kFinish) void finish_sum_kernel(const double *__restrict__ partials, int64_t n,
                                                             float *out, double *out64) {
  __shared__ double lw[kFinish / 64];
  double acc = 0.0;
  const int64_t pairs = n / 2;
  const d2 *p2 = reinterpret_cast<const d2 *>(partials);  // partials are 16-byte aligned
  int64_t i = threadIdx.x;
  // eight 16-byte loads in flight per thread: one memory round trip for up to 16384 partials
  for (; i + 7 * kFinish < pairs; i += 8 * kFinish) {
    d2 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = p2[i + k * kFinish];
#pragma unroll
    for (int k = 0; k < 8; ++k) acc += v[k].x + v[k].y;
  }
  for (; i < pairs; i += kFinish) {
    const d2 v = p2[i];
    acc += v.x + v.y;
  }
  if (threadIdx.x == 0 && (n & 1)) acc += partials[n - 1];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if ((threadIdx.x & 63) == 0) lw[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = lw[0];
#pragma unroll
    for (int w = 1; w < kFinish / 64; ++w) t += lw[w];
    if (out) *out = float(t);
    if (out64) *out64 = t;
  }
}

__global__ __launch_bounds__(kFinish) void finish_max_kernel(const float *__restrict__ partials, int64_t n,
                                                             float *out) {
  __shared__ float lw[kFinish / 64];
  float m = __builtin_nanf("");
  for (int64_t i = threadIdx.x; i < n; i += kFinish) m = nanmax(m, partials[i]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = nanmax(m, __shfl_xor(m, off, 64));
  if ((threadIdx.x & 63) == 0) lw[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = lw[0];
#pragma unroll
    for (int w = 1; w < kFinish / 64; ++w) t = nanmax(t, lw[w]);
    *out = t;
  }
}

// A pass of a single workgroup writes its result itself, as the combine of one partial would.
__device__ __forceinline__ void write_total(double total, float *out, double *out64) {
  if (out) *out = float(total);
  if (out64) *out64 = total;
}

// ----------------------------------------------------------------------------- full sum/max
// With one workgroup *out and *out64 get the result, else each workgroup its partial.
template <bool kMax>
__global__ __launch_bounds__(kBlock) void reduce_all_kernel(const float *__restrict__ in, int64_t n,
                                                            double *partial64, float *partialmax, float *out,
                                                            double *out64) {
  Acc a;
  float m = __builtin_nanf("");
  const int64_t nvec = ((reinterpret_cast<uintptr_t>(in) & 15) == 0) ? n / 4 : 0;
  const f4 *in4 = reinterpret_cast<const f4 *>(in);
  // Block-strided chunks of kBlock vectors: consecutive threads read consecutive vectors.
  const int64_t stride = int64_t(gridDim.x) * kBlock;
  int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  for (; i + 3 * stride < nvec; i += 4 * stride) {
    f4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = __builtin_nontemporal_load(in4 + i + k * stride);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (kMax) {
        m = nanmax(m, nanmax(nanmax(v[k].x, v[k].y), nanmax(v[k].z, v[k].w)));
      } else {
        a.add(v[k].x); a.add(v[k].y); a.add(v[k].z); a.add(v[k].w);
      }
    }
  }
  for (; i < nvec; i += stride) {
    f4 v = __builtin_nontemporal_load(in4 + i);
    if (kMax) {
      m = nanmax(m, nanmax(nanmax(v.x, v.y), nanmax(v.z, v.w)));
    } else {
      a.add(v.x); a.add(v.y); a.add(v.z); a.add(v.w);
    }
  }
  for (int64_t j = nvec * 4 + int64_t(blockIdx.x) * kBlock + threadIdx.x; j < n; j += stride) {
    float x = in[j];
    if (kMax) m = nanmax(m, x); else a.add(x);
  }
  block_reduce(a, m);
  if (threadIdx.x == 0) {
    if (gridDim.x == 1) {
      if (kMax) *out = m;
      else write_total(a.result64(), out, out64);
    } else if (kMax) {
      partialmax[blockIdx.x] = m;
    } else {
      partial64[blockIdx.x] = a.result64();
    }
  }
}

// ----------------------------------------------------------------------------- rows
// A row starts at any 4-byte boundary (cols need not be a multiple of 4): 16-byte loads take
// four-byte alignment on this hardware, so rows are read in vectors of four from their first
// element, with cols % 4 single elements at the end.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// Adds four elements: pairwise inside the vector, then one compensated add.
__device__ __forceinline__ void add_vector(f4u v, Acc &a, float &m) {
  float s01, e01, s23, e23, s, e;
  two_sum(v.x, v.y, s01, e01);
  two_sum(v.z, v.w, s23, e23);
  two_sum(s01, s23, s, e);
  a.merge(s, e + e01 + e23);
  m = nanmax(m, nanmax(nanmax(v.x, v.y), nanmax(v.z, v.w)));
}

// Where the row kernels write, each nullable: a row's sum and maximum, and the workgroups' partial sums or,
// where there is one workgroup, the total. One argument, and no look at the grid, since a small call takes as
// long as its launches: a kernel that reads gridDim has 256 more bytes of arguments to write (22 x 607 4.2 us a
// call with them, 3.7 without).
struct RowOutputs {
  float *row_sum, *row_max;
  double *partial64;
  float *total;
  double *total64;
};

// One row's share of a lane: vectors lane, lane + kStep, ... of p, four loads in flight. The
// cols % 4 elements after the last whole vector ride with the other loads: in a wave or less as the end
// of one more vector that overlaps it (120011 x 77 12.0 us, one by one 13.1), in a workgroup one by one,
// which is shorter (3000 x 2500 8.9 us, as a vector 9.2). kShort: at most one vector per lane; what a
// launch of few short rows waits for is mostly its own instructions, so it gets a kernel of few.
template <int kStep, bool kShort, class Index>
__device__ __forceinline__ void read_row(const float *__restrict__ p, Index cols, int lane, Acc &a, float &m) {
  const Index nv = cols / 4;
  Index i = lane;
  if (!kShort) {
    const f4u *p4 = reinterpret_cast<const f4u *>(p);
    for (; i + 3 * kStep < nv; i += 4 * kStep) {
      f4u v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = __builtin_nontemporal_load(p4 + i + k * kStep);
#pragma unroll
      for (int k = 0; k < 4; ++k) add_vector(v[k], a, m);
    }
  }
  constexpr int kVecs = kShort ? 1 : 4;
  f4u v[kVecs];
  if constexpr (kStep > 64) {
    float x;
    const bool one = 4 * nv + lane < cols;
    if (one) x = p[4 * nv + lane];
    if (i < nv) {
#pragma unroll
      for (int k = 0; k < kVecs; ++k)
        if (i + k * kStep < nv)
          v[k] = __builtin_nontemporal_load(reinterpret_cast<const f4u *>(p + 4 * (i + k * kStep)));
#pragma unroll
      for (int k = 0; k < kVecs; ++k)
        if (i + k * kStep < nv) {
#pragma unroll
          for (int e = 0; e < 4; ++e) a.add(v[k][e]);
          m = nanmax(m, nanmax(nanmax(v[k].x, v[k].y), nanmax(v[k].z, v[k].w)));
        }
    }
    if (one) {
      a.add(x);
      m = nanmax(m, x);
    }
  } else {
    const int tail = static_cast<int>(cols % 4);
    if (nv == 0) {
      for (int j = lane; j < tail; j += kStep) {
        a.add(p[j]);
        m = nanmax(m, p[j]);
      }
      return;
    }
    const Index all = nv + (tail ? 1 : 0);
    if (i >= all) return;
#pragma unroll
    for (int k = 0; k < kVecs; ++k) {
      const Index c = i + k * kStep;
      if (c < all) v[k] = __builtin_nontemporal_load(reinterpret_cast<const f4u *>(p + (c < nv ? 4 * c : cols - 4)));
    }
#pragma unroll
    for (int k = 0; k < kVecs; ++k) {
      const Index c = i + k * kStep;
      if (c < all) {
        const int again = c < nv ? 0 : 4 - tail;  // elements that the vector before has added
#pragma unroll
        for (int e = 0; e < 4; ++e) a.add(e >= again ? v[k][e] : 0.0f);
        m = nanmax(m, nanmax(nanmax(v[k].x, v[k].y), nanmax(v[k].z, v[k].w)));  // twice changes no maximum
      }
    }
  }
}

// One workgroup per row: row sum (compensated FP32, rounded once), row max, and the FP64
// partial of the row for the total.
template <int kThreads, bool kShort>
__global__ __launch_bounds__(kThreads) void reduce_rows_kernel(const float *__restrict__ in, int64_t cols,
                                                               RowOutputs out) {
  const int64_t row = blockIdx.x;
  Acc a;
  float m = __builtin_nanf("");
  read_row<kThreads, kShort>(in + row * cols, cols, threadIdx.x, a, m);
  block_reduce<kThreads / 64>(a, m);
  if (threadIdx.x == 0) {
    if (out.row_sum) out.row_sum[row] = a.result();
    if (out.row_max) out.row_max[row] = m;
    if (out.partial64) out.partial64[row] = a.result64();
    else write_total(a.result64(), out.total, out.total64);
  }
}

// Short rows: kG lanes per row, kBlock / kG consecutive rows per workgroup at a time, so that a
// wave reads whole rows one after another; `tiles` such groups of rows per workgroup. The FP64
// values of its rows are added in a fixed order into one partial per workgroup. Bound by HBM once
// the grid fills the chip: 120011 x 77 (37 MB) takes 12.0 us with its combine, 3.1 TB/s, against
// 109 us when every row had a workgroup; 16000 x 1025 15.7 us (4.2 TB/s) against 25.2.
template <int kG, bool kShort>
__global__ __launch_bounds__(kBlock) void reduce_short_rows_kernel(const float *__restrict__ in, int64_t rows,
                                                                   int64_t cols, int tiles, RowOutputs out) {
  __shared__ double lw[kWaves];
  const int lane = threadIdx.x % kG, group = threadIdx.x / kG;
  double sum = 0.0;  // of this lane's rows
  for (int t = 0; t < tiles; ++t) {
    const int64_t row = (int64_t(blockIdx.x) * tiles + t) * (kBlock / kG) + group;
    Acc a;
    float m = __builtin_nanf("");
    if (row < rows) read_row<kG, kShort>(in + row * cols, static_cast<int>(cols), lane, a, m);
#pragma unroll
    for (int off = kG / 2; off >= 1; off >>= 1) {
      const float s2 = __shfl_xor(a.s, off, 64), c2 = __shfl_xor(a.c, off, 64), m2 = __shfl_xor(m, off, 64);
      a.merge(s2, c2);
      m = nanmax(m, m2);
    }
    if (lane == 0 && row < rows) {
      if (out.row_sum) out.row_sum[row] = a.result();
      if (out.row_max) out.row_max[row] = m;
      sum += a.result64();
    }
  }
  if (!out.partial64 && !out.total && !out.total64) return;
#pragma unroll
  for (int off = 32; off >= kG; off >>= 1) sum += __shfl_xor(sum, off, 64);  // lane 0 of each row group holds a value
  if ((threadIdx.x & 63) == 0) lw[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = lw[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) s += lw[w];
    if (out.partial64) out.partial64[blockIdx.x] = s;
    else write_total(s, out.total, out.total64);
  }
}

// ----------------------------------------------------------------------------- columns
// Column sums. A thread owns four adjacent columns (16-byte loads at any 4-byte boundary; the
// last four columns overlap the group before when cols % 4 != 0) and every `lanes`-th row of the
// workgroup's slice of rows: `across` threads side by side, kBlock / across row lanes, so that a
// workgroup reads whole rows of a narrow matrix. Eight rows of loads are in flight before the
// first addition. The row lanes meet in LDS in FP64, in order: one partial per column and slice
// (or, with one slice, the column's sum itself). Bound by HBM: 16384 x 4096 takes 45.7 us with its
// combine (5.9 TB/s), 20011 x 1003 19.0 us against 26.3 us with one column per thread and one
// thread per column in the combine, 524288 x 8 9.9 us against 169 us (a wave with two active
// lanes).
template <bool kFew>
__global__ __launch_bounds__(kBlock) void reduce_cols_kernel(const float *__restrict__ in, int64_t rows,
                                                             int64_t cols, int across, int64_t rows_per_slice,
                                                             double *partial64, float *col_sum) {
  __shared__ double part[kBlock * 4];
  const int lanes = kBlock / across;
  const int rl = threadIdx.x / across, cl = threadIdx.x % across;
  const int64_t first = (int64_t(blockIdx.x) * across + cl) * 4;  // of this thread's four columns
  const int64_t r0 = int64_t(blockIdx.y) * rows_per_slice;
  const int64_t r1 = r0 + rows_per_slice < rows ? r0 + rows_per_slice : rows;
  Acc a[4];
  if (rl < lanes && first < cols) {
    if (cols >= 4) {
      const int64_t c = first + 4 <= cols ? first : cols - 4;
      const int64_t step = int64_t(lanes) * cols;
      int64_t r = r0 + rl;
      const float *p = in + r * cols + c;
      for (; r + 7 * lanes < r1; r += 8 * lanes, p += 8 * step) {
        f4u v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = __builtin_nontemporal_load(reinterpret_cast<const f4u *>(p + k * step));
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          a[0].add(v[k].x);
          a[1].add(v[k].y);
          a[2].add(v[k].z);
          a[3].add(v[k].w);
        }
      }
      f4u v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (r + k * lanes < r1) v[k] = __builtin_nontemporal_load(reinterpret_cast<const f4u *>(p + k * step));
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (r + k * lanes < r1) {
          a[0].add(v[k].x);
          a[1].add(v[k].y);
          a[2].add(v[k].z);
          a[3].add(v[k].w);
        }
    } else {
      // the slice is one run of values: a thread takes every 256th (255th of three columns), all of one column
      // (5054 x 2 one row at a time 9.2 us)
      const int span = cols == 3 ? 255 : 256, mine = cols == 1 ? 0 : cols == 2 ? rl & 1 : rl % 3;
      const int64_t n = rl < span ? (r1 - r0) * cols : 0;
      const float *p = in + r0 * cols;
      Acc b;
      for (int64_t i = rl; i < n; i += 8 * span) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = i + k * span < n ? p[i + k * span] : 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) b.add(v[k]);
      }
#pragma unroll
      for (int k = 0; k < 3; ++k)
        if (mine == k) a[k] = b;
    }
  }
  if (rl < lanes) {
#pragma unroll
    for (int k = 0; k < 4; ++k) part[(rl * across + cl) * 4 + k] = a[k].result64();
  }
  __syncthreads();
  for (int t = threadIdx.x; t < across * 4; t += kBlock) {
    // column t of the workgroup's columns; in an overlapping group the column sits nearer to the
    // group's end
    const int64_t col = int64_t(blockIdx.x) * across * 4 + t;
    if (col < cols) {
      const int64_t group = col - t % 4;
      const int k = cols >= 4 && group + 4 > cols ? static_cast<int>(col - (cols - 4)) : t % 4;
      double s = part[(t / 4) * 4 + k];
      for (int l = 1; l < lanes; ++l) s += part[(l * across + t / 4) * 4 + k];
      if (col_sum) col_sum[col] = float(s);
      else partial64[int64_t(blockIdx.y) * cols + col] = s;
    }
    if (!kFew) break;  // at most 64 threads across
  }
}

// Adds each column's slices: `lanes` threads per column take every lanes-th slice in order, eight
// loads in flight, and meet in LDS in order.
__global__ __launch_bounds__(kBlock) void finish_cols_kernel(const double *__restrict__ partial64, int64_t cols,
                                                             int64_t slices, int lanes, float *col_sum) {
  __shared__ double part[kBlock];
  const int width = kBlock / lanes, cl = threadIdx.x % width, sl = threadIdx.x / width;
  const int64_t col = int64_t(blockIdx.x) * width + cl;
  double s = 0.0;
  if (col < cols) {
    const double *p = partial64 + int64_t(sl) * cols + col;
    const int64_t step = int64_t(lanes) * cols;
    int64_t y = sl;
    for (; y + 7 * lanes < slices; y += 8 * lanes, p += 8 * step) {
      double v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = p[k * step];
#pragma unroll
      for (int k = 0; k < 8; ++k) s += v[k];
    }
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = y + k * lanes < slices ? p[k * step] : 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (y + k * lanes < slices) s += v[k];
  }
  part[threadIdx.x] = s;
  __syncthreads();
  if (sl == 0 && col < cols) {
    for (int l = 1; l < lanes; ++l) s += part[l * width + cl];
    col_sum[col] = float(s);
  }
}

}  // namespace

// Per-stream scratch holding the FP64 (or FP32 max) partials.
struct ReduceScratch {
  double *partial64;
  float *partialmax;
};

}  // namespace csmi

using namespace csmi;

static ReduceScratch scratch_for(cs_stream *stream, size_t partial_doubles) {
  char *base = static_cast<char *>(stream_scratch(stream, partial_doubles * 8 + 4096));
  ReduceScratch r;
  r.partial64 = reinterpret_cast<double *>(base);
  r.partialmax = reinterpret_cast<float *>(base);
  return r;
}

namespace csmi {
double *sum_partials(cs_stream *stream, size_t n) { return scratch_for(stream, n).partial64; }

void launch_finish_sum(cs_stream *stream, const double *partials, int64_t n, float *out, double *out64) {
  hipLaunchKernelGGL(finish_sum_kernel, dim3(1), dim3(kFinish), 0, stream->stream, partials, n, out, out64);
}
}  // namespace csmi

// ----------------------------------------------------------------------------- no allocation
// cs_reduce_rows_noalloc keeps its row partials in this file-scope device array (one copy per
// GPU, held until the process ends). Host code reaches it only through the address
// hipGetSymbolAddress returns on each device.
constexpr int64_t kNoallocMaxRows = int64_t(1) << 20;
static __device__ __align__(256) double scratch[kNoallocMaxRows];

namespace {
std::mutex g_noalloc_mu;
std::map<int, double *> g_noalloc_scratch;  // device ordinal -> address of `scratch` there

// The device address of `scratch` on `device`, looked up once per device with that device
// current.
double *noalloc_scratch(cs_device *device) {
  std::lock_guard<std::mutex> l(g_noalloc_mu);
  auto it = g_noalloc_scratch.find(device->ordinal);
  if (it != g_noalloc_scratch.end()) return it->second;
  set_device(device);
  void *p = nullptr;
  CS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  if (!p) fail(CS_OUT_OF_RESOURCES, "no device address for the reduction scratch");
  g_noalloc_scratch[device->ordinal] = static_cast<double *>(p);
  return static_cast<double *>(p);
}
}  // namespace

namespace {
// How a [rows, cols] matrix is cut for the row kernels.
struct RowPlan {
  int lanes = 0;        // lanes per row of the short-row kernel; 0: a workgroup per row
  bool wide = false;    // with a workgroup per row: 1024 threads instead of 256
  int tiles = 1;        // groups of kBlock / lanes rows per workgroup
  int64_t grid = 0;     // workgroups, each with one FP64 partial
};

// Where the lines lie (whole calls with the total, in us: a workgroup per row against the rule):
//   * up to 2048 columns a row is 8 vectors per lane of one wave, so a workgroup per row spends
//     its time starting and combining: 120011 x 77 109.0 / 12.0, 524288 x 8 464 / 8.7,
//     60000 x 128 57.8 / 8.9, 16384 x 1024 19.5 / 14.3, 16000 x 1025 21.6 / 15.7; equal at
//     2047 columns (15.4 / 15.6); at 4096 the workgroup per row is ahead (43.3 / 45.8).
//   * few rows (at most 8 per CU, all resident at once) of more than 256 columns keep a workgroup
//     per row, since nothing else fills the chip: 2000 x 2000 7.5 / 7.2.
//   * as many lanes as take a row in at most four vectors each, all in flight together: half as
//     many (eight vectors) 14.1 at 120011 x 77 against 12.4, twice as many 15.5.
//     More where the rows leave the chip idle otherwise, down to one vector each.
//   * at most 8192 partials, which the combine adds in one round of loads.
//   * at most one row per CU and long rows: 1024 threads per row, since nothing else fills the
//     chip (64 x 65536 14.9 / 9.0, 256 x 16384 7.4 / 6.5); from two rows per CU on 256 threads
//     are ahead (512 x 16384 8.8 against 9.4, 2000 x 8192 13.4 against 16.9).
constexpr int64_t kShortCols = 2048, kMaxPartials = 8192, kWideCols = 8192, kFewRows = 8;

RowPlan plan_rows(cs_stream *stream, int64_t rows, int64_t cols) {
  RowPlan p;
  const int64_t cus = stream->device->props.multiProcessorCount;
  if (cols > kShortCols || (rows <= kFewRows * cus && cols > 256)) {
    p.grid = rows;
    p.wide = rows <= cus && cols >= kWideCols;
    return p;
  }
  p.lanes = 2;
  while (p.lanes < 64 && p.lanes * 16 < cols) p.lanes *= 2;
  while (p.lanes < 64 && p.lanes * 4 < cols && rows * p.lanes < 2 * cus * kBlock) p.lanes *= 2;
  const int64_t per = kBlock / p.lanes, groups = (rows + per - 1) / per;
  p.tiles = static_cast<int>((groups + kMaxPartials - 1) / kMaxPartials);
  p.grid = (groups + p.tiles - 1) / p.tiles;
  return p;
}

template <int kG, bool kShort>
void launch_short_rows(cs_stream *stream, const RowPlan &p, const float *in, int64_t rows, int64_t cols,
                       const RowOutputs &out) {
  hipLaunchKernelGGL((reduce_short_rows_kernel<kG, kShort>), dim3(static_cast<unsigned>(p.grid)), dim3(kBlock), 0,
                     stream->stream, in, rows, cols, p.tiles, out);
}

template <int kThreads, bool kShort>
void launch_long_rows(cs_stream *stream, const RowPlan &p, const float *in, int64_t cols,
                      const RowOutputs &out) {
  hipLaunchKernelGGL((reduce_rows_kernel<kThreads, kShort>), dim3(static_cast<unsigned>(p.grid)), dim3(kThreads), 0,
                     stream->stream, in, cols, out);
}

// The row pass of a plan and, where a total is wanted, the combine of its plan.grid partials (one workgroup
// writes the total itself).
void launch_rows(cs_stream *stream, const RowPlan &p, const float *in, int64_t rows, int64_t cols, float *row_sum,
                 float *row_max, double *partial64, float *total, double *total64) {
  const bool combine = (total || total64) && p.grid > 1;
  const RowOutputs out = combine ? RowOutputs{row_sum, row_max, partial64, nullptr, nullptr}
                                 : RowOutputs{row_sum, row_max, nullptr, total, total64};
#define CSMI_ROWS(kG) \
  (cols <= 4 * kG ? launch_short_rows<kG, true> : launch_short_rows<kG, false>)(stream, p, in, rows, cols, out)
  switch (p.lanes) {
    case 2: CSMI_ROWS(2); break;
    case 4: CSMI_ROWS(4); break;
    case 8: CSMI_ROWS(8); break;
    case 16: CSMI_ROWS(16); break;
    case 32: CSMI_ROWS(32); break;
    case 64: CSMI_ROWS(64); break;
    default:
      (p.wide                ? launch_long_rows<1024, false>
       : cols <= 4 * kBlock  ? launch_long_rows<kBlock, true>
                             : launch_long_rows<kBlock, false>)(stream, p, in, cols, out);
  }
#undef CSMI_ROWS
  if (combine) launch_finish_sum(stream, partial64, p.grid, total, total64);
}
}  // namespace

namespace {
// How a [rows, cols] matrix is cut for column sums.
struct ColPlan {
  int across = 1;          // threads side by side, four columns each
  int64_t groups = 1;      // workgroups side by side
  int64_t slices = 1, rows_per_slice = 1;
  int finish_lanes = 1;    // threads per column of the combine
};

// Where the lines lie (whole calls, in us):
//   * one workgroup per CU, never a few more: four waves of eight rows of loads keep the memory
//     busy, and each further slice adds partials to write and read (20011 x 1003: 19.0 with one,
//     19.5 with two, 20.3 with four per CU; 16384 x 4096: 45.8, 51.0, 55.8). Rounding the slices
//     up left a second round of a few workgroups (10000 x 3000: 31.2 against 25.6).
//   * at least eight rows per row lane (60000 x 128: 11.0; with 32 13.8).
//   * up to 32 rows per row lane in one slice, which needs no combine (116 x 2588: 4.2 against
//     6.8 with two launches); 128 leave one workgroup busy too long (1000 x 100: 13.3 against 6.7).
//   * 64 threads across, for whole rows of 1 KiB per wave, more where there are fewer rows than row
//     lanes (1 x 16000000: 27.3 against 72.8, 2 x 8000000 25.0 against 39.9); up to 1024 rows fewer, down to 16, as
//     long as that brings workgroups (300 x 16384: 6.1 against 7.9; 116 x 2588: 4.2 against 6.4).
//     Taller matrices lose by it (20011 x 1003: 22.8 against 19.0). Where that would leave a few CUs with two
//     workgroups, as many as the CUs' number needs (1022 x 19058: 19 across 17.8, 16 across 22.2).
//   * from half as many groups as CUs on, one slice leaves CUs idle, or a few with two workgroups: up to
//     eight slices there, as the estimate has it, by which 0.8 of the CUs fill the memory and a slice costs
//     3% (4000 x 33000, 129 groups: 1 slice 122.8, 2 110.6, 3 89.2, 4 106.6; 4000 x 44000, 172 groups: 125.6,
//     112.3, 127.7, 108.5; 2000 x 70000, 274 groups: 107.1, 105.8, 98.4, 95.5; 4000 x 60000, 235 groups: 137.1,
//     141.0, 145.0, 146.2).
constexpr int64_t kMinRowsPerLane = 8, kOneSliceRowsPerLane = 32, kNarrowRows = 1024;
constexpr int kMaxWideSlices = 8;

ColPlan plan_cols(cs_stream *stream, int64_t rows, int64_t cols) {
  ColPlan p;
  const int64_t cus = stream->device->props.multiProcessorCount;
  const int64_t quads = (cols + 3) / 4;
  int64_t most = 64;
  while (most * 2 * std::max<int64_t>(rows, 1) <= kBlock) most *= 2;
  if (rows <= kNarrowRows) {
    while (most > 16 && (quads + most - 1) / most < cus) most /= 2;
    if (most < 64 && quads > most * cus && quads * 5 < most * cus * 6) most = (quads + cus - 1) / cus;
  }
  p.groups = (quads + most - 1) / most;
  if (p.groups > 0x7fffffff) fail(CS_INVALID_VALUE, "too many columns");
  p.across = static_cast<int>((quads + p.groups - 1) / p.groups);
  const int64_t lanes = kBlock / p.across;
  // of fewer than four columns a thread has values, not rows: 64 each in one slice (8191 x 3 9.7 us cut, 11.0 whole)
  if (cols < 4 ? rows * cols > 2 * lanes * kOneSliceRowsPerLane : rows > lanes * kOneSliceRowsPerLane) {
    int64_t slices = cus / p.groups;
    if (slices <= 1 && rows > kNarrowRows) {
      // the time of s slices in rounds over all rows: what memory delivers, or the CU with most workgroups
      const double full = double(p.groups) / (0.8 * double(cus));
      double least = 1e30;
      for (int s = 1; s <= kMaxWideSlices; ++s) {
        const double t = std::max(full, double((p.groups * s + cus - 1) / cus) / s) + 0.03 * s;
        if (t < 0.95 * least) least = t, slices = s;
      }
    }
    slices = std::min(slices, rows / (lanes * kMinRowsPerLane));
    slices = std::max<int64_t>(1, std::min<int64_t>(slices, 65535));
    p.rows_per_slice = (rows + slices - 1) / slices;
    p.slices = (rows + p.rows_per_slice - 1) / p.rows_per_slice;
  } else {
    p.rows_per_slice = std::max<int64_t>(rows, 1);
  }
  while (p.finish_lanes < 32 && p.finish_lanes * 8 < p.slices) p.finish_lanes *= 2;
  return p;
}
}  // namespace

static int reduce_grid(cs_stream *stream, int64_t n) {
  int cus = stream->device->props.multiProcessorCount;
  int64_t want = (n / 4 + kBlock * 4 - 1) / (kBlock * 4);  // >= 4 vectors per thread
  int64_t cap = int64_t(cus) * 8;
  if (want > cap) want = cap;
  if (want < 1) want = 1;
  return static_cast<int>(want);
}

extern "C" {

cs_status cs_reduce_sum(cs_stream *stream, const float *in, int64_t n, float *out, double *out64) {
  return guard([&] {
    if (!stream) fail(CS_INVALID_VALUE, "stream is null");
    if (n < 0) fail(CS_INVALID_VALUE, "negative length");
    if (n > 0 && !in) fail(CS_INVALID_VALUE, "input is null");
    if (!out && !out64) fail(CS_INVALID_VALUE, "no output");
    set_device(stream->device);
    int grid = reduce_grid(stream, n);
    ReduceScratch s = scratch_for(stream, static_cast<size_t>(grid));
    hipLaunchKernelGGL(reduce_all_kernel<false>, dim3(grid), dim3(kBlock), 0, stream->stream, in, n,
                       s.partial64, s.partialmax, out, out64);
    if (grid > 1) launch_finish_sum(stream, s.partial64, grid, out, out64);
    CS_HIP(hipGetLastError());
  });
}

cs_status cs_reduce_max(cs_stream *stream, const float *in, int64_t n, float *out) {
  return guard([&] {
    if (!stream) fail(CS_INVALID_VALUE, "stream is null");
    if (n < 0) fail(CS_INVALID_VALUE, "negative length");
    if (n > 0 && !in) fail(CS_INVALID_VALUE, "input is null");
    if (!out) fail(CS_INVALID_VALUE, "output is null");
    set_device(stream->device);
    int grid = reduce_grid(stream, n);
    ReduceScratch s = scratch_for(stream, static_cast<size_t>(grid));
    hipLaunchKernelGGL(reduce_all_kernel<true>, dim3(grid), dim3(kBlock), 0, stream->stream, in, n,
                       s.partial64, s.partialmax, out, static_cast<double *>(nullptr));
    if (grid > 1)
      hipLaunchKernelGGL(finish_max_kernel, dim3(1), dim3(kFinish), 0, stream->stream, s.partialmax,
                         int64_t(grid), out);
    CS_HIP(hipGetLastError());
  });
}

cs_status cs_reduce_rows(cs_stream *stream, const float *in, int64_t rows, int64_t cols, float *row_sum,
                         float *row_max, float *total, double *total64) {
  return guard([&] {
    if (!stream) fail(CS_INVALID_VALUE, "stream is null");
    if (rows < 0 || cols < 0) fail(CS_INVALID_VALUE, "negative shape");
    if (rows > 0x7fffffff) fail(CS_INVALID_VALUE, "more than 2^31-1 rows");
    if (rows > 0 && cols > 0 && !in) fail(CS_INVALID_VALUE, "input is null");
    set_device(stream->device);
    bool want_total = total || total64;
    if (rows == 0) {
      // no rows: the total is an empty sum, written by the combine over zero partials
      if (want_total)
        hipLaunchKernelGGL(finish_sum_kernel, dim3(1), dim3(kFinish), 0, stream->stream, nullptr, int64_t(0), total,
                           total64);
      CS_HIP(hipGetLastError());
      return;
    }
    const RowPlan plan = plan_rows(stream, rows, cols);
    // sized for calls of up to as many rows under capture, which may have a partial per row
    if (want_total) reserve_scratch(stream, static_cast<size_t>(rows) * 8 + 4096);
    ReduceScratch s = scratch_for(stream, want_total ? static_cast<size_t>(plan.grid) : 0);
    launch_rows(stream, plan, in, rows, cols, row_sum, row_max, s.partial64, total, total64);
    CS_HIP(hipGetLastError());
  });
}

cs_status cs_reduce_rows_noalloc(cs_stream *stream, const float *in, int64_t rows, int64_t cols, float *row_sum,
                                 float *row_max, float *total, double *total64) {
  return guard([&] {
    if (!stream) fail(CS_INVALID_VALUE, "stream is null");
    if (rows < 0 || cols < 0) fail(CS_INVALID_VALUE, "negative shape");
    if (rows > 0x7fffffff) fail(CS_INVALID_VALUE, "more than 2^31-1 rows");
    if (rows > 0 && cols > 0 && !in) fail(CS_INVALID_VALUE, "input is null");
    const bool want_total = total || total64;
    if (want_total && rows > kNoallocMaxRows)
      fail(CS_INVALID_BUFFER_SIZE, "cs_reduce_rows_noalloc takes at most " + std::to_string(kNoallocMaxRows) +
                                       " rows when a total is asked for, got " + std::to_string(rows));
    set_device(stream->device);
    if (rows == 0) {
      // no rows: the total is an empty sum, written by the combine over zero partials
      if (want_total)
        hipLaunchKernelGGL(finish_sum_kernel, dim3(1), dim3(kFinish), 0, stream->stream, nullptr, int64_t(0), total,
                           total64);
      CS_HIP(hipGetLastError());
      return;
    }
    // every partial the combine reads is written by this call's row kernel first
    double *partial64 = want_total ? noalloc_scratch(stream->device) : nullptr;
    launch_rows(stream, plan_rows(stream, rows, cols), in, rows, cols, row_sum, row_max, partial64, total, total64);
    CS_HIP(hipGetLastError());
  });
}

cs_status cs_reduce_cols(cs_stream *stream, const float *in, int64_t rows, int64_t cols, float *col_sum) {
  return guard([&] {
    if (!stream) fail(CS_INVALID_VALUE, "stream is null");
    if (rows < 0 || cols < 0) fail(CS_INVALID_VALUE, "negative shape");
    if (cols == 0) return;
    if (!col_sum || (rows > 0 && !in)) fail(CS_INVALID_VALUE, "null pointer");
    set_device(stream->device);
    const ColPlan p = plan_cols(stream, rows, cols);
    const dim3 grid(static_cast<unsigned>(p.groups), static_cast<unsigned>(p.slices));
    // sized for smaller calls under capture as well: only matrices of up to two groups per CU are cut into
    // slices that take more than the least scratch
    const int64_t widest = rows > kNarrowRows ? std::min<int64_t>(cols, 512 * stream->device->props.multiProcessorCount) : 0;
    reserve_scratch(stream, static_cast<size_t>(widest * kMaxWideSlices * 8 + 4096));
    if (p.slices == 1) {
      hipLaunchKernelGGL((p.across > 64 ? reduce_cols_kernel<true> : reduce_cols_kernel<false>), grid, dim3(kBlock), 0,
                         stream->stream, in, rows, cols, p.across, p.rows_per_slice, static_cast<double *>(nullptr),
                         col_sum);
    } else {
      ReduceScratch s = scratch_for(stream, static_cast<size_t>(p.slices * cols));
      hipLaunchKernelGGL(reduce_cols_kernel<false>, grid, dim3(kBlock), 0, stream->stream, in, rows, cols, p.across,
                         p.rows_per_slice, s.partial64, static_cast<float *>(nullptr));
      const int64_t width = kBlock / p.finish_lanes;
      hipLaunchKernelGGL(finish_cols_kernel, dim3(static_cast<unsigned>((cols + width - 1) / width)), dim3(kBlock), 0,
                         stream->stream, s.partial64, cols, p.slices, p.finish_lanes, col_sum);
    }
    CS_HIP(hipGetLastError());
  });
}

}  // extern "C"
