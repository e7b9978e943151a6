// Random number kernels: the reference's Wang-hash `random` and Box-Muller `randomNormal`
// (Tensors.scala:106-117, 397-443), plus FP64-exact synthetic-input generators on the same
// hash.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "internal.h"

#pragma clang fp contract(off)

namespace csmi {
namespace {

// Thomas Wang's 32-bit integer hash, in the variant the reference emits
// (Tensors.scala:107-115).
__device__ __forceinline__ uint32_t wang_hash(uint32_t v) {
  v = (v ^ 61u) ^ (v >> 16);
  v *= 9u;
  v ^= v << 4;
  v *= 0x27d4eb2du;
  v ^= v >> 15;
  return v;
}

// Marsaglia xorshift step used by random_normal (Tensors.scala:403-407).
__device__ __forceinline__ uint32_t xorshift32(uint32_t s) {
  uint32_t t1 = s ^ (s << 13);
  uint32_t t2 = t1 ^ (t1 >> 17);
  return t2 ^ (t2 << 5);
}

constexpr int kBlock = 256;

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// buffer[i] = hash(i ^ seed) / 2^32, converted to float then scaled (Tensors.scala:436-439); four
// consecutive elements per thread, one 16-byte store (16777259 values: 11.7 us against 18.2 us with
// one element per thread).
__global__ __launch_bounds__(kBlock) void random_kernel(float *out, int64_t n, uint32_t seed) {
  const int64_t i = (int64_t(blockIdx.x) * kBlock + threadIdx.x) * 4;
  if (i >= n) return;
  f4u v;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    v[k] = static_cast<float>(wang_hash(static_cast<uint32_t>(i + k) ^ seed)) / 4294967296.0f;
  if (i + 4 <= n) {
    *reinterpret_cast<f4u *>(out + i) = v;
  } else {
    for (int k = 0; k < n - i; ++k) out[i + k] = v[k];
  }
}

// Tables of the normal generator, one copy per workgroup in LDS.
constexpr int kLogIntervals = 128, kSectors = 64;
struct NormalTables {
  struct {
    double inv, ln;  // 1 / c, ln c
  } log[kLogIntervals];
  struct {
    double sin, cos;  // of k 2 pi / kSectors
  } turn[kSectors + 1];
};

__device__ __forceinline__ void fill_tables(NormalTables &t) {
  for (int k = threadIdx.x; k < kLogIntervals; k += kBlock) {
    const double c = k + 1 == kLogIntervals ? 1.0 : 0.5 + (k + 0.5) / 256.0;
    t.log[k] = {1.0 / c, log(c)};
  }
  for (int k = threadIdx.x; k <= kSectors; k += kBlock) {
    double sine, cosine;
    sincospi(k * (2.0 / kSectors), &sine, &cosine);  // exact at the quarters
    t.turn[k] = {sine, cosine};
  }
  __syncthreads();
}

// ln(f 2^-32) in FP64 for f = 0 or a single-precision f in [1, 2^32], by Tang's table-driven method
// (ACM TOMS 16(4), 1990): f = m 2^e with m in [1/2, 1), c the middle of m's interval of width 2^-8
// (1 for the last one, so that the result keeps its relative accuracy just below 2^32), z = m / c - 1
// and ln(f 2^-32) = (e - 32) ln 2 + ln c + ln(1 + z). |z| <= 2^-8, so the series to z^7 is within
// 2^-58 of |z|.
__device__ __forceinline__ double log_unit(float f, const NormalTables &tables) {
  const float m = __builtin_amdgcn_frexp_mantf(f);
  const int e = __builtin_amdgcn_frexp_expf(f) - 32;
  const auto t = tables.log[(__float_as_uint(m) >> 16) & (kLogIntervals - 1)];
  const double z = fma(static_cast<double>(m), t.inv, -1.0);
  double p = fma(z, 1.0 / 7.0, -1.0 / 6.0);
  p = fma(p, z, 1.0 / 5.0);
  p = fma(p, z, -1.0 / 4.0);
  p = fma(p, z, 1.0 / 3.0);
  p = fma(p, z, -1.0 / 2.0);
  p = fma(p * z, z, z);
  p += fma(static_cast<double>(e), 0.69314718055994530942, t.ln);
  return f < 4294967296.0f ? p : 0.0;
}

// sin and cos in FP64 of a single-precision theta in [0, 2 pi], each rounded once to FP32: theta is
// n 2 pi / 64 + y (2 pi / 64 as a 33-bit part, whose multiples are exact, and the rest), |y| <= pi / 64,
// and the Taylor series of y turn the table's values for n. The first terms left out are below 2^-57.
__device__ __forceinline__ void sincos_turn(float theta, const NormalTables &tables, float &sine, float &cosine) {
  const float n = rintf(theta * float(kSectors / 6.28318530717958647693));
  const double nd = static_cast<double>(n);
  const auto t = tables.turn[static_cast<int>(n)];
  double y = fma(nd, -0x1.921fb544p-4, static_cast<double>(theta));
  y = fma(nd, -0x1.0b4611a626331p-38, y);
  const double y2 = y * y;
  double s = fma(y2, -1.0 / 5040.0, 1.0 / 120.0);
  s = fma(s, y2, -1.0 / 6.0);
  s = fma(s * y2, y, y);
  double c = fma(y2, 1.0 / 40320.0, -1.0 / 720.0);
  c = fma(c, y2, 1.0 / 24.0);
  c = fma(c, y2, -1.0 / 2.0);
  c *= y2;  // cos y - 1
  sine = static_cast<float>(fma(t.cos, s, fma(t.sin, c, t.sin)));
  cosine = static_cast<float>(fma(-t.sin, s, fma(t.cos, c, t.cos)));
}

// Pair i writes buffer[2i], buffer[2i+1] (Tensors.scala:409-425). Every FP32 operation is
// correctly rounded: log, cos and sin are evaluated in FP64 and rounded once, as a correctly
// rounded libm does on the host. Two pairs per thread and step, one 16-byte store. Bound by
// arithmetic, a third of it FP64: 16777259 values (67 MB) take 25.0 us, against 58.4 us with the
// device library's log, cos and sin, which serve the whole range of their arguments. (One copy of the
// tables per LDS lane, against bank conflicts, took 32.5 us: filling them costs more than it saves.)
__global__ __launch_bounds__(kBlock) void random_normal_kernel(float *out, int64_t pairs, uint32_t seed,
                                                                int64_t stride) {
  __shared__ NormalTables tables;
  fill_tables(tables);
  for (int64_t i = (int64_t(blockIdx.x) * kBlock + threadIdx.x) * 2; i < pairs; i += stride) {
    f4u v;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t r1 = wang_hash(static_cast<uint32_t>(i + k) ^ seed);
      const uint32_t r2 = xorshift32(r1);
      // the uniform draws are these over 2^32; the scaling is exact, so it is left to what follows
      const float f1 = static_cast<float>(r1), f2 = static_cast<float>(r2);
      const float ln = f1 > 0.0f ? static_cast<float>(log_unit(f1, tables)) : -__builtin_huge_valf();
      const float r = sqrtf(-2.0f * ln);
      float sine, cosine;
      sincos_turn(2.0f * 3.14159274101257324219f / 4294967296.0f * f2, tables, sine, cosine);
      v[2 * k] = r * cosine;
      v[2 * k + 1] = r * sine;
    }
    if (i + 2 <= pairs) {
      *reinterpret_cast<f4u *>(out + 2 * i) = v;
    } else {
      out[2 * i] = v[0];
      out[2 * i + 1] = v[1];
    }
  }
}

// Synthetic inputs: u = hash(i ^ seed) / 2^32 exactly in FP64; x = lo + (hi - lo) * u,
// rounded once to FP32.
__global__ __launch_bounds__(kBlock) void fill_uniform_kernel(float *out, int64_t n, uint32_t seed,
                                                              double lo, double hi) {
  int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  double u = static_cast<double>(wang_hash(static_cast<uint32_t>(i) ^ seed)) * (1.0 / 4294967296.0);
  double w = hi - lo;
  double t = w * u;
  out[i] = static_cast<float>(lo + t);
}

// N(0,1): u1 = (hash + 1) / 2^32 in (0, 1], u2 = xorshift(hash) / 2^32;
// z = sqrt(-2 ln u1) * cos(2 pi u2) in FP64, rounded once to FP32.
__global__ __launch_bounds__(kBlock) void fill_normal_kernel(float *out, int64_t n, uint32_t seed) {
  int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  uint32_t h = wang_hash(static_cast<uint32_t>(i) ^ seed);
  double u1 = (static_cast<double>(h) + 1.0) * (1.0 / 4294967296.0);
  double u2 = static_cast<double>(xorshift32(h)) * (1.0 / 4294967296.0);
  double r = sqrt(-2.0 * log(u1));
  double th = 6.283185307179586 * u2;
  out[i] = static_cast<float>(r * cos(th));
}

unsigned blocks_for(int64_t n) { return static_cast<unsigned>((n + kBlock - 1) / kBlock); }

}  // namespace
}  // namespace csmi

using namespace csmi;

extern "C" {

cs_status cs_random(cs_stream *stream, float *out, int64_t n, uint32_t seed) {
  return guard([&] {
    if (!stream) fail(CS_INVALID_VALUE, "stream is null");
    if (n < 0 || n > 0xffffffffll) fail(CS_INVALID_VALUE, "length out of range");
    if (n == 0) return;
    if (!out) fail(CS_INVALID_VALUE, "out is null");
    set_device(stream->device);
    hipLaunchKernelGGL(random_kernel, dim3(blocks_for((n + 3) / 4)), dim3(kBlock), 0, stream->stream, out, n, seed);
    CS_HIP(hipGetLastError());
  });
}

cs_status cs_random_normal(cs_stream *stream, float *out, int64_t n, uint32_t seed) {
  return guard([&] {
    if (!stream) fail(CS_INVALID_VALUE, "stream is null");
    if (n < 0 || n > 0xffffffffll) fail(CS_INVALID_VALUE, "length out of range");
    if (n == 0) return;
    if (!out) fail(CS_INVALID_VALUE, "out is null");
    set_device(stream->device);
    int64_t pairs = (n + 1) / 2;
    // workgroups to fill every CU, each with pairs enough to pay for its table
    const unsigned grid = std::min<unsigned>(blocks_for((pairs + 1) / 2), 8 * stream->device->props.multiProcessorCount);
    hipLaunchKernelGGL(random_normal_kernel, dim3(grid), dim3(kBlock), 0, stream->stream, out,
                       pairs, seed, int64_t(grid) * kBlock * 2);
    CS_HIP(hipGetLastError());
  });
}

cs_status cs_fill_uniform(cs_stream *stream, float *out, int64_t n, uint32_t seed, double lo, double hi) {
  return guard([&] {
    if (!stream) fail(CS_INVALID_VALUE, "stream is null");
    if (n < 0 || n > 0xffffffffll) fail(CS_INVALID_VALUE, "length out of range");
    if (n == 0) return;
    if (!out) fail(CS_INVALID_VALUE, "out is null");
    set_device(stream->device);
    hipLaunchKernelGGL(fill_uniform_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, stream->stream, out, n, seed,
                       lo, hi);
    CS_HIP(hipGetLastError());
  });
}

cs_status cs_fill_normal(cs_stream *stream, float *out, int64_t n, uint32_t seed) {
  return guard([&] {
    if (!stream) fail(CS_INVALID_VALUE, "stream is null");
    if (n < 0 || n > 0xffffffffll) fail(CS_INVALID_VALUE, "length out of range");
    if (n == 0) return;
    if (!out) fail(CS_INVALID_VALUE, "out is null");
    set_device(stream->device);
    hipLaunchKernelGGL(fill_normal_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, stream->stream, out, n, seed);
    CS_HIP(hipGetLastError());
  });
}

}  // extern "C"
