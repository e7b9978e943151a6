// A small fully connected network (the cost model's predictor), trained and evaluated on
// the device: forward, mean-squared-error gradient, backward and Adam, all in FP32.
//
// The reference has no counterpart (it has no tuning). Layout: parameters are one flat
// FP32 array [W1 (d0 x d1), b1 (d1), W2 (d1 x d2), b2, ...]; W is row-major [in][out]; ReLU
// follows every layer but the last. Every sum has a fixed order, so results are
// deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <utility>
#include <vector>

#include "internal.h"

struct cs_mlp {
  cs_device *device = nullptr;
  std::vector<int> widths;
  std::vector<int64_t> w_off, b_off;  // offsets of each layer's W and b in the flat arrays
  int64_t count = 0;
  float *params = nullptr, *m = nullptr, *v = nullptr;
  float *acts = nullptr;  // activations of every layer for the last forward pass
  int64_t acts_capacity = 0;
  float *deltas = nullptr;  // two ping-pong gradient buffers of n x max width
  int64_t deltas_capacity = 0;
  std::vector<float *> retired;  // workspaces outgrown under capture
};

namespace csmi {
namespace {

constexpr int kB = 256;

__global__ __launch_bounds__(kB) void linear_fwd(const float *__restrict__ X, int64_t n, int din,
                                                 const float *__restrict__ W, const float *__restrict__ b, int dout,
                                                 int relu, float *__restrict__ Y) {
  int64_t t = int64_t(blockIdx.x) * kB + threadIdx.x;
  if (t >= n * dout) return;
  int64_t s = t / dout;
  int j = static_cast<int>(t % dout);
  const float *x = X + s * din;
  float acc = b[j];
  for (int i = 0; i < din; ++i) acc = fmaf(x[i], W[int64_t(i) * dout + j], acc);
  Y[t] = relu ? fmaxf(acc, 0.0f) : acc;
}

// dpred = 2 (pred - target) / n; loss = sum (pred - target)^2 / n (one workgroup, fixed order).
__global__ __launch_bounds__(1024) void mse_grad(const float *__restrict__ pred, const float *__restrict__ target,
                                                 int64_t n, float *__restrict__ dpred, float *loss) {
  __shared__ double part[1024];
  double acc = 0.0;
  for (int64_t s = threadIdx.x; s < n; s += 1024) {
    float d = pred[s] - target[s];
    dpred[s] = 2.0f * d / float(n);
    acc += double(d) * double(d);
  }
  part[threadIdx.x] = acc;
  __syncthreads();
  for (int off = 512; off > 0; off >>= 1) {
    if (int(threadIdx.x) < off) part[threadIdx.x] += part[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0 && loss) *loss = float(part[0] / double(n));
}

// g = dY * relu'(Y) is formed on the fly. dX[s][i] = sum_j g[s][j] W[i][j].
__global__ __launch_bounds__(kB) void linear_bwd_dx(const float *__restrict__ dY, const float *__restrict__ Y,
                                                    int relu, const float *__restrict__ W, int64_t n, int din,
                                                    int dout, float *__restrict__ dX) {
  int64_t t = int64_t(blockIdx.x) * kB + threadIdx.x;
  if (t >= n * din) return;
  int64_t s = t / din;
  int i = static_cast<int>(t % din);
  float acc = 0.0f;
  for (int j = 0; j < dout; ++j) {
    float g = dY[s * dout + j];
    if (relu && Y[s * dout + j] <= 0.0f) g = 0.0f;
    acc = fmaf(g, W[int64_t(i) * dout + j], acc);
  }
  dX[t] = acc;
}

// dW[i][j] = sum_s X[s][i] g[s][j] for i < din; row i == din holds db[j] = sum_s g[s][j].
__global__ __launch_bounds__(kB) void linear_bwd_dw(const float *__restrict__ X, const float *__restrict__ dY,
                                                    const float *__restrict__ Y, int relu, int64_t n, int din,
                                                    int dout, float *__restrict__ dW, float *__restrict__ db) {
  int64_t t = int64_t(blockIdx.x) * kB + threadIdx.x;
  if (t >= int64_t(din + 1) * dout) return;
  int i = static_cast<int>(t / dout), j = static_cast<int>(t % dout);
  float acc = 0.0f;
  for (int64_t s = 0; s < n; ++s) {
    float g = dY[s * dout + j];
    if (relu && Y[s * dout + j] <= 0.0f) g = 0.0f;
    acc = fmaf(i < din ? X[s * din + i] : 1.0f, g, acc);
  }
  if (i < din) dW[int64_t(i) * dout + j] = acc;
  else db[j] = acc;
}

__global__ __launch_bounds__(kB) void adam_kernel(float *__restrict__ p, const float *__restrict__ g,
                                                  float *__restrict__ m, float *__restrict__ v, int64_t count,
                                                  float lr, float b1, float b2, float eps, float c1, float c2) {
  int64_t t = int64_t(blockIdx.x) * kB + threadIdx.x;
  if (t >= count) return;
  float gi = g[t];
  float mi = b1 * m[t] + (1.0f - b1) * gi;
  float vi = b2 * v[t] + (1.0f - b2) * gi * gi;
  m[t] = mi;
  v[t] = vi;
  p[t] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ------------------------------------------------------------------------ whole network
// Networks whose layers fit LDS run in one kernel: a workgroup takes kSamples samples through
// every layer, forward and back, with the activations and deltas in LDS, so that nothing but the
// inputs, the parameters and the gradients' partial sums crosses memory. With the gradient, each
// workgroup adds its samples' share of every parameter's gradient into its own row of `partial`,
// and reduce_grads_kernel adds the rows.
//
// All three products run on the FP32 matrix instructions of K = 1, each a fused multiply-add per
// element, so a sum keeps the order of its chain of them: the forward sums that of linear_fwd (bias
// first, inputs in order), so activations are the same bits on either path. The 4x4x1 form, whose 16
// blocks take one block's rows, multiplies four samples by 64 units, with the weights read from LDS
// once for four samples and 16 inputs of the samples in one register; with a thread per sum each
// multiply-add read its weight and its input, and LDS was the bound. The 16x16x1 form adds the outer
// products of the weights' gradient, 16 inputs by 64 units. Bound by latency, that of the chain of layers
// in one workgroup (18 cycles for each of a sum's terms), of the first loads and of fetching its
// instructions, for which the loops are short (29 KiB unrolled 22.8 us, 10 KiB 17.5, at 512 samples of
// 23-64-64-64-1; with a thread per sum 19.7). A gradient of 92 samples of 14-99-99-99-1 22.0 us (with a
// thread per sum 37.7), of 512 of 32-128-128-128-1 38.8 (42.4); 512 samples of 23-64-64-64-1 took 820 us
// in twelve launches with one thread per weight summing over all samples.
// Eight samples and 512 threads a workgroup: four samples double the rows to add.
// Evaluation of more than kManySamples takes four times as many, so that every wave has units of its own
// (262144 samples of 23-64-64-64-1 191 us, with eight 406; at 4096 11.9 and 11.8, below eight are ahead).
constexpr int kSamples = 8;  // per workgroup
constexpr int kManySamples = 4096;
constexpr int kNet = 512;      // threads of its kernel
constexpr int kNetWaves = kNet / 64;
constexpr int kMaxLayers = 15;

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16 __attribute__((ext_vector_type(16)));

// A layer: its widths, its parameters (W, then b) in the flat array and in LDS, and the LDS offsets of
// its input and output activations.
struct NetLayer {
  int din, dout, params, lds, in, out, unused[2];
};
struct NetShape {
  int layers;  // L
  int count;   // parameters
  int unit_floats, delta_floats, weight_floats;  // LDS floats of all activations, one delta buffer, parameters
  int resident;  // all parameters stay in LDS, else one layer's at a time
  NetLayer layer[kMaxLayers];
};

// In LDS widths are padded with zeros to a multiple of 16, the steps of sum_units. Rows of weights are an
// odd number of 16-byte pieces: 64 consecutive floats of a row, and pieces of 16 rows, lie in different banks.
__host__ __device__ __forceinline__ int padded(int width) { return (width + 15) & ~15; }
__host__ __device__ __forceinline__ int pitch(int width) { return padded(width) + 4; }

// Copies the parameters of layers from .. to (any 4-byte boundary) to LDS, that of layer l to dst + its lds:
// the bias first, then W. The waves take 1024 floats each in turn, through the layers.
__device__ __forceinline__ void copy_to_lds(float *dst, const float *__restrict__ params, const NetShape &net,
                                            int from, int to, int wave, int lane) {
  typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
  int mine = wave;  // chunks until this wave's next one
#pragma unroll 1
  for (int l = from; l <= to; ++l) {
    const NetLayer y = net.layer[l - 1];
    const int width = y.dout, n = y.din * width, chunks = (n + 1023) / 1024, row = pitch(width);
    const float *const src = params + y.params;
    float *const out = dst + y.lds;
    const float inverse = 1.0f / float(width);
    // (e + 0.5) / width is at least 0.5 / width from a whole number, and e < 2^16
    auto at = [&](int e) {
      const int r = int((float(e) + 0.5f) * inverse);
      return e + (r + 1) * row - r * width;
    };
    if (mine == 0) {
      for (int j = lane; j < width; j += 64) out[j] = src[n + j];
      if (n < 4 && lane < n) out[at(lane)] = src[lane];
    }
#pragma unroll 1
    for (; n >= 4 && mine < chunks; mine += kNetWaves) {  // the last vector overlaps the one before
      const int e0 = mine * 1024 + 4 * lane;
      f4u v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const f4u *>(src + min(e0 + 256 * k, n - 4));
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int e = min(e0 + 256 * k, n - 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) out[at(e + i)] = v[k][i];
      }
    }
    mine = (mine - chunks) & (kNetWaves - 1);
  }
}

// acc[r] += x[k][r] w[k] for 16 units k in order: a holds unit k of sample r in lane 4 k + r.
template <int... I>
__device__ __forceinline__ void chain(float a, const float (&w)[16], f4 &acc, std::integer_sequence<int, I...>) {
  ((acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a, w[I], acc, 4, I, 0)), ...);
}

// acc[r] + sum_k x[k][r] v[k], k = 0 .. n - 1 in order, for four samples r and each lane's v: consecutive
// values (kRow, 16-byte aligned) or values `stride` apart. x: the samples' values by unit, kS apart.
// Both are zeros from n to the next multiple of 16.
template <bool kRow, int kS>
__device__ __forceinline__ f4 sum_units(const float *x, const float *v, int stride, int n, f4 acc) {
  const int lane = threadIdx.x & 63;
  const float *p = x + (lane >> 2) * kS + (lane & 3);
#pragma unroll 1
  for (int k0 = 0; k0 < n; k0 += 16) {
    const float a = p[k0 * kS];
    float w[16];
    if constexpr (kRow) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const f4 q = reinterpret_cast<const f4 *>(v + k0)[k];
#pragma unroll
        for (int e = 0; e < 4; ++e) w[4 * k + e] = q[e];
      }
    } else {
#pragma unroll
      for (int k = 0; k < 16; ++k) w[k] = v[k * stride];
      v += 16 * stride;
    }
    chain(a, w, acc, std::make_integer_sequence<int, 16>());
  }
  return acc;
}

// LDS: activations [layer][unit][sample], two delta buffers [unit][sample], parameters by layer: the bias,
// then W's rows.
template <bool kGrad, int kS>
__global__ __launch_bounds__(kNet) void network_kernel(NetShape net, const float *__restrict__ params,
                                                       const float *__restrict__ X, const float *__restrict__ target,
                                                       int64_t n, float *__restrict__ result,
                                                       float *__restrict__ partial, double *__restrict__ partial_loss) {
  static_assert(!kGrad || kS == 8, "the weights' gradient adds two registers of four samples");
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float *const units = lds, *const deltas = units + net.unit_floats, *const weights = deltas + 2 * net.delta_floats;
  const int t = threadIdx.x, L = net.layers;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const int last = net.layer[L - 1].dout, din0 = net.layer[0].din;
  // In sums over units a wave takes four samples and 64 units, then the next units that no wave has taken.
  constexpr int kQuads = kS / 4, kStep = kNetWaves / kQuads * 64;
  const int q = wave % kQuads * 4, first_unit = wave / kQuads * 64 + lane;
  // Layer l's parameters in LDS, for every thread of the workgroup.
  auto layer_weights = [&](int l, const NetLayer &layer) -> const float * {
    if (net.resident) return weights + layer.lds;
    __syncthreads();  // the previous layer's are no longer read
    for (int i = t * 4; i < net.weight_floats; i += kNet * 4) *reinterpret_cast<f4 *>(weights + i) = f4{};
    __syncthreads();
    copy_to_lds(weights - layer.lds, params, net, l, l, wave, lane);
    return weights;
  };
  for (int i = t * 4; i < net.unit_floats + 2 * net.delta_floats + net.weight_floats; i += kNet * 4)
    *reinterpret_cast<f4 *>(lds + i) = f4{};
  __syncthreads();
  double loss = 0.0;
  bool first = true;
#pragma unroll 1
  for (int64_t s0 = int64_t(blockIdx.x) * kS; s0 < n; s0 += int64_t(gridDim.x) * kS, first = false) {
    const int live = n - s0 < kS ? static_cast<int>(n - s0) : kS;  // samples past n are zeros
    const float wanted = kGrad && t < live ? target[s0 + t] : 0.0f;
    if (!first) __syncthreads();  // the activations of the samples before are no longer read
    for (int s = wave; s < kS; s += kNetWaves)
      for (int c = lane; c < din0; c += 64) units[c * kS + s] = s < live ? X[(s0 + s) * din0 + c] : 0.0f;
    if (first && net.resident) copy_to_lds(weights, params, net, 1, L, wave, lane);
    NetLayer y = net.layer[0];
#pragma unroll 1
    for (int l = 1; l <= L; ++l) {
      const NetLayer following = net.layer[l < L ? l : L - 1];  // read while this layer runs
      const float *const w = layer_weights(l, y);
      __syncthreads();
#pragma unroll 1
      for (int j = first_unit; j - lane < y.dout; j += kStep) {
        const float *const wj = w + min(j, y.dout - 1);
        const float b = wj[0];
        f4 acc = sum_units<false, kS>(units + y.in + q, wj + pitch(y.dout), pitch(y.dout), y.din, f4{b, b, b, b});
        if (l < L)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[e] = fmaxf(acc[e], 0.0f);
        if (j < y.dout) *reinterpret_cast<f4 *>(units + y.out + j * kS + q) = acc;
      }
      y = following;
    }
    __syncthreads();
    const float *const pred = units + y.out;
    if constexpr (!kGrad) {
      for (int s = wave; s < live; s += kNetWaves)
        for (int c = lane; c < last; c += 64) result[(s0 + s) * last + c] = pred[c * kS + s];
    } else {
      // samples past n add nothing, whatever infinite parameters have made of their zeros
      if (live < kS)
        for (int i = t; i < net.unit_floats; i += kNet)
          if (i % kS >= live) units[i] = 0.0f;
      // delta[j][s]: the loss's gradient by layer l's output before its ReLU
      float *cur = deltas, *next = deltas + net.delta_floats;
      if (t < 16 * kS) {
        const float d = t < live ? pred[t] - wanted : 0.0f;
        cur[t] = 2.0f * d / float(n);
        loss += double(d) * double(d);
      }
#pragma unroll 1
      for (int l = L; l >= 1; --l) {
        const NetLayer following = net.layer[l > 1 ? l - 2 : 0];
        const int din = y.din, dout = y.dout;
        const float *const in = units + y.in;
        const float *const w = l > 1 ? layer_weights(l, y) : nullptr;
        __syncthreads();
        // dX[s][i] = sum_j delta[s][j] W[i][j], then the ReLU of layer l - 1: 64 inputs at a time
        if (l > 1)
#pragma unroll 1
          for (int i = first_unit; i - lane < din; i += kStep) {
            f4 acc = sum_units<true, kS>(cur + q, w + (min(i, din - 1) + 1) * pitch(dout), 1, dout, f4{});
            const f4 x = *reinterpret_cast<const f4 *>(in + min(i, din - 1) * kS + q);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = x[e] <= 0.0f || i >= din ? 0.0f : acc[e];
            if (i < padded(din)) *reinterpret_cast<f4 *>(next + i * kS + q) = acc;
          }
        // dW[i][j] = sum_s in[s][i] delta[s][j]; row din is the bias's, whose input is 1. 16 inputs and 64
        // units at a time, from the first wave without a sum above on. Inputs and units past the end have
        // results of their own, which lie out of the buffer's range.
        const __amdgpu_buffer_rsrc_t row = __builtin_amdgcn_make_buffer_rsrc(
            partial + int64_t(blockIdx.x) * net.count + y.params, 0, (din + 1) * dout * 4, 0x00020000);
        const int l16 = lane & 15, quad = lane >> 4, busy = l > 1 ? (din + 63) / 64 * kQuads : 0;
#pragma unroll 1
        for (int i0 = ((wave - busy) & (kNetWaves - 1)) * 16; i0 <= din; i0 += kNetWaves * 16) {
          const int i = i0 + l16;
          const float *const x = in + min(i, din - 1) * kS + quad;
          const float a0 = i < din ? x[0] : 1.0f, a1 = i < din ? x[4] : 1.0f;
#pragma unroll 1
          for (int j0 = 0; j0 < dout; j0 += 64) {
            const f4 *const d = reinterpret_cast<const f4 *>(cur + min(j0 + lane, dout - 1) * kS);
            const f4 d0 = d[0], d1 = d[1];
            int at[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int j = j0 + e / 4 * 16 + l16;
              at[e] = j < dout ? ((i0 + 4 * quad + e % 4) * dout + j) * 4 : 0x7ffffffc;
            }
            f16 acc = {};
            if (!first)
#pragma unroll
              for (int e = 0; e < 16; ++e)
                acc[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(row, at[e], 0, 0));
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a0, d0[0], acc, 2, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a0, d0[1], acc, 2, 1, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a0, d0[2], acc, 2, 2, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a0, d0[3], acc, 2, 3, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a1, d1[0], acc, 2, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a1, d1[1], acc, 2, 1, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a1, d1[2], acc, 2, 2, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a1, d1[3], acc, 2, 3, 0);
#pragma unroll
            for (int e = 0; e < 16; ++e)
              __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[e]), row, at[e], 0, 0);
          }
        }
        float *const swap = cur;
        cur = next;
        next = swap;
        y = following;
      }
    }
  }
  if constexpr (kGrad) {
    // the samples' losses are in the first kS lanes of wave 0
#pragma unroll
    for (int off = kS / 2; off >= 1; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (t == 0) partial_loss[blockIdx.x] = loss;
  }
}

// grads[i] = the sum of the workgroups' rows in a fixed order: kGradLanes lanes per parameter take
// every kGradLanes-th row, eight loads in flight, in FP64, and meet in LDS. The last workgroup adds
// the losses.
constexpr int kGradLanes = 16;
__global__ __launch_bounds__(kB) void reduce_grads_kernel(const float *__restrict__ partial, int count, int rows,
                                                          const double *__restrict__ partial_loss, int64_t n,
                                                          float *__restrict__ grads, float *loss) {
  constexpr int kWidth = kB / kGradLanes;
  __shared__ double part[kB];
  const int t = threadIdx.x;
  if (blockIdx.x == gridDim.x - 1) {
    double s = 0.0;
    for (int r = t; r < rows; r += kB) s += partial_loss[r];
    part[t] = s;
    __syncthreads();
    for (int off = kB / 2; off > 0; off >>= 1) {
      if (t < off) part[t] += part[t + off];
      __syncthreads();
    }
    if (t == 0 && loss) *loss = float(part[0] / double(n));
    return;
  }
  const int i = int(blockIdx.x) * kWidth + t % kWidth, lane = t / kWidth;
  double s = 0.0;
  if (i < count) {
    for (int r = lane; r < rows; r += 8 * kGradLanes) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int at = r + k * kGradLanes;
        v[k] = at < rows ? partial[int64_t(at) * count + i] : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) s += double(v[k]);
    }
  }
  part[t] = s;
  __syncthreads();
  if (lane == 0 && i < count) {
#pragma unroll
    for (int l = 1; l < kGradLanes; ++l) s += part[l * kWidth + t];
    grads[i] = float(s);
  }
}

unsigned blocks(int64_t n) { return static_cast<unsigned>((n + kB - 1) / kB); }

uint32_t hash32(uint32_t v) {
  v = (v ^ 61u) ^ (v >> 16);
  v *= 9u;
  v ^= v << 4;
  v *= 0x27d4eb2du;
  v ^= v >> 15;
  return v;
}

// A workspace of `need` floats. Under capture one that grows is kept as well, since the calls captured
// before use it; allocating there needs the relaxed capture mode.
void ensure(cs_stream *stream, cs_mlp *net, float **buf, int64_t *cap, int64_t need) {
  if (*cap >= need) return;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  CS_HIP(hipStreamIsCapturing(stream->stream, &status));
  const bool capturing = status != hipStreamCaptureStatusNone;
  if (*buf && capturing) net->retired.push_back(*buf);
  if (*buf && !capturing) CS_HIP(hipFree(*buf));
  *buf = nullptr;
  *cap = 0;
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  if (capturing) CS_HIP(hipThreadExchangeStreamCaptureMode(&mode));
  const hipError_t r = hipMalloc(reinterpret_cast<void **>(buf), static_cast<size_t>(need) * 4);
  if (capturing) (void)hipThreadExchangeStreamCaptureMode(&mode);
  CS_HIP(r);
  *cap = need;
}

int64_t act_offset(const cs_mlp *net, int layer, int64_t n) {  // layer 1..L outputs
  int64_t off = 0;
  for (int l = 1; l < layer; ++l) off += n * net->widths[l];
  return off;
}

void forward(cs_stream *stream, cs_mlp *net, const float *X, int64_t n) {
  const int L = static_cast<int>(net->widths.size()) - 1;
  int64_t total = 0;
  for (int l = 1; l <= L; ++l) total += n * net->widths[l];
  ensure(stream, net, &net->acts, &net->acts_capacity, total);
  const float *in = X;
  for (int l = 1; l <= L; ++l) {
    float *out = net->acts + act_offset(net, l, n);
    int din = net->widths[l - 1], dout = net->widths[l];
    hipLaunchKernelGGL(linear_fwd, dim3(blocks(n * dout)), dim3(kB), 0, stream->stream, in, n, din,
                       net->params + net->w_off[l - 1], net->params + net->b_off[l - 1], dout, l < L ? 1 : 0, out);
    in = out;
  }
  CS_HIP(hipGetLastError());
}

// The whole-network kernel's shape, and its LDS bytes: 0 when the network does not fit.
size_t network_shape(const cs_mlp *net, bool grad, int samples, NetShape *shape) {
  const int L = static_cast<int>(net->widths.size()) - 1;
  if (L > kMaxLayers || net->count > (1 << 24)) return 0;
  shape->layers = L;
  shape->count = static_cast<int>(net->count);
  int unit = samples * padded(net->widths[0]), from = 0, weights = 0, widest = net->widths[0], layer = 0;
  for (int l = 1; l <= L; ++l) {
    NetLayer &y = shape->layer[l - 1];
    y.din = net->widths[l - 1], y.dout = net->widths[l];
    y.params = static_cast<int>(net->w_off[l - 1]);
    y.lds = weights;
    y.in = from, y.out = from = unit;
    unit += samples * padded(y.dout);
    widest = std::max(widest, y.dout);
    const int size = (padded(y.din) + 1) * pitch(y.dout);
    if (size > (1 << 16)) return 0;
    weights += size;
    layer = std::max(layer, size);
  }
  shape->unit_floats = unit;
  shape->delta_floats = grad ? samples * padded(widest) : 0;
  const size_t fixed = size_t(unit + 2 * shape->delta_floats) * 4, budget = net->device->props.sharedMemPerBlock;
  shape->resident = fixed + size_t(weights) * 4 <= budget;
  shape->weight_floats = shape->resident ? weights : layer;
  const size_t bytes = fixed + size_t(shape->weight_floats) * 4;
  return bytes <= budget ? bytes : 0;
}

// Workgroups for n samples: one each kS, up to `per_cu` on every CU (they take further samples in turn).
// With the gradient one: each has a row of `partial` to write and to add.
template <int kS>
unsigned network_grid(cs_stream *stream, int64_t n, int64_t per_cu) {
  return static_cast<unsigned>(
      std::min<int64_t>((n + kS - 1) / kS, per_cu * stream->device->props.multiProcessorCount));
}

template <bool kGrad, int kS>
void launch_network(cs_stream *stream, const NetShape &shape, size_t lds, unsigned grid, const cs_mlp *net,
                    const float *X, const float *target, int64_t n, float *y, float *partial, double *partial_loss) {
  static std::atomic<uint64_t> allowed{0};
  allow_lds(allowed, stream->device->ordinal, reinterpret_cast<const void *>(&network_kernel<kGrad, kS>), 160 << 10);
  hipLaunchKernelGGL((network_kernel<kGrad, kS>), dim3(grid), dim3(kNet), lds, stream->stream, shape, net->params, X,
                     target, n, y, partial, partial_loss);
}

// Whether the layer kernels, a thread per unit and sample, are ahead of the whole-network kernel in evaluating
// many samples on a network of few units: by estimates in us, of which the layers' is 2.2 for a launch and, for
// each input of a unit, the latency of one step of its loop or the rate of all CUs (1.7 times slower where rows
// of inputs straddle lines), or what L2 delivers where the rows that the waves of a CU read together outgrow
// its L1. The whole network's is per sample and 4 us. Measured (layers / whole; samples): 64-8-1 17.8 / 25.2
// (65536), 71 / 108 (300000); 1000-1 199 / 595, 2934 / 3042; 512-8 109 / 160, 585 / 889; 32-16-1 18.1 / 19.7,
// 62 / 84; 16-8-8-1 13.5 / 22.7 (65536); 256-4-1 52 / 71, 353 / 329; 200-8-1 59 / 55, 280 / 248; 64-16-1
// 27 / 25, 111 / 108; 12-14-14-1 26 / 23; 30-30-1 37 / 21. Above 65536 samples networks of up to 400
// parameters stay with the layers.
bool prefer_layers(const cs_mlp *net, const NetShape &shape, size_t lds, int samples, int64_t n) {
  const double cus = net->device->props.multiProcessorCount;
  double layers = 0.0;
  for (int l = 0; l < shape.layers; ++l) {
    const int din = shape.layer[l].din, dout = shape.layer[l].dout;
    const double threads = double(n) * dout, waves = std::min(32.0, threads / 64 / cus);
    double step = std::max(0.17, (din % 16 && dout <= 16 ? 1.7e-4 : 1e-4) * threads / cus);
    if (waves * std::max(1, 64 / dout) * std::min(128, 4 * din) > 36000)
      step = std::max(step, 4.9e-6 * double(n) * std::min(1.0, din / 32.0));
    layers += 2.2 + step * din;
  }
  const double crowded = samples < 4 * kSamples && n > kManySamples ? 2.4 : size_t(160 << 10) / lds < 2 ? 1.35 : 1.0;
  const double whole = 4 + double(n) * (1e-4 + 3.6e-6 * shape.layer[0].din + 6e-5 * (shape.layers - 1)) * crowded;
  return layers < 0.95 * whole || (n > 65536 && shape.count <= 400);
}

// Evaluation with kS samples per workgroup, where the network fits.
template <int kS>
bool evaluate(cs_stream *stream, cs_mlp *net, const float *X, int64_t n, float *y) {
  NetShape shape;
  const size_t lds = network_shape(net, false, kS, &shape);
  if (!lds || prefer_layers(net, shape, lds, kS, n)) return false;
  const int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>(4, int64_t(160 << 10) / int64_t(lds)));
  launch_network<false, kS>(stream, shape, lds, network_grid<kS>(stream, n, per_cu), net, X, nullptr, n, y, nullptr,
                            nullptr);
  CS_HIP(hipGetLastError());
  return true;
}

}  // namespace
}  // namespace csmi

using namespace csmi;

extern "C" {

cs_status cs_mlp_create(cs_device *device, const int32_t *widths, int nw, uint32_t seed, cs_mlp **mlp) {
  return guard([&] {
    if (!device || !widths || !mlp) fail(CS_INVALID_VALUE, "null argument");
    if (nw < 2 || nw > 16) fail(CS_INVALID_VALUE, "a network has 2 to 16 widths");
    for (int i = 0; i < nw; ++i)
      if (widths[i] < 1 || widths[i] > 4096) fail(CS_INVALID_VALUE, "layer width out of range");
    // freed with its device arrays if a later step fails
    std::unique_ptr<cs_mlp, void (*)(cs_mlp *)> net(new cs_mlp(), [](cs_mlp *x) {
      for (float *p : {x->params, x->m, x->v})
        if (p) (void)hipFree(p);
      delete x;
    });
    net->device = device;
    for (int i = 0; i < nw; ++i) net->widths.push_back(widths[i]);
    std::vector<float> host;
    for (int l = 1; l < nw; ++l) {
      int din = widths[l - 1], dout = widths[l];
      net->w_off.push_back(static_cast<int64_t>(host.size()));
      // He-uniform: U(-sqrt(6/din), sqrt(6/din)) from the Wang hash of (seed, index)
      double a = std::sqrt(6.0 / din);
      for (int64_t k = 0; k < int64_t(din) * dout; ++k) {
        uint32_t h = hash32(static_cast<uint32_t>(host.size()) ^ hash32(seed + 0x9e3779b9u * l));
        host.push_back(static_cast<float>(-a + 2.0 * a * (h * (1.0 / 4294967296.0))));
      }
      net->b_off.push_back(static_cast<int64_t>(host.size()));
      for (int j = 0; j < dout; ++j) host.push_back(0.0f);
    }
    net->count = static_cast<int64_t>(host.size());
    set_device(device);
    CS_HIP(hipMalloc(reinterpret_cast<void **>(&net->params), host.size() * 4));
    CS_HIP(hipMalloc(reinterpret_cast<void **>(&net->m), host.size() * 4));
    CS_HIP(hipMalloc(reinterpret_cast<void **>(&net->v), host.size() * 4));
    CS_HIP(hipMemcpy(net->params, host.data(), host.size() * 4, hipMemcpyHostToDevice));
    CS_HIP(hipMemset(net->m, 0, host.size() * 4));
    CS_HIP(hipMemset(net->v, 0, host.size() * 4));
    *mlp = net.release();
  });
}

cs_status cs_mlp_param_count(cs_mlp *mlp, int64_t *count) {
  return guard([&] {
    if (!mlp || !count) fail(CS_INVALID_VALUE, "null argument");
    *count = mlp->count;
  });
}

cs_status cs_mlp_get_params(cs_stream *stream, cs_mlp *mlp, float *host, int64_t count) {
  return guard([&] {
    if (!stream || !mlp || !host) fail(CS_INVALID_VALUE, "null argument");
    if (count != mlp->count) fail(CS_INVALID_VALUE, "parameter count mismatch");
    set_device(stream->device);
    CS_HIP(hipMemcpyAsync(host, mlp->params, size_t(count) * 4, hipMemcpyDeviceToHost, stream->stream));
    CS_HIP(hipStreamSynchronize(stream->stream));
  });
}

cs_status cs_mlp_set_params(cs_stream *stream, cs_mlp *mlp, const float *host, int64_t count) {
  return guard([&] {
    if (!stream || !mlp || !host) fail(CS_INVALID_VALUE, "null argument");
    if (count != mlp->count) fail(CS_INVALID_VALUE, "parameter count mismatch");
    set_device(stream->device);
    CS_HIP(hipMemcpyAsync(mlp->params, host, size_t(count) * 4, hipMemcpyHostToDevice, stream->stream));
    CS_HIP(hipStreamSynchronize(stream->stream));
  });
}

cs_status cs_mlp_forward(cs_stream *stream, cs_mlp *mlp, const float *X, int64_t n, float *y) {
  return guard([&] {
    if (!stream || !mlp || !X || !y) fail(CS_INVALID_VALUE, "null argument");
    if (n <= 0) fail(CS_INVALID_VALUE, "no samples");
    set_device(stream->device);
    // y over X's memory: the layer kernels have read X before y is written
    const bool over = y < X + n * mlp->widths.front() && X < y + n * mlp->widths.back();
    if (!over && ((n > kManySamples && evaluate<4 * kSamples>(stream, mlp, X, n, y)) ||
                  evaluate<kSamples>(stream, mlp, X, n, y)))
      return;
    forward(stream, mlp, X, n);
    const int L = static_cast<int>(mlp->widths.size()) - 1;
    CS_HIP(hipMemcpyAsync(y, mlp->acts + act_offset(mlp, L, n), size_t(n) * mlp->widths[L] * 4,
                          hipMemcpyDeviceToDevice, stream->stream));
  });
}

cs_status cs_mlp_backward(cs_stream *stream, cs_mlp *mlp, const float *X, const float *target, int64_t n,
                          float *loss, float *grads) {
  return guard([&] {
    if (!stream || !mlp || !X || !target || !grads) fail(CS_INVALID_VALUE, "null argument");
    if (n <= 0) fail(CS_INVALID_VALUE, "no samples");
    const int L = static_cast<int>(mlp->widths.size()) - 1;
    if (mlp->widths[L] != 1) fail(CS_INVALID_VALUE, "the loss needs a single output");
    set_device(stream->device);
    NetShape shape;
    if (const size_t lds = network_shape(mlp, true, kSamples, &shape)) {
      const unsigned grid = network_grid<kSamples>(stream, n, 1);
      // partial losses (FP64), then one row of gradients per workgroup
      ensure(stream, mlp, &mlp->deltas, &mlp->deltas_capacity, int64_t(grid) * (2 + mlp->count));
      double *partial_loss = reinterpret_cast<double *>(mlp->deltas);
      float *partial = mlp->deltas + 2 * grid;
      launch_network<true, kSamples>(stream, shape, lds, grid, mlp, X, target, n, nullptr, partial, partial_loss);
      hipLaunchKernelGGL(reduce_grads_kernel, dim3(blocks(kGradLanes * mlp->count) + 1), dim3(kB), 0, stream->stream,
                         partial,
                         static_cast<int>(mlp->count), static_cast<int>(grid), partial_loss, n, grads, loss);
      CS_HIP(hipGetLastError());
      return;
    }
    forward(stream, mlp, X, n);
    int wmax = 1;
    for (int w : mlp->widths) wmax = std::max(wmax, w);
    ensure(stream, mlp, &mlp->deltas, &mlp->deltas_capacity, 2 * n * wmax);
    float *d_cur = mlp->deltas, *d_next = mlp->deltas + n * wmax;
    const float *pred = mlp->acts + act_offset(mlp, L, n);
    hipLaunchKernelGGL(mse_grad, dim3(1), dim3(1024), 0, stream->stream, pred, target, n, d_cur, loss);
    for (int l = L; l >= 1; --l) {
      int din = mlp->widths[l - 1], dout = mlp->widths[l];
      const float *Y = mlp->acts + act_offset(mlp, l, n);
      const float *Xin = l == 1 ? X : mlp->acts + act_offset(mlp, l - 1, n);
      int relu = l < L ? 1 : 0;
      hipLaunchKernelGGL(linear_bwd_dw, dim3(blocks(int64_t(din + 1) * dout)), dim3(kB), 0, stream->stream, Xin,
                         d_cur, Y, relu, n, din, dout, grads + mlp->w_off[l - 1], grads + mlp->b_off[l - 1]);
      if (l > 1) {
        hipLaunchKernelGGL(linear_bwd_dx, dim3(blocks(n * din)), dim3(kB), 0, stream->stream, d_cur, Y, relu,
                           mlp->params + mlp->w_off[l - 1], n, din, dout, d_next);
        std::swap(d_cur, d_next);
      }
    }
    CS_HIP(hipGetLastError());
  });
}

cs_status cs_mlp_adam(cs_stream *stream, cs_mlp *mlp, const float *grads, float lr, int t) {
  return guard([&] {
    if (!stream || !mlp || !grads) fail(CS_INVALID_VALUE, "null argument");
    if (t < 1) fail(CS_INVALID_VALUE, "Adam steps count from 1");
    const float b1 = 0.9f, b2 = 0.999f;
    float c1 = 1.0f - std::pow(b1, float(t)), c2 = 1.0f - std::pow(b2, float(t));
    set_device(stream->device);
    hipLaunchKernelGGL(adam_kernel, dim3(blocks(mlp->count)), dim3(kB), 0, stream->stream, mlp->params, grads, mlp->m,
                       mlp->v, mlp->count, lr, b1, b2, 1e-8f, c1, c2);
    CS_HIP(hipGetLastError());
  });
}

cs_status cs_mlp_release(cs_mlp *mlp) {
  return guard([&] {
    if (!mlp) fail(CS_INVALID_VALUE, "mlp is null");
    set_device(mlp->device);
    for (float *p : {mlp->params, mlp->m, mlp->v, mlp->acts, mlp->deltas})
      if (p) (void)hipFree(p);
    for (float *p : mlp->retired) (void)hipFree(p);
    delete mlp;
  });
}

}  // extern "C"
