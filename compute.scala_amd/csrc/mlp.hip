// A small fully connected network (the cost model's predictor), trained and evaluated on
// the device: forward, mean-squared-error gradient, backward and Adam, all in FP32.
//
// The reference has no counterpart (it has no tuning). Layout: parameters are one flat
// FP32 array [W1 (d0 x d1), b1 (d1), W2 (d1 x d2), b2, ...]; W is row-major [in][out]; ReLU
// follows every layer but the last. Every reduction runs in a fixed order (one thread per
// output sum), so results are deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
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
// and reduce_grads_kernel adds the rows. The forward sums run in the order of linear_fwd (bias
// first, inputs in order), so activations are the same bits on either path. Bound by the latency of
// the chain of layers in one workgroup (about 13 us for 23-64-64-64-1, of which the forward pass
// takes 5): a gradient of 512 samples takes 19.7 us in two launches, against 820 us in twelve with
// one thread per weight summing over all samples. Eight samples and 512 threads a workgroup: four
// samples double the rows to add (25.5 us), 1024 threads change nothing.
constexpr int kSamples = 8;  // per workgroup
constexpr int kNet = 512;      // threads of its kernel
constexpr int kMaxLayers = 15;

struct NetShape {
  int layers;                      // L: widths[0] -> ... -> widths[L]
  int widths[kMaxLayers + 1];
  int w_off[kMaxLayers];           // of layer l + 1 in the flat parameters: W, then b
  int act_off[kMaxLayers + 1];     // LDS offset of layer l's activations (0: the input)
  int unit_off[kMaxLayers + 1];    // likewise of the activations by unit
  int act_floats, unit_floats, delta_floats;  // LDS floats of both forms and of one delta buffer
  int count;                       // parameters
  int resident;                    // all parameters stay in LDS, else one layer's at a time
};

__host__ __device__ __forceinline__ int padded(int width) { return (width + 3) & ~3; }

// Copies n floats of global memory to LDS, four 16-byte loads of a thread in flight (src at any
// 4-byte boundary, dst at 16 bytes).
__device__ __forceinline__ void copy_to_lds(float *dst, const float *__restrict__ src, int n) {
  typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
  const f4u *s4 = reinterpret_cast<const f4u *>(src);
  f4u *d4 = reinterpret_cast<f4u *>(dst);
  const int nv = n / 4;
  int i = threadIdx.x;
  for (; i + 3 * kNet < nv; i += 4 * kNet) {
    f4u v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = s4[i + k * kNet];
#pragma unroll
    for (int k = 0; k < 4; ++k) d4[i + k * kNet] = v[k];
  }
  for (; i < nv; i += kNet) d4[i] = s4[i];
  for (int j = nv * 4 + threadIdx.x; j < n; j += kNet) dst[j] = src[j];
}

// LDS: activations by sample [layer][sample][padded width] and by unit [layer][unit, then a one for
// the bias][sample], two delta buffers [sample][widest], parameters.
template <bool kGrad>
__global__ __launch_bounds__(kNet) void network_kernel(NetShape net, const float *__restrict__ params,
                                                       const float *__restrict__ X, const float *__restrict__ target,
                                                       int64_t n, float *__restrict__ y, float *__restrict__ partial,
                                                       double *__restrict__ partial_loss) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float *const acts = lds, *const by_unit = lds + net.act_floats;
  float *const deltas = by_unit + net.unit_floats, *const weights = deltas + 2 * net.delta_floats;
  const int t = threadIdx.x, L = net.layers;
  const int last = net.widths[L];
  if (net.resident) copy_to_lds(weights, params, net.count);
  // Layer l's parameters in LDS, for every thread of the workgroup.
  auto layer_weights = [&](int l) -> const float * {
    const int from = net.w_off[l - 1];
    if (net.resident) return weights + from;
    __syncthreads();  // the previous layer's are no longer read
    copy_to_lds(weights, params + from, (net.widths[l - 1] + 1) * net.widths[l]);
    return weights;
  };
  double loss = 0.0;
  bool first = true;
  for (int64_t s0 = int64_t(blockIdx.x) * kSamples; s0 < n; s0 += int64_t(gridDim.x) * kSamples, first = false) {
    const int live = n - s0 < kSamples ? static_cast<int>(n - s0) : kSamples;  // samples past n are zeros
    const int din0 = net.widths[0], pad0 = padded(din0);
    __syncthreads();  // the activations of the samples before are no longer read
    if (kGrad && first)
      for (int l = 0; l < L; ++l)  // the bias's input, after each layer's units
        if (t < kSamples) by_unit[net.unit_off[l] + net.widths[l] * kSamples + t] = 1.0f;
    for (int i = t; i < kSamples * pad0; i += kNet) {
      const int s = i / pad0, c = i % pad0;
      const float x = s < live && c < din0 ? X[(s0 + s) * din0 + c] : 0.0f;
      acts[i] = x;
      if (kGrad && c < din0) by_unit[c * kSamples + s] = x;
    }
    for (int l = 1; l <= L; ++l) {
      const int din = net.widths[l - 1], dout = net.widths[l], pin = padded(din), pout = padded(dout);
      const float *const w = layer_weights(l), *const b = w + din * dout;
      const float *const in = acts + net.act_off[l - 1];
      float *const out = acts + net.act_off[l], *const out_unit = by_unit + net.unit_off[l];
      __syncthreads();
      for (int o = t; o < dout * kSamples; o += kNet) {
        const int s = o / dout, j = o - s * dout;
        const float *const x = in + s * pin, *wj = w + j;
        float acc = b[j];
        int i = 0;
        for (; i + 16 <= din; i += 16, wj += 16 * dout) {
          float4 xs[4];
          float v[16];
#pragma unroll
          for (int k = 0; k < 4; ++k) xs[k] = *reinterpret_cast<const float4 *>(x + i + 4 * k);
#pragma unroll
          for (int k = 0; k < 16; ++k) v[k] = wj[k * dout];
          __builtin_amdgcn_sched_barrier(0);  // all reads out before the first use
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            acc = fmaf(xs[k].x, v[4 * k], acc);
            acc = fmaf(xs[k].y, v[4 * k + 1], acc);
            acc = fmaf(xs[k].z, v[4 * k + 2], acc);
            acc = fmaf(xs[k].w, v[4 * k + 3], acc);
          }
        }
        for (; i < din; ++i, wj += dout) acc = fmaf(x[i], *wj, acc);
        if (l < L) acc = fmaxf(acc, 0.0f);
        out[s * pout + j] = acc;
        if (kGrad) out_unit[j * kSamples + s] = acc;
      }
    }
    __syncthreads();
    const float *const pred = acts + net.act_off[L];
    if constexpr (!kGrad) {
      for (int i = t; i < live * last; i += kNet) y[s0 * last + i] = pred[(i / last) * padded(last) + i % last];
    } else {
      // delta[s][j]: the loss's gradient by layer l's output before its ReLU
      float *cur = deltas, *next = deltas + net.delta_floats;
      if (t < kSamples) {
        const float d = t < live ? pred[t * padded(last)] - target[s0 + t] : 0.0f;
        cur[t] = 2.0f * d / float(n);
        loss += double(d) * double(d);
      }
      for (int l = L; l >= 1; --l) {
        const int din = net.widths[l - 1], dout = net.widths[l], pin = padded(din);
        const float *const in = acts + net.act_off[l - 1], *const in_unit = by_unit + net.unit_off[l - 1];
        const float *const w = l > 1 ? layer_weights(l) : nullptr;
        __syncthreads();
        // dW[i][j] = sum_s in[s][i] delta[s][j]; row din is the bias's, whose input is 1. A thread
        // keeps a column j (several in turn where there are more than threads) and takes every
        // `rows`-th row.
        float *const row = partial + int64_t(blockIdx.x) * net.count + net.w_off[l - 1];
        const int rows = dout < kNet ? kNet / dout : 1, side = dout < kNet ? dout : kNet;
        const int i0 = t / side;
        for (int j = t - i0 * side; j < dout && i0 < rows; j += side) {
          float g[kSamples];
#pragma unroll
          for (int s = 0; s < kSamples; ++s) g[s] = cur[s * dout + j];
          auto add = [&](int i, float acc) {
            const float4 *const u = reinterpret_cast<const float4 *>(in_unit + i * kSamples);
#pragma unroll
            for (int s = 0; s < kSamples / 4; ++s) {
              const float4 x = u[s];
              acc = fmaf(x.x, g[4 * s], acc);
              acc = fmaf(x.y, g[4 * s + 1], acc);
              acc = fmaf(x.z, g[4 * s + 2], acc);
              acc = fmaf(x.w, g[4 * s + 3], acc);
            }
            return acc;
          };
          if (first) {
#pragma unroll 4
            for (int i = i0; i <= din; i += rows) row[i * dout + j] = add(i, 0.0f);
          } else {
            for (int i = i0; i <= din; i += rows) row[i * dout + j] = add(i, row[i * dout + j]);
          }
        }
        if (l > 1) {
          // dX[s][i] = sum_j delta[s][j] W[i][j], from a different j on for each i and round, so
          // that the rows of W that a wave reads at once lie in different banks; then the ReLU of
          // layer l - 1
          const bool quads = dout % 4 == 0 && net.w_off[l - 1] % 4 == 0;
          for (int o = t; o < kSamples * din; o += kNet) {
            const int s = o / din, i = o - s * din;
            const float *const wi = w + i * dout, *const gs = cur + s * dout;
            float acc = 0.0f;
            if (quads) {
              const int nq = dout / 4;
              int q = i % nq;
#pragma unroll 4
              for (int k = 0; k < nq; ++k) {
                const float4 g = reinterpret_cast<const float4 *>(gs)[q], v = reinterpret_cast<const float4 *>(wi)[q];
                acc = fmaf(g.x, v.x, acc);
                acc = fmaf(g.y, v.y, acc);
                acc = fmaf(g.z, v.z, acc);
                acc = fmaf(g.w, v.w, acc);
                q = q + 1 == nq ? 0 : q + 1;
              }
            } else {
              int j = i % dout;
#pragma unroll 8
              for (int k = 0; k < dout; ++k) {
                acc = fmaf(gs[j], wi[j], acc);
                j = j + 1 == dout ? 0 : j + 1;
              }
            }
            next[s * din + i] = in[s * pin + i] <= 0.0f ? 0.0f : acc;
          }
          float *const swap = cur;
          cur = next;
          next = swap;
        }
      }
    }
  }
  if constexpr (kGrad) {
    // the samples' losses are in the first kSamples lanes of wave 0
#pragma unroll
    for (int off = kSamples / 2; off >= 1; off >>= 1) loss += __shfl_xor(loss, off, 64);
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

void ensure(float **buf, int64_t *cap, int64_t need) {
  if (*cap >= need) return;
  if (*buf) CS_HIP(hipFree(*buf));
  *buf = nullptr;
  CS_HIP(hipMalloc(reinterpret_cast<void **>(buf), static_cast<size_t>(need) * 4));
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
  ensure(&net->acts, &net->acts_capacity, total);
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
size_t network_shape(const cs_mlp *net, bool grad, NetShape *shape) {
  const int L = static_cast<int>(net->widths.size()) - 1;
  if (L > kMaxLayers || net->count > (1 << 24)) return 0;
  shape->layers = L;
  shape->count = static_cast<int>(net->count);
  int act = 0, unit = 0, widest = 1, layer = 0;
  for (int l = 0; l <= L; ++l) {
    const int w = net->widths[l];
    shape->widths[l] = w;
    shape->act_off[l] = act;
    shape->unit_off[l] = unit;
    act += kSamples * padded(w);
    if (grad) unit += kSamples * padded(w + 1);
    widest = std::max(widest, w);
    if (l == 0) continue;
    shape->w_off[l - 1] = static_cast<int>(net->w_off[l - 1]);
    layer = std::max(layer, (net->widths[l - 1] + 1) * w);
  }
  shape->act_floats = act;
  shape->unit_floats = unit;
  shape->delta_floats = grad ? kSamples * padded(widest) : 0;
  const size_t fixed = size_t(act + unit + 2 * shape->delta_floats) * 4, budget = net->device->props.sharedMemPerBlock;
  shape->resident = fixed + size_t(net->count) * 4 <= budget;
  const size_t bytes = fixed + size_t(shape->resident ? shape->count : layer) * 4;
  return bytes <= budget ? bytes : 0;
}

template <bool kGrad>
void launch_network(cs_stream *stream, const NetShape &shape, size_t lds, unsigned grid, const cs_mlp *net,
                    const float *X, const float *target, int64_t n, float *y, float *partial, double *partial_loss) {
  static const bool configured = [] {
    CS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&network_kernel<kGrad>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 << 10));
    return true;
  }();
  (void)configured;
  hipLaunchKernelGGL(network_kernel<kGrad>, dim3(grid), dim3(kNet), lds, stream->stream, shape, net->params, X, target, n,
                     y, partial, partial_loss);
}

// Workgroups for n samples: one each kSamples, up to `per_cu` on every CU (they take further samples
// in turn). With the gradient one: each has a row of `partial` to write and to add.
unsigned network_grid(cs_stream *stream, int64_t n, int64_t per_cu) {
  return static_cast<unsigned>(std::min<int64_t>((n + kSamples - 1) / kSamples,
                                                 per_cu * stream->device->props.multiProcessorCount));
}

// Evaluation alone, of very many samples on a network too narrow to give every thread a unit: the
// layer kernels, whose threads do not wait for one another, are ahead (262144 samples through
// 8-16-1: 34 us against 45; through 23-64-64-64-1 they are behind, 872 against 650).
bool prefer_layers(const NetShape &shape, int64_t n) {
  int widest = 1;
  for (int l = 1; l <= shape.layers; ++l) widest = std::max(widest, shape.widths[l]);
  return n > 65536 && widest * kSamples < kNet;
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
    NetShape shape;
    const size_t lds = network_shape(mlp, false, &shape);
    // y over X's memory: the layer kernels have read X before y is written
    const bool over = y < X + n * mlp->widths.front() && X < y + n * mlp->widths.back();
    if (lds && !over && !prefer_layers(shape, n)) {
      const int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>(4, int64_t(160 << 10) / int64_t(lds)));
      launch_network<false>(stream, shape, lds, network_grid(stream, n, per_cu), mlp, X, nullptr, n, y, nullptr, nullptr);
      CS_HIP(hipGetLastError());
      return;
    }
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
    if (const size_t lds = network_shape(mlp, true, &shape)) {
      const unsigned grid = network_grid(stream, n, 1);
      // partial losses (FP64), then one row of gradients per workgroup
      ensure(&mlp->deltas, &mlp->deltas_capacity, int64_t(grid) * (2 + mlp->count));
      double *partial_loss = reinterpret_cast<double *>(mlp->deltas);
      float *partial = mlp->deltas + 2 * grid;
      launch_network<true>(stream, shape, lds, grid, mlp, X, target, n, nullptr, partial, partial_loss);
      hipLaunchKernelGGL(reduce_grads_kernel, dim3(blocks(kGradLanes * mlp->count) + 1), dim3(kB), 0, stream->stream, partial,
                         static_cast<int>(mlp->count), static_cast<int>(grid), partial_loss, n, grads, loss);
      CS_HIP(hipGetLastError());
      return;
    }
    forward(stream, mlp, X, n);
    int wmax = 1;
    for (int w : mlp->widths) wmax = std::max(wmax, w);
    ensure(&mlp->deltas, &mlp->deltas_capacity, 2 * n * wmax);
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
    delete mlp;
  });
}

}  // extern "C"
