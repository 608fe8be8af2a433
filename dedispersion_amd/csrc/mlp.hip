// mlp.hip -- the cost model of the learned tuner: a small fully connected
// network (inputs -> hidden x layers, ReLU -> 1) in FP32, with forward,
// backward (mean squared error) and Adam kernels, all on the device.
//
// Parameters are one flat device array: for each layer l with fan-in a and
// fan-out b, W_l (a x b, row-major: W_l[i * b + j] connects input i to unit
// j) followed by its bias (b).  Gradients use the same layout.
//
// The reference has no learned tuner: its tuner (src/DedispersionTuning.cpp)
// is exhaustive.  This network ranks configurations so that only the most
// promising ones are timed; the exhaustive sweep stays the fallback.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "dedispersion_amd.h"
#include "internal.hpp"

namespace {

using ddamd::set_error;

constexpr uint32_t kMaxWidth = 256;

// The network's shape: dense layers 0 .. layers (the last has one unit).
struct Shape {
  uint32_t inputs, hidden, layers;
  __host__ __device__ uint32_t fan_in(uint32_t l) const { return l == 0 ? inputs : hidden; }
  __host__ __device__ uint32_t fan_out(uint32_t l) const { return l == layers ? 1 : hidden; }
  __host__ __device__ uint32_t offset(uint32_t l) const {  // of layer l's weights; its biases follow
    return l == 0 ? 0 : inputs * hidden + hidden + (l - 1) * (hidden * hidden + hidden);
  }
  // the same in LDS, where every row of weights is followed by an unused float
  // so that neither a walk along a row nor one down a column meets bank conflicts
  __host__ __device__ uint32_t lds_offset(uint32_t l) const {
    return l == 0 ? 0 : inputs * (hidden + 1) + hidden + (l - 1) * (hidden * (hidden + 1) + hidden);
  }
  __host__ __device__ uint32_t lds_floats() const { return (lds_offset(layers) + 2 * hidden + 1 + 3) & ~3u; }
};

constexpr uint32_t kColumns = 32;       // columns of a weight matrix transposed through LDS at a time
constexpr uint32_t kMaxGroups = 512;    // workgroups of the gradient pass (partial gradients)
constexpr uint32_t kMaxParts = 1u << 27;  // floats of their partial gradients (512 MiB; 1 GiB is 1.5x faster at most)
constexpr uint32_t kHalfLds = 80 * 1024;      // LDS of a workgroup that shares a compute unit with another
constexpr uint32_t kResidentLds = 64 * 1024;  // ... whose weights stay in LDS

// A layer's weights W[i * ld + j] and biases, in LDS or in the parameter array.
struct Layer {
  const float *W, *b;
  uint32_t ld;
};

template <bool RESIDENT>
__device__ __forceinline__ Layer layer_of(const Shape &s, uint32_t l, const float *params, const float *weights) {
  const uint32_t a = s.fan_in(l), b = s.fan_out(l);
  if (RESIDENT) return Layer{weights + s.lds_offset(l), weights + s.lds_offset(l) + a * (b + 1), b + 1};
  return Layer{params + s.offset(l), params + s.offset(l) + a * b, b};
}

constexpr uint32_t kBatch = 8;  // reads sent for together, before any of them is used

// All parameters to LDS: wavefronts take rows of weights (row a: the biases) and
// lanes their columns.
__device__ __forceinline__ void read_weights(const Shape &s, const float *__restrict__ params, float *weights) {
  const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64, waves = blockDim.x / 64;
  for (uint32_t l = 0; l <= s.layers; ++l) {
    const uint32_t a = s.fan_in(l), b = s.fan_out(l);
    const float *from = params + s.offset(l);
    float *to = weights + s.lds_offset(l);
    for (uint32_t j = lane; j < b; j += 64)
      for (uint32_t i0 = wave; i0 <= a; i0 += waves * kBatch) {
        float v[kBatch];
#pragma unroll
        for (uint32_t k = 0; k < kBatch; ++k) v[k] = from[min(i0 + k * waves, a) * b + j];
#pragma unroll
        for (uint32_t k = 0; k < kBatch; ++k)
          if (i0 + k * waves <= a) to[(i0 + k * waves) * (b + 1) + j] = v[k];
      }
  }
}

// acc += sum over c < n, in order, of e[c * R .. + 3] w[c * ld].
template <uint32_t R>
__device__ __forceinline__ void add_products(float4 &acc, const float *e, const float *w, uint32_t n, uint32_t ld) {
  auto add = [&](const float4 &x, float y) {
    acc.x += x.x * y;
    acc.y += x.y * y;
    acc.z += x.z * y;
    acc.w += x.w * y;
  };
  uint32_t c = 0;
  for (; c + kBatch <= n; c += kBatch) {
    float4 x[kBatch];
    float y[kBatch];
#pragma unroll
    for (uint32_t k = 0; k < kBatch; ++k) {
      y[k] = w[(c + k) * ld];
      x[k] = *reinterpret_cast<const float4 *>(e + (c + k) * R);
    }
    __builtin_amdgcn_sched_barrier(0);  // the scheduler would read each next to its use
#pragma unroll
    for (uint32_t k = 0; k < kBatch; ++k) add(x[k], y[k]);
  }
  for (; c < n; ++c) add(*reinterpret_cast<const float4 *>(e + c * R), w[c * ld]);
}

// One layer over R rows held unit by unit (in[i * R + r]): out[j][r] = act(b[j]
// + sum over i, in order, of in[i][r] W[i][j]); a thread takes four rows of a
// unit, and consecutive threads consecutive units.  CUT: rows from `rows` on are zero.
template <uint32_t R, bool CUT>
__device__ __forceinline__ void dense(const Layer &y, uint32_t din, uint32_t dout, bool relu, const float *in, float *out,
                                      uint32_t rows = R) {
  for (uint32_t idx = threadIdx.x; idx < dout * (R / 4); idx += blockDim.x) {
    const uint32_t j = idx % dout, q = 4 * (idx / dout);
    const float bias = y.b[j];
    float4 acc = make_float4(bias, bias, bias, bias);
    add_products<R>(acc, in + q, y.W + j, din, y.ld);
    if (relu) acc = make_float4(fmaxf(acc.x, 0.0f), fmaxf(acc.y, 0.0f), fmaxf(acc.z, 0.0f), fmaxf(acc.w, 0.0f));
    if (CUT && q + 4 > rows)
      acc = make_float4(q < rows ? acc.x : 0.0f, q + 1 < rows ? acc.y : 0.0f, q + 2 < rows ? acc.z : 0.0f, 0.0f);
    *reinterpret_cast<float4 *>(out + j * R + q) = acc;
  }
}

// Rows r0 .. r0 + R - 1 of X (n x inputs) to in[i * R + r]; zeros past row n.  Few
// rows are read in the order of the input.  Of 64, a thread takes four inputs of a
// row and consecutive threads consecutive rows, whose places in LDS lie side by side
// (in the input's order they are 64 floats apart, all on one bank: 260 against 210 us
// for 200000 rows of 256 x 8 x 1; over 16 rows it costs 0.7 us more latency).
template <uint32_t R>
__device__ __forceinline__ void read_rows(const float *__restrict__ X, uint32_t n, uint32_t inputs, uint64_t r0, float *in) {
  if constexpr (R < 64) {
    for (uint32_t idx = threadIdx.x; idx < inputs * R; idx += blockDim.x) {
      const uint32_t r = idx / inputs, i = idx % inputs;
      in[i * R + r] = r0 + r < n ? X[(r0 + r) * inputs + i] : 0.0f;
    }
  } else {
    struct __attribute__((packed, aligned(4))) Four {
      float v[4];
    };
    for (uint32_t idx = threadIdx.x; idx < (inputs + 3) / 4 * R; idx += blockDim.x) {
      const uint32_t r = idx % R, i = 4 * (idx / R);
      const float *x = X + (r0 + r) * inputs + i;
      Four f = {{0.0f, 0.0f, 0.0f, 0.0f}};
      if (r0 + r < n) {
        if (i + 4 <= inputs) {
          f = *reinterpret_cast<const Four *>(x);
        } else {
#pragma unroll
          for (uint32_t k = 0; k < 3; ++k)
            if (i + k < inputs) f.v[k] = x[k];
        }
      }
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k)
        if (i + k < inputs) in[(i + k) * R + r] = f.v[k];
    }
  }
}

// The whole network over R rows per workgroup; activations stay in LDS (two
// buffers in turn), as do the weights where they fit (RESIDENT).
template <uint32_t R, bool RESIDENT>
__global__ void __launch_bounds__(256) mlp_forward(const Shape s, const float *__restrict__ X, uint32_t n,
                                                   const float *__restrict__ params, float *__restrict__ Y) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const uint32_t width = s.inputs > s.hidden ? s.inputs : s.hidden;
  float *in = lds, *out = lds + width * R;
  float *weights = out + s.hidden * R;
  if (RESIDENT) read_weights(s, params, weights);
  const uint64_t r0 = (uint64_t)blockIdx.x * R;
  read_rows<R>(X, n, s.inputs, r0, in);
  __syncthreads();
  for (uint32_t l = 0; l <= s.layers; ++l) {
    dense<R, false>(layer_of<RESIDENT>(s, l, params, weights), s.fan_in(l), s.fan_out(l), l < s.layers, in, out);
    __syncthreads();
    float *t = in;
    in = out;
    out = t;
  }
  if (threadIdx.x < R && r0 + threadIdx.x < n) Y[r0 + threadIdx.x] = in[threadIdx.x];
}

// Threads of a workgroup of the gradient pass.  Weights that are not in LDS are
// waited for; twice the threads have twice the reads under way (four rows of
// 256 x 256 x 8 networks: 802 us with 256 threads, 16 columns at a time and one
// read after another; 691 with the reads in batches; 347 with 512 threads and 32
// columns; one launch per layer and operation took 458).
constexpr uint32_t gradient_threads(bool resident) { return resident ? 256 : 512; }

// Forward and backward pass of L = (1/n) sum_r (y_r - t_r)^2 over R rows at a
// time.  Activations and errors stay in LDS.  Workgroup g takes row blocks g, g
// + gridDim.x, ... and leaves its part of dL/dparams in part[g * (count + 1)],
// followed by its sum of squared errors.
//
// A pass over 2880 rows of the tuner's 9217 parameters took 2860 us as one
// launch per layer and operation, with one thread per weight walking all rows in
// 17 workgroups; as this pass and the sum of its parts it takes 39 us (70 with the
// weights read through the caches in every layer).  It is bound by the latency of
// one workgroup's chain of layers, so a workgroup takes as few rows as still
// share a weight read.
template <uint32_t R, bool RESIDENT>
__global__ void __launch_bounds__(gradient_threads(RESIDENT)) mlp_gradient(const Shape s, const float *__restrict__ X,
                                                    const float *__restrict__ T, uint32_t n,
                                                    const float *__restrict__ params, uint32_t count,
                                                    float *__restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float *act = lds;  // the input rows, then every hidden layer's output
  float *G = act + (s.inputs + s.layers * s.hidden) * R, *GX = G + s.hidden * R;
  // all weights, or [hidden][kColumns + 1] of a layer's; the squares
  float *weights = GX + s.hidden * R, *cols = weights;
  float *squares = weights + (RESIDENT ? s.lds_floats() : s.hidden * (kColumns + 1));
  if (RESIDENT) read_weights(s, params, weights);
  float *mine = part + (uint64_t)blockIdx.x * (count + 1);
  auto input_of = [&](uint32_t l) { return act + (l == 0 ? 0 : (s.inputs + (l - 1) * s.hidden) * R); };
  bool first = true;
  for (uint64_t r0 = (uint64_t)blockIdx.x * R; r0 < n; r0 += (uint64_t)gridDim.x * R, first = false) {
    // rows past n stay zero in every layer: their errors are zero, and zero times
    // an activation that is not finite would not be
    const uint32_t rows = (uint32_t)min((uint64_t)R, n - r0);
    read_rows<R>(X, n, s.inputs, r0, act);
    __syncthreads();
    for (uint32_t l = 0; l <= s.layers; ++l) {
      dense<R, true>(layer_of<RESIDENT>(s, l, params, weights), s.fan_in(l), s.fan_out(l), l < s.layers, input_of(l),
                     l < s.layers ? input_of(l + 1) : GX, rows);
      __syncthreads();
    }
    // the output's error 2 (y - t) / n, and the squares
    if (threadIdx.x < R) {
      const bool row = r0 + threadIdx.x < n;
      const float d = row ? GX[threadIdx.x] - T[r0 + threadIdx.x] : 0.0f;
      G[threadIdx.x] = 2.0f * d / (float)n;
      squares[threadIdx.x] = d * d;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      float e = first ? 0.0f : mine[count];
      for (uint32_t r = 0; r < R; ++r) e += squares[r];
      mine[count] = e;
    }
    for (uint32_t l = s.layers + 1; l-- > 0;) {
      const uint32_t a = s.fan_in(l), b = s.fan_out(l);
      const Layer y = layer_of<RESIDENT>(s, l, params, weights);
      const float *in = input_of(l);
      // weights W[i][j] and, as row i = a, the biases
      uint32_t held = ~0u;
      float4 g[R / 4];
      const uint32_t di = blockDim.x / b, dj = blockDim.x % b;
      uint32_t i = threadIdx.x / b, j = threadIdx.x % b;
      for (uint32_t idx = threadIdx.x; idx < (a + 1) * b; idx += blockDim.x) {
        if (j != held) {
          held = j;
#pragma unroll
          for (uint32_t q = 0; q < R / 4; ++q) g[q] = *reinterpret_cast<const float4 *>(G + j * R + 4 * q);
        }
        float sum = 0.0f;
#pragma unroll
        for (uint32_t q = 0; q < R / 4; ++q) {
          const float4 x = i < a ? *reinterpret_cast<const float4 *>(in + i * R + 4 * q) : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
          sum += x.x * g[q].x;
          sum += x.y * g[q].y;
          sum += x.z * g[q].z;
          sum += x.w * g[q].w;
        }
        float *slot = mine + s.offset(l) + idx;
        *slot = first ? sum : *slot + sum;
        i += di;
        j += dj;
        if (j >= b) {
          j -= b;
          ++i;
        }
      }
      if (l == 0) break;
      // the layer input's error, through the ReLU of the layer below: GX[i][r] =
      // (in[i][r] > 0) * sum over j, in order, of G[j][r] W[i][j].  Threads take
      // consecutive i, whose weights lie a row apart: where they are not in LDS,
      // they come through it, kColumns columns at a time.
      const uint32_t step = RESIDENT ? b : kColumns;
      for (uint32_t j0 = 0; j0 < b; j0 += step) {
        const uint32_t nj = b - j0 < step ? b - j0 : step;
        if (!RESIDENT) {
          __syncthreads();
          constexpr uint32_t kInFlight = 16;
          for (uint32_t x0 = threadIdx.x; x0 < a * kColumns; x0 += kInFlight * blockDim.x) {
            float v[kInFlight];
#pragma unroll
            for (uint32_t k = 0; k < kInFlight; ++k) {
              const uint32_t idx = min(x0 + k * blockDim.x, a * kColumns - 1);
              v[k] = y.W[idx / kColumns * y.ld + j0 + min(idx % kColumns, nj - 1)];
            }
#pragma unroll
            for (uint32_t k = 0; k < kInFlight; ++k) {
              const uint32_t idx = x0 + k * blockDim.x;
              if (idx < a * kColumns) cols[idx / kColumns * (kColumns + 1) + idx % kColumns] = v[k];
            }
          }
          __syncthreads();
        }
        for (uint32_t idx = threadIdx.x; idx < a * (R / 4); idx += blockDim.x) {
          const uint32_t i = idx % a, q = 4 * (idx / a);
          const float *row = RESIDENT ? weights + s.lds_offset(l) + i * (b + 1) : cols + i * (kColumns + 1);
          float4 *gx = reinterpret_cast<float4 *>(GX + i * R + q);
          float4 acc = j0 == 0 ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : *gx;
          add_products<R>(acc, G + j0 * R + q, row, nj, 1);
          if (j0 + nj == b) {
            const float4 h = *reinterpret_cast<const float4 *>(in + i * R + q);
            acc = make_float4(h.x <= 0.0f ? 0.0f : acc.x, h.y <= 0.0f ? 0.0f : acc.y, h.z <= 0.0f ? 0.0f : acc.z,
                              h.w <= 0.0f ? 0.0f : acc.w);
          }
          *gx = acc;
        }
      }
      __syncthreads();
      float *t = G;
      G = GX;
      GX = t;
    }
    __syncthreads();
  }
}

// grad[k] = the sum of the workgroups' parts, four threads per parameter; the
// element past the last parameter is the loss.
__global__ void __launch_bounds__(256) mlp_sum_parts(const float *__restrict__ part, uint32_t groups, uint32_t count,
                                                     uint32_t n, float *__restrict__ grad, float *__restrict__ loss) {
  __shared__ float sums[4][64];
  const uint32_t lane = threadIdx.x % 64, seg = threadIdx.x / 64, k = blockIdx.x * 64 + lane;
  float sum = 0.0f;
  if (k <= count) {
#pragma unroll 8
    for (uint32_t g = seg; g < groups; g += 4) sum += part[(uint64_t)g * (count + 1) + k];
  }
  sums[seg][lane] = sum;
  __syncthreads();
  if (seg == 0 && k <= count) {
    const float all = (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
    if (k < count) grad[k] = all;
    else loss[0] = all / (float)n;
  }
}

// Adam (Kingma and Ba, 2015) with bias correction factors c1 = 1 - beta1^t,
// c2 = 1 - beta2^t computed on the host.
__global__ void adam_update(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                            float *__restrict__ v, uint32_t count, float lr, float beta1, float beta2, float eps,
                            float c1, float c2) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= count) return;
  const float gk = g[k];
  const float mk = beta1 * m[k] + (1.0f - beta1) * gk;
  const float vk = beta2 * v[k] + (1.0f - beta2) * gk * gk;
  m[k] = mk;
  v[k] = vk;
  p[k] -= lr * (mk / c1) / (sqrtf(vk / c2) + eps);
}

inline uint32_t blocks_for(uint64_t n, uint32_t threads) { return (uint32_t)((n + threads - 1) / threads); }

} // namespace

struct dd_mlp {
  Shape shape{};
  size_t count = 0;
  float *params = nullptr, *m = nullptr, *v = nullptr, *grad_tmp = nullptr;
  uint32_t step = 0;
  // parts of the gradient, one per workgroup, the losses of a training run, and
  // the outputs of a forward pass whose caller wants them inside its input
  float *part = nullptr, *losses = nullptr, *outputs = nullptr;
  uint32_t part_groups = 0, losses_cap = 0, outputs_cap = 0;

  ~dd_mlp() {
    for (float *p : {params, m, v, grad_tmp, part, losses, outputs}) (void)hipFree(p);
  }
};

namespace {

dd_status fail_mlp(dd_status s, const std::string &msg) {
  set_error(msg);
  return s;
}

#define MLP_HIP(call)                                                                                 \
  do {                                                                                                \
    hipError_t e_ = (call);                                                                           \
    if (e_ != hipSuccess) return fail_mlp(DD_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

// LDS of a gradient and of a forward pass over R rows per workgroup.
uint32_t gradient_lds(const Shape &s, uint32_t R, bool resident) {
  return 4 * ((s.inputs + s.layers * s.hidden + 2 * s.hidden + 1) * R +
              (resident ? s.lds_floats() : s.hidden * (kColumns + 1)));
}
uint32_t forward_lds(const Shape &s, uint32_t R, bool resident) {
  return 4 * ((std::max(s.inputs, s.hidden) + s.hidden) * R + (resident ? s.lds_floats() : 0));
}

// The weights are kept in LDS where 16 rows' activations fit beside them (up to
// three hidden layers of 64, or one of 100); else a workgroup takes four rows.
bool resident(const Shape &s) { return gradient_lds(s, 16, true) <= kResidentLds; }
uint32_t gradient_rows(const Shape &s) { return resident(s) ? 16 : 4; }

// The parts of all workgroups take at most kMaxParts floats, which networks of more
// than 262143 parameters reach below kMaxGroups.
uint32_t gradient_groups(const Shape &s, uint32_t n) {
  const uint32_t count = s.offset(s.layers) + s.hidden + 1;
  return std::min(blocks_for(n, gradient_rows(s)), std::min(kMaxGroups, kMaxParts / (count + 1)));
}

dd_status reserve(float *&p, uint32_t &have, uint32_t want, size_t each) {
  if (want <= have) return DD_OK;
  (void)hipFree(p);
  p = nullptr;
  have = 0;
  MLP_HIP(hipMalloc(reinterpret_cast<void **>(&p), (size_t)want * each * sizeof(float)));
  have = want;
  return DD_OK;
}

dd_status reserve_parts(dd_mlp *net, uint32_t n) {
  return reserve(net->part, net->part_groups, gradient_groups(net->shape, n), net->count + 1);
}

// Rows per workgroup of the forward pass.  Its weights are kept in LDS where the
// gradient's are and they fit; else a workgroup takes four rows.  Sixteen rows of up to
// 16 units are too little work for a workgroup: many rows go 64 at a time (200000 rows
// of 1 x 1 x 1 21.9 -> 8.6 us, of 5 x 8 x 1 26.6 -> 11.5, of 256 x 8 x 1 321 -> 210; one
// launch per layer 10.4, 16.0 and 206).
bool forward_resident(const Shape &s) { return resident(s) && forward_lds(s, 16, true) <= kResidentLds; }
uint32_t forward_rows(const Shape &s, uint32_t n) {
  if (!forward_resident(s)) return 4;
  return s.hidden <= 16 && n >= 64 * 1024 && forward_lds(s, 64, true) <= kHalfLds ? 64 : 16;
}

dd_status forward(dd_mlp *net, const float *d_x, uint32_t n, float *d_y, hipStream_t s) {
  const Shape &sh = net->shape;
  const uint32_t R = forward_rows(sh, n);
  auto kernel = R == 64 ? mlp_forward<64, true> : R == 16 ? mlp_forward<16, true> : mlp_forward<4, false>;
  hipLaunchKernelGGL(kernel, dim3(blocks_for(n, R)), dim3(256), forward_lds(sh, R, R != 4), s, sh, d_x, n, net->params, d_y);
  MLP_HIP(hipGetLastError());
  return DD_OK;
}

dd_status loss_grad(dd_mlp *net, const float *d_x, const float *d_t, uint32_t n, float *d_loss, float *d_grad,
                    hipStream_t s) {
  const Shape &sh = net->shape;
  const uint32_t groups = gradient_groups(sh, n);
  const bool keep = resident(sh);
  auto kernel = keep ? mlp_gradient<16, true> : mlp_gradient<4, false>;
  hipLaunchKernelGGL(kernel, dim3(groups), dim3(gradient_threads(keep)), gradient_lds(sh, gradient_rows(sh), keep), s, sh, d_x, d_t, n,
                     net->params, (uint32_t)net->count, net->part);
  MLP_HIP(hipGetLastError());
  hipLaunchKernelGGL(mlp_sum_parts, dim3(blocks_for(net->count + 1, 64)), dim3(256), 0, s, net->part, groups,
                     (uint32_t)net->count, n, d_grad, d_loss);
  MLP_HIP(hipGetLastError());
  return DD_OK;
}

dd_status adam(dd_mlp *net, const float *d_grad, float lr, hipStream_t s) {
  const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
  net->step += 1;
  const float c1 = 1.0f - (float)std::pow((double)beta1, (double)net->step);
  const float c2 = 1.0f - (float)std::pow((double)beta2, (double)net->step);
  hipLaunchKernelGGL(adam_update, dim3(blocks_for(net->count, 256)), dim3(256), 0, s, net->params, d_grad, net->m,
                     net->v, (uint32_t)net->count, lr, beta1, beta2, eps, c1, c2);
  MLP_HIP(hipGetLastError());
  return DD_OK;
}

} // namespace

extern "C" {

dd_status dd_mlp_create(dd_mlp **out, uint32_t inputs, uint32_t hidden, uint32_t hidden_layers) {
  if (!out) return fail_mlp(DD_ERR_INVALID_ARGUMENT, "null argument");
  *out = nullptr;
  if (inputs == 0 || inputs > kMaxWidth || hidden == 0 || hidden > kMaxWidth || hidden_layers == 0 ||
      hidden_layers > 8)
    return fail_mlp(DD_ERR_INVALID_ARGUMENT, "network shape out of range");
  dd_mlp *net = new dd_mlp();
  net->shape = Shape{inputs, hidden, hidden_layers};
  const size_t off = net->shape.offset(hidden_layers) + hidden + 1;
  net->count = off;
  hipError_t e = hipMalloc(reinterpret_cast<void **>(&net->params), off * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(&net->m), off * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(&net->v), off * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(&net->grad_tmp), off * sizeof(float));
  if (e == hipSuccess) e = hipMemset(net->params, 0, off * sizeof(float));
  if (e == hipSuccess) e = hipMemset(net->m, 0, off * sizeof(float));
  if (e == hipSuccess) e = hipMemset(net->v, 0, off * sizeof(float));
  if (e != hipSuccess) {
    delete net;
    return fail_mlp(DD_ERR_HIP, std::string("allocating the network: ") + hipGetErrorString(e));
  }
  *out = net;
  return DD_OK;
}

dd_status dd_mlp_destroy(dd_mlp *net) {
  delete net;
  return DD_OK;
}

dd_status dd_mlp_param_count(const dd_mlp *net, uint32_t *count) {
  if (!net || !count) return fail_mlp(DD_ERR_INVALID_ARGUMENT, "null argument");
  *count = (uint32_t)net->count;
  return DD_OK;
}

dd_status dd_mlp_set_params(dd_mlp *net, const float *params) {
  if (!net || !params) return fail_mlp(DD_ERR_INVALID_ARGUMENT, "null argument");
  MLP_HIP(hipMemcpy(net->params, params, net->count * sizeof(float), hipMemcpyHostToDevice));
  MLP_HIP(hipMemset(net->m, 0, net->count * sizeof(float)));
  MLP_HIP(hipMemset(net->v, 0, net->count * sizeof(float)));
  net->step = 0;
  return DD_OK;
}

dd_status dd_mlp_get_params(const dd_mlp *net, float *params) {
  if (!net || !params) return fail_mlp(DD_ERR_INVALID_ARGUMENT, "null argument");
  MLP_HIP(hipMemcpy(params, net->params, net->count * sizeof(float), hipMemcpyDeviceToHost));
  return DD_OK;
}

dd_status dd_mlp_init(dd_mlp *net, uint64_t seed) {
  if (!net) return fail_mlp(DD_ERR_INVALID_ARGUMENT, "null argument");
  // He-uniform weights (bound sqrt(6 / fan_in)), zero biases.
  std::mt19937_64 rng(seed);
  std::vector<float> p(net->count, 0.0f);
  for (uint32_t l = 0; l <= net->shape.layers; ++l) {
    const uint32_t a = net->shape.fan_in(l), b = net->shape.fan_out(l);
    const float bound = std::sqrt(6.0f / (float)a);
    std::uniform_real_distribution<float> u(-bound, bound);
    for (size_t k = 0; k < (size_t)a * b; ++k) p[net->shape.offset(l) + k] = u(rng);
  }
  return dd_mlp_set_params(net, p.data());
}

dd_status dd_mlp_forward(dd_mlp *net, const float *d_x, uint32_t n, float *d_y, void *stream) {
  if (!net || !d_x || !d_y) return fail_mlp(DD_ERR_INVALID_ARGUMENT, "null argument");
  if (n == 0) return DD_OK;
  // A workgroup stores its rows' outputs while others still read their inputs, so
  // outputs inside the input are written once the pass is over.
  const uintptr_t x0 = reinterpret_cast<uintptr_t>(d_x), x1 = x0 + (size_t)n * net->shape.inputs * sizeof(float);
  const uintptr_t y0 = reinterpret_cast<uintptr_t>(d_y), y1 = y0 + (size_t)n * sizeof(float);
  if (y1 <= x0 || x1 <= y0) return forward(net, d_x, n, d_y, (hipStream_t)stream);
  dd_status s = reserve(net->outputs, net->outputs_cap, n, 1);
  if (s == DD_OK) s = forward(net, d_x, n, net->outputs, (hipStream_t)stream);
  if (s != DD_OK) return s;
  MLP_HIP(hipMemcpyAsync(d_y, net->outputs, (size_t)n * sizeof(float), hipMemcpyDeviceToDevice, (hipStream_t)stream));
  return DD_OK;
}

dd_status dd_mlp_loss_grad(dd_mlp *net, const float *d_x, const float *d_target, uint32_t n, float *d_loss,
                           float *d_grad, void *stream) {
  if (!net || !d_x || !d_target || !d_loss || !d_grad || n == 0)
    return fail_mlp(DD_ERR_INVALID_ARGUMENT, "invalid argument");
  dd_status s = reserve_parts(net, n);
  return s != DD_OK ? s : loss_grad(net, d_x, d_target, n, d_loss, d_grad, (hipStream_t)stream);
}

dd_status dd_mlp_adam_step(dd_mlp *net, const float *d_grad, float lr, void *stream) {
  if (!net || !d_grad) return fail_mlp(DD_ERR_INVALID_ARGUMENT, "null argument");
  return adam(net, d_grad, lr, (hipStream_t)stream);
}

dd_status dd_mlp_train(dd_mlp *net, const float *d_x, const float *d_target, uint32_t n, uint32_t steps, float lr,
                       float *losses, void *stream) {
  if (!net || !d_x || !d_target || n == 0) return fail_mlp(DD_ERR_INVALID_ARGUMENT, "invalid argument");
  dd_status s = reserve_parts(net, n);
  // the losses stay on the device until the run is over
  if (s == DD_OK) s = reserve(net->losses, net->losses_cap, std::max(steps, 1u), 1);
  if (s != DD_OK) return s;
  hipStream_t st = (hipStream_t)stream;
  for (uint32_t k = 0; k < steps; ++k) {
    s = loss_grad(net, d_x, d_target, n, net->losses + k, net->grad_tmp, st);
    if (s == DD_OK) s = adam(net, net->grad_tmp, lr, st);
    if (s != DD_OK) return s;
  }
  if (losses && steps)
    MLP_HIP(hipMemcpyAsync(losses, net->losses, (size_t)steps * sizeof(float), hipMemcpyDeviceToHost, st));
  MLP_HIP(hipStreamSynchronize(st));
  return DD_OK;
}

} // extern "C"
