// Cost-model MLP on the GPU: a 3-layer perceptron (in -> H -> H -> 1, ReLU,
// FP32) trained with mean-squared error and Adam by this file's own forward
// and backward kernels. It maps features of a part to its predicted kernel
// time; the planner uses it to choose the part width.
//
// Parameter layout (one flat FP32 array, as hsv_mlp_get_params returns it):
//   W1[in][H] | b1[H] | W2[H][H] | b2[H] | W3[H] | b3
// Forward:  a1 = relu(X W1 + b1); a2 = relu(a1 W2 + b2); y = a2 W3 + b3.
// Every reduction runs in a fixed order, so training is deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/hsv.h"

void hsv_set_last_error(const std::string& msg);

namespace {

int mfail(int code, const std::string& m) {
  hsv_set_last_error(m);
  return code;
}
#define MCHK(expr)                                                                     \
  do {                                                                                 \
    hipError_t e_ = (expr);                                                            \
    if (e_ != hipSuccess) return mfail(HSV_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

typedef float v4f __attribute__((ext_vector_type(4)));

// The three contractions of a layer on the FP32 matrix cores, one 16x16
// result tile per wave, the operands read straight from L2 (a layer of the
// cost model is 14..64 wide: every array but the samples stays cached).
// v_mfma_f32_16x16x4_f32: lane l holds A[l%16][l/16] and B[l/16][l%16], result
// item i is D[4*(l/16) + i][l%16]; FP32 products and accumulation. Entries
// outside a matrix are read as 0 and never stored.
//
// What bounds them is latency: a wave's loads and its chain of K/4 MFMAs.
// So a contraction over many samples is split until about kMlpWaves waves
// are in flight. Measured at 6000 samples, 14-64-64-1, against one thread
// per result element: weight gradients of the three layers 38 us
// against 4390 us, forward 17 us against 31 us, input gradients 14 us
// against 52 us.
constexpr int kMlpWaves = 2048;       // wanted in flight: 2 per SIMD
constexpr int kMlpMinSlice = 32;      // samples per slice: 8 MFMAs to one store
constexpr int kMlpBlock = 256;

struct Mat {  // element (row, col) at p[row * rs + col * cs]
  const float* p;
  int rs, cs;
};

// acc += A[m0..m0+15][k0..k1) * B[k0..k1)[n0..n0+15]. ONES: row M - 1 of A is
// all ones (the bias of a weight gradient).
template <bool ONES>
__device__ __forceinline__ v4f mlp_tile(const Mat& A, const Mat& B, int m0, int n0, int k0, int k1, int M, int N,
                                        v4f acc) {
  const int lane = threadIdx.x & 63;
  const int m = m0 + (lane & 15), n = n0 + (lane & 15), g = lane >> 4;
  const bool one = ONES && m == M - 1;
  const bool am = m < M && !one, bn = n < N;
  for (int kb = k0; kb < k1; kb += 16) {  // 16 at a time: eight loads in flight per lane
    float a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = kb + 4 * u + g;
      const bool in = k < k1;
      a[u] = one && in ? 1.0f : 0.0f;
      b[u] = 0.0f;
      if (am && in) a[u] = A.p[(size_t)m * A.rs + (size_t)k * A.cs];
      if (bn && in) b[u] = B.p[(size_t)k * B.rs + (size_t)n * B.cs];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b[u], acc, 0, 0, 0);
  }
  return acc;
}

// Y[n][o] = act(b[o] + sum_i X[n][i] W[i][o])
__global__ __launch_bounds__(kMlpBlock) void k_linear_fwd(const float* __restrict__ X, const float* __restrict__ W,
                                                          const float* __restrict__ b, float* __restrict__ Y, int N,
                                                          int I, int O, int relu) {
  const int to = (O + 15) / 16, tn = (N + 15) / 16;
  const int t = blockIdx.x * (kMlpBlock / 64) + (threadIdx.x >> 6);
  if (t >= to * tn) return;
  const int lane = threadIdx.x & 63, n0 = t / to * 16, o0 = t % to * 16, o = o0 + (lane & 15);
  const float bias = o < O ? b[o] : 0.0f;
  v4f acc = {bias, bias, bias, bias};
  acc = mlp_tile<false>(Mat{X, I, 1}, Mat{W, O, 1}, n0, o0, 0, I, N, O, acc);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = n0 + 4 * (lane >> 4) + i;
    if (n < N && o < O) Y[(size_t)n * O + o] = relu ? fmaxf(acc[i], 0.0f) : acc[i];
  }
}

// dX[n][i] = (sum_o dY[n][o] W[i][o]) * (A[n][i] > 0), A = the layer input's
// post-ReLU activation (mask = 1 when A is the network input).
__global__ __launch_bounds__(kMlpBlock) void k_linear_bwd_in(const float* __restrict__ dY, const float* __restrict__ W,
                                                             const float* __restrict__ A, float* __restrict__ dX,
                                                             int N, int I, int O, int relu_mask) {
  const int ti = (I + 15) / 16, tn = (N + 15) / 16;
  const int t = blockIdx.x * (kMlpBlock / 64) + (threadIdx.x >> 6);
  if (t >= ti * tn) return;
  const int lane = threadIdx.x & 63, n0 = t / ti * 16, i0 = t % ti * 16, c = i0 + (lane & 15);
  v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
  acc = mlp_tile<false>(Mat{dY, O, 1}, Mat{W, 1, O}, n0, i0, 0, O, N, I, acc);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = n0 + 4 * (lane >> 4) + i;
    if (n >= N || c >= I) continue;
    const size_t at = (size_t)n * I + c;
    dX[at] = (relu_mask && !(A[at] > 0.0f)) ? 0.0f : acc[i];
  }
}

// dW[i][o] = sum_n X[n][i] dY[n][o], and db[o] = sum_n dY[n][o] as row I (the
// parameter layout puts a layer's bias behind its weights): the samples
// [slice * per, +per) of one result tile per wave. out: the gradient itself
// with one slice, else part[slice][(I + 1) * O].
__global__ __launch_bounds__(kMlpBlock) void k_linear_bwd_w(const float* __restrict__ X, const float* __restrict__ dY,
                                                            float* __restrict__ out, int N, int I, int O, int per,
                                                            int slices) {
  const int ti = (I + 1 + 15) / 16, to = (O + 15) / 16;
  const int t = blockIdx.x * (kMlpBlock / 64) + (threadIdx.x >> 6);
  if (t >= ti * to * slices) return;
  const int s = t / (ti * to), r = t % (ti * to), i0 = r / to * 16, o0 = r % to * 16;
  const int n0 = s * per, n1 = min(N, n0 + per), lane = threadIdx.x & 63, o = o0 + (lane & 15);
  v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
  acc = mlp_tile<true>(Mat{X, 1, I}, Mat{dY, O, 1}, i0, o0, n0, n1, I + 1, O, acc);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = i0 + 4 * (lane >> 4) + j;
    if (i <= I && o < O) out[(size_t)s * (I + 1) * O + (size_t)i * O + o] = acc[j];
  }
}

// the slices' partial gradients, added in order
__global__ __launch_bounds__(kMlpBlock) void k_slice_sum(const float* __restrict__ part, float* __restrict__ g, int P,
                                                         int slices) {
  const int t = blockIdx.x * kMlpBlock + threadIdx.x;
  if (t >= P) return;
  float acc = part[t];
#pragma unroll 8
  for (int s = 1; s < slices; ++s) acc += part[(size_t)s * P + t];
  g[t] = acc;
}

// d = 2 (y - target) / N and the per-sample squared error
__global__ void k_mse_grad(const float* __restrict__ y, const float* __restrict__ target, float* __restrict__ d,
                           float* __restrict__ sq, int N) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const float e = y[n] - target[n];
  d[n] = 2.0f * e / (float)N;
  sq[n] = e * e;
}

__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, int P, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P) return;
  const float gi = g[t];
  m[t] = b1 * m[t] + (1.0f - b1) * gi;
  v[t] = b2 * v[t] + (1.0f - b2) * gi * gi;
  const float mh = m[t] / c1, vh = v[t] / c2;
  w[t] -= lr * mh / (sqrtf(vh) + eps);
}

inline int blocks(long long n, int bs = 256) { return (int)((n + bs - 1) / bs); }

}  // namespace

struct hsv_mlp {
  int in = 0, H = 0;
  size_t P = 0;
  float* w = nullptr;   // parameters; the four arrays below lie behind them
  float* g = nullptr;   // gradients (same layout)
  float* m = nullptr;   // Adam moments
  float* v = nullptr;
  float* part = nullptr;  // partial weight gradients of a layer's sample slices
  int step = 0;
  // activations / scratch for up to cap samples
  int cap = 0;
  float *X = nullptr, *T = nullptr, *a1 = nullptr, *a2 = nullptr, *y = nullptr;
  float *d1 = nullptr, *d2 = nullptr, *d3 = nullptr, *sq = nullptr;
  hipStream_t stream = nullptr;
  size_t off_b1() const { return (size_t)in * H; }
  size_t off_W2() const { return off_b1() + H; }
  size_t off_b2() const { return off_W2() + (size_t)H * H; }
  size_t off_W3() const { return off_b2() + H; }
  size_t off_b3() const { return off_W3() + H; }
};

namespace {

void free_scratch(hsv_mlp* m) {
  float** bufs[] = {&m->X, &m->T, &m->a1, &m->a2, &m->y, &m->d1, &m->d2, &m->d3, &m->sq};
  for (float** b : bufs) {
    if (*b) (void)hipFree(*b);
    *b = nullptr;
  }
  m->cap = 0;
}

int ensure_cap(hsv_mlp* m, int n) {
  if (n <= m->cap) return HSV_OK;
  free_scratch(m);
  const size_t N = (size_t)n;
  struct { float** p; size_t cnt; } want[] = {{&m->X, N * m->in}, {&m->T, N}, {&m->a1, N * m->H}, {&m->a2, N * m->H},
                                              {&m->y, N}, {&m->d1, N * m->H}, {&m->d2, N * m->H}, {&m->d3, N},
                                              {&m->sq, N}};
  for (auto& w : want)
    if (hipMalloc(reinterpret_cast<void**>(w.p), std::max<size_t>(w.cnt, 1) * sizeof(float)) != hipSuccess)
      return mfail(HSV_ERR_ALLOC, "MLP scratch allocation failed");
  m->cap = n;
  return HSV_OK;
}

inline int tiles16(int n) { return (n + 15) / 16; }

void linear_fwd(hsv_mlp* m, const float* X, const float* W, const float* b, float* Y, int n, int I, int O, int relu) {
  hipLaunchKernelGGL(k_linear_fwd, blocks((long long)tiles16(n) * tiles16(O), kMlpBlock / 64), kMlpBlock, 0, m->stream,
                     X, W, b, Y, n, I, O, relu);
}

void linear_bwd_in(hsv_mlp* m, const float* dY, const float* W, const float* A, float* dX, int n, int I, int O) {
  hipLaunchKernelGGL(k_linear_bwd_in, blocks((long long)tiles16(n) * tiles16(I), kMlpBlock / 64), kMlpBlock, 0,
                     m->stream, dY, W, A, dX, n, I, O, 1);
}

// g: the layer's weights and, behind them, its bias. Slices of the samples
// until kMlpWaves waves are in flight; kMlpMinSlice samples at least, so that
// a slice's work is worth its store. slices * tiles <= kMlpWaves bounds the
// partials by kMlpPart floats; a layer with more tiles than that takes one
// slice and writes the gradient itself.
constexpr size_t kMlpPart = size_t(kMlpWaves) * 256;
void linear_bwd_w(hsv_mlp* m, const float* X, const float* dY, float* g, int n, int I, int O) {
  const long long tiles = (long long)tiles16(I + 1) * tiles16(O);
  const long long want = std::max<long long>(1, std::min<long long>(kMlpWaves / tiles, (n + kMlpMinSlice - 1) / kMlpMinSlice));
  const int per = (int)(((n + want - 1) / want + 15) / 16 * 16);
  const int slices = (n + per - 1) / per, P = (I + 1) * O;
  hipLaunchKernelGGL(k_linear_bwd_w, blocks(tiles * slices, kMlpBlock / 64), kMlpBlock, 0, m->stream, X, dY,
                     slices > 1 ? m->part : g, n, I, O, per, slices);
  if (slices > 1)
    hipLaunchKernelGGL(k_slice_sum, blocks(P, kMlpBlock), kMlpBlock, 0, m->stream, m->part, g, P, slices);
}

void forward(hsv_mlp* m, int n, const float* Xd) {
  const float* w = m->w;
  linear_fwd(m, Xd, w, w + m->off_b1(), m->a1, n, m->in, m->H, 1);
  linear_fwd(m, m->a1, w + m->off_W2(), w + m->off_b2(), m->a2, n, m->H, m->H, 1);
  linear_fwd(m, m->a2, w + m->off_W3(), w + m->off_b3(), m->y, n, m->H, 1, 0);
}

void backward(hsv_mlp* m, int n, const float* Xd, const float* Td) {
  const float* w = m->w;
  float* g = m->g;
  hipLaunchKernelGGL(k_mse_grad, blocks(n), 256, 0, m->stream, m->y, Td, m->d3, m->sq, n);
  // layer 3: y = a2 W3 + b3
  linear_bwd_w(m, m->a2, m->d3, g + m->off_W3(), n, m->H, 1);
  linear_bwd_in(m, m->d3, w + m->off_W3(), m->a2, m->d2, n, m->H, 1);
  // layer 2: a2 = relu(a1 W2 + b2)
  linear_bwd_w(m, m->a1, m->d2, g + m->off_W2(), n, m->H, m->H);
  linear_bwd_in(m, m->d2, w + m->off_W2(), m->a1, m->d1, n, m->H, m->H);
  // layer 1: a1 = relu(X W1 + b1)
  linear_bwd_w(m, Xd, m->d1, g, n, m->in, m->H);
}

}  // namespace

extern "C" {

int hsv_mlp_create(int in_features, int hidden, uint64_t seed, hsv_mlp** out) {
  if (!out || in_features < 1 || in_features > 256 || hidden < 1 || hidden > 1024)
    return mfail(HSV_ERR_ARG, "bad MLP shape");
  *out = nullptr;
  auto* m = new hsv_mlp();
  m->in = in_features;
  m->H = hidden;
  m->P = (size_t)in_features * hidden + hidden + (size_t)hidden * hidden + hidden + hidden + 1;
  if (hipStreamCreate(&m->stream) != hipSuccess) { delete m; return mfail(HSV_ERR_DEVICE, "stream"); }
  // parameters, gradients, Adam moments and slice partials in one allocation
  if (hipMalloc(reinterpret_cast<void**>(&m->w), (4 * m->P + kMlpPart) * sizeof(float)) != hipSuccess) {
    hsv_mlp_destroy(m);
    return mfail(HSV_ERR_ALLOC, "MLP parameter allocation failed");
  }
  m->g = m->w + m->P;
  m->m = m->g + m->P;
  m->v = m->m + m->P;
  m->part = m->v + m->P;
  // He-uniform initialisation from a splitmix64 stream, zero biases
  std::vector<float> h(4 * m->P, 0.0f);  // gradients and moments start at zero
  uint64_t s = seed ? seed : 0x9E3779B97F4A7C15ull;
  auto uni = [&]() {
    s += 0x9E3779B97F4A7C15ull;
    uint64_t z = s;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) / 9007199254740992.0 * 2.0 - 1.0;
  };
  const double a1 = std::sqrt(6.0 / in_features), a2 = std::sqrt(6.0 / hidden);
  for (size_t i = 0; i < (size_t)in_features * hidden; ++i) h[i] = (float)(a1 * uni());
  for (size_t i = 0; i < (size_t)hidden * hidden; ++i) h[m->off_W2() + i] = (float)(a2 * uni());
  for (int i = 0; i < hidden; ++i) h[m->off_W3() + i] = (float)(a2 * uni());
  MCHK(hipMemcpy(m->w, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice));
  *out = m;
  return HSV_OK;
}

int hsv_mlp_destroy(hsv_mlp* m) {
  if (!m) return HSV_OK;
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  free_scratch(m);
  if (m->w) (void)hipFree(m->w);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return HSV_OK;
}

int hsv_mlp_num_params(hsv_mlp* m, uint64_t* count) {
  if (!m || !count) return mfail(HSV_ERR_ARG, "null argument");
  *count = m->P;
  return HSV_OK;
}

int hsv_mlp_get_params(hsv_mlp* m, float* out) {
  if (!m || !out) return mfail(HSV_ERR_ARG, "null argument");
  MCHK(hipMemcpyAsync(out, m->w, m->P * sizeof(float), hipMemcpyDeviceToHost, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  return HSV_OK;
}

int hsv_mlp_set_params(hsv_mlp* m, const float* in) {
  if (!m || !in) return mfail(HSV_ERR_ARG, "null argument");
  MCHK(hipMemcpyAsync(m->w, in, m->P * sizeof(float), hipMemcpyHostToDevice, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  m->step = 0;
  return HSV_OK;
}

int hsv_mlp_forward(hsv_mlp* m, const float* X, int n, float* y_out) {
  if (!m || n < 0 || (n && (!X || !y_out))) return mfail(HSV_ERR_ARG, "bad arguments");
  if (!n) return HSV_OK;
  if (int rc = ensure_cap(m, n)) return rc;
  MCHK(hipMemcpyAsync(m->X, X, sizeof(float) * n * m->in, hipMemcpyHostToDevice, m->stream));
  forward(m, n, m->X);
  MCHK(hipGetLastError());
  MCHK(hipMemcpyAsync(y_out, m->y, sizeof(float) * n, hipMemcpyDeviceToHost, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  return HSV_OK;
}

// Forward + backward on (X, target); the mean squared error in *loss and,
// when grads_out is not null, the gradient of every parameter.
int hsv_mlp_gradient(hsv_mlp* m, const float* X, const float* target, int n, float* loss, float* grads_out) {
  if (!m || n <= 0 || !X || !target) return mfail(HSV_ERR_ARG, "bad arguments");
  if (int rc = ensure_cap(m, n)) return rc;
  MCHK(hipMemcpyAsync(m->X, X, sizeof(float) * n * m->in, hipMemcpyHostToDevice, m->stream));
  MCHK(hipMemcpyAsync(m->T, target, sizeof(float) * n, hipMemcpyHostToDevice, m->stream));
  forward(m, n, m->X);
  backward(m, n, m->X, m->T);
  MCHK(hipGetLastError());
  if (loss) {
    std::vector<float> sq(n);
    MCHK(hipMemcpyAsync(sq.data(), m->sq, sizeof(float) * n, hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    double s = 0;
    for (float x : sq) s += x;
    *loss = (float)(s / n);
  }
  if (grads_out) {
    MCHK(hipMemcpyAsync(grads_out, m->g, m->P * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
  }
  return HSV_OK;
}

// Full-batch Adam for `epochs` steps over mini-batches of `batch` samples
// taken in order (the caller shuffles). Final mean squared error in *loss.
int hsv_mlp_train(hsv_mlp* m, const float* X, const float* target, int n, int epochs, int batch, float lr,
                  float* loss) {
  if (!m || n <= 0 || !X || !target || epochs < 0 || batch <= 0 || !(lr > 0))
    return mfail(HSV_ERR_ARG, "bad arguments");
  const int nb = std::min(batch, n);
  if (int rc = ensure_cap(m, nb)) return rc;
  // the whole training set goes to the device once
  float *Xall = nullptr, *Tall = nullptr;
  if (hipMalloc(reinterpret_cast<void**>(&Xall), sizeof(float) * (size_t)n * m->in) != hipSuccess ||
      hipMalloc(reinterpret_cast<void**>(&Tall), sizeof(float) * (size_t)n) != hipSuccess) {
    if (Xall) (void)hipFree(Xall);
    return mfail(HSV_ERR_ALLOC, "training set allocation failed");
  }
  MCHK(hipMemcpyAsync(Xall, X, sizeof(float) * (size_t)n * m->in, hipMemcpyHostToDevice, m->stream));
  MCHK(hipMemcpyAsync(Tall, target, sizeof(float) * (size_t)n, hipMemcpyHostToDevice, m->stream));
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (int e = 0; e < epochs; ++e) {
    for (int s0 = 0; s0 < n; s0 += nb) {
      const int cnt = std::min(nb, n - s0);
      forward(m, cnt, Xall + (size_t)s0 * m->in);
      backward(m, cnt, Xall + (size_t)s0 * m->in, Tall + s0);
      ++m->step;
      const float c1 = 1.0f - std::pow(b1, (float)m->step), c2 = 1.0f - std::pow(b2, (float)m->step);
      hipLaunchKernelGGL(k_adam, blocks((long long)m->P), 256, 0, m->stream, m->w, m->g, m->m, m->v, (int)m->P, lr,
                         b1, b2, eps, c1, c2);
    }
  }
  (void)hipStreamSynchronize(m->stream);
  (void)hipFree(Xall);
  (void)hipFree(Tall);
  MCHK(hipGetLastError());
  MCHK(hipStreamSynchronize(m->stream));
  if (loss) {
    float l = 0;
    if (int rc = hsv_mlp_gradient(m, X, target, std::min(n, 65536), &l, nullptr)) return rc;
    *loss = l;
  }
  return HSV_OK;
}

}  // extern "C"
