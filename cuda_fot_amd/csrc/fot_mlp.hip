// fot_mlp.hip -- the learned cost model: a small FP32 MLP
// (in -> hidden -> hidden -> out, ReLU) trained and evaluated on the GPU by
// hand-written kernels.  Every matrix product runs on the matrix cores
// (v_mfma_f32_16x16x4_f32, one 16x16 tile per workgroup, K split across its
// waves); bias, ReLU, the masked MSE gradient and Adam are elementwise
// kernels.  A training step of a network that fits one workgroup's LDS (the
// cost model's does) is two launches instead: mlp_step_kernel and
// mlp_update_kernel.  No reference counterpart.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "fot_hip.hpp"

using fot::fail;

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

// C[m][n] = sum_k A(m,k) B(k,n) (+ bias[n]) (ReLU), with A(m,k) =
// A[m*sam + k*sak] and B(k,n) = B[k*sbk + n*sbn]: any transpose through the
// strides.  One 16x16 tile of C per workgroup of kGemmWaves waves; wave w
// takes the K steps w, w + kGemmWaves, ... (four k each), so a long K (the
// weight gradients reduce over the whole batch) is split across the waves,
// and the partial tiles are summed in wave order through LDS.
// MFMA 16x16x4 f32 operand layout: lane l supplies A(i = l%16, k = l/16) and
// B(k = l/16, j = l%16); its four results are C(4*(l/16) + v, l%16).
constexpr uint32_t kGemmWaves = 8;

__global__ __launch_bounds__(64 * kGemmWaves) void gemm_mfma_kernel(
    const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C,
    const float *__restrict__ bias, uint32_t M, uint32_t N, uint32_t K, uint32_t sam,
    uint32_t sak, uint32_t sbk, uint32_t sbn, uint32_t ldc, int relu, int accumulate) {
  __shared__ v4f part[kGemmWaves][64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t m0 = blockIdx.x * 16u, n0 = blockIdx.y * 16u;
  const uint32_t r = lane & 15u, q = lane >> 4;
  const uint32_t am = m0 + r, bn = n0 + r;
  v4f acc = {0.f, 0.f, 0.f, 0.f};
  for (uint32_t k0 = 4u * wave; k0 < K; k0 += 4u * kGemmWaves) {
    const uint32_t k = k0 + q;
    const float a = (am < M && k < K) ? A[size_t(am) * sam + size_t(k) * sak] : 0.f;
    const float b = (bn < N && k < K) ? B[size_t(k) * sbk + size_t(bn) * sbn] : 0.f;
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
  }
  part[wave][lane] = acc;
  __syncthreads();
  if (wave != 0) return;
  v4f sum = part[0][lane];
#pragma unroll
  for (uint32_t w = 1; w < kGemmWaves; ++w) sum += part[w][lane];
  const uint32_t col = n0 + r;
  if (col >= N) return;
  const float bb = bias ? bias[col] : 0.f;
#pragma unroll
  for (uint32_t v = 0; v < 4; ++v) {
    const uint32_t row = m0 + 4u * q + v;
    if (row >= M) continue;
    float x = sum[v] + bb;
    if (relu) x = x > 0.f ? x : 0.f;
    float *c = C + size_t(row) * ldc + col;
    *c = accumulate ? *c + x : x;
  }
}

// dY = 2 (Y - T) mask / count; per-block partial sums of mask (Y - T)^2
__global__ __launch_bounds__(256) void mse_grad_kernel(const float *__restrict__ Y,
                                                       const float *__restrict__ T,
                                                       const float *__restrict__ mask,
                                                       float *__restrict__ dY, uint32_t n,
                                                       float inv_count,
                                                       float *__restrict__ partial) {
  __shared__ float s[256];
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  float l = 0.f;
  if (i < n) {
    const float w = mask ? mask[i] : 1.f;
    const float e = (Y[i] - T[i]) * w;
    dY[i] = 2.f * e * inv_count;
    l = e * (Y[i] - T[i]);
  }
  s[threadIdx.x] = l;
  __syncthreads();
  for (uint32_t o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// dZ = dH * (Z > 0) in place on dH (Z is the pre-activation's output after
// ReLU: H > 0 exactly where Z > 0)
__global__ __launch_bounds__(256) void relu_grad_kernel(float *__restrict__ dH,
                                                        const float *__restrict__ H, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n && !(H[i] > 0.f)) dH[i] = 0.f;
}

// column sums: db[j] = sum_i dZ[i][j]
__global__ __launch_bounds__(256) void colsum_kernel(const float *__restrict__ dZ,
                                                     float *__restrict__ db, uint32_t rows,
                                                     uint32_t cols) {
  __shared__ float s[256];
  const uint32_t j = blockIdx.x;
  float acc = 0.f;
  for (uint32_t i = threadIdx.x; i < rows; i += 256) acc += dZ[size_t(i) * cols + j];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (uint32_t o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) db[j] = s[0];
}

// Adam (Kingma & Ba 2015) with bias correction folded into the step size
__global__ __launch_bounds__(256) void adam_kernel(float *__restrict__ p, const float *__restrict__ g,
                                                   float *__restrict__ m, float *__restrict__ v,
                                                   uint32_t n, float lr_t, float b1, float b2,
                                                   float eps, float wd) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i] + wd * p[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi, v[i] = vi;
  p[i] -= lr_t * mi / (sqrtf(vi) + eps);
}

// ---- a training step in two launches --------------------------------------
// Layer by layer a step is 16 launches of 2-6 us each for 25 MFLOP, and the
// loss read back every epoch drains the queue: 113 us per epoch at 695 rows
// of 24 -> 64 -> 64 -> 6, all of it latency.  Here the whole network sits in
// one workgroup's LDS (63 KB) and a workgroup carries a tile of 16 rows
// through the forward pass, the loss and the backward pass without leaving
// it; its parts of the weight gradients stay in MFMA accumulators over all its
// tiles and are stored once.  A second launch sums the workgroups' parts and
// applies Adam: 9.5 + 3.8 us per epoch at 695 rows (44 workgroups), bound by
// the chain of loads, products and barriers, and 20 epochs as one call 2216 ->
// 350 us.
constexpr uint32_t kStepWidth = 64;   // most inputs and hidden units
constexpr uint32_t kStepOutputs = 16; // most outputs
constexpr uint32_t kStepRows = 16;    // rows of a tile (one MFMA tile's)
// at most one workgroup per CU: beyond 4096 rows a workgroup takes several
// tiles, so the gradient parts stay under 256 x the parameters
constexpr uint32_t kStepBlocks = 256;
// LDS row stride: lanes l of an operand read word (l % 16) * 68 + l / 16, 64
// different banks
constexpr uint32_t kStepStride = kStepWidth + 4;

struct MlpShape {
  uint32_t I, H, O;
  __host__ __device__ uint32_t b1() const { return H * I; }
  __host__ __device__ uint32_t w2() const { return b1() + H; }
  __host__ __device__ uint32_t b2() const { return w2() + H * H; }
  __host__ __device__ uint32_t w3() const { return b2() + H; }
  __host__ __device__ uint32_t b3() const { return w3() + O * H; }
  __host__ __device__ uint32_t params() const { return b3() + O; }
};

// dst[row][col] (stride kStepStride) = src[row][col], zero outside rows x cols
template <uint32_t ROWS>
__device__ __forceinline__ void step_load(float *dst, const float *__restrict__ src, uint32_t rows,
                                          uint32_t cols, uint32_t t) {
  float v[ROWS / 4];
#pragma unroll
  for (uint32_t i = 0; i < ROWS / 4; ++i) {
    const uint32_t r = (t >> 6) + 4 * i, c = t & 63u;
    v[i] = (r < rows && c < cols) ? src[size_t(r) * cols + c] : 0.f;
  }
#pragma unroll
  for (uint32_t i = 0; i < ROWS / 4; ++i) dst[((t >> 6) + 4 * i) * kStepStride + (t & 63u)] = v[i];
}

// acc += A B over k < K (a multiple of 4), A(i,k) = a[i * sai + k * sak] and
// B(k,j) = b[k * sbk + j * sbj] in LDS, zero-padded to whole tiles
template <uint32_t K>
__device__ __forceinline__ v4f step_mfma(v4f acc, const float *a, uint32_t sai, uint32_t sak,
                                         const float *b, uint32_t sbk, uint32_t sbj,
                                         uint32_t lane) {
  const float *pa = a + (lane & 15u) * sai + (lane >> 4) * sak;
  const float *pb = b + (lane & 15u) * sbj + (lane >> 4) * sbk;
  // two chains, so that one product's latency hides the other's
  v4f odd = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (uint32_t k = 0; k < K; k += 8) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[k * sak], pb[k * sbk], acc, 0, 0, 0);
    if (k + 4 < K)
      odd = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[(k + 4) * sak], pb[(k + 4) * sbk], odd, 0, 0,
                                                 0);
  }
  return acc + odd;
}

// the sum of a C tile's column, in every lane of the column
__device__ __forceinline__ float step_colsum(const float *v) {
  float s = (v[0] + v[1]) + (v[2] + v[3]);
  s += __shfl_xor(s, 16);
  s += __shfl_xor(s, 32);
  return s;
}

// Forward, loss and backward of the rows of tiles blockIdx.x, + gridDim.x,
// ...; part[blockIdx.x][params] gets the workgroup's sums of the gradients,
// loss_part[blockIdx.x] its sum of mask (y - t)^2.  Four waves; wave w owns
// columns 16 w .. 16 w + 15 of each layer.  Rows past the end carry zeros
// through every layer, whatever the biases are: their products with the zero
// gradients must not be 0 x infinity.  IN: the inputs
// rounded up to 32 or 64 (half the first layer's products at 24 inputs).
template <uint32_t IN>
__global__ __launch_bounds__(256) void mlp_step_kernel(MlpShape s, const float *__restrict__ p,
                                                       const float *__restrict__ X,
                                                       const float *__restrict__ T,
                                                       const float *__restrict__ mask,
                                                       uint32_t rows, float inv_count,
                                                       float *__restrict__ part,
                                                       double *__restrict__ loss_part) {
  constexpr uint32_t S = kStepStride, W = kStepWidth;
  __shared__ float w1[W * S], w2[W * S], w3[kStepOutputs * S];
  __shared__ float xs[kStepRows * S], h1[kStepRows * S], h2[kStepRows * S];
  __shared__ float d1[kStepRows * S], d2[kStepRows * S], dy[kStepRows * 20];
  __shared__ double wave_loss[4];
  const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6, r = lane & 15u, q = lane >> 4;
  const uint32_t col = 16 * w + r; // this lane's column of a hidden layer
  step_load<W>(w1, p, s.H, s.I, t);
  step_load<W>(w2, p + s.w2(), s.H, s.H, t);
  step_load<kStepOutputs>(w3, p + s.w3(), s.O, s.H, t);
  const float b1 = col < s.H ? p[s.b1() + col] : 0.f, b2 = col < s.H ? p[s.b2() + col] : 0.f;
  const uint32_t yr = t >> 4, yc = t & 15u; // this thread's output value
  const float b3 = yc < s.O ? p[s.b3() + yc] : 0.f;
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
  v4f g1[IN / 16], g2[4] = {zero, zero, zero, zero}, g3 = zero;
#pragma unroll
  for (uint32_t j = 0; j < IN / 16; ++j) g1[j] = zero;
  float gb1 = 0.f, gb2 = 0.f, gb3 = 0.f;
  double loss = 0.0; // as many FP32 terms per thread as tiles: summed in FP64
  for (uint32_t row0 = blockIdx.x * kStepRows; row0 < rows; row0 += gridDim.x * kStepRows) {
    const uint32_t n = min(kStepRows, rows - row0);
    step_load<kStepRows>(xs, X + size_t(row0) * s.I, n, s.I, t);
    const size_t yi = size_t(row0 + yr) * s.O + yc;
    const bool live = yr < n && yc < s.O;
    const float target = live ? T[yi] : 0.f, weight = live ? (mask ? mask[yi] : 1.f) : 0.f;
    __syncthreads();
    v4f a = step_mfma<IN>(zero, xs, S, 1, w1 + 16 * w * S, 1, S, lane);
#pragma unroll
    for (uint32_t v = 0; v < 4; ++v) {
      const float z = a[v] + b1;
      h1[(4 * q + v) * S + col] = z > 0.f && 4 * q + v < n ? z : 0.f;
    }
    __syncthreads();
    a = step_mfma<W>(zero, h1, S, 1, w2 + 16 * w * S, 1, S, lane);
#pragma unroll
    for (uint32_t v = 0; v < 4; ++v) {
      const float z = a[v] + b2;
      h2[(4 * q + v) * S + col] = z > 0.f && 4 * q + v < n ? z : 0.f;
    }
    __syncthreads();
    // the one output tile: each wave a quarter of its sum, through d1
    a = step_mfma<W / 4>(zero, h2 + 16 * w, S, 1, w3 + 16 * w, 1, S, lane);
#pragma unroll
    for (uint32_t v = 0; v < 4; ++v) d1[w * 256 + (4 * q + v) * 16 + r] = a[v];
    __syncthreads();
    const float y = ((d1[t] + d1[256 + t]) + (d1[512 + t] + d1[768 + t])) + b3;
    const float e = live ? (y - target) * weight : 0.f;
    if (live) loss += e * (y - target);
    dy[yr * 20 + yc] = 2.f * e * inv_count;
    __syncthreads();
    a = step_mfma<kStepOutputs>(zero, dy, 20, 1, w3 + 16 * w, S, 1, lane);
    float dz[4];
#pragma unroll
    for (uint32_t v = 0; v < 4; ++v) {
      const uint32_t row = 4 * q + v;
      dz[v] = (row < n && h2[row * S + col] > 0.f) ? a[v] : 0.f;
      d2[row * S + col] = dz[v];
    }
    gb2 += step_colsum(dz);
    g3 = step_mfma<kStepRows>(g3, dy, 1, 20, h2 + 16 * w, S, 1, lane);
    if (w == 0) gb3 += step_colsum((const float[4]){dy[(4 * q) * 20 + r], dy[(4 * q + 1) * 20 + r],
                                                    dy[(4 * q + 2) * 20 + r],
                                                    dy[(4 * q + 3) * 20 + r]});
    __syncthreads();
    a = step_mfma<W>(zero, d2, S, 1, w2 + 16 * w, S, 1, lane);
#pragma unroll
    for (uint32_t v = 0; v < 4; ++v) {
      const uint32_t row = 4 * q + v;
      dz[v] = (row < n && h1[row * S + col] > 0.f) ? a[v] : 0.f;
      d1[row * S + col] = dz[v];
    }
    gb1 += step_colsum(dz);
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
      g2[j] = step_mfma<kStepRows>(g2[j], d2 + 16 * w, 1, S, h1 + 16 * j, S, 1, lane);
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < IN / 16; ++j)
      g1[j] = step_mfma<kStepRows>(g1[j], d1 + 16 * w, 1, S, xs + 16 * j, S, 1, lane);
    __syncthreads(); // xs, h1 and d1 are free for the next tile
  }
  float *g = part + size_t(blockIdx.x) * s.params();
#pragma unroll
  for (uint32_t v = 0; v < 4; ++v) {
    const uint32_t row = 16 * w + 4 * q + v; // g1, g2: this wave's 16 rows
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t c = 16 * j + r;
      if (j < IN / 16 && row < s.H && c < s.I) g[row * s.I + c] = g1[j][v];
      if (row < s.H && c < s.H) g[s.w2() + row * s.H + c] = g2[j][v];
    }
    if (4 * q + v < s.O && col < s.H) g[s.w3() + (4 * q + v) * s.H + col] = g3[v];
  }
  if (q == 0 && col < s.H) g[s.b1() + col] = gb1, g[s.b2() + col] = gb2;
  if (w == 0 && q == 0 && r < s.O) g[s.b3() + r] = gb3;
#pragma unroll
  for (uint32_t o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o);
  if (lane == 0) wave_loss[w] = loss;
  __syncthreads();
  if (t == 0)
    loss_part[blockIdx.x] = (wave_loss[0] + wave_loss[1]) + (wave_loss[2] + wave_loss[3]);
}

// Sums the workgroups' gradient parts (in FP64, four slices of them per
// parameter) and either applies Adam or, with grad, stores the sums; the last
// workgroup also sums the loss.  64 parameters per workgroup.
__global__ __launch_bounds__(256) void mlp_update_kernel(
    float *__restrict__ p, float *__restrict__ m, float *__restrict__ v,
    const float *__restrict__ part, const double *__restrict__ loss_part, uint32_t n,
    uint32_t parts, float lr_t, float b1, float b2, float eps, float wd, float count,
    float *__restrict__ grad, float *__restrict__ loss) {
  __shared__ double sum[256];
  const uint32_t t = threadIdx.x, i = blockIdx.x * 64u + (t & 63u);
  const uint32_t at = min(i, n - 1);
  const float pi = p[at], m0 = m[at], v0 = v[at];
  double acc = 0.0;
#pragma unroll 8
  for (uint32_t j = t >> 6; j < parts; j += 4) acc += double(part[size_t(j) * n + at]);
  sum[t] = acc;
  __syncthreads();
  if (t < 64 && i < n) {
    const float g0 = float((sum[t] + sum[t + 64]) + (sum[t + 128] + sum[t + 192]));
    if (grad) {
      grad[i] = g0;
    } else {
      const float gi = g0 + wd * pi;
      const float mi = b1 * m0 + (1.f - b1) * gi;
      const float vi = b2 * v0 + (1.f - b2) * gi * gi;
      m[i] = mi, v[i] = vi;
      p[i] = pi - lr_t * mi / (sqrtf(vi) + eps);
    }
  }
  if (!loss || blockIdx.x + 1 != gridDim.x) return;
  __syncthreads();
  sum[t] = t < parts ? loss_part[t] : 0.0; // parts <= kStepBlocks
  __syncthreads();
  for (uint32_t o = 128; o > 0; o >>= 1) {
    if (t < o) sum[t] += sum[t + o];
    __syncthreads();
  }
  if (t == 0) *loss = float(sum[0] / count);
}

uint32_t cdiv(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// C (MxN) = op(A) op(B) through strides; see gemm_mfma_kernel
fot_status gemm(const float *A, const float *B, float *C, const float *bias, uint32_t M,
                uint32_t N, uint32_t K, uint32_t sam, uint32_t sak, uint32_t sbk, uint32_t sbn,
                uint32_t ldc, bool relu, bool accumulate, hipStream_t s) {
  if (M == 0 || N == 0) return FOT_OK;
  hipLaunchKernelGGL(gemm_mfma_kernel, dim3(cdiv(M, 16), cdiv(N, 16)), dim3(64 * kGemmWaves), 0, s,
                     A, B, C,
                     bias, M, N, K, sam, sak, sbk, sbn, ldc, relu ? 1 : 0, accumulate ? 1 : 0);
  FOT_HIP(hipGetLastError());
  return FOT_OK;
}

struct SplitMix {
  uint64_t s;
  uint64_t next() {
    uint64_t z = (s += 0x9e3779b97f4a7c15ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
  }
  double uniform() { return double(next() >> 11) * 0x1.0p-53; }
};

} // namespace

// parameter layout (flat, row-major): W1 [H][I], b1 [H], W2 [H][H], b2 [H],
// W3 [O][H], b3 [O]
struct fot_mlp {
  int device = 0; // the device holding the parameters
  uint32_t I = 0, H = 0, O = 0;
  size_t nparam = 0;
  size_t off_w1 = 0, off_b1 = 0, off_w2 = 0, off_b2 = 0, off_w3 = 0, off_b3 = 0;
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
  // activations for up to `cap` rows: X, H1, H2, Y, T, mask, dY, dH2, dH1, partials
  uint32_t cap = 0;
  float *X = nullptr, *H1 = nullptr, *H2 = nullptr, *Y = nullptr, *T = nullptr, *Mk = nullptr;
  float *dY = nullptr, *dH2 = nullptr, *dH1 = nullptr, *part = nullptr;
  // two-launch training steps: gradient and loss parts of the workgroups, the
  // epochs' losses
  float *gpart = nullptr, *losses = nullptr;
  double *lpart = nullptr;
  uint32_t gcap = 0, lcap = 0;
  uint64_t step = 0;
  std::vector<void *> owned;

  ~fot_mlp() {
    for (void *q : owned) (void)hipFree(q);
  }
  template <class T> fot_status alloc(T **q, size_t n) {
    void *r = nullptr;
    FOT_HIP(hipMalloc(&r, std::max<size_t>(1, n) * sizeof(T)));
    owned.push_back(r);
    *q = static_cast<T *>(r);
    return FOT_OK;
  }
  fot_status reserve(uint32_t rows) {
    if (rows <= cap) return FOT_OK;
    for (float **q : {&X, &H1, &H2, &Y, &T, &Mk, &dY, &dH2, &dH1, &part}) {
      if (*q) {
        owned.erase(std::find(owned.begin(), owned.end(), static_cast<void *>(*q)));
        (void)hipFree(*q);
        *q = nullptr;
      }
    }
    const size_t r = rows;
    fot_status st;
    if ((st = alloc(&X, r * I)) || (st = alloc(&H1, r * H)) || (st = alloc(&H2, r * H)) ||
        (st = alloc(&Y, r * O)) || (st = alloc(&T, r * O)) || (st = alloc(&Mk, r * O)) ||
        (st = alloc(&dY, r * O)) || (st = alloc(&dH2, r * H)) || (st = alloc(&dH1, r * H)) ||
        (st = alloc(&part, cdiv(uint32_t(r * O), 256) + 1)))
      return st;
    cap = rows;
    return FOT_OK;
  }
  // forward over `rows` rows of x (device) through the hidden activations
  // h1, h2 (rows x H each) into y
  fot_status forward_into(const float *x, float *h1, float *h2, float *y, uint32_t rows,
                          hipStream_t s) const {
    fot_status st;
    if ((st = gemm(x, p + off_w1, h1, p + off_b1, rows, H, I, I, 1, 1, I, H, true, false, s)))
      return st;
    if ((st = gemm(h1, p + off_w2, h2, p + off_b2, rows, H, H, H, 1, 1, H, H, true, false, s)))
      return st;
    return gemm(h2, p + off_w3, y, p + off_b3, rows, O, H, H, 1, 1, H, O, false, false, s);
  }
  fot_status forward(uint32_t rows, hipStream_t s) { return forward_into(X, H1, H2, Y, rows, s); }
  // gradients of the masked MSE into g; returns the loss
  fot_status backward(uint32_t rows, bool masked, float count, float *loss, hipStream_t s) {
    const uint32_t n = rows * O, nb = cdiv(n, 256);
    hipLaunchKernelGGL(mse_grad_kernel, dim3(nb), dim3(256), 0, s, Y, T, masked ? Mk : nullptr,
                       dY, n, 1.f / count, part);
    FOT_HIP(hipGetLastError());
    fot_status st;
    // layer 3: dW3 = dY^T H2, db3 = colsum dY, dH2 = dY W3
    if ((st = gemm(dY, H2, g + off_w3, nullptr, O, H, rows, 1, O, H, 1, H, false, false, s)))
      return st;
    hipLaunchKernelGGL(colsum_kernel, dim3(O), dim3(256), 0, s, dY, g + off_b3, rows, O);
    if ((st = gemm(dY, p + off_w3, dH2, nullptr, rows, H, O, O, 1, H, 1, H, false, false, s)))
      return st;
    hipLaunchKernelGGL(relu_grad_kernel, dim3(cdiv(rows * H, 256)), dim3(256), 0, s, dH2, H2,
                       rows * H);
    // layer 2
    if ((st = gemm(dH2, H1, g + off_w2, nullptr, H, H, rows, 1, H, H, 1, H, false, false, s)))
      return st;
    hipLaunchKernelGGL(colsum_kernel, dim3(H), dim3(256), 0, s, dH2, g + off_b2, rows, H);
    if ((st = gemm(dH2, p + off_w2, dH1, nullptr, rows, H, H, H, 1, H, 1, H, false, false, s)))
      return st;
    hipLaunchKernelGGL(relu_grad_kernel, dim3(cdiv(rows * H, 256)), dim3(256), 0, s, dH1, H1,
                       rows * H);
    // layer 1
    if ((st = gemm(dH1, X, g + off_w1, nullptr, H, I, rows, 1, H, I, 1, I, false, false, s)))
      return st;
    hipLaunchKernelGGL(colsum_kernel, dim3(H), dim3(256), 0, s, dH1, g + off_b1, rows, H);
    FOT_HIP(hipGetLastError());
    if (loss) {
      std::vector<float> h(nb);
      FOT_HIP(hipMemcpyAsync(h.data(), part, nb * sizeof(float), hipMemcpyDeviceToHost, s));
      FOT_HIP(hipStreamSynchronize(s));
      double acc = 0;
      for (float x : h) acc += x;
      *loss = float(acc / count);
    }
    return FOT_OK;
  }
  // Whether a training step runs as two launches: the network fits the LDS of
  // mlp_step_kernel.  Wider networks go layer by layer.
  bool fits_step() const { return I <= kStepWidth && H <= kStepWidth && O <= kStepOutputs; }
  fot_status resize(float **q, uint32_t *have, uint32_t want, size_t each) {
    if (want <= *have) return FOT_OK;
    if (*q) {
      owned.erase(std::find(owned.begin(), owned.end(), static_cast<void *>(*q)));
      (void)hipFree(*q);
      *q = nullptr;
      *have = 0;
    }
    if (fot_status st = alloc(q, want * each)) return st;
    *have = want;
    return FOT_OK;
  }
  fot_status reserve_step(uint32_t rows, uint32_t epochs) {
    fot_status st;
    if (!lpart && (st = alloc(&lpart, kStepBlocks))) return st;
    if ((st = resize(&gpart, &gcap, step_blocks(rows), nparam))) return st;
    return resize(&losses, &lcap, epochs, 1);
  }
  static uint32_t step_blocks(uint32_t rows) { return std::min(cdiv(rows, kStepRows), kStepBlocks); }
  // One step over the loaded rows (reserve_step first): Adam with lr_t, or the
  // gradient into g when `gradient`; the loss into losses[e] when wanted.
  fot_status fused_step(uint32_t rows, bool masked, float count, bool gradient, float lr_t,
                        float b1, float b2, float eps, float wd, bool want_loss, uint32_t e,
                        hipStream_t s) {
    const uint32_t nb = step_blocks(rows), n = uint32_t(nparam);
    hipLaunchKernelGGL(I <= 32 ? mlp_step_kernel<32> : mlp_step_kernel<64>, dim3(nb), dim3(256), 0,
                       s, (MlpShape{I, H, O}), p, X, T, masked ? Mk : nullptr, rows, 1.f / count,
                       gpart, lpart);
    hipLaunchKernelGGL(mlp_update_kernel, dim3(cdiv(n, 64)), dim3(256), 0, s, p, m, v, gpart,
                       lpart, n, nb, lr_t, b1, b2, eps, wd, count, gradient ? g : nullptr,
                       want_loss ? losses + e : nullptr);
    FOT_HIP(hipGetLastError());
    return FOT_OK;
  }
  fot_status load_rows(const float *x, const float *t, const float *mask, uint32_t rows) {
    if (fot_status st = reserve(rows)) return st;
    FOT_HIP(hipMemcpy(X, x, sizeof(float) * rows * I, hipMemcpyHostToDevice));
    if (t) FOT_HIP(hipMemcpy(T, t, sizeof(float) * rows * O, hipMemcpyHostToDevice));
    if (mask) FOT_HIP(hipMemcpy(Mk, mask, sizeof(float) * rows * O, hipMemcpyHostToDevice));
    return FOT_OK;
  }
};

static float mask_count(const float *mask, size_t n) {
  if (!mask) return float(n);
  double c = 0;
  for (size_t i = 0; i < n; ++i) c += mask[i];
  return float(std::max(c, 1.0));
}

static fot_status fot_mlp_create_impl(uint32_t in, uint32_t hidden, uint32_t out, uint64_t seed,
                                     fot_mlp **mlp) {
  if (!mlp || in == 0 || hidden == 0 || out == 0 || in > 4096 || hidden > 4096 || out > 4096)
    return fail(FOT_ERR_INVALID_ARGUMENT, "bad MLP shape");
  *mlp = nullptr;
  std::unique_ptr<fot_mlp> M(new fot_mlp);
  FOT_HIP(hipGetDevice(&M->device));
  M->I = in, M->H = hidden, M->O = out;
  M->off_w1 = 0;
  M->off_b1 = M->off_w1 + size_t(hidden) * in;
  M->off_w2 = M->off_b1 + hidden;
  M->off_b2 = M->off_w2 + size_t(hidden) * hidden;
  M->off_w3 = M->off_b2 + hidden;
  M->off_b3 = M->off_w3 + size_t(out) * hidden;
  M->nparam = M->off_b3 + out;
  fot_status st;
  if ((st = M->alloc(&M->p, M->nparam)) || (st = M->alloc(&M->g, M->nparam)) ||
      (st = M->alloc(&M->m, M->nparam)) || (st = M->alloc(&M->v, M->nparam)))
    return st;
  // He-uniform weights (fan in), zero biases
  std::vector<float> h(M->nparam, 0.f);
  SplitMix r{seed};
  auto init = [&](size_t off, uint32_t rows, uint32_t fan_in) {
    const double a = std::sqrt(6.0 / fan_in);
    for (size_t i = 0; i < size_t(rows) * fan_in; ++i) h[off + i] = float((2 * r.uniform() - 1) * a);
  };
  init(M->off_w1, hidden, in);
  init(M->off_w2, hidden, hidden);
  init(M->off_w3, out, hidden);
  FOT_HIP(hipMemcpy(M->p, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice));
  FOT_HIP(hipMemset(M->m, 0, M->nparam * sizeof(float)));
  FOT_HIP(hipMemset(M->v, 0, M->nparam * sizeof(float)));
  *mlp = M.release();
  return FOT_OK;
}
extern "C" fot_status fot_mlp_create(uint32_t in, uint32_t hidden, uint32_t out, uint64_t seed,
                                     fot_mlp **mlp) {
  return fot::guarded("fot_mlp_create", [&] {
    return fot_mlp_create_impl(in, hidden, out, seed, mlp);
  });
}

static fot_status fot_mlp_destroy_impl(fot_mlp *mlp) {
  delete mlp;
  return FOT_OK;
}
extern "C" fot_status fot_mlp_destroy(fot_mlp *mlp) {
  return fot::guarded("fot_mlp_destroy", [&] { return fot_mlp_destroy_impl(mlp); });
}

static fot_status fot_mlp_num_params_impl(const fot_mlp *mlp, uint64_t *n) {
  if (!mlp || !n) return fail(FOT_ERR_INVALID_ARGUMENT, "null argument");
  *n = mlp->nparam;
  return FOT_OK;
}
extern "C" fot_status fot_mlp_num_params(const fot_mlp *mlp, uint64_t *n) {
  return fot::guarded("fot_mlp_num_params", [&] { return fot_mlp_num_params_impl(mlp, n); });
}

static fot_status fot_mlp_get_params_impl(const fot_mlp *mlp, float *host, uint64_t n) {
  if (!mlp || !host || n != mlp->nparam) return fail(FOT_ERR_INVALID_ARGUMENT, "bad params");
  FOT_HIP(hipMemcpy(host, mlp->p, n * sizeof(float), hipMemcpyDeviceToHost));
  return FOT_OK;
}
extern "C" fot_status fot_mlp_get_params(const fot_mlp *mlp, float *host, uint64_t n) {
  return fot::guarded("fot_mlp_get_params", [&] { return fot_mlp_get_params_impl(mlp, host, n); });
}

static fot_status fot_mlp_set_params_impl(fot_mlp *mlp, const float *host, uint64_t n) {
  if (!mlp || !host || n != mlp->nparam) return fail(FOT_ERR_INVALID_ARGUMENT, "bad params");
  FOT_HIP(hipMemcpy(mlp->p, host, n * sizeof(float), hipMemcpyHostToDevice));
  FOT_HIP(hipMemset(mlp->m, 0, mlp->nparam * sizeof(float)));
  FOT_HIP(hipMemset(mlp->v, 0, mlp->nparam * sizeof(float)));
  mlp->step = 0;
  return FOT_OK;
}
extern "C" fot_status fot_mlp_set_params(fot_mlp *mlp, const float *host, uint64_t n) {
  return fot::guarded("fot_mlp_set_params", [&] { return fot_mlp_set_params_impl(mlp, host, n); });
}

static fot_status fot_mlp_forward_impl(fot_mlp *mlp, const float *x, uint32_t rows, float *y) {
  if (!mlp || !x || !y) return fail(FOT_ERR_INVALID_ARGUMENT, "null argument");
  if (rows == 0) return FOT_OK;
  fot_status st;
  if ((st = mlp->load_rows(x, nullptr, nullptr, rows))) return st;
  if ((st = mlp->forward(rows, nullptr))) return st;
  FOT_HIP(hipMemcpy(y, mlp->Y, sizeof(float) * rows * mlp->O, hipMemcpyDeviceToHost));
  return FOT_OK;
}
extern "C" fot_status fot_mlp_forward(fot_mlp *mlp, const float *x, uint32_t rows, float *y) {
  return fot::guarded("fot_mlp_forward", [&] { return fot_mlp_forward_impl(mlp, x, rows, y); });
}

// ---- inference that allocates nothing ------------------------------------
// The two hidden activations of one fot_mlp_forward_noalloc call live in a
// fixed device array instead of buffers the library allocates: each device
// holds its own copy from first use until the process ends.  Host code never
// uses the array's name as an address (on the host it is a stand-in, not
// device memory); it uses the address hipGetSymbolAddress returns for the
// current device, looked up once per device on the entry point's first call
// there.
constexpr size_t kNoAllocScratchFloats = size_t(1) << 20; // 4 MiB per device
static __device__ __align__(256) float scratch[kNoAllocScratchFloats];

constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static float *g_scratch_ptr[kMaxScratchDevices] = {};

static fot_status scratch_of_current_device(float **out) {
  int dev = 0;
  FOT_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxScratchDevices)
    return fail(FOT_ERR_UNSUPPORTED, "device %d beyond the %d scratch slots", dev,
                kMaxScratchDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *q = nullptr;
    const hipError_t e = hipGetSymbolAddress(&q, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !q)
      return fail(FOT_ERR_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = static_cast<float *>(q);
  }
  *out = g_scratch_ptr[dev];
  return FOT_OK;
}

static fot_status fot_mlp_forward_noalloc_impl(const fot_mlp *mlp, const float *x,
                                              uint32_t rows, float *y, void *stream) {
  if (!mlp) return fail(FOT_ERR_INVALID_ARGUMENT, "null MLP");
  if (rows == 0) return FOT_OK;
  if (!x || !y) return fail(FOT_ERR_INVALID_ARGUMENT, "null device buffer");
  if (2 * uint64_t(rows) * mlp->H > kNoAllocScratchFloats)
    return fail(FOT_ERR_INVALID_ARGUMENT,
                "rows %u x hidden %u needs %llu activation floats; the scratch holds %zu "
                "(at most %llu rows)",
                rows, mlp->H, (unsigned long long)(2 * uint64_t(rows) * mlp->H),
                kNoAllocScratchFloats,
                (unsigned long long)(kNoAllocScratchFloats / (2 * uint64_t(mlp->H))));
  int dev = 0;
  FOT_HIP(hipGetDevice(&dev));
  if (dev != mlp->device)
    return fail(FOT_ERR_INVALID_ARGUMENT, "current device %d, the MLP lives on device %d", dev,
                mlp->device);
  float *h = nullptr;
  if (fot_status st = scratch_of_current_device(&h)) return st;
  // every element of both activations is written before it is read: no
  // clearing needed
  return mlp->forward_into(x, h, h + size_t(rows) * mlp->H, y, rows,
                           static_cast<hipStream_t>(stream));
}
extern "C" fot_status fot_mlp_forward_noalloc(const fot_mlp *mlp, const float *x, uint32_t rows,
                                              float *y, void *stream) {
  return fot::guarded("fot_mlp_forward_noalloc", [&] {
    return fot_mlp_forward_noalloc_impl(mlp, x, rows, y, stream);
  });
}

static fot_status fot_mlp_loss_grad_impl(fot_mlp *mlp, const float *x, const float *t,
                                        const float *mask, uint32_t rows, float *loss,
                                        float *grad) {
  if (!mlp || !x || !t || !loss || !grad || rows == 0)
    return fail(FOT_ERR_INVALID_ARGUMENT, "null argument");
  fot_status st;
  if ((st = mlp->load_rows(x, t, mask, rows))) return st;
  const float count = mask_count(mask, size_t(rows) * mlp->O);
  if (mlp->fits_step()) {
    if ((st = mlp->reserve_step(rows, 1))) return st;
    if ((st = mlp->fused_step(rows, mask != nullptr, count, true, 0.f, 0.f, 0.f, 0.f, 0.f, true, 0,
                              nullptr)))
      return st;
    FOT_HIP(hipMemcpy(loss, mlp->losses, sizeof(float), hipMemcpyDeviceToHost));
  } else {
    if ((st = mlp->forward(rows, nullptr))) return st;
    if ((st = mlp->backward(rows, mask != nullptr, count, loss, nullptr))) return st;
  }
  FOT_HIP(hipMemcpy(grad, mlp->g, mlp->nparam * sizeof(float), hipMemcpyDeviceToHost));
  return FOT_OK;
}
extern "C" fot_status fot_mlp_loss_grad(fot_mlp *mlp, const float *x, const float *t,
                                        const float *mask, uint32_t rows, float *loss,
                                        float *grad) {
  return fot::guarded("fot_mlp_loss_grad", [&] {
    return fot_mlp_loss_grad_impl(mlp, x, t, mask, rows, loss, grad);
  });
}

static fot_status fot_mlp_train_impl(fot_mlp *mlp, const float *x, const float *t,
                                    const float *mask, uint32_t rows, uint32_t epochs, float lr,
                                    float weight_decay, float *loss_per_epoch) {
  if (!mlp || !x || !t || rows == 0) return fail(FOT_ERR_INVALID_ARGUMENT, "null argument");
  fot_status st;
  if ((st = mlp->load_rows(x, t, mask, rows))) return st;
  const float count = mask_count(mask, size_t(rows) * mlp->O);
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const bool fused = mlp->fits_step();
  if (fused && (st = mlp->reserve_step(rows, loss_per_epoch ? epochs : 0))) return st;
  for (uint32_t e = 0; e < epochs; ++e) {
    if (!fused) {
      if ((st = mlp->forward(rows, nullptr))) return st;
      float l = 0;
      if ((st = mlp->backward(rows, mask != nullptr, count, loss_per_epoch ? &l : nullptr,
                              nullptr)))
        return st;
      if (loss_per_epoch) loss_per_epoch[e] = l;
    }
    ++mlp->step;
    const double c1 = 1.0 - std::pow(double(b1), double(mlp->step));
    const double c2 = 1.0 - std::pow(double(b2), double(mlp->step));
    const float lr_t = float(lr * std::sqrt(c2) / c1);
    if (fused) {
      if ((st = mlp->fused_step(rows, mask != nullptr, count, false, lr_t, b1, b2, eps,
                                weight_decay, loss_per_epoch != nullptr, e, nullptr)))
        return st;
      continue;
    }
    hipLaunchKernelGGL(adam_kernel, dim3(cdiv(uint32_t(mlp->nparam), 256)), dim3(256), 0, nullptr,
                       mlp->p, mlp->g, mlp->m, mlp->v, uint32_t(mlp->nparam), lr_t, b1, b2, eps,
                       weight_decay);
    FOT_HIP(hipGetLastError());
  }
  FOT_HIP(hipDeviceSynchronize());
  if (fused && loss_per_epoch && epochs)
    FOT_HIP(hipMemcpy(loss_per_epoch, mlp->losses, sizeof(float) * epochs, hipMemcpyDeviceToHost));
  return FOT_OK;
}
extern "C" fot_status fot_mlp_train(fot_mlp *mlp, const float *x, const float *t,
                                    const float *mask, uint32_t rows, uint32_t epochs, float lr,
                                    float weight_decay, float *loss_per_epoch) {
  return fot::guarded("fot_mlp_train", [&] {
    return fot_mlp_train_impl(mlp, x, t, mask, rows, epochs, lr, weight_decay, loss_per_epoch);
  });
}

// The MFMA GEMM on device buffers: C[M][N] = op(A) op(B) with row-major A
// (M x K, or K x M when trans_a) and B (K x N, or N x K when trans_b).
static fot_status fot_gemm_f32_impl(const float *A, const float *B, float *C, uint32_t M,
                                   uint32_t N, uint32_t K, int trans_a, int trans_b,
                                   void *stream) {
  if ((!A || !B || !C) && M && N) return fail(FOT_ERR_INVALID_ARGUMENT, "null matrix");
  const uint32_t sam = trans_a ? 1 : K, sak = trans_a ? M : 1;
  const uint32_t sbk = trans_b ? 1 : N, sbn = trans_b ? K : 1;
  return gemm(A, B, C, nullptr, M, N, K, sam, sak, sbk, sbn, N, false, false,
              static_cast<hipStream_t>(stream));
}
extern "C" fot_status fot_gemm_f32(const float *A, const float *B, float *C, uint32_t M,
                                   uint32_t N, uint32_t K, int trans_a, int trans_b,
                                   void *stream) {
  return fot::guarded("fot_gemm_f32", [&] {
    return fot_gemm_f32_impl(A, B, C, M, N, K, trans_a, trans_b, stream);
  });
}
