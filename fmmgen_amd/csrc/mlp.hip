// Kernels of the order-selection network (layout and semantics in mlp.h).
#include "mlp.h"

#include <mutex>

namespace fmm {
namespace {

constexpr int F = kMlpF, H = kMlpH, O = kMlpO;

__device__ __forceinline__ void stage_params(const float* __restrict__ P, float* sP) {
  for (int i = threadIdx.x; i < kMlpParams; i += blockDim.x) sP[i] = P[i];
  __syncthreads();
}

// Forward pass, one thread per sample.
__global__ __launch_bounds__(64) void k_mlp_fwd(int B, const float* __restrict__ X, const float* __restrict__ P,
                                                float* __restrict__ Y) {
  __shared__ float sP[kMlpParams];
  stage_params(P, sP);
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  float x[F], h1[H], h2[H];
#pragma unroll
  for (int f = 0; f < F; ++f) x[f] = X[(size_t)b * F + f];
#pragma unroll
  for (int j = 0; j < H; ++j) {
    float a = sP[kMlpB1 + j];
#pragma unroll
    for (int f = 0; f < F; ++f) a += sP[kMlpW1 + j * F + f] * x[f];
    h1[j] = a > 0.f ? a : 0.f;
  }
#pragma unroll
  for (int j = 0; j < H; ++j) {
    float a = sP[kMlpB2 + j];
#pragma unroll
    for (int i = 0; i < H; ++i) a += sP[kMlpW2 + j * H + i] * h1[i];
    h2[j] = a > 0.f ? a : 0.f;
  }
#pragma unroll
  for (int o = 0; o < O; ++o) {
    float a = sP[kMlpB3 + o];
#pragma unroll
    for (int i = 0; i < H; ++i) a += sP[kMlpW3 + o * H + i] * h2[i];
    Y[(size_t)b * O + o] = a;
  }
}

// Gradient of the masked mean-square loss: forward, backward and weight
// gradients of 16 samples at a time on the FP32 matrix cores (16x16x4), one
// block of 4 waves per run of sample tiles, every product a 16-row tile.
//   forward   H1 = relu(X W1^T + b1), H2 = relu(H1 W2^T + b2), Y = H2 W3^T + b3
//             (wave w: hidden units 16w .. 16w + 15; the 11 outputs: wave 0)
//   backward  D2 = (dY W3) [H2 > 0], D1 = (D2 W2) [H1 > 0]
//   weights   dW3 += dY^T H2, dW2 += D2^T H1, dW1 += D1^T X, in accumulators
//             that stay in registers over the block's tiles
// dY is the unscaled error; the block's sums, its loss and its count of valid
// outputs go to its row of `part`, and k_mlp_grad_sum adds the rows in a fixed
// order and scales by 2 / count, so the gradient and the loss are the same on
// every run.  A grid of one block finishes by itself and needs no `part`.
// The work is 0.07 GFLOP at 2048 samples: launches and the chain of a block
// bound it, so the batch is spread over many blocks and takes two launches.
// One thread per weight summing the whole batch took 2230 us at 2048 samples
// (three launches), with a forward and a backward of one thread per sample
// another 85 us; the call went from 2299 to 19 us, its error against FP64 from
// 5.6e-7 to 1.1e-7.
// Operand layout of the 16x16x4 MFMA: lane l holds A[l%16][l/16],
// B[l/16][l%16] and rows 4 (l/16) + r of column l%16 of the result.
constexpr int kGradWaves = 4;
constexpr int kOP = 16;  // outputs padded to a tile
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__global__ __launch_bounds__(64 * kGradWaves) void k_mlp_grad(int B, int per, const float* __restrict__ X,
                                                              const float* __restrict__ T,
                                                              const float* __restrict__ mask,
                                                              const float* __restrict__ P, float* __restrict__ part,
                                                              float* __restrict__ grad, float* __restrict__ loss) {
  constexpr int HS = H + 1, FS = F + 1, XS = 17;  // odd row strides: conflict-free column reads
  static_assert(kGradWaves * 16 == H && F % 4 == 0 && O < kOP, "one wave per 16 hidden units");
  __shared__ float sW1[H * FS], sW2[H * HS], sW3[kOP * HS], sb1[H], sb2[H], sb3[kOP];
  __shared__ float sX[16 * XS], sH1[16 * HS], sH2[16 * HS], sY[16 * XS], sD2[16 * HS], sD1[16 * HS];
  __shared__ float red[2][64 * kGradWaves];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = lane & 15, q = lane >> 4;
  constexpr int NT = 64 * kGradWaves;
  for (int i = tid; i < H * F; i += NT) sW1[(i / F) * FS + i % F] = P[kMlpW1 + i];
  for (int i = tid; i < H * H; i += NT) sW2[(i / H) * HS + i % H] = P[kMlpW2 + i];
  for (int i = tid; i < kOP * H; i += NT) sW3[(i / H) * HS + i % H] = i < O * H ? P[kMlpW3 + i] : 0.f;
  if (tid < H) {
    sb1[tid] = P[kMlpB1 + tid];
    sb2[tid] = P[kMlpB2 + tid];
  }
  if (tid < kOP) sb3[tid] = tid < O ? P[kMlpB3 + tid] : 0.f;
  f32x4 g1 = {0, 0, 0, 0}, g3 = {0, 0, 0, 0}, g2[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
  float gb = 0.f, lsum = 0.f, cnt = 0.f;  // gb: a bias sum of threads 0 .. 2H + O - 1
  const int j = 16 * w + c;               // this lane's hidden unit (column)
  const int s0 = blockIdx.x * per * kGradTile;
  for (int t = 0; t < per; ++t) {
    const int base = s0 + t * kGradTile;
    if (base >= B) break;  // uniform over the block
    __syncthreads();       // parameters staged; the previous tile consumed
    for (int i = tid; i < 16 * F; i += NT) {
      const int s = i / F, f = i % F;
      sX[s * XS + f] = base + s < B ? X[(size_t)(base + s) * F + f] : 0.f;
    }
    __syncthreads();
    f32x4 a = {sb1[j], sb1[j], sb1[j], sb1[j]};
#pragma unroll
    for (int k = 0; k < F / 4; ++k) a = mma(sX[c * XS + 4 * k + q], sW1[j * FS + 4 * k + q], a);
#pragma unroll
    for (int r = 0; r < 4; ++r) sH1[(4 * q + r) * HS + j] = a[r] > 0.f ? a[r] : 0.f;
    __syncthreads();
    a = f32x4{sb2[j], sb2[j], sb2[j], sb2[j]};
#pragma unroll
    for (int k = 0; k < H / 4; ++k) a = mma(sH1[c * HS + 4 * k + q], sW2[j * HS + 4 * k + q], a);
#pragma unroll
    for (int r = 0; r < 4; ++r) sH2[(4 * q + r) * HS + j] = a[r] > 0.f ? a[r] : 0.f;
    __syncthreads();
    if (w == 0) {
      a = f32x4{sb3[c], sb3[c], sb3[c], sb3[c]};
#pragma unroll
      for (int k = 0; k < H / 4; ++k) a = mma(sH2[c * HS + 4 * k + q], sW3[c * HS + 4 * k + q], a);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int b = base + 4 * q + r;
        const bool valid = c < O && b < B && mask[(size_t)b * O + c] != 0.f;
        const float e = valid ? a[r] - T[(size_t)b * O + c] : 0.f;
        sY[(4 * q + r) * XS + c] = e;
        lsum += e * e;
        cnt += valid ? 1.f : 0.f;
      }
    }
    __syncthreads();
    a = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < (O + 3) / 4; ++k) a = mma(sY[c * XS + 4 * k + q], sW3[(4 * k + q) * HS + j], a);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int s = 4 * q + r;
      sD2[s * HS + j] = sH2[s * HS + j] > 0.f ? a[r] : 0.f;
    }
    __syncthreads();
    a = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < H / 4; ++k) a = mma(sD2[c * HS + 4 * k + q], sW2[(4 * k + q) * HS + j], a);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int s = 4 * q + r;
      sD1[s * HS + j] = sH1[s * HS + j] > 0.f ? a[r] : 0.f;
    }
    __syncthreads();
    // weight gradients: rows of the left factor's transpose, summed over samples
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int s = 4 * k + q;
      g3 = mma(sY[s * XS + c], sH2[s * HS + j], g3);            // dW3[c rows][16w cols]
      const float d2 = sD2[s * HS + j];
#pragma unroll
      for (int n = 0; n < 4; ++n) g2[n] = mma(d2, sH1[s * HS + 16 * n + c], g2[n]);  // dW2[16w rows][16n cols]
      g1 = mma(sD1[s * HS + j], c < F ? sX[s * XS + c] : 0.f, g1);                   // dW1[16w rows][F cols]
    }
    if (tid < 2 * H + O) {
      const float* col = tid < H ? sD1 + tid : (tid < 2 * H ? sD2 + tid - H : sY + tid - 2 * H);
      const int st = tid < 2 * H ? HS : XS;
#pragma unroll
      for (int s = 0; s < 16; ++s) gb += col[s * st];
    }
  }
  red[0][tid] = lsum;
  red[1][tid] = cnt;
  __syncthreads();
  for (int s = NT / 2; s > 0; s >>= 1) {
    if (tid < s) {
      red[0][tid] += red[0][tid + s];
      red[1][tid] += red[1][tid + s];
    }
    __syncthreads();
  }
  const bool last = gridDim.x == 1;
  const float inv = red[1][0] > 0.f ? 1.f / red[1][0] : 0.f;
  const float sc = last ? 2.f * inv : 1.f;
  float* out = last ? grad : part + (size_t)blockIdx.x * kGradRow;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 16 * w + 4 * q + r;
    if (c < F) out[kMlpW1 + row * F + c] = g1[r] * sc;
#pragma unroll
    for (int n = 0; n < 4; ++n) out[kMlpW2 + row * H + 16 * n + c] = g2[n][r] * sc;
    if (4 * q + r < O) out[kMlpW3 + (4 * q + r) * H + j] = g3[r] * sc;
  }
  if (tid < H) out[kMlpB1 + tid] = gb * sc;
  else if (tid < 2 * H) out[kMlpB2 + tid - H] = gb * sc;
  else if (tid < 2 * H + O) out[kMlpB3 + tid - 2 * H] = gb * sc;
  if (tid == 0) {
    if (last) loss[0] = red[0][0] * inv;
    else {
      out[kMlpParams] = red[0][0];
      out[kMlpParams + 1] = red[1][0];
    }
  }
}

// Sum of the blocks' rows, scaled: 64 columns a block, 4 threads a column.
__global__ __launch_bounds__(256) void k_mlp_grad_sum(int nrow, const float* __restrict__ part,
                                                      float* __restrict__ grad, float* __restrict__ loss) {
  __shared__ float red[4][64];
  const int c = threadIdx.x & 63, g = threadIdx.x >> 6, k = blockIdx.x * 64 + c;
  double n = 0.0;  // the count of valid outputs, a whole number
  for (int r = c; r < nrow; r += 64) n += (double)part[(size_t)r * kGradRow + kMlpParams + 1];
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) n += __shfl_xor(n, m, 64);
  float a = 0.f;
  if (k <= kMlpParams)
    for (int r = g; r < nrow; r += 4) a += part[(size_t)r * kGradRow + k];
  red[g][c] = a;
  __syncthreads();
  if (g != 0 || k > kMlpParams) return;
  const float inv = n > 0.0 ? (float)(1.0 / n) : 0.f;
  const float s = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
  if (k < kMlpParams) grad[k] = 2.f * inv * s;
  else loss[0] = s * inv;
}

__global__ void k_adam(int n, const float* __restrict__ g, float* __restrict__ p, float* __restrict__ m,
                       float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ void k_to_half(int n, const float* __restrict__ a, _Float16* __restrict__ h) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) h[i] = (_Float16)a[i];
}

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot2(h2_t a, h2_t b, float c) { return __builtin_amdgcn_fdot2(a, b, c, false); }

// FP16 inference, one thread per sample: activations and weights in FP16,
// products accumulated in FP32 by v_dot2_f32_f16.
__global__ __launch_bounds__(64) void k_mlp_infer(int B, const float* __restrict__ X,
                                                  const _Float16* __restrict__ HP, float* __restrict__ Y,
                                                  int* __restrict__ order, float log10_tol, float margin,
                                                  int min_order, int max_order) {
  __shared__ h2_t sW[(kMlpParams + 1) / 2];
  const _Float16* sP = reinterpret_cast<const _Float16*>(sW);
  for (int i = threadIdx.x; i < kMlpParams; i += blockDim.x) reinterpret_cast<_Float16*>(sW)[i] = HP[i];
  __syncthreads();
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  h2_t x[F / 2], h1[H / 2], h2[H / 2];
#pragma unroll
  for (int f = 0; f < F / 2; ++f) x[f] = h2_t{(_Float16)X[(size_t)b * F + 2 * f], (_Float16)X[(size_t)b * F + 2 * f + 1]};
  auto w2 = [&](int off) { return h2_t{sP[off], sP[off + 1]}; };
#pragma unroll
  for (int j = 0; j < H; j += 2) {
    float a0 = (float)sP[kMlpB1 + j], a1 = (float)sP[kMlpB1 + j + 1];
#pragma unroll
    for (int f = 0; f < F / 2; ++f) {
      a0 = dot2(w2(kMlpW1 + j * F + 2 * f), x[f], a0);
      a1 = dot2(w2(kMlpW1 + (j + 1) * F + 2 * f), x[f], a1);
    }
    h1[j / 2] = h2_t{(_Float16)(a0 > 0.f ? a0 : 0.f), (_Float16)(a1 > 0.f ? a1 : 0.f)};
  }
#pragma unroll
  for (int j = 0; j < H; j += 2) {
    float a0 = (float)sP[kMlpB2 + j], a1 = (float)sP[kMlpB2 + j + 1];
#pragma unroll
    for (int i = 0; i < H / 2; ++i) {
      a0 = dot2(w2(kMlpW2 + j * H + 2 * i), h1[i], a0);
      a1 = dot2(w2(kMlpW2 + (j + 1) * H + 2 * i), h1[i], a1);
    }
    h2[j / 2] = h2_t{(_Float16)(a0 > 0.f ? a0 : 0.f), (_Float16)(a1 > 0.f ? a1 : 0.f)};
  }
  int q = -1;
#pragma unroll
  for (int o = 0; o < O; ++o) {
    float a = (float)sP[kMlpB3 + o];
#pragma unroll
    for (int i = 0; i < H / 2; ++i) a = dot2(w2(kMlpW3 + o * H + 2 * i), h2[i], a);
    if (Y) Y[(size_t)b * O + o] = a;
    if (q < 0 && a + margin <= log10_tol) q = o + kMlpOrder0;
  }
  if (order) {
    if (q < 0) q = max_order;
    order[b] = q < min_order ? min_order : (q > max_order ? max_order : q);
  }
}

inline int nb(long long n, int bs) { return (int)((n + bs - 1) / bs); }

// Workspace of the allocation-free gradient.  In host code `scratch` names
// a host-side stand-in, never the device array: host code uses only the
// per-device address from hipGetSymbolAddress.  Nothing in it has to start
// at zero (every kernel writes what it later reads).
static __device__ __align__(256) float scratch[kGradBlocks * kGradRow];

constexpr int kMaxDevices = 64;

}  // namespace

float* mlp_scratch() {
  static std::mutex mu;
  static float* addr[kMaxDevices] = {};
  int dev = 0;
  FMM_HIP(hipGetDevice(&dev));
  FMM_CHECK(dev >= 0 && dev < kMaxDevices, kUnsupported, "device index beyond the workspace table");
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    FMM_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    FMM_CHECK(p != nullptr, kHipError, "no device address for the gradient workspace");
    addr[dev] = static_cast<float*>(p);
  }
  return addr[dev];
}

void mlp_forward(int B, const float* X, const float* params, float* Y, hipStream_t st) {
  if (B <= 0) return;
  k_mlp_fwd<<<nb(B, 64), 64, 0, st>>>(B, X, params, Y);
}

void mlp_grad(int B, const float* X, const float* T, const float* mask, const float* params, float* grad,
              float* loss, float* work, hipStream_t st) {
  FMM_CHECK(B > 0, kInvalidArgument, "empty batch");
  const GradGrid g = mlp_grad_grid(B);
  k_mlp_grad<<<g.blocks, 64 * kGradWaves, 0, st>>>(B, g.per, X, T, mask, params, work, grad, loss);
  if (g.blocks > 1) k_mlp_grad_sum<<<nb(kMlpParams + 1, 64), 256, 0, st>>>(g.blocks, work, grad, loss);
}

void mlp_adam(const float* grad, float* params, float* m, float* v, float lr, float beta1, float beta2, float eps,
              int step, hipStream_t st) {
  FMM_CHECK(step >= 1, kInvalidArgument, "Adam step must be >= 1");
  const float c1 = 1.f - powf(beta1, (float)step), c2 = 1.f - powf(beta2, (float)step);
  k_adam<<<nb(kMlpParams, 256), 256, 0, st>>>(kMlpParams, grad, params, m, v, lr, beta1, beta2, eps, c1, c2);
}

void mlp_to_half(const float* params, _Float16* hparams, hipStream_t st) {
  k_to_half<<<nb(kMlpParams, 256), 256, 0, st>>>(kMlpParams, params, hparams);
}

void mlp_infer_f16(int B, const float* X, const _Float16* hparams, float* Y, int* order, float log10_tol,
                   float margin, int min_order, int max_order, hipStream_t st) {
  if (B <= 0) return;
  k_mlp_infer<<<nb(B, 64), 64, 0, st>>>(B, X, hparams, Y, order, log10_tol, margin, min_order, max_order);
}

}  // namespace fmm
