// FP32 training kernels of the learned RK5 step-size proposer.
//
// One training step = one minibatch, two launches:
//   grad_kernel    forward and backward pass of the 6-32-32-1 ReLU MLP on
//                  the matrix cores, 32 samples a wave at a time; every
//                  block writes its sums of the gradients and the loss as
//                  one row of partial sums;
//   update_kernel  adds the rows in block order, then SGD or Adam on the
//                  1313 parameters; refreshes the BF16 inference copy.
// The sums have a fixed order, so a training run is reproducible.
#include <hip/hip_runtime.h>

#include "ngpu_device.h"
#include "proposer.h"

namespace ngpu {

namespace {

constexpr int kTB = 256;

__device__ __forceinline__ uint16_t to_bf16(float f) {
  // round to nearest even
  uint32_t u = __float_as_uint(f);
  uint32_t lsb = (u >> 16) & 1u;
  u += 0x7FFFu + lsb;
  return (uint16_t)(u >> 16);
}

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kTile = 32;              // samples of one wave's pass
constexpr int kPad = kTile + 1;        // row stride of a transposed tile
constexpr int kGradWaves = kTB / 64;

// Minibatch gradient, all FP32 (v_mfma_f32_32x32x2_f32: FP32 products and
// sums).  A layer is H^T = W X^T with the tile's 32 samples as columns; the
// accumulator layout (lane l, value r: row 8 (r / 4) + 4 (l / 32) + r % 4,
// column l % 32) is the next product's B operand when its contraction runs
// in the order k = (8 g + c, 8 g + 4 + c), so activations and their
// gradients stay in registers from layer to layer.  The weight gradients
// contract over the samples: their A operands are read back transposed from
// LDS.  Each lane of that read passes over a whole row of the tile, which
// also gives the bias sums.
// The bound is latency (8192 samples are 256 tiles, one a wave on 64 CUs,
// 68 MFMAs of 64 clocks each); the atomic-add version it replaces put 64
// lanes on one LDS address per parameter: 1030 us per step of 8192 samples.
__global__ __launch_bounds__(kTB) void grad_kernel(PropTrainArgs A) {
  __shared__ float s_t[kGradWaves][3][kPropHid * kPad];
  __shared__ float s_g[kPropGradRow];
  const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
  const int col = lane & 31, half = lane >> 5;
  float *td2 = s_t[wave][0], *th1 = s_t[wave][1], *tx = s_t[wave][2];
  // A operands: W1 with the bias as input 6, W2, W2 transposed; b2 and w3
  // in the accumulator layout
  float w1[4], w2[16], w2t[16];
  v16f b2;
  float w3[16];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int k = 4 * half + c;
    w1[c] = k < kPropIn ? A.w[kPropW1 + col * kPropIn + k]
                        : (k == kPropIn ? A.w[kPropB1 + col] : 0.0f);
  }
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int k = 8 * (r / 4) + 4 * half + r % 4;
    w2[r] = A.w[kPropW2 + col * kPropHid + k];
    w2t[r] = A.w[kPropW2 + k * kPropHid + col];
    b2[r] = A.w[kPropB2 + k];
    w3[r] = A.w[kPropW3 + k];
  }
  const float b3 = A.w[kPropB3];
  v16f g2, g1;                          // dW2 and dW1 (columns 0-5, 6: db1)
#pragma unroll
  for (int r = 0; r < 16; r++) g2[r] = g1[r] = 0.0f;
  float gb2 = 0.0f, gw3 = 0.0f;         // of unit col, samples of this half
  float gb3 = 0.0f, loss = 0.0f;
  const int tiles = (int)(((uint32_t)A.batch + kTile - 1u) / kTile);
  // every wave of the block makes the same number of passes
  for (int t0 = blockIdx.x * kGradWaves; t0 < tiles;
       t0 += gridDim.x * kGradWaves) {
    const long long b = (long long)(t0 + wave) * kTile + col;
    const bool valid = b < A.batch;
    float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (valid) {
      unsigned long long idx;
      if (A.full_batch) {
        idx = (unsigned long long)b % A.n;
      } else {
        const uint32_t u0 = dev_philox_w0((uint32_t)b, A.iter, 0x70726F70u,
                                          0u, A.seed, 0x74726169u);
        const uint32_t u1 = dev_philox_w0((uint32_t)b, A.iter, 0x70726F70u,
                                          1u, A.seed, 0x74726169u);
        idx = (((unsigned long long)u1 << 32) | u0) % A.n;
      }
      // inputs 0-3 in the lower half, inputs 4, 5 and the target above
      q = *reinterpret_cast<const float4 *>(A.samples + idx * kPropSample +
                                            4 * half);
    }
    const float target = __shfl(q.z, 32 + col);
    const float x[4] = {q.x, q.y, half ? 1.0f : q.z, half ? 0.0f : q.w};
    v16f z1, z2 = b2, h1, h2;
#pragma unroll
    for (int r = 0; r < 16; r++) z1[r] = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; c++)
      z1 = __builtin_amdgcn_mfma_f32_32x32x2f32(w1[c], x[c], z1, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; r++) h1[r] = z1[r] > 0.0f ? z1[r] : 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r++)
      z2 = __builtin_amdgcn_mfma_f32_32x32x2f32(w2[r], h1[r], z2, 0, 0, 0);
    float y = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      h2[r] = z2[r] > 0.0f ? z2[r] : 0.0f;
      y = __builtin_fmaf(w3[r], h2[r], y);
    }
    y = (y + __shfl_xor(y, 32)) + b3;
    const float dy = valid ? y - target : 0.0f;  // d(0.5 (y - t)^2)/dy
    if (half == 0) {
      loss += 0.5f * dy * dy;
      gb3 += dy;
    }
    v16f d2, d1;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      d2[r] = z2[r] > 0.0f ? dy * w3[r] : 0.0f;
      d1[r] = 0.0f;
    }
#pragma unroll
    for (int r = 0; r < 16; r++)
      d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(w2t[r], d2[r], d1, 0, 0, 0);
    // transposed tiles: row = unit, column = sample
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int k = 8 * (r / 4) + 4 * half + r % 4;
      td2[k * kPad + col] = d2[r];
      th1[k * kPad + col] = h1[r];
      tx[k * kPad + col] = dy * h2[r];
      d1[r] = z1[r] > 0.0f ? d1[r] : 0.0f;
    }
    __syncthreads();
    // contraction over the samples 2 s + half: dW2 = D2 H1^T
#pragma unroll
    for (int s = 0; s < 16; s++) {
      const float a = td2[col * kPad + 2 * s + half];
      gb2 += a;
      gw3 += tx[col * kPad + 2 * s + half];
      g2 = __builtin_amdgcn_mfma_f32_32x32x2f32(
          a, th1[col * kPad + 2 * s + half], g2, 0, 0, 0);
    }
    __syncthreads();
    // dW1 = D1 X^T: the inputs as rows 0-7 of a tile, its other rows 0
#pragma unroll
    for (int r = 0; r < 16; r++)
      td2[(8 * (r / 4) + 4 * half + r % 4) * kPad + col] = d1[r];
#pragma unroll
    for (int c = 0; c < 4; c++) th1[(4 * half + c) * kPad + col] = x[c];
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 16; s++)
      g1 = __builtin_amdgcn_mfma_f32_32x32x2f32(
          td2[col * kPad + 2 * s + half],
          col < 8 ? th1[col * kPad + 2 * s + half] : 0.0f, g1, 0, 0, 0);
    __syncthreads();
  }
  gb2 += __shfl_xor(gb2, 32);
  gw3 += __shfl_xor(gw3, 32);
#pragma unroll
  for (int off = 1; off < 32; off <<= 1) {
    gb3 += __shfl_xor(gb3, off);
    loss += __shfl_xor(loss, off);
  }
  // the block's row: its waves' sums in wave order
  for (int k = threadIdx.x; k < kPropGradRow; k += kTB) s_g[k] = 0.0f;
  for (int w = 0; w < kGradWaves; w++) {
    __syncthreads();
    if (wave != w) continue;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int k = 8 * (r / 4) + 4 * half + r % 4;
      s_g[kPropW2 + k * kPropHid + col] += g2[r];
      if (col < kPropIn) s_g[kPropW1 + k * kPropIn + col] += g1[r];
      if (col == kPropIn) s_g[kPropB1 + k] += g1[r];
    }
    if (half == 0) {
      s_g[kPropB2 + col] += gb2;
      s_g[kPropW3 + col] += gw3;
    }
    if (lane == 0) {
      s_g[kPropB3] += gb3;
      s_g[kPropNParam] += loss;
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < kPropGradRow; k += kTB)
    A.grad[(size_t)blockIdx.x * kPropGradRow + k] = s_g[k];
}

// 64 parameters a block, four threads each a quarter of the rows.
__global__ __launch_bounds__(kTB) void update_kernel(PropTrainArgs A,
                                                     uint32_t step,
                                                     int rows) {
  __shared__ float s_p[kTB];
  const int k = blockIdx.x * 64 + (threadIdx.x & 63);
  const int part = threadIdx.x / 64;
  float sum = 0.0f;
  if (k < kPropGradRow) {
    const int per = (rows + 3) / 4;
    const int r1 = (part + 1) * per < rows ? (part + 1) * per : rows;
#pragma unroll 8
    for (int r = part * per; r < r1; r++)
      sum += A.grad[(size_t)r * kPropGradRow + k];
  }
  s_p[threadIdx.x] = sum;
  __syncthreads();
  if (part != 0 || k >= kPropGradRow) return;
  sum = (s_p[threadIdx.x] + s_p[threadIdx.x + 64]) +
        (s_p[threadIdx.x + 128] + s_p[threadIdx.x + 192]);
  if (k == kPropNParam) {
    *A.loss = sum;
    return;
  }
  float g = sum / (float)A.batch;
  float w = A.w[k];
  if (A.adam) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    float m = b1 * A.m[k] + (1.0f - b1) * g;
    float v = b2 * A.v[k] + (1.0f - b2) * g * g;
    A.m[k] = m;
    A.v[k] = v;
    float mh = m / (1.0f - powf(b1, (float)step));
    float vh = v / (1.0f - powf(b2, (float)step));
    w -= A.lr * mh / (sqrtf(vh) + eps);
  } else {
    w -= A.lr * g;
  }
  A.w[k] = w;
  A.w_bf16[k] = to_bf16(w);
}

__global__ void pack_kernel(const float *w, unsigned char *pk) {
  int l = threadIdx.x;  // 64 threads
  if (l >= 64) return;
  uint16_t *w1p = reinterpret_cast<uint16_t *>(pk + kPropPkW1);
  uint16_t *w2p = reinterpret_cast<uint16_t *>(pk + kPropPkW2);
  float *b1p = reinterpret_cast<float *>(pk + kPropPkB1);
  float *b2p = reinterpret_cast<float *>(pk + kPropPkB2);
  float *w3p = reinterpret_cast<float *>(pk + kPropPkW3);
  int row = l % 32, half = l / 32;
  for (int j = 0; j < 4; j++) {
    int k = 4 * half + j;
    w1p[l * 4 + j] = k < kPropIn ? to_bf16(w[kPropW1 + row * kPropIn + k])
                                 : (uint16_t)0;
    for (int c = 0; c < 4; c++)
      w2p[(c * 64 + l) * 4 + j] =
          to_bf16(w[kPropW2 + row * kPropHid + 8 * c + 4 * half + j]);
  }
  for (int r = 0; r < 16; r++) {
    int unit = 8 * (r / 4) + 4 * half + (r % 4);
    b1p[l * 16 + r] = w[kPropB1 + unit];
    b2p[l * 16 + r] = w[kPropB2 + unit];
    w3p[l * 16 + r] = w[kPropW3 + unit];
  }
  if (l == 0) *reinterpret_cast<float *>(pk + kPropPkB3) = w[kPropB3];
}

__global__ void to_bf16_kernel(const float *w, uint16_t *o) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < kPropNParam) o[k] = to_bf16(w[k]);
}

}  // namespace

const char *LaunchPropTrainStep(const PropTrainArgs &a, void *stream) {
  hipStream_t s = (hipStream_t)stream;
  if (a.batch <= 0) return "batch must be positive";
  // a wave per tile up to one block per CU
  const int tiles = (int)(((uint32_t)a.batch + kTile - 1u) / kTile);
  int rows = tiles / kGradWaves + (tiles % kGradWaves ? 1 : 0);
  if (rows > kPropGradRows) rows = kPropGradRows;
  hipLaunchKernelGGL(grad_kernel, dim3(rows), dim3(kTB), 0, s, a);
  hipLaunchKernelGGL(update_kernel, dim3((kPropGradRow + 63) / 64), dim3(kTB),
                     0, s, a, a.iter + 1u, rows);
  return nullptr;
}

void LaunchPropPack(const float *w, unsigned char *packed, void *stream) {
  hipLaunchKernelGGL(pack_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream,
                     w, packed);
}

void LaunchPropToBf16(const float *w, uint16_t *w_bf16, void *stream) {
  hipLaunchKernelGGL(to_bf16_kernel, dim3((kPropNParam + 255) / 256),
                     dim3(256), 0, (hipStream_t)stream, w, w_bf16);
}

}  // namespace ngpu
