// The learned controller's network on gfx950: FP32 training kernels
// (forward + hand-written backward + Adam) and BF16 matrix-core inference,
// with the odehip_mlp_* C ABI (declarations in odehip.h).
//
// Training: a mini-batch is split over workgroups of 256 threads; each
// workgroup takes its samples in chunks of 64, runs the forward and backward
// pass for the chunk as FP32 matrix-core products, and keeps its share of the
// weight gradient in registers; the per-workgroup partial gradients are then
// summed in a fixed order by the Adam kernel (the run is deterministic).  Samples are visited in the order
// of an affine permutation i -> (a i + c) mod n per epoch.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <random>
#include <vector>

#include "context.hpp"
#include "mlp.hpp"

struct odehip_mlp {
  int device = 0;
  float* w = nullptr;  // FP32 master weights
  float* m = nullptr;  // Adam moments
  float* v = nullptr;
  float* mean = nullptr;  // input normalisation (device, kMlpIn each)
  float* inv_std = nullptr;
  odehip::MlpInfer* infer = nullptr;  // published inference copy
  float* partial = nullptr;           // [kMaxGradBlocks][kMlpParams]
  float* loss_part = nullptr;         // [kMaxGradBlocks]
  float* grad = nullptr;              // [kMlpParams]
  double* loss_acc = nullptr;         // device scalar
  long step = 0;
};

namespace odehip {

const MlpInfer* mlp_infer_ptr(const odehip_mlp* m) { return m ? m->infer : nullptr; }
int mlp_device(const odehip_mlp* m) { return m ? m->device : -1; }

namespace {

constexpr int kGradThreads = 256;
constexpr int kChunk = 64;
constexpr int kMaxGradBlocks = 256;

struct GradArgs {
  const float* w;
  const float* mean;
  const float* inv_std;
  const float* x;  // [n][kMlpIn] raw features
  const float* t;  // [n] targets
  long n;
  unsigned long long perm_a, perm_c;  // sample of position i: (a i + c) mod n
  long first;                         // first position of this batch
  int count;                          // samples in this batch
  float inv_count;
  float* partial;
  float* loss_part;
};

// One chunk is 64 samples; wave w computes the samples 16 w .. 16 w + 15
// forward and back, and rows 16 w .. of the weight gradients over all 64.  The
// five products run on v_mfma_f32_16x16x4_f32 (FP32 operands, products and
// sums); lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and D[4 (l / 16) +
// i][l % 16].  220 of them per wave and chunk, 3 us; as LDS-fed multiply-adds,
// one LDS read each, a chunk took 36 us, and 4096 samples ran on 16 workgroups
// of 4 chunks (145 us a batch, now 7).
// Row strides: 72 floats keep the operand reads along rows and along columns
// at two lanes per bank.
constexpr int kRow = 72;

struct GradLds {
  float w2[kMlpHid][kRow];
  float h1[kChunk][kRow];
  float d2[kChunk][kRow];
  float d1[kChunk][kRow];
  float xs[kChunk][20];  // normalised inputs, columns 10 .. 15 zero
  float tgt[kChunk];
  long idx[kChunk];  // -1: past the end
  float red[4][3][kMlpHid];
  float red1[4][2];
};

__device__ __forceinline__ mlp_float4 mfma4(float a, float b, mlp_float4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__global__ __launch_bounds__(kGradThreads) void k_mlp_grad(GradArgs g) {
  __shared__ GradLds L;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, kq = lane >> 4;
  for (int e = tid; e < kMlpHid * kMlpHid; e += kGradThreads)
    L.w2[e / kMlpHid][e % kMlpHid] = g.w[kMlpOffW2 + e];
  float w1f[4][3], b1[4], b2[4], w3[4];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    const int u = 16 * nb + r;
#pragma unroll
    for (int ks = 0; ks < 3; ++ks) {
      const int i = 4 * ks + kq;
      w1f[nb][ks] = i < kMlpIn ? g.w[kMlpOffW1 + u * kMlpIn + i] : 0.0f;
    }
    b1[nb] = g.w[kMlpOffB1 + u];
    b2[nb] = g.w[kMlpOffB2 + u];
    w3[nb] = g.w[kMlpOffW3 + u];
  }
  const float b3 = g.w[kMlpOffB3];
  const mlp_float4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  // this wave's rows of the gradients: W2 (4 column tiles), W1; and its
  // samples' share of b1, b2, w3 (column 16 nb + r), b3 and the loss
  mlp_float4 gw2[4] = {zero, zero, zero, zero}, gw1 = zero;
  float gb1[4] = {}, gb2[4] = {}, gw3[4] = {}, gb3 = 0.0f, loss = 0.0f;
  const int per = ((g.count + static_cast<int>(gridDim.x) * kChunk - 1) /
                   (static_cast<int>(gridDim.x) * kChunk)) * kChunk;
  const int begin = blockIdx.x * per;
  const int end = min(g.count, begin + per);
  for (int c0 = begin; c0 < end; c0 += kChunk) {
    __syncthreads();
    if (tid < kChunk) {
      const int b = c0 + tid;
      long idx = -1;
      if (b < end) {
        const unsigned long long pos = static_cast<unsigned long long>(g.first + b);
        idx = static_cast<long>((g.perm_a * pos + g.perm_c) % g.n);
      }
      L.idx[tid] = idx;
      L.tgt[tid] = idx >= 0 ? g.t[idx] : 0.0f;
    }
    __syncthreads();
    for (int e = tid; e < kChunk * 16; e += kGradThreads) {
      const int s = e >> 4, i = e & 15;
      const long idx = L.idx[s];
      float v = 0.0f;
      if (idx >= 0 && i < kMlpIn) v = (g.x[idx * kMlpIn + i] - g.mean[i]) * g.inv_std[i];
      L.xs[s][i] = v;
    }
    __syncthreads();
    // layer 1
    const int row = 16 * wave + r;  // the sample of this lane's A operands
    mlp_float4 h1[4], h2[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) h1[nb] = zero;
#pragma unroll
    for (int ks = 0; ks < 3; ++ks) {
      const float a = L.xs[row][4 * ks + kq];
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) h1[nb] = mfma4(a, w1f[nb][ks], h1[nb]);
    }
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        h1[nb][i] = tanhf(h1[nb][i] + b1[nb]);
        L.h1[16 * wave + 4 * kq + i][16 * nb + r] = h1[nb][i];
      }
    __syncthreads();
    // layer 2
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) h2[nb] = zero;
#pragma unroll 4
    for (int ks = 0; ks < 16; ++ks) {
      const float a = L.h1[row][4 * ks + kq];
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) h2[nb] = mfma4(a, L.w2[16 * nb + r][4 * ks + kq], h2[nb]);
    }
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) h2[nb][i] = tanhf(h2[nb][i] + b2[nb]);
    // output, residual and the last layer's gradients, for the samples 4 kq + i
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float y = 0.0f;
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) y += w3[nb] * h2[nb][i];
#pragma unroll
      for (int m = 1; m < 16; m <<= 1) y += __shfl_xor(y, m, 64);
      const int s = 16 * wave + 4 * kq + i;
      const float res = L.idx[s] >= 0 ? y + b3 - L.tgt[s] : 0.0f;
      const float dy = res * g.inv_count;
      if (r == 0) {
        loss += 0.5f * res * res;
        gb3 += dy;
      }
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        const float hv = h2[nb][i];
        const float d = dy * w3[nb] * (1.0f - hv * hv);
        L.d2[s][16 * nb + r] = d;
        gw3[nb] += dy * hv;
        gb2[nb] += d;
      }
    }
    __syncthreads();
    // back through layer 2
    mlp_float4 d1[4] = {zero, zero, zero, zero};
#pragma unroll 4
    for (int ks = 0; ks < 16; ++ks) {
      const float a = L.d2[row][4 * ks + kq];
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) d1[nb] = mfma4(a, L.w2[4 * ks + kq][16 * nb + r], d1[nb]);
    }
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float hv = h1[nb][i];
        const float d = d1[nb][i] * (1.0f - hv * hv);
        L.d1[16 * wave + 4 * kq + i][16 * nb + r] = d;
        gb1[nb] += d;
      }
    __syncthreads();
    // weight gradients: rows 16 wave + ., summed over the chunk's samples
#pragma unroll 4
    for (int ks = 0; ks < 16; ++ks) {
      const int s = 4 * ks + kq;
      const float a = L.d2[s][row];
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) gw2[nb] = mfma4(a, L.h1[s][16 * nb + r], gw2[nb]);
      gw1 = mfma4(L.d1[s][row], L.xs[s][r], gw1);
    }
  }
  float* P = g.partial + static_cast<size_t>(blockIdx.x) * kMlpParams;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = 16 * wave + 4 * kq + i;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) P[kMlpOffW2 + j * kMlpHid + 16 * nb + r] = gw2[nb][i];
    if (r < kMlpIn) P[kMlpOffW1 + j * kMlpIn + r] = gw1[i];
  }
  // the vectors: over the wave's sample rows, then over the waves
#pragma unroll
  for (int m = 16; m < 64; m <<= 1) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      gb1[nb] += __shfl_xor(gb1[nb], m, 64);
      gb2[nb] += __shfl_xor(gb2[nb], m, 64);
      gw3[nb] += __shfl_xor(gw3[nb], m, 64);
    }
    gb3 += __shfl_xor(gb3, m, 64);
    loss += __shfl_xor(loss, m, 64);
  }
  if (kq == 0) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      L.red[wave][0][16 * nb + r] = gb1[nb];
      L.red[wave][1][16 * nb + r] = gb2[nb];
      L.red[wave][2][16 * nb + r] = gw3[nb];
    }
  }
  if (lane == 0) {
    L.red1[wave][0] = gb3;
    L.red1[wave][1] = loss;
  }
  __syncthreads();
  if (tid < 192) {
    const int v = tid >> 6;
    const float sum = (L.red[0][v][lane] + L.red[1][v][lane]) +
                      (L.red[2][v][lane] + L.red[3][v][lane]);
    P[(v == 0 ? kMlpOffB1 : v == 1 ? kMlpOffB2 : kMlpOffW3) + lane] = sum;
  } else if (tid < 194) {
    const int v = tid - 192;
    const float sum = (L.red1[0][v] + L.red1[1][v]) + (L.red1[2][v] + L.red1[3][v]);
    if (v == 0)
      P[kMlpOffB3] = sum;
    else
      g.loss_part[blockIdx.x] = sum;
  }
}

// Sums the partial gradients in a fixed order (four interleaved shares of the
// workgroups' partials per parameter, then the shares); optionally one Adam
// step.  A share of 16 partials at 4096 samples is one round trip of loads.
constexpr int kAdamParams = 64;  // parameters per workgroup
__global__ __launch_bounds__(4 * kAdamParams) void k_mlp_adam(
    const float* partial, int nblk, float* w, float* m, float* v, float* grad, float lr,
    float b1, float b2, float eps, float bc1, float bc2, int apply, const float* loss_part,
    double* loss_acc) {
  __shared__ float part[4][kAdamParams];
  const int lane = threadIdx.x & 63, share = threadIdx.x >> 6;
  const int p = blockIdx.x * kAdamParams + lane;
  float s = 0.0f;
  if (p < kMlpParams) {
    const float* src = partial + p;
#pragma unroll 16
    for (int b = share; b < nblk; b += 4) s += src[static_cast<size_t>(b) * kMlpParams];
  }
  part[share][lane] = s;
  if (blockIdx.x == 0 && share == 3) {
    double l = 0.0;
    for (int b = lane; b < nblk; b += 64) l += loss_part[b];
#pragma unroll
    for (int k = 32; k >= 1; k >>= 1) l += __shfl_xor(l, k, 64);
    if (lane == 0) *loss_acc += l;
  }
  __syncthreads();
  if (share != 0 || p >= kMlpParams) return;
  const float gsum = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
  grad[p] = gsum;
  if (!apply) return;
  const float mm = b1 * m[p] + (1.0f - b1) * gsum;
  const float vv = b2 * v[p] + (1.0f - b2) * gsum * gsum;
  m[p] = mm;
  v[p] = vv;
  w[p] -= lr * (mm / bc1) / (sqrtf(vv / bc2) + eps);
}

__global__ void k_mlp_publish(const float* w, const float* mean,
                              const float* inv_std, MlpInfer* out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < 16) {
    out->mean[t] = t < kMlpIn ? mean[t] : 0.0f;
    out->inv_std[t] = t < kMlpIn ? inv_std[t] : 0.0f;
  }
  if (t < 64 * 16) {
    const int j = t / 16, i = t % 16;
    out->w1[j][i] = i < kMlpIn ? float_to_bf16(w[kMlpOffW1 + j * kMlpIn + i]) : 0;
  }
  if (t < 64 * 64) {
    const int j = t / 64, i = t % 64;
    out->w2[j][i] = float_to_bf16(w[kMlpOffW2 + j * kMlpHid + i]);
    // w3: 16 x 64, row 0 the weights
    if (j < 16) out->w3[j][i] = j == 0 ? float_to_bf16(w[kMlpOffW3 + i]) : 0;
  }
  if (t < 64) {
    out->b1[t] = w[kMlpOffB1 + t];
    out->b2[t] = w[kMlpOffB2 + t];
  }
  if (t == 0) {
    out->b3 = w[kMlpOffB3];
    out->pad[0] = out->pad[1] = out->pad[2] = 0.0f;
  }
}

// One wave per 16 samples.
__global__ __launch_bounds__(64) void k_mlp_infer(const MlpInfer* M,
                                                  const float* x, long n,
                                                  float* y) {
  __shared__ MlpTileLds t;
  const int lane = threadIdx.x;
  const long row = static_cast<long>(blockIdx.x) * 16 + lane;
  if (lane < 16) {
    float raw[kMlpIn];
    for (int i = 0; i < kMlpIn; ++i) raw[i] = row < n ? x[row * kMlpIn + i] : 0.0f;
    mlp_tile_set_row(M, t, lane, raw);
  }
  __syncthreads();
  mlp_tile_forward(M, t);
  if (lane < 16 && row < n) y[row] = t.y[lane];
}

unsigned long long gcd_u(unsigned long long a, unsigned long long b) {
  while (b) {
    const unsigned long long t = a % b;
    a = b;
    b = t;
  }
  return a;
}

int publish(odehip_context* ctx, odehip_mlp* m, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_publish, dim3(16), dim3(256), 0, s, m->w, m->mean, m->inv_std,
                     m->infer);
  HIP_TRY(ctx, hipGetLastError());
  return ODEHIP_OK;
}

// Gradient of one batch (positions [first, first + count) of the
// permutation) into m->grad; with apply, one Adam step.
int batch_step(odehip_context* ctx, odehip_mlp* m, const float* x, const float* t, long n,
               unsigned long long a, unsigned long long c, long first, int count,
               bool apply, float lr, float b1, float b2, float eps, hipStream_t s) {
  const int nblk = std::min(kMaxGradBlocks, std::max(1, (count + kChunk - 1) / kChunk));
  GradArgs g{};
  g.w = m->w;
  g.mean = m->mean;
  g.inv_std = m->inv_std;
  g.x = x;
  g.t = t;
  g.n = n;
  g.perm_a = a;
  g.perm_c = c;
  g.first = first;
  g.count = count;
  g.inv_count = 1.0f / static_cast<float>(count);
  g.partial = m->partial;
  g.loss_part = m->loss_part;
  hipLaunchKernelGGL(k_mlp_grad, dim3(nblk), dim3(kGradThreads), 0, s, g);
  HIP_TRY(ctx, hipGetLastError());
  float bc1 = 1.0f, bc2 = 1.0f;
  if (apply) {
    m->step += 1;
    bc1 = 1.0f - std::pow(b1, static_cast<float>(m->step));
    bc2 = 1.0f - std::pow(b2, static_cast<float>(m->step));
  }
  hipLaunchKernelGGL(k_mlp_adam, dim3((kMlpParams + kAdamParams - 1) / kAdamParams),
                     dim3(4 * kAdamParams), 0, s,
                     m->partial, nblk, m->w, m->m, m->v, m->grad, lr, b1, b2, eps, bc1, bc2,
                     apply ? 1 : 0, m->loss_part, m->loss_acc);
  HIP_TRY(ctx, hipGetLastError());
  return ODEHIP_OK;
}

}  // namespace
}  // namespace odehip

using namespace odehip;

extern "C" {

int odehip_mlp_create(odehip_context* ctx, const float* params, uint64_t seed,
                      const float* mean, const float* stdv, odehip_mlp** out) {
  ODEHIP_USE_DEVICE(ctx);
  if (!ctx) return ODEHIP_ERR_INVALID;
  if (!out || !mean || !stdv) return fail(ctx, ODEHIP_ERR_INVALID, "null argument");
  float inv[kMlpIn];
  for (int i = 0; i < kMlpIn; ++i) {
    if (!(stdv[i] > 0.0f) || !std::isfinite(mean[i]))
      return fail(ctx, ODEHIP_ERR_INVALID, "std must be positive and mean finite");
    inv[i] = 1.0f / stdv[i];
  }
  std::vector<float> p(kMlpParams, 0.0f);
  if (params) {
    std::memcpy(p.data(), params, sizeof(float) * kMlpParams);
  } else {
    // Glorot-uniform weights, zero biases
    std::mt19937_64 gen(seed);
    auto fill = [&](int off, int fan_in, int fan_out, int count) {
      const double lim = std::sqrt(6.0 / (fan_in + fan_out));
      std::uniform_real_distribution<double> d(-lim, lim);
      for (int k = 0; k < count; ++k) p[off + k] = static_cast<float>(d(gen));
    };
    fill(kMlpOffW1, kMlpIn, kMlpHid, kMlpHid * kMlpIn);
    fill(kMlpOffW2, kMlpHid, kMlpHid, kMlpHid * kMlpHid);
    fill(kMlpOffW3, kMlpHid, 1, kMlpHid);
  }
  auto* m = new (std::nothrow) odehip_mlp();
  if (!m) return fail(ctx, ODEHIP_ERR_NOMEM, "mlp");
  m->device = ctx->device;
  auto cleanup = [&](int rc) {
    odehip_mlp_destroy(m);
    return rc;
  };
  hipError_t e;
  if ((e = hipMalloc(&m->w, sizeof(float) * kMlpParams)) != hipSuccess ||
      (e = hipMalloc(&m->m, sizeof(float) * kMlpParams)) != hipSuccess ||
      (e = hipMalloc(&m->v, sizeof(float) * kMlpParams)) != hipSuccess ||
      (e = hipMalloc(&m->grad, sizeof(float) * kMlpParams)) != hipSuccess ||
      (e = hipMalloc(&m->mean, sizeof(float) * 16)) != hipSuccess ||
      (e = hipMalloc(&m->inv_std, sizeof(float) * 16)) != hipSuccess ||
      (e = hipMalloc(&m->infer, sizeof(MlpInfer))) != hipSuccess ||
      (e = hipMalloc(&m->partial, sizeof(float) * kMlpParams * kMaxGradBlocks)) != hipSuccess ||
      (e = hipMalloc(&m->loss_part, sizeof(float) * kMaxGradBlocks)) != hipSuccess ||
      (e = hipMalloc(&m->loss_acc, sizeof(double))) != hipSuccess)
    return cleanup(hip_fail(ctx, e, "mlp allocation"));
  std::vector<float> zeros(kMlpParams, 0.0f);
  if ((e = hipMemcpy(m->w, p.data(), sizeof(float) * kMlpParams, hipMemcpyHostToDevice)) ||
      (e = hipMemcpy(m->m, zeros.data(), sizeof(float) * kMlpParams, hipMemcpyHostToDevice)) ||
      (e = hipMemcpy(m->v, zeros.data(), sizeof(float) * kMlpParams, hipMemcpyHostToDevice)) ||
      (e = hipMemcpy(m->mean, mean, sizeof(float) * kMlpIn, hipMemcpyHostToDevice)) ||
      (e = hipMemcpy(m->inv_std, inv, sizeof(float) * kMlpIn, hipMemcpyHostToDevice)))
    return cleanup(hip_fail(ctx, e, "mlp upload"));
  hipStream_t s = begin_work(ctx);
  int rc = publish(ctx, m, s);
  if (rc) return cleanup(rc);
  if ((e = hipStreamSynchronize(s)) != hipSuccess) return cleanup(hip_fail(ctx, e, "mlp init"));
  end_work(ctx);
  *out = m;
  return ODEHIP_OK;
}

int odehip_mlp_destroy(odehip_mlp* m) {
  if (!m) return ODEHIP_OK;
  (void)hipSetDevice(m->device);
  (void)hipDeviceSynchronize();
  for (void* p : {static_cast<void*>(m->w), static_cast<void*>(m->m), static_cast<void*>(m->v),
                  static_cast<void*>(m->grad), static_cast<void*>(m->mean),
                  static_cast<void*>(m->inv_std), static_cast<void*>(m->infer),
                  static_cast<void*>(m->partial), static_cast<void*>(m->loss_part),
                  static_cast<void*>(m->loss_acc)})
    if (p) (void)hipFree(p);
  delete m;
  return ODEHIP_OK;
}

int odehip_mlp_get_params(odehip_context* ctx, const odehip_mlp* m,
                          float* params_out) {
  ODEHIP_USE_DEVICE(ctx);
  if (!ctx) return ODEHIP_ERR_INVALID;
  if (!m || !params_out) return fail(ctx, ODEHIP_ERR_INVALID, "null argument");
  if (m->device != ctx->device)
    return fail(ctx, ODEHIP_ERR_INVALID, "the network lives on another device");
  HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  HIP_TRY(ctx, hipMemcpy(params_out, m->w, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost));
  return ODEHIP_OK;
}

int odehip_mlp_loss_grad(odehip_context* ctx, odehip_mlp* m, const float* x,
                         const float* t, long n, float* grad_out,
                         double* loss_out) {
  ODEHIP_USE_DEVICE(ctx);
  if (!ctx) return ODEHIP_ERR_INVALID;
  if (!m || !x || !t || !grad_out) return fail(ctx, ODEHIP_ERR_INVALID, "null argument");
  if (m->device != ctx->device)
    return fail(ctx, ODEHIP_ERR_INVALID, "the network lives on another device");
  if (n <= 0 || n > (1L << 30)) return fail(ctx, ODEHIP_ERR_INVALID, "bad sample count");
  hipStream_t s = begin_work(ctx);
  HIP_TRY(ctx, hipMemsetAsync(m->loss_acc, 0, sizeof(double), s));
  int rc = batch_step(ctx, m, x, t, n, 1, 0, 0, static_cast<int>(n), false, 0.f, 0.f, 0.f,
                      0.f, s);
  if (rc) return rc;
  double loss = 0.0;
  HIP_TRY(ctx, hipMemcpyAsync(grad_out, m->grad, sizeof(float) * kMlpParams,
                              hipMemcpyDeviceToHost, s));
  HIP_TRY(ctx, hipMemcpyAsync(&loss, m->loss_acc, sizeof(double), hipMemcpyDeviceToHost, s));
  HIP_TRY(ctx, hipStreamSynchronize(s));
  end_work(ctx);
  if (loss_out) *loss_out = loss / static_cast<double>(n);
  return ODEHIP_OK;
}

int odehip_mlp_train(odehip_context* ctx, odehip_mlp* m, const float* x,
                     const float* t, long n, const odehip_mlp_train_options* o,
                     double* epoch_loss) {
  ODEHIP_USE_DEVICE(ctx);
  if (!ctx) return ODEHIP_ERR_INVALID;
  if (!m || !x || !t || !o) return fail(ctx, ODEHIP_ERR_INVALID, "null argument");
  if (m->device != ctx->device)
    return fail(ctx, ODEHIP_ERR_INVALID, "the network lives on another device");
  if (n <= 0 || n > (1L << 34)) return fail(ctx, ODEHIP_ERR_INVALID, "bad sample count");
  if (o->epochs < 0 || o->batch <= 0 || !(o->lr > 0.0f))
    return fail(ctx, ODEHIP_ERR_INVALID, "bad training options");
  hipStream_t s = begin_work(ctx);
  std::mt19937_64 gen(o->seed);
  const float b1 = o->beta1 > 0.0f ? o->beta1 : 0.9f;
  const float b2 = o->beta2 > 0.0f ? o->beta2 : 0.999f;
  const float eps = o->eps > 0.0f ? o->eps : 1e-8f;
  const unsigned long long un = static_cast<unsigned long long>(n);
  for (int ep = 0; ep < o->epochs; ++ep) {
    unsigned long long a = 1, c = 0;
    if (n > 1) {
      do {
        a = 1 + gen() % (un - 1);
      } while (gcd_u(a, un) != 1);
      c = gen() % un;
    }
    HIP_TRY(ctx, hipMemsetAsync(m->loss_acc, 0, sizeof(double), s));
    for (long first = 0; first < n; first += o->batch) {
      const int count = static_cast<int>(std::min<long>(o->batch, n - first));
      int rc = batch_step(ctx, m, x, t, n, a, c, first, count, true, o->lr, b1, b2, eps, s);
      if (rc) return rc;
    }
    double loss = 0.0;
    HIP_TRY(ctx, hipMemcpyAsync(&loss, m->loss_acc, sizeof(double), hipMemcpyDeviceToHost, s));
    HIP_TRY(ctx, hipStreamSynchronize(s));
    if (epoch_loss) epoch_loss[ep] = loss / static_cast<double>(n);
  }
  int rc = publish(ctx, m, s);
  if (rc) return rc;
  HIP_TRY(ctx, hipStreamSynchronize(s));
  end_work(ctx);
  return ODEHIP_OK;
}

int odehip_mlp_infer(odehip_context* ctx, const odehip_mlp* m, const float* x,
                     long n, float* y) {
  ODEHIP_USE_DEVICE(ctx);
  if (!ctx) return ODEHIP_ERR_INVALID;
  if (!m || !x || !y) return fail(ctx, ODEHIP_ERR_INVALID, "null argument");
  if (m->device != ctx->device)
    return fail(ctx, ODEHIP_ERR_INVALID, "the network lives on another device");
  if (n <= 0 || n > (1L << 34)) return fail(ctx, ODEHIP_ERR_INVALID, "bad sample count");
  hipStream_t s = begin_work(ctx);
  const long blocks = (n + 15) / 16;
  hipLaunchKernelGGL(k_mlp_infer, dim3(static_cast<unsigned>(blocks)), dim3(64), 0, s,
                     m->infer, x, n, y);
  HIP_TRY(ctx, hipGetLastError());
  end_work(ctx);
  return ODEHIP_OK;
}

}  // extern "C"
