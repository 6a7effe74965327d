// The learned step-size controller's network: layout, controller features
// and the BF16 matrix-core inference of a tile of 16 systems.
//
// Network: 10 -> 64 -> 64 -> 1, tanh hidden layers, linear output = the log
// of the proposed step ratio dt_new / dt.  Training keeps FP32 master
// weights in the flat layout
//   W1[64][10] | b1[64] | W2[64][64] | b2[64] | w3[64] | b3     (kParams)
// and publishes an MlpInfer copy: weights in bfloat16, padded to the 16 x 16
// x 16 matrix-core shape, biases and the input normalisation in FP32.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "rk_device.hpp"

namespace odehip {

constexpr int kMlpIn = ODEHIP_MLP_IN;
constexpr int kMlpHid = ODEHIP_MLP_HIDDEN;
constexpr int kMlpOffW1 = 0;
constexpr int kMlpOffB1 = kMlpOffW1 + kMlpHid * kMlpIn;
constexpr int kMlpOffW2 = kMlpOffB1 + kMlpHid;
constexpr int kMlpOffB2 = kMlpOffW2 + kMlpHid * kMlpHid;
constexpr int kMlpOffW3 = kMlpOffB2 + kMlpHid;
constexpr int kMlpOffB3 = kMlpOffW3 + kMlpHid;
constexpr int kMlpParams = kMlpOffB3 + 1;
static_assert(kMlpParams == ODEHIP_MLP_PARAMS, "parameter count");

// Step ratio limits of the learned proposal: [0.2, 5].
constexpr double kMlpLogRatioMin = -1.6094379124341003;
constexpr double kMlpLogRatioMax = 1.6094379124341003;

// Inference copy (device).  Rows are output units, columns inputs, so a
// 16 x 16 B operand (k, n) reads W[n][k .. k+3] contiguously.
struct MlpInfer {
  float mean[16];
  float inv_std[16];
  uint16_t w1[64][16];  // K padded 10 -> 16 with zeros
  float b1[64];
  uint16_t w2[64][64];
  float b2[64];
  uint16_t w3[16][64];  // row 0 = w3, rows 1..15 zero (N padded to 16)
  float b3;
  float pad[3];
};

__host__ __device__ inline uint16_t float_to_bf16(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  if ((u & 0x7f800000u) != 0x7f800000u) u += 0x7fffu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(u >> 16);
}

typedef short mlp_short4 __attribute__((ext_vector_type(4)));
typedef float mlp_float4 __attribute__((ext_vector_type(4)));

// LDS scratch of one wave's tile.
struct MlpTileLds {
  float x[16][16];
  float h[16][65];
  float y[16];
};

// Network output for the 16 rows of t.x (normalised features, written by the
// caller; columns 10..15 zero).  Must be called by all 64 lanes of a wave,
// in a workgroup of exactly one wave (the barriers are workgroup barriers).
// v_mfma_f32_16x16x16_bf16 operand layout: lane l holds A[l % 16][4 (l / 16)
// + i], B[4 (l / 16) + i][l % 16] and D[4 (l / 16) + i][l % 16], i = 0..3.
__device__ inline void mlp_tile_forward(const MlpInfer* M, MlpTileLds& t) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int kq = lane >> 4;
  // layer 1: [16 x 16] x [16 x 64]
  mlp_short4 a;
#pragma unroll
  for (int i = 0; i < 4; ++i) a[i] = static_cast<short>(float_to_bf16(t.x[r][4 * kq + i]));
  mlp_float4 z[4];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    mlp_short4 b;
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = static_cast<short>(M->w1[16 * nb + r][4 * kq + i]);
    const mlp_float4 c = {0.0f, 0.0f, 0.0f, 0.0f};
    z[nb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
  }
  __syncthreads();
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      t.h[4 * kq + i][16 * nb + r] = tanhf(z[nb][i] + M->b1[16 * nb + r]);
  __syncthreads();
  // layer 2: [16 x 64] x [64 x 64]
  mlp_short4 a2[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      a2[ks][i] = static_cast<short>(float_to_bf16(t.h[r][16 * ks + 4 * kq + i]));
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    mlp_float4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      mlp_short4 b;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        b[i] = static_cast<short>(M->w2[16 * nb + r][16 * ks + 4 * kq + i]);
      c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a2[ks], b, c, 0, 0, 0);
    }
    z[nb] = c;
  }
  __syncthreads();
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      t.h[4 * kq + i][16 * nb + r] = tanhf(z[nb][i] + M->b2[16 * nb + r]);
  __syncthreads();
  // layer 3: [16 x 64] x [64 x 16] (only column 0 is the output)
  mlp_float4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    mlp_short4 a3, b;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a3[i] = static_cast<short>(float_to_bf16(t.h[r][16 * ks + 4 * kq + i]));
      b[i] = static_cast<short>(M->w3[r][16 * ks + 4 * kq + i]);
    }
    c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a3, b, c, 0, 0, 0);
  }
  if (r == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) t.y[4 * kq + i] = c[i] + M->b3;
  }
  __syncthreads();
}

// One system's forward pass by one wave, row 0 of the same tile: every weight is
// loaded up front (no load waits for an activation) and only row 0's activations
// go through tanh, 8 of them per lane instead of 32.  The row's products and
// sums are those of mlp_tile_forward.  `x`: the 16 normalised features, `h`: 64
// floats, both in LDS and used by this wave alone.  The result is in lane 0.
struct MlpRowWeights {
  mlp_short4 w1[4], w2[4][4], w3[4];
  float b1[4], b2[4], b3;
};

__device__ inline MlpRowWeights mlp_row_weights(const MlpInfer* M) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int kq = lane >> 4;
  MlpRowWeights w;
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    const int o = 16 * nb + r;
    w.w1[nb] = *reinterpret_cast<const mlp_short4*>(&M->w1[o][4 * kq]);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      w.w2[nb][ks] = *reinterpret_cast<const mlp_short4*>(&M->w2[o][16 * ks + 4 * kq]);
    w.w3[nb] = *reinterpret_cast<const mlp_short4*>(&M->w3[r][16 * nb + 4 * kq]);
    w.b1[nb] = M->b1[o];
    w.b2[nb] = M->b2[o];
  }
  w.b3 = M->b3;
  return w;
}

__device__ inline float mlp_row_forward(const MlpRowWeights& w, const float* x, float* h) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int kq = lane >> 4;
  auto operand = [&](const float* v, int k0) {  // row 0 of A, the other rows zero
    mlp_short4 a;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      a[i] = r == 0 ? static_cast<short>(float_to_bf16(v[k0 + 4 * kq + i])) : short{0};
    return a;
  };
  const mlp_float4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  float z[4];
  wave_lds_fence();
  const mlp_short4 a1 = operand(x, 0);
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
    z[nb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1, w.w1[nb], zero, 0, 0, 0)[0];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    const float t = tanhf(z[nb] + w.b1[nb]);
    if (kq == 0) h[16 * nb + r] = t;
  }
  wave_lds_fence();
  mlp_short4 a[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) a[ks] = operand(h, 16 * ks);
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    mlp_float4 c = zero;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[ks], w.w2[nb][ks], c, 0, 0, 0);
    z[nb] = c[0];
  }
  wave_lds_fence();
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    const float t = tanhf(z[nb] + w.b2[nb]);
    if (kq == 0) h[16 * nb + r] = t;
  }
  wave_lds_fence();
  mlp_float4 c = zero;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(operand(h, 16 * ks), w.w3[ks], c, 0, 0, 0);
  return c[0] + w.b3;
}

// The step ratio the network's output stands for (NaN if it is not finite).
__device__ inline double mlp_ratio(double y) {
  y = y < kMlpLogRatioMin ? kMlpLogRatioMin : (y > kMlpLogRatioMax ? kMlpLogRatioMax : y);
  return std::isfinite(y) ? std::exp(y) : NAN;
}

// LDS of one wave's learned controller.
struct MlpRowLds {
  double arg[16];
  float x[16];
  float h[64];
};

// Controller features of one system after an attempt: log error norms of the
// last three attempts, log(dt / (tf - t0)) of the last, the log ratios of the two
// before to it, the three accept flags, log N; non-finite ones (history not
// filled yet) are 0.  Lane 0 gathers what they are made of, then 16 lanes take one
// each (0 from kMlpIn on), so the logarithms run side by side.
__device__ inline void mlp_gather(const SolverState* st, int n_particles, double* arg) {
  const double d0 = st->hist_dt[0];
#pragma unroll
  for (int h = 0; h < 3; ++h) {
    const double e = st->hist_err[h];
    arg[h] = e < 1.0e-12 ? 1.0e-12 : (e > 1.0e12 ? 1.0e12 : e);
    arg[6 + h] = st->hist_acc[h];
  }
  arg[3] = d0 / (st->tf - st->t0);
  arg[4] = st->hist_dt[1] / d0;
  arg[5] = st->hist_dt[2] / d0;
  arg[9] = static_cast<double>(n_particles);
}
__device__ inline float mlp_feature(const MlpInfer* M, const double* arg, int i) {
  if (i >= kMlpIn) return 0.0f;
  const double f = i >= 6 && i < 9 ? arg[i] : std::log(arg[i]);
  const float raw = std::isfinite(f) ? static_cast<float>(f) : 0.0f;
  return (raw - M->mean[i]) * M->inv_std[i];
}

// An attempt's end by one wave (every lane calls): judge and step on lane 0
// (`sum` is read there), the learned controller's features and network on all
// lanes.  `st`, in LDS, is this wave's alone to change.
__device__ inline void ctrl_attempt_wave(SolverState* st, const Tableau& T, double sum,
                                         size_t n_var, double* times, double* trace,
                                         const MlpInfer* M, int n_particles, MlpRowLds* lds) {
  const int lane = threadIdx.x & 63;
  const MlpRowWeights w = mlp_row_weights(M);
  bool accept = false, judged = false;
  if (lane == 0) {
    judged = ctrl_judge(st, T, sum, n_var, times, trace, &accept);
    mlp_gather(st, n_particles, lds->arg);
  }
  wave_lds_fence();
  const float f = mlp_feature(M, lds->arg, lane < 16 ? lane : 15);
  if (lane < 16) lds->x[lane] = f;
  const float out = mlp_row_forward(w, lds->x, lds->h);
  ctrl_step_wave(st, judged, accept, mlp_ratio(out));
}

// The solve state from global memory to LDS and back, by one wave: the
// controller's reads and writes of it follow one another, each a memory latency.
static_assert(sizeof(SolverState) % 8 == 0 && sizeof(SolverState) <= 64 * 8, "one word a lane");
__device__ inline void state_words(SolverState* to, const SolverState* from) {
  const int lane = threadIdx.x & 63;
  if (lane < static_cast<int>(sizeof(SolverState) / 8))
    reinterpret_cast<uint64_t*>(to)[lane] = reinterpret_cast<const uint64_t*>(from)[lane];
  wave_lds_fence();
}

// The published inference copy of a network handle (mlp_kernels.hip).
const MlpInfer* mlp_infer_ptr(const odehip_mlp* m);
// Device the network was created on (its buffers live there).
int mlp_device(const odehip_mlp* m);

// Stores the normalised features of row `row` (0..15) of a tile.
__device__ inline void mlp_tile_set_row(const MlpInfer* M, MlpTileLds& t,
                                        int row, const float* raw) {
#pragma unroll
  for (int i = 0; i < 16; ++i)
    t.x[row][i] = i < kMlpIn ? (raw[i] - M->mean[i]) * M->inv_std[i] : 0.0f;
}

}  // namespace odehip
