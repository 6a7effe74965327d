// Partner chunks of the batched kernels' reorderable right-hand sides (fast,
// mixed): device functions shared by the lockstep kernels, whose partners are
// read at wave-uniform addresses through scalar loads, and the one-workgroup
// kernel, whose partners are in LDS.
#pragma once

#include "ensemble.hpp"
#include "nbody_terms.hpp"

namespace odehip {

// Each target's sum is the sum, in order, of the sums over chunks of kEnsChunk
// partners, and a chunk's is the sum, in order, of the sums over its groups of
// kEnsGroup partners taken in increasing j.  The order does not depend on who
// computes which group or chunk, so one wave walking every chunk, several
// waves sharing a tile and the one-workgroup kernel give the same bits.
constexpr int kEnsGroup = 32;
static_assert(kEnsChunk % kEnsGroup == 0, "chunks are whole groups");

// U partners of one lane, coordinates c and masses m already loaded: displacements
// and m r^-3 of fast_term (nbody_terms.hpp) step by step for all of them, so that a
// wave that has its SIMD to itself does not wait out each partner's chain of a dozen
// instructions (one partner after the other took 200 cycles each).
template <bool kMass, int U>
__device__ __forceinline__ void fast_weights(const double (&c)[3 * U], const double (&m)[U],
                                             double xi, double yi, double zi, double eps2,
                                             double (&dx)[U], double (&dy)[U], double (&dz)[U],
                                             double (&w)[U]) {
  double r2[U], y0[U], y2[U], e[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    dx[u] = c[3 * u] - xi;
    dy[u] = c[3 * u + 1] - yi;
    dz[u] = c[3 * u + 2] - zi;
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
    r2[u] = __builtin_fma(dx[u], dx[u],
                          __builtin_fma(dy[u], dy[u], __builtin_fma(dz[u], dz[u], eps2)));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < U; ++u) y0[u] = __builtin_amdgcn_rsq(r2[u]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < U; ++u) y2[u] = y0[u] * y0[u];
#pragma unroll
  for (int u = 0; u < U; ++u) e[u] = __builtin_fma(-r2[u], y2[u], 1.0);
#pragma unroll
  for (int u = 0; u < U; ++u) y0[u] = y2[u] * (kMass ? y0[u] * m[u] : y0[u]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < U; ++u) e[u] = e[u] * __builtin_fma(e[u], 1.25, 1.0);
#pragma unroll
  for (int u = 0; u < U; ++u) w[u] = __builtin_fma(y0[u] * e[u], 1.5, y0[u]);
}

// Their terms summed in increasing j.
template <bool kMass, bool kGuard, int U>
__device__ __forceinline__ void fast_terms(const double (&c)[3 * U], const double (&m)[U], int j,
                                           int i, double xi, double yi, double zi, double eps2,
                                           double& ax, double& ay, double& az) {
  double dx[U], dy[U], dz[U], w[U];
  fast_weights<kMass, U>(c, m, xi, yi, zi, eps2, dx, dy, dz, w);
  if (kGuard) {
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = j + u == i ? 0.0 : w[u];
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    ax = __builtin_fma(dx[u], w[u], ax);
    ay = __builtin_fma(dy[u], w[u], ay);
    az = __builtin_fma(dz[u], w[u], az);
  }
}

// The same for mixed_term_fp32.
template <bool kMass, bool kGuard, int U>
__device__ __forceinline__ void mixed_terms(const double (&c)[3 * U], const double (&m)[U], int j,
                                            int i, double xi, double yi, double zi, float eps2f,
                                            float& fx, float& fy, float& fz) {
  float dx[U], dy[U], dz[U], r2[U], w[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    dx[u] = static_cast<float>(c[3 * u] - xi);
    dy[u] = static_cast<float>(c[3 * u + 1] - yi);
    dz[u] = static_cast<float>(c[3 * u + 2] - zi);
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
    r2[u] = __builtin_fmaf(dx[u], dx[u],
                           __builtin_fmaf(dy[u], dy[u], __builtin_fmaf(dz[u], dz[u], eps2f)));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float rinv = __builtin_amdgcn_rsqf(r2[u]);
    w[u] = (rinv * rinv) * rinv;
    if (kMass) w[u] *= static_cast<float>(m[u]);
    if (kGuard) w[u] = j + u == i ? 0.0f : w[u];
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    fx = __builtin_fmaf(dx[u], w[u], fx);
    fy = __builtin_fmaf(dy[u], w[u], fy);
    fz = __builtin_fmaf(dz[u], w[u], fz);
  }
}

// The sum over one group of `count` partners from j0 on, in LDS at p (3 doubles
// each) with masses at m; p, m, j0 and count may differ between the lanes.  U
// partners a step: more of them hide a lone wave's latencies, fewer leave room for
// other waves.
template <int kVariant, bool kMass, bool kGuard, int U>
__device__ __forceinline__ void lds_group(const __attribute__((address_space(3))) double* p,
                                          const __attribute__((address_space(3))) double* m,
                                          int j0, int count, int i, double xi, double yi,
                                          double zi, double eps2, double& ax, double& ay,
                                          double& az) {
  float fx = 0.0f, fy = 0.0f, fz = 0.0f;
  ax = ay = az = 0.0;
  const float eps2f = static_cast<float>(eps2);
  int q = 0;
  for (; q + U <= count; q += U) {
    double c[3 * U], ms[U];
#pragma unroll
    for (int v = 0; v < 3 * U; ++v) c[v] = p[3 * q + v];
#pragma unroll
    for (int u = 0; u < U; ++u) ms[u] = kMass ? m[q + u] : 1.0;
    if constexpr (kVariant == ODEHIP_NBODY_FAST)
      fast_terms<kMass, kGuard, U>(c, ms, j0 + q, i, xi, yi, zi, eps2, ax, ay, az);
    else
      mixed_terms<kMass, kGuard, U>(c, ms, j0 + q, i, xi, yi, zi, eps2f, fx, fy, fz);
  }
  for (; q < count; ++q) {
    const double mj = kMass ? m[q] : 1.0;
    if constexpr (kVariant == ODEHIP_NBODY_FAST)
      fast_term<kMass, kGuard>(p[3 * q], p[3 * q + 1], p[3 * q + 2], mj, j0 + q, i, xi, yi, zi,
                               eps2, ax, ay, az);
    else
      mixed_term_fp32<kMass, kGuard>(p[3 * q], p[3 * q + 1], p[3 * q + 2],
                                     static_cast<float>(mj), j0 + q, i, xi, yi, zi, eps2f, fx,
                                     fy, fz);
  }
  if constexpr (kVariant != ODEHIP_NBODY_FAST) {
    ax = static_cast<double>(fx);
    ay = static_cast<double>(fy);
    az = static_cast<double>(fz);
  }
}

// P: pointer to the partners' coordinates and masses (scalar loads or LDS).

// fast: partners j0 .. j1 - 1 (of one group) summed into p* (which the caller
// zeroes).
template <bool kMass, bool kGuard, int TPL, typename P>
__device__ inline void fast_group(P yu, P mu, int j0, int j1,
                                  const int* ic, const double* xi, const double* yi,
                                  const double* zi, double eps2, double* px, double* py,
                                  double* pz) {
  constexpr int U = TPL == 1 ? 8 : 4;
  int j = j0;
  for (; j + U <= j1; j += U) {
    const P pp = yu + 3 * j;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const double mj = kMass ? mu[j + u] : 1.0;
#pragma unroll
      for (int t = 0; t < TPL; ++t)
        fast_term<kMass, kGuard>(pp[3 * u], pp[3 * u + 1], pp[3 * u + 2], mj, j + u,
                                 ic[t], xi[t], yi[t], zi[t], eps2, px[t], py[t], pz[t]);
    }
  }
  for (; j < j1; ++j) {
    const double mj = kMass ? mu[j] : 1.0;
#pragma unroll
    for (int t = 0; t < TPL; ++t)
      fast_term<kMass, kGuard>(yu[3 * j], yu[3 * j + 1], yu[3 * j + 2], mj, j, ic[t],
                               xi[t], yi[t], zi[t], eps2, px[t], py[t], pz[t]);
  }
}

// fast: partners j0 .. j1 - 1 (j0 a multiple of kEnsGroup) summed by groups into
// p* (which the caller zeroes).
template <bool kMass, bool kGuard, int TPL, typename P>
__device__ inline void fast_chunk(P yu, P mu, int j0, int j1, const int* ic, const double* xi,
                                  const double* yi, const double* zi, double eps2, double* px,
                                  double* py, double* pz) {
  for (int g0 = j0; g0 < j1; g0 += kEnsGroup) {
    double gx[TPL], gy[TPL], gz[TPL];
#pragma unroll
    for (int t = 0; t < TPL; ++t) gx[t] = gy[t] = gz[t] = 0.0;
    fast_group<kMass, kGuard, TPL>(yu, mu, g0, min(j1, g0 + kEnsGroup), ic, xi, yi, zi, eps2,
                                   gx, gy, gz);
#pragma unroll
    for (int t = 0; t < TPL; ++t) {
      px[t] += gx[t];
      py[t] += gy[t];
      pz[t] += gz[t];
    }
  }
}

// mixed: FP64 displacement rounded to FP32, FP32 pair force, partial sums
// in FP32 flushed into FP64 after every group.  kNear: near pairs (FP32
// r^2 < near2) are left out of the FP32 sums and their FP64 term is added
// into the FP64 sums; without it every pair is FP32.
// Partners j0 .. j1 - 1 (j0 a multiple of kEnsGroup) summed into the FP64
// sums a* (which the caller zeroes).
template <bool kMass, bool kGuard, bool kNear, int TPL, typename P>
__device__ inline void mixed_chunk(P yu, P mu, int j0, int j1,
                                   const int* ic, const double* xi, const double* yi,
                                   const double* zi, double eps2, float near2, double* ax,
                                   double* ay, double* az) {
  constexpr int U = 8;
  const float eps2f = static_cast<float>(eps2);
  int j = j0;
  while (j < j1) {
    const int jstop = min(j1, j + kEnsGroup);
    float fx[TPL], fy[TPL], fz[TPL];
#pragma unroll
    for (int t = 0; t < TPL; ++t) fx[t] = fy[t] = fz[t] = 0.0f;
    if constexpr (!kNear) {
      for (; j + U <= jstop; j += U) {
        const P pp = yu + 3 * j;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float mj = kMass ? static_cast<float>(mu[j + u]) : 1.0f;
#pragma unroll
          for (int t = 0; t < TPL; ++t)
            mixed_term_fp32<kMass, kGuard>(pp[3 * u], pp[3 * u + 1], pp[3 * u + 2], mj,
                                           j + u, ic[t], xi[t], yi[t], zi[t], eps2f, fx[t],
                                           fy[t], fz[t]);
        }
      }
      for (; j < jstop; ++j) {
        const float mj = kMass ? static_cast<float>(mu[j]) : 1.0f;
#pragma unroll
        for (int t = 0; t < TPL; ++t)
          mixed_term_fp32<kMass, kGuard>(yu[3 * j], yu[3 * j + 1], yu[3 * j + 2], mj, j,
                                         ic[t], xi[t], yi[t], zi[t], eps2f, fx[t], fy[t],
                                         fz[t]);
      }
    } else {
      for (; j + U <= jstop; j += U) {
        const P pp = yu + 3 * j;
        // bit u: some lane has partner j + u in the near field of one of its targets
        uint32_t near = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const double mj = kMass ? mu[j + u] : 1.0;
          uint64_t lanes = 0;
#pragma unroll
          for (int t = 0; t < TPL; ++t)
            lanes |= ballot_not(mixed_term<kMass, kGuard>(pp[3 * u], pp[3 * u + 1],
                                                          pp[3 * u + 2], mj, j + u, ic[t],
                                                          xi[t], yi[t], zi[t], eps2f, near2,
                                                          fx[t], fy[t], fz[t]));
          near |= lanes ? (1u << u) : 0u;
        }
#pragma unroll
        for (int t = 0; t < TPL; ++t) {
          fx[t] = opaque(fx[t]);
          fy[t] = opaque(fy[t]);
          fz[t] = opaque(fz[t]);
        }
        if (near) {
          double xo[TPL], yo[TPL], zo[TPL];
#pragma unroll
          for (int t = 0; t < TPL; ++t) {
            xo[t] = opaque(xi[t]);
            yo[t] = opaque(yi[t]);
            zo[t] = opaque(zi[t]);
          }
          do {
            const int u = __builtin_ctz(near);
            near &= near - 1;
            const double mj = kMass ? mu[j + u] : 1.0;
#pragma unroll
            for (int t = 0; t < TPL; ++t)
              mixed_near_term<kMass, kGuard>(pp[3 * u], pp[3 * u + 1], pp[3 * u + 2], mj,
                                             j + u, ic[t], xo[t], yo[t], zo[t], eps2f, eps2,
                                             near2, ax[t], ay[t], az[t]);
          } while (near);
        }
      }
      for (; j < jstop; ++j) {
        const double mj = kMass ? mu[j] : 1.0;
#pragma unroll
        for (int t = 0; t < TPL; ++t)
          if (!mixed_term<kMass, kGuard>(yu[3 * j], yu[3 * j + 1], yu[3 * j + 2], mj, j,
                                         ic[t], xi[t], yi[t], zi[t], eps2f, near2, fx[t],
                                         fy[t], fz[t]))
            mixed_near_term<kMass, kGuard>(yu[3 * j], yu[3 * j + 1], yu[3 * j + 2], mj, j,
                                           ic[t], xi[t], yi[t], zi[t], eps2f, eps2, near2,
                                           ax[t], ay[t], az[t]);
      }
    }
#pragma unroll
    for (int t = 0; t < TPL; ++t) {
      ax[t] += static_cast<double>(fx[t]);
      ay[t] += static_cast<double>(fy[t]);
      az[t] += static_cast<double>(fz[t]);
    }
  }
}

}  // namespace odehip
