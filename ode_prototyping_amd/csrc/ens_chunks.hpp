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
