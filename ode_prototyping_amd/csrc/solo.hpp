// One-workgroup solves of small systems (solo_kernels.hip): arguments, LDS use
// and the sizes they take.
#pragma once

#include <algorithm>

#include "ensemble.hpp"
#include "mlp.hpp"

namespace odehip {

constexpr int kSoloWaves = 16;    // at most, per workgroup
constexpr int kSoloTerms = 4;     // exact: partners per wave and block
constexpr int kSoloMaxN = 320;    // fast, mixed: 192 threads per 64 targets
constexpr int kSoloExactN = 128;  // an ensemble's systems: sizes up to which it takes them
constexpr int kSoloSumN = 256;
// exact, a solve of its own: one tile of targets (DOPRI5 / DOP853, launched attempts
// against one workgroup: 64 bodies 21.6 / 24.4 against 12.8 / 16.1 ms; with a second
// tile, 80 bodies 21.5 / 25.2 against 23.4 / 30.7, 128 bodies 11.7 / 14.2 against 17.3 /
// 27.9)
constexpr int kSoloOneExactN = 64;
// fast, a solve of its own: two tiles of targets by 16 waves (DOPRI5 / DOP853,
// launched attempts against one workgroup: 64 bodies 22.3 / 25.2 against 8.6 /
// 10.3 ms, 128 bodies 10.2 / 11.9 against 8.6 / 11.4; with three tiles on, 180 bodies,
// 7.2 / 9.1 against 17.4 / 25.4)
constexpr int kSoloOneFastN = 128;
constexpr uint64_t kSoloTicks = 200000;  // of the 100 MHz clock: 2 ms a launch
constexpr int kSoloMaxQuads = 4 * ((6 * kSoloMaxN + ODEHIP_REDUCE_GROUP - 1) / ODEHIP_REDUCE_GROUP);
// LDS of a CU less the kernel's static use and some to spare.
constexpr int kSoloLdsDoubles = (160 * 1024 - 2048) / 8;

struct SoloArgs {
  const EnsSys* sys;   // systems' table, or null: the one system `one`
  const int* list;     // system per workgroup, or null (with sys null)
  EnsSys one;
  SolverState* st;
  double* xb0;
  double* xb1;
  double* ks;          // its first stage vector holds a kept k1 between launches
  double* kfsal;
  const double* mass;
  const double* atol_v;  // per element (one system), or null: atol, rtol
  const double* rtol_v;
  double atol, rtol;
  double* times;
  double* trace;
  long trace_cap;      // per system of `trace`
  const MlpInfer* mlp;
  int* n_active;       // counted down as systems end, or null
  double eps2;
  double near_c;
  int tableau;
  int lds_doubles;     // set by launch_solo
};

// LDS of a system of n bodies: state, stage input, S stage vectors, masses, the
// partial sums of the waves and the learned controller's network.
__host__ __device__ constexpr int solo_sums(int variant) {
  return variant == ODEHIP_NBODY_EXACT ? 3 * 64 * kSoloTerms : 192;
}
__host__ __device__ inline int solo_lds_doubles(int n, int S, int variant, int waves,
                                                bool learned) {
  static_assert(sizeof(MlpInfer) % 8 == 0, "copied by doubles");
  return (S + 2) * 6 * n + ((n + 1) & ~1) + waves * solo_sums(variant) +
         (learned ? static_cast<int>(sizeof(MlpInfer) / 8) : 0);
}

// Waves of the workgroup for systems of up to n bodies, 0 if they do not fit.
inline int solo_waves(int n, int S, int variant, bool learned) {
  if (n < 1 || n > kSoloMaxN) return 0;
  for (int w : {kSoloWaves, 8}) {
    // fast, mixed: a thread per target and coordinate; more waves than units
    // of 64 targets and 32 partners would only wait
    if (variant != ODEHIP_NBODY_EXACT) {
      if (w == kSoloWaves && n <= 128) continue;
      if (192 * ((n + 63) / 64) > 64 * w) continue;
    }
    if (solo_lds_doubles(n, S, variant, w, learned) <= kSoloLdsDoubles) return w;
  }
  return 0;
}

// Bodies up to which a solve is one workgroup's.
inline int solo_limit(int S, int variant, bool learned) {
  const int want = variant == ODEHIP_NBODY_EXACT ? kSoloExactN : kSoloSumN;
  for (int n = want; n > 0; --n)
    if (solo_waves(n, S, variant, learned) > 0) return n;
  return 0;
}

// The same for a solve of its own (odehip_rk_solve).
inline int solo_one_limit(int S, int variant, bool learned) {
  const int all = solo_limit(S, variant, learned);
  switch (variant) {
    case ODEHIP_NBODY_EXACT: return std::min(all, kSoloOneExactN);
    case ODEHIP_NBODY_FAST: return std::min(all, kSoloOneFastN);
    default: return 0;  // mixed: the launched kernels' sums have another order
  }
}

// One launch: `blocks` systems of at most n_max bodies.
hipError_t launch_solo(const SoloArgs& a, int n_max, int variant, unsigned blocks,
                       hipStream_t s);
hipError_t upload_solo_tableau(int id, const Tableau& T);

}  // namespace odehip
