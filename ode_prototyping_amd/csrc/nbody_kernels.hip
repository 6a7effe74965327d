// N-body gravity right-hand side on gfx950 (CDNA4): dxdt = [vel | acc(pos)]
// for the state layout of src/ode/NBodyODE.hpp:12-19 (positions then
// velocities, xyz interleaved per particle), G = 1, Plummer softening.
//
// The reference evaluates the N(N-1)/2 pairs in parallel and scatters six
// FP64 atomic adds per pair (NBodyODE.hpp:68-133).  Here every kernel is an
// atomic-free gather: a workgroup owns a tile of 64 target particles (one per
// lane) and streams the partner particles j; partner coordinates are
// wave-uniform, so they arrive through scalar loads into SGPRs and cost no
// VGPR bandwidth or LDS (the exact kernels for smaller grids have their own
// layouts).
//
//  * exact:  the reference's FP64 expression (((dx^2 + dy^2) + dz^2) + eps^2,
//            correctly rounded sqrt, den = dist * dist_sq, three correctly
//            rounded divisions) and, per target, the partners summed in
//            increasing j -- the order the single-threaded pair loop adds into
//            acc[i] (nbody_exact.hpp).  Result: bit-identical to NBodyODE with
//            SingleThreadedExecutor, but for the few quotients that
//            nbody_terms.hpp names.  Must be compiled with -ffp-contract=off.
//  * fast:   FP64, r^-3 from the hardware reciprocal square root with a
//            third-order correction (a few ulp), FMA accumulation, the j range
//            split over 16 waves per workgroup and the partial sums combined
//            in a fixed order (deterministic, not bit-identical).
//  * mixed:  displacement computed in FP64 and rounded to FP32, r^-3 and the
//            pair force in FP32 (hardware rsqrt), per-wave partial sums in
//            FP32 flushed into FP64 accumulators every 32 partners; near pairs
//            (r^2 below a per-launch threshold) in FP64, summed in FP64.
#include <algorithm>

#include "internal.hpp"
#include "nbody_terms.hpp"
#include "rk_device.hpp"

namespace odehip {
namespace {

// Partner data is read at wave-uniform addresses and never written during a
// launch; reading it through the constant address space lets the compiler
// use scalar loads (SGPR results broadcast to all lanes for free).
typedef const __attribute__((address_space(4))) double* uniform_ptr;
__device__ inline uniform_ptr as_uniform(const double* p) {
  return (uniform_ptr)(p);
}

__device__ inline const double* select_input(const NBodyArgs& a) {
  if (a.y) return a.y;
  return a.st->cur ? a.xb1 : a.xb0;
}

// built-in tableaux, then the slots of registered ones
__constant__ Tableau n_tab[ODEHIP_MAX_TABLEAUS] = {
    kTableaus[0], kTableaus[1], kTableaus[2],
    kTableaus[3], kTableaus[4], kTableaus[5]};

// The kernel's arguments (NBodyArgs its only parameter), read again: what only
// the end of a kernel needs does not hold SGPRs through the partner loop.
__device__ inline NBodyArgs late_args() {
  typedef const __attribute__((address_space(4))) NBodyArgs* args_ptr;
  args_ptr p = (args_ptr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  NBodyArgs a;
  __builtin_memcpy(&a, (const void*)p, sizeof a);
  return a;
}

// Element e of the result, and of the next stage's input (L: next_stage).
template <int L>
__device__ inline void put(const NBodyArgs& a, long e, double v) {
  a.k[e] = v;
  if (!a.next.y) return;
  if (a.next.n >= 0) {
    next_stage<L>(a.next, n_tab[a.next.tab], 6 * static_cast<size_t>(a.n), e, v,
                  (a.st->cur ? a.xb1 : a.xb0)[e], a.st->dt);
    return;
  }
  // update_velocity_kernel, then the next step's update_position_kernel
  // (LeapfrogParallel.hpp:57-68)
  const long p = e - 3L * a.n;
  if (p < 0) return;
  const double dt = a.leap_dt, x = a.y[p];
  const double vel = a.y[e] + 0.5 * dt * (a.next.ks[p] + v);
  a.next.y[e] = vel;
  a.next.y[p] = a.next.n == kLeapMove ? x + dt * (vel + 0.5 * dt * v) : x;
}

// Returns true if the launch has nothing to compute (solve finished, or k1
// of this attempt is reused, or a dense-output evaluation whose pass does not
// run).  On k1 reuse the launch copies k1 instead, unless it is in place, and
// forms the next stage's input.
__device__ inline bool prologue_skip(const NBodyArgs& a) {
  if (!a.st) return false;
  if (a.stage0 == 2) return a.st->dense_go == 0;
  if (a.st->done) return true;
  if (a.stage0 && a.st->k1_valid) {
    const double* from = a.st->k1_valid == 1 ? a.kfsal : a.k;
    const long n_var = static_cast<long>(a.n) * 6;
    for (long e = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; e < n_var;
         e += static_cast<long>(gridDim.x) * blockDim.x)
      put<kStageLoadsLean>(a, e, from[e]);
    return true;
  }
  return false;
}

// dxdt[0:3N] = x[3N:6N] for `count` particles from i0
// (nbody_init_dxdt_kernel, NBodyODE.hpp:51-56): one element per thread, loaded
// at the start and written at the end (the load's latency passes meanwhile).
// The threads before `first` write accelerations; a workgroup too small for
// both starts from thread 0.
struct Velocity {
  long e;  // -1: none
  double v;
};
__device__ inline Velocity load_velocity(const NBodyArgs& a, const double* __restrict__ y,
                                         int i0, int count, int first) {
  const int t = static_cast<int>(threadIdx.x) -
                (first + 3 * count <= static_cast<int>(blockDim.x) ? first : 0);
  const long e = 3L * i0 + t, lim = 3L * a.n;
  if (t < 0 || t >= 3 * count || e >= lim) return Velocity{-1, 0.0};
  return Velocity{e, y[lim + e]};
}
template <int L>
__device__ inline void put_velocity(const NBodyArgs& a, const Velocity& v) {
  if (v.e >= 0) put<L>(a, v.e, v.v);
}

// Whether every position coordinate of the state passes coord_shared_ok:
// all threads of the workgroup test a strided share of the 3N coordinates.
__device__ inline bool all_positions_shared_ok(const double* __restrict__ y, int n) {
  const bool ok = strided_all_shared_ok(y, 3L * n, threadIdx.x, blockDim.x);
  return __syncthreads_and(ok) != 0;
}

// The common mass when all n masses are one power of two 2^k with |k| <= 300,
// else 0 (every thread tests a strided share).  Then the per-term mass factor
// can move out of the sum: 2^k t is exact, and scaling by 2^k commutes with
// every rounding of the in-order sum while the values stay normal, so
// sum_j (2^k t_j) equals 2^k (sum_j t_j) bit for bit.  On the shared-
// reciprocal path every nonzero term is >= 2^-602 in magnitude and every
// nonzero partial sum >= 2^-654 (a multiple of its operands' ulp), at most
// 2^430, so |k| <= 300 keeps all of them normal and finite.
__device__ inline double uniform_pow2_mass(const double* __restrict__ mass, int n) {
  const uint64_t b0 = __builtin_bit_cast(uint64_t, mass[0]);
  const uint64_t ex = b0 >> 52;  // sign 0 and the biased exponent
  bool ok = (b0 & 0x000fffffffffffffull) == 0 && ex >= 1023 - 300 && ex <= 1023 + 300;
  ok = ok & strided_all_bits(mass, n, threadIdx.x, blockDim.x, b0);
  return __syncthreads_and(ok) != 0 ? mass[0] : 0.0;
}

// ------------------------------------------------------------------- fast --
constexpr int kFastWaves = 16;

// Two 16-wave workgroups share a CU only while a wave's SGPRs fit eighty: the
// SIMD's 800 hold eight waves of 80 and the 16 the trap handler keeps per wave.
// (With 88, which the compiler counts as eight waves too, 65536 bodies took 2584
// instead of 2391 us.)
#define ODEHIP_EIGHT_WAVES_SGPRS __attribute__((amdgpu_num_sgpr(80)))

// kFastSet partners' coordinates (and masses), wave-uniform in SGPRs.
constexpr int kFastSet = 4;
template <bool kMass>
struct FastSet {
  double c[3 * kFastSet];
  double m[kMass ? kFastSet : 1];
};

template <bool kMass>
__device__ __forceinline__ void fast_load(FastSet<kMass>& s, uniform_ptr yu, uniform_ptr mass,
                                          int j) {
  const uniform_ptr pp = yu + 3 * j;
#pragma unroll
  for (int e = 0; e < 3 * kFastSet; ++e) s.c[e] = pp[e];
  if constexpr (kMass) {
#pragma unroll
    for (int u = 0; u < kFastSet; ++u) s.m[u] = mass[j + u];
  }
}

template <bool kMass, bool kGuard>
__device__ __forceinline__ void fast_set_terms(const FastSet<kMass>& s, int j, int i, double xi,
                                               double yi, double zi, double eps2, double& ax,
                                               double& ay, double& az) {
#pragma unroll
  for (int u = 0; u < kFastSet; ++u)
    fast_term<kMass, kGuard>(s.c[3 * u], s.c[3 * u + 1], s.c[3 * u + 2], kMass ? s.m[u] : 1.0,
                             j + u, i, xi, yi, zi, eps2, ax, ay, az);
}

// Waits for every scalar load issued so far.  Scalar loads complete out of
// order, so the wait counter cannot single out an older set while a newer one
// is in flight: the partner loop therefore drains the set it is about to use
// (issued one set earlier) before it issues the next.  The scheduling
// barriers keep the wait where it is written: after the previous set's terms
// and before the next set's loads.
__device__ __forceinline__ void scalar_loads_drain() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); vector and export counters untouched
  __builtin_amdgcn_sched_barrier(0);
}

}  // namespace
}  // namespace odehip

#include "nbody_exact.hpp"

namespace odehip {
namespace {

// Partners jbeg .. jend - 1 of target i in increasing j (wave-uniform scalar
// loads); kMass: per-term masses.  kPrefetch: full sets of kFastSet partners
// alternate between two SGPR sets, each loaded while the other's terms are
// computed -- worth it with 4 waves per SIMD (one workgroup per CU), whose
// scalar-load waits the other waves cannot cover; with 8 waves per SIMD the
// extra waits cost more than they hide, and steps of 8 partners that load and
// then wait are faster.  Both add the terms in the same order.
template <bool kMass, bool kGuard, bool kPrefetch>
__device__ __forceinline__ void fast_partners(uniform_ptr yu, uniform_ptr mass, int jbeg,
                                              int jend, int i, double xi, double yi,
                                              double zi, double eps2, double& ax, double& ay,
                                              double& az) {
  constexpr int U = kFastSet;
  int j = jbeg;
  if constexpr (!kPrefetch) {
    for (; j + 8 <= jend; j += 8) {
      const uniform_ptr pp = yu + 3 * j;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const double mj = kMass ? mass[j + u] : 1.0;
        fast_term<kMass, kGuard>(pp[3 * u], pp[3 * u + 1], pp[3 * u + 2], mj, j + u, i, xi,
                                 yi, zi, eps2, ax, ay, az);
      }
    }
  } else if (j + U <= jend) {
    FastSet<kMass> a, b;
    fast_load<kMass>(a, yu, mass, j);
    // a holds partners j .. j + U - 1 (j + U <= jend); the next two sets are in range
    for (; j + 3 * U <= jend; j += 2 * U) {
      scalar_loads_drain();
      fast_load<kMass>(b, yu, mass, j + U);
      __builtin_amdgcn_sched_barrier(0);  // issue the loads before the terms
      fast_set_terms<kMass, kGuard>(a, j, i, xi, yi, zi, eps2, ax, ay, az);
      scalar_loads_drain();
      fast_load<kMass>(a, yu, mass, j + 2 * U);
      __builtin_amdgcn_sched_barrier(0);
      fast_set_terms<kMass, kGuard>(b, j + U, i, xi, yi, zi, eps2, ax, ay, az);
    }
    scalar_loads_drain();
    fast_set_terms<kMass, kGuard>(a, j, i, xi, yi, zi, eps2, ax, ay, az);
    j += U;
  }
  for (; j < jend; ++j) {
    const double mj = kMass ? mass[j] : 1.0;
    fast_term<kMass, kGuard>(yu[3 * j], yu[3 * j + 1], yu[3 * j + 2], mj, j, i, xi,
                             yi, zi, eps2, ax, ay, az);
  }
}

// The common mass when all n masses are equal (finite, nonzero), else 0
// (a workgroup vote over strided shares).
__device__ inline double workgroup_uniform_mass(const double* __restrict__ mass, int n) {
  const bool ok = lane_masses_uniform<kScanLoadsLean>(mass, n, threadIdx.x, blockDim.x);
  return __syncthreads_and(ok) != 0 ? mass[0] : 0.0;
}

template <bool kMass, bool kGuard, bool kPrefetch>
__device__ __forceinline__ void fast_kernel(const NBodyArgs& a) {
  if (prologue_skip(a)) return;
  __shared__ double red[kFastWaves][3][64];
  const double* __restrict__ y = select_input(a);
  const uniform_ptr yu = as_uniform(y);
  const uniform_ptr mass = as_uniform(a.mass);
  const int n = a.n;
  const double eps2 = a.eps2;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = blockIdx.x * 64;
  const int i = i0 + lane;
  const bool valid_i = i < n;
  const int ic = valid_i ? i : n - 1;
  const double xi = y[3 * ic], yi = y[3 * ic + 1], zi = y[3 * ic + 2];
  const int seg = (n + kFastWaves - 1) / kFastWaves;
  const int jbeg = min(n, wave * seg);
  const int jend = min(n, jbeg + seg);
  // equal masses: unit-mass terms and one scale of each finished sum
  const double m_uni = kMass ? workgroup_uniform_mass(a.mass, n) : 0.0;
  double ax = 0.0, ay = 0.0, az = 0.0;
  if (kMass && m_uni == 0.0)
    fast_partners<true, kGuard, kPrefetch>(yu, mass, jbeg, jend, i, xi, yi, zi, eps2, ax, ay,
                                           az);
  else
    fast_partners<false, kGuard, kPrefetch>(yu, mass, jbeg, jend, i, xi, yi, zi, eps2, ax, ay,
                                            az);
  red[wave][0][lane] = ax;
  red[wave][1][lane] = ay;
  red[wave][2][lane] = az;
  const NBodyArgs late = late_args();
  __syncthreads();
  if (wave < 3 && valid_i) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kFastWaves; ++w) s += red[w][wave][lane];
    put<kStageLoadsLean>(late, 3L * n + 3 * i + wave, kMass && m_uni != 0.0 ? s * m_uni : s);
  }
  // (loaded only here: held through the loop, two VGPRs cost it 1.5 %)
  put_velocity<kStageLoadsLean>(late, load_velocity(late, select_input(late), i0, 64, 192));
}

template <bool kMass, bool kGuard>
__global__ __launch_bounds__(64 * kFastWaves) ODEHIP_EIGHT_WAVES_SGPRS
void k_nbody_fast(NBodyArgs a) {
  fast_kernel<kMass, kGuard, false>(a);
}
// (one workgroup per CU: the two SGPR sets may take what they need)
template <bool kMass, bool kGuard>
__global__ __launch_bounds__(64 * kFastWaves) void k_nbody_fast_prefetch(NBodyArgs a) {
  fast_kernel<kMass, kGuard, true>(a);
}

// The fast sum for grids of 64-target workgroups that would leave CUs empty: R
// targets per workgroup, wave-uniform; each lane takes one partner of every 64
// and sums its terms for the R targets, and the lanes' sums are folded at the
// end.  n / R workgroups of W waves: 1000 bodies take 3.3 us instead of 13, 4096
// 17 instead of 40, 8192 57 instead of 85.  Per-term masses throughout: finding
// that they are equal would cost a second memory latency.
constexpr int kFastRowsWaves = 8;

// {a's lower half | b's lower half} and {a's upper | b's upper}, halves of the
// wave (32 lanes) or of each pair of rows (16 lanes).
__device__ __forceinline__ void swap_halves(double a, double b, double& lo, double& hi) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
  const auto l = __builtin_amdgcn_permlane32_swap(static_cast<uint32_t>(x),
                                                  static_cast<uint32_t>(y), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(static_cast<uint32_t>(x >> 32),
                                                  static_cast<uint32_t>(y >> 32), false, false);
  lo = __builtin_bit_cast(double, (static_cast<uint64_t>(h[0]) << 32) | l[0]);
  hi = __builtin_bit_cast(double, (static_cast<uint64_t>(h[1]) << 32) | l[1]);
}
__device__ __forceinline__ void swap_rows(double a, double b, double& lo, double& hi) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
  const auto l = __builtin_amdgcn_permlane16_swap(static_cast<uint32_t>(x),
                                                  static_cast<uint32_t>(y), false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(static_cast<uint32_t>(x >> 32),
                                                  static_cast<uint32_t>(y >> 32), false, false);
  lo = __builtin_bit_cast(double, (static_cast<uint64_t>(h[0]) << 32) | l[0]);
  hi = __builtin_bit_cast(double, (static_cast<uint64_t>(h[1]) << 32) | l[1]);
}
template <int kRotate>
__device__ __forceinline__ double rotated_in_row(double v) {
  const uint64_t x = __builtin_bit_cast(uint64_t, v);
  const uint32_t l = __builtin_amdgcn_update_dpp(0, static_cast<int>(x), 0x120 + kRotate, 0xf,
                                                 0xf, true);
  const uint32_t h = __builtin_amdgcn_update_dpp(0, static_cast<int>(x >> 32), 0x120 + kRotate,
                                                 0xf, 0xf, true);
  return __builtin_bit_cast(double, (static_cast<uint64_t>(h) << 32) | l);
}

// Sums v[0 .. V - 1] over the wave's lanes into out[0 .. V - 1] (LDS).  Two
// values share each swap, so halving the lanes halves the values.
template <int V>
__device__ __forceinline__ void wave_sums(const double (&v)[V], double* out, int lane) {
  constexpr int V1 = (V + 1) / 2, V2 = (V1 + 1) / 2;
  double u[V1], w[V2];
#pragma unroll
  for (int m = 0; m < V1; ++m) {
    double lo, hi;
    swap_halves(v[2 * m], 2 * m + 1 < V ? v[2 * m + 1] : 0.0, lo, hi);
    u[m] = lo + hi;
  }
#pragma unroll
  for (int m = 0; m < V2; ++m) {
    double lo, hi;
    swap_rows(u[2 * m], 2 * m + 1 < V1 ? u[2 * m + 1] : 0.0, lo, hi);
    w[m] = lo + hi;
  }
  // row r of w[m] holds the sums of value 4 m + 2 (r & 1) + (r >> 1)
  const int r = lane >> 4;
#pragma unroll
  for (int m = 0; m < V2; ++m) {
    double s = w[m];
    s += rotated_in_row<8>(s);
    s += rotated_in_row<4>(s);
    s += rotated_in_row<2>(s);
    s += rotated_in_row<1>(s);
    const int id = 4 * m + 2 * (r & 1) + (r >> 1);
    if ((lane & 15) == 0 && id < V) out[id] = s;
  }
}

// The last workgroup's targets are the last R bodies (n >= R).
template <int R, bool kMass, bool kGuard>
__global__ __launch_bounds__(64 * kFastRowsWaves) void k_nbody_fast_rows(NBodyArgs a) {
  if (prologue_skip(a)) return;
  __shared__ double red[kFastRowsWaves][3 * R];
  const double* __restrict__ y = select_input(a);
  const uniform_ptr yu = as_uniform(y);
  const double* __restrict__ mass = a.mass;
  const int n = a.n;
  const double eps2 = a.eps2;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int step = blockDim.x;
  const int i0 = min(static_cast<int>(blockIdx.x) * R, n - R);
  const int j = min(wave * 64 + lane, n - 1);
  double px = y[3 * j], py = y[3 * j + 1], pz = y[3 * j + 2];
  double pm = kMass ? mass[j] : 1.0;
  double tx[R], ty[R], tz[R], v[3 * R];
#pragma unroll
  for (int t = 0; t < R; ++t) {
    tx[t] = yu[3 * (i0 + t)];
    ty[t] = yu[3 * (i0 + t) + 1];
    tz[t] = yu[3 * (i0 + t) + 2];
    v[3 * t] = v[3 * t + 1] = v[3 * t + 2] = 0.0;
  }
  const int e = threadIdx.x;
  const Velocity vel = load_velocity(a, y, i0, R, 3 * R);
  for (int b = wave * 64; b < n; b += step) {
    const int jn = min(b + step + lane, n - 1);  // the next partner, loaded ahead
    const double qx = y[3 * jn], qy = y[3 * jn + 1], qz = y[3 * jn + 2];
    const double qm = kMass ? mass[jn] : 1.0;
    if (b + 64 <= n) {
#pragma unroll
      for (int t = 0; t < R; ++t)
        fast_term<kMass, kGuard>(px, py, pz, pm, b + lane, i0 + t, tx[t], ty[t], tz[t], eps2,
                                 v[3 * t], v[3 * t + 1], v[3 * t + 2]);
    } else {
      // lanes past the end pass as the target itself: their terms are left out
      const bool in = b + lane < n;
#pragma unroll
      for (int t = 0; t < R; ++t)
        fast_term<kMass, true>(px, py, pz, pm, in ? (kGuard ? b + lane : -1) : i0 + t, i0 + t,
                               tx[t], ty[t], tz[t], eps2, v[3 * t], v[3 * t + 1], v[3 * t + 2]);
    }
    px = qx;
    py = qy;
    pz = qz;
    pm = qm;
  }
  wave_sums<3 * R>(v, red[wave], lane);
  __syncthreads();
  if (e < 3 * R) {
    double s = 0.0;
    for (int w = 0; w < step / 64; ++w) s += red[w][e];
    put<kStageLoads>(a, 3L * n + 3L * i0 + e, s);
  }
  put_velocity<kStageLoads>(a, vel);
}

// ------------------------------------------------------------------ mixed --
constexpr int kMixedWaves = 16;
constexpr int kMixedFlush = 32;

// Partners jbeg .. jend - 1 of target i into the FP64 sums a*: FP32 terms
// flushed every kMixedFlush partners; kNear: near pairs (FP32 r^2 < near2) in
// FP64; kMass: per-term masses.
template <bool kMass, bool kGuard, bool kNear>
__device__ __forceinline__ void mixed_partners(uniform_ptr yu, uniform_ptr mass, int jbeg,
                                               int jend, int i, double xi, double yi,
                                               double zi, float eps2f, double eps2,
                                               float near2, double& ax, double& ay,
                                               double& az) {
  int j = jbeg;
  while (j < jend) {
    const int jstop = min(jend, j + kMixedFlush);
    float fx = 0.0f, fy = 0.0f, fz = 0.0f;
    if constexpr (!kNear) {
      for (; j + 8 <= jstop; j += 8) {
        const uniform_ptr pp = yu + 3 * j;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const float mj = kMass ? static_cast<float>(mass[j + u]) : 1.0f;
          mixed_term_fp32<kMass, kGuard>(pp[3 * u], pp[3 * u + 1], pp[3 * u + 2], mj, j + u,
                                         i, xi, yi, zi, eps2f, fx, fy, fz);
        }
      }
      for (; j < jstop; ++j) {
        const float mj = kMass ? static_cast<float>(mass[j]) : 1.0f;
        mixed_term_fp32<kMass, kGuard>(yu[3 * j], yu[3 * j + 1], yu[3 * j + 2], mj, j, i, xi,
                                       yi, zi, eps2f, fx, fy, fz);
      }
    }
    for (; kNear && j + 8 <= jstop; j += 8) {
      const uniform_ptr pp = yu + 3 * j;
      // bit u: some lane has partner j + u in its near field
      uint32_t near = 0;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const double mj = kMass ? mass[j + u] : 1.0;
        const bool far = mixed_term<kMass, kGuard>(pp[3 * u], pp[3 * u + 1], pp[3 * u + 2], mj,
                                                   j + u, i, xi, yi, zi, eps2f, near2, fx, fy,
                                                   fz);
        near |= ballot_not(far) ? (1u << u) : 0u;
      }
      fx = opaque(fx);
      fy = opaque(fy);
      fz = opaque(fz);
      if (near) {
        const double xo = opaque(xi), yo = opaque(yi), zo = opaque(zi);
        do {
          const int u = __builtin_ctz(near);
          near &= near - 1;
          const double mj = kMass ? mass[j + u] : 1.0;
          mixed_near_term<kMass, kGuard>(pp[3 * u], pp[3 * u + 1], pp[3 * u + 2], mj, j + u,
                                         i, xo, yo, zo, eps2f, eps2, near2, ax, ay, az);
        } while (near);
      }
    }
    for (; kNear && j < jstop; ++j) {
      const double mj = kMass ? mass[j] : 1.0;
      if (!mixed_term<kMass, kGuard>(yu[3 * j], yu[3 * j + 1], yu[3 * j + 2], mj, j, i, xi,
                                     yi, zi, eps2f, near2, fx, fy, fz))
        mixed_near_term<kMass, kGuard>(yu[3 * j], yu[3 * j + 1], yu[3 * j + 2], mj, j, i,
                                       xi, yi, zi, eps2f, eps2, near2, ax, ay, az);
    }
    ax += static_cast<double>(fx);
    ay += static_cast<double>(fy);
    az += static_cast<double>(fz);
  }
}

// kNear: near pairs (a.near2 > 0) in FP64; without it every pair is FP32.
// kNext: a.next is set; without its code in the epilogue the partner loop is
// scheduled 3 % faster (65536 bodies 1485 -> 1430 us).
template <bool kMass, bool kGuard, bool kNear, bool kNext>
__device__ __forceinline__ void mixed_body(const NBodyArgs& a) {
  if (prologue_skip(a)) return;
  __shared__ double red[kMixedWaves][3][64];
  const double* __restrict__ y = select_input(a);
  const uniform_ptr yu = as_uniform(y);
  const uniform_ptr mass = as_uniform(a.mass);
  const int n = a.n;
  const float eps2f = static_cast<float>(a.eps2);
  const float near2 = a.near2;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = blockIdx.x * 64;
  const int i = i0 + lane;
  const bool valid_i = i < n;
  const int ic = valid_i ? i : n - 1;
  const double xi = y[3 * ic], yi = y[3 * ic + 1], zi = y[3 * ic + 2];
  const int seg = (n + kMixedWaves - 1) / kMixedWaves;
  const int jbeg = min(n, wave * seg);
  const int jend = min(n, jbeg + seg);
  // equal masses: unit-mass terms and one FP64 scale of each finished sum
  const double m_uni = kMass ? workgroup_uniform_mass(a.mass, n) : 0.0;
  double ax = 0.0, ay = 0.0, az = 0.0;
  if (kMass && m_uni == 0.0)
    mixed_partners<true, kGuard, kNear>(yu, mass, jbeg, jend, i, xi, yi, zi, eps2f, a.eps2,
                                        near2, ax, ay, az);
  else
    mixed_partners<false, kGuard, kNear>(yu, mass, jbeg, jend, i, xi, yi, zi, eps2f, a.eps2,
                                         near2, ax, ay, az);
  red[wave][0][lane] = ax;
  red[wave][1][lane] = ay;
  red[wave][2][lane] = az;
  if constexpr (kNext) {
    const NBodyArgs late = late_args();
    __syncthreads();
    if (wave < 3 && valid_i) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < kMixedWaves; ++w) s += red[w][wave][lane];
      put<kStageLoadsLean>(late, 3L * n + 3 * i + wave, kMass && m_uni != 0.0 ? s * m_uni : s);
    }
    put_velocity<kStageLoadsLean>(late, load_velocity(late, select_input(late), i0, 64, 192));
  } else {
    __syncthreads();
    if (wave < 3 && valid_i) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < kMixedWaves; ++w) s += red[w][wave][lane];
      a.k[3L * n + 3 * i + wave] = kMass && m_uni != 0.0 ? s * m_uni : s;
    }
    const long e = 3L * i0 + threadIdx.x, lim = 3L * n;
    if (threadIdx.x < 192 && e < lim) a.k[e] = y[lim + e];
  }
}

// Held to eighty SGPRs, the loop over unequal masses spills (16384 bodies with near
// field 157 instead of 151 us).  Only launches that form the next stage's input in
// more than one workgroup a CU gain by the limit; with masses they leave that to a
// launch of its own (nbody_rhs_forms_next), without them they keep it (leapfrog, 20
// steps at 65536 bodies, 37.6 instead of 38.3 ms).
template <bool kMass, bool kGuard, bool kNear, bool kNext>
__global__ __launch_bounds__(64 * kMixedWaves) void k_nbody_mixed(NBodyArgs a) {
  mixed_body<kMass, kGuard, kNear, kNext>(a);
}
template <bool kGuard, bool kNear>
__global__ __launch_bounds__(64 * kMixedWaves) ODEHIP_EIGHT_WAVES_SGPRS
void k_nbody_mixed_unit_next(NBodyArgs a) {
  mixed_body<false, kGuard, kNear, true>(a);
}

// ----------------------------------------------------------------- energy --
// Kinetic 0.5 sum m_i v_i^2 and potential -sum over pairs m_i m_j /
// sqrt(r^2 + eps^2).  A workgroup owns 64 targets, one per lane; its waves share
// the partners in units of 32 (wave-uniform scalar loads).  Each unordered pair
// of 64-body tiles is met once: tile a meets the tiles a + d, d = 0 ... nt / 2
// around the ring, with weight 1/2 for its own tile (both directions are summed
// there) and for the opposite tile of an even ring (met from both ends).
// 12 full-rate FP64 instructions and a rsqrt per pair bound it: one thread per
// target over all partners with IEEE square roots and divisions took 3600 us at
// 16384 bodies (64 workgroups), this 97, the sums and the copy out included.
constexpr int kEnergyWaves = 16;
constexpr int kEnergyUnit = 32;

// 1 / sqrt(r2) to the last bit or so; the guarded form also for r2 = 0, inf.
template <bool kGuarded>
__device__ __forceinline__ double inverse_root(double r2) {
  const double y = __builtin_amdgcn_rsq(r2);
  const double e = __builtin_fma(-(r2 * y), y, 1.0);
  const double c = __builtin_fma(e, 0.375, 0.5);
  const double z = __builtin_fma(y * e, c, y);
  return kGuarded && e != e ? y : z;
}

// sum over the unit's partners of m_j / sqrt(r^2 + eps^2), j != i.
template <bool kMass, bool kGuarded>
__device__ __forceinline__ double energy_unit(uniform_ptr yu, uniform_ptr mu, int j0, int j1,
                                              int i, bool own, double xi, double yi, double zi,
                                              double eps2) {
  double pe = 0.0;
#pragma unroll 4
  for (int j = j0; j < j1; ++j) {
    const double dx = yu[3 * j] - xi, dy = yu[3 * j + 1] - yi, dz = yu[3 * j + 2] - zi;
    const double r2 =
        __builtin_fma(dx, dx, __builtin_fma(dy, dy, __builtin_fma(dz, dz, eps2)));
    double inv = inverse_root<kGuarded>(r2);
    if (own) inv = j == i ? 0.0 : inv;
    pe = kMass ? __builtin_fma(mu[j], inv, pe) : pe + inv;
  }
  return pe;
}

// kin[tile] and pot[tile + nt blockIdx.y]: this workgroup's sums.
template <bool kMass>
__global__ __launch_bounds__(64 * kEnergyWaves) void k_energy(const double* __restrict__ y,
                                                              int n, double eps2,
                                                              const double* __restrict__ mass,
                                                              double* __restrict__ kin,
                                                              double* __restrict__ pot) {
  __shared__ double red[kEnergyWaves];
  const uniform_ptr yu = as_uniform(y);
  const uniform_ptr mu = as_uniform(mass);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nt = gridDim.x, tile = blockIdx.x;
  const int i = 64 * tile + lane;
  const int ic = i < n ? i : n - 1;
  const double xi = y[3 * ic], yi = y[3 * ic + 1], zi = y[3 * ic + 2];
  const double mi = i < n ? (kMass ? mass[ic] : 1.0) : 0.0;
  const int units = 2 * (nt / 2 + 1);
  double pe = 0.0;
  for (int u = blockIdx.y * kEnergyWaves + wave; u < units; u += gridDim.y * kEnergyWaves) {
    const int d = u >> 1;
    const int b = tile + d < nt ? tile + d : tile + d - nt;
    const int j0 = min(n, 64 * b + (u & 1) * kEnergyUnit);
    const int j1 = min(n, j0 + kEnergyUnit);
    double part = energy_unit<kMass, false>(yu, mu, j0, j1, i, d == 0, xi, yi, zi, eps2);
    // coincident bodies without softening, or separations whose square overflows
    if (__any(part != part))
      part = energy_unit<kMass, true>(yu, mu, j0, j1, i, d == 0, xi, yi, zi, eps2);
    pe = __builtin_fma(d == 0 || 2 * d == nt ? 0.5 : 1.0, part, pe);
  }
  double e = i < n ? -(mi * pe) : 0.0;
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) e += __shfl_xor(e, s, 64);
  if (lane == 0) red[wave] = e;
  __syncthreads();
  if (threadIdx.x == 0) {
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < kEnergyWaves; ++w) sum += red[w];
    pot[tile + static_cast<size_t>(nt) * blockIdx.y] = sum;
  }
  if (blockIdx.y == 0 && wave == 1) {
    const double* v = y + 3L * n;
    const double v2 =
        v[3 * ic] * v[3 * ic] + v[3 * ic + 1] * v[3 * ic + 1] + v[3 * ic + 2] * v[3 * ic + 2];
    double ke = 0.5 * mi * v2;
    ke = i < n ? ke : 0.0;
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) ke += __shfl_xor(ke, s, 64);
    if (lane == 0) kin[tile] = ke;
  }
}

// out[0] = sum of kin (nk entries), out[1] = sum of pot (np).
__global__ __launch_bounds__(256) void k_energy_sums(const double* __restrict__ kin, long nk,
                                                     const double* __restrict__ pot, long np,
                                                     double* __restrict__ out) {
  __shared__ double red[2][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double s0 = 0.0, s1 = 0.0;
  for (long e = threadIdx.x; e < nk; e += 256) s0 += kin[e];
  for (long e = threadIdx.x; e < np; e += 256) s1 += pot[e];
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) {
    s0 += __shfl_xor(s0, s, 64);
    s1 += __shfl_xor(s1, s, 64);
  }
  if (lane == 0) {
    red[0][wave] = s0;
    red[1][wave] = s1;
  }
  __syncthreads();
  if (threadIdx.x < 2)
    out[threadIdx.x] = (red[threadIdx.x][0] + red[threadIdx.x][1]) +
                       (red[threadIdx.x][2] + red[threadIdx.x][3]);
}

// m_i v_i per component: out[c * n + i].
__global__ void k_momentum_terms(const double* __restrict__ y, int n,
                                 const double* __restrict__ mass,
                                 double* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const double mi = mass ? mass[i] : 1.0;
  const double* v = y + 3L * n;
  for (int c = 0; c < 3; ++c) out[static_cast<long>(c) * n + i] = mi * v[3 * i + c];
}

// Eight independent FMA chains per lane; lane 0 of block 0 records the
// shader-clock and 100 MHz real-time counters around the loop.
__global__ __launch_bounds__(1024) void k_probe_fp64(double* out, long long* clk,
                                                     int iters) {
  double a[8];
  for (int u = 0; u < 8; ++u) a[u] = threadIdx.x * 1e-9 + u;
  const double b = 0.999999, c = 1e-7;
  long long t0 = 0, r0 = 0;
  const bool rec = threadIdx.x == 0 && blockIdx.x == 0;
  if (rec) {
    t0 = __builtin_amdgcn_s_memtime();
    r0 = __builtin_amdgcn_s_memrealtime();
  }
  for (int i = 0; i < iters; ++i) {
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = __builtin_fma(a[u], b, c);
  }
  if (rec) {
    clk[0] = __builtin_amdgcn_s_memtime() - t0;
    clk[1] = __builtin_amdgcn_s_memrealtime() - r0;
  }
  double s = 0.0;
  for (int u = 0; u < 8; ++u) s += a[u];
  out[static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x] = s;
}

}  // namespace

hipError_t launch_probe_fp64(double* out, long long* clk, int blocks, int iters,
                             hipStream_t s) {
  hipLaunchKernelGGL(k_probe_fp64, dim3(blocks), dim3(1024), 0, s, out, clk, iters);
  return hipGetLastError();
}

hipError_t launch_momentum_terms(const double* x, int n, const double* mass,
                                 double* out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_momentum_terms, dim3((n + 255) / 256), dim3(256), 0, s,
                     x, n, mass, out);
  return hipGetLastError();
}

namespace {
// Compute units of the current device (cached per device id).
int device_cus() {
  static int cache[64] = {};
  int d = 0;
  if (hipGetDevice(&d) != hipSuccess || d < 0 || d >= 64) return 256;
  if (cache[d] <= 0) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, d) != hipSuccess ||
        v <= 0)
      v = 256;
    cache[d] = v;
  }
  return cache[d];
}
}  // namespace

namespace {
template <int R>
void launch_fast_rows(const NBodyArgs& a, bool guard, int waves, hipStream_t s) {
  auto* kern = a.mass ? (guard ? k_nbody_fast_rows<R, true, true> : k_nbody_fast_rows<R, true, false>)
                      : (guard ? k_nbody_fast_rows<R, false, true>
                               : k_nbody_fast_rows<R, false, false>);
  hipLaunchKernelGGL(kern, dim3((a.n + R - 1) / R), dim3(64 * waves), 0, s, a);
}
// R so that up to 4 bodies per CU the grid is one workgroup per CU; more waves
// than steps of 64 partners would idle.
void launch_fast_rows(const NBodyArgs& a, bool guard, hipStream_t s) {
  const int cus = device_cus(), steps = (a.n + 63) / 64;
  if (a.n <= cus) return launch_fast_rows<1>(a, guard, std::min(4, steps), s);
  if (a.n <= 2 * cus) return launch_fast_rows<2>(a, guard, std::min(4, steps), s);
  launch_fast_rows<4>(a, guard, std::min(kFastRowsWaves, steps), s);
}
}  // namespace

namespace {
template <bool kMass, bool kNext>
auto* mixed_kernel(bool guard, bool near) {
  return guard ? (near ? k_nbody_mixed<kMass, true, true, kNext>
                       : k_nbody_mixed<kMass, true, false, kNext>)
               : (near ? k_nbody_mixed<kMass, false, true, kNext>
                       : k_nbody_mixed<kMass, false, false, kNext>);
}
auto* mixed_unit_next(bool guard, bool near) {
  return guard ? (near ? k_nbody_mixed_unit_next<true, true> : k_nbody_mixed_unit_next<true, false>)
               : (near ? k_nbody_mixed_unit_next<false, true>
                       : k_nbody_mixed_unit_next<false, false>);
}
}  // namespace

// With masses, the mixed kernel's partner loop is slower beside that code; the launch
// it saves makes up for that up to one workgroup a CU with near field and half as
// many without.  A DOP853 solve of 10 steps, formed here / by a launch behind: unequal
// masses 2000 bodies 4.16 / 4.47 ms, 8192 12.19 / 12.06, 16384 23.2 / 22.6 (with near
// field 28.6 / 28.4), 65536 276 / 265 (292 / 289); equal ones 8192 11.13 / 11.14, 16384
// 21.0 / 20.7 (24.1 / 24.3), 65536 235 / 230 (261 / 261).  Without masses 16384 26.7 /
// 27.2, 65536 367 / 373.
bool nbody_rhs_forms_next(int n, int variant, float near2, bool masses) {
  if (variant != ODEHIP_NBODY_MIXED || !masses) return true;
  return (n + 63L) / 64 <= device_cus() / (near2 > 0.0f ? 1 : 2);
}

hipError_t launch_nbody_rhs(const NBodyArgs& a, int variant, hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  const unsigned blocks = static_cast<unsigned>((a.n + 63) / 64);
  const bool mass = a.mass != nullptr;
  const bool guard = !(a.eps2 >= 1e-150);
  switch (variant) {
    case ODEHIP_NBODY_EXACT: {
      launch_exact(a, device_cus(), s);
      break;
    }
    case ODEHIP_NBODY_FAST: {
      // 64-target workgroups for less than 0.7 of the CUs (MI355X: up to 11468
      // bodies; at 8192 57 us against 85, at 16384 220 against 157)
      if (10L * blocks < 7L * device_cus()) {
        launch_fast_rows(a, guard, s);
        break;
      }
      // one workgroup per CU at most: 4 waves per SIMD, prefetching partner loop
      const bool prefetch = static_cast<long>(blocks) <= device_cus();
      auto* kern = mass ? (guard ? (prefetch ? k_nbody_fast_prefetch<true, true>
                                             : k_nbody_fast<true, true>)
                                 : (prefetch ? k_nbody_fast_prefetch<true, false>
                                             : k_nbody_fast<true, false>))
                        : (guard ? (prefetch ? k_nbody_fast_prefetch<false, true>
                                             : k_nbody_fast<false, true>)
                                 : (prefetch ? k_nbody_fast_prefetch<false, false>
                                             : k_nbody_fast<false, false>));
      hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * kFastWaves), 0, s, a);
      break;
    }
    case ODEHIP_NBODY_MIXED: {
      const bool guardf = !(static_cast<float>(a.eps2) >= 1e-12f);
      const bool near = a.near2 > 0.0f;
      const dim3 g(blocks), th(64 * kMixedWaves);
      auto* kern = a.next.y ? (mass ? mixed_kernel<true, true>(guardf, near)
                                    : mixed_unit_next(guardf, near))
                            : (mass ? mixed_kernel<true, false>(guardf, near)
                                    : mixed_kernel<false, false>(guardf, near));
      hipLaunchKernelGGL(kern, g, th, 0, s, a);
      break;
    }
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Workgroups per tile of k_energy: enough of them for four per CU, each wave
// with at least one unit.
static int energy_parts(int n) {
  const long nt = (n + 63) / 64, units = 2 * (nt / 2 + 1);
  const long want = (4L * device_cus() + nt - 1) / nt;
  return static_cast<int>(std::max(1L, std::min(want, (units + kEnergyWaves - 1) / kEnergyWaves)));
}

size_t nbody_energy_scratch(int n) {
  const size_t nt = (static_cast<size_t>(n) + 63) / 64;
  return nt * (1 + energy_parts(n));
}

hipError_t launch_nbody_energy(const double* x, int n, double eps2, const double* mass,
                               double* scratch, double* out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const unsigned nt = static_cast<unsigned>((n + 63) / 64);
  const unsigned parts = static_cast<unsigned>(energy_parts(n));
  double* kin = scratch;
  double* pot = scratch + nt;
  const dim3 g(nt, parts), th(64 * kEnergyWaves);
  if (mass)
    hipLaunchKernelGGL(k_energy<true>, g, th, 0, s, x, n, eps2, mass, kin, pot);
  else
    hipLaunchKernelGGL(k_energy<false>, g, th, 0, s, x, n, eps2, mass, kin, pot);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_energy_sums, dim3(1), dim3(256), 0, s, kin, static_cast<long>(nt), pot,
                     static_cast<long>(nt) * parts, out);
  return hipGetLastError();
}

hipError_t upload_nbody_tableau(int id, const Tableau& T) {
  if (id < ODEHIP_NUM_TABLEAUS || id >= ODEHIP_MAX_TABLEAUS) return hipErrorInvalidValue;
  return hipMemcpyToSymbol(HIP_SYMBOL(n_tab), &T, sizeof(Tableau), id * sizeof(Tableau),
                           hipMemcpyHostToDevice);
}

}  // namespace odehip
