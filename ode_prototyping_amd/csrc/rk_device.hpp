// Device-side arithmetic of the embedded Runge-Kutta method shared by the
// single-system kernels (rk_kernels.hip) and the ensemble kernels
// (ensemble_kernels.hip): per-element stage / update formulas, the canonical
// group reduction, and the accept/reject + step-size controller.  Both solve
// paths call these same functions, so an ensemble member is computed with
// exactly the arithmetic of a single-system solve.
#pragma once

#include <cmath>

#include "crpow.hpp"
#include "internal.hpp"

namespace odehip {

__device__ inline double max_abs(double a, double b) {
  // std::max(std::abs(x), std::abs(x0)): the first argument unless it is
  // less than the second.
  const double fa = std::fabs(a), fb = std::fabs(b);
  return (fa < fb) ? fb : fa;
}

// Canonical group reduction (odehip.h, ODEHIP_REDUCE_GROUP): 256 threads; each
// 64-lane quad reduced with halving xor strides (lane 0 holds
// v0 + v32, + (v16 + v48), ...), then (q0 + q1) + (q2 + q3).
__device__ inline double group_reduce(double v) {
  __shared__ double q[4];
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) v = v + __shfl_xor(v, s, 64);
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  if (lane == 0) q[wave] = v;
  __syncthreads();
  return (q[0] + q[1]) + (q[2] + q[3]);
}

// Sequential fold of group partials from 0.0 (the last level of the
// canonical order).
__device__ inline double fold_partials(const double* p, int n_groups) {
  double r = 0.0;
  for (int g = 0; g < n_groups; ++g) r = r + p[g];
  return r;
}

// The same fold, called by every thread of a block: the partials are first
// staged through LDS (coalesced), kFoldLds at a time, then thread 0 adds them in
// order from LDS.  Returns the sum in thread 0.
// kCoherent: of partials that other workgroups of this launch have written
// (last_group).
constexpr int kFoldLds = 512;
template <bool kCoherent = false>
__device__ inline double fold_partials_block(const double* p, int n_groups) {
  __shared__ double buf[kFoldLds];
  double r = 0.0;
  for (int g0 = 0; g0 < n_groups; g0 += kFoldLds) {
    const int cnt = min(kFoldLds, n_groups - g0);
    if (g0 > 0) __syncthreads();
    for (int g = threadIdx.x; g < cnt; g += blockDim.x)
      buf[g] = kCoherent ? __hip_atomic_load(p + g0 + g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                         : p[g0 + g];
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll 8
      for (int g = 0; g < cnt; ++g) r = r + buf[g];
    }
  }
  return r;
}

// detail::rk_stage_kernel (RKEmbeddedParallel.hpp:91-101): element i of
// x0 + dt * sum_{j<stage} a[stage-1][j] k_j, stage vectors n_var apart.
__device__ inline double stage_value(const Tableau& T, int stage, double dt,
                                     const double* ks, const double* x0,
                                     size_t i, size_t n_var) {
  double tmp = 0.0;
  for (int j = 0; j < stage; ++j) tmp += T.a[stage - 1][j] * ks[j * n_var + i];
  return x0[i] + tmp * dt;
}

// The same for element e of the next stage by the launch that writes its last
// stage vector (NextStage), whose element is k: the sum in the same order, L
// loads per round trip (a load per step of the sum would wait for each in turn).
// All of them for kernels whose launch is a chain of latencies; few for those
// that fill the chip, whose occupancy the loads' registers would take.
constexpr int kStageLoads = kMaxStages - 1;
constexpr int kStageLoadsLean = 2;
template <int L>
__device__ inline void next_stage(const NextStage& N, const Tableau& T, size_t n_var, size_t e,
                                  double k, double x0, double dt) {
  double tmp = 0.0;
  for (int j0 = 0; j0 < N.n; j0 += L) {
    double v[L];
#pragma unroll
    for (int u = 0; u < L; ++u)
      v[u] = N.ks[static_cast<size_t>(j0 + u < N.n ? j0 + u : j0) * n_var + e];
#pragma unroll
    for (int u = 0; u < L; ++u)
      if (j0 + u < N.n) tmp += T.a[N.n][j0 + u] * v[u];
  }
  tmp += T.a[N.n][N.n] * k;
  N.y[e] = x0 + tmp * dt;
}

// detail::update_state_and_error_kernel (RKEmbeddedParallel.hpp:103-123).
__device__ inline void update_values(const Tableau& T, double dt,
                                     const double* ks, const double* x0,
                                     size_t i, size_t n_var, double& x,
                                     double& err) {
  double xs = 0.0, es = 0.0;
  for (int j = 0; j < T.S; ++j) {
    const double kj = ks[j * n_var + i];
    xs += T.b[j] * kj;
    es += T.db[j] * kj;
  }
  x = x0[i] + xs * dt;
  err = es * dt;
}

// Called by every thread of a workgroup of an attempt's final pass, `partial` (its
// group's sum, in thread 0) going to *slot: true in the last of the n_groups
// workgroups, which then may fold every partial (fold_partials_block<true>) and
// change the solve's state.  The partials alone pass between workgroups here, so
// they are written and read past the XCDs' L2s, each store complete before its
// group is counted; a fence would write the whole L2 back, which 1000 groups made
// 50 us of.
__device__ inline bool last_group(SolverState* st, int n_groups, double* slot, double partial) {
  __shared__ int last;
  if (threadIdx.x == 0) {
    __hip_atomic_store(slot, partial, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last = __hip_atomic_fetch_add(&st->arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           n_groups - 1;
    if (last) st->arrived = 0;
  }
  __syncthreads();
  return last != 0;
}

// ---------------------------------------------------------- controller ----

// Solver scalars before the first attempt (RKEmbeddedParallel.hpp:13-33).
__device__ inline void ctrl_init(SolverState* st, const Tableau& T, double t0,
                                 double tf, long max_acc, long max_att,
                                 int fsal, int tab, int n_groups,
                                 long times_cap, long trace_cap,
                                 int controller) {
  const int q = T.p < T.pt ? T.p : T.pt;
  st->t = t0;
  st->t0 = t0;
  st->tf = tf;
  st->dt = 0.0;
  st->err = 0.0;
  st->dt_initial = 0.0;
  st->inv_q1 = 1.0 / (1.0 + q);
  st->root_k = 1 + q;
  st->safety = cr_root(0.38, st->inv_q1, st->root_k);
  st->dt0 = 0.0;
  st->d1 = 0.0;
  st->err_prev = 1.0e-4;
  for (int h = 0; h < 3; ++h) {
    st->hist_err[h] = 0.0;
    st->hist_dt[h] = 0.0;
    st->hist_acc[h] = 0.0;
  }
  st->accepted = 0;
  st->rejected = 0;
  st->attempts = 0;
  st->rhs_evals = 0;
  st->max_accepted = max_acc;
  st->max_attempts = max_att;
  st->times_cap = times_cap;
  st->trace_cap = trace_cap;
  st->learned_steps = 0;
  st->dt_acc = 0.0;
  st->dense_next = 0;
  st->dense_lo = 0;
  st->dense_hi = 0;
  st->dense_seen = 0;
  st->dense_steps = 0;
  st->dense_rhs_evals = 0;
  st->dense_go = 0;
  st->arrived = 0;
  st->cur = 0;
  st->fsal = fsal;
  st->tableau = tab;
  st->n_groups = n_groups;
  st->k1_valid = 0;
  st->controller = controller;
  st->rejects_in_row = 0;
  st->just_accepted = 0;
  st->status = ODEHIP_STATUS_RUNNING;
  st->done = (t0 < tf) ? 0 : 1;
  if (st->done) st->status = ODEHIP_STATUS_REACHED_END;
}

// First half of an attempt's end (RKEmbeddedParallel.hpp:56-63): the scaled
// error norm from the sum of squares, counters, trace, accept/reject, the
// time update and the x0 = x swap.  Returns false when the solve stops on a
// non-finite error norm (nothing else to do for this attempt).
__device__ inline bool ctrl_judge(SolverState* st, const Tableau& T,
                                  double sum, size_t n_var, double* times,
                                  double* trace, bool* accepted_out) {
  const double scaled_error =
      std::sqrt(sum / static_cast<double>(static_cast<long>(n_var)));
  const long attempt = st->attempts;
  st->attempts = attempt + 1;
  st->rhs_evals += st->k1_valid ? (T.S - 1) : T.S;
  st->err = scaled_error;
  const double dt = st->dt;
  const bool finite = std::isfinite(scaled_error);
  const bool accept = finite && scaled_error <= 1.0;
  *accepted_out = accept;
  st->just_accepted = accept ? 1 : 0;
  if (trace && attempt < st->trace_cap) {
    trace[3 * attempt] = scaled_error;
    trace[3 * attempt + 1] = dt;
    trace[3 * attempt + 2] = accept ? 1.0 : 0.0;
  }
  // attempt history, most recent first (controller features)
  for (int h = 2; h > 0; --h) {
    st->hist_err[h] = st->hist_err[h - 1];
    st->hist_dt[h] = st->hist_dt[h - 1];
    st->hist_acc[h] = st->hist_acc[h - 1];
  }
  st->hist_err[0] = scaled_error;
  st->hist_dt[0] = dt;
  st->hist_acc[0] = accept ? 1.0 : 0.0;
  if (!finite) {
    st->rejected += 1;
    st->status = ODEHIP_STATUS_NONFINITE;
    st->done = 1;
    return false;
  }
  if (accept) {
    st->t = st->t + dt;
    st->dt_acc = dt;
    st->cur ^= 1;  // x0 = x (the ping-pong buffers swap roles)
    const long acc = st->accepted + 1;
    st->accepted = acc;
    if (times && acc < st->times_cap) times[acc] = st->t;
    st->k1_valid = (st->fsal && T.fsal) ? 1 : 0;
    st->rejects_in_row = 0;
  } else {
    st->rejected += 1;
    st->k1_valid = st->fsal ? 2 : 0;
    st->rejects_in_row += 1;
  }
  return true;
}

// Step-size proposal of the PI controller (Gustafsson's PI.3.4; Hairer &
// Wanner, Solving ODEs II, IV.2): dt * (0.38/err)^(0.3/k) *
// (err_prev/err)^(0.4/k), k = 1 + q -- the reference controller's steady
// error 0.38 --, err_prev the error of the last accepted step (1e-4 before
// the first one, floored at 1e-4), no growth right after a rejection.
// The two powers, `which` = 0, 1: a wave's first two lanes take one each.
__device__ inline double pi_power(const SolverState* st, double err, int which) {
  const double k_inv = st->inv_q1;
  return cr_pow((which ? st->err_prev : 0.38) / err, (which ? 0.4 : 0.3) * k_inv);
}
__device__ inline double pi_proposal(const SolverState* st, double power0, double power1,
                                     bool accept) {
  double fac = power0 * power1;
  if (!accept && fac > 1.0) fac = 1.0;
  return st->dt * fac;
}

// Whether a judged attempt's step comes from the PI controller: always its own,
// the learned one's before three attempts of history exist, after two rejections
// in a row or when its ratio is not finite.
__device__ inline bool pi_steps(const SolverState* st, double learned_ratio) {
  if (st->controller == ODEHIP_CONTROLLER_PI) return true;
  return st->controller == ODEHIP_CONTROLLER_LEARNED &&
         !(std::isfinite(learned_ratio) && st->attempts >= 3 && st->rejects_in_row < 2);
}

// Second half (RKEmbeddedParallel.hpp:64-79): the new step size, its clamps
// and the clip to tf, then the termination tests.  `learned_ratio` is the
// learned controller's proposed dt_new / dt (ODEHIP_CONTROLLER_LEARNED only,
// capped at 1 right after a rejection); `power0` and `power1` (pi_power) are
// read where pi_steps says so.
__device__ inline void ctrl_step(SolverState* st, bool accept, double learned_ratio,
                                 double power0, double power1) {
  const double scaled_error = st->err;
  double dt = st->dt;
  const double t = st->t;
  double dtnew;
  if (pi_steps(st, learned_ratio)) {
    dtnew = pi_proposal(st, power0, power1, accept);
  } else if (st->controller == ODEHIP_CONTROLLER_LEARNED) {
    // no growth right after a rejection
    dtnew = dt * ((!accept && learned_ratio > 1.0) ? 1.0 : learned_ratio);
    st->learned_steps += 1;
  } else {
    dtnew = dt * st->safety / cr_root(scaled_error, st->inv_q1, st->root_k);
  }
  if (accept) st->err_prev = scaled_error < 1.0e-4 ? 1.0e-4 : scaled_error;
  const double max_step_scale = 6.0;
  const double min_step_scale = 0.33;
  const double tf = st->tf, t0 = st->t0;
  if (std::fabs(dtnew) > max_step_scale * std::fabs(dt)) {
    dt *= max_step_scale;
  } else if (std::fabs(dtnew) < min_step_scale * std::fabs(dt)) {
    dt *= min_step_scale;
  } else if (dtnew / (tf - t0) < 1.0e-12) {
    dt = (tf - t0) * 1.0e-12;
  } else {
    dt = dtnew;
  }
  if (t + dt > tf) dt = tf - t;
  st->dt = dt;
  if (!(t < tf)) {
    st->status = ODEHIP_STATUS_REACHED_END;
    st->done = 1;
  } else if (accept && st->max_accepted > 0 && st->accepted >= st->max_accepted) {
    st->status = ODEHIP_STATUS_MAX_ACCEPTED;
    st->done = 1;
  } else if (st->max_attempts > 0 && st->attempts >= st->max_attempts) {
    st->status = ODEHIP_STATUS_MAX_ATTEMPTS;
    st->done = 1;
  }
}

// Orders a wave's own LDS writes before its later reads.
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The step of a judged attempt by one wave (every lane calls; `judged` and
// `learned_ratio` are lane 0's).  `st`, in LDS, is this wave's alone to change.
__device__ inline void ctrl_step_wave(SolverState* st, bool judged, bool accept,
                                      double learned_ratio) {
  const int lane = threadIdx.x & 63;
  double power = 1.0;
  wave_lds_fence();
  if (__any(lane == 0 && judged && pi_steps(st, learned_ratio)) && lane < 2)
    power = pi_power(st, st->err, lane);
  const double power1 = __shfl(power, 1, 64);
  if (lane == 0 && judged) ctrl_step(st, accept, learned_ratio, power, power1);
}

// A whole attempt end with the reference or PI controller, by one wave (`sum` is
// read in lane 0).
__device__ inline void ctrl_attempt(SolverState* st, const Tableau& T,
                                    double sum, size_t n_var, double* times,
                                    double* trace) {
  bool accept = false, judged = false;
  if ((threadIdx.x & 63) == 0) judged = ctrl_judge(st, T, sum, n_var, times, trace, &accept);
  ctrl_step_wave(st, judged, accept, NAN);
}

// ------------------------------------------------------- dense output ----

// DenseOutput::save's test (NumericalRecipes/Output.hpp:109) after an
// attempt: if it was accepted and ended strictly after the next output
// time(s), rows [dense_lo, dense_hi) are this step's and dense_go is set.
// extra_rhs: RHS evaluations the pass costs (counted; with DOP853 f at the
// step's end also becomes the next k1 when k1 reuse is on).
__device__ inline void dense_gate(SolverState* st, const double* times, long n_dense,
                                  int extra_rhs) {
  int go = 0;
  if (st->just_accepted && st->accepted != st->dense_seen) {
    st->dense_seen = st->accepted;
    const long lo = st->dense_next;
    long hi = lo;
    const double t = st->t;
    while (hi < n_dense && t > times[hi]) ++hi;
    if (hi > lo) {
      go = 1;
      st->dense_lo = lo;
      st->dense_hi = hi;
      st->dense_next = hi;
      st->dense_steps += 1;
      st->dense_rhs_evals += extra_rhs;
      if (extra_rhs && st->fsal) st->k1_valid = 1;
    }
  }
  st->dense_go = go;
}

// By one thread of the final pass of an attempt enqueued behind a solve's last one,
// whose own dense pass has run: the passes from here on find the gate shut (left
// open, each of them would evaluate and write the last step's rows again).
__device__ inline void dense_over(SolverState* st) { st->dense_go = 0; }

// DOP853's stage vector j of a dense pass: 0..11 the accepted attempt's
// stages (nv apart in ks), 12 = f at the step's end (k13), 13..15 the extra
// stages, kept in the slots of stages 1..3, which the extension never reads.
__device__ inline const double* dop853_dense_vec(const double* ks, const double* k13, int j,
                                                 size_t nv) {
  if (j < 12) return ks + static_cast<size_t>(j) * nv;
  if (j == 12) return k13;
  return ks + static_cast<size_t>(j - 12) * nv;
}

// Element e of the input of extra stage 13 + x (StepperDopr853.hpp:239-262):
// y + h (w_0 k_{i0} + ... + w_7 k_{i7}), the sum left to right.
__device__ inline double dop853_dense_stage(const Dop853Dense& D, int x, const double* ks,
                                            const double* k13, size_t nv, size_t e,
                                            const double* y, double h) {
  double acc = D.extra_w[x][0] * dop853_dense_vec(ks, k13, D.extra_idx[x][0], nv)[e];
  for (int m = 1; m < 8; ++m)
    acc = acc + D.extra_w[x][m] * dop853_dense_vec(ks, k13, D.extra_idx[x][m], nv)[e];
  return y[e] + h * acc;
}

// StepperDopr853::prepare_dense / dense_out (StepperDopr853.hpp:214-237,
// 263-289) for element e: the eight polynomial coefficients from 14 stage
// vectors, then out[row * row_stride + e] for the pass's rows.
__device__ inline void dop853_dense_rows(const Dop853Dense& D, const SolverState* st,
                                         const double* ks, const double* k13, size_t nv,
                                         size_t e, const double* y, const double* yout,
                                         const double* times, double* out,
                                         size_t row_stride) {
  const double h = st->dt_acc;
  const double yi = y[e];
  const double ydiff = yout[e] - yi;
  const double bspl = h * ks[e] - ydiff;
  const double rc3 = ydiff - h * k13[e] - bspl;
  double rc[4];
  for (int r = 0; r < 4; ++r) {
    double acc = D.d_w[r][0] * dop853_dense_vec(ks, k13, D.d_idx[0], nv)[e];
    for (int m = 1; m < 12; ++m)
      acc = acc + D.d_w[r][m] * dop853_dense_vec(ks, k13, D.d_idx[m], nv)[e];
    rc[r] = h * acc;
  }
  const double t_end = st->t;
  const long hi = st->dense_hi;
  for (long row = st->dense_lo; row < hi; ++row) {
    const double s = (times[row] - (t_end - h)) / h;
    const double s1 = 1.0 - s;
    out[static_cast<size_t>(row) * row_stride + e] =
        yi + s * (ydiff + s1 * (bspl + s * (rc3 + s1 * (rc[0] + s * (rc[1] + s1 * (rc[2] + s * rc[3]))))));
  }
}

// StepperDopr5::prepare_dense / dense_out (StepperDopr5.hpp:195-221) for
// element e of a state whose stage vectors are nv apart in ks (stage 7 = f at
// the new state): the step went from y to yout over st->dt_acc ending at
// st->t; writes out[row * row_stride + e] for the pass's rows.
__device__ inline void dopri5_dense_rows(const Dopri5Dense& D, const SolverState* st,
                                         const double* ks, size_t nv, size_t e,
                                         const double* y, const double* yout,
                                         const double* times, double* out,
                                         size_t row_stride) {
  const double h = st->dt_acc;
  const double yi = y[e];
  const double ydiff = yout[e] - yi;
  const double bspl = h * ks[e] - ydiff;
  const double rc3 = ydiff - h * ks[6 * nv + e] - bspl;
  double acc = D.d[0] * ks[static_cast<size_t>(D.idx[0]) * nv + e];
  for (int m = 1; m < 6; ++m) acc = acc + D.d[m] * ks[static_cast<size_t>(D.idx[m]) * nv + e];
  const double rc4 = h * acc;
  const double t_end = st->t;
  const long hi = st->dense_hi;
  for (long row = st->dense_lo; row < hi; ++row) {
    const double s = (times[row] - (t_end - h)) / h;
    const double s1 = 1.0 - s;
    out[static_cast<size_t>(row) * row_stride + e] =
        yi + s * (ydiff + s1 * (bspl + s * (rc3 + s1 * rc4)));
  }
}

// estimate_initial_step (RKEmbeddedParallel.hpp:183-185): d0, d1, dt0 from
// the sums of squares of x0/sc and f0/sc.
__device__ inline void ctrl_init_step_a(SolverState* st, double sa, double sb,
                                        size_t n_var) {
  const double nv = static_cast<double>(static_cast<long>(n_var));
  const double d0 = std::sqrt(sa / nv);
  const double d1 = std::sqrt(sb / nv);
  const double dt0 = (d0 < 1.0e-5 or d1 < 1.0e-5) ? 1.0e-6 : 0.01 * (d0 / d1);
  st->dt0 = dt0;
  st->d1 = d1;
}

// (:193-199): d2, dt1, the initial step, from the sum of squares of
// (f1 - f0)/sc.
__device__ inline void ctrl_init_step_b(SolverState* st, const Tableau& T,
                                        double sa, size_t n_var) {
  const double nv = static_cast<double>(static_cast<long>(n_var));
  const double dt0 = st->dt0;
  const double d1 = st->d1;
  const double d2 = std::sqrt(sa / nv) / dt0;
  const int p = T.p;
  const double m = (d1 < d2) ? d2 : d1;
  const double hi = 1.0e-6, lo = dt0 * 1.0e-3;
  const double dt1 = (m <= 1.0e-15) ? ((hi < lo) ? lo : hi)
                                    : cr_root(0.01 / m, 1.0 / (1.0 + p), 1 + p);
  const double cap = 100.0 * dt0;
  const double dt = (dt1 < cap) ? dt1 : cap;
  st->dt = dt;
  st->dt_initial = dt;
  st->rhs_evals += 2;
}

}  // namespace odehip
