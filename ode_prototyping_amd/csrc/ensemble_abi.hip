// C ABI of the ensemble solve (declarations in odehip.h): layout and tile
// tables, the tile autotuner, and the lockstep-round driver.
//
// The driver mirrors odehip_rk_solve: initial step for every system, then K
// lockstep rounds (one attempt of each active system per round) captured in
// a HIP graph and replayed until the device-side count of running systems
// reaches zero; the host polls that count one replay behind.  Systems small
// enough for one workgroup run beside the rounds, on a stream of their own,
// each at its own pace (solo_kernels.hip).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <numeric>
#include <vector>

#include "context.hpp"
#include "ensemble.hpp"
#include "ensemble_plan.hpp"
#include "mlp.hpp"
#include "solo.hpp"

namespace odehip {

struct EnsembleWorkspace {
  char* dev = nullptr;  // device arena
  size_t cap = 0;       // bytes
  int* h_active = nullptr;  // pinned, 2 slots for the rounds, 2 for `side`
  hipEvent_t ev[2] = {nullptr, nullptr};
  // the one-workgroup solves' stream
  hipStream_t side = nullptr;
  hipEvent_t ev_side[2] = {nullptr, nullptr};
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  hipEvent_t t0 = nullptr, t1 = nullptr;
  // cached graph of K rounds and the arguments it was captured with
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  EnsBufs graph_bufs{};
  int graph_k = 0;
  // tables currently on the device
  TableKey tables;
  // autotuner cache
  std::vector<int> tuned_sizes;
  int tuned_variant = -1;
  bool tuned_mass = false;
  double tuned_eps2 = -1.0;
  double tuned_near = -1.0;
  int tuned_cfg = -1;
  double tuned_ms[ODEHIP_ENS_TILE_CONFIGS] = {};
};

void destroy_ensemble_workspace(EnsembleWorkspace* w) {
  if (!w) return;
  if (w->side) {
    (void)hipStreamSynchronize(w->side);
    (void)hipStreamDestroy(w->side);
  }
  for (auto& e : w->ev_side)
    if (e) (void)hipEventDestroy(e);
  if (w->ev_fork) (void)hipEventDestroy(w->ev_fork);
  if (w->ev_join) (void)hipEventDestroy(w->ev_join);
  if (w->exec) (void)hipGraphExecDestroy(w->exec);
  if (w->graph) (void)hipGraphDestroy(w->graph);
  if (w->dev) (void)hipFree(w->dev);
  if (w->h_active) (void)hipHostFree(w->h_active);
  for (auto& e : w->ev)
    if (e) (void)hipEventDestroy(e);
  if (w->t0) (void)hipEventDestroy(w->t0);
  if (w->t1) (void)hipEventDestroy(w->t1);
  delete w;
}

}  // namespace odehip

using namespace odehip;

namespace {

int make_layout(odehip_context* ctx, int n_systems, const int* n_particles,
                Layout* L) {
  const char* why = build_layout(n_systems, n_particles, L);
  return why ? fail(ctx, ODEHIP_ERR_INVALID, why) : ODEHIP_OK;
}

int workspace(odehip_context* ctx, size_t bytes, EnsembleWorkspace** out) {
  if (!ctx->ens) {
    auto* made = new (std::nothrow) EnsembleWorkspace();
    if (!made) return fail(ctx, ODEHIP_ERR_NOMEM, "ensemble workspace");
    // the context holds it once all of it is there
    const int rc = [&]() -> int {
      HIP_TRY(ctx, hipHostMalloc(reinterpret_cast<void**>(&made->h_active), 4 * sizeof(int)));
      HIP_TRY(ctx, hipStreamCreateWithFlags(&made->side, hipStreamNonBlocking));
      for (hipEvent_t* e : {&made->ev[0], &made->ev[1], &made->ev_side[0], &made->ev_side[1],
                            &made->ev_fork, &made->ev_join})
        HIP_TRY(ctx, hipEventCreateWithFlags(e, hipEventDisableTiming));
      HIP_TRY(ctx, hipEventCreate(&made->t0));
      HIP_TRY(ctx, hipEventCreate(&made->t1));
      return ODEHIP_OK;
    }();
    if (rc != ODEHIP_OK) {
      destroy_ensemble_workspace(made);
      return rc;
    }
    ctx->ens = made;
  }
  EnsembleWorkspace* w = ctx->ens;
  if (w->cap < bytes) {
    HIP_TRY(ctx, hipDeviceSynchronize());
    if (w->exec) (void)hipGraphExecDestroy(w->exec);
    if (w->graph) (void)hipGraphDestroy(w->graph);
    w->exec = nullptr;
    w->graph = nullptr;
    if (w->dev) HIP_TRY(ctx, hipFree(w->dev));
    w->dev = nullptr;
    w->cap = 0;
    w->tables.invalidate();
    HIP_TRY(ctx, hipMalloc(reinterpret_cast<void**>(&w->dev), bytes));
    w->cap = bytes;
  }
  *out = w;
  return ODEHIP_OK;
}

// Uploads the system/group tables and the tile list of `cfg` (skipped when
// the device already holds exactly these tables at these offsets).
int upload_tables(odehip_context* ctx, EnsembleWorkspace* w, const Plan& p,
                  const Layout& L, size_t tiles_cap, int cfg, int* n_tiles,
                  hipStream_t s) {
  const std::vector<EnsTile> tiles = make_tiles(L, kEnsTileConfigs[cfg]);
  if (const char* why = check_tiles(tiles, L, tiles_cap))
    return fail(ctx, ODEHIP_ERR_INVALID, why);
  *n_tiles = static_cast<int>(tiles.size());
  if (w->tables.matches(cfg, w->dev, p, L)) return ODEHIP_OK;
  HIP_TRY(ctx, hipStreamSynchronize(s));  // no kernel may still read them
  HIP_TRY(ctx, hipMemcpy(w->dev + p.sys, L.sys.data(), L.sys.size() * sizeof(EnsSys),
                         hipMemcpyHostToDevice));
  HIP_TRY(ctx, hipMemcpy(w->dev + p.groups, L.groups.data(),
                         L.groups.size() * sizeof(int2), hipMemcpyHostToDevice));
  HIP_TRY(ctx, hipMemcpy(w->dev + p.tiles, tiles.data(), tiles.size() * sizeof(EnsTile),
                         hipMemcpyHostToDevice));
  w->tables.set(cfg, w->dev, p, L);
  return ODEHIP_OK;
}

EnsBufs make_bufs(EnsembleWorkspace* w, const Plan& p, const Layout& L,
                  bool with_state) {
  EnsBufs b;
  std::memset(&b, 0, sizeof b);  // padding too: the graph cache compares bytes
  char* d = w->dev;
  b.sys = reinterpret_cast<const EnsSys*>(d + p.sys);
  b.groups = reinterpret_cast<const int2*>(d + p.groups);
  b.tiles = reinterpret_cast<const EnsTile*>(d + p.tiles);
  b.n_active = reinterpret_cast<int*>(d + p.n_active);
  if (with_state) {
    b.st = reinterpret_cast<SolverState*>(d + p.st);
    b.xb0 = reinterpret_cast<double*>(d + p.xb0);
    b.xb1 = reinterpret_cast<double*>(d + p.xb1);
    b.ks = reinterpret_cast<double*>(d + p.ks);
    b.ytmp = reinterpret_cast<double*>(d + p.ytmp);
    b.kfsal = reinterpret_cast<double*>(d + p.kfsal);
    b.ytmp2 = reinterpret_cast<double*>(d + p.sc0);
    b.sc0 = reinterpret_cast<double*>(d + p.sc0);
    b.partA = reinterpret_cast<double*>(d + p.partA);
    b.partB = reinterpret_cast<double*>(d + p.partB);
  }
  b.nv = L.nv;
  b.n_sys = static_cast<int>(L.sys.size());
  b.n_groups = L.n_groups;
  return b;
}

// `solve`: of a solve, or timed for one.
void set_tile_cfg(EnsBufs* b, int cfg, int n_tiles, const Layout& L, bool solve) {
  b->fine = solve ? n_tiles <= kEnsFineTiles
                  : plain_fine(n_tiles, tail_shape(L, nullptr).longest, kEnsTileConfigs[cfg].split);
  b->wpb = kEnsTileConfigs[cfg].wpb;
  b->tpl2_min_n = kEnsTileConfigs[cfg].tpl2_min_n;
  b->split = kEnsTileConfigs[cfg].split;
  b->n_tiles = n_tiles;
}

// Waits for a stream when a call that put work on it returns early, so that the next
// call may set up the same buffers.
struct DrainOnReturn {
  hipStream_t stream = nullptr;  // null: nothing to wait for
  ~DrainOnReturn() {
    if (stream) (void)hipStreamSynchronize(stream);
  }
};

bool tune_cache_hit(const EnsembleWorkspace* w, const Layout& L, int variant,
                    bool mass, double eps2, double near_c) {
  return w->tuned_cfg >= 0 && w->tuned_variant == variant && w->tuned_mass == mass &&
         std::memcmp(&w->tuned_eps2, &eps2, sizeof eps2) == 0 &&
         std::memcmp(&w->tuned_near, &near_c, sizeof near_c) == 0 && w->tuned_sizes == L.sizes;
}

// Times one right-hand side of the state `y` into `k` for every candidate
// configuration (one warm-up, best of two).  Among the candidates within 3 %
// of the fastest it keeps the one with the most target tiles (then the
// fastest of those): on the full ensemble 128-target tiles often tie with
// 64-target ones, but they halve the waves once compaction leaves a few
// large systems running.
int autotune(odehip_context* ctx, EnsembleWorkspace* w, const Plan& p,
             const Layout& L, size_t tiles_cap, EnsBufs b, const double* y,
             double* k, hipStream_t s) {
  double best = 1e300;
  int best_cfg = kEnsDefaultTileConfig;
  for (int c = 0; c < ODEHIP_ENS_TILE_CONFIGS; ++c) {
    int n_tiles = 0;
    int rc = upload_tables(ctx, w, p, L, tiles_cap, c, &n_tiles, s);
    if (rc) return rc;
    set_tile_cfg(&b, c, n_tiles, L, true);
    HIP_TRY(ctx, ens_launch_rhs(b, y, k, 0, s));
    double ms_best = 1e300;
    for (int r = 0; r < 2; ++r) {
      HIP_TRY(ctx, hipEventRecord(w->t0, s));
      HIP_TRY(ctx, ens_launch_rhs(b, y, k, 0, s));
      HIP_TRY(ctx, hipEventRecord(w->t1, s));
      HIP_TRY(ctx, hipEventSynchronize(w->t1));
      float ms = 0.0f;
      HIP_TRY(ctx, hipEventElapsedTime(&ms, w->t0, w->t1));
      ms_best = std::min(ms_best, static_cast<double>(ms));
    }
    w->tuned_ms[c] = ms_best;
    if (ms_best < best) {
      best = ms_best;
      best_cfg = c;
    }
  }
  long most = -1;
  for (int c = 0; c < ODEHIP_ENS_TILE_CONFIGS; ++c) {
    if (!(w->tuned_ms[c] <= 1.03 * best)) continue;
    const long t = real_tiles(L, kEnsTileConfigs[c]);
    if (t > most || (t == most && w->tuned_ms[c] < w->tuned_ms[best_cfg])) {
      most = t;
      best_cfg = c;
    }
  }
  w->tuned_cfg = best_cfg;
  return ODEHIP_OK;
}

int check_common(odehip_context* ctx, int nbody_variant, double softening,
                 int tile_config) {
  if (nbody_variant < 0 || nbody_variant > 2)
    return fail(ctx, ODEHIP_ERR_INVALID, "bad nbody_variant");
  if (!(softening >= 0.0)) return fail(ctx, ODEHIP_ERR_INVALID, "bad softening");
  if (tile_config < ODEHIP_ENS_TILE_AUTO || tile_config >= ODEHIP_ENS_TILE_CONFIGS)
    return fail(ctx, ODEHIP_ERR_INVALID, "bad tile_config");
  return ODEHIP_OK;
}

}  // namespace

extern "C" {

int odehip_ensemble_rhs(odehip_context* ctx, int n_systems,
                        const int* n_particles, int nbody_variant,
                        double softening, const double* masses,
                        int tile_config, const double* x, double* dxdt,
                        double* ms_out) {
  ODEHIP_USE_DEVICE(ctx);
  if (!ctx) return ODEHIP_ERR_INVALID;
  if (!x || !dxdt) return fail(ctx, ODEHIP_ERR_INVALID, "null argument");
  int rc = check_common(ctx, nbody_variant, softening, tile_config);
  if (rc) return rc;
  Layout L;
  if ((rc = make_layout(ctx, n_systems, n_particles, &L))) return rc;
  const size_t tcap = tiles_capacity(L);
  const Plan p = plan(L, tcap, 0, 0, false);
  EnsembleWorkspace* w = nullptr;
  if ((rc = workspace(ctx, p.total, &w))) return rc;
  const double eps2 = softening * softening;
  const double near_c = nbody_variant == ODEHIP_NBODY_MIXED ? ctx->near_c : 0.0;
  int cfg = tile_config;
  if (cfg == ODEHIP_ENS_TILE_AUTO)
    cfg = tune_cache_hit(w, L, nbody_variant, masses != nullptr, eps2, near_c)
              ? w->tuned_cfg
              : kEnsDefaultTileConfig;
  hipStream_t s = begin_work(ctx);
  int n_tiles = 0;
  if ((rc = upload_tables(ctx, w, p, L, tcap, cfg, &n_tiles, s))) return rc;
  EnsBufs b = make_bufs(w, p, L, false);
  b.mass = masses;
  b.variant = nbody_variant;
  b.eps2 = eps2;
  b.near_c = near_c;
  set_tile_cfg(&b, cfg, n_tiles, L, false);
  HIP_TRY(ctx, hipEventRecord(w->t0, s));
  HIP_TRY(ctx, ens_launch_rhs(b, x, dxdt, 0, s));
  HIP_TRY(ctx, hipEventRecord(w->t1, s));
  if (ms_out) {
    HIP_TRY(ctx, hipEventSynchronize(w->t1));
    float ms = 0.0f;
    HIP_TRY(ctx, hipEventElapsedTime(&ms, w->t0, w->t1));
    *ms_out = ms;
  }
  end_work(ctx);
  return ODEHIP_OK;
}

int odehip_ensemble_solve(odehip_context* ctx, int tableau, int n_systems,
                          const int* n_particles, int nbody_variant,
                          double softening, const double* masses,
                          const odehip_ensemble_options* opt,
                          const double* x0, double* x_out,
                          odehip_ensemble_stats* stats,
                          odehip_system_stats* per_system) {
  ODEHIP_USE_DEVICE(ctx);
  if (!ctx) return ODEHIP_ERR_INVALID;
  if (!opt || !x0 || !x_out) return fail(ctx, ODEHIP_ERR_INVALID, "null argument");
  if (const int trc = use_tableau(ctx, tableau)) return trc;
  int rc = check_common(ctx, nbody_variant, softening, opt->tile_config);
  if (rc) return rc;
  if (opt->max_accepted < 0 || opt->max_attempts < 0 || opt->trace_cap < 0)
    return fail(ctx, ODEHIP_ERR_INVALID, "negative budget or capacity");
  if (opt->controller < ODEHIP_CONTROLLER_REFERENCE ||
      opt->controller > ODEHIP_CONTROLLER_LEARNED)
    return fail(ctx, ODEHIP_ERR_INVALID, "bad controller");
  if (opt->controller == ODEHIP_CONTROLLER_LEARNED && !opt->mlp)
    return fail(ctx, ODEHIP_ERR_INVALID, "the learned controller needs a network (mlp)");
  if (opt->controller == ODEHIP_CONTROLLER_LEARNED && mlp_device(opt->mlp) != ctx->device)
    return fail(ctx, ODEHIP_ERR_INVALID, "the network lives on another device");
  const long n_dense = opt->n_dense;
  if (n_dense < 0) return fail(ctx, ODEHIP_ERR_INVALID, "negative n_dense");
  if (n_dense > 0) {
    if (tableau != ODEHIP_TABLEAU_DOPRI5 && tableau != ODEHIP_TABLEAU_DOP853)
      return fail(ctx, ODEHIP_ERR_INVALID, "ensemble dense output needs DOPRI5 or DOP853");
    if (!opt->dense_times || !opt->dense_states)
      return fail(ctx, ODEHIP_ERR_INVALID, "dense_times / dense_states null");
    double prev = opt->t0;
    for (long r = 0; r < n_dense; ++r) {
      const double tr = opt->dense_times[r];
      if (!std::isfinite(tr) || !(tr > prev))
        return fail(ctx, ODEHIP_ERR_INVALID,
                    "dense_times must be finite and strictly increasing after t0");
      prev = tr;
    }
  }
  Layout L;
  if ((rc = make_layout(ctx, n_systems, n_particles, &L))) return rc;
  const int S = host_tableau(tableau).S;
  const long trace_cap = opt->trace ? opt->trace_cap : 0;
  const size_t tcap = tiles_capacity(L);
  const Plan p = plan(L, tcap, S, trace_cap, true, n_dense);
  EnsembleWorkspace* w = nullptr;
  // (after the plan's regions: the list of one-workgroup systems)
  if ((rc = workspace(ctx, p.total + L.sys.size() * sizeof(int), &w))) return rc;
  const double eps2 = softening * softening;
  const double near_c = nbody_variant == ODEHIP_NBODY_MIXED ? ctx->near_c : 0.0;
  hipStream_t s = begin_work(ctx);

  EnsBufs b = make_bufs(w, p, L, true);
  b.trace = trace_cap > 0 ? reinterpret_cast<double*>(w->dev + p.trace) : nullptr;
  b.trace_cap = trace_cap;
  b.mass = masses;
  b.atol = opt->atol;
  b.rtol = opt->rtol;
  b.tableau = tableau;
  b.variant = nbody_variant;
  b.eps2 = eps2;
  b.near_c = near_c;
  b.controller = opt->controller;
  b.mlp = opt->controller == ODEHIP_CONTROLLER_LEARNED ? mlp_infer_ptr(opt->mlp) : nullptr;
  if (n_dense > 0) {
    b.dense_t = reinterpret_cast<const double*>(w->dev + p.dense_t);
    b.dense_out = reinterpret_cast<double*>(w->dev + p.dense_out);
    b.n_dense = n_dense;
    HIP_TRY(ctx, hipMemcpyAsync(w->dev + p.dense_t, opt->dense_times, n_dense * sizeof(double),
                                hipMemcpyHostToDevice, s));
    HIP_TRY(ctx, launch_fill(b.dense_out, NAN, static_cast<size_t>(n_dense) * L.nv, s));
  }

  // tile configuration
  int cfg = opt->tile_config;
  if (cfg == ODEHIP_ENS_TILE_AUTO) {
    if (!tune_cache_hit(w, L, nbody_variant, masses != nullptr, eps2, near_c)) {
      std::fill(w->tuned_ms, w->tuned_ms + ODEHIP_ENS_TILE_CONFIGS, 0.0);
      EnsBufs tb = b;
      tb.st = nullptr;  // plain evaluations of x0 into the k1 slot
      if ((rc = autotune(ctx, w, p, L, tcap, tb, x0, b.ks, s))) return rc;
      w->tuned_variant = nbody_variant;
      w->tuned_mass = masses != nullptr;
      w->tuned_eps2 = eps2;
      w->tuned_near = near_c;
      w->tuned_sizes = L.sizes;
    }
    cfg = w->tuned_cfg;
  }
  const bool tuned = tune_cache_hit(w, L, nbody_variant, masses != nullptr, eps2, near_c);
  if (opt->tune_ms) {
    for (int c = 0; c < ODEHIP_ENS_TILE_CONFIGS; ++c)
      opt->tune_ms[c] = tuned ? w->tuned_ms[c] : 0.0;
  }
  // Small systems are solved by one workgroup each (solo.hpp) unless the caller
  // names a tile configuration; dense output is written by the rounds only.
  const bool exact = nbody_variant == ODEHIP_NBODY_EXACT;
  std::vector<int> solo;
  std::vector<char> live(L.sys.size(), 1);
  int solo_max = 0;
  if (opt->tile_config == ODEHIP_ENS_TILE_AUTO && n_dense == 0) {
    b.solo_n = solo_limit(S, nbody_variant, b.mlp != nullptr);
    for (size_t k = 0; k < L.sys.size(); ++k) {
      if (L.sys[k].n > b.solo_n) continue;
      solo.push_back(static_cast<int>(k));
      live[k] = 0;
      solo_max = std::max(solo_max, L.sys[k].n);
    }
    // the longest evaluations first
    std::stable_sort(solo.begin(), solo.end(),
                     [&](int p, int q) { return L.sys[p].n > L.sys[q].n; });
  }
  b.n_solo = static_cast<int>(solo.size());
  const int n_rounds = n_systems - b.n_solo;

  // a tile's partners are shared by several waves from the start when the
  // ensemble's tiles would leave SIMDs idle
  int run_cfg = tail_config(L, nullptr, cfg, exact);
  int n_tiles = 0;
  if ((rc = upload_tables(ctx, w, p, L, tcap, run_cfg, &n_tiles, s))) return rc;
  set_tile_cfg(&b, run_cfg, n_tiles, L, true);

  HIP_TRY(ctx, ens_enqueue_init(b, x0, opt->t0, opt->tf, opt->max_accepted,
                                opt->max_attempts, opt->fsal ? 1 : 0, opt->controller, s));
  HIP_TRY(ctx, ens_enqueue_initial_step(b, s));

  // The one-workgroup solves: launches of kSoloTicks, two ahead of the host,
  // until their count of running systems has been seen at zero.
  SoloArgs sa{};
  long solo_pushed = 0, solo_seen = 0;
  bool solo_done = solo.empty();
  DrainOnReturn drain;
  auto push_solo = [&]() -> int {
    const int at = static_cast<int>(solo_pushed & 1);
    HIP_TRY(ctx, launch_solo(sa, solo_max, nbody_variant, static_cast<unsigned>(solo.size()),
                             w->side));
    HIP_TRY(ctx, hipMemcpyAsync(&w->h_active[2 + at], b.n_active + 1, sizeof(int),
                                hipMemcpyDeviceToHost, w->side));
    HIP_TRY(ctx, hipEventRecord(w->ev_side[at], w->side));
    ++solo_pushed;
    return ODEHIP_OK;
  };
  // Takes in finished launches (waiting for the oldest one if `wait`) and keeps
  // two in flight.
  auto poll_solo = [&](bool wait) -> int {
    while (!solo_done) {
      if (solo_pushed - solo_seen < 2) {
        if (const int prc = push_solo()) return prc;
        continue;
      }
      const int at = static_cast<int>(solo_seen & 1);
      const hipError_t q = wait ? hipEventSynchronize(w->ev_side[at])
                                : hipEventQuery(w->ev_side[at]);
      if (q == hipErrorNotReady) return ODEHIP_OK;
      if (q != hipSuccess) return hip_fail(ctx, q, "one-workgroup solves");
      ++solo_seen;
      solo_done = w->h_active[2 + at] == 0;
    }
    return ODEHIP_OK;
  };
  if (!solo.empty()) {
    HIP_TRY(ctx, hipStreamSynchronize(s));  // earlier launches read the list's region
    HIP_TRY(ctx, hipMemcpy(w->dev + p.total, solo.data(), solo.size() * sizeof(int),
                           hipMemcpyHostToDevice));
    sa.sys = b.sys;
    sa.list = reinterpret_cast<const int*>(w->dev + p.total);
    sa.st = b.st;
    sa.xb0 = b.xb0;
    sa.xb1 = b.xb1;
    sa.ks = b.ks;
    sa.kfsal = b.kfsal;
    sa.mass = b.mass;
    sa.atol = b.atol;
    sa.rtol = b.rtol;
    sa.trace = b.trace;
    sa.trace_cap = b.trace_cap;
    sa.mlp = static_cast<const MlpInfer*>(b.mlp);
    sa.n_active = b.n_active + 1;
    sa.eps2 = b.eps2;
    sa.near_c = b.near_c;
    sa.tableau = tableau;
    HIP_TRY(ctx, hipEventRecord(w->ev_fork, s));
    HIP_TRY(ctx, hipStreamWaitEvent(w->side, w->ev_fork, 0));
    drain.stream = w->side;
    if ((rc = poll_solo(false))) return rc;
  }

  // Rounds run on lists of the running systems' workgroups: every system at
  // first, rebuilt (and the graph re-captured) each time the number of
  // running systems has fallen to 7/8 of the last list's, so the long tail of
  // a few slow systems does not launch workgroups for all the finished ones
  // (on 2048 systems 3/4 measured 1-1.5 % faster than 1/2, and 7/8 another
  // 0-1 %; same results), but where launches bound a round (kEnsListWork pairs or
  // less), no sooner than kEnsListRounds rounds after the last time: new lists gain
  // little there, and their graph costs as much as a dozen rounds.  (64 systems of 64
  // bodies in rounds, DOPRI5 fast 5.5 -> 4.2 ms; 128 of up to 1024, DOP853 exact 44.9 ->
  // 33.9; with 1e8 pairs 141 of up to 233, DOP853 exact, take 108 ms instead of 105,
  // with 1e7 the second example stays at 44.)
  constexpr long kEnsListRounds = 64;
  constexpr double kEnsListWork = 3.0e7;
  auto rounds_per_replay = [&](double sum_n2) {
    int k = opt->rounds_per_launch;
    if (k <= 0) {
      const double work = static_cast<double>(S) * sum_n2;
      k = work > 1.0e10 ? 2 : (work > 1.0e9 ? 4 : 8);  // (a recapture costs by its launches)
    }
    return k;
  };
  auto capture = [&](const EnsBufs& rb, int k) -> int {
    if (w->exec && w->graph_k == k && std::memcmp(&w->graph_bufs, &rb, sizeof rb) == 0)
      return ODEHIP_OK;
    // a replay of the cached graph may still run (e.g. after a failed call)
    HIP_TRY(ctx, hipStreamSynchronize(s));
    if (w->exec) (void)hipGraphExecDestroy(w->exec);
    if (w->graph) (void)hipGraphDestroy(w->graph);
    w->exec = nullptr;
    w->graph = nullptr;
    HIP_TRY(ctx, hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    hipError_t ce = hipSuccess;
    for (int r = 0; r < k && ce == hipSuccess; ++r) ce = ens_enqueue_round(rb, s);
    hipGraph_t g = nullptr;
    hipError_t ee = hipStreamEndCapture(s, &g);
    if (ce != hipSuccess || ee != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      return ce != hipSuccess ? hip_fail(ctx, ce, "capture round")
                              : hip_fail(ctx, ee, "hipStreamEndCapture");
    }
    w->graph = g;
    HIP_TRY(ctx, hipGraphInstantiate(&w->exec, g, nullptr, nullptr, 0));
    w->graph_bufs = rb;
    w->graph_k = k;
    return ODEHIP_OK;
  };
  EnsBufs rb = b;  // run_cfg: the tile shape of the running systems
  int K = 0, n_live = n_rounds;
  double work = S * L.work;  // of a round of the present lists
  // Lists and graph for the systems `live` marks (the stream is idle).
  auto set_running = [&]() -> int {
    std::vector<int2> act;
    double sum_n2 = 0.0;
    for (size_t k = 0; k < L.sys.size(); ++k) {
      if (!live[k]) continue;
      sum_n2 += static_cast<double>(L.sys[k].n) * L.sys[k].n;
      for (int g = 0; g < L.sys[k].n_groups; ++g) act.push_back(L.groups[L.sys[k].gbase + g]);
    }
    // once the running systems' tiles no longer give every SIMD four
    // waves: 64-target tiles, then partners shared by several waves per
    // tile; same results
    run_cfg = tail_config(L, &live, run_cfg, exact);
    const std::vector<EnsTile> tiles = make_tiles(L, kEnsTileConfigs[run_cfg], &live);
    if (const char* why = check_tiles(tiles, L, tcap)) return fail(ctx, ODEHIP_ERR_INVALID, why);
    HIP_TRY(ctx, hipMemcpy(w->dev + p.groups_act, act.data(), act.size() * sizeof(int2),
                           hipMemcpyHostToDevice));
    HIP_TRY(ctx, hipMemcpy(w->dev + p.tiles, tiles.data(), tiles.size() * sizeof(EnsTile),
                           hipMemcpyHostToDevice));
    w->tables.invalidate();  // the tile region now holds the running systems' tiles
    rb.groups = reinterpret_cast<const int2*>(w->dev + p.groups_act);
    rb.n_groups = static_cast<int>(act.size());
    set_tile_cfg(&rb, run_cfg, static_cast<int>(tiles.size()), L, true);
    K = rounds_per_replay(sum_n2);
    work = S * sum_n2;
    return capture(rb, K);
  };
  if (n_rounds == n_systems) {
    K = rounds_per_replay(L.work);
    if ((rc = capture(rb, K))) return rc;
  } else if (n_rounds > 0) {
    HIP_TRY(ctx, hipStreamSynchronize(s));
    if ((rc = set_running())) return rc;
  }

  const long cap_rounds = opt->max_attempts > 0 ? opt->max_attempts : (1L << 40);
  long launched = 0;
  int slot = 0;
  bool have_prev = false;
  int compact_below = n_rounds * 7 / 8;
  auto next_lists = [&] { return launched + (work > kEnsListWork ? 0 : kEnsListRounds); };
  long compact_from = next_lists();
  int seen = n_rounds;  // systems running at the last look
  std::vector<SolverState> hst;
  while (n_rounds > 0) {
    HIP_TRY(ctx, hipGraphLaunch(w->exec, s));
    launched += K;
    HIP_TRY(ctx, hipMemcpyAsync(&w->h_active[slot], b.n_active, sizeof(int),
                                hipMemcpyDeviceToHost, s));
    HIP_TRY(ctx, hipEventRecord(w->ev[slot], s));
    if ((rc = poll_solo(false))) return rc;
    if (launched >= cap_rounds + 2L * K) break;
    if (have_prev) {
      HIP_TRY(ctx, hipEventSynchronize(w->ev[slot ^ 1]));
      const int running = w->h_active[slot ^ 1];
      if (running == 0) break;
      if (running <= compact_below && launched < compact_from && running < seen) {
        // systems are ending: whether the last has is seen before another replay is
        // launched, whose empty rounds would cost more than the wait
        HIP_TRY(ctx, hipEventSynchronize(w->ev[slot]));
        if (w->h_active[slot] == 0) break;
      }
      seen = running;
      if (running <= compact_below && launched >= compact_from) {
        HIP_TRY(ctx, hipStreamSynchronize(s));
        hst.resize(L.sys.size());
        HIP_TRY(ctx, hipMemcpy(hst.data(), b.st, hst.size() * sizeof(SolverState),
                               hipMemcpyDeviceToHost));
        n_live = 0;
        for (size_t k = 0; k < L.sys.size(); ++k) {
          live[k] = live[k] && !hst[k].done;
          n_live += live[k];
        }
        if (n_live == 0) break;
        if ((rc = set_running())) return rc;
        compact_below = n_live * 7 / 8;
        compact_from = next_lists();
        have_prev = false;
        slot = 0;
        continue;
      }
    }
    have_prev = true;
    slot ^= 1;
  }
  if (!solo.empty()) {
    if ((rc = poll_solo(true))) return rc;
    HIP_TRY(ctx, hipEventRecord(w->ev_join, w->side));
    HIP_TRY(ctx, hipStreamWaitEvent(s, w->ev_join, 0));
    drain.stream = nullptr;  // `s` goes on behind it
  }
  HIP_TRY(ctx, ens_enqueue_copy_out(b, x_out, s));
  std::vector<SolverState> hs(L.sys.size());
  HIP_TRY(ctx, hipMemcpyAsync(hs.data(), b.st, hs.size() * sizeof(SolverState),
                              hipMemcpyDeviceToHost, s));
  HIP_TRY(ctx, hipStreamSynchronize(s));
  if (opt->trace && trace_cap > 0)
    HIP_TRY(ctx, hipMemcpy(opt->trace, b.trace,
                           hs.size() * static_cast<size_t>(trace_cap) * 3 * sizeof(double),
                           hipMemcpyDeviceToHost));
  if (n_dense > 0)
    HIP_TRY(ctx, hipMemcpy(opt->dense_states, b.dense_out,
                           static_cast<size_t>(n_dense) * L.nv * sizeof(double),
                           hipMemcpyDeviceToHost));
  end_work(ctx);
  odehip_ensemble_stats agg{};
  agg.tile_config = cfg;
  agg.interactions = L.interactions;
  agg.rhs_ms = tuned ? w->tuned_ms[cfg] : 0.0;
  for (size_t k = 0; k < hs.size(); ++k) {
    const SolverState& h = hs[k];
    agg.rounds = std::max(agg.rounds, h.attempts);
    agg.accepted += h.accepted;
    agg.rejected += h.rejected;
    agg.attempts += h.attempts;
    agg.rhs_evals += h.rhs_evals;
    agg.learned_steps += h.learned_steps;
    agg.particle_steps += static_cast<double>(L.sys[k].n) * h.accepted;
    if (h.status == ODEHIP_STATUS_RUNNING) agg.n_unfinished += 1;
    if (per_system) {
      odehip_system_stats& o = per_system[k];
      o.accepted = h.accepted;
      o.rejected = h.rejected;
      o.attempts = h.attempts;
      o.rhs_evals = h.rhs_evals;
      o.n_trace = std::min(h.attempts, trace_cap);
      o.learned_steps = h.learned_steps;
      o.status = h.status;
      o.pad = 0;
      o.t = h.t;
      o.dt = h.dt;
      o.dt_initial = h.dt_initial;
      o.last_err = h.err;
      o.n_dense = n_dense > 0 ? h.dense_next : 0;
    }
  }
  if (stats) *stats = agg;
  if (agg.n_unfinished)
    return fail(ctx, ODEHIP_ERR_INVALID, "ensemble did not finish within the attempt cap");
  return ODEHIP_OK;
}

}  // extern "C"
