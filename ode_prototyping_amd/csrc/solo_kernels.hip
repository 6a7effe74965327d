// Whole solves of small N-body systems, one workgroup per system: stages,
// right-hand sides, error norm and controller of attempt after attempt in one
// launch, the state and the stage vectors in LDS.
//
// A small system's attempt is a chain of short steps.  Spread over launches,
// every one of them costs the 2.4 ... 3 us a kernel takes from its start to the
// next one's (a 64-body DOPRI5 attempt: 16 launches, 50 us), and in an ensemble
// every system waits for the slowest of each round; here a step ends with a
// workgroup barrier, and every system goes its own pace.  What bounds an attempt
// is that chain: barriers, LDS reads and the dependent arithmetic of one
// wave's partners, not throughput (a CU holds one or two such workgroups).
//
// Every number is computed by the functions and in the order of the kernels that
// run the same solve by launches -- for a solve of its own those of rk_kernels.hip and
// nbody_kernels.hip, for an ensemble's system the lockstep ones of
// ensemble_kernels.hip, whose fast sums have another order --, so which form runs a
// solve changes no bit of its result (tests/test_gpu_solve_forms.py,
// tests/test_gpu_solo.py).  A workgroup starts no attempt once kSoloTicks have passed
// and keeps what the next launch needs in the state's global buffers: launches
// of bounded time, whose systems need not wait for one another's attempts.
#include <type_traits>

#include "ens_chunks.hpp"
#include "mlp.hpp"
#include "rk_device.hpp"
#include "solo.hpp"

namespace odehip {
namespace {

__constant__ Tableau s_tab[ODEHIP_MAX_TABLEAUS] = {
    kTableaus[0], kTableaus[1], kTableaus[2],
    kTableaus[3], kTableaus[4], kTableaus[5]};

#define ODEHIP_LDS __attribute__((address_space(3)))
typedef ODEHIP_LDS double* lds_ptr;
typedef const ODEHIP_LDS double* lds_cptr;

extern __shared__ __attribute__((aligned(16))) double solo_lds[];

// f(std::integral_constant<int, J>) for J = count in [Lo, Hi]: sums over the
// stages unrolled, so that their loads go out together.
template <int Lo, int Hi, typename F>
__device__ __forceinline__ void with_count(int count, F&& f) {
  if constexpr (Lo <= Hi) {
    if (count == Lo)
      f(std::integral_constant<int, Lo>{});
    else
      with_count<Lo + 1, Hi>(count, f);
  }
}

// exact: the terms of blocks of kSoloTerms partners per wave go to LDS, waves
// 0, 1, 2 add the block's x, y, z terms in partner order.  A target's own index
// and the partners past the end contribute +0, which leaves a sum that starts at
// +0 unchanged.
template <bool kMass, bool kShared>
__device__ __forceinline__ void solo_exact(lds_cptr in, lds_cptr mass, lds_ptr kout, lds_ptr term,
                                           int n, double eps2, int wave, int waves, int lane) {
  const int B = waves * kSoloTerms;
  for (int i0 = 0; i0 < n; i0 += 64) {
    const int i = i0 + lane, ic = i < n ? i : n - 1;
    const double xi = in[3 * ic], yi = in[3 * ic + 1], zi = in[3 * ic + 2];
    double acc = 0.0;
    for (int jb = 0; jb < n; jb += B) {
      const int j0 = jb + wave * kSoloTerms;
      if (j0 < n) {
#pragma unroll
        for (int p = 0; p < kSoloTerms; ++p) {
          const int j = j0 + p, jc = j < n ? j : n - 1;
          double tx, ty, tz;
          exact_term<kMass, kShared>(in[3 * jc] - xi, in[3 * jc + 1] - yi, in[3 * jc + 2] - zi,
                                     kMass ? mass[jc] : 1.0, eps2, tx, ty, tz);
          const bool out = j >= n || j == i;
          lds_ptr t = term + (wave * kSoloTerms + p) * 64 + lane;
          t[0] = out ? 0.0 : tx;
          t[B * 64] = out ? 0.0 : ty;
          t[2 * B * 64] = out ? 0.0 : tz;
        }
      }
      __syncthreads();
      if (wave < 3) {
        // whole groups of kSoloTerms partners (a group's slots past n hold +0)
        const int cnt = min(B, (n - jb + kSoloTerms - 1) / kSoloTerms * kSoloTerms);
        lds_cptr t = term + wave * B * 64 + lane;
        int q = 0;
        if (cnt >= 16) {  // the next 16 terms come in while 16 are added
          double v[2][16];
#pragma unroll
          for (int u = 0; u < 16; ++u) v[0][u] = t[u * 64];
          for (; q + 32 <= cnt; q += 16) {
#pragma unroll
            for (int u = 0; u < 16; ++u) v[1][u] = t[(q + 16 + u) * 64];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 16; ++u) acc += v[0][u];
#pragma unroll
            for (int u = 0; u < 16; ++u) v[0][u] = v[1][u];
          }
#pragma unroll
          for (int u = 0; u < 16; ++u) acc += v[0][u];
          q += 16;
        }
        for (; q < cnt; q += kSoloTerms) {
#pragma unroll
          for (int u = 0; u < kSoloTerms; ++u) acc += t[(q + u) * 64];
        }
      }
      __syncthreads();
    }
    if (wave < 3 && i < n) kout[3 * n + 3 * i + wave] = acc;
  }
}

// fast, mixed: one wave per (64 targets, group of partners); thread (tile,
// coordinate, target) adds the groups' sums in order, chunk by chunk.  The
// near field adds FP64 terms into the chunk's sum between its groups, so there
// a chunk is one wave's.
template <int kVariant, bool kMass, bool kGuard, bool kNear>
__device__ __forceinline__ void solo_groups(lds_cptr in, lds_cptr mass, lds_ptr kout,
                                            lds_ptr part, int n, double eps2, float near2,
                                            double scale, int wave, int waves, int lane) {
  constexpr int U = kNear ? kEnsChunk : kEnsGroup;
  constexpr int kPerChunk = kEnsChunk / U;
  const int tiles = (n + 63) / 64, units = tiles * ((n + U - 1) / U);
  const int q = threadIdx.x, ft = q / 192, fc = q % 192;
  double acc = 0.0, chunk = 0.0;
  int g = 0;
  for (int r = 0; r < units; r += waves) {
    const int u = r + wave;
    if (u < units) {
      const int t = u % tiles, j0 = u / tiles * U, j1 = min(n, j0 + U);
      const int i = 64 * t + lane;
      const int ic[1] = {i < n ? i : n - 1};
      const double xi[1] = {in[3 * ic[0]]}, yi[1] = {in[3 * ic[0] + 1]},
                   zi[1] = {in[3 * ic[0] + 2]};
      double px[1] = {0.0}, py[1] = {0.0}, pz[1] = {0.0};
      if constexpr (!kNear)
        lds_group<kVariant, kMass, kGuard, kMass || kGuard ? 4 : 8>(in + 3 * j0, mass + j0, j0, j1 - j0, ic[0], xi[0],
                                           yi[0], zi[0], eps2, px[0], py[0], pz[0]);
      else
        mixed_chunk<kMass, kGuard, kNear, 1>(in, mass, j0, j1, ic, xi, yi, zi, eps2, near2, px,
                                             py, pz);
      lds_ptr o = part + wave * 192 + lane;
      o[0] = px[0];
      o[64] = py[0];
      o[128] = pz[0];
    }
    __syncthreads();
    if (ft < tiles) {
      int w = ft - r % tiles;
      if (w < 0) w += tiles;
      for (; w < waves && r + w < units; w += tiles) {
        chunk += part[w * 192 + fc];
        if (++g % kPerChunk == 0) {
          acc += chunk;
          chunk = 0.0;
        }
      }
    }
    if (r + waves < units) __syncthreads();  // part is written again
  }
  if (g % kPerChunk != 0) acc += chunk;
  const int i = 64 * ft + fc % 64;
  if (ft < tiles && i < n) kout[3 * n + 3 * i + fc / 64] = acc * scale;
}

// fast, one system: the order of k_nbody_fast_rows (nbody_kernels.hip), which
// evaluates such systems wherever attempts are launched (dense output, kept states,
// attempts_per_launch), so that a solve's bits do not depend on these.  Up to four
// sets of 64 partners each has a wave of its own there, a lane per partner, which
// folds lanes l with l + 32, then + 16, 8, 4, 2 and 1: the sum of the lanes
// l = c mod B is, level by level, the same whoever computes it.  Lanes past the last
// partner add +0 there, which changes at most the sign of a zero, and the fold over
// the sets starts at +0; so they are left out here where that is a whole level.
static_assert(kSoloOneFastN <= 2 * 64, "a share of 8 or 16 lanes per wave");

// Lanes c, c + 8, ... of a set, the first kLive of them, j the first one's partner.
// (Unclamped loads in sets that are whole spill, and take 10 % longer.)
template <bool kMass, bool kGuard, int kLive>
__device__ __forceinline__ void row_lanes(lds_cptr in, lds_cptr mass, int j, int n, int i,
                                          double xi, double yi, double zi, double eps2,
                                          double (&s)[3]) {
  double c[3 * kLive], m[kLive], dx[kLive], dy[kLive], dz[kLive], w[kLive];
#pragma unroll
  for (int u = 0; u < kLive; ++u) {
    const int q = min(j + 8 * u, n - 1);
    c[3 * u] = in[3 * q];
    c[3 * u + 1] = in[3 * q + 1];
    c[3 * u + 2] = in[3 * q + 2];
    m[u] = kMass ? mass[q] : 1.0;
  }
  fast_weights<kMass, kLive>(c, m, xi, yi, zi, eps2, dx, dy, dz, w);
#pragma unroll
  for (int u = 0; u < kLive; ++u) {
    const bool out = (j + 8 * u >= n) | (kGuard & (j + 8 * u == i));
    w[u] = out ? 0.0 : w[u];
    dx[u] = __builtin_fma(dx[u], w[u], 0.0);  // (a lane's sum starts at +0)
    dy[u] = __builtin_fma(dy[u], w[u], 0.0);
    dz[u] = __builtin_fma(dz[u], w[u], 0.0);
  }
#pragma unroll
  for (int h = kLive / 2; h >= 1; h /= 2) {
#pragma unroll
    for (int u = 0; u < h; ++u) {
      dx[u] += dx[u + h];
      dy[u] += dy[u + h];
      dz[u] += dz[u + h];
    }
  }
  s[0] = dx[0];
  s[1] = dy[0];
  s[2] = dz[0];
}

// kTiles tiles of 64 targets and sets of 64 partners (n / 64, rounded up), one wave for
// the lanes l = c mod P of a set and a tile: eight waves and P = 8 at up to 64
// bodies, sixteen and P = 4 at up to 128.  Thread (tile, coordinate, target) folds the
// shares of a set, then adds the sets.
template <bool kMass, bool kGuard, int kTiles>
__device__ __forceinline__ void solo_rows(lds_cptr in, lds_cptr mass, lds_ptr kout, lds_ptr part,
                                          int n, double eps2, int wave, int lane) {
  static_assert(kTiles == 1 || kTiles == 2, "shares of 8 or 16 lanes");
  constexpr int P = kTiles == 1 ? 8 : 4;
  {
    const int i = min(64 * (wave / P % kTiles) + lane, n - 1);
    const int j = 64 * (wave / P / kTiles) + wave % P;
    const double xi = in[3 * i], yi = in[3 * i + 1], zi = in[3 * i + 2];
    double s[3], t[3];
    if constexpr (kTiles == 1) {
      if (n > 32)
        row_lanes<kMass, kGuard, 8>(in, mass, j, n, i, xi, yi, zi, eps2, s);
      else if (n > 16)
        row_lanes<kMass, kGuard, 4>(in, mass, j, n, i, xi, yi, zi, eps2, s);
      else
        row_lanes<kMass, kGuard, 2>(in, mass, j, n, i, xi, yi, zi, eps2, s);
    } else {
#pragma unroll 1  // (the loads of both halves together would spill)
      for (int h = 0; h < 2; ++h) {
        row_lanes<kMass, kGuard, 8>(in, mass, j + 4 * h, n, i, xi, yi, zi, eps2, s);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          if (h == 0)
            t[k] = s[k];
          else
            s[k] += t[k];
        }
      }
    }
    lds_ptr o = part + wave * 192 + lane;
#pragma unroll
    for (int k = 0; k < 3; ++k) o[64 * k] = s[k];
  }
  __syncthreads();
  const int ft = threadIdx.x / 192, fc = threadIdx.x % 192, i = 64 * ft + fc % 64;
  if (ft >= kTiles || i >= n) return;
  double acc = 0.0;
#pragma unroll
  for (int set = 0; set < kTiles; ++set) {
    double v[P];
#pragma unroll
    for (int c = 0; c < P; ++c) v[c] = part[(P * (kTiles * set + ft) + c) * 192 + fc];
#pragma unroll
    for (int h = P / 2; h >= 1; h /= 2)
#pragma unroll
      for (int c = 0; c < h; ++c) v[c] += v[c + h];
    acc += v[0];
  }
  kout[3 * n + 3 * i + fc / 64] = acc;
}

// Sum over the workgroup's elements of 64-element quads and groups in the
// canonical order (rk_device.hpp): quad[] holds the quads' sums.
__device__ __forceinline__ double solo_fold(lds_cptr quad, int n_groups) {
  double r = 0.0;
  for (int g = 0; g < n_groups; ++g)
    r = r + ((quad[4 * g] + quad[4 * g + 1]) + (quad[4 * g + 2] + quad[4 * g + 3]));
  return r;
}

// kRows: fast, one system (solo_rows); an ensemble's systems have the lockstep
// kernels' order (solo_groups).
template <int kVariant, bool kMass, bool kSpecial, bool kNear, bool kRows>
__global__ __launch_bounds__(64 * kSoloWaves) void k_solo(SoloArgs a) {
  __shared__ SolverState st;
  __shared__ double quad_[kSoloMaxQuads];
  __shared__ int wide[kMaxStages];  // exact: a coordinate of the stage fails coord_shared_ok
  __shared__ MlpRowLds mlp_lds;
  __shared__ int stop;  // no further attempt in this launch
  lds_ptr quad = (lds_ptr)quad_;
  const int slot = a.list ? a.list[blockIdx.x] : 0;
  SolverState* gst = a.st + slot;
  if (gst->done) return;
  const EnsSys sy = a.sys ? a.sys[slot] : a.one;
  const int n = sy.n, nv = 6 * n, threads = blockDim.x, tid = threadIdx.x;
  if (n < 1 || solo_lds_doubles(n, s_tab[a.tableau].S, kVariant, threads / 64, a.mlp) > a.lds_doubles)
    return;  // does not fit what the launch set aside (uniform)
  const int lane = tid & 63, waves = threads >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Tableau& T = s_tab[a.tableau];
  const int S = T.S;
  lds_ptr x0 = (lds_ptr)solo_lds, y = x0 + nv, ks = y + nv, mass = ks + S * nv,
          work = mass + ((n + 1) & ~1);
  for (int e = tid; e < static_cast<int>(sizeof(SolverState) / 8); e += threads)
    reinterpret_cast<uint64_t*>(&st)[e] = reinterpret_cast<const uint64_t*>(gst)[e];
  __syncthreads();
  {
    const double* g = (st.cur ? a.xb1 : a.xb0) + sy.eoff;
    for (int e = tid; e < nv; e += threads) x0[e] = g[e];
    if (st.k1_valid) {
      const double* k1 = (st.k1_valid == 1 ? a.kfsal : a.ks) + sy.eoff;
      lds_ptr to = st.k1_valid == 1 ? ks + (S - 1) * nv : ks;
      for (int e = tid; e < nv; e += threads) to[e] = k1[e];
    }
  }
  double m_uni = 0.0;
  if (kMass) {
    const double* m = a.mass + sy.eoff / 6;
    for (int e = tid; e < n; e += threads) mass[e] = m[e];
    if (kVariant != ODEHIP_NBODY_EXACT && !kRows) m_uni = st.mass_uniform;
  }
  const bool per_term = kMass && m_uni == 0.0;
  const double scale = per_term || !kMass ? 1.0 : m_uni;
  const float near2 = kNear ? mixed_near2(a.near_c, n) : 0.0f;
  double* trace = a.trace ? a.trace + static_cast<size_t>(slot) * a.trace_cap * 3 : nullptr;
  const int n_quads = 4 * sy.n_groups;
  // the network beside the system, for the same reason
  const bool learned = st.controller == ODEHIP_CONTROLLER_LEARNED;
  const MlpInfer* net = (const MlpInfer*)(work + waves * solo_sums(kVariant));
  if (learned) {
    uint64_t* to = (uint64_t*)net;
    for (int e = tid; e < static_cast<int>(sizeof(MlpInfer) / 8); e += threads)
      to[e] = reinterpret_cast<const uint64_t*>(a.mlp)[e];
  }

  const uint64_t start = __builtin_amdgcn_s_memrealtime();
  for (;;) {
    const double dt = st.dt;
    const int k1_valid = st.k1_valid;
    if (kVariant == ODEHIP_NBODY_EXACT && kSpecial) {
      // (read last before the final pass's barrier of the attempt before)
      if (tid < kMaxStages) wide[tid] = 0;
      __syncthreads();
    }
    for (int stage = 0; stage < S; ++stage) {
      lds_cptr in = stage == 0 ? x0 : y;
      lds_ptr kout = ks + stage * nv;
      bool ok = true;
      if (stage == 0) {
        if (k1_valid == 1)
          for (int e = tid; e < nv; e += threads) ks[e] = ks[(S - 1) * nv + e];
        if (k1_valid) continue;
        if (kVariant == ODEHIP_NBODY_EXACT && kSpecial)
          for (int e = tid; e < 3 * n; e += threads) ok = ok & coord_shared_ok(x0[e]);
      } else {
        with_count<1, kMaxStages - 1>(stage, [&](auto J) {
          const double* row = T.a[J - 1];
          for (int e = tid; e < nv; e += threads) {
            double k[J], tmp = 0.0;  // stage_value (rk_device.hpp)
#pragma unroll
            for (int j = 0; j < J; ++j) k[j] = ks[j * nv + e];
#pragma unroll
            for (int j = 0; j < J; ++j) tmp += row[j] * k[j];
            const double v = x0[e] + tmp * dt;
            y[e] = v;
            if (kVariant == ODEHIP_NBODY_EXACT && kSpecial)
              ok = ok & ((e >= 3 * n) | coord_shared_ok(v));
          }
        });
      }
      if (kVariant == ODEHIP_NBODY_EXACT && kSpecial && !__all(ok) && lane == 0) wide[stage] = 1;
      __syncthreads();
      const bool shared = kVariant == ODEHIP_NBODY_EXACT && kSpecial && wide[stage] == 0;
      for (int e = tid; e < 3 * n; e += threads) kout[e] = in[3 * n + e];
      if constexpr (kVariant == ODEHIP_NBODY_EXACT) {
        if (shared)
          solo_exact<kMass, true>(in, mass, kout, work, n, a.eps2, wave, waves, lane);
        else
          solo_exact<kMass, false>(in, mass, kout, work, n, a.eps2, wave, waves, lane);
      } else if constexpr (kRows) {
        if (n <= 64)
          solo_rows<kMass, kSpecial, 1>(in, mass, kout, work, n, a.eps2, wave, lane);
        else
          solo_rows<kMass, kSpecial, 2>(in, mass, kout, work, n, a.eps2, wave, lane);
      } else {
        if (kMass && per_term)
          solo_groups<kVariant, true, kSpecial, kNear>(in, mass, kout, work, n, a.eps2, near2,
                                                       1.0, wave, waves, lane);
        else
          solo_groups<kVariant, false, kSpecial, kNear>(in, mass, kout, work, n, a.eps2, near2,
                                                        scale, wave, waves, lane);
      }
      __syncthreads();
    }
    // new state, embedded error, scaled squared error by quads (k_ens_final);
    // whole waves, so that a quad is one wave's pass
    with_count<2, kMaxStages>(S, [&](auto J) {
    for (int e0 = 64 * wave; e0 < 64 * n_quads; e0 += threads) {
      const int e = e0 + lane;
      double term = 0.0;
      if (e < nv) {
        double k[J], xs = 0.0, es = 0.0;
#pragma unroll
        for (int j = 0; j < J; ++j) k[j] = ks[j * nv + e];
#pragma unroll
        for (int j = 0; j < J; ++j) {
          xs += T.b[j] * k[j];
          es += T.db[j] * k[j];
        }
        const double xo = x0[e];
        const double xv = xo + xs * dt, ev = es * dt;
        y[e] = xv;
        const double at = a.atol_v ? a.atol_v[e] : a.atol, rt = a.rtol_v ? a.rtol_v[e] : a.rtol;
        const double sc = at + rt * max_abs(xv, xo);
        const double scaled = ev / sc;
        term = scaled * scaled;
      }
#pragma unroll
      for (int s = 32; s >= 1; s >>= 1) term = term + __shfl_xor(term, s, 64);
      if (lane == 0) quad[e0 / 64] = term;
    }
    });
    __syncthreads();
    if (wave == 0) {
      const double sum = lane == 0 ? solo_fold(quad, sy.n_groups) : 0.0;
      if (learned)
        ctrl_attempt_wave(&st, T, sum, nv, a.times, trace, net, n, &mlp_lds);
      else
        ctrl_attempt(&st, T, sum, nv, a.times, trace);
      if (lane == 0) stop = st.done || __builtin_amdgcn_s_memrealtime() - start >= kSoloTicks;
    }
    __syncthreads();
    if (st.just_accepted)
      for (int e = tid; e < nv; e += threads) x0[e] = y[e];
    if (stop) break;
  }
  // the next launch's (or the caller's) state
  double* g = (st.cur ? a.xb1 : a.xb0) + sy.eoff;
  for (int e = tid; e < nv; e += threads) g[e] = x0[e];
  if (st.k1_valid && !st.done) {
    double* k1 = (st.k1_valid == 1 ? a.kfsal : a.ks) + sy.eoff;
    lds_cptr from = st.k1_valid == 1 ? ks + (S - 1) * nv : ks;
    for (int e = tid; e < nv; e += threads) k1[e] = from[e];
  }
  __syncthreads();  // (st is read above)
  for (int e = tid; e < static_cast<int>(sizeof(SolverState) / 8); e += threads)
    reinterpret_cast<uint64_t*>(gst)[e] = reinterpret_cast<const uint64_t*>(&st)[e];
  if (tid == 0 && st.done && a.n_active) atomicSub(a.n_active, 1);
}

template <int kVariant, bool kNear, bool kRows = false>
void* solo_kernel(bool mass, bool special) {
  return mass ? (special ? (void*)k_solo<kVariant, true, true, kNear, kRows>
                         : (void*)k_solo<kVariant, true, false, kNear, kRows>)
              : (special ? (void*)k_solo<kVariant, false, true, kNear, kRows>
                         : (void*)k_solo<kVariant, false, false, kNear, kRows>);
}

}  // namespace

hipError_t launch_solo(const SoloArgs& args, int n_max, int variant, unsigned blocks,
                       hipStream_t s) {
  SoloArgs a = args;
  const int S = host_tableau(a.tableau).S;
  const bool rows = variant == ODEHIP_NBODY_FAST && !a.sys;
  int waves = solo_waves(n_max, S, variant, a.mlp);
  if (rows) waves = n_max > kSoloOneFastN ? 0 : n_max > 64 ? kSoloWaves : 8;
  if (waves == 0 || (variant == ODEHIP_NBODY_MIXED && !a.sys)) return hipErrorInvalidValue;
  if (blocks == 0) return hipSuccess;
  a.lds_doubles = solo_lds_doubles(n_max, S, variant, waves, a.mlp);
  if (a.lds_doubles > kSoloLdsDoubles) return hipErrorInvalidValue;
  void* k = nullptr;
  if (variant == ODEHIP_NBODY_EXACT)
    k = solo_kernel<ODEHIP_NBODY_EXACT, false>(a.mass, a.eps2 >= 0x1p-200 && a.eps2 <= 0x1p100);
  else if (rows)
    k = solo_kernel<ODEHIP_NBODY_FAST, false, true>(a.mass, !(a.eps2 >= 1e-150));
  else if (variant == ODEHIP_NBODY_FAST)
    k = solo_kernel<ODEHIP_NBODY_FAST, false>(a.mass, !(a.eps2 >= 1e-150));
  else if (a.near_c > 0.0)
    k = solo_kernel<ODEHIP_NBODY_MIXED, true>(a.mass, !(static_cast<float>(a.eps2) >= 1e-12f));
  else
    k = solo_kernel<ODEHIP_NBODY_MIXED, false>(a.mass, !(static_cast<float>(a.eps2) >= 1e-12f));
  const size_t bytes = static_cast<size_t>(a.lds_doubles) * sizeof(double);
  hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     static_cast<int>(bytes));
  if (e != hipSuccess) return e;
  void* p[] = {&a};
  return hipLaunchKernel(k, dim3(blocks), dim3(64 * waves), p, bytes, s);
}

hipError_t upload_solo_tableau(int id, const Tableau& T) {
  if (id < ODEHIP_NUM_TABLEAUS || id >= ODEHIP_MAX_TABLEAUS) return hipErrorInvalidValue;
  return hipMemcpyToSymbol(HIP_SYMBOL(s_tab), &T, sizeof(Tableau), id * sizeof(Tableau),
                           hipMemcpyHostToDevice);
}

}  // namespace odehip
