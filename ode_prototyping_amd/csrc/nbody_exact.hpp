// The bit-exact right-hand side of one system: for every target the pair terms
// of the reference's FP64 expression, summed in increasing partner index from
// +0 -- the order in which the single-threaded pair loop adds into acc[i].
// Included by nbody_kernels.hip.
//
// The sums are chains of dependent adds, so the parallelism beyond one lane per
// target has to come from computing the terms elsewhere and bringing them to
// the chain in order.  What that costs sets the shapes (MI355X, 256 CUs, unit
// masses; the arithmetic alone is 33 full-rate FP64 instructions and a
// transcendental, 149 cycles of a SIMD per 64 terms):
//
//  * k_exact_relay: 64 targets per workgroup, one per lane.  Every wave computes
//    P partners' terms into registers, takes the three running sums from LDS
//    when the wave before it is done, adds its terms and passes the sums on.
//    Nothing but the sums goes through LDS: a form that hands every term
//    through LDS moves 48 bytes per term, more than LDS delivers at the rate
//    the terms are made, and its fold waves also unbalance the SIMDs (16384
//    bodies: 450 us that way, 350 us here, 0.9 of the issue bound).
//  * k_exact_slot: the same with 32 or 16 targets per workgroup and 2 or 4
//    partner slots per wave, for sizes whose 64-target grid would leave CUs
//    empty (8192 bodies: 109 us against 167 us with 64 targets; 4096: 37
//    against 87 us).  The slots' sums follow each other inside a wave, so the
//    adds cost 2 or 4 times as many instructions.
//  * k_exact_tile: 1 to 8 targets, for the smallest systems, whose time is the
//    chain of n adds and the latency around it.  Producer waves write a tile's
//    terms to LDS, one wave adds the previous tile's (1000 bodies: 23 -> 9 us;
//    64: 5.4 -> 3.5 us).
//
// Partners past the end and a target's own index contribute +0: the running
// sum starts at +0 and is never -0, so adding +0 leaves its bits unchanged.
#pragma once

namespace odehip {
namespace {

#define ODEHIP_LDS __attribute__((address_space(3)))

typedef double double2_t __attribute__((ext_vector_type(2)));

// Polls a wave makes for its turn before it gives up with NaN sums.  Turns
// always come (every wave before it only waits for earlier ones), so the
// limit is never met; it bounds the kernel whatever happens.
constexpr int kTurnPolls = 1 << 22;

// The workgroup's vote on the two shortcuts: whether every position coordinate
// admits the shared-reciprocal terms and, from `uni_min_n` bodies on, the
// masses' common power of two (uniform_pow2_mass), else 0.
struct ExactForm {
  bool shared;
  double m_uni;
};
template <bool kMass, bool kSharedRcp>
__device__ inline ExactForm exact_form(const double* __restrict__ y,
                                       const double* __restrict__ mass, int n, int uni_min_n) {
  ExactForm f{false, 0.0};
  if constexpr (kSharedRcp) {
    f.shared = all_positions_shared_ok(y, n);
    if constexpr (kMass) {
      if (f.shared && n >= uni_min_n) f.m_uni = uniform_pow2_mass(mass, n);
    }
  } else {
    __syncthreads();  // the callers' LDS set-up
  }
  return f;
}
// Below this size the second pass over the masses costs more than the three
// products per term it saves.
constexpr int kUniformMassMinN = 2048;

// ------------------------------------------------------------------ relay --
struct RelaySums {
  double x[64], y[64], z[64];
  int turn;  // chunk whose wave may add next
};

// W waves, P partners per chunk; chunk c belongs to wave c % W.  The polls
// read the turn before the sums and a pass writes it after them: a wave's LDS
// operations execute in order, so a wave that sees its turn has the sums.
template <bool kMass, bool kShared, int W, int P>
__device__ __forceinline__ void relay_sum(volatile ODEHIP_LDS RelaySums* box, uniform_ptr yu,
                                          uniform_ptr mu, int n, double eps2, double xi,
                                          double yi, double zi, int wave, int lane, int i0,
                                          int i) {
  constexpr int U = kFastSet;
  static_assert(P % (2 * U) == 0, "chunks are pairs of sets");
  const int n_full = n / P;
  FastSet<kMass> sa, sb;
  double tx[P], ty[P], tz[P];
  auto terms = [&](const FastSet<kMass>& s, int base) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      exact_term<kMass, kShared>(s.c[3 * u] - xi, s.c[3 * u + 1] - yi, s.c[3 * u + 2] - zi,
                                 kMass ? s.m[u] : 1.0, eps2, tx[base + u], ty[base + u],
                                 tz[base + u]);
      // complete here: sunk past the wait for the turn, the terms would be
      // computed one wave at a time
      tx[base + u] = opaque(tx[base + u]);
      ty[base + u] = opaque(ty[base + u]);
      tz[base + u] = opaque(tz[base + u]);
    }
  };
  auto take = [&](int c, double& ax, double& ay, double& az) {
    for (int polls = 0;; ++polls) {
      const int turn = box->turn;
      ax = box->x[lane];
      ay = box->y[lane];
      az = box->z[lane];
      if (__builtin_amdgcn_readfirstlane(turn) == c) break;
      if (polls == kTurnPolls) {
        ax = ay = az = __builtin_nan("");
        break;
      }
    }
    __builtin_amdgcn_s_setprio(3);  // the other waves wait for these adds
  };
  auto pass = [&](int c, double ax, double ay, double az) {
    box->x[lane] = ax;
    box->y[lane] = ay;
    box->z[lane] = az;
    if (lane == 0) box->turn = c + 1;
    __builtin_amdgcn_s_setprio(0);
  };
  int c = wave;
  if (c < n_full) fast_load<kMass>(sa, yu, mu, c * P);
  for (; c < n_full; c += W) {
    const int j0 = c * P;
#pragma unroll
    for (int b = 0; b < P / U; b += 2) {
      scalar_loads_drain();
      fast_load<kMass>(sb, yu, mu, j0 + (b + 1) * U);
      __builtin_amdgcn_sched_barrier(0);
      terms(sa, b * U);
      scalar_loads_drain();
      fast_load<kMass>(sa, yu, mu,
                       b + 2 < P / U ? j0 + (b + 2) * U : min((c + W) * P, n - U));
      __builtin_amdgcn_sched_barrier(0);
      terms(sb, (b + 1) * U);
    }
    double ax, ay, az;
    take(c, ax, ay, az);
    if (j0 + P <= i0 || j0 >= i0 + 64) {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        ax += tx[p];
        ay += ty[p];
        az += tz[p];
      }
    } else {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const bool self = j0 + p == i;
        ax += self ? 0.0 : tx[p];
        ay += self ? 0.0 : ty[p];
        az += self ? 0.0 : tz[p];
      }
    }
    pass(c, ax, ay, az);
  }
  // the partners past the last whole chunk, one at a time
  if (c == n_full && n_full * P < n) {
    double ax, ay, az;
    take(c, ax, ay, az);
    for (int j = n_full * P; j < n; ++j) {
      double ux, uy, uz;
      exact_term<kMass, kShared>(yu[3 * j] - xi, yu[3 * j + 1] - yi, yu[3 * j + 2] - zi,
                                 kMass ? mu[j] : 1.0, eps2, ux, uy, uz);
      const bool self = j == i;
      ax += self ? 0.0 : ux;
      ay += self ? 0.0 : uy;
      az += self ? 0.0 : uz;
    }
    pass(c, ax, ay, az);
  }
}

template <bool kMass, bool kSharedRcp, int W, int P>
__global__ __launch_bounds__(64 * W) void k_exact_relay(NBodyArgs a) {
  if (prologue_skip(a)) return;
  __shared__ RelaySums box;
  const double* __restrict__ y = select_input(a);
  const uniform_ptr yu = as_uniform(y);
  const uniform_ptr mu = as_uniform(a.mass);
  const int n = a.n;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = blockIdx.x * 64;
  const int i = i0 + lane;
  const int ic = i < n ? i : n - 1;
  const double xi = y[3 * ic], yi = y[3 * ic + 1], zi = y[3 * ic + 2];
  const Velocity vel = load_velocity(a, y, i0, 64, 192);
  if (threadIdx.x < 64) {
    box.x[lane] = box.y[lane] = box.z[lane] = 0.0;
    box.turn = 0;
  }
  const ExactForm f = exact_form<kMass, kSharedRcp>(y, a.mass, n, kUniformMassMinN);
  volatile ODEHIP_LDS RelaySums* sums = (volatile ODEHIP_LDS RelaySums*)&box;
  double scale = 1.0;
  if (kMass && kSharedRcp && f.m_uni != 0.0) {
    relay_sum<false, true, W, P>(sums, yu, mu, n, a.eps2, xi, yi, zi, wave, lane, i0, i);
    scale = f.m_uni;
  } else if (kSharedRcp && f.shared) {
    relay_sum<kMass, true, W, P>(sums, yu, mu, n, a.eps2, xi, yi, zi, wave, lane, i0, i);
  } else {
    relay_sum<kMass, false, W, P>(sums, yu, mu, n, a.eps2, xi, yi, zi, wave, lane, i0, i);
  }
  __syncthreads();
  if (wave < 3 && i < n) {
    const double acc = wave == 0 ? box.x[lane] : wave == 1 ? box.y[lane] : box.z[lane];
    put<kStageLoads>(a, 3L * n + 3 * i + wave, acc * scale);
  }
  put_velocity<kStageLoads>(a, vel);
}

// ------------------------------------------------------------------- slot --
// T = 64 / Q targets, lane (slot q, target t); a chunk is Q P partners, slot q
// taking its P from q P on.  Sums and turns per coordinate, so that the next
// wave may add x while this one adds y.
template <int T>
struct SlotSums {
  double v[3][T];
  int turn[4];
};

// The value each 16-lane row (32-lane half) holds, in both rows of a pair
// (both halves): which = 0 the lower one's, 1 the upper one's.
__device__ __forceinline__ double pair_rows(double x, int which) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = static_cast<uint32_t>(b), hi = static_cast<uint32_t>(b >> 32);
  const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  return __builtin_bit_cast(double, (static_cast<uint64_t>(h[which]) << 32) | l[which]);
}
__device__ __forceinline__ double lower_half(double x) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = static_cast<uint32_t>(b), hi = static_cast<uint32_t>(b >> 32);
  const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return __builtin_bit_cast(double, (static_cast<uint64_t>(h[0]) << 32) | l[0]);
}
// The sums of slot q's lanes in the lanes of slot q + 1.
template <int Q>
__device__ __forceinline__ double to_next_slot(double sum, int q) {
  if (Q == 2) return lower_half(sum);
  if (q == 1) return lower_half(pair_rows(sum, 1));
  return pair_rows(sum, 0);
}

template <bool kMass, bool kShared, int Q, int P, int W>
__device__ __forceinline__ void slot_sum(volatile ODEHIP_LDS SlotSums<64 / Q>* box,
                                         ODEHIP_LDS double2_t (*stage)[2],
                                         const double* __restrict__ y,
                                         const double* __restrict__ mass, int n, double eps2,
                                         double xi, double yi, double zi, int wave, int lane,
                                         int i0, int i) {
  constexpr int T = 64 / Q, C = Q * P;
  const int n_chunks = (n + C - 1) / C;
  const int q = lane / T, t = lane % T;
  const int sl = lane % C;  // the partner of the chunk this lane stages
  // a wave's partners of one chunk: loaded once, read by the slots' lanes
  auto put = [&](double px, double py, double pz, double pm) {
    stage[sl][0] = double2_t{px, py};
    stage[sl][1] = double2_t{pz, pm};
  };
  {
    const int j = min(wave * C + sl, n - 1);
    put(y[3 * j], y[3 * j + 1], y[3 * j + 2], kMass ? mass[j] : 1.0);
  }
  for (int c = wave; c < n_chunks; c += W) {
    const int j0 = c * C;
    const int jn = min(j0 + W * C + sl, n - 1);  // this wave's next chunk
    const double nx = y[3 * jn], ny = y[3 * jn + 1], nz = y[3 * jn + 2];
    const double nm = kMass ? mass[jn] : 1.0;
    double v[3][P];
    ODEHIP_LDS double2_t (*mine)[2] = stage + q * P;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const double2_t xy = mine[p][0], zm = mine[p][1];
      exact_term<kMass, kShared>(xy[0] - xi, xy[1] - yi, zm[0] - zi, kMass ? zm[1] : 1.0, eps2,
                                 v[0][p], v[1][p], v[2][p]);
    }
    if (j0 + C > n || (j0 < i0 + T && j0 + C > i0)) {
      const int jq = j0 + q * P;
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const bool out = jq + p >= n || jq + p == i;
#pragma unroll
        for (int k = 0; k < 3; ++k) v[k][p] = out ? 0.0 : v[k][p];
      }
    }
    // complete before the wait for the turn (as in relay_sum)
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int k = 0; k < 3; ++k) v[k][p] = opaque(v[k][p]);
    put(nx, ny, nz, nm);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      double acc;
      for (int polls = 0;; ++polls) {
        const int turn = box->turn[k];
        acc = box->v[k][t];
        if (__builtin_amdgcn_readfirstlane(turn) == c) break;
        if (polls == kTurnPolls) {
          acc = __builtin_nan("");
          break;
        }
      }
      if (k == 0) __builtin_amdgcn_s_setprio(3);
#pragma unroll
      for (int s = 0; s < Q; ++s) {
        if (s > 0) acc = to_next_slot<Q>(acc, s - 1);
#pragma unroll
        for (int p = 0; p < P; ++p) acc += v[k][p];
      }
      if (lane >= 64 - T) box->v[k][t] = acc;  // the last slot's lanes
      if (lane == 0) box->turn[k] = c + 1;
    }
    __builtin_amdgcn_s_setprio(0);
  }
}

// The last workgroup's targets are the last T bodies (some of them twice, with
// the same bits), so every lane has a target: n >= T.
template <bool kMass, bool kSharedRcp, int Q, int P, int W>
__global__ __launch_bounds__(64 * W) void k_exact_slot(NBodyArgs a) {
  if (prologue_skip(a)) return;
  constexpr int T = 64 / Q, C = Q * P;
  __shared__ SlotSums<T> box;
  __shared__ double2_t stage[W][C][2];
  const double* __restrict__ y = select_input(a);
  const double* __restrict__ mass = a.mass;
  const int n = a.n;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = min(static_cast<int>(blockIdx.x) * T, n - T);
  const int i = i0 + lane % T;
  const double xi = y[3 * i], yi = y[3 * i + 1], zi = y[3 * i + 2];
  const int e = threadIdx.x;
  const Velocity vel = load_velocity(a, y, i0, T, 3 * T);
  if (e < 3 * T) (&box.v[0][0])[e] = 0.0;
  if (e < 4) box.turn[e] = 0;
  const ExactForm f = exact_form<kMass, kSharedRcp>(y, mass, n, kUniformMassMinN);
  auto* sums = (volatile ODEHIP_LDS SlotSums<T>*)&box;
  auto* mine = (ODEHIP_LDS double2_t (*)[2])stage[wave];
  double scale = 1.0;
  if (kMass && kSharedRcp && f.m_uni != 0.0) {
    slot_sum<false, true, Q, P, W>(sums, mine, y, mass, n, a.eps2, xi, yi, zi, wave, lane, i0, i);
    scale = f.m_uni;
  } else if (kSharedRcp && f.shared) {
    slot_sum<kMass, true, Q, P, W>(sums, mine, y, mass, n, a.eps2, xi, yi, zi, wave, lane, i0, i);
  } else {
    slot_sum<kMass, false, Q, P, W>(sums, mine, y, mass, n, a.eps2, xi, yi, zi, wave, lane, i0,
                                    i);
  }
  __syncthreads();
  if (e < 3 * T) put<kStageLoads>(a, 3L * n + 3 * (i0 + e % T) + e / T, (&box.v[0][0])[e] * scale);
  put_velocity<kStageLoads>(a, vel);
}

// ------------------------------------------------------------------- tile --
// T targets as H groups of R; a producer lane computes partner lane % PL
// against the R targets of group lane / PL.  A tile is NP PL partners.  Wave 0
// adds, so the producers are the waves off its SIMD (waves are dealt to the
// four SIMDs in turn).
template <int T_, int H_, int NP_>
struct TileShape {
  static constexpr int T = T_, H = H_, NP = NP_;
  static constexpr int R = T / H, PL = 64 / H, TJ = NP * PL;
  static constexpr int S = TJ + 2;  // row stride: 16-byte reads of 3 T rows without conflicts
  static constexpr int W = NP == 1 ? 2 : NP / 3 * 4;
  static_assert(NP == 1 || NP % 3 == 0, "producers sit on three SIMDs");
};

template <typename Sh, bool kMass>
struct TileLane {
  double tx[Sh::R], ty[Sh::R], tz[Sh::R];  // this lane's targets
  double px, py, pz, pm;                   // its partner of the coming tile
};

template <typename Sh, bool kMass, bool kShared>
__device__ __forceinline__ double tile_sum(double (*term)[3 * Sh::T][Sh::S],
                                           TileLane<Sh, kMass> L, const double* __restrict__ y,
                                           const double* __restrict__ mass, int n, double eps2,
                                           int wave, int pw, int lane, int i0) {
  constexpr int T = Sh::T, R = Sh::R, PL = Sh::PL, TJ = Sh::TJ, S = Sh::S;
  const int n_tiles = (n + TJ - 1) / TJ;
  const int p = lane % PL, h = lane / PL;
  const int row = lane < 3 * T ? lane : 0;
  double acc = 0.0;
  for (int t = 0; t <= n_tiles; ++t) {
    if (pw >= 0 && t < n_tiles) {
      const int jw = t * TJ + pw * PL;  // this wave's first partner of the tile
      const int j = min(jw + TJ + p, n - 1);
      const double qx = y[3 * j], qy = y[3 * j + 1], qz = y[3 * j + 2];
      const double qm = kMass ? mass[j] : 1.0;
      double(*dst)[S] = term[t & 1];
      const int col = pw * PL + p;
      const bool plain = jw + PL <= n && (jw + PL <= i0 || jw >= i0 + T);
#pragma unroll
      for (int u = 0; u < R; ++u) {
        double ax, ay, az;
        exact_term<kMass, kShared>(L.px - L.tx[u], L.py - L.ty[u], L.pz - L.tz[u], L.pm, eps2,
                                   ax, ay, az);
        if (!plain) {
          const bool out = jw + p >= n || jw + p == i0 + h * R + u;
          ax = out ? 0.0 : ax;
          ay = out ? 0.0 : ay;
          az = out ? 0.0 : az;
        }
        dst[h * R + u][col] = ax;
        dst[T + h * R + u][col] = ay;
        dst[2 * T + h * R + u][col] = az;
      }
      L.px = qx;
      L.py = qy;
      L.pz = qz;
      L.pm = qm;
    }
    if (wave == 0 && t > 0) {
      // Straight-line adds, 16 partners' terms read ahead: with the reads a
      // step behind (or a branch in between, which makes the wait drain them
      // all) a partner costs 15-20 cycles instead of 10.
      constexpr int Q = 8;
      const double2_t* src = reinterpret_cast<const double2_t*>(&term[(t - 1) & 1][row][0]);
      double2_t v[2][Q];
#pragma unroll
      for (int m = 0; m < Q; ++m) v[0][m] = src[m];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < TJ / 2; b += Q) {
        const int cur = (b / Q) & 1;
        if (b + Q < TJ / 2) {
#pragma unroll
          for (int m = 0; m < Q; ++m) v[cur ^ 1][m] = src[b + Q + m];
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int m = 0; m < Q; ++m) {
          acc += v[cur][m][0];
          acc += v[cur][m][1];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
  }
  return acc;
}

// n >= T, as for k_exact_slot.
template <typename Sh, bool kMass, bool kSharedRcp>
__global__ __launch_bounds__(64 * Sh::W) void k_exact_tile(NBodyArgs a) {
  if (prologue_skip(a)) return;
  constexpr int T = Sh::T, PL = Sh::PL;
  __shared__ __attribute__((aligned(16))) double term[2][3 * T][Sh::S];
  const double* __restrict__ y = select_input(a);
  const double* __restrict__ mass = a.mass;
  const int n = a.n;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = min(static_cast<int>(blockIdx.x) * T, n - T);
  const int pw = Sh::NP == 1 ? wave - 1 : (wave & 3) ? (wave >> 2) * 3 + (wave & 3) - 1 : -1;
  // the first partners and the targets come in with the range test's loads
  TileLane<Sh, kMass> L{};
  if (pw >= 0) {
    const int j = min(pw * PL + lane % PL, n - 1);
    L.px = y[3 * j];
    L.py = y[3 * j + 1];
    L.pz = y[3 * j + 2];
    L.pm = kMass ? mass[j] : 1.0;
#pragma unroll
    for (int u = 0; u < Sh::R; ++u) {
      const int i = i0 + lane / PL * Sh::R + u;
      L.tx[u] = y[3 * i];
      L.ty[u] = y[3 * i + 1];
      L.tz[u] = y[3 * i + 2];
    }
  }
  const Velocity vel = load_velocity(a, y, i0, T, 64);
  ExactForm f{false, 0.0};
  if (kSharedRcp && n <= Sh::TJ)  // the producers hold every partner
    f.shared = __syncthreads_and(pw < 0 || point_shared_ok(L.px, L.py, L.pz)) != 0;
  else
    f = exact_form<kMass, kSharedRcp>(y, mass, n, kUniformMassMinN);
  double acc, scale = 1.0;
  if (kMass && kSharedRcp && f.m_uni != 0.0) {
    TileLane<Sh, false> U;
    __builtin_memcpy(&U, &L, sizeof U);
    acc = tile_sum<Sh, false, true>(term, U, y, mass, n, a.eps2, wave, pw, lane, i0);
    scale = f.m_uni;
  } else if (kSharedRcp && f.shared) {
    acc = tile_sum<Sh, kMass, true>(term, L, y, mass, n, a.eps2, wave, pw, lane, i0);
  } else {
    acc = tile_sum<Sh, kMass, false>(term, L, y, mass, n, a.eps2, wave, pw, lane, i0);
  }
  if (wave == 0 && lane < 3 * T) put<kStageLoads>(a, 3L * n + 3 * (i0 + lane % T) + lane / T, acc * scale);
  put_velocity<kStageLoads>(a, vel);
}

// --------------------------------------------------------------- dispatch --
// Launches kernel template K<kMass, kSharedRcp, ...> for the call's masses and
// softening (the shared-reciprocal form needs softening^2 in [2^-200, 2^100]).
template <int W, int P>
void launch_exact_relay(const NBodyArgs& a, bool shared, hipStream_t s) {
  auto* kern = a.mass ? (shared ? k_exact_relay<true, true, W, P> : k_exact_relay<true, false, W, P>)
                      : (shared ? k_exact_relay<false, true, W, P>
                                : k_exact_relay<false, false, W, P>);
  hipLaunchKernelGGL(kern, dim3((a.n + 63) / 64), dim3(64 * W), 0, s, a);
}
// Without the shared reciprocal a partner's term takes more registers: with 16 of
// them the instance with masses spilled (softening 0, 8192 bodies 230 us, 24576 2.04 ms;
// with 12 186 us and 1.64 ms, without masses 182 / 181 us).
template <int Q, int P, int W>
void launch_exact_slot(const NBodyArgs& a, bool shared, hipStream_t s) {
  constexpr int T = 64 / Q, kIeeeP = 12;
  auto* kern = a.mass ? (shared ? k_exact_slot<true, true, Q, P, W>
                                : k_exact_slot<true, false, Q, kIeeeP, W>)
                      : (shared ? k_exact_slot<false, true, Q, P, W>
                                : k_exact_slot<false, false, Q, kIeeeP, W>);
  hipLaunchKernelGGL(kern, dim3((a.n + T - 1) / T), dim3(64 * W), 0, s, a);
}
template <typename Sh>
void launch_exact_tile(const NBodyArgs& a, bool shared, hipStream_t s) {
  auto* kern = a.mass ? (shared ? k_exact_tile<Sh, true, true> : k_exact_tile<Sh, true, false>)
                      : (shared ? k_exact_tile<Sh, false, true> : k_exact_tile<Sh, false, false>);
  hipLaunchKernelGGL(kern, dim3((a.n + Sh::T - 1) / Sh::T), dim3(64 * Sh::W), 0, s, a);
}

// The shape with the least time by rounds: a launch runs its workgroups on the
// CUs in ceil(workgroups / CUs) rounds.  Up to 8 targets a workgroup the grid
// is one round (T targets for n <= T CUs); beyond, a round of the 16- and
// 32-target kernels costs 0.425 and 0.63 of a 64-target round (sweep over
// n = 4096 ... 20001), so e.g. 8192 bodies take one round of 32 targets and
// 20001 three of them rather than two of 64.
void launch_exact(const NBodyArgs& a, long device_cus, hipStream_t s) {
  const long cus = device_cus < 4 ? 4 : device_cus;  // every shape's targets <= n below
  const bool shared = a.eps2 >= 0x1p-200 && a.eps2 <= 0x1p100;
  const long n = a.n;
  if (n <= cus) return launch_exact_tile<TileShape<1, 1, 1>>(a, shared, s);
  if (n <= 2 * cus) return launch_exact_tile<TileShape<2, 1, 3>>(a, shared, s);
  if (n <= 4 * cus) return launch_exact_tile<TileShape<4, 1, 3>>(a, shared, s);
  if (n <= 8 * cus) return launch_exact_tile<TileShape<8, 2, 6>>(a, shared, s);
  auto rounds = [&](long targets) {
    return static_cast<double>(((n + targets - 1) / targets + cus - 1) / cus);
  };
  const double c16 = 0.425 * rounds(16), c32 = 0.63 * rounds(32), c64 = rounds(64);
  if (c16 < c32 && c16 < c64) return launch_exact_slot<4, 16, 8>(a, shared, s);
  if (c32 < c64) return launch_exact_slot<2, 16, 8>(a, shared, s);
  // two or more workgroups per CU: four waves each, three workgroups resident
  // (65536 bodies: 5.1 against 5.3 ms with eight); fewer: eight waves (16384
  // bodies: 350 against 395 us with four)
  if (rounds(64) >= 2.0) return launch_exact_relay<4, 16>(a, shared, s);
  launch_exact_relay<8, 16>(a, shared, s);
}

}  // namespace
}  // namespace odehip
