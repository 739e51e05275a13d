// HIP kernels for gfx950 (MI355X): LocVolCalib prices by separation of the
// x direction (the grids' modes), FP64.
//
// What separates.  MuX = MuY = 0 and VarX = x^(2 beta) * exp(2 y - nu^2 t),
// VarY = nu^2 (LocVolCalib.fut:50-66), so with d2 the plain second difference
// (uniform grids, zero on the boundary nodes, :26-44) a time step of
// `rollback` (:180-209) works with
//     Lx = E_j(t) * B,  B = x^(2 beta) / (4 dx^2) * d2x,  E_j = exp(2 y_j - nu^2 t)
//     Ly = nu^2 / (4 dy^2) * d2y
// and, for s = 1/dt, u = (s + Lx + 2 Ly) r; (s - Lx) u' = u;
// (s - Ly) r' = s u' - Ly r.  B is the same for every row and step and is
// similar to a symmetric matrix, so B z_k = -lambda_k z_k with a complete set
// of modes, orthogonal in the weights m_i = 4 dx^2 / x_i^(2 beta).  In that
// basis x is diagonal: mode k is a system of its own in y alone, with no
// exchange between modes at any step.  Eliminating u from the two solves
// gives, with A = (s - Ly) / 2s and eps_jk = E_j lambda_k / 2s,
//     r' = r + A^-1 (1/2 + eps)^-1 (Ly / 2s - eps) r
// (the same scheme in exact arithmetic: (1/2 + eps) is (s - Lx) / 2s).
//
// What every option shares.  The payoff max(x - K, 0) (:46-47) does not
// depend on y, and linear functions of x are left unchanged by every step,
// so the payoff minus its chord through the grid's ends is a sum of modes
// times the constant 1 in y: one scalar f_k per mode, the value at y = NY/2
// after all steps from 1 everywhere, serves every strike.  Summation by
// parts leaves the payoff's second difference, which is zero except at the
// two nodes around K in [x_i, x_i+1):
//     price = chord(x_idx) - sum_k f_k z_k(x_idx)
//             * (z_k(i) (x_i+1 - K) + z_k(i+1) (K - x_i)) / (lambda_k sum_j m_j z_k(j)^2).
// The work is one grid's point steps in FP64 for any number of strikes, at
// one launch for all time steps, in place of two launches per step that each
// move every option's grid (63 steps, 128 options of 256 x 256: 126 launches,
// 8.5 GB).  The price is what is left of the chord, with the chord's rounding.
// The host takes this path where the scalars allow it, the steps are worth three
// launches (lvc_modes_fit) and the price is not lost that way (lvc_modes_strike).
//
// Three kernels: lvc_modes_kernel (eigenvalues, eigenvectors, the options'
// coefficients), lvc_evolve_kernel (f_k: every time step), lvc_price_kernel
// (the sums over k).
//
// Rounding: compiled without contraction, every fused multiply-add written
// as fma(), each mode's and option's operations depending on its own grid
// alone: a price has the same bits alone and in any batch.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "lvc_internal.h"

namespace {

__device__ __forceinline__ uint32_t hi_word(double v) {
  return (uint32_t)((unsigned long long)__double_as_longlong(v) >> 32);
}
__device__ __forceinline__ double from_hi(uint32_t hi) {
  return __longlong_as_double((long long)((unsigned long long)hi << 32));
}

// 1/d for normal d of moderate size: v_rcp_f64 (relative error e up to
// 2^-24.4, measured over 67 million values) times 1 + e + e^2.
__device__ __forceinline__ double recip(double d) {
  const double x0 = __builtin_amdgcn_rcp(d);
  const double e = fma(-d, x0, 1.0);
  return fma(x0, fma(e, e, e), x0);
}

// The grid in scalar registers: the one in the kernel's arguments (main), or
// grids[i], i uniform.
template <bool ONE>
__device__ __forceinline__ lvc_mgrid load_grid(const lvc_modes_args &a, int i) {
  if constexpr (ONE)
    return a.one;
  else
    return a.grids[__builtin_amdgcn_readfirstlane(i)];
}

// Grid node i of initGrid (LocVolCalib.fut:21).
__device__ __forceinline__ double node(const lvc_mgrid &g, int i) {
  return (double)i * g.dx - (double)g.xindex * g.dx + g.s0;
}

__device__ __forceinline__ double strike_of(const lvc_modes_args &a, int option) {
  if (a.strikes) return a.strikes[option];
  // main's strikes (LocVolCalib.fut:247)
  return a.strike_f32 ? (double)(0.001f * (float)option) : 0.001 * (double)option;
}

__device__ __forceinline__ double payoff(double x, double k) {
  const double v = x - k;
  return v > 0.0 ? v : 0.0;  // f32.max v 0 (:47); 0 for a NaN strike
}

// ---- modes -------------------------------------------------------------------
//
// lambda_k from the left shooting recurrence of B z = -lambda z in flux form,
//     G_i = G_(i-1) - m_i z_i,  z_(i+1) = z_i + lambda G_i,  z_0 = 0, G_0 = 1:
// the sign changes of z_1 .. z_(N+1) count the eigenvalues below lambda
// (Sturm), and z_(N+1) = 0 exactly at one.  Two dependent FP64 operations per
// node and no division; the flux form keeps small eigenvalues to full
// relative accuracy, and since m falls with x (beta >= 0) the modes grow from
// the left boundary, the stable direction.  (z_(N+1)/G_N) has the exact
// derivative sum G^2 / G_N^2, so a Newton step costs one more operation per
// node; the sum is also the mode's norm (sum m z^2 = lambda sum G^2).
//
// One wavefront takes kModes consecutive modes, 16 lanes each.  Two rounds of
// 64 points over the modes' common interval, two of 16 points per mode (in
// sqrt(lambda), where modes are evenly spaced), the last one ending in a
// Newton step, then Newton passes guarded by the count's bracket, two as a
// rule.  A pass is a serial chain of 3 or 4 operations per node at 4.8 cycles
// each (a dependent FP64 operation issues right behind the last one), so what
// matters is that nothing else is in it: a block's weights come into
// registers ahead of the block before, and the values kept go out a block at
// a time.  (With the weights read and the values written node by node the
// kernel took 60 us on 256 nodes, most of it LDS latency.)  64 lanes per mode
// would save one pass in six and cost the batched form four times the work.

constexpr int kLanes = 16, kModes = LVC_MODES_PER_WAVE;
static_assert(kLanes * kModes == 64, "a wavefront's modes fill it");
constexpr int kBlk = 16;  // nodes between rescalings

struct Shot {
  double z, g, q;  // z_(N+1), G_N, sum of G^2, at scale 2^-e
  int e, count;
};

// One shooting pass over the N interior nodes for this lane's lambda; node i's
// weight is mass[i - 1], and mass is readable for two blocks past the last
// node's.  SUM: with q.  KEEP: the nodes' values to zs[0 .. N-1] and each
// block's scale to es[], by the lanes with `writer`.
template <bool SUM, bool KEEP>
__device__ __forceinline__ Shot shoot(double lambda, const double *mass, int N, double *zs,
                                      int *es, bool writer) {
  double z = lambda, g = 1.0, q = 1.0;
  int e = 0, count = 0;
  uint32_t signs = 0;  // bit 0: the sign of z_1, positive
  double kept[KEEP ? kBlk : 1];
  auto load = [&](double (&m)[kBlk], int i0) {
#pragma unroll
    for (int i = 0; i < kBlk; ++i) m[i] = mass[i0 + i];
  };
  auto step = [&](const double (&m)[kBlk], int i) {
    if constexpr (KEEP) kept[i] = z;
    g = fma(-m[i], z, g);
    z = fma(lambda, g, z);
    if constexpr (SUM) q = fma(g, g, q);
    signs = __builtin_amdgcn_alignbit(signs, hi_word(z), 31);
  };
  auto finish = [&](int i0, int taken) {
    // bit `taken` is the sign before the block, bit 0 the last one
    count += __popc((signs ^ (signs >> 1)) & ((1u << taken) - 1u));
    if constexpr (KEEP) {
      if (writer) {
        es[i0 / kBlk] = e;
#pragma unroll
        for (int i = 0; i < kBlk; ++i) zs[i0 + i] = kept[i];
      }
    }
    // a block grows z and G by at most (lambda m)^16: bring the larger to [1, 2)
    const uint32_t hz = hi_word(z) & 0x7ff00000u, hg = hi_word(g) & 0x7ff00000u;
    const int x = (int)((hz > hg ? hz : hg) >> 20) - 1023;
    const double sc = from_hi((uint32_t)(1023 - x) << 20);
    z *= sc;
    g *= sc;
    if constexpr (SUM) q *= sc * sc;
    e += x;
  };
  auto block = [&](const double (&m)[kBlk], int i0) {
#pragma unroll
    for (int i = 0; i < kBlk; ++i) step(m, i);
    finish(i0, kBlk);
  };
  auto tail = [&](const double (&m)[kBlk], int i0) {
#pragma unroll
    for (int i = 0; i < kBlk - 1; ++i)
      if (i < N - i0) step(m, i);
    finish(i0, N - i0);
  };
  double m0[kBlk], m1[kBlk];
  load(m0, 0);
  int i0 = 0;
  for (; i0 + 2 * kBlk <= N; i0 += 2 * kBlk) {
    load(m1, i0 + kBlk);
    block(m0, i0);
    load(m0, i0 + 2 * kBlk);
    block(m1, i0 + kBlk);
  }
  if (i0 + kBlk <= N) {
    load(m1, i0 + kBlk);
    block(m0, i0);
    i0 += kBlk;
    if (i0 < N) tail(m1, i0);
  } else if (i0 < N) {
    tail(m0, i0);
  }
  return Shot{z, g, q, e, count};
}

// The point l+1 of n parts of [lo, hi].
__device__ __forceinline__ double part(double lo, double hi, int l, double inv) {
  return fma(hi - lo, (double)(l + 1) * inv, lo);
}

template <bool ONE>
__global__ __launch_bounds__(64) void lvc_modes_kernel(lvc_modes_args a) {
  extern __shared__ double lds[];
  const int lane = threadIdx.x, grp = lane / kLanes, l = lane % kLanes;
  int gi = 0, first = blockIdx.x * kModes;
  if constexpr (!ONE) {
    gi = a.mode_tiles[blockIdx.x].grid;
    first = a.mode_tiles[blockIdx.x].first;
  }
  const lvc_mgrid G = load_grid<ONE>(a, gi);
  const int nx = G.nx, N = nx - 2;
  const int nb = LVC_MODES_BLOCKS(nx), padded = kBlk * nb;
  double *mass = lds;
  double *zs = lds + padded + 2 * kBlk + grp * padded;
  int *es = (int *)(lds + (1 + kModes) * padded + 2 * kBlk) + grp * nb;
  __shared__ double wa[64], wb[64];
  __shared__ int at[64];

  // m_i over its smallest value, m_N (x grows with i, beta >= 0): lambda is
  // then below 4
  const double xN = node(G, N), tb = 2.0 * G.beta;
  const double logN = log(xN);
  for (int i = lane; i < padded + 2 * kBlk; i += 64)
    mass[i] = i < N ? exp(tb * (logN - log(node(G, i + 1)))) : 0.0;
  __syncthreads();

  int k = first + grp;
  const bool live = k < N;
  if (!live) k = N - 1;
  const int klast = (first + kModes <= N ? first + kModes : N) - 1;
  // brackets in sigma = sqrt(lambda)
  double lo = 0.0, hi = 2.0000001;
  for (int round = 0; round < 2; ++round) {
    // all lanes over the modes' common interval (brackets are ordered by k)
    const double wlo = __shfl(lo, 0), whi = __shfl(hi, (klast - first) * kLanes);
    const double sg = part(wlo, whi, lane, 1.0 / 65.0);
    const Shot s = shoot<false, false>(sg * sg, mass, N, nullptr, nullptr, false);
    int below = 0;
#pragma unroll
    for (int m = 0; m < kModes; ++m) {
      const int km = first + m < N ? first + m : N - 1;
      const int p = __popcll(__ballot(s.count <= km));
      if (m == grp) below = p;
    }
    const double nlo = below > 0 ? part(wlo, whi, below - 1, 1.0 / 65.0) : wlo;
    const double nhi = below < 64 ? part(wlo, whi, below, 1.0 / 65.0) : whi;
    lo = nlo > lo ? nlo : lo;
    hi = nhi < hi ? nhi : hi;
  }
  double lambda = 0.0;
  for (int round = 0; round < 2; ++round) {
    const double sg = part(lo, hi, l, 1.0 / 17.0);
    Shot s;
    if (round == 0)
      s = shoot<false, false>(sg * sg, mass, N, nullptr, nullptr, false);
    else
      s = shoot<true, false>(sg * sg, mass, N, nullptr, nullptr, false);
    const uint64_t mask = __ballot(s.count <= k) >> (grp * kLanes);
    const int p = __popcll(mask & ((1ull << kLanes) - 1));
    if (round == 1) lambda = __shfl(fma(sg, sg, -(s.z * s.g) / s.q), grp * kLanes + (p ? p - 1 : 0));
    const double nlo = p > 0 ? part(lo, hi, p - 1, 1.0 / 17.0) : lo;
    const double nhi = p < kLanes ? part(lo, hi, p, 1.0 / 17.0) : hi;
    lo = nlo;
    hi = nhi;
  }
  // Newton on z_(N+1)/G_N inside the bracket; a step that leaves it bisects.
  // The last pass leaves the mode's values in zs (a mode that is done early
  // repeats its last pass).  At most 64 passes.
  double llo = lo * lo, lhi = hi * hi;
  if (!(lambda > llo && lambda < lhi)) lambda = 0.5 * (llo + lhi);
  Shot s = shoot<true, false>(lambda, mass, N, nullptr, nullptr, false);
  bool done = false;
  for (int it = 0;; ++it) {
    if (!done) {
      if (s.count <= k) {
        llo = lambda;
      } else {
        lhi = lambda;
      }
      const double next = lambda - (s.z * s.g) / s.q;
      lambda = next > llo && next < lhi ? next : 0.5 * (llo + lhi);
    }
    s = shoot<true, true>(lambda, mass, N, zs, es, l == 0);
    done = done || fabs(s.z * s.g) <= 1e-13 * lambda * s.q || it >= 63;
    if (__ballot(!done) == 0) break;
  }
  __syncthreads();

  // z_k(i) at the scale of the norm's sum, 0 on the boundary
  auto value = [&](int i) {
    if (i <= 0 || i > N) return 0.0;
    return ldexp(zs[i - 1], es[(i - 1) / kBlk] - s.e);
  };
  if (live && l == 0) {
    const double inv_mass = exp(tb * logN) / (4.0 * G.dx * G.dx);
    a.lambda[G.mode0 + k] = lambda * inv_mass;
  }
  // the options' coefficients, 64 at a time: each lane finds one strike's
  // nodes and weights (node 0, whose value is 0, for none), then every mode's
  // lanes go over them
  const double base = value(G.xindex) / (lambda * lambda * s.q);
  const double x0 = node(G, 0), xe = node(G, nx - 1);
  for (int o0 = 0; o0 < G.count; o0 += 64) {
    const int here = G.count - o0 < 64 ? G.count - o0 : 64;
    if (lane < here) {
      const double K = strike_of(a, G.first + o0 + lane);
      int i = 0;
      double da = 0.0, db = 0.0;
      if (K >= x0 && K < xe) {
        i = (int)((K - x0) / G.dx);
        i = i < 0 ? 0 : (i > nx - 2 ? nx - 2 : i);
        while (i > 0 && node(G, i) > K) --i;
        while (i < nx - 2 && node(G, i + 1) <= K) ++i;
        da = node(G, i + 1) - K;
        db = K - node(G, i);
      }
      at[lane] = i;
      wa[lane] = da;
      wb[lane] = db;
    }
    __syncthreads();
    for (int o = l; o < here && live; o += kLanes) {
      const int i = at[o];
      a.coef[G.coef_off + (int64_t)(o0 + o) * N + k] =
          base * fma(value(i), wa[o], value(i + 1) * wb[o]);
    }
    __syncthreads();
  }
}

// ---- time steps ----------------------------------------------------------------
//
// f_k: mode k's ny unknowns live in registers for all time steps, M rows per
// lane, `lanes` (a power of two) lanes per mode, and no memory is touched in
// the loop.  A's taps are the same at every step, so its factorisation
// (Thomas inside a lane's rows, parallel cyclic reduction of the lanes' last
// rows, every quantity a sum of positive terms) is made once and a step only
// substitutes.  The step is taken as a correction,
//     r' = r + A^-1 d,  d = (Ly r / 2s - eps r) / (1/2 + eps),
// with Ly r from neighbour differences: rounding is then relative to the
// change of a step (f_k to 1e-15; the form r' = A^-1 h', q = r' - h' saves 3
// of 17 operations per row and left 1e-14 to 3e-14).
//
// Bound by FP64 issue of one wavefront per SIMD (14 operations of 4.8 cycles
// and a v_rcp_f64, 20, per row), so a mode is spread over as many lanes as
// exchange cheaply.  Up to 16 lanes (128 rows) the lanes' last rows are
// reduced by DPP shifts within a row of 16 lanes.  Taller columns take a whole
// wavefront: its four rows of 16 are reduced each by itself, then coupled in
// pairs and the pairs to each other, through the two unknowns on either side
// of a seam, which every lane takes by v_readlane.

template <int CTRL>
__device__ __forceinline__ double dpp(double old, double v) {
  const long long o = __double_as_longlong(old), s = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)s, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(s >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// 0 where the source lane is out of reach
template <int CTRL>
__device__ __forceinline__ double dpp0(double v) {
  const long long s = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)s, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(s >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double lane_value(double v, int lane) {
  const long long s = __double_as_longlong(v);
  return __longlong_as_double(
      ((long long)__builtin_amdgcn_readlane((int)(s >> 32), lane) << 32) |
      (unsigned int)__builtin_amdgcn_readlane((int)s, lane));
}

// The value of the next lane below / above: within a row of 16 lanes, or
// (WAVE) the wavefront; 0 where there is none.  Lanes of other modes may be
// read: their taps towards them are zero.
template <bool WAVE>
__device__ __forceinline__ double below(double v) {
  return WAVE ? dpp0<0x138>(v) : dpp0<0x111>(v);  // wave_shr, row_shr
}
template <bool WAVE>
__device__ __forceinline__ double above(double v) {
  return WAVE ? dpp0<0x130>(v) : dpp0<0x101>(v);  // wave_shl, row_shl
}

// The reduced system over the lanes, -A X_below + (A + C + S) X - C X_above = y
// with A, C, S >= 0: factored once, then solved for each y.
template <int V>
struct Int {
  static constexpr int value = V;
};

template <bool WAVE>
struct Reduced {
  double alpha[4], gamma[4], invd;
  // WAVE: what the unknowns at the seams (lanes 15 | 16, 47 | 48, then
  // 31 | 32) add to this lane's
  double seam[6];

  __device__ __forceinline__ double solve_rows(double y) const {
    y = fma(alpha[0], dpp0<0x111>(y), fma(gamma[0], dpp0<0x101>(y), y));
    y = fma(alpha[1], dpp0<0x112>(y), fma(gamma[1], dpp0<0x102>(y), y));
    y = fma(alpha[2], dpp0<0x114>(y), fma(gamma[2], dpp0<0x104>(y), y));
    y = fma(alpha[3], dpp0<0x118>(y), fma(gamma[3], dpp0<0x108>(y), y));
    return y * invd;
  }
  __device__ __forceinline__ double solve_pairs(double y) const {
    const double x = solve_rows(y);
    return fma(seam[0], lane_value(x, 15), fma(seam[1], lane_value(x, 16),
           fma(seam[2], lane_value(x, 47), fma(seam[3], lane_value(x, 48), x))));
  }
  __device__ __forceinline__ double solve(double y) const {
    if constexpr (!WAVE) return solve_rows(y);
    const double x = solve_pairs(y);
    return fma(seam[4], lane_value(x, 31), fma(seam[5], lane_value(x, 32), x));
  }
  // Couples the blocks on either side of the seam lo | lo + 1, this lane in
  // the `mine` one of them (0 lower, 1 upper, else neither): with p a block's
  // response to the unknown below it, r above it and z to the shift
  // (p + r + z = 1), u_lo and u_hi the blocks' own solutions at the seam,
  // x += r (u_hi + p_hi u_lo) / (1 - r_lo p_hi) in the lower block and
  // x += p (u_lo + r_lo u_hi) / (1 - r_lo p_hi) in the upper, the divisor as
  // the sum (1 - r_lo) + r_lo (1 - p_hi).
  __device__ __forceinline__ void couple(double p, double r, double z, int lo, int mine, double &c_lo,
                                         double &c_hi) {
    const double r_lo = lane_value(r, lo), p_hi = lane_value(p, lo + 1);
    const double inv = recip(lane_value(z + p, lo) + r_lo * lane_value(z + r, lo + 1));
    c_lo = mine == 0 ? r * p_hi * inv : mine == 1 ? p * inv : 0.0;
    c_hi = mine == 0 ? r * inv : mine == 1 ? p * r_lo * inv : 0.0;
  }
  __device__ __forceinline__ void factor(double A, double C, double S) {
    const int lane = threadIdx.x, pos = lane & 15;
    double outA = 0.0, outC = 0.0;
    const double S0 = S;
    if constexpr (WAVE) {
      // the taps across the rows' ends wait for the coupling; a row of 16
      // keeps their part of the diagonal
      outA = pos == 0 ? A : 0.0;
      outC = pos == 15 ? C : 0.0;
      A -= outA;
      C -= outC;
      S += outA + outC;
    }
    auto level = [&](auto shr, auto shl, int d) {
      constexpr int kShr = decltype(shr)::value, kShl = decltype(shl)::value;
      const double D = A + C + S;
      alpha[d] = A * recip(dpp<kShr>(1.0, D));
      gamma[d] = C * recip(dpp<kShl>(1.0, D));
      S = S + alpha[d] * dpp0<kShr>(S) + gamma[d] * dpp0<kShl>(S);
      A = alpha[d] * dpp0<kShr>(A);
      C = gamma[d] * dpp0<kShl>(C);
    };
    level(Int<0x111>{}, Int<0x101>{}, 0);
    level(Int<0x112>{}, Int<0x102>{}, 1);
    level(Int<0x114>{}, Int<0x104>{}, 2);
    level(Int<0x118>{}, Int<0x108>{}, 3);
    invd = recip(A + C + S);
    if constexpr (WAVE) {
      const int row = lane >> 4;
      const double p = solve_rows(outA), r = solve_rows(outC), z = solve_rows(S0);
      couple(p, r, z, 15, row, seam[0], seam[1]);
      couple(p, r, z, 47, row - 2, seam[2], seam[3]);
      const double p2 = solve_pairs(lane == 32 ? outA : 0.0);
      const double r2 = solve_pairs(lane == 31 ? outC : 0.0);
      const double z2 = solve_pairs(S0);
      couple(p2, r2, z2, 31, lane >> 5, seam[4], seam[5]);
    }
  }
};

template <int KIND, bool ONE>
__global__ __launch_bounds__(64, KIND == LVC_MODES_WAVE16 ? 1 : 2) void lvc_evolve_kernel(
    lvc_modes_args a) {
  constexpr int M = KIND == LVC_MODES_ROW4 || KIND == LVC_MODES_WAVE4 ? 4
                    : KIND == LVC_MODES_WAVE16 ? 16 : 8;
  constexpr bool WAVE = KIND >= LVC_MODES_WAVE4;
  int gi = 0, first = 0;
  if constexpr (ONE) {
    first = blockIdx.x * (64 / a.one.lanes);
  } else {
    const lvc_mtile t = a.tiles[KIND][blockIdx.x];
    gi = t.grid;
    first = t.first;
  }
  const lvc_mgrid G = load_grid<ONE>(a, gi);
  const int lane = threadIdx.x;
  const int lanes = WAVE ? 64 : G.lanes;
  const int seg = lane & (lanes - 1), k = first + lane / lanes;
  const int ny = G.ny, steps = G.nt - 1;
  const bool live = k < G.nx - 2;
  const double half_dt = 0.5 * (G.t / (double)steps);  // 1 / 2s
  const double lam = live ? a.lambda[G.mode0 + k] * half_dt : 0.0;
  const double tap = half_dt * (G.nu * G.nu / (4.0 * G.dy * G.dy));
  const int row0 = seg * M;
  auto tap_of = [&](int j) { return j >= 1 && j <= ny - 2 ? tap : 0.0; };

  // Thomas on the lane's rows 0 .. M-2: pivots p_j = g_j + c_j with
  // g_j = 1/2 + a_j g_(j-1) / p_(j-1), b_j = c_j / p_j; responses v to the
  // unknown before the lane, w to its own last one, sh to 1/2 in every row
  // (v + w + sh = 1).  el, ep: eps at t = 0, and over the pivot.
  double el[M], ep[M], b[M], v[M - 1], w[M - 1];
  Reduced<WAVE> red;
  {
    double sh[M - 1];
    double g = 0.5 + tap_of(row0), rp = 0.0;
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const int row = row0 + j;
      const double y = (double)row * G.dy - (double)G.yindex * G.dy + G.log_alpha;
      el[j] = row < ny ? lam * exp(2.0 * y) : 0.0;
      if (j == M - 1) break;
      const double c = tap_of(row);
      if (j > 0) g = 0.5 + c * (g * rp);
      rp = recip(g + c);
      ep[j] = el[j] * rp;
      b[j] = c * rp;
      v[j] = j == 0 ? b[0] : b[j] * v[j - 1];
      sh[j] = j == 0 ? 0.5 * rp : fma(b[j], sh[j - 1], 0.5 * rp);
    }
    const double al = tap_of(row0 + M - 1);
    ep[M - 1] = el[M - 1];
    b[M - 1] = al;
    w[M - 2] = b[M - 2];
#pragma unroll
    for (int j = M - 3; j >= 0; --j) {
      w[j] = b[j] * w[j + 1];
      v[j] = fma(b[j], v[j + 1], v[j]);
      sh[j] = fma(b[j], sh[j + 1], sh[j]);
    }
    // the lanes' last rows
    red.factor(al * v[M - 2], al * above<WAVE>(w[0]),
               0.5 + al * (sh[M - 2] + above<WAVE>(sh[0])));
  }

  // exp(-nu^2 t_k), k = steps - 1 - n, for 64 steps n at a time in the lanes
  // (lanes past the last step hold values that are not used)
  double tau64 = exp(-(G.nu * G.nu) * (G.t * (double)(steps - 1 - lane) / (double)steps));
  const double next64 = exp((G.nu * G.nu) * (G.t * 64.0 / (double)steps));
  double r[M];
#pragma unroll
  for (int j = 0; j < M; ++j) r[j] = 1.0;
  for (int n = 0; n < steps; ++n) {
    if ((n & 63) == 0 && n > 0) tau64 *= next64;
    const double tau = lane_value(tau64, n & 63);
    // d over the pivots (the last row's: 1)
    double x[M];
    const double prev = below<WAVE>(r[M - 1]), next = above<WAVE>(r[0]);
    double lo = r[0] - prev;
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const double hi = (j < M - 1 ? r[j + 1] : next) - r[j];
      const double X = recip(fma(el[j], tau, 0.5));
      x[j] = X * fma(b[j], hi - lo, -((ep[j] * tau) * r[j]));
      lo = hi;
    }
#pragma unroll
    for (int j = 1; j < M - 1; ++j) x[j] = fma(b[j], x[j - 1], x[j]);
#pragma unroll
    for (int j = M - 3; j >= 0; --j) x[j] = fma(b[j], x[j + 1], x[j]);
    const double X = red.solve(fma(b[M - 1], x[M - 2] + above<WAVE>(x[0]), x[M - 1]));
    const double Xp = below<WAVE>(X);
#pragma unroll
    for (int j = 0; j < M - 1; ++j) r[j] += fma(v[j], Xp, fma(w[j], X, x[j]));
    r[M - 1] += X;
  }
  const int yj = G.yindex - row0;
#pragma unroll
  for (int j = 0; j < M; ++j)
    if (live && j == yj) a.f[G.mode0 + k] = r[j];
}

// ---- prices --------------------------------------------------------------------

// One wavefront per option: the chord's value at the price node minus the
// sum over the modes, lane l the modes l, l + 64, ...
template <bool ONE, typename O>
__global__ __launch_bounds__(256) void lvc_price_kernel(lvc_modes_args a, int n, O *out) {
  const int o = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (o >= n || (o >= a.far && o < a.far_end)) return;
  const lvc_mgrid G = load_grid<ONE>(a, ONE ? 0 : a.grid_of[o]);
  const int N = G.nx - 2;
  const double *c = a.coef + G.coef_off + (int64_t)(o - G.first) * N, *f = a.f + G.mode0;
  double sum = 0.0;
  for (int k = lane; k < N; k += 256) {
    // four of a lane's modes at once, for one memory round trip
    double fk[4], ck[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kk = k + 64 * i;
      fk[i] = kk < N ? f[kk] : 0.0;
      ck[i] = kk < N ? c[kk] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) sum = fma(fk[i], ck[i], sum);
  }
  for (int st = 32; st > 0; st >>= 1) sum += __shfl_xor(sum, st);
  if (lane == 0) {
    const double K = strike_of(a, o);
    const double x0 = node(G, 0), x1 = node(G, G.nx - 1), x = node(G, G.xindex);
    const double p0 = payoff(x0, K), p1 = payoff(x1, K);
    const double chord = p0 + (p1 - p0) * ((x - x0) / (x1 - x0));
    out[a.out_index ? a.out_index[o] : o] = (O)(chord - sum);
  }
}

}  // namespace

extern "C" {

int lvc_launch_modes(void *stream, const lvc_modes_args *a, int tiles, int max_nx) {
  const size_t lds = LVC_MODES_LDS(max_nx);
  if (a->grids)
    lvc_modes_kernel<false><<<tiles, 64, lds, (hipStream_t)stream>>>(*a);
  else
    lvc_modes_kernel<true><<<tiles, 64, lds, (hipStream_t)stream>>>(*a);
  return (int)hipGetLastError();
}

int lvc_launch_evolve(void *stream, const lvc_modes_args *a, int kind, int tiles) {
  hipStream_t st = (hipStream_t)stream;
#define LAUNCH(KIND)                                             \
  case KIND:                                                     \
    if (a->grids)                                                \
      lvc_evolve_kernel<KIND, false><<<tiles, 64, 0, st>>>(*a);  \
    else                                                         \
      lvc_evolve_kernel<KIND, true><<<tiles, 64, 0, st>>>(*a);   \
    break
  switch (kind) {
    LAUNCH(LVC_MODES_ROW4);
    LAUNCH(LVC_MODES_ROW8);
    LAUNCH(LVC_MODES_WAVE4);
    LAUNCH(LVC_MODES_WAVE8);
    LAUNCH(LVC_MODES_WAVE16);
    default: return (int)hipErrorInvalidValue;
  }
#undef LAUNCH
  return (int)hipGetLastError();
}

int lvc_launch_price(void *stream, const lvc_modes_args *a, int n, void *out, int out_f64) {
  hipStream_t st = (hipStream_t)stream;
  const int blocks = (n + 3) / 4;
  if (a->grids && out_f64)
    lvc_price_kernel<false><<<blocks, 256, 0, st>>>(*a, n, (double *)out);
  else if (a->grids)
    lvc_price_kernel<false><<<blocks, 256, 0, st>>>(*a, n, (float *)out);
  else if (out_f64)
    lvc_price_kernel<true><<<blocks, 256, 0, st>>>(*a, n, (double *)out);
  else
    lvc_price_kernel<true><<<blocks, 256, 0, st>>>(*a, n, (float *)out);
  return (int)hipGetLastError();
}

}  // extern "C"
