// InterestCalib (finpar/InterestCalib.fut) kernels for MI355X (gfx950).
//
// The calibration evaluates, per MCMC iteration, every genome of the
// population on every swaption quote (evalGenomeOnSwap, :484-602): a G2++
// model price from three Brent root finds over the swaption's schedule and
// a Gauss-Hermite sum over it.  That work is independent per (genome,
// swaption) and bounded by the schedule length n (2..60 periods in the
// datasets), so one evaluation runs on a group of lanes holding K schedule
// periods each (K = 1, 2, 4 or 8, a template parameter; the group is a power
// of two of 1..64 lanes), a wavefront holds 64/lanes evaluations of the same
// swaption for consecutive genomes, and every sum, maximum and Brent
// iteration over the schedule is a sum over the lane's K periods followed by
// a butterfly within the group.  The butterfly hands every lane of the group
// the same bits, so a group's control flow (the root finder's branches and
// iteration counts) stays uniform within the group.  The lanes of a group are
// virtual: a physical lane stands for V = 1, 2 or 4 of them, and the sums are
// added in the butterfly's order whatever V, so every result has the same bits
// for every V.  What a group does once (the root finder's own
// arithmetic, the quadrature's terms without a period) is done by each of its
// physical lanes, so fewer of them is less work, and the host packs as far as
// enough wavefronts remain.
//
// What does not depend on the genome (dates, discount factors, the Black
// quote, each period's c_i * zc(end) / zc(maturity)) is computed once per
// call by ic_setup_kernel into per-swaption and per-period tables.  The
// log-likelihood terms land in [swaption][genome] order; ic_step_kernel sums
// them per genome in a fixed order, accepts or rejects and draws the next
// proposals, so an iteration is two launches, each spread over the device.
//
// Arithmetic is f32 in the reference's order of operations, compiled
// without contraction; expf/logf/sqrtf are the device library's, so results
// differ from a host libm in the last bits.
//
// Divisions.  An IEEE division is 11 instructions; half of the evaluation's
// were that.  rcp_rn's v_rcp_f32 and one Newton step give the correctly
// rounded reciprocal for every significand (checked over all 2^23), and
// Markstein's theorem then makes q = a r corrected by one residual step the
// correctly rounded quotient, in 7 instructions, where neither the reciprocal
// nor the residual underflows: |b| and |a / b| within 2^+-125, |a| above
// 2^-101 or 0.  v_div_fixup gives the quotients of zeros, infinities and NaN.
// With the calibration's genomes (1e-3 .. 1) the evaluation's operands are far
// inside (root finder: |f| below 600, every difference an ulp of 1 or more).
// interestcalib_eval takes any genome: where one is outside 2^-12 .. 2^4
// (ic_entry.c) the kernels divide by the operator.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "ic_internal.h"

namespace {

constexpr float kEps0 = 1.0e-3f;  // :20
constexpr float kEps = 1.0e-5f;   // :21
constexpr float kCauchyOffs = 5.0f;
constexpr float kR = 0.03f;       // :27
constexpr float kPi = 3.14159265358979323846f;

// ---- the calendar (lib/github.com/diku-dk/date/date.fut:48-150) ----------
// Integer / and % of Futhark round towards negative infinity.
__device__ inline int32_t fdiv(int32_t a, int32_t b) {
  int32_t q = a / b;
  if ((a % b != 0) && ((a < 0) != (b < 0))) q--;
  return q;
}
__device__ inline int32_t fmod_(int32_t a, int32_t b) {
  int32_t r = a % b;
  if (r != 0 && ((r < 0) != (b < 0))) r += b;
  return r;
}

constexpr int32_t kMinutesInDay = 24 * 60;
constexpr int32_t kMinutesToNoon = 12 * 60;

// minutes since the epoch of (y, m, d, hour, minute), date.fut:65-75
__device__ int32_t date_of_gregorian(int32_t y, int32_t m, int32_t d, int32_t hr, int32_t mn) {
  int32_t j;
  if (m == 1 || m == 2)
    j = fdiv(1461 * (y + 4800 - 1), 4) + fdiv(367 * (m + 10), 12) -
        fdiv(3 * fdiv(y + 4900 - 1, 100), 4);
  else
    j = fdiv(1461 * (y + 4800), 4) + fdiv(367 * (m - 2), 12) - fdiv(3 * fdiv(y + 4900, 100), 4);
  return (j + d - 32075 - 2444238) * kMinutesInDay + hr * 60 + mn;
}

__device__ int32_t end_of_month(int32_t y, int32_t m) {  // date.fut:93-100
  const bool leap = fmod_(y, 4) == 0 && (fmod_(y, 400) == 0 || fmod_(y, 100) != 0);
  if (m == 2) return leap ? 29 : 28;
  if (m == 4 || m == 6 || m == 9 || m == 11) return 30;
  return 31;
}

// add_months (date.fut:128-137) over gregorian_of_date (:77-91)
__device__ int32_t add_months(int32_t t, int32_t nbmonths) {
  const int32_t jul = fdiv(t, kMinutesInDay);
  int32_t l = jul + 68569 + 2444238;
  const int32_t n = fdiv(4 * l, 146097);
  l = l - fdiv(146097 * n + 3, 4);
  const int32_t i = fdiv(4000 * (l + 1), 1461001);
  l = l - fdiv(1461 * i, 4) + 31;
  const int32_t j = fdiv(80 * l, 2447);
  const int32_t day = l - fdiv(2447 * j, 80);
  l = fdiv(j, 11);
  const int32_t month = j + 2 - 12 * l;
  const int32_t year = 100 * (n - 49) + i + l;
  const int32_t daytime = fmod_(t, kMinutesInDay);
  int32_t hr = 12, mn = 0;
  if (daytime != kMinutesToNoon) {
    hr = fdiv(daytime, 60);
    mn = fmod_(daytime, 60);
  }
  int32_t m = month + nbmonths;
  int32_t y = year + fdiv(m - 1, 12);
  m = fmod_(m - 1, 12) + 1;
  if (m <= 0) {
    y -= 1;
    m += 12;
  }
  const int32_t eom = end_of_month(y, m);
  return date_of_gregorian(y, m, day < eom ? day : eom, hr, mn);
}

// date_act_365(t1, t2) = f32.f64 (diff_dates t2 t1) (:31, date.fut:139-143)
__device__ inline float act365(int32_t t1, int32_t t2) {
  const double inv_minutes_in_day = 1.0 / (double)kMinutesInDay;
  return (float)((double)(t1 - t2) * inv_minutes_in_day / 365.0);
}

__device__ inline int32_t today() { return date_of_gregorian(2012, 1, 1, 12, 0); }

__device__ inline float zc(int32_t t) { return expf(-kR * act365(t, today())); }  // :48

// The two forms of the divisions: by these steps where every operand is in
// range (Short), and IEEE's (Ieee).
struct Short {
  static __device__ __forceinline__ float rcp_rn(float b) {
    const float r = __builtin_amdgcn_rcpf(b);
    return fmaf(fmaf(-b, r, 1.0f), r, r);
  }
  static __device__ __forceinline__ float quot(float a, float b) {
    const float r = rcp_rn(b), q = a * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-b, q, a), r, q), b, a);
  }
  static __device__ __forceinline__ float recip(float b) {
    return __builtin_amdgcn_div_fixupf(rcp_rn(b), b, 1.0f);
  }
  // x / sqrt(2) (the divisor's correctly rounded reciprocal is a constant)
  static __device__ __forceinline__ float over_sqrt2(float x) {
    constexpr float c = 1.41421354f, r = 1.0f / c;  // sqrtf(2.0f)
    const float q = x * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-c, q, x), r, q), c, x);
  }
};
struct Ieee {
  static __device__ __forceinline__ float quot(float a, float b) { return a / b; }
  static __device__ __forceinline__ float recip(float b) { return 1.0f / b; }
  static __device__ __forceinline__ float over_sqrt2(float x) { return x / sqrtf(2.0f); }
};

// ---- the math module (:56-101) --------------------------------------------
// Abramowitz & Stegun 7.1.26 without its exp factor
template <typename D>
__device__ inline float erf_poly(float x) {
  const float p = 0.3275911f;
  const float a1 = 0.254829592f, a2 = -0.284496736f, a3 = 1.421413741f, a4 = -1.453152027f,
              a5 = 1.061405429f;
  const float t = D::recip(1.0f + p * x);
  const float t2 = t * t;
  const float t3 = t * t2;
  const float t4 = t2 * t2;
  const float t5 = t2 * t3;
  return a1 * t + a2 * t2 + a3 * t3 + a4 * t4 + a5 * t5;
}

template <typename D>
__device__ inline float ugaussian_P(float x) {  // :60-93
  const float u = D::over_sqrt2(x);
  const float e = u < 0.0f ? -(1.0f - erf_poly<D>(-u) * expf(-(u * u)))
                           : 1.0f - erf_poly<D>(u) * expf(-(u * u));
  return 0.5f * (1.0f + e);
}

template <typename D>
__device__ inline float ugaussian_P_exp(float x, float exp_factor) {  // :95-101
  const float u = fabsf(D::over_sqrt2(x));
  const float e = erf_poly<D>(u);
  const float res = 0.5f * e * expf(exp_factor - u * u);
  return 0.0f <= x ? expf(exp_factor) - res : res;
}

template <typename D>
__device__ inline float log_likelihood(float y_ref, float y) {  // Cauchy, :606-625
  const float gamma = (fabsf(y_ref) / 50.0f) * kCauchyOffs + 0.01f;
  const float x = D::quot(y - y_ref, gamma);
  const float pdf = D::recip(kPi * gamma * (1.0f + x * x));
  return logf(pdf + 1.0e-20f);
}

// ---- Sobol numbers (:190-202) ------------------------------------------------
// Unrolled over the largest vector so the direction numbers load once, up
// front, rather than one scalar load and wait per bit.
__device__ inline float sobol(const ic_dirvec &dv, int32_t n) {
  const float norm_fact = 1.0f / ((float)((int64_t)1 << dv.bits) + 1.0f);
  const int32_t n_gray = (n >> 1) ^ n;
  int32_t res = 0;
#pragma unroll
  for (int i = 0; i < IC_MAX_BITS; i++) {
    const int32_t t = (int32_t)(1u << i);
    if (i < dv.bits && (n_gray & t) == t) res ^= dv.dir[i];
  }
  return (float)res * norm_fact;
}

// ---- genomes (:220-320) -------------------------------------------------------
__device__ inline float gene_min(int j) { return j == 2 ? kEps0 - 1.0f : kEps0; }
__device__ inline float gene_max(int j) { return j < 3 ? 1.0f - kEps0 : 0.2f; }
constexpr float kAmplRatio = 0.005f;  // moves_unif_ampl_ratio, :248

// ---- G2++ (:322-413) -------------------------------------------------------------
template <typename D>
__device__ inline float b_fun(float z, float tau) {
  return D::quot(1.0f - expf(-z * tau), z);
}

template <typename D>
__device__ inline float t_fun(float sigma, float x, float tau) {
  const float expxtau = expf(-x * tau);
  const float exp2xtau = expxtau * expxtau;
  return D::quot(sigma * sigma, x * x) *
         (tau + D::quot(2.0f, x) * expxtau - D::recip(2.0f * x) * exp2xtau - D::quot(3.0f, 2.0f * x));
}

struct Genome {
  float a, b, rho, nu, sigma;
};

// bigv (:336-352): V(tau) and B_a(tau), B_b(tau)
template <typename D>
__device__ inline float bigv(const Genome &g, float tau, float *ba, float *bb) {
  const float sigma = g.sigma == 0.0f ? 1.0e-10f : g.sigma;
  *ba = b_fun<D>(g.a, tau);
  *bb = b_fun<D>(g.b, tau);
  const float t1 = t_fun<D>(sigma, g.a, tau);
  const float t2 = t_fun<D>(g.nu, g.b, tau);
  const float t3 = D::quot(2.0f * g.rho * g.nu * sigma, g.a * g.b) *
                   (tau - *ba - *bb + b_fun<D>(g.a + g.b, tau));
  return t1 + t2 + t3;
}

// bigmx / bigmy (:364-413) over (today, maturity, today, maturity): ts =
// tmat0 = tmats = t0, tmatt = s0 = 0
template <typename D>
__device__ inline float bigmx(const Genome &g, float tmat0) {
  const float a = g.a, b = g.b, rho = g.rho, nu = g.nu, sigma = g.sigma;
  const float ts = tmat0, tmatt = 0.0f, tmats = tmat0, t0 = tmat0, s0 = 0.0f;
  const float tmp1 = D::quot(sigma * sigma, a * a) + D::quot(sigma * rho * nu, a * b);
  const float tmp2 = 1.0f - expf(-a * ts);
  const float tmp3 = D::quot(sigma * sigma, 2.0f * a * a);
  const float tmp4 = D::quot(rho * sigma * nu, b * (a + b));
  const float tmp5 = expf(-a * tmatt) - expf(-a * (tmats + ts));
  const float tmp6 = expf(-b * tmatt) - expf(-b * tmat0 - a * t0 + (a + b) * s0);
  return tmp1 * tmp2 - (tmp3 * tmp5) - (tmp4 * tmp6);
}

template <typename D>
__device__ inline float bigmy(const Genome &g, float tmat0) {
  const float a = g.a, b = g.b, rho = g.rho, nu = g.nu, sigma = g.sigma;
  const float ts = tmat0, tmatt = 0.0f, tmats = tmat0, t0 = tmat0, s0 = 0.0f;
  const float tmp1 = D::quot(nu * nu, b * b) + D::quot(sigma * rho * nu, a * b);
  const float tmp2 = 1.0f - expf(-b * ts);
  const float tmp3 = D::quot(nu * nu, 2.0f * b * b);
  const float tmp4 = D::quot(sigma * rho * nu, a * (a + b));
  const float tmp5 = expf(-b * tmatt) - expf(-b * (tmats + ts));
  const float tmp6 = expf(-a * tmatt) - expf(-a * tmat0 - b * t0 + (a + b) * s0);
  return tmp1 * tmp2 - (tmp3 * tmp5) - (tmp4 * tmp6);
}

// ---- group reductions ---------------------------------------------------------------
// Butterflies over the `lanes` physical lanes of an evaluation group (a power
// of two, wave-uniform); every lane of the group ends with the same bits.
// Level m adds the lane j ^ m; the levels before it have left the same value
// in m lanes each, so any lane of the partner's block does: mirrors within 8
// and 16 lanes, row and half swaps past that, all VALU operands (the
// ds_bpermute form waited for LDS at each level).
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <typename Op>
__device__ __forceinline__ float group_all(float v, int lanes, Op op) {
  if (lanes >= 2) v = op(v, dpp<0xB1>(v));   // quad_perm [1,0,3,2]
  if (lanes >= 4) v = op(v, dpp<0x4E>(v));   // quad_perm [2,3,0,1]
  if (lanes >= 8) v = op(v, dpp<0x141>(v));  // row_half_mirror
  if (lanes >= 16) v = op(v, dpp<0x140>(v)); // row_mirror
  if (lanes >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  if (lanes >= 64) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  return v;
}
__device__ __forceinline__ float group_max(float v, int lanes) {
  return group_all(v, lanes, [](float a, float b) { return fmaxf(a, b); });
}
// The sum over the group of the V virtual lanes' sums on each lane, virtual
// lane j + lanes * v on lane j: the physical lanes are the butterfly's first
// levels, each v by itself, then the v.
template <int V>
__device__ __forceinline__ float group_sum(const float (&s)[V], int lanes) {
  float t[V];
#pragma unroll
  for (int v = 0; v < V; v++) t[v] = group_all(s[v], lanes, [](float a, float b) { return a + b; });
  if constexpr (V == 1) return t[0];
  if constexpr (V == 2) return t[0] + t[1];
  if constexpr (V == 4) return (t[0] + t[1]) + (t[2] + t[3]);
}

// One lane's schedule periods (K for each of its V virtual lanes) and their
// genome-dependent values.
template <int K, int V>
struct Periods {
  float bai[K * V], bbi[K * V], aici[K * V], log_aici[K * V], scale[K * V], t1cs[K * V], cs[K * V];
  bool valid[K * V];
  int32_t n;  // the slots whose first period (slot0) is below n hold any: wave-uniform
  int32_t slot0[K * V];
};

// expf(x) for |x| < 87 by the device library's method, so as to have its bits:
// the exponent's integer part and the rest of x log2(e), its product in two
// parts, by v_exp_f32; without the range handling, a third of the instructions.  Equal to expf for every float of
// that range (compared over all of them).
__device__ __forceinline__ float exp_mid(float x) {
  constexpr float c = 0x1.715476p+0f, cc = 0x1.4ae0bep-26f;  // log2(e)
  const float t = x * c, n = __builtin_rintf(t);
  const float r = (t - n) + fmaf(x, cc, fmaf(x, c, -t));
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(r), (int)n);
}

// sum over the group of scales * exp(-bbi * y), minus 1 (:108-117, fid 1).
// MID: every |bbi * y| is below 87.
template <bool MID, int K, int V>
__device__ __forceinline__ float to_solve(const Periods<K, V> &P, const float (&ups)[K * V],
                                          float y, int lanes) {
  float s[V];
#pragma unroll
  for (int v = 0; v < V; v++) {
    s[v] = 0.0f;
#pragma unroll
    for (int k = 0; k < K; k++) {
      if (P.slot0[v * K + k] >= P.n) continue;
      const float x = -P.bbi[v * K + k] * y;
      const float t = ups[v * K + k] * (MID ? exp_mid(x) : expf(x));
      s[v] += P.valid[v * K + k] ? t : 0.0f;
    }
  }
  return group_sum<V>(s, lanes) - 1.0f;
}

// rootFinding_Brent (:124-185); the loop ends where the reference's
// iterations stop changing its state
template <typename D, bool MID, int K, int V>
__device__ float brent(const Periods<K, V> &P, const float (&ups)[K * V], int lanes, float lb, float ub,
                       float tol, int32_t iter_max, float *err) {
  tol = tol <= 0.0f ? 1.0e-9f : tol;
  iter_max = iter_max <= 0 ? 10000 : iter_max;
  float a = lb, b = ub;
  float fa = to_solve<MID>(P, ups, a, lanes), fb = to_solve<MID>(P, ups, b, lanes);
  if (0.0f <= fa * fb) {
    *err = 0.0f <= a ? INFINITY : -INFINITY;
    return 0.0f;
  }
  if (fabsf(fa) < fabsf(fb)) {
    float t = fa; fa = fb; fb = t;
    t = a; a = b; b = t;
  }
  // x: |b - c| after a bisection, |c - d| after an interpolation
  float c = a, fc = fa, x = fabsf(b - c);
  for (int32_t i = 0; i < iter_max; i++) {
    if (fb == 0.0f || fabsf(b - a) < tol) break;
    float s;
    if (fa == fc || fb == fc) {
      s = b - D::quot(fb * (b - a), fb - fa);
    } else {
      // each difference once: negation is exact
      const float ab = fa - fb, ac = fa - fc, bc = fb - fc;
      const float s1 = D::quot(a * fb * fc, ab * ac);
      const float s2 = D::quot(b * fa * fc, -ab * bc);
      const float s3 = D::quot(c * fa * fb, ac * bc);
      s = s1 + s2 + s3;
    }
    const bool bisect = !((3.0f * a + b) / 4.0f <= s && s <= b) || x / 2.0f <= fabsf(s - b) ||
                        x <= fabsf(tol);
    s = bisect ? (a + b) / 2.0f : s;
    const float fs = to_solve<MID>(P, ups, s, lanes);
    const float was_c = c;
    c = b;
    fc = fb;
    const bool left = fa * fs < 0.0f;
    b = left ? s : b;
    fb = left ? fs : fb;
    a = left ? a : s;
    fa = left ? fa : fs;
    const bool swap = fabsf(fa) < fabsf(fb);
    const float t = a, ft = fa;
    a = swap ? b : a;
    fa = swap ? fb : fa;
    b = swap ? t : b;
    fb = swap ? ft : fb;
    x = fabsf(bisect ? b - c : c - was_c);
  }
  *err = fb;
  return b;
}

struct Scals {
  float b, sigmax, sigmay, rhoxy, rhoxyc, rhoxycs, mux, muy, bb_first, bb_last;
};

// exactYhat (:418-481); bb_first and bb_last are bbi[0] and bbi[n-1]
template <typename D, int K, int V>
__device__ float exact_yhat(const Periods<K, V> &P, int n, int lanes, const Scals &sc, float x) {
  const float k = -3.71901648545568f;
  float ups[K * V], part[V], lo = -INFINITY;
#pragma unroll
  for (int v = 0; v < V; v++) {
    part[v] = 0.0f;
#pragma unroll
    for (int q = v * K; q < (v + 1) * K; q++) {
      ups[q] = 0.0f;
      if (P.slot0[q] >= P.n) continue;
      if (P.valid[q]) {
        const float baix = P.bai[q] * x;
        ups[q] = P.aici[q] * expf(-baix);
        part[v] += ups[q];
        lo = fmaxf(lo, D::quot(P.log_aici[q] - baix, P.bbi[q]));
      }
    }
  }
  const float up = group_sum<V>(part, lanes);
  lo = group_max(lo, lanes);
  if (n < 2) return lo;
  const float log_s = logf(up);
  float tmp = D::quot(log_s, sc.bb_last);
  if (!(tmp <= 0.0f)) {
    tmp = D::quot(log_s, sc.bb_first);
    tmp = 0.0f <= tmp ? tmp : -INFINITY;
  }
  const float yl = lo - kEps, yu = tmp + kEps;
  const float rx = D::quot(sc.rhoxy * (x - sc.mux), sc.sigmax);
  const float y0 = sc.sigmay * (rx + k * sc.rhoxycs) - D::quot(sc.rhoxyc, sc.b) + sc.muy;
  const float y1 = sc.sigmay * (rx - k * sc.rhoxycs) + sc.muy;
  if (y1 <= yl) return y1 + 1.0f;
  if (yu <= y0) return y0 - 1.0f;
  const float ya = fmaxf(yl, y0), yb = fminf(yu, y1);
  // every iterate lies between the two, so the wavefront knows its range of
  // exponents (a NaN is in none)
  float bb = 0.0f;
#pragma unroll
  for (int q = 0; q < K * V; q++) bb = fmaxf(bb, P.bbi[q]);
  float err, root;
  if (__ballot(!(bb * fabsf(ya) < 86.0f && bb * fabsf(yb) < 86.0f)) == 0)
    root = brent<D, true>(P, ups, lanes, ya, yb, 1.0e-4f, 1000, &err);
  else
    root = brent<D, false>(P, ups, lanes, ya, yb, 1.0e-4f, 1000, &err);
  if (err == -INFINITY) return y0 - 1.0f;
  if (err == INFINITY) return y1 + 1.0f;
  return root;
}

}  // namespace

// ---- per-call setup: what does not depend on the genome (:486-525, :533-547)
// One workgroup per swaption, its periods spread over the threads; the
// quote's level is summed in period order by one thread, as the reference's
// sequential reduction.
constexpr int kSetupThreads = 64;

__global__ __launch_bounds__(kSetupThreads) void ic_setup_kernel(
    const float *__restrict__ swp, int64_t stride, int32_t nswap, ic_swaption *__restrict__ sw,
    ic_period *__restrict__ per) {
  __shared__ float a12s[IC_MAX_PERIODS];
  __shared__ int32_t a1s[IC_MAX_PERIODS], a2s[IC_MAX_PERIODS];
  __shared__ float strike_sh;
  const int32_t s = blockIdx.x;
  if (s >= nswap) return;
  const float *row = swp + (int64_t)s * stride;
  const ic_swaption S0 = sw[s];
  const int32_t n = S0.n;
  const int32_t t_today = today();
  const float swap_freq = row[1];
  const int32_t maturity = add_months(t_today, (int32_t)(row[0] * 12.0f));  // add_years, :33
  const float tmat0 = act365(maturity, t_today);
  for (int32_t i = threadIdx.x; i < n; i += kSetupThreads) {
    const int32_t a1 = add_months(maturity, (int32_t)(swap_freq * (float)(int64_t)i));
    const int32_t a2 = add_months(a1, (int32_t)swap_freq);
    a1s[i] = a1;
    a2s[i] = a2;
    a12s[i] = zc(a2) * act365(a2, a1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float lvl = 0.0f;
    int32_t t0 = date_of_gregorian(2229, 12, 31, 12, 0), tn = date_of_gregorian(1980, 1, 1, 12, 0);
    for (int32_t i = 0; i < n; i++) {
      lvl = lvl + a12s[i];
      t0 = t0 < a1s[i] ? t0 : a1s[i];
      tn = tn > a2s[i] ? tn : a2s[i];
    }
    const float strike = (zc(t0) - zc(tn)) / lvl;
    const float d1 = 0.5f * row[3] * tmat0;
    ic_swaption S = S0;
    S.quote = lvl * strike * (ugaussian_P<Ieee>(d1) - ugaussian_P<Ieee>(-d1));
    S.tmat0 = tmat0;
    S.zc_mat = zc(maturity);
    sw[s] = S;
    strike_sh = strike;
  }
  __syncthreads();
  const float strike = strike_sh;
  const float zc_mat = zc(maturity);
  for (int32_t i = threadIdx.x; i < n; i += kSetupThreads) {
    const int32_t beg = a1s[i], end = a2s[i];  // the same dates as the quote's (:533-536)
    const float res = act365(end, beg) * strike;
    const float cii = i == n - 1 ? 1.0f + res : res;
    ic_period p;
    p.tod1 = act365(end, t_today);
    p.tod2 = act365(end, maturity);
    p.fact = cii * zc(end) / zc_mat;
    p.log_fact = logf(p.fact);
    per[S0.off + i] = p;
  }
}

__global__ void ic_init_kernel(int32_t pop, ic_dirvec dv, float *__restrict__ genomes,
                               float *__restrict__ props) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= pop) return;
  for (int j = 0; j < 5; j++) {  // initGenome (:233-238) of sobolInd at 5i+1 .. 5i+5
    const float r01 = sobol(dv, 5 * i + 1 + j);
    const float g = r01 * (gene_max(j) - gene_min(j)) + gene_min(j);
    genomes[5 * i + j] = g;
    props[5 * i + j] = g;
  }
}

// ---- the evaluation ------------------------------------------------------------------
struct EvalArgs {
  const ic_swaption *sw;
  const ic_period *per;
  const ic_work *work;
  int32_t nwork;
  const float *genomes;
  int32_t npop;
  const float *hx, *hw;
  int32_t nherm, nswap, mode;
  float *out0, *out1;
};

// One wavefront's evaluations, K schedule periods for each of a lane's V
// virtual lanes: period jv + S.lanes * k for virtual lane jv = j + lanes * v.
// (With neighbouring virtual lanes on one physical lane the sums are shorter,
// but a schedule of 20 periods on 16 lanes of 2 then keeps 8 slots busy for
// lane 0's sake, where this needs 5.)
template <typename D, int K, int V>
__device__ __forceinline__ void eval_wave(const EvalArgs &A, const ic_work wk, const ic_swaption S,
                                          const int lane) {
  const int lanes = S.lanes / V;  // physical lanes of a group
  const int n = S.n;
  const int j = lane & (lanes - 1), group0 = lane & ~(lanes - 1);
  int32_t gi = wk.genome0 + lane / lanes;
  const bool store = gi < A.npop && j == 0;
  gi = gi < A.npop ? gi : A.npop - 1;
  const Genome g = {A.genomes[5 * gi], A.genomes[5 * gi + 1], A.genomes[5 * gi + 2],
                    A.genomes[5 * gi + 3], A.genomes[5 * gi + 4]};
  const float tmat0 = S.tmat0;

  // :528-546
  float dum1, dum2;
  const float v0_mat = bigv<D>(g, tmat0, &dum1, &dum2);
  const float mux = 0.0f - bigmx<D>(g, tmat0);
  const float muy = 0.0f - bigmy<D>(g, tmat0);
  const float sqrt_bfun_a = sqrtf(b_fun<D>(2.0f * g.a, tmat0));
  const float sqrt_bfun_b = sqrtf(b_fun<D>(2.0f * g.b, tmat0));
  const float rhoxy = D::quot(g.rho * b_fun<D>(g.a + g.b, tmat0), sqrt_bfun_a * sqrt_bfun_b);
  const float sigmax = g.sigma * sqrt_bfun_a;
  const float sigmay = g.nu * sqrt_bfun_b;
  const float rhoxyc = 1.0f - rhoxy * rhoxy;
  const float rhoxycs = sqrtf(rhoxyc);
  const float sigmay_rhoxycs = sigmay * rhoxycs;
  const float t4 = D::quot(rhoxy * sigmay, sigmax);

  // the schedule's periods (:549-583)
  Periods<K, V> P;
  P.n = n;
#pragma unroll
  for (int q = 0; q < K * V; q++) {
    P.slot0[q] = lanes * (q / K) + S.lanes * (q % K);
    const int i = P.slot0[q] + j;
    P.valid[q] = i < n;
    P.bai[q] = P.bbi[q] = P.aici[q] = P.log_aici[q] = P.scale[q] = P.t1cs[q] = P.cs[q] = 0.0f;
    if (P.valid[q]) {
      const ic_period pe = A.per[S.off + i];
      float bai, bbi;
      const float v0_end = bigv<D>(g, pe.tod1, &dum1, &dum2);
      const float vt_end = bigv<D>(g, pe.tod2, &bai, &bbi);
      const float expo_aici = 0.5f * (vt_end - v0_end + v0_mat);
      P.bai[q] = bai;
      P.bbi[q] = bbi;
      P.aici[q] = pe.fact * expf(expo_aici);
      P.log_aici[q] = pe.log_fact + expo_aici;
      P.scale[q] = 0.0f - (bai + bbi * t4);
      P.cs[q] = pe.fact;
      P.t1cs[q] = bbi * (mux * t4 - (muy - 0.5f * rhoxyc * sigmay * sigmay * bbi)) + expo_aici;
    }
  }
  Scals sc;
  sc.b = g.b;
  sc.sigmax = sigmax;
  sc.sigmay = sigmay;
  sc.rhoxy = rhoxy;
  sc.rhoxyc = rhoxyc;
  sc.rhoxycs = rhoxycs;
  sc.mux = mux;
  sc.muy = muy;
  sc.bb_first = n > 0 ? b_fun<D>(g.b, A.per[S.off].tod2) : 0.0f;
  sc.bb_last = n > 0 ? b_fun<D>(g.b, A.per[S.off + n - 1].tod2) : 0.0f;

  // :586-591
  const float eps = 0.5f * sigmax;
  // one copy of the root search for the three: a launch's wavefronts run four
  // instantiations of this function, which have to share the instruction cache
  float f = 0.0f, gg = 0.0f, h = 0.0f;
#pragma unroll 1
  for (int r = 0; r < 3; r++) {
    const float x = r == 0 ? mux : r == 1 ? mux + eps : mux - eps;
    const float y = exact_yhat<D>(P, n, lanes, sc, x);
    f = r == 0 ? y : f;
    gg = r == 1 ? y : gg;
    h = r == 2 ? y : h;
  }
  const float df = D::quot(0.5f * (gg - h), eps);
  const float sqrt2sigmax = sqrtf(2.0f) * sigmax;
  const float t2 = D::quot(rhoxy, sigmax * rhoxycs);

  // Gauss-Hermite (:594-620).  A point's terms without a period, h1 and
  // P(-h1), are made by one lane of the group each, `lanes` points at a time,
  // and its weight by one lane of the wavefront, 64 points at a time.
  float accum = 0.0f;
  for (int q64 = 0; q64 < A.nherm; q64 += 64) {
    const int end64 = A.nherm - q64 < 64 ? A.nherm - q64 : 64;
    const int mine = q64 + (lane < end64 ? lane : 0);
    const float hx = A.hx[mine];
    const float tmp = sqrtf(2.0f) * hx;
    const float hw = A.hw[mine] * expf(-0.5f * tmp * tmp);
    for (int q0 = 0; q0 < end64; q0 += lanes) {
      float own_h1, own_p;
      {
        const float x = sqrt2sigmax * __shfl(hx, q0 + j) + mux;
        const float yhat_x = f + df * (x - mux);
        own_h1 = D::quot(yhat_x - muy, sigmay_rhoxycs) - t2 * (x - mux);
        own_p = ugaussian_P<D>(-own_h1);
      }
      const int here = end64 - q0 < lanes ? end64 - q0 : lanes;
      for (int t = 0; t < here; t++) {
        const float h1 = __shfl(own_h1, group0 + t), p1 = __shfl(own_p, group0 + t);
        const float x_quad = __int_as_float(
            __builtin_amdgcn_readlane(__float_as_int(hx), q0 + t));
        const float w_t1 = __int_as_float(
            __builtin_amdgcn_readlane(__float_as_int(hw), q0 + t));
        const float x = sqrt2sigmax * x_quad + mux;
        float part[V];
#pragma unroll
        for (int v = 0; v < V; v++) {
          part[v] = 0.0f;
#pragma unroll
          for (int q = v * K; q < (v + 1) * K; q++) {
            if (P.slot0[q] >= n) continue;
            const float h2 = h1 + P.bbi[q] * sigmay_rhoxycs;
            const float expo_aici = P.t1cs[q] + P.scale[q] * x;
            const float term = P.cs[q] * ugaussian_P_exp<D>(-h2, expo_aici);
            part[v] += P.valid[q] ? term : 0.0f;
          }
        }
        accum = accum + w_t1 * (p1 - group_sum<V>(part, lanes));
      }
    }
  }
  const float price = S.zc_mat * (accum / sqrtf(kPi));
  if (!store) return;
  const int32_t s = wk.swaption;
  if (A.mode == IC_OUT_TERMS) {
    A.out0[(int64_t)s * A.npop + gi] = log_likelihood<D>(S.quote, price);
  } else if (A.mode == IC_OUT_PRICES) {
    A.out0[(int64_t)gi * A.nswap + s] = S.quote;
    A.out1[(int64_t)gi * A.nswap + s] = price;
  } else {  // makeSummary (:205-213)
    const float err_ratio = (price - S.quote) / S.quote;
    A.out0[3 * s] = 10000.0f * price;
    A.out0[3 * s + 1] = 10000.0f * S.quote;
    A.out0[3 * s + 2] = 100.0f * fabsf(err_ratio);
  }
}

// Swaptions of 1 or 2 periods a virtual lane (up to 128 periods) in one
// launch, so the classes share the device; a class is uniform per wavefront.
template <typename D>
__global__ __launch_bounds__(256) void ic_eval_kernel(EvalArgs A) {
  const int32_t wv = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (wv >= A.nwork) return;  // wave-uniform
  const ic_work wk = A.work[wv];
  const ic_swaption S = A.sw[wk.swaption];
  const int lane = threadIdx.x & 63;
  if (S.per_lane == 1)
    eval_wave<D, 1, 1>(A, wk, S, lane);
  else if (wk.pack == 1)
    eval_wave<D, 2, 1>(A, wk, S, lane);
  else if (wk.pack == 2)
    eval_wave<D, 2, 2>(A, wk, S, lane);
  else
    eval_wave<D, 2, 4>(A, wk, S, lane);
}

// Longer schedules (4 or 8 periods a lane, up to 512 periods): more registers.
template <typename D>
__global__ __launch_bounds__(256) void ic_eval_long_kernel(EvalArgs A) {
  const int32_t wv = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (wv >= A.nwork) return;
  const ic_work wk = A.work[wv];
  const ic_swaption S = A.sw[wk.swaption];
  if (S.per_lane == 4)
    eval_wave<D, 4, 1>(A, wk, S, threadIdx.x & 63);
  else
    eval_wave<D, 8, 1>(A, wk, S, threadIdx.x & 63);
}

// ---- accept / propose ------------------------------------------------------------------
struct StepArgs {
  int32_t pop, nswap;
  const float *terms;
  ic_state from, to;
  int32_t init, acc, it, conv;
  ic_move next;
  ic_dirvec dv;
  ic_trace trace;
};

constexpr int kSumLanes = 32;  // threads per genome of the step kernel

// The log-likelihoods (:639-645) of N genomes ids[]: 32 lanes per genome, lane
// t summing the swaptions t, t + 32, ... in order, the 32 partial sums added
// pairwise with the same bits on every lane.  Eight terms of every genome are
// loaded before their sums (a lane has ceil(nswap / 32) terms: 7 for 196
// swaptions, so one memory round trip).
template <int N>
__device__ __forceinline__ void loglik_sums(const StepArgs &A, const int32_t (&ids)[N], int t,
                                            float (&s)[N]) {
#pragma unroll
  for (int m = 0; m < N; m++) s[m] = 0.0f;
  for (int32_t w = t; w < A.nswap; w += 8 * kSumLanes) {
    float v[N][8];
#pragma unroll
    for (int m = 0; m < N; m++)
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int32_t wk = w + k * kSumLanes;
        v[m][k] = wk < A.nswap ? A.terms[(int64_t)wk * A.pop + ids[m]] : 0.0f;
      }
#pragma unroll
    for (int m = 0; m < N; m++)
#pragma unroll
      for (int k = 0; k < 8; k++)
        if (w + k * kSumLanes < A.nswap) s[m] += v[m][k];
  }
#pragma unroll
  for (int m = 0; m < N; m++)
    for (int b = 1; b < kSumLanes; b <<= 1) s[m] += __shfl_xor(s[m], b, 64);
}

// What the step reads of a genome, gene j: all of it asked for beside the terms,
// not after the sums and again after the decision (three memory round trips
// of a launch that is little else: 8.9 us, and 8.2 with one).
struct Member {
  float loglik, fb, gene, prop;
};
__device__ __forceinline__ Member read_member(const StepArgs &A, int32_t i, int j) {
  return {A.from.logliks[i], A.from.fb[i], A.from.genomes[5 * i + j], A.from.props[5 * i + j]};
}

// Whether the genome's proposal, of log-likelihood s, is accepted on its draw
// (:733-745).
__device__ __forceinline__ bool accepted(const Member &g, float s, float draw) {
  return draw < fminf(1.0f, expf(s - g.loglik) * g.fb);
}

// One step of the population: each genome's log-likelihood and acceptance,
// then its next proposal (:655-724), 32 lanes per genome, a lane per gene.
// Differential evolution reads two other genomes after their accept steps;
// their log-likelihoods are summed here again, so that no second launch has
// to wait for all of the first (which took 6 us of an iteration).  The old
// state is only read and the new one only written: nothing races.
__global__ __launch_bounds__(256) void ic_step_kernel(StepArgs A) {
  const int32_t pop = A.pop;
  const int t = threadIdx.x & (kSumLanes - 1);
  const int32_t at = (int32_t)(blockIdx.x * (256 / kSumLanes) + threadIdx.x / kSumLanes);
  const int32_t i = at < pop ? at : pop - 1;  // spare lanes follow the last genome
  const ic_move mv = A.next;
  const bool de = mv.type == 3;
  // DE's genomes k and l and its gamma (:700-712)
  int32_t k = i, l = i;
  float gamma1 = 0.0f;
  const int32_t kk = 8 * i + mv.base;
  // The genome's Sobol numbers, a lane each (one after the other they were seven
  // chains of 31 bits in DE's step, 8.2 us, and 6.4 with two): the genes' in
  // lanes 0 .. 4, the accept step's, then DE's three.
  const int first = threadIdx.x & 63 & ~(kSumLanes - 1);
  const float draws =
      sobol(A.dv, t < 5 ? (de ? kk + 3 : 5 * i + mv.base) + t : t == 5 ? A.acc + i : kk + t - 6);
  const float draw = __shfl(draws, first + 5), s1 = __shfl(draws, first + 6);
  const float s2 = __shfl(draws, first + 7), s3 = __shfl(draws, first + 8);
  if (de) {
    k = (int32_t)(s1 * (float)(pop - 1));
    int32_t cand_ub = pop - 1;
    if (k == i) {
      k = pop - 1;
      cand_ub = pop - 2;
    }
    l = (int32_t)(s2 * (float)cand_ub);
    if (l == i || l == k) l = cand_ub;
    const float gamma_avg = 2.38f / sqrtf(2.0f * 5.0f);
    gamma1 = gamma_avg - 0.5f + s3;
  }
  const int j = t < 5 ? t : 0;  // this lane's gene
  const Member own = read_member(A, i, j);
  float s, gene_k = 0.0f, gene_l = 0.0f;
  bool take = false;
  if (de) {
    const Member gk = read_member(A, k, j), gl = read_member(A, l, j);
    const float theirs = sobol(A.dv, A.acc + (t & 1 ? l : k));
    const float draw_k = __shfl(theirs, first), draw_l = __shfl(theirs, first + 1);
    const int32_t ids[3] = {i, k, l};
    float sums[3];
    loglik_sums<3>(A, ids, t, sums);
    s = sums[0];
    take = !A.init && accepted(own, s, draw);
    gene_k = !A.init && accepted(gk, sums[1], draw_k) ? gk.prop : gk.gene;
    gene_l = !A.init && accepted(gl, sums[2], draw_l) ? gl.prop : gl.gene;
  } else {
    const int32_t ids[1] = {i};
    float sums[1];
    loglik_sums<1>(A, ids, t, sums);
    s = sums[0];
    take = !A.init && accepted(own, s, draw);
  }
  const float gene = take ? own.prop : own.gene;
  const float loglik = A.init || take ? s : own.loglik;
  float out = 0.0f, bf = 1.0f;
  if (mv.type == 1 || mv.type == 2) {  // mutate_dims_all / mutate_dims_one (:278-306)
    const float r01 = draws;
    const float ampl = mv.type == 1 || j == mv.dim ? kAmplRatio : 0.0f;
    const float g_min = gene_min(j), g_max = gene_max(j);
    const float prop = own.prop;
    const float amplitude = fabsf((g_max - g_min) * ampl);  // mutateHelper, :250-266
    const float semiamplitude = amplitude / 2.0f;
    float tmp_min_max = fminf(g_max, gene + semiamplitude);
    float tmp_max_min = fmaxf(g_min, gene - semiamplitude);
    const float forward_range = tmp_min_max - tmp_max_min;
    tmp_min_max = fminf(g_max, prop + semiamplitude);
    tmp_max_min = fmaxf(g_min, prop - semiamplitude);
    const float backward_range = tmp_min_max - tmp_max_min;
    bf = 0.0f < semiamplitude ? backward_range / forward_range : 1.0f;
    const float ng = gene + amplitude * r01 - semiamplitude;
    out = fmaxf(g_min, fminf(g_max, ng));  // constrainDim, :268-270
  } else if (de) {  // :713-723, mcmc_DE :309-320
    const float ampl_ratio = 0.1f * kAmplRatio;
    const float r01 = draws;
    const float mm_diff = gene_max(j) - gene_min(j);
    const float amplitude = fabsf(mm_diff * ampl_ratio);
    const float semiamplitude = amplitude / 2.0f;
    const float perturb = amplitude * r01 - semiamplitude;
    const float ng = gene + perturb + gamma1 * (gene_k - gene_l);
    out = fmaxf(gene_min(j), fminf(gene_max(j), ng));
  }
  // the genes' ratios multiplied in order
  float fb = __shfl(bf, first);
  for (int m = 1; m < 5; m++) fb = fb * __shfl(bf, first + m);
  if (at >= pop) return;
  const int64_t row = (int64_t)(A.it + 1) * pop + i;
  if (t < 5) {
    A.to.genomes[5 * i + j] = gene;
    if (mv.type) A.to.props[5 * i + j] = out;
    if (A.trace.genomes) A.trace.genomes[5 * row + j] = gene;
    if (mv.type && A.trace.props && A.it + 1 < A.conv) A.trace.props[5 * row + j] = out;
  }
  if (t == 0) {
    A.to.logliks[i] = loglik;
    if (mv.type) A.to.fb[i] = fb;
    if (A.trace.newl && !A.init) A.trace.newl[(int64_t)A.it * pop + i] = s;
    if (A.trace.genomes) A.trace.logliks[row] = loglik;
    if (mv.type && A.trace.props && A.it + 1 < A.conv) A.trace.fb[row] = fb;
  }
}

// The winner (:752-756): the reduction read as a left fold, so the first of the
// largest log-likelihoods (a NaN is never one, and genome 0 wins where nothing
// is above -inf).  One workgroup: a lane folds its genomes in order, the lanes
// are joined by value, then by the smaller index.  (One thread over them all
// was 17.6 us at 256 genomes, 4.6 now.)
constexpr int kWinnerThreads = 256;
__global__ __launch_bounds__(kWinnerThreads) void ic_winner_kernel(
    int32_t pop, const float *__restrict__ genomes, const float *__restrict__ logliks,
    float *__restrict__ out, float *__restrict__ winner) {
  __shared__ float values[kWinnerThreads / 64];
  __shared__ int32_t indexes[kWinnerThreads / 64];
  const int t = threadIdx.x;
  int32_t wi = 0;
  float wv = -INFINITY;
  for (int32_t i = t; i < pop; i += kWinnerThreads) {
    const float v = logliks[i];
    if (wv < v) {
      wi = i;
      wv = v;
    }
  }
  auto join = [&](float v, int32_t i) {
    if (wv < v || (wv == v && i < wi)) {
      wi = i;
      wv = v;
    }
  };
#pragma unroll
  for (int b = 1; b < 64; b <<= 1) join(__shfl_xor(wv, b), __shfl_xor(wi, b));
  if ((t & 63) == 0) {
    values[t >> 6] = wv;
    indexes[t >> 6] = wi;
  }
  __syncthreads();
  if (t != 0) return;
#pragma unroll
  for (int k = 1; k < kWinnerThreads / 64; k++) join(values[k], indexes[k]);
  const float *w = genomes + 5 * wi;
  out[0] = w[0];
  out[1] = w[1];
  out[2] = w[4];
  out[3] = w[3];
  out[4] = w[2];
  out[5] = wv;
  for (int j = 0; j < 5; j++) winner[j] = w[j];
}

// ---- launchers ---------------------------------------------------------------------------
extern "C" int ic_launch_setup(void *stream, const float *swaptions, int64_t stride,
                               int32_t nswap, ic_swaption *sw, ic_period *periods) {
  if (nswap <= 0) return 0;
  hipLaunchKernelGGL(ic_setup_kernel, dim3(nswap), dim3(kSetupThreads), 0, (hipStream_t)stream,
                     swaptions, stride, nswap, sw, periods);
  return (int)hipGetLastError();
}

extern "C" int ic_launch_init(void *stream, int32_t pop, const ic_dirvec *dv, float *genomes,
                              float *props) {
  if (pop <= 0) return 0;
  hipLaunchKernelGGL(ic_init_kernel, dim3((pop + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                     pop, *dv, genomes, props);
  return (int)hipGetLastError();
}

extern "C" int ic_launch_eval(void *stream, const ic_swaption *sw, const ic_period *periods,
                              const ic_worklists *wl, const float *genomes, int32_t npop,
                              const float *herm_x, const float *herm_w, int32_t nherm,
                              int32_t nswap, int mode, int ieee, float *out0, float *out1) {
  EvalArgs A;
  A.sw = sw;
  A.per = periods;
  A.genomes = genomes;
  A.npop = npop;
  A.hx = herm_x;
  A.hw = herm_w;
  A.nherm = nherm;
  A.nswap = nswap;
  A.mode = mode;
  A.out0 = out0;
  A.out1 = out1;
  for (int c = IC_LAUNCHES - 1; c >= 0; c--) {
    if (wl->nwork[c] <= 0) continue;
    A.work = wl->work[c];
    A.nwork = wl->nwork[c];
    const dim3 grid((A.nwork + 3) / 4), block(256);
    void (*const kernel)(EvalArgs) = c == 0 ? (ieee ? ic_eval_kernel<Ieee> : ic_eval_kernel<Short>)
                                     : ieee ? ic_eval_long_kernel<Ieee>
                                            : ic_eval_long_kernel<Short>;
    hipLaunchKernelGGL(kernel, grid, block, 0, (hipStream_t)stream, A);
  }
  return (int)hipGetLastError();
}

extern "C" int ic_launch_step(void *stream, int32_t pop, int32_t nswap, const float *terms,
                              const ic_state *from, const ic_state *to, int init, int32_t acc,
                              const ic_move *next, const ic_dirvec *dv, int32_t it, int32_t conv,
                              const ic_trace *trace) {
  StepArgs A;
  A.pop = pop;
  A.nswap = nswap;
  A.terms = terms;
  A.from = *from;
  A.to = *to;
  A.init = init;
  A.acc = acc;
  A.it = it;
  A.conv = conv;
  A.next = *next;
  A.dv = *dv;
  if (trace) {
    A.trace = *trace;
  } else {
    A.trace.genomes = A.trace.logliks = A.trace.props = A.trace.fb = A.trace.newl = nullptr;
  }
  if (pop <= 0) return 0;
  const int64_t per_block = 256 / kSumLanes;
  hipLaunchKernelGGL(ic_step_kernel, dim3((unsigned)((pop + per_block - 1) / per_block)),
                     dim3(256), 0, (hipStream_t)stream, A);
  return (int)hipGetLastError();
}

extern "C" int ic_launch_winner(void *stream, int32_t pop, const float *genomes,
                                const float *logliks, float *out, float *winner) {
  hipLaunchKernelGGL(ic_winner_kernel, dim3(1), dim3(kWinnerThreads), 0, (hipStream_t)stream, pop, genomes,
                     logliks, out, winner);
  return (int)hipGetLastError();
}
