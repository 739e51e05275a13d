// HIP kernels for gfx950: finpar/OptionPricing.fut's `main`.
//
// One lane per Monte-Carlo path, a wave per 64 consecutive Sobol indices n =
// 64 w + 1 + lane.  The Sobol number is linear in the Gray code over GF(2)
// (:17-27), so of the wave's 64 numbers of a dimension one part is the
// wave's (the Gray code of 64 w) and one the lane's (that of lane + 1; lane
// 63, whose index ends in six zeros, takes the change of the wave's part to
// w + 1 instead).  A path runs the reference's pipeline in f32: the inverse
// Gaussian (:40-140) of each Sobol number as the Brownian bridge (:145-183)
// consumes it, then per market model the Black-Scholes path (:190-225), the
// bridge's differences taken on the fly, streamed date by date into the
// contract's payoff (:230-293).  The shapes are fixed by the contract
// (:289-293), so each contract is its own instantiation.
//
// All three contracts are bound by VALU issue: there is nothing to read but
// tables that every wave shares.  What the layout is after is therefore few
// instructions per dimension and nothing in private memory:
//   * the inverse Gaussian is one polynomial in log2(p (1 - p)) for all but
//     0.02 % of the numbers (gauss below): 17 instructions for about 80;
//   * contracts 1 and 2 keep a lane's Sobol numbers in registers and walk
//     w upwards, one exclusive or per dimension and path;
//   * contract 3 (367 dates x 3 underlyings) keeps only the bridge's dates
//     that are still to be read, in LDS (op_tables_kernel's schedule);
//   * prices are kept as logarithms: the barriers are compared there, and an
//     exponential is taken only where a payoff needs the price itself.
// Payoffs accumulate in f64 per lane, then per wave, workgroup and over the
// workgroups in a fixed order, so a result depends only on the inputs (the
// reference leaves the order of this sum, :318, to its backend).

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "op_internal.h"

namespace {

constexpr int kThreads = 256, kWaves = kThreads / 64;

template <int C>
struct Shape;
template <>
struct Shape<1> {
  static constexpr int D = 1, U = 1;
};
template <>
struct Shape<2> {
  static constexpr int D = 5, U = 3;
};
template <>
struct Shape<3> {
  static constexpr int D = 367, U = 3;
};

// OptionPricing.fut:40-56 (polyAppr), Horner as written, IEEE division.
__device__ __forceinline__ float poly_appr(float x, const float (&a)[8], const float (&b)[8]) {
  const float num =
      x * (x * (x * (x * (x * (x * (x * a[7] + a[6]) + a[5]) + a[4]) + a[3]) + a[2]) + a[1]) +
      a[0];
  const float den =
      x * (x * (x * (x * (x * (x * (x * b[7] + b[6]) + b[5]) + b[4]) + b[3]) + b[2]) + b[1]) +
      b[0];
  return num / den;
}

// OptionPricing.fut:121-136 (ugaussianEl), the tail's value before its sign,
// with the coefficients of intermediate (:81-99).  Those of tail (:101-119) are
// for sqrt(-log pp) > 5, and pp = 0.5 - |p - 0.5| is 0 or at least 2^-25 in
// f32, where that root is 4.2: what is left of that branch is its NaN for a pp
// that is not positive.
constexpr float kIa[8] = {1.42343711074968357734f, 4.6303378461565452959f,
                          5.7694972214606914055f, 3.64784832476320460504f,
                          1.27045825245236838258f, 0.24178072517745061177f,
                          0.0227238449892691845833f, 7.7454501427834140764e-4f};
constexpr float kIb[8] = {1.0f, 2.05319162663775882187f, 1.6763848301838038494f,
                          0.68976733498510000455f, 0.14810397642748007459f,
                          0.0151986665636164571966f, 5.475938084995344946e-4f,
                          1.05075007164441684324e-9f};

__device__ __forceinline__ float gauss_tail(float pp) {
  const float x = poly_appr(sqrtf(-logf(pp)) - 1.6f, kIa, kIb);
  return pp > 0.0f ? x : __builtin_nanf("");
}

// The inverse Gaussian of p = x / 2 ** num_bits (:31-35, :121-140), from d4 =
// 4 (p - 1/2) (every p is a float times a power of two, so the fused multiply
// and add that makes d4 rounds as p - 0.5 does).  With u = log2(16 p (1 - p))
// = log2(4 - d4 * d4), the quotient of the inverse Gaussian by d4 is a smooth
// function of u: kG is its minimax fit of degree 11 for u >= -9 (p between
// 1.2e-4 and 1 - 1.2e-4), relative error 1.9e-8.  Against 64 bits over all
// multiples of 2^-23 there the result is within 1.7e-7, 4.2e-8 rms; the
// rational functions of :58-99 in f32 are within 4.3e-7, 8.4e-8 rms.  Beyond
// that the reference's own tail runs, in a branch that 5 % of the waves take
// per date; a p outside (0, 1) is NaN there as in the reference.
constexpr float kG[12] = {0.8652234077453613f,      -0.12257158011198044f,
                          0.0005459203966893256f,   0.0005110175698064268f,
                          2.668678280315362e-05f,   -3.055389242945239e-06f,
                          -4.226185978950525e-07f,  8.659843508951326e-09f,
                          5.638087330339658e-09f,   5.215573528616346e-10f,
                          2.160310992593839e-11f,   3.478511153166136e-13f};
constexpr float kGTail = 0x1p-9f;

template <int U>
__device__ __forceinline__ void gauss(const int32_t (&x)[U], float scale4, float (&z)[U]) {
  float d4[U], t[U], u[U];
#pragma unroll
  for (int i = 0; i < U; ++i) {
    d4[i] = fmaf((float)x[i], scale4, -2.0f);
    t[i] = fmaf(-d4[i], d4[i], 4.0f);
    u[i] = __builtin_amdgcn_logf(t[i]);
    z[i] = kG[11];
  }
#pragma unroll
  for (int k = 10; k >= 0; --k) {
#pragma unroll
    for (int i = 0; i < U; ++i) z[i] = fmaf(z[i], u[i], kG[k]);
  }
  float least = t[0];
#pragma unroll
  for (int i = 0; i < U; ++i) {
    z[i] *= d4[i];
    least = fminf(least, t[i]);
  }
  if (least < kGTail) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      if (t[i] < kGTail) z[i] = copysignf(gauss_tail(fmaf(-0.25f, fabsf(d4[i]), 0.5f)), d4[i]);
    }
  }
}

// OptionPricing.fut:230-236 (fminPayoff)
__device__ __forceinline__ float fmin_payoff(float x0, float x1, float x2) {
  const float a = x0 / 3758.05f, b = x1 / 11840.0f, c = x2 / 1200.0f;
  return a < b ? (a < c ? a : c) : (b < c ? b : c);
}

// The levels that the payoffs compare prices with: contract 2's are the
// starts of fmin_payoff (1 <= x / level exactly where level <= x),
// contract 3's the barriers (:270), kShift of their logarithms above.
template <int C>
__device__ constexpr float level(int u) {
  return C == 2 ? (u == 0 ? 3758.05f : u == 1 ? 11840.0f : 1200.0f)
                : (u == 0 ? 2630.6349999999998f : u == 1 ? 8288.0f : 840.0f);
}
__device__ __forceinline__ constexpr float shift(int u) {  // log(level<3> / level<2>)
  return u == 0 ? -0.35667494393873245f : u == 1 ? -0.35667494393873245f : -0.35667494393873245f;
}

// One market model set (OptionPricing.fut:299-304), row-major; the kernel's
// __restrict__ parameters, so that wave-uniform reads of them become scalar
// loads.
struct Market {
  const float *cs, *vols, *drifts, *sts, *detvals, *discts;
  int K;
};

// The log return of underlying u at date d (:190-213) from the differences dz
// of the bridge rows.
template <int C>
__device__ __forceinline__ float log_return(const Market &mk, int m, int d, int u,
                                            const float (&dz)[Shape<C>::U]) {
  constexpr int D = Shape<C>::D, U = Shape<C>::U;
  const float *cs = mk.cs + (m * U + u) * U;
  const int at = (m * D + d) * U + u;
  float noise = dz[0] * cs[0];  // (:194-197), from the left
#pragma unroll
  for (int k = 1; k < U; ++k)
    if (k <= u) noise = fmaf(dz[k], cs[k], noise);
  return fmaf(noise, mk.vols[at], mk.drifts[at]);
}

// payoff2's amount times its discount (:246-265): `date` is the first date on
// which all prices are at their starts (4 if none of 0 .. 3), x50 the last
// date's fmin_payoff.
__device__ __forceinline__ float payoff2(const float *disc, int date, float x50) {
  float pay = (1.0f <= x50 ? 1750.0f : (0.75f < x50 ? 1000.0f : x50 * 1000.0f)) * disc[4];
#pragma unroll
  for (int d = 3; d >= 0; --d)
    if (date == d) pay = (1150.0f + 150.0f * (float)d) * disc[d];
  return pay;
}

// payoff3 (:267-283): goto40 where a barrier was reached and x, the last
// date's fmin_payoff, is below 1
__device__ __forceinline__ float payoff3(const float *disc, bool goto40, float x) {
  const float price1 = 100.0f * disc[0];
  const float amount = goto40 ? 1000.0f * x : 1000.0f;
  return price1 + amount * disc[1];
}

// The payoff of one path under model m with the prices as the reference
// makes them, the running product of the exponentials (:214-225), date by date
// into payoff1-3 (:238-293).  row(u, d): the bridge rows.
template <int C, typename Row>
__device__ __forceinline__ float product_payoff(const Market &mk, int m, Row row) {
  constexpr int D = Shape<C>::D, U = Shape<C>::U;
  const float *sts = mk.sts + m * U, *disc = mk.discts + m * mk.K;
  float acc[U], price[U], prev[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    acc[u] = 1.0f;
    prev[u] = 0.0f;
  }
  bool cond = false;
  int date = D - 1;
  float x = 0.0f;
  for (int d = 0; d < D; ++d) {
    float dz[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float r = row(u, d);
      dz[u] = d == 0 ? r : r - prev[u];  // bbrow[i] - bbrow[i - 1] (:181)
      prev[u] = r;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      acc[u] = acc[u] * expf(log_return<C>(mk, m, d, u, dz));  // the scan from 1 (:218)
      price[u] = sts[u] * acc[u];                              // (:219)
    }
    if constexpr (C == 2) {
      x = fmin_payoff(price[0], price[1], price[2]);
      if (date == D - 1 && 1.0f <= x) date = d;
    }
    if constexpr (C == 3)
      cond = cond || price[0] <= level<3>(0) || price[1] <= level<3>(1) ||
             price[2] <= level<3>(2);
  }
  if constexpr (C == 1) {  // payoff1 (:240-244)
    const float amount = (price[0] - 4000.0f) * mk.detvals[m];
    const float amount0 = 0.0f < amount ? amount : 0.0f;
    return amount0 * disc[0];
  } else if constexpr (C == 2) {
    return payoff2(disc, date, x);
  } else {
    const bool goto40 =
        cond && (price[0] < 3758.05f || price[1] < 11840.0f || price[2] < 1200.0f);
    return payoff3(disc, goto40, fmin_payoff(price[0], price[1], price[2]));
  }
}

// Minima and maxima that ignore a NaN, without the compiler's quieting of
// their operands (one instruction more each).
__device__ __forceinline__ float least3(float a, float b, float c) {
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float most3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// A date of a market model: an underlying's volatility times its row of
// md_cs (the lower triangle, by rows), and its drift.
struct Date {
  float a[6], drift[3];
};
template <int C>
__device__ __forceinline__ Date make_date(const Market &mk, int m, int d) {
  constexpr int D = Shape<C>::D;
  Date r = {};
  for (int u = 0, e = 0; u < 3; ++u) {
    const int at = (m * D + d) * 3 + u;
    r.drift[u] = mk.drifts[at];
    for (int k = 0; k <= u; ++k, ++e) r.a[e] = mk.cs[(m * 3 + u) * 3 + k] * mk.vols[at];
  }
  return r;
}

// The payoffs of contracts 2 and 3 from log prices: s is the running sum of
// the log returns from log(start / level), so that a price stands at its
// level where s is 0, and no exponential is taken before the last date.
// Where the product form could not leave the range of normal numbers the
// two agree to rounding (the sum's is the smaller: 367 dates round at 2^-26
// of a price each, the product at 2^-24); pay() says whether that held, and
// a path where it did not, NaN included, is priced by product_payoff.
template <int C>
struct LogPath {
  static constexpr int D = Shape<C>::D;
  float s[3], least, most;
  int date;
  __device__ __forceinline__ void start(const float (&s0)[3]) {
#pragma unroll
    for (int u = 0; u < 3; ++u) s[u] = s0[u];
    least = __builtin_inff();
    most = -__builtin_inff();
    date = D - 1;
  }
  // date d from the differences dz of the bridge rows (:190-213)
  __device__ __forceinline__ void step(const Date &at, int d, const float (&dz)[3]) {
    s[0] = fmaf(dz[0], at.a[0], s[0] + at.drift[0]);
    s[1] = fmaf(dz[1], at.a[2], fmaf(dz[0], at.a[1], s[1] + at.drift[1]));
    s[2] = fmaf(dz[2], at.a[5], fmaf(dz[1], at.a[4], fmaf(dz[0], at.a[3], s[2] + at.drift[2])));
    if constexpr (C == 2) {
      const float low = least3(s[0], s[1], s[2]);
      if (date == D - 1 && 0.0f <= low) date = d;
      least = least3(least, low, low);
    } else {
      least = least3(least3(least, s[0], s[1]), s[2], s[2]);
    }
    most = most3(most3(most, s[0], s[1]), s[2], s[2]);
  }
  __device__ __forceinline__ bool pay(const float *disc, float *out) const {
    // the worst price over its start (fmin_payoff, :230-236)
    if constexpr (C == 2) {
      *out = payoff2(disc, date, expf(least3(s[0], s[1], s[2])));
    } else {
      const float x =
          expf(least3(s[0] + shift(0), s[1] + shift(1), s[2] + shift(2)));
      *out = payoff3(disc, least <= 0.0f && x < 1.0f, x);
    }
    return least > -60.0f && most < 60.0f && fabsf(s[0] + s[1] + s[2]) < 200.0f;
  }
};

// log(start / level), |.| < 20; another start makes it NaN, so that
// LogPath::pay refuses its paths
template <int C>
__device__ __forceinline__ float log_start(const Market &mk, int m, int u) {
  const float s = mk.sts[m * 3 + u];
  return s > 1e-4f && s < 1e8f ? -logf(level<C>(u) / s) : __builtin_nanf("");
}

// Step t of the bridge, and the dates that step t - 1 completed.  Slots as
// offsets in bytes, so that the path kernel spends no instruction on them.
struct Step {
  uint32_t k, j, l;   // the slots of the right and left neighbour and the date
  uint32_t r[2];      // of the first two dates to stream
  uint32_t stream;    // bytes of the records of all the dates to stream
  float sd, lw, rw;   // bb_data
  int32_t pad[3];
};

// Contract 3's tables: the lanes' and the waves' parts of the Sobol numbers
// and the bridge's schedule.
constexpr int kD3 = Shape<3>::D;
constexpr int kLo = 63 + 26;  // lanes 0 .. 62, then lane 63's 26 possible changes
constexpr int kHi = 7;        // a wave's 27 Gray code bits, in groups of 4
constexpr int kSlots = 12;    // live dates in LDS; one slot more is always zero
struct Tables {
  // the path kernel reads ahead: one step and two dates more, zero
  Step step[kD3 + 1];
  Date date[OP_MAX_MODELS][kD3 + 2];
  uint32_t slot[kD3];  // of a date
  int32_t fits;
  int32_t pad[3];
  int32_t lo[kD3][kLo][3];
  int32_t hi[kHi][16][kD3][3];
};

__device__ __forceinline__ int clamp_date(int i, int D) {
  return i < 0 ? 0 : (i >= D ? D - 1 : i);
}

// x ^ (mask & v), one instruction of gfx950
__device__ __forceinline__ int32_t xor_and(int32_t x, int32_t mask, int32_t v) {
  return (int32_t)__builtin_amdgcn_bitop3_b32((uint32_t)mask, (uint32_t)v, (uint32_t)x, 0x6a);
}

// Contracts 1 and 2 (few dimensions).  Each wave walks a run of consecutive
// w, its lanes' Sobol numbers in registers: from w to w + 1 the Gray code of
// 64 w changes in bit 5 and bit 6 + ctz(w + 1), so every dimension takes one
// exclusive or with a row of `change`, read from LDS (lane 63 is one w
// ahead).  4096 waves at most (OP_FEW_BLOCKS): at 2^20 paths 4 per SIMD with 4
// paths a lane, which hide the LDS and share the 350 instructions of a wave's
// start; half, 3/4 and twice as many measured 4, 2 and 5 us more.  Bound by VALU
// issue: 2^20 paths of contract 2 take 21 us, against 73.5 with the numbers
// looked up per path and the rational functions.
template <int C, int MC>
__global__ __launch_bounds__(kThreads) void op_few_kernel(
    const int32_t *__restrict__ dir_vs, const int32_t *__restrict__ bbi,
    const float *__restrict__ bbd, const float *__restrict__ cs,
    const float *__restrict__ vols, const float *__restrict__ drifts,
    const float *__restrict__ sts, const float *__restrict__ detvals,
    const float *__restrict__ discts, int bits, int K, int M, int64_t N,
    double *__restrict__ partial) {
  const Market mk = {cs, vols, drifts, sts, detvals, discts, K};
  constexpr int D = Shape<C>::D, U = Shape<C>::U, DIMS = D * U, PAD = DIMS > 1 ? 16 : 1;
  static_assert(DIMS <= PAD, "a row of the tables");
  __shared__ int32_t vec[32][PAD], change[26][PAD];
  // the bridge rows: a lane reads and writes its own column only
  __shared__ float4 rows[C == 1 ? 1 : kWaves][C == 1 ? 1 : D][C == 1 ? 1 : 64];
  // the models' dates
  __shared__ Date dates[C == 1 ? 1 : MC][C == 1 ? 1 : D];
  __shared__ float starts[MC][3];
  __shared__ double red[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if constexpr (C == 2) {
    if (tid < M * D) dates[tid / D][tid % D] = make_date<C>(mk, tid / D, tid % D);
    if (tid >= 64 && tid < 64 + 3 * M)
      starts[(tid - 64) / 3][(tid - 64) % 3] = log_start<C>(mk, (tid - 64) / 3, (tid - 64) % 3);
  }
  for (int i = tid; i < 32 * PAD; i += kThreads) {
    const int b = i / PAD, d = i % PAD;
    vec[b][d] = b < bits && d < DIMS ? dir_vs[d * bits + b] : 0;
  }
  __syncthreads();
  for (int i = tid; i < 26 * PAD; i += kThreads) {
    const int t = i / PAD, d = i % PAD;
    change[t][d] = vec[5][d] ^ vec[6 + t][d];
  }
  __syncthreads();
  const float scale4 = ldexpf(4.0f, -bits);
  float s0[MC][3];
  if constexpr (C == 2) {
#pragma unroll
    for (int m = 0; m < MC; ++m)
#pragma unroll
      for (int u = 0; u < 3; ++u) s0[m][u] = starts[m][u];
  }
  // the bridge (:145-177) may skip the rows' zero start (:153) where no step
  // reads a date that no earlier one wrote and every date is written
  const int32_t *bi = bbi, *li = bbi + D, *ri = bbi + 2 * D;
  const float *sd = bbd, *lw = bbd + D, *rw = bbd + 2 * D;
  uint32_t written = 0;
  bool zero_free = true;
#pragma unroll
  for (int i = 0; i < D; ++i) {
    const int j = li[i] - 1;
    if (i > 0)
      zero_free = zero_free && (written >> clamp_date(ri[i] - 1, D) & 1u) &&
                  (j == -1 || (written >> clamp_date(j, D) & 1u));
    written |= 1u << clamp_date(bi[i] - 1, D);
  }
  zero_free = zero_free && written == (1u << D) - 1u;
  // a lane's places of the bridge's reads and writes
  uint32_t at_l[D], at_k[D], at_j[D];
#pragma unroll
  for (int i = 0; i < D; ++i) {
    at_l[i] = (uint32_t)(clamp_date(bi[i] - 1, D) * 64 + lane);
    at_k[i] = (uint32_t)(clamp_date(ri[i] - 1, D) * 64 + lane);
    at_j[i] = (uint32_t)(clamp_date(li[i] - 1, D) * 64 + lane);
    asm("" : "+v"(at_l[i]), "+v"(at_k[i]), "+v"(at_j[i]));
  }
  double sum[MC];
#pragma unroll
  for (int m = 0; m < MC; ++m) sum[m] = 0.0;
  // this wave's run of w
  const int64_t blocks = (N + 63) / 64, waves = (int64_t)gridDim.x * kWaves;
  const int64_t self = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWaves + wave));
  const int w0 = (int)(self * blocks / waves), w1 = (int)((self + 1) * blocks / waves);
  int32_t x[DIMS];
  {
    const uint32_t c = (uint32_t)w0 << 6, hi = c ^ (c >> 1);
    const uint32_t n = (uint32_t)lane + 1u, g = lane == 63 ? 0u : n ^ (n >> 1);
    // the wave's part, dimension d in lane d, and lane 63's change
    int32_t part = 0;
    for (uint32_t left = hi; left; left &= left - 1u)
      part ^= vec[__builtin_ctz(left)][lane % PAD];
    const int32_t *ch = change[__builtin_ctz((uint32_t)w0 + 1u)];
    const int32_t last = -(int32_t)(lane == 63);
#pragma unroll
    for (int d = 0; d < DIMS; ++d)
      x[d] = xor_and(__builtin_amdgcn_readlane(part, d), last, ch[d]);
#pragma unroll
    for (int b = 0; b < 6; ++b) {
      const int32_t mask = -(int32_t)(g >> b & 1u);
#pragma unroll
      for (int d = 0; d < DIMS; ++d) x[d] = xor_and(x[d], mask, vec[b][d]);
    }
  }
  for (int w = w0; w < w1; ++w) {
    const bool live = (int64_t)w * 64 + lane < N;
    if constexpr (C == 1) {
      float z[1];
      gauss<1>(x, scale4, z);
      const float r = sd[0] * z[0];
#pragma unroll
      for (int m = 0; m < MC; ++m) {
        if (m < M) {
          const float pay = product_payoff<1>(mk, m, [&](int, int) { return r; });
          if (live) sum[m] += (double)pay;
        }
      }
    } else {
      // the dates are read from LDS for each path: kept in registers, their 45
      // values cost a wave of four per SIMD (28.5 against 22.6 us, 2^20 paths)
      asm volatile("" ::: "memory");
      float4 *const mine = rows[wave][0];
      if (!zero_free) {
#pragma unroll
        for (int d = 0; d < D; ++d) mine[d * 64 + lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      }
#pragma unroll
      for (int i = 0; i < D; ++i) {
        const int32_t xi[3] = {x[3 * i], x[3 * i + 1], x[3 * i + 2]};
        float z[3];
        gauss<3>(xi, scale4, z);
        float4 v = make_float4(sd[i] * z[0], sd[i] * z[1], sd[i] * z[2], 0.0f);
        if (i > 0) {
          const float4 k = mine[at_k[i]];
          v.x = fmaf(rw[i], k.x, v.x);
          v.y = fmaf(rw[i], k.y, v.y);
          v.z = fmaf(rw[i], k.z, v.z);
          if (li[i] != 0) {
            const float4 q = mine[at_j[i]];
            v.x = fmaf(lw[i], q.x, v.x);
            v.y = fmaf(lw[i], q.y, v.y);
            v.z = fmaf(lw[i], q.z, v.z);
          }
        }
        mine[at_l[i]] = v;
      }
      LogPath<C> path[MC];
#pragma unroll
      for (int m = 0; m < MC; ++m) path[m].start(s0[m]);
      float4 prev = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const float4 r = mine[d * 64 + lane];
        const float dz[3] = {r.x - prev.x, r.y - prev.y, r.z - prev.z};
        prev = r;
#pragma unroll
        for (int m = 0; m < MC; ++m)
          if (m < M) path[m].step(dates[m][d], d, dz);
      }
#pragma unroll
      for (int m = 0; m < MC; ++m) {
        if (m < M) {
          float pay;
          if (!path[m].pay(discts + m * K, &pay))
            pay = product_payoff<C>(mk, m, [&](int u, int d) {
              return reinterpret_cast<const float *>(&mine[d * 64 + lane])[u];
            });
          if (live) sum[m] += (double)pay;
        }
      }
    }
    const int32_t *ch = change[__builtin_ctz((uint32_t)(w + 1 + (lane == 63)))];
#pragma unroll
    for (int d = 0; d < DIMS; ++d) x[d] ^= ch[d];
  }
  // the workgroup's sums, model by model
#pragma unroll
  for (int m = 0; m < MC; ++m) {
    if (m < M) {
      double s = sum[m];
#pragma unroll
      for (int k = 32; k > 0; k >>= 1) s += __shfl_xor(s, k);
      if (lane == 0) red[wave] = s;
      __syncthreads();
      if (tid == 0)
        partial[(int64_t)blockIdx.x * M + m] = (red[0] + red[1]) + (red[2] + red[3]);
      __syncthreads();
    }
  }
}

// A record at a wave-uniform offset of tables that this launch does not
// write, through the constant address space: scalar loads, which the
// compiler does not find by itself beside the stores to LDS.
template <typename T>
__device__ __forceinline__ T scalar_load(const Tables *tab, uint32_t at) {
  typedef const __attribute__((address_space(4))) char Const;
  typedef const __attribute__((address_space(4))) uint32_t Word;
  union {
    uint32_t w[sizeof(T) / 4];
    T t;
  } r;
  Word *const p = (Word *)((Const *)(uintptr_t)tab + at);
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) / 4); ++i) r.w[i] = p[i];
  return r.t;
}

// three ints at a lane's address
__device__ __forceinline__ void load3(const char *at, int32_t (&v)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) v[i] = ((const int32_t *)at)[i];
}

// Contract 3.  A path's 1101 bridge values in private memory are 590 MB for
// 2^17 paths, written and read once each.  But the reference's tables build
// the bridge's middle dates left first, so that after each step the dates up to
// some point are complete and can be streamed into the prices, and only a
// path's ancestors in the bridge's tree (at most 10 of 367 dates) are still to
// be read.  op_tables_kernel finds that schedule, and a wave keeps those dates in
// LDS: 13 slots of 16 bytes a lane, 52 KB a workgroup, 3 workgroups (12 waves) a
// CU.  Tables that need more slots, or read dates that are not written, and
// prices outside the log form's range keep the rows in private memory.
// 2^17 paths are 2 waves per SIMD, so a step's latencies are hidden by its
// order and not by other waves, and its 101 VALU cycles of 4 (60 the
// Gaussians, 20 the date) are 96 % of the time: 157 us, against 1064 with the
// rows in private memory and the rational functions.  Loads a step ahead
// (211 -> 197 us), records as byte offsets in scalar registers and the wave's
// part of the numbers by groups of 4 bits (197 -> 188) came after that.
template <int MC>
__global__ __launch_bounds__(kThreads) void op_many_kernel(
    const Tables *__restrict__ tab, const int32_t *__restrict__ bbi,
    const float *__restrict__ bbd, const float *__restrict__ cs,
    const float *__restrict__ vols, const float *__restrict__ drifts,
    const float *__restrict__ sts, const float *__restrict__ detvals,
    const float *__restrict__ discts, int bits, int K, int M, int64_t N,
    double *__restrict__ partial) {
  const Market mk = {cs, vols, drifts, sts, detvals, discts, K};
  constexpr int D = kD3, U = 3, kChunks = (D + 63) / 64;
  static_assert(sizeof(Step) == 48 && sizeof(Date) == 36, "table records");
  __shared__ float4 slots[kWaves][kSlots + 1][64];
  __shared__ double red[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float scale4 = ldexpf(4.0f, -bits);
  const bool fits = __builtin_amdgcn_readfirstlane(tab->fits) != 0;
  float s0[MC][U];
#pragma unroll
  for (int m = 0; m < MC; ++m)
#pragma unroll
    for (int u = 0; u < U; ++u) s0[m][u] = m < M ? log_start<3>(mk, m, u) : 0.0f;
  // The tables come from another launch, so they are in no XCD's L2, and a wave
  // that reads them date by date would wait for memory 367 times: the first
  // workgroups of an XCD read them through once, 128 bytes a lane.
  int32_t seen = 0;
  {
    const int parts = min(8, max(1, (int)gridDim.x / 32));
    const int lines = (int)(offsetof(Tables, hi) / 128);
    for (int i = (int)(blockIdx.x / 8) % parts * kThreads + tid; i < lines; i += parts * kThreads)
      seen ^= ((const int32_t *)tab)[i * 32];
  }
  double sum[MC];
#pragma unroll
  for (int m = 0; m < MC; ++m) sum[m] = 0.0;
  float4 *const mine = &slots[wave][0][lane];
  mine[kSlots * 64] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const int64_t blocks = (N + 63) / 64, waves = (int64_t)gridDim.x * kWaves;
  const int64_t self = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWaves + wave));
  const int w0 = (int)(self * blocks / waves), w1 = (int)((self + 1) * blocks / waves);
  for (int w = w0; w < w1; ++w) {
    const bool live = (int64_t)w * 64 + lane < N;
    const uint32_t c = (uint32_t)w << 6, ghi = (c ^ (c >> 1)) >> 5;
    const int at = lane < 63 ? lane : 63 + __builtin_ctz((uint32_t)w + 1u);
    // the wave's parts of all dates, date 64 c + lane in this lane's part[c]
    int32_t part[kChunks][U] = {};
    for (uint32_t g = 0; ghi >> (4 * g) != 0u; ++g) {
      const int32_t(*const v)[3] = tab->hi[g][ghi >> (4 * g) & 15u];
#pragma unroll
      for (int c = 0; c < kChunks; ++c) {
        const int t = c * 64 + lane < D ? c * 64 + lane : D - 1;
#pragma unroll
        for (int u = 0; u < U; ++u) part[c][u] ^= v[t][u];
      }
    }
    int32_t h[U] = {};
    auto wave_part = [&](int t0) {
#pragma unroll
      for (int c = 0; c < kChunks; ++c)
#pragma unroll
        for (int u = 0; u < U; ++u) h[u] = t0 == c * 64 ? part[c][u] : h[u];
    };
    asm volatile("" ::"v"(seen));
    float pay[MC];
    // the models whose payoff stands: a model's path is repriced for its own
    // prices' sake only, so its mean does not depend on which share the pass
    bool good[MC], all = false;
#pragma unroll
    for (int m = 0; m < MC; ++m) good[m] = false;
    if (fits) {
      LogPath<3> path[MC];
#pragma unroll
      for (int m = 0; m < MC; ++m) path[m].start(s0[m]);
      float prev[U] = {0.0f, 0.0f, 0.0f};
      // One step's order: everything that is read for it is asked for, then the
      // Gaussians, then the dates that the step before completed, then this
      // step's date.  So the latencies pass under the Gaussians.
      const char *const here = (const char *)mine;
      const char *lo = (const char *)tab->lo[0][at];
      uint32_t step_at = 0, date_at = 0;  // bytes
      auto step_of = [&](uint32_t at_t) {
        return scalar_load<Step>(tab, (uint32_t)offsetof(Tables, step) + at_t);
      };
      auto date_of = [&](int m, uint32_t at_d) {
        return scalar_load<Date>(
            tab, (uint32_t)(offsetof(Tables, date) + m * sizeof(tab->date[0])) + at_d);
      };
      auto stream = [&](const Date (&at_d)[MC], const float4 &r) {
        const float dz[U] = {r.x - prev[0], r.y - prev[1], r.z - prev[2]};
        prev[0] = r.x;
        prev[1] = r.y;
        prev[2] = r.z;
#pragma unroll
        for (int m = 0; m < MC; ++m)
          if (MC == 1 || m < M) path[m].step(at_d[m], 0, dz);
      };
      auto stream_rest = [&](uint32_t from, uint32_t to) {
        for (uint32_t e = from; e < to; e += sizeof(Date)) {
          Date at_d[MC];
#pragma unroll
          for (int m = 0; m < MC; ++m) at_d[m] = date_of(m, e);
          stream(at_d, *(const float4 *)(here + tab->slot[e / sizeof(Date)]));
        }
      };
      Step ahead = step_of(0);
      // the lane parts two steps ahead, in two sets of registers
      int32_t even[U], odd[U];
      load3(lo, even);
      load3(lo + kLo * 12, odd);
      lo += 2 * kLo * 12;
      auto step = [&](int t, int32_t(&mine_x)[U]) {
        const Step st = ahead;
        const float4 k = *(const float4 *)(here + st.k), j = *(const float4 *)(here + st.j);
        const float4 r0 = *(const float4 *)(here + st.r[0]);
        const float4 r1 = *(const float4 *)(here + st.r[1]);
        step_at += sizeof(Step);
        ahead = step_of(step_at);
        Date near[2][MC];
#pragma unroll
        for (int m = 0; m < MC; ++m) {
          near[0][m] = date_of(m, date_at);
          near[1][m] = date_of(m, date_at + (uint32_t)sizeof(Date));
        }
        int32_t x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = mine_x[u] ^ __builtin_amdgcn_readlane(h[u], t);
        load3(lo, mine_x);  // the last two steps': past the table, in tab->hi
        lo += kLo * 12;
        __builtin_amdgcn_sched_barrier(0);
        float z[U];
        gauss<U>(x, scale4, z);
        float4 v;
        v.x = fmaf(st.lw, j.x, fmaf(st.rw, k.x, st.sd * z[0]));
        v.y = fmaf(st.lw, j.y, fmaf(st.rw, k.y, st.sd * z[1]));
        v.z = fmaf(st.lw, j.z, fmaf(st.rw, k.z, st.sd * z[2]));
        v.w = 0.0f;
        if (st.stream != 0) {
          stream(near[0], r0);
          if (st.stream > sizeof(Date)) {
            stream(near[1], r1);
            // before this step's date takes a slot
            stream_rest(date_at + 2 * sizeof(Date), date_at + st.stream);
          }
          date_at += st.stream;
        }
        *(float4 *)((char *)mine + st.l) = v;
      };
      for (int t0 = 0; t0 < D; t0 += 64) {
        wave_part(t0);
        const int t1 = t0 + 64 < D ? t0 + 64 : D - 1;
        for (int t = t0; t < t1; t += 2) {
          step(t, even);
          step(t + 1, odd);
        }
      }
      static_assert(D % 2 == 1, "a last step");
      step(D - 1, even);
      stream_rest(date_at, D * sizeof(Date));
      all = true;
#pragma unroll
      for (int m = 0; m < MC; ++m)
        if (m < M) {
          good[m] = path[m].pay(discts + m * K, &pay[m]);
          all = good[m] && all;
        }
    }
    if (__any(!all)) {
      // any tables, any values: all rows in private memory, starting at zero
      // (:153), indexes clamped to the row so that no input makes an access out
      // of bounds (the reference reads bb_inds unchecked, :156)
      const int32_t *bi = bbi, *li = bbi + D, *ri = bbi + 2 * D;
      const float *sd = bbd, *lw = bbd + D, *rw = bbd + 2 * D;
      float rows[U][D];
      for (int i = 0; i < D; ++i) {
#pragma unroll
        for (int u = 0; u < U; ++u) rows[u][i] = 0.0f;
      }
      for (int i = 0; i < D; ++i) {
        if ((i & 63) == 0) wave_part(i);
        const int l = clamp_date(bi[i] - 1, D), k = clamp_date(ri[i] - 1, D), j = li[i] - 1;
        int32_t x[U];
        float z[U], v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          x[u] = tab->lo[i][at][u] ^ __builtin_amdgcn_readlane(h[u], i & 63);
        gauss<U>(x, scale4, z);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          v[u] = sd[i] * z[u];
          if (i > 0) {
            v[u] = fmaf(rw[i], rows[u][k], v[u]);
            if (j != -1) v[u] = fmaf(lw[i], rows[u][clamp_date(j, D)], v[u]);
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) rows[u][l] = v[u];
      }
#pragma unroll
      for (int m = 0; m < MC; ++m) {
        if (m < M) {
          const float p = product_payoff<3>(mk, m, [&](int u, int d) { return rows[u][d]; });
          if (!good[m]) pay[m] = p;
        }
      }
    }
#pragma unroll
    for (int m = 0; m < MC; ++m)
      if (m < M && live) sum[m] += (double)pay[m];
  }
#pragma unroll
  for (int m = 0; m < MC; ++m) {
    if (m < M) {
      double s = sum[m];
#pragma unroll
      for (int k = 32; k > 0; k >>= 1) s += __shfl_xor(s, k);
      if (lane == 0) red[wave] = s;
      __syncthreads();
      if (tid == 0)
        partial[(int64_t)blockIdx.x * M + m] = (red[0] + red[1]) + (red[2] + red[3]);
      __syncthreads();
    }
  }
}

// Contract 3's tables, one launch: workgroup 0 makes the bridge's schedule,
// the others the parts of the Sobol numbers and the models' dates.  It is the
// schedule's chain of LDS and barriers, 8.9 us; the dates made at its end, and a
// second search for the step before, were 1.2 us of it.
//
// The schedule: with the path kernel's clamped indexes step i (of D) writes
// date l_i and, for i >= 1, reads dates k_i and (when li != 0) j_i.  Every date
// must be written by exactly one step and every read date by an earlier
// one (then no read sees the rows' zero start).  A date's slot is its depth, the
// longest chain of reads below it; date d is streamed after the first step that
// completes the dates up to d.  That fits when no slot is written again before
// its date's last read or its streaming, which is checked, not assumed: next()
// is the first later step that writes a step's slot.
constexpr int kTabThreads = 512;
__global__ __launch_bounds__(kTabThreads) void op_tables_kernel(
    const int32_t *__restrict__ dir_vs, const int32_t *__restrict__ bbi,
    const float *__restrict__ bbd, const float *__restrict__ cs,
    const float *__restrict__ vols, const float *__restrict__ drifts, int bits, int groups,
    int M, Tables *__restrict__ tab) {
  constexpr int D = kD3;
  static_assert(D + 2 <= kTabThreads, "one step per thread");
  const int tid = threadIdx.x;
  if (blockIdx.x > 0) {
    const int i = (int)(blockIdx.x - 1) * kTabThreads + tid;
    // bit b's vector where `on`, read in any case: the loads are independent
    auto vec = [&](int t, int u, int b, bool on) {
      const int32_t v = bits > 0 ? dir_vs[(t * 3 + u) * bits + min(b, bits - 1)] : 0;
      return on && b < bits ? v : 0;
    };
    if (i < D * kLo) {
      const int t = i / kLo, at = i % kLo;
      const uint32_t g = (uint32_t)(at + 1) ^ (uint32_t)(at + 1) >> 1;
      for (int u = 0; u < 3; ++u) {
        int32_t x = 0;
        if (at < 63) {
#pragma unroll
          for (int b = 0; b < 6; ++b) x ^= vec(t, u, b, g >> b & 1u);
        } else {
          x = vec(t, u, 5, true) ^ vec(t, u, 6 + at - 63, true);
        }
        tab->lo[t][at][u] = x;
      }
    } else if (i < D * (kLo + 16 * groups)) {
      const int e = i - D * kLo, row = e / D, t = e % D;
      for (int u = 0; u < 3; ++u) {
        int32_t x = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) x ^= vec(t, u, 5 + row / 16 * 4 + b, row >> b & 1);
        tab->hi[row / 16][row % 16][t][u] = x;
      }
    } else {
      // the models' dates, and two zero ones that the path kernel reads past them
      const int e = i - D * (kLo + 16 * groups), m = e / (D + 2), d = e % (D + 2);
      const Market mk = {cs, vols, drifts, nullptr, nullptr, nullptr, 0};
      if (m < M) tab->date[m][d] = d < D ? make_date<3>(mk, m, d) : Date{};
    }
    return;
  }
  constexpr int kWords = (D + 31) / 32;
  __shared__ int32_t first[D], count[D], depth[2][D], ready[kTabThreads];
  __shared__ int32_t most[kTabThreads / 64];
  __shared__ uint32_t uses[kSlots][kWords];
  __shared__ int32_t bad;
  const int i = tid;
  const bool on = i < D;
  int l = 0, k = 0, j = 0;
  float sd = 0.0f, lw = 0.0f, rw = 0.0f;
  if (on) {
    sd = bbd[i];
    lw = bbd[D + i];
    rw = bbd[2 * D + i];
    l = clamp_date(bbi[i] - 1, D);
    j = bbi[D + i] - 1;
    k = clamp_date(bbi[2 * D + i] - 1, D);
    if (i == 0) j = -1;
    if (j != -1) j = clamp_date(j, D);
    first[i] = D;
    count[i] = 0;
    depth[0][i] = 0;
  }
  for (int e = tid; e < kSlots * kWords; e += kTabThreads) (&uses[0][0])[e] = 0u;
  if (tid == 0) bad = 0;
  __syncthreads();
  if (on) {
    atomicMin(&first[l], i);
    atomicAdd(&count[l], 1);
  }
  __syncthreads();
  bool ok = true;
  if (on) {
    ok = count[i] == 1;
    if (i > 0) ok = ok && first[k] < i && (j == -1 || first[j] < i);
    if (!ok) bad = 1;
  }
  __syncthreads();
  if (bad) {
    if (tid == 0) tab->fits = 0;
    return;  // uniform, as every later return here
  }
  const int fk = on && i > 0 ? first[k] : 0, fj = on && j != -1 ? first[j] : 0;
  // depths: after r rounds every depth below r is final
  int r = 0, deep = 0;
  for (; r <= kSlots; ++r) {
    if (on && i > 0) {
      deep = depth[r & 1][fk] + 1;
      if (j != -1) deep = max(deep, depth[r & 1][fj] + 1);
    }
    if (on) depth[(r + 1) & 1][i] = deep;
    __syncthreads();
  }
  if (on && deep >= kSlots) bad = 1;
  // the step that completes the dates up to i: a running maximum
  int done = on ? first[i] : 0;
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) {
    const int v = __shfl_up(done, s);
    if ((tid & 63) >= s) done = max(done, v);
  }
  if ((tid & 63) == 63) most[tid >> 6] = done;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kTabThreads / 64; ++w) {
    const int v = most[w];  // read whether it counts or not: the reads are independent
    done = w < tid >> 6 ? max(done, v) : done;
  }
  ready[tid] = done;
  if (bad) {
    if (tid == 0) tab->fits = 0;
    return;
  }
  const int32_t *dep = depth[r & 1];
  if (on) atomicOr(&uses[deep][i >> 5], 1u << (i & 31));
  __syncthreads();
  auto next = [&](int step) {
    const uint32_t *m = uses[dep[step]];
    int word = (step + 1) >> 5;
    uint32_t left = word < kWords ? m[word] & (~0u << ((step + 1) & 31)) : 0u;
    while (left == 0u && ++word < kWords) left = m[word];
    return left ? word * 32 + __builtin_ctz(left) : D;
  };
  // the dates complete after step i: ready is ascending
  int upto = 0;
  for (int hi = D; upto < hi;) {
    const int mid = (upto + hi) >> 1;
    if (ready[mid] <= i)
      upto = mid + 1;
    else
      hi = mid;
  }
  if (on) count[i] = upto;
  __syncthreads();
  if (on) {
    ok = next(first[i]) > done;
    if (i > 0) ok = ok && next(fk) >= i && (j == -1 || next(fj) >= i);
    if (!ok) bad = 1;
    const int from = i > 0 ? count[i - 1] : 0;
    auto offset = [](int slot) { return (uint32_t)(slot * 64 * (int)sizeof(float4)); };
    auto slot_of = [&](int d) { return offset(d < D ? dep[first[d]] : kSlots); };
    // the half of a record that streams comes from the thread of the step before
    Step *const st = &tab->step[i];
    st->k = offset(i > 0 ? dep[fk] : kSlots);
    st->j = offset(j != -1 ? dep[fj] : kSlots);
    st->l = offset(deep);
    st->sd = sd;
    st->lw = j != -1 ? lw : 0.0f;
    st->rw = i > 0 ? rw : 0.0f;
    st[1].r[0] = slot_of(from);
    st[1].r[1] = slot_of(from + 1);
    st[1].stream = (uint32_t)(upto - from) * (uint32_t)sizeof(Date);
    if (i == 0) {
      st->r[0] = st->r[1] = offset(kSlots);
      st->stream = 0u;
    }
    tab->slot[i] = slot_of(i);
  }
  __syncthreads();
  if (tid == 0) tab->fits = !bad;
}

// The mean per model: the workgroups' partial sums in a fixed order, / N.
constexpr int kMeanThreads = 256;
__global__ __launch_bounds__(kMeanThreads) void op_mean_kernel(const double *partial, int nblocks,
                                                               int M, int64_t N, float *out) {
  constexpr int kEach = (OP_MANY_BLOCKS + kMeanThreads - 1) / kMeanThreads;
  static_assert(OP_FEW_BLOCKS <= OP_MANY_BLOCKS, "partial sums per thread");
  __shared__ double red[kMeanThreads / 64];
  const int tid = threadIdx.x;
  for (int m = 0; m < M; ++m) {
    double v[kEach], s = 0.0;
#pragma unroll
    for (int k = 0; k < kEach; ++k) {  // in flight together
      const int b = tid + k * kMeanThreads;
      v[k] = b < nblocks ? partial[(int64_t)b * M + m] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kEach; ++k) s += v[k];
#pragma unroll
    for (int k = 32; k > 0; k >>= 1) s += __shfl_xor(s, k);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0)
      out[m] = (float)(((red[0] + red[1]) + (red[2] + red[3])) / (double)N);
    __syncthreads();
  }
}

}  // namespace

extern "C" {

int op_blocks(int contract, int64_t paths) {
  const int64_t b = (paths + kThreads - 1) / kThreads;
  const int64_t most = contract == 3 ? OP_MANY_BLOCKS : OP_FEW_BLOCKS;
  return (int)(b < most ? b : most);
}

size_t op_table_bytes(int contract) { return contract == 3 ? sizeof(Tables) : 0; }

int op_launch(void *stream, int contract, const op_args *A, const int32_t *dir_vs,
              void *tables, double *partial, float *out) {
  hipStream_t st = (hipStream_t)stream;
  if (contract < 1 || contract > 3 || A->M < 1 || A->bits < 0 || A->bits > OP_MAX_BITS ||
      A->N < 1 || A->N > INT32_MAX)
    return (int)hipErrorInvalidValue;
  const int nblocks = op_blocks(contract, A->N);
  const int D = contract == 1 ? 1 : contract == 2 ? 5 : kD3, U = contract == 1 ? 1 : 3;
  Tables *tab = (Tables *)tables;
  // the models in chunks of OP_MAX_MODELS (a lane's sums are registers): each
  // chunk reruns the paths with its models' market data and writes its means
  for (int m0 = 0; m0 < A->M; m0 += OP_MAX_MODELS) {
    const int mc = A->M - m0 < OP_MAX_MODELS ? A->M - m0 : OP_MAX_MODELS;
    if (contract == 3) {
      // the groups of bits that a wave's base has
      int groups = 0;
      while (groups < kHi && (((uint32_t)A->N + 63u) >> 5) >> (4 * groups) != 0u) ++groups;
      const int entries = kD3 * (kLo + 16 * groups) + mc * (kD3 + 2);
      op_tables_kernel<<<1 + (entries + kTabThreads - 1) / kTabThreads, kTabThreads, 0, st>>>(
          dir_vs, A->bbi, A->bbd, A->cs + (int64_t)m0 * U * U, A->vols + (int64_t)m0 * D * U,
          A->drifts + (int64_t)m0 * D * U, A->bits, groups, mc, tab);
    }
#define OP_PATHS(KERNEL, FIRST)                                                          \
  KERNEL<<<nblocks, kThreads, 0, st>>>(                                                  \
      FIRST, A->bbi, A->bbd, A->cs + (int64_t)m0 * U * U, A->vols + (int64_t)m0 * D * U, \
      A->drifts + (int64_t)m0 * D * U, A->sts + (int64_t)m0 * U, A->detvals + m0,        \
      A->discts + (int64_t)m0 * A->K, A->bits, A->K, mc, A->N, partial)
    // one model is the common call; more share the bridge
    if (contract == 1) {
      if (mc == 1) OP_PATHS((op_few_kernel<1, 1>), dir_vs);
      else OP_PATHS((op_few_kernel<1, OP_MAX_MODELS>), dir_vs);
    } else if (contract == 2) {
      if (mc == 1) OP_PATHS((op_few_kernel<2, 1>), dir_vs);
      else OP_PATHS((op_few_kernel<2, OP_MAX_MODELS>), dir_vs);
    } else {
      if (mc == 1) OP_PATHS(op_many_kernel<1>, tab);
      else OP_PATHS(op_many_kernel<OP_MAX_MODELS>, tab);
    }
#undef OP_PATHS
    op_mean_kernel<<<1, kMeanThreads, 0, st>>>(partial, nblocks, mc, A->N, out + m0);
  }
  return (int)hipGetLastError();
}

}  // extern "C"
