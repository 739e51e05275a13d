/*
 * Host side of the prices by separation of x (lvc_modes_kernels.hip): which
 * problems take it, and the launches of main's one grid and of a batch.
 */
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include "lvc_runtime.h"

/* Time steps from which this path is taken: three launches against two per step
 * of the sweeps.  main with one strike and 7 steps, us by the sweeps / by the
 * modes: 32 x 4 points 142 / 36, 256 x 256 187 / 52, 1024 x 4 183 / 123; with 15
 * steps 224 / 37, 318 / 54, 319 / 125. */
#define MODES_MIN_STEPS 6

static int64_t align64(int64_t v) { return (v + 63) & ~(int64_t)63; }

/* Whether a problem (its initGrid scalars set) separates, in FP64, to the
 * accuracy of the sweeps.  The weights 4 dx^2 / x^(2 beta) of the interior
 * nodes have to be positive, fall with x and stay within 1e8 of each other
 * (the kernel rescales its recurrence every 16 nodes), and x^beta at the
 * price node within 256 times the first node's (the factor by which the sum
 * over modes can amplify rounding there); every exponential has to stay far
 * from the range's ends.  x[0] enters the reference's log(x) too (:63): where
 * that is not finite every price is NaN, and the sweeps give that. */
int lvc_modes_fit(const lvc_problem *q) {
  if (q->status != 0 || q->nt - 1 < MODES_MIN_STEPS)
    return 0;
  const double s0 = q->s0, t = q->t, alpha = q->alpha, nu = q->nu, beta = q->beta;
  const int in_range = s0 > 1e-30 && s0 < 1e30 && t > 1e-30 && t < 1e30 && alpha > 1e-30 &&
                       alpha < 1e30 && nu > 1e-6 && nu < 1e6 && beta >= 0.0 && beta < 1e3 &&
                       q->dx > 1e-60 && q->dx < 1e60 && q->dy > 1e-30 && q->dy < 1e30;
  if (!in_range || !(q->x0log > 0.0 || (q->x0log == 0.0 && beta > 0.0)))
    return 0;
  /* 2 y reaches 10 nu sqrt(t) + 2 log(alpha), the time factor nu^2 t */
  if (!(10.0 * nu * sqrt(t) < 100.0 && nu * nu * t < 100.0))
    return 0;
  const double x1 = q->dx - (double)q->xindex * q->dx + s0;
  const double xn = (double)(q->nx - 2) * q->dx - (double)q->xindex * q->dx + s0;
  if (!(x1 > 0.0) || !(fabs(2.0 * beta * log(x1)) < 100.0) ||
      !(fabs(2.0 * beta * log(xn)) < 100.0))
    return 0;
  return 2.0 * beta * log(xn / x1) < log(1e8) && beta * log(s0 / x1) < log(256.0);
}

/* Whether a problem of a batch costs less by its modes than by the sweeps.  A
 * grid's modes are numX / 4 waves that each pass over numX nodes some seven
 * times whatever numY and the steps are (and from 512 nodes on their LDS leaves
 * few waves per CU), and its sweeps numX numY points per step.  Measured, ms
 * by the sweeps / by the modes, numX x numY x steps:
 *   512 problems   192 x 16 x 8 0.68 / 0.83, 192 x 8 x 31 1.15 / 0.84,
 *                  256 x 64 x 8 1.03 / 1.15, 256 x 128 x 8 1.64 / 1.20,
 *                  512 x 128 x 8 3.15 / 3.44, 512 x 32 x 63 5.78 / 4.46,
 *                  768 x 128 x 8 6.8 / 8.3, 768 x 32 x 63 13.2 / 9.5,
 *                  1024 x 16 x 8 1.5 / 16.2, 1024 x 32 x 63 15.4 / 18.1,
 *                  1024 x 64 x 63 28.9 / 19.1
 *   8192 problems  64 x 16 x 8 2.10 / 2.11, 128 x 16 x 8 2.95 / 4.41,
 *                  128 x 8 x 31 5.93 / 4.30, 256 x 8 x 31 8.4 / 11.2,
 *                  256 x 16 x 31 12.2 / 11.7
 * A few problems alone, which two launches a step leave waiting, are faster by
 * the modes everywhere (16 of 256 x 8 x 31 0.80 / 0.37); the rule is on the
 * problem's own sizes, so that its price does not depend on its batch.  main's
 * strikes share one grid's modes, which are faster at every size (one strike on
 * 1024 x 4 x 7 0.18 / 0.12). */
int lvc_modes_pay(const lvc_problem *q) {
  const double nx = q->nx, rows = (double)q->ny * (double)(q->nt - 1);
  return nx <= 64.0 || (rows >= 2.25 * (nx - 48.0) && rows >= nx * nx / 300.0);
}

/* The normal call price in units of the standard deviation, struck d above
 * the mean (less than 1e-20 past 9). */
static double normal_call(double d) {
  if (!(d < 9.0))
    return d >= 9.0 ? 0.0 : d; /* a NaN stays one */
  return 0.3989422804014327 * exp(-0.5 * d * d) - 0.5 * d * erfc(0.7071067811865476 * d);
}

/* A floor of the price of an option of q's grid, over the spot, as far as it
 * takes to reach `enough`.  The chord
 * through the grid's ends, of which the modes take their sum, does not get
 * small where the price does, so what they leave of a far strike is rounding.
 * Given the volatility's path, x is the elastic process in the clock
 * V = integral of exp(2y - nu^2 t), stopped at the grid's ends: in u = the
 * integral of dx / x^beta a Brownian motion whose drift towards the strike is
 * minus the mean of beta/2 x^(beta-1), and the price at least strike^beta times
 * the normal call spread up to the grid's last node, less its image behind the
 * first.  V is at least
 * alpha^2 t times the geometric mean of the same path, whose logarithm is
 * normal, -nu^2 t / 2 with variance 4/3 nu^2 t; a price grows with V, so three
 * levels of it with the probabilities between them bound the mean.  Against
 * the scheme in 128 bits (19,000 prices, beta 0 .. 1.6, nu .01 .. 1.6, 6 .. 512
 * nodes): median 0.4 of the price, at most 1.5 times it in 99 % and 10 times on
 * grids of under 10 nodes at beta 1.5. */
static double price_floor(const lvc_problem *q, double strike, double xe, double enough) {
  static const double level[3] = {1.3, 0.3, -0.7}, weight[3] = {0.097, 0.285, 0.376};
  const double s0 = q->s0, beta = q->beta, inner = (s0 - strike) / s0;
  if (inner > 0.0)
    strike = s0;
  const double g = 1.0 - beta, sg = pow(s0, g);
  const int lognormal = fabs(g) < 1e-6;
  const double up = lognormal ? log(strike / s0) : (pow(strike, g) - sg) / g;
  const double end = lognormal ? log(xe / s0) : (pow(xe, g) - sg) / g;
  const double low = lognormal ? log(q->x0log / s0) : (pow(q->x0log, g) - sg) / g;
  const double drift =
      0.5 * beta * (strike > s0 * (1.0 + 1e-6) ? log(strike / s0) / up : sg / s0);
  const double root = sqrt(q->t), nt = q->nu * root, scale = pow(strike, beta) / s0;
  double sum = 0.0;
  for (int i = 0; i < 3 && !(scale * sum >= enough); i++) {
    const double sd = q->alpha * root * exp(nt * (level[i] / sqrt(3.0) - 0.25 * nt));
    const double m = drift * sd;
    const double v = normal_call(up / sd + m) - normal_call(end / sd + m) -
                     normal_call((up - 2.0 * low) / sd + m) +
                     normal_call((end - 2.0 * low) / sd + m);
    sum += v > 0.0 ? weight[i] * sd * v : v > -1.0 ? 0.0 : v; /* a NaN stays one */
  }
  return inner > scale * sum ? inner : scale * sum;
}

/* Whether the modes give the price of a strike on q's grid (lvc_modes_fit)
 * to the accuracy that the sweeps give it.  Their error is up to 10 ulp of the
 * spot times (x_N / x_1)^beta, the sweeps' a few ulp of the price itself, so the
 * rule is on the price's floor.  Error against 128 bits over the accepted ones
 * of the 19,000 prices above, modes / sweeps:
 *   FP64 (beta <= 0.7, floor 1/48 and (x_N / x_1)^beta / 250 of the spot):
 *     worst 8.5e-14 / 1.2e-13, 1 % above 2.7e-14 / 5.4e-14, rms 5.6e-15 / 1.2e-14,
 *     median 3.6e-16 / 1.5e-15; with beta up to 0.75 the worst is 2.1e-13
 *   f32 (2^-24 (x_N / x_1)^beta of the spot): before the price is rounded to f32,
 *     worst 3.0e-8, 0.1 % above 2.8e-9; the FP32 sweeps with refinement had a
 *     median of 6e-8 and a worst of 2.3e-6.
 * From the grid's last node on a price is exactly 0 either way. */
int lvc_modes_strike(const lvc_problem *q, double strike, int out_f64) {
  const double x0 = q->s0 - (double)q->xindex * q->dx;
  const double xe = (double)(q->nx - 1) * q->dx + x0;
  if (strike >= xe)
    return 1;
  if (out_f64 && !(q->beta <= 0.7))
    return 0;
  const double spread = pow((xe - q->dx) / (x0 + q->dx), q->beta);
  const double least = out_f64 ? fmax(1.0 / 48.0, spread / 250.0)
                               : 0x1p-24 * fmax(1.0, spread);
  return q->s0 - strike >= least * q->s0 || price_floor(q, strike, xe, least) >= least;
}

/* main's strike i (LocVolCalib.fut:247), in f32 for the f32 entry */
double lvc_main_strike(int i, int f32) {
  return f32 ? (double)(0.001f * (float)i) : 0.001 * (double)i;
}

/* How many of main's strikes, from the first, are below the grid's last node. */
static int strikes_inside(const lvc_problem *q, int f32) {
  const double xe = (double)(q->nx - 1) * q->dx - (double)q->xindex * q->dx + q->s0;
  const double n = 1000.0 * xe;
  int i = n < 2147483647.0 ? (int)n : INT32_MAX;
  while (i > 0 && lvc_main_strike(i - 1, f32) >= xe)
    i--;
  while (i < INT32_MAX && lvc_main_strike(i, f32) < xe)
    i++;
  return i;
}

/* Whether main's last strike within the grid is too far: then lvc_modes_far is
 * worth waiting for before the launches.  A strike within so many deviations of
 * the spot is not even looked at here (half a microsecond of a call of 40);
 * should it be far, it is found behind the launches. */
int lvc_modes_ends_far(const lvc_problem *q, int outer, int f32) {
  const int inside = strikes_inside(q, f32), last = outer < inside ? outer : inside;
  const double strike = lvc_main_strike(last > 0 ? last - 1 : 0, f32);
  if (strike - q->s0 < (f32 ? 8.0 : 0.5) * q->alpha * sqrt(q->t) * pow(q->s0, q->beta))
    return 0;
  return !lvc_modes_strike(q, strike, !f32);
}

/* main's options [*first, *end), of `outer`, that the modes leave to the
 * sweeps: above the last strike that a bisection finds accepted by
 * lvc_modes_strike (a price falls with the strike, so those below it are worth
 * more) to the grid's last node.  Which way an option goes does not depend on
 * `outer`. */
void lvc_modes_far(const lvc_problem *q, int outer, int f32, int *first, int *end) {
  const int inside = strikes_inside(q, f32);
  int near = -1, far = inside; /* options known to be near, and not */
  if (far > 0 && lvc_modes_strike(q, lvc_main_strike(far - 1, f32), !f32))
    near = far - 1;
  while (far - near > 1) {
    const int i = near + (far - near) / 2;
    if (lvc_modes_strike(q, lvc_main_strike(i, f32), !f32))
      near = i;
    else
      far = i;
  }
  *end = outer < inside ? outer : inside;
  *first = far < *end ? far : *end;
}

/* The lanes per mode of a column of ny rows, and how its rows lie in them. */
static int modes_kind(int ny, int32_t *lanes) {
  *lanes = ny <= 64 ? lvc_lanes_for(ny, 4) : ny <= 128 ? 16 : 64;
  return ny <= 64 ? LVC_MODES_ROW4 : ny <= 128 ? LVC_MODES_ROW8
                  : ny <= 256 ? LVC_MODES_WAVE4 : ny <= 512 ? LVC_MODES_WAVE8
                  : LVC_MODES_WAVE16;
}

static lvc_mgrid make_grid(const lvc_problem *q, int first, int count) {
  lvc_mgrid g;
  memset(&g, 0, sizeof(g));
  g.nx = q->nx;
  g.ny = q->ny;
  g.nt = q->nt;
  g.xindex = q->xindex;
  g.yindex = q->yindex;
  g.first = first;
  g.count = count;
  g.kind = modes_kind(q->ny, &g.lanes);
  g.s0 = q->s0;
  g.t = q->t;
  g.nu = q->nu;
  g.beta = q->beta;
  g.dx = q->dx;
  g.dy = q->dy;
  g.log_alpha = log(q->alpha);
  return g;
}

static int launch(struct futhark_context *ctx, hipStream_t stream, const lvc_modes_args *a,
                  int mode_tiles, int max_nx, const int64_t tiles[LVC_MODES_KINDS], int n,
                  void *out, int out_f64) {
  void *st = (void *)stream;
  int tok = lvc_prof_begin(ctx, "lvc_modes");
  int e = lvc_launch_modes(st, a, mode_tiles, max_nx);
  lvc_prof_end(ctx, tok);
  for (int kind = LVC_MODES_KINDS - 1; kind >= 0 && !e; kind--) {
    if (tiles[kind] == 0)
      continue;
    tok = lvc_prof_begin(ctx, "lvc_evolve");
    e = lvc_launch_evolve(st, a, kind, (int)tiles[kind]);
    lvc_prof_end(ctx, tok);
  }
  if (!e) {
    tok = lvc_prof_begin(ctx, "lvc_price");
    e = lvc_launch_price(st, a, n, out, out_f64);
    lvc_prof_end(ctx, tok);
  }
  return lvc_check_hip(ctx, e, "price kernels");
}

/* Doubles of work memory of main: lambda and f per mode, one coefficient per
 * mode and option. */
int64_t lvc_modes_main_work(int outer, int nx) {
  return 2 * align64(nx - 2) + (int64_t)outer * (nx - 2);
}

/* main's options on q's grid, strikes 0.001 * i: prices into out, those of the
 * options [far, far_end) left out. */
int lvc_modes_main(struct futhark_context *ctx, hipStream_t stream, const lvc_problem *q,
                   int outer, int far, int far_end, int strike_f32, double *work, void *out,
                   int out_f64) {
  lvc_modes_args a;
  memset(&a, 0, sizeof(a));
  a.one = make_grid(q, 0, outer);
  a.strike_f32 = strike_f32;
  a.far = far;
  a.far_end = far_end;
  const int modes = q->nx - 2, per = 64 / a.one.lanes;
  a.lambda = work;
  a.f = work + align64(modes);
  a.coef = work + 2 * align64(modes);
  int64_t tiles[LVC_MODES_KINDS] = {0};
  tiles[a.one.kind] = (modes + per - 1) / per;
  return launch(ctx, stream, &a, (modes + LVC_MODES_PER_WAVE - 1) / LVC_MODES_PER_WAVE, q->nx,
                tiles, outer, out, out_f64);
}

static int by_steps(const void *x, const void *y) {
  const int64_t a = *(const int64_t *)x, b = *(const int64_t *)y;
  return (a < b) - (a > b);
}

/* n problems (initGrid scalars set, lvc_modes_fit) on `stream` (ctx->stream, or
 * ctx->stream2 after lvc_fork), each one's price to out[out_index].  Runs of
 * consecutive problems that differ only in the strike share their modes.  `m`
 * keeps the device memory, for lvc_modes_release once ctx->stream has joined. */
int lvc_modes_batch(struct futhark_context *ctx, int beside, int n, const lvc_problem *probs,
                    void *out, int out_f64, lvc_modes_mem *m) {
  memset(m, 0, sizeof(*m));
  if (n == 0)
    return 0;
  /* the grids, then tiles counted per kind */
  lvc_mgrid *grids = malloc((size_t)n * sizeof(*grids));
  int64_t *order = malloc((size_t)n * sizeof(*order));
  if (!grids || !order) {
    free(grids);
    free(order);
    lvc_set_error(ctx, "host allocation failed");
    return 1;
  }
  int ng = 0, max_nx = 0;
  int64_t modes = 0, coefs = 0, nmode = 0, tiles[LVC_MODES_KINDS] = {0};
  for (int p = 0; p < n;) {
    int c = 1;
    while (p + c < n && lvc_same_factor(&probs[p], &probs[p + c]))
      c++;
    lvc_mgrid g = make_grid(&probs[p], p, c);
    const int m = g.nx - 2, per = 64 / g.lanes;
    g.mode0 = (int32_t)modes;
    g.coef_off = coefs;
    modes += m;
    coefs += (int64_t)c * m;
    nmode += (m + LVC_MODES_PER_WAVE - 1) / LVC_MODES_PER_WAVE;
    tiles[g.kind] += (m + per - 1) / per;
    if (g.nx > max_nx)
      max_nx = g.nx;
    order[ng] = (int64_t)g.nt << 32 | ng; /* most steps first */
    grids[ng++] = g;
    p += c;
  }
  if (modes > INT32_MAX) {
    free(grids);
    free(order);
    lvc_set_error(ctx, "batch too large");
    return 1;
  }
  qsort(order, (size_t)ng, sizeof(*order), by_steps);
  /* one upload: grids, strikes, tiles, each option's grid and output place */
  const size_t o_strikes = (size_t)ng * sizeof(lvc_mgrid);
  const size_t o_mode = o_strikes + (size_t)n * sizeof(double);
  size_t o_tiles[LVC_MODES_KINDS + 1] = {o_mode + (size_t)nmode * sizeof(lvc_mtile)};
  for (int i = 0; i < LVC_MODES_KINDS; i++)
    o_tiles[i + 1] = o_tiles[i] + (size_t)tiles[i] * sizeof(lvc_mtile);
  const size_t o_grid = o_tiles[LVC_MODES_KINDS];
  const size_t o_out = o_grid + (size_t)n * sizeof(int32_t);
  const size_t up = o_out + (size_t)n * sizeof(int32_t);
  const size_t work = (size_t)(2 * align64(modes) + coefs) * sizeof(double);
  char *h = malloc(up);
  int rc = !h;
  if (rc) {
    lvc_set_error(ctx, "host allocation failed");
  } else {
    memcpy(h, grids, o_strikes);
    lvc_mtile *mt = (lvc_mtile *)(h + o_mode), *et[LVC_MODES_KINDS];
    for (int i = 0; i < LVC_MODES_KINDS; i++)
      et[i] = (lvc_mtile *)(h + o_tiles[i]);
    for (int i = 0; i < ng; i++) {
      const int gi = (int)(order[i] & 0xffffffff);
      const lvc_mgrid *g = &grids[gi];
      const int m = g->nx - 2, per = 64 / g->lanes;
      for (int k = 0; k < m; k += LVC_MODES_PER_WAVE)
        *mt++ = (lvc_mtile){gi, k};
      for (int k = 0; k < m; k += per)
        *et[g->kind]++ = (lvc_mtile){gi, k};
      for (int p = g->first; p < g->first + g->count; p++) {
        ((double *)(h + o_strikes))[p] = probs[p].strike;
        ((int32_t *)(h + o_grid))[p] = gi;
        ((int32_t *)(h + o_out))[p] = probs[p].out_index;
      }
    }
    m->tables_bytes = up;
    m->work_bytes = work;
    rc = lvc_dev_alloc(ctx, up, &m->tables) || lvc_dev_alloc(ctx, work, &m->work) ||
         lvc_upload(ctx, m->tables, h, up) || (beside && lvc_fork(ctx));
  }
  if (!rc) {
    char *d = m->tables;
    double *w = m->work;
    lvc_modes_args a;
    memset(&a, 0, sizeof(a));
    a.grids = (const lvc_mgrid *)d;
    a.strikes = (const double *)(d + o_strikes);
    a.mode_tiles = (const lvc_mtile *)(d + o_mode);
    for (int i = 0; i < LVC_MODES_KINDS; i++)
      a.tiles[i] = (const lvc_mtile *)(d + o_tiles[i]);
    a.grid_of = (const int32_t *)(d + o_grid);
    a.out_index = (const int32_t *)(d + o_out);
    a.lambda = w;
    a.f = w + align64(modes);
    a.coef = w + 2 * align64(modes);
    m->forked = beside;
    rc = launch(ctx, beside ? ctx->stream2 : ctx->stream, &a, (int)nmode, max_nx, tiles, n, out,
                out_f64);
    if (!rc && lvc_debugging(ctx) && probs[0].out_index == 0) {
      lvc_mgrid g;
      rc = lvc_download(ctx, &g, a.grids, sizeof(g));
      if (!rc)
        lvc_note_index(ctx, g.yindex, g.xindex);
    }
  }
  free(h);
  free(grids);
  free(order);
  return rc;
}

/* Joins a batch that ran beside ctx->stream and gives its memory back. */
int lvc_modes_release(struct futhark_context *ctx, lvc_modes_mem *m) {
  const int rc = m->forked && lvc_join(ctx);
  lvc_dev_free(ctx, m->tables, m->tables_bytes);
  lvc_dev_free(ctx, m->work, m->work_bytes);
  memset(m, 0, sizeof(*m));
  return rc;
}
