/*
 * grs_nm.h -- bounded Nelder-Mead as a resumable state: start, the points to
 * score, result.  The steps between are nm_lanes' (grs_nm_lanes.h).
 *
 * fminsearchbnd (fminsearchbnd.m:152-165 start point, :263-268 sine
 * transform for two-sided bounds) over MATLAB's fminsearch.  The method
 * (Lagarias, Reeds, Wright, Wright, SIAM J. Optim. 9 (1998) 112-147, with
 * fminsearch's documented constants) is restated here:
 *   simplex x0 and x0 with coordinate j scaled by 1.05 (0.00025 when 0),
 *   sorted by f (stable, NaN last), iteration count 1;
 *   loop while evaluations < MaxFunEvals and iterations < MaxIter; stop when
 *   max|f1-fj| <= max(TolFun, 10 eps(f1)) and max|vj-v1| <= max(TolX,
 *   10 eps(max(v1))) (max ignores NaN);
 *   xbar = (sum of the n best) / n; reflect 2 xbar - v_end; expand 3 xbar -
 *   2 v_end if the reflection beats the best; keep the reflection if it beats
 *   the second worst; else contract outside 1.5 xbar - 0.5 v_end (reflection
 *   beats the worst; kept if <= the reflection) or inside 0.5 xbar +
 *   0.5 v_end (kept if it beats the worst); otherwise shrink towards the best
 *   by 1/2; sort again.
 * The points of a request are scored in any order and their values fed back
 * together, so each fit follows the sequential method exactly.  sin/asin are
 * the engine's FP64 functions.  Everything is host and device code (and plain
 * C++ for the tests), with the same operations and so the same results.
 */
#ifndef GRS_NM_H
#define GRS_NM_H

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define GRS_NM_FN __host__ __device__
#else
#define GRS_NM_FN
#endif

#include <cmath>

#include "grs_math.h"

#define GRS_NM_NMAX 8

/* eps(x) of MATLAB: the spacing of doubles at |x| */
GRS_NM_FN static inline double grs_nm_eps(double x) {
  if (x != x) return x;
  x = fabs(x);
  if (__builtin_isinf(x)) return __builtin_nan("");
  if (x < 2.2250738585072014e-308) return 4.9406564584124654e-324;
  int e;
  frexp(x, &e);
  return ldexp(1.0, e - 53);
}

/* MATLAB max of two values: NaN ignored unless both are NaN */
GRS_NM_FN static inline double grs_nm_max(double a, double b) {
  if (a != a) return b;
  if (b != b) return a;
  return a > b ? a : b;
}

/* coordinate of the expansion (q = 1), the outside (2) and the inside
 * contraction (3) from the centroid's and the worst vertex's (a macro: as a
 * function, inlined, it cost k_com_nm 1%) */
#define GRS_NM_FOLLOW_UP(q, xbar, vn)          \
  ((q) == 1   ? (1.0 + 2.0) * (xbar) - 2.0 * (vn) \
   : (q) == 2 ? (1.0 + 0.5) * (xbar) - 0.5 * (vn) \
              : (1.0 - 0.5) * (xbar) + 0.5 * (vn))

struct grs_nm {
  enum State { INIT, REFLECT, EXPAND, CONTRACT_OUT, CONTRACT_IN, SHRINK, DONE };
  int n = 0;
  double lb[GRS_NM_NMAX], ub[GRS_NM_NMAX];
  int max_fe = 2000, max_it = 500;
  double tol_f = 1e-10, tol_x = 1e-4;
  double v[GRS_NM_NMAX + 1][GRS_NM_NMAX], fv[GRS_NM_NMAX + 1];
  double xbar[GRS_NM_NMAX], xr[GRS_NM_NMAX], fxr = 0.0;
  int nf = 0, it = 0;
  State st = DONE;
  int npend = 0;
  double pend[GRS_NM_NMAX + 1][GRS_NM_NMAX]; /* requested points, transformed (u) space */

  /* coordinate k of u -> x (fminsearchbnd.m:263-268) */
  GRS_NM_FN void xform1(const double *u, int k, double *xk) const {
    GRS_NO_CONTRACT
    double t = (grs_sin(u[k]) + 1.0) / 2.0;
    t = t * (ub[k] - lb[k]) + lb[k];
    *xk = fmax(lb[k], fmin(ub[k], t));
  }

  GRS_NM_FN void xform(const double *u, double *x) const {
    for (int k = 0; k < n; k++) xform1(u, k, &x[k]);
  }

  GRS_NM_FN void start(int dims, const double *x0, const double *lo, const double *hi) {
    GRS_NO_CONTRACT
    n = dims;
    double u0[GRS_NM_NMAX];
    for (int k = 0; k < n; k++) {
      lb[k] = lo[k];
      ub[k] = hi[k];
      if (x0[k] <= lb[k]) {
        u0[k] = -GRS_PI / 2.0;
      } else if (x0[k] >= ub[k]) {
        u0[k] = GRS_PI / 2.0;
      } else {
        double z = 2.0 * (x0[k] - lb[k]) / (ub[k] - lb[k]) - 1.0;
        z = z < -1.0 ? -1.0 : (z > 1.0 ? 1.0 : z);
        u0[k] = 2.0 * GRS_PI + grs_asin(z);
      }
    }
    for (int j = 0; j <= n; j++)
      for (int k = 0; k < n; k++)
        pend[j][k] = k != j - 1 ? u0[k] : (u0[k] != 0.0 ? (1.0 + 0.05) * u0[k] : 0.00025);
    npend = n + 1;
    st = INIT;
  }

  GRS_NM_FN bool done() const { return st == DONE; }

  /* the points to score: the requested ones, and with a reflection the three
   * that its value can lead to next (GRS_NM_FOLLOW_UP), so that an iteration
   * is one round; their values are used where the method goes on to request
   * them */
  GRS_NM_FN int points() const { return done() ? 0 : (st == REFLECT ? 4 : npend); }

  /* result in the original variables */
  GRS_NM_FN void result(double *x, double *fval) const {
    xform(v[0], x);
    *fval = fv[0];
  }
};

#endif /* GRS_NM_H */
