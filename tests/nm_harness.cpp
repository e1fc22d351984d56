/*
 * Host-side driver of the engine's Nelder-Mead for the CPU tests: the state
 * of grs_nm.h is stepped by nm_lanes (grs_nm_lanes.h), the code that the
 * kernels run, with the lanes of a wave as threads and an objective given by
 * the caller (a ctypes callback).  A step's cross-lane operations stay within
 * 8 lanes.  Plain C++, built by tests/test_nm_kat.py.
 */
#include <pthread.h>

#include <cstring>
#include <thread>

#include "grs_nm.h"

#define LANES 8

/* the lanes' exchange: every lane leaves its value, then reads another's */
static thread_local int g_lane;
static double g_slot[LANES];
static pthread_barrier_t g_meet;

static double exchange(double x, int from) {
  g_slot[g_lane] = x;
  pthread_barrier_wait(&g_meet);
  const double y = g_slot[from];
  pthread_barrier_wait(&g_meet);
  return y;
}
static double __shfl_xor(double x, int mask, int) { return exchange(x, g_lane ^ mask); }
static double __shfl(double x, int lane, int) { return exchange(x, lane); }

#include "grs_nm_lanes.h"

typedef double (*nm_objective)(const double *u, int n);

/* one step of the wave on the values of all points, or of the requested ones
 * alone */
template <int N>
static void wave_step(grs_nm *s, const double *f, bool follow_ups) {
  pthread_barrier_init(&g_meet, nullptr, LANES);
  std::thread lane[LANES];
  for (int l = 0; l < LANES; l++)
    lane[l] = std::thread([=]() {
      g_lane = l;
      nm_lanes<N> L(s, l);
      L.step(f, follow_ups);
      /* the lanes store one after the other */
      for (int t = 0; t < LANES; t++) {
        pthread_barrier_wait(&g_meet);
        if (t == l) L.store();
      }
    });
  for (int l = 0; l < LANES; l++) lane[l].join();
  pthread_barrier_destroy(&g_meet);
}

static void step(grs_nm *s, const double *f, bool follow_ups) {
  switch (s->n) {
    case 1: return wave_step<1>(s, f, follow_ups);
    case 2: return wave_step<2>(s, f, follow_ups);
    case 3: return wave_step<3>(s, f, follow_ups);
    case 4: return wave_step<4>(s, f, follow_ups);
    case 5: return wave_step<5>(s, f, follow_ups);
    case 6: return wave_step<6>(s, f, follow_ups);
    case 7: return wave_step<7>(s, f, follow_ups);
    default: return wave_step<8>(s, f, follow_ups);
  }
}

static void start_simplex(grs_nm *s, int n, const double *sim0, int max_fe, int max_it, double tol_f, double tol_x) {
  s->n = n;
  for (int k = 0; k < n; k++) {
    s->lb[k] = -1.0;
    s->ub[k] = 1.0;
  }
  s->max_fe = max_fe;
  s->max_it = max_it;
  s->tol_f = tol_f;
  s->tol_x = tol_x;
  for (int j = 0; j <= n; j++)
    for (int k = 0; k < n; k++) s->pend[j][k] = sim0[j * n + k];
  s->npend = n + 1;
  s->st = grs_nm::INIT;
}

/* coordinate k of point q, as the kernels form it */
static double point(const grs_nm &s, int q, int k) {
  return s.st == grs_nm::REFLECT && q > 0 ? GRS_NM_FOLLOW_UP(q, s.xbar[k], s.v[s.n][k]) : s.pend[q][k];
}

static void end_simplex(const grs_nm &s, double *sim_out, double *fv_out, int *nf, int *it) {
  for (int j = 0; j <= s.n; j++) {
    fv_out[j] = s.fv[j];
    for (int k = 0; k < s.n; k++) sim_out[j * s.n + k] = s.v[j][k];
  }
  *nf = s.nf;
  *it = s.it;
}

/* the states agree bit for bit in everything a later step reads */
static bool same_state(const grs_nm &a, const grs_nm &b) {
  bool same = a.st == b.st && a.nf == b.nf && a.it == b.it && a.npend == b.npend;
  const size_t row = sizeof(double) * (size_t)a.n;
  for (int j = 0; j <= a.n; j++) same = same && !memcmp(a.v[j], b.v[j], row) && !memcmp(&a.fv[j], &b.fv[j], sizeof(double));
  for (int j = 0; j < a.npend; j++) same = same && !memcmp(a.pend[j], b.pend[j], row);
  if (a.st == grs_nm::REFLECT) same = same && !memcmp(a.xbar, b.xbar, row) && !memcmp(a.xr, b.xr, row);
  return same;
}

extern "C" {

/* fminsearch's iteration from an explicit starting simplex sim0 ((n+1) x n,
 * row-major), objective in the transformed variables; every point is
 * evaluated when the method requests it. */
int nm_run_simplex(int n, const double *sim0, int max_fe, int max_it, double tol_f, double tol_x, nm_objective f,
                   double *sim_out, double *fv_out, int *nf, int *it) {
  if (n < 1 || n > GRS_NM_NMAX) return -1;
  grs_nm s;
  start_simplex(&s, n, sim0, max_fe, max_it, tol_f, tol_x);
  double vals[GRS_NM_NMAX + 1];
  while (!s.done()) {
    for (int j = 0; j < s.npend; j++) vals[j] = f(s.pend[j], n);
    step(&s, vals, false);
  }
  end_simplex(s, sim_out, fv_out, nf, it);
  return 0;
}

/* The same iteration driven as the kernels drive it: every requested
 * reflection is evaluated together with its three follow-ups (grs_nm::points)
 * and a step takes what the method goes on to request from those values.  A
 * second state requests and is fed point by point: -2 if the two ever differ,
 * or if a request is not the follow-up evaluated for it.  fed receives the
 * points fed to the method, in order (up to fed_cap of them); hits[0..2] count
 * the expansions, outside and inside contractions taken from the follow-ups. */
int nm_run_follow_ups(int n, const double *sim0, int max_fe, int max_it, double tol_f, double tol_x, nm_objective f,
                      double *sim_out, double *fv_out, int *nf, int *it, double *fed, int fed_cap, int *n_fed,
                      int *hits) {
  if (n < 1 || n > GRS_NM_NMAX) return -1;
  grs_nm s, one;
  start_simplex(&s, n, sim0, max_fe, max_it, tol_f, tol_x);
  start_simplex(&one, n, sim0, max_fe, max_it, tol_f, tol_x);
  double u[GRS_NM_NMAX + 1][GRS_NM_NMAX], vals[GRS_NM_NMAX + 1];
  *n_fed = 0;
  hits[0] = hits[1] = hits[2] = 0;
  auto log_fed = [&](const double *p) {
    if (*n_fed < fed_cap)
      for (int k = 0; k < n; k++) fed[*n_fed * n + k] = p[k];
    *n_fed += 1;
  };
  while (!s.done()) {
    const int np = s.points();
    for (int q = 0; q < np; q++) {
      for (int k = 0; k < n; k++) u[q][k] = point(s, q, k);
      vals[q] = f(u[q], n);
    }
    const bool refl = s.st == grs_nm::REFLECT;
    step(&s, vals, true);
    for (int j = 0; j < one.npend; j++) log_fed(one.pend[j]);
    step(&one, vals, false);
    const int q = !refl ? 0 : one.st == grs_nm::EXPAND ? 1 : one.st == grs_nm::CONTRACT_OUT ? 2 : one.st == grs_nm::CONTRACT_IN ? 3 : 0;
    if (q) {
      if (memcmp(one.pend[0], u[q], sizeof(double) * (size_t)n)) return -2;
      hits[q - 1] += 1;
      log_fed(one.pend[0]);
      step(&one, vals + q, false);
    }
    if (!same_state(s, one)) return -2;
  }
  end_simplex(s, sim_out, fv_out, nf, it);
  return 0;
}

/* The starting simplex fminsearchbnd builds for x0 within [lb, ub]. */
int nm_start(int n, const double *x0, const double *lb, const double *ub, double *sim_out) {
  if (n < 1 || n > GRS_NM_NMAX) return -1;
  grs_nm s;
  s.start(n, x0, lb, ub);
  for (int j = 0; j <= n; j++)
    for (int k = 0; k < n; k++) sim_out[j * n + k] = s.pend[j][k];
  return 0;
}

/* Whole fminsearchbnd with the objective in the original variables, with the
 * kernels' rounds of points. */
int nm_fminsearchbnd(int n, const double *x0, const double *lb, const double *ub, int max_fe, int max_it,
                     double tol_f, double tol_x, nm_objective f, double *x, double *fval, int *nf, int *it) {
  if (n < 1 || n > GRS_NM_NMAX) return -1;
  grs_nm s;
  s.max_fe = max_fe;
  s.max_it = max_it;
  s.tol_f = tol_f;
  s.tol_x = tol_x;
  s.start(n, x0, lb, ub);
  double vals[GRS_NM_NMAX + 1], u[GRS_NM_NMAX], xx[GRS_NM_NMAX];
  while (!s.done()) {
    for (int q = 0; q < s.points(); q++) {
      for (int k = 0; k < n; k++) u[k] = point(s, q, k);
      s.xform(u, xx);
      vals[q] = f(xx, n);
    }
    step(&s, vals, true);
  }
  s.result(x, fval);
  *nf = s.nf;
  *it = s.it;
  return 0;
}

}  // extern "C"
