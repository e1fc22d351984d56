/*
 * grs_nm_lanes.h -- the Nelder-Mead of grs_nm.h stepped by one wave inside a
 * kernel (k_com_nm, k_fit_nm).  Outside of HIP, __shfl and __shfl_xor are the
 * includer's (the tests run a wave's lanes as threads).
 */
#ifndef GRS_NM_LANES_H
#define GRS_NM_LANES_H

#include "grs_nm.h"

#ifdef __HIPCC__
#define GRS_NM_LANES_FN __device__ __forceinline__
#else
#define GRS_NM_LANES_FN inline
#endif

/* The steps of the method for N coordinates, taken by the 64 lanes of one
 * wave in registers: lane k holds coordinate k of the simplex, xbar and xr,
 * and every lane holds the values, counts and state and takes the method's
 * decisions on them.  The constructor and store() move the state between the
 * registers and the grs_nm in LDS around a step (so that it costs no registers
 * between steps), each one round of independent accesses; all loops are
 * unrolled over N.  The results are the sequential method's, bit for bit: its
 * statements for the coordinate, the stopping test's largest vertex distance
 * and largest coordinate reduced across the lanes (a maximum is exact), and
 * the stable insertion sort as exchanges of neighbours.  Stepped by one lane
 * on the grs_nm in LDS, one dependent access after the other, a step of six
 * coordinates with its follow-up took 11,900 cycles; three fits of six
 * coordinates went from 1.61 to 1.22 ms with this. */
template <int N>
struct nm_lanes {
  grs_nm *s;
  int k;
  bool on;
  double v[N + 1], fv[N + 1], xbar, xr, pend0, fxr;
  int nf, it, npend, max_fe, max_it;
  double tol_f, tol_x;
  grs_nm::State st;

  GRS_NM_LANES_FN nm_lanes(grs_nm *nm, int lane) : s(nm), k(lane < N ? lane : N - 1), on(lane < N) {
#pragma unroll
    for (int j = 0; j <= N; j++) {
      v[j] = s->v[j][k];
      fv[j] = s->fv[j];
    }
    xbar = s->xbar[k];
    xr = s->xr[k];
    pend0 = s->pend[0][k];
    fxr = s->fxr;
    nf = s->nf;
    it = s->it;
    npend = s->npend;
    max_fe = s->max_fe;
    max_it = s->max_it;
    tol_f = s->tol_f;
    tol_x = s->tol_x;
    st = s->st;
  }

  GRS_NM_LANES_FN void store() {
    if (on) {
#pragma unroll
      for (int j = 0; j <= N; j++) s->v[j][k] = v[j];
      s->xbar[k] = xbar;
      s->xr[k] = xr;
      s->pend[0][k] = pend0;
      if (st == grs_nm::SHRINK) {
#pragma unroll
        for (int j = 1; j <= N; j++) s->pend[j - 1][k] = v[j];
      }
    }
#pragma unroll
    for (int j = 0; j <= N; j++) s->fv[j] = fv[j];
    s->fxr = fxr;
    s->nf = nf;
    s->it = it;
    s->npend = npend;
    s->st = st;
  }

  /* largest of the N lanes' values (the lanes beyond repeat lane N - 1's) */
  GRS_NM_LANES_FN static double lanes_max(double x) {
    for (int off = 4; off > 0; off >>= 1) x = grs_nm_max(x, __shfl_xor(x, off, 64));
    return __shfl(x, 0, 64);
  }

  /* entry i into the sorted entries 0 .. i - 1 (stable, NaN last) */
  template <int I>
  GRS_NM_LANES_FN void insert() {
#pragma unroll
    for (int j = I - 1; j >= 0; j--) {
      const double a = fv[j], b = fv[j + 1];
      const bool sw = (b == b) && (a != a || a > b);
      fv[j] = sw ? b : a;
      fv[j + 1] = sw ? a : b;
      const double va = v[j], vb = v[j + 1];
      v[j] = sw ? vb : va;
      v[j + 1] = sw ? va : vb;
    }
  }

  template <int I = 1>
  GRS_NM_LANES_FN void sort() {
    insert<I>();
    if constexpr (I < N) sort<I + 1>();
  }

  GRS_NM_LANES_FN void begin() {
    GRS_NO_CONTRACT
    if (!(nf < max_fe && it < max_it)) {
      st = grs_nm::DONE;
      npend = 0;
      return;
    }
    double dfv = __builtin_nan(""), dx = __builtin_nan("");
#pragma unroll
    for (int j = 1; j <= N; j++) {
      dfv = grs_nm_max(dfv, fabs(fv[0] - fv[j]));
      dx = grs_nm_max(dx, fabs(v[j] - v[0]));
    }
    dx = lanes_max(dx);
    const double vmax = lanes_max(v[0]);
    if (dfv <= grs_nm_max(tol_f, 10.0 * grs_nm_eps(fv[0])) && dx <= grs_nm_max(tol_x, 10.0 * grs_nm_eps(vmax))) {
      st = grs_nm::DONE;
      npend = 0;
      return;
    }
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < N; j++) acc += v[j];
    xbar = acc / (double)N;
    xr = (1.0 + 1.0) * xbar - 1.0 * v[N];
    pend0 = xr;
    npend = 1;
    st = grs_nm::REFLECT;
  }

  /* the last entry replaced: it alone can be out of order */
  GRS_NM_LANES_FN void end_iter() {
    insert<N>();
    it += 1;
    begin();
  }

  GRS_NM_LANES_FN void shrink() {
    GRS_NO_CONTRACT
#pragma unroll
    for (int j = 1; j <= N; j++) v[j] = v[0] + 0.5 * (v[j] - v[0]);
    npend = N;
    st = grs_nm::SHRINK;
  }

  GRS_NM_LANES_FN void feed(const double *f) {
    GRS_NO_CONTRACT
    switch (st) {
      case grs_nm::INIT:
#pragma unroll
        for (int j = 0; j <= N; j++) {
          v[j] = s->pend[j][k];
          fv[j] = f[j];
        }
        nf = N + 1;
        sort();
        it = 1;
        begin();
        return;
      case grs_nm::REFLECT:
        fxr = f[0];
        nf += 1;
        if (fxr < fv[0]) {
          pend0 = GRS_NM_FOLLOW_UP(1, xbar, v[N]);
          npend = 1;
          st = grs_nm::EXPAND;
          return;
        }
        if (fxr < fv[N - 1]) {
          v[N] = xr;
          fv[N] = fxr;
          end_iter();
          return;
        }
        if (fxr < fv[N]) {
          pend0 = GRS_NM_FOLLOW_UP(2, xbar, v[N]);
          st = grs_nm::CONTRACT_OUT;
        } else {
          pend0 = GRS_NM_FOLLOW_UP(3, xbar, v[N]);
          st = grs_nm::CONTRACT_IN;
        }
        npend = 1;
        return;
      case grs_nm::EXPAND:
        nf += 1;
        if (f[0] < fxr) {
          v[N] = pend0;
          fv[N] = f[0];
        } else {
          v[N] = xr;
          fv[N] = fxr;
        }
        end_iter();
        return;
      case grs_nm::CONTRACT_OUT:
      case grs_nm::CONTRACT_IN:
        nf += 1;
        if (st == grs_nm::CONTRACT_OUT ? f[0] <= fxr : f[0] < fv[N]) {
          v[N] = pend0;
          fv[N] = f[0];
          end_iter();
        } else {
          shrink();
        }
        return;
      case grs_nm::SHRINK:
#pragma unroll
        for (int j = 1; j <= N; j++) fv[j] = f[j - 1];
        nf += N;
        sort();
        it += 1;
        begin();
        return;
      case grs_nm::DONE:
        return;
    }
  }

  /* a step with the values f (in LDS) of grs_nm's points: a reflection's
   * follow-ups stand behind its own value (without follow_ups: of the
   * requested points alone).  One call site of feed, so that it is inlined
   * and the state stays in registers. */
  GRS_NM_LANES_FN void step(const double *f, bool follow_ups = true) {
    for (int q = 0;;) {
      const bool refl = st == grs_nm::REFLECT;
      feed(f + q);
      if (!refl || !follow_ups) return;
      q = st == grs_nm::EXPAND ? 1 : st == grs_nm::CONTRACT_OUT ? 2 : st == grs_nm::CONTRACT_IN ? 3 : 0;
      if (q == 0) return;
    }
  }
};

#endif
