/*
 * grs_resolve.h -- deciding an event without the exact FP64 pipeline where
 * that is safe (device code of the scoring, pairing, G-vector matching and
 * centre-of-mass kernels).
 */
#ifndef GRS_RESOLVE_H
#define GRS_RESOLVE_H

#include "grs_internal.h"

/* P = S * [pos0, pos1 - RotAxisOffset, pos2] of a voxel: SamposW at omega is
 * Omega * P (forward_comp.m:17,22 up to the order of the products, which
 * only the exact pipeline needs). */
__device__ __forceinline__ void voxel_P(const grs_dgeo *g, const double *pos, double *P) {
  const double x = pos[0], y = pos[1] - g->RAO, z = pos[2];
  for (int i = 0; i < 3; i++) P[i] = __builtin_fma(g->S[3 * i], x, __builtin_fma(g->S[3 * i + 1], y, g->S[3 * i + 2] * z));
}

/* SamposW and the unit beam direction u = grainpos / |grainpos| at
 * (cos omega, sin omega), to a few 1e-15 relative (filters only). */
__device__ __forceinline__ void beam_terms(const grs_dgeo *g, const double *P, double c, double s, double *sw,
                                           double *u) {
  sw[0] = c * P[0] - s * P[1];
  sw[1] = s * P[0] + c * P[1];
  sw[2] = P[2];
  const double gp0 = g->Lss + sw[0], gp1 = (sw[1] - g->P0y) + g->RAO, gp2 = sw[2] - g->P0z;
  const double n2 = __builtin_fma(gp0, gp0, __builtin_fma(gp1, gp1, gp2 * gp2));
  double r = __builtin_amdgcn_rsq(n2);
  r = r * __builtin_fma(-0.5 * n2, r * r, 1.5);
  u[0] = gp0 * r;
  u[1] = gp1 * r;
  u[2] = gp2 * r;
}

/* Refined hardware reciprocal / reciprocal square root (one Newton step,
 * relative error below 5e-15): used only by the conservative filters, whose
 * margins are 1e-12 or wider. */
__device__ __forceinline__ double fast_rcp(double x) {
  double y = __builtin_amdgcn_rcp(x);
  return y * __builtin_fma(-x, y, 2.0);
}
__device__ __forceinline__ double fast_rsq(double x) {
  double y = __builtin_amdgcn_rsq(x);
  return y * __builtin_fma(-0.5 * x, y * y, 1.5);
}

/* Phase B1: resolve an event without the exact pipeline where that is safe.
 *
 * The spot position is recomputed from the same quantities through exact
 * identities -- sin(theta) = -cos(beta), cos(theta) = sqrt(1 - cos^2 beta),
 * lambda = -4 pi cos(beta) / |G|, sin(phix) = sqrt(1 - cos^2 phix),
 * sin(phix - 2 theta) by the difference formula -- with refined hardware
 * reciprocals (relative error below 5e-15).  Guards send ill-conditioned
 * events to the exact pipeline: |sin(phiy)| < 1e-3, |t denominator| < 1e-3,
 * |cos(phix)| > 0.99, G nearly along the beam.  Under the guards both this
 * value and the exact pipeline's are within about 1e-8 pixel of the true spot
 * position, so when the unrounded coordinate is at least GRS_RES_TAU (1e-4
 * pixel) from every half-integer the two round to the same pixel; the window
 * tests are decided here when cos(beta) and lambda clear their bounds by the
 * phase-A margins (1e-12 on cos(beta), 1e-9 lambda_max on lambda), either
 * way.  Everything else (and every NaN) returns 2 and goes
 * through the exact pipeline, so the decisions are those of forward_comp.m.
 * Returns 0 (not selected), 1 (selected, pixel in *dy, *dz) or 2 (exact). */
#define GRS_RES_TAU 1e-4

struct b1_out {
  double ry, rz;
  int32_t dy, dz;
  int32_t win; /* cleared by the caller; 1 once the event enters the spot construction */
};

__device__ __forceinline__ bool res_round(double r, double *k) {
  const double f = r + 0.5;
  const double fl = __builtin_floor(f);
  const double fr = f - fl;
  *k = fl;
  return (fr >= GRS_RES_TAU) & (fr <= 1.0 - GRS_RES_TAU);
}

/* the per (voxel, omega) terms of the spot construction (forward_comp.m:
 * 36-54): the beam direction u, k0 = Lsd - SamposW(1), d = center(2:3) -
 * SamposW(2:3) with center(2:3) = L u(2:3) / u0, L2 = (Lsd - SamposW(1)) /
 * u0 (cos(alpha) = u0), the t numerator and the offsets of the
 * tilted-detector intersection */
struct om_terms {
  double u0, u1, u2, k0, d1, d2, L2, tnum, ov1, ov2;
};

__device__ __forceinline__ void omega_terms(const grs_dgeo *g, const double *P, double c, double s, om_terms *w) {
  double swv[3], uv[3];
  beam_terms(g, P, c, s, swv, uv);
  const double iu0 = fast_rcp(uv[0]);
  w->u0 = uv[0];
  w->u1 = uv[1];
  w->u2 = uv[2];
  w->k0 = g->Lsd - swv[0];
  w->d1 = g->L * uv[1] * iu0 - swv[1];
  w->d2 = g->L * uv[2] * iu0 - swv[2];
  w->L2 = w->k0 * iu0;
  const double *R = g->R;
  w->tnum = __builtin_fma(R[0], w->k0, __builtin_fma(R[3], (g->dety00 - g->RAO) - swv[1], R[6] * (g->detz00 - swv[2])));
  w->ov1 = (swv[1] - g->dety00) + g->RAO;
  w->ov2 = swv[2] - g->detz00;
}

/* The unrounded spot coordinates of an event from cos(beta) = cb, its rotated
 * G (G1, G2; g2 = |G|^2) and the terms w; false where a guard sends it to
 * the exact pipeline.  STRAIGHT: no branches at the guards, which nearly
 * always hold; a branch at each keeps the loads and products behind it from
 * starting early (without them 1,024 voxels x 343 x 7.9 samples: 26.7 ->
 * 26.0 ms, 262,144 orientations of a voxel: 2.82 -> 2.73 ms, 24 fits: 1.39 ->
 * 1.27 ms).  It holds more registers, which costs a kernel that spills them
 * (k_gt_score: 3.4 -> 4.3 ms). */
template <bool STRAIGHT>
__device__ __forceinline__ bool b1_spot(const grs_dgeo *g, const om_terms &w, double G1, double G2, double cb,
                                        double g2, const double *thr, double *ry, double *rz) {
  const double omc = __builtin_fma(-cb, cb, 1.0);
  const double cth = omc * fast_rsq(omc);
  const double s2t = -2.0 * cb * cth;
  const double c2t = __builtin_fma(-2.0 * cb, cb, 1.0);
  const double nv2 = __builtin_fma(G1, G1, G2 * G2);
  bool ok = nv2 >= 1e-12 * g2;
  if (!STRAIGHT && !ok) return false;
  /* the remaining per (voxel, omega) terms from u and SamposW: center is
   * grainpos * L / grainpos(1), so center/|center| = u, center(2:3) =
   * L u(2:3) / u0, L2 = (Lsd - SW1) / u0 (cos(alpha) = u0); K_out(2:3) =
   * (dety22, detz22) - SamposW(2:3) = d + diffvec e; and the t numerator
   * and offsets of forward_comp.m:51-54 */
  const double k0 = w.k0, d1 = w.d1, d2 = w.d2, L2 = w.L2;
  const double *R = g->R;
  const double tnum = w.tnum;
  const double ov1 = w.ov1, ov2 = w.ov2;
  const double inv = fast_rsq(nv2);
  const double ap = __builtin_fma(G1, w.u1, G2 * w.u2) * inv;
  ok = ok & (__builtin_fabs(ap) <= 0.99);
  if (!STRAIGHT && !ok) return false;
  const double oma = __builtin_fma(-ap, ap, 1.0);
  const double sph = oma * fast_rsq(oma);
  const double sphy = __builtin_fma(sph, c2t, -ap * s2t);
  ok = ok & (__builtin_fabs(sphy) >= 1e-3);
  if (!STRAIGHT && !ok) return false;
  const double diffvec = L2 * s2t * fast_rcp(sphy);
  /* K_out = (Lsd, y22, z22) - SamposW unnormalised: t K_out is the same
   * vector for K_out and K_out / |K_out|, and the guard |R(:,1) . K_out| >=
   * 1e-3 |K_out| is taken squared */
  const double k1 = __builtin_fma(diffvec * G1, inv, d1);
  const double k2 = __builtin_fma(diffvec * G2, inv, d2);
  const double kk = __builtin_fma(k0, k0, __builtin_fma(k1, k1, k2 * k2));
  const double tden = __builtin_fma(R[0], k0, __builtin_fma(R[3], k1, R[6] * k2));
  ok = ok & (tden * tden >= 1e-6 * kk);
  if (!STRAIGHT && !ok) return false;
  const double t = tnum * fast_rcp(tden);
  const double w0 = __builtin_fma(t, k0, -k0), w1 = __builtin_fma(t, k1, ov1), w2 = __builtin_fma(t, k2, ov2);
  /* thr[6..11]: -R(:,2) / pixelysize and -R(:,3) / pixelzsize */
  *ry = __builtin_fma(thr[6], w0, __builtin_fma(thr[7], w1, __builtin_fma(thr[8], w2, g->dety0)));
  *rz = __builtin_fma(thr[9], w0, __builtin_fma(thr[10], w1, __builtin_fma(thr[11], w2, g->detz0)));
  return ok;
}

template <bool STRAIGHT>
__device__ __forceinline__ int b1_classify(const grs_dgeo *g, double c, double s, const double *P, const double *bt,
                                           const double *gt, const double *thr, b1_out *o) {
  om_terms w;
  if (bt) {
    /* the beam table row of this omega: the same values as omega_terms */
    w.u0 = bt[0];
    w.u1 = bt[1];
    w.u2 = bt[2];
    w.k0 = bt[3];
    w.d1 = bt[4];
    w.d2 = bt[5];
    w.L2 = bt[6];
    w.tnum = bt[7];
    w.ov1 = bt[8];
    w.ov2 = bt[9];
  } else {
    omega_terms(g, P, c, s, &w);
  }
  const double gw0 = gt[0], gw1 = gt[1], gw2 = gt[2];
  const double u0 = w.u0, u1 = w.u1, u2 = w.u2;
  const double G0 = c * gw0 - s * gw1, G1 = s * gw0 + c * gw1, G2 = gw2;
  /* |G| is invariant under the rotation: 1/|G| and |G|^2 of the reflection */
  const double rg = gt[3], g2 = gt[4];
  const double cb = __builtin_fma(u0, G0, __builtin_fma(u1, G1, u2 * G2)) * rg;
  const double lam = (-4.0 * GRS_PI) * cb * rg;
  /* outside the window by more than the margins: not selected */
  const bool outer = (cb < 1e-12) & (cb > thr[0]) & (lam > thr[1]) & (lam < thr[2]);
  const int out = ((cb == cb) & (lam == lam)) ? 0 : 2;
  if (!STRAIGHT && !outer) return out;
  /* inside by less than the margins: the exact pipeline decides */
  const bool inner = (cb < -1e-12) & (cb > thr[3]) & (lam > thr[4]) & (lam < thr[5]);
  o->win = outer & inner;
  if (!STRAIGHT && !inner) return 2;
  double ry, rz, ky, kz;
  bool ok = b1_spot<STRAIGHT>(g, w, G1, G2, cb, g2, thr, &ry, &rz);
  ok = ok & res_round(ry, &ky);
  ok = ok & res_round(rz, &kz);
  if (!STRAIGHT && !ok) return 2;
  /* ky, kz are the rounded pixel: floor(r + 0.5) equals round-half-away for
   * every r that is not a half-integer, and negative values are off anyway */
  const bool on = (ky >= 1.0) & (ky <= g->detysize) & (kz >= 1.0) & (kz <= g->detzsize);
  const bool stop = (ky >= g->bsy0) & (ky <= g->bsy1) & (kz >= g->bsz0) & (kz <= g->bsz1);
  o->ry = ry;
  o->rz = rz;
  o->dy = on ? (int32_t)ky : 0;
  o->dz = on ? (int32_t)kz : 0;
  const int in = (inner & ok) ? ((on & !stop) ? 1 : 0) : 2;
  return outer ? in : out;
}

/* b1_classify's thresholds: the window with the outer, then the inner margins,
 * and the detector rows scaled to pixels */
__device__ __forceinline__ void b1_thresholds(const grs_dgeo *g, double *thr) {
  const double lm = 1e-9 * g->lambda_max;
  thr[0] = g->cos_beta_max - 1e-12;
  thr[1] = g->lambda_min - lm;
  thr[2] = g->lambda_max + lm;
  thr[3] = g->cos_beta_max + 1e-12;
  thr[4] = g->lambda_min + lm;
  thr[5] = g->lambda_max - lm;
  for (int k = 0; k < 3; k++) {
    thr[6 + k] = -g->R[3 * k + 1] * g->ipy;
    thr[9 + k] = -g->R[3 * k + 2] * g->ipz;
  }
}

#endif
