/*
 * grs_com.hip -- the objective of fit_grain_COM.m on the GPU.
 *
 * fit_grain_COM_fun (fit_grain_COM.m:32-89) for x = [position (mm), ZXZ
 * Euler angles (degrees)]: for every paired spot of the grain the event of
 * its (hkl, omega) is forward-simulated from pos = [x1, x2-RotAxisOffset,
 * x3] and U = euler2u(x(4:6)) through the forward_comp.m statements
 * (grs_event_pixel; its shortcut b1_spot where that rounds to the same
 * pixel), its pixel rounded, and the distance to the measured centroid
 * (columns 19:20 of the pair row) taken; ErrMean is the mean.
 * k_com_nm runs fminsearchbnd's Nelder-Mead for each grain inside the
 * kernel (one block per grain, its first wave stepping the method with one
 * lane per coordinate), so a fit costs no host round trip per simplex step.
 */
#include <hip/hip_runtime.h>

#include "grs_internal.h"
#include "grs_nm.h"
#include "grs_nm_lanes.h"
#include "grs_resolve.h"

/* cos/sin of every pair row's omega (column 17), once per call */
__global__ __launch_bounds__(256) void k_com_prep(const double *rows, int64_t total, double *cs) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < total) grs_omega_cs(rows[23 * i + 16], &cs[2 * i], &cs[2 * i + 1]);
}

/* distance of one pair row r to its event simulated at x (SUB of x's U, cs
 * the cos/sin of the row's omega): the exact pipeline */
__device__ static __noinline__ double com_pair_exact(const grs_dgeo *g, const double *r, const double *xp,
                                                     const double *SUB, double c, double s) {
  GRS_NO_CONTRACT
  grs_vw v;
  grs_vw_terms(g, xp, c, s, &v);
  double gw[3], Gt[3], Glen;
  grs_Gw(SUB, r + 12, gw);
  grs_Gt(v.c, v.s, gw[0], gw[1], gw[2], Gt);
  const double beta = grs_event_beta(&v, Gt, &Glen);
  double ry, rz;
  grs_event_pixel(g, &v, Gt, Glen, beta, &ry, &rz);
  const double ey = grs_round(ry) - r[17], ez = grs_round(rz) - r[18];
  return grs_sqrt(ey * ey + ez * ez);
}

/* The same distance.  Only the rounded pixel enters it, so the spot comes
 * from the identities and reciprocals of b1_spot where its coordinates
 * clear every half-integer by 1e-5 (the exact pipeline's are within 5e-7
 * pixel of them while both stay below 1e5 pixels: the guards leave
 * relative errors of 5e-12); everything else, NaN included, goes through the
 * exact pipeline.  The margin is smaller than k_fast's because one event in the exact pipeline
 * delays the whole round: at 1e-4 every other round had one. */
__device__ __forceinline__ bool com_round(double r, double *k) {
  const double f = r + 0.5, fl = __builtin_floor(f), fr = f - fl;
  *k = fl;
  return fr >= 1e-5 && fr <= 1.0 - 1e-5;
}

__device__ __forceinline__ double com_pair_dist(const grs_dgeo *g, const double *thr, const double *r,
                                                const double *xp, const double *P, const double *SUB,
                                                const double *cs) {
  const double c = cs[0], s = cs[1];
  om_terms w;
  omega_terms(g, P, c, s, &w);
  double gw[3];
  grs_Gw(SUB, r + 12, gw);
  const double G0 = c * gw[0] - s * gw[1], G1 = s * gw[0] + c * gw[1], G2 = gw[2];
  const double g2 = __builtin_fma(gw[0], gw[0], __builtin_fma(gw[1], gw[1], gw[2] * gw[2]));
  const double cb = __builtin_fma(w.u0, G0, __builtin_fma(w.u1, G1, w.u2 * G2)) * fast_rsq(g2);
  double ry, rz, ky, kz;
  if (__builtin_fabs(cb) <= 0.99 && b1_spot<true>(g, w, G1, G2, cb, g2, thr, &ry, &rz) && __builtin_fabs(ry) <= 1e5 &&
      __builtin_fabs(rz) <= 1e5 && com_round(ry, &ky) && com_round(rz, &kz)) {
    GRS_NO_CONTRACT
    const double ey = ky - r[17], ez = kz - r[18];
    return grs_sqrt(ey * ey + ez * ez);
  }
  return com_pair_exact(g, r, xp, SUB, c, s);
}

#define COM_THREADS 512

/* values of the (point, pair) distances kept in LDS (as one sequential sum
 * waits on every load of them); more pairs than fit use device memory */
#define COM_LDS_DIST 6144

/* pairs up to which a reflection is evaluated together with its follow-ups:
 * a round then takes about as long for four points as for one; beyond, the
 * distances of the two or three points that the method does not request cost more
 * than the rounds saved.  Three fits, with and without, in ms: 373 pairs 1.61
 * and 1.76, 724 2.80 and 2.84, 746 2.43 and 2.49, 1,119 3.42 and 3.25, 1,448 5.77 and
 * 4.52, 2,984 9.74 and 7.16; one of 20,000 474 and 240. */
#define COM_FOLLOW_PAIRS 1024

/* One block per fit m: the first wave steps the Nelder-Mead state machine
 * (started on the host) in registers (nm_lanes); for the requested points - up
 * to COM_FOLLOW_PAIRS pairs a reflection together with the three points its
 * value can lead to (grs_nm::points), so that an iteration is one round - the
 * point coordinates and the six cosines and sines of each point's angles are
 * computed one per thread, the first threads build each point's U and SUB,
 * all threads compute the (point, pair) distances, and thread p adds point
 * p's distances in pair order, so ErrMean is the sequential sum over the
 * count.  Bound: the chain of one round (trigonometry, distances, the
 * sequential sum of a few hundred values, the simplex step).  Three grains of
 * about 400 pairs: 1.2 ms for the launch; 1.6 with the simplex stepped in
 * LDS; 2.4 with also the exact pipeline for every distance, the distances
 * in device memory and a round per requested point.  The state machine ends
 * after at most max_iter iterations, so every block exits. */
__global__ __launch_bounds__(COM_THREADS) void k_com_nm(const grs_dgeo *g, const double *rows, const int64_t *rptr,
                                                        const double *cs, double *dis, grs_nm *nms) {
  GRS_NO_CONTRACT
  __shared__ __align__(16) unsigned char nm_buf[sizeof(grs_nm)];
  __shared__ double xs[GRS_NM_NMAX + 1][6];
  __shared__ double Ps[GRS_NM_NMAX + 1][3];
  __shared__ double sub[GRS_NM_NMAX + 1][9];
  __shared__ double trig[GRS_NM_NMAX + 1][6];
  __shared__ double fs[GRS_NM_NMAX + 1];
  __shared__ double ldist[COM_LDS_DIST];
  __shared__ double thr[12];
  __shared__ grs_dgeo sg;
  __shared__ int npts;
  grs_nm *nm = reinterpret_cast<grs_nm *>(nm_buf);
  const int t = threadIdx.x;
  const int64_t m = blockIdx.x;
  const int64_t r0 = rptr[m];
  const int n = (int)(rptr[m + 1] - r0);
  const bool follow_ups = n <= COM_FOLLOW_PAIRS;
  if (t == 0) {
    *nm = nms[m];
    sg = *g;
    b1_thresholds(&sg, thr);
  }
  __syncthreads();
  for (;;) {
    if (t == 0) npts = follow_ups ? nm->points() : nm->npend;
    __syncthreads();
    const int np = npts;
    if (np == 0) break;
    if (t < 6 * np) { /* one coordinate per thread, with the cos and sin of an angle */
      const int p = t / 6, k = t - 6 * p;
      double u = nm->pend[p][k];
      if (nm->st == grs_nm::REFLECT && p > 0) {
        const double xb = nm->xbar[k], vn = nm->v[nm->n][k];
        u = GRS_NM_FOLLOW_UP(p, xb, vn);
      }
      double u6[6], x;
      u6[k] = u;
      nm->xform1(u6, k, &x);
      xs[p][k] = x;
      if (k >= 3) {
        const double a = grs_deg2rad(x);
        trig[p][2 * (k - 3)] = grs_cos(a);
        trig[p][2 * (k - 3) + 1] = grs_sin(a);
      }
    }
    __syncthreads();
    if (t < np) {
      double U[9];
      grs_U_from_trig(trig[t][0], trig[t][1], trig[t][2], trig[t][3], trig[t][4], trig[t][5], U);
      grs_SUB(g, U, sub[t]);
    } else if (t >= 64 && t < 64 + np) {
      voxel_P(&sg, xs[t - 64], Ps[t - 64]);
    }
    __syncthreads();
    const bool local = np * n <= COM_LDS_DIST;
    double *dm = dis + (GRS_NM_NMAX + 1) * r0;
    for (int w = t; w < np * n; w += COM_THREADS) {
      const int p = w / n, i = w - p * n;
      const double d = com_pair_dist(&sg, thr, rows + 23 * (r0 + i), xs[p], Ps[p], sub[p], cs + 2 * (r0 + i));
      if (local) ldist[w] = d;
      else dm[w] = d;
    }
    __syncthreads();
    if (t < np) {
      /* loads 16 ahead of the in-order additions */
      auto sum = [n](const double *d) {
        double acc = 0.0;
        int i = 0;
        for (; i + 16 <= n; i += 16) {
          double b[16];
#pragma unroll
          for (int k = 0; k < 16; k++) b[k] = d[i + k];
#pragma unroll
          for (int k = 0; k < 16; k++) acc = acc + b[k];
        }
        for (; i < n; i++) acc = acc + d[i];
        return acc;
      };
      fs[t] = (local ? sum(ldist + t * n) : sum(dm + t * n)) / (double)n;
    }
    __syncthreads();
    if (t < 64) { /* the first wave steps the method */
      nm_lanes<6> L(nm, t);
      L.step(fs, follow_ups);
      L.store();
    }
    __syncthreads();
  }
  if (t == 0) nms[m] = *nm;
}

hipError_t grs_launch_com_nm(const grs_dgeo *d_g, const double *d_rows, const int64_t *d_rptr, int64_t M,
                             int64_t total, double *d_cs, double *d_dis, grs_nm *d_nm, hipStream_t st) {
  if (M <= 0) return hipSuccess;
  if (M > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_com_prep, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, d_rows, total, d_cs);
  hipLaunchKernelGGL(k_com_nm, dim3((unsigned)M), dim3(COM_THREADS), 0, st, d_g, d_rows, d_rptr, d_cs, d_dis, d_nm);
  return hipGetLastError();
}
