/*
 * grs_kernels.hip -- gfx950 kernels of the completeness-scoring engine.
 *
 * Hot path: for every evaluation (voxel, orientation) and every event
 * (omega, hkl) decide whether the reflection lands on the detector
 * (forward_comp.m:28-65), look the pixel up in the distance stack
 * (forward_comp.m:69-72) and reduce the integer counts and the median
 * distance (forward_comp.m:67, 86-90).
 *
 * k_fast  -- one 64-wide wavefront per evaluation (two or four share one in
 *            small launches).
 *   solve:   with uniform rotation angles each reflection's candidate ranges
 *            of omega are solved for (om_ranges) and go straight to phase B1.
 *   phase A: otherwise lanes walk the flattened (omega, hkl) event space 64 events at a
 *            time and apply a conservative Bragg/wavelength filter that only
 *            needs 4 multiplies and 3 FMAs per event; it rejects an event only
 *            when the exact test is proven to fail (margins 1e-12 on cos(beta),
 *            1e-9 relative on lambda, far above the FP64 rounding of the exact
 *            path).  Survivors are compacted into a 128-slot LDS ring with
 *            ballot + mbcnt.
 *   phase B1: whenever 64 survivors are queued the wave recomputes their
 *            spot positions through exact identities and refined hardware
 *            reciprocals (b1_classify) and decides every event whose pixel
 *            and window tests are unambiguous by a wide margin; the rest
 *            (about 1e-4 of them) are queued for
 *   phase B2: the exact FP64 event pipeline of forward_comp.m, 64 at a time.
 *   gather:  selected events are queued as stack indices; 64 at a time the
 *            wave gathers their distance keys (or hit bits), consumed one
 *            batch later, and counts hits with ballot/popcount.
 *   median : selected keys go to a per-wave list in HBM; the median is found
 *            by a 32-step radix bisection over the keys held in registers.
 *   Decisions are those of the exact pipeline, so the counts are bit-exact.
 *
 * k_plain -- the straightforward port: one thread per evaluation, the whole
 *   event pipeline for every event, per-thread key list and quickselect.
 *   It is the denominator of the batched-vs-plain speedup.
 */
#include <hip/hip_runtime.h>

#include "grs_internal.h"
#include "grs_nm_lanes.h"
#include "grs_resolve.h"

#define GRS_WPB 8      /* largest number of waves per block of k_fast (the launch chooses 1, 2, 4 or 8) */
#ifndef GRS_FAST_MIN_WAVES
#define GRS_FAST_MIN_WAVES 4 /* resident waves per SIMD k_fast is compiled for (128 VGPRs) */
#endif
#define GRS_QCAP 128   /* LDS ring slots per wave */
#define GRS_GWT 5      /* doubles per hkl row in LDS: G (3), 1/|G|, |G|^2 */
#define GRS_RING_DOUBLES (3 * GRS_QCAP * 4 / 8) /* three u32 rings per wave */
#define GRS_RANGE_DOUBLES(H) (4 * (int64_t)(H) + 1) /* 8H + 2 u32: omega-solve ranges */
#define GRS_REG_KEYS 16 /* keys per lane kept in registers for the median */

/* LDS doubles of one wave's region of k_fast: the G table, the rings, the
 * omega-solve ranges, S*pos of the voxel (4) and S*U*B (9) */
__host__ __device__ inline int64_t fast_wave_doubles(int32_t H) {
  return (int64_t)H * GRS_GWT + GRS_RING_DOUBLES + GRS_RANGE_DOUBLES(H) + 4 + 9;
}

/* k_fast's static LDS: the geometry, the thresholds of b1_classify and a
 * team's counters, rounded up */
#define GRS_FAST_STATIC_LDS ((int64_t)((sizeof(grs_dgeo) + 12 * sizeof(double) + 3 * sizeof(int32_t) + 127) / 128 * 128))

/* LDS doubles of the one-voxel beam table behind the wave regions: the
 * table is kept when the block's LDS stays within 160 KB (one CU's
 * LDS; with 8 waves per block two blocks, 16 waves, share a CU) */
__host__ __device__ inline int64_t fast_tab_doubles(int32_t map, int32_t nrot, int32_t H, int wpb) {
  if (map != GRS_MAP_ONE_VOXEL || nrot <= 0) return 0;
  const int64_t t = (int64_t)GRS_BT * nrot;
  return ((int64_t)wpb * fast_wave_doubles(H) + t) * (int64_t)sizeof(double) <= 163840 - GRS_FAST_STATIC_LDS ? t : 0;
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint32_t lane_prefix(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
  for (int off = 32; off >= 1; off >>= 1) {
    uint32_t o = (uint32_t)__shfl_xor((int)v, off, 64);
    v = o < v ? o : v;
  }
  return v;
}

__device__ __forceinline__ float key_to_float(uint32_t k) { return __uint_as_float(k); }

/* ---------------------------------------------------------------------- */
/* small set-up kernels                                                    */

__global__ void k_omega_cs(const double *rot, int32_t nrot, double *cs) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nrot) return;
  double c, s;
  grs_omega_cs(rot[i], &c, &s);
  cs[2 * i] = c;
  cs[2 * i + 1] = s;
}

__global__ void k_voxel_pos(const double *rows, int64_t M, int32_t stride, const double *p1, double *pos) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  const double *r = rows + i * stride;
  grs_voxel_pos(r[0], r[1], r[2], p1, pos + 3 * i);
}

/* Per-voxel bounds of the omega-solve candidate filter (GRS_VB doubles per
 * voxel).  With u(omega) the unit beam direction at the voxel
 * (grainpos / norm(grainpos), forward_comp.m:26) and P = S*pos' (RotAxisOffset
 * taken off pos(2)), the first-order beam direction has
 * u1 ~ al sin(omega) + be cos(omega) + ga with al = P0/Lss, be = P1/Lss,
 * ga = (RotAxisOffset - P0y)/Lss; u0 ~ 1 and u2 varies only through the norm.
 *   vb[0] W  >= max |u0 - 1| + max |u1 - (al sin + be cos + ga)| + hypot(al, be)/2
 *   vb[1], vb[2]  min and max of u2 (widened by 1e-12)
 *   vb[3] K  >= sin^2(theta) = cos^2(beta) of every event that can reach the
 *            detector; 1 (no bound) when a detector corner is 90 degrees or
 *            more off the beam or when the window admits
 *            2 theta + angle(u, x) >= pi/2 - 1e-3
 *   vb[4..6] al, be, ga
 *   vb[7], vb[8]  Zt >= and Zb <= the detector rows term of every event
 *            (below); +-1e300 (no bound) where K is 1
 *   vb[9], vb[10], vb[11] sin(eta), cos(eta), tan(eta): eta >= asin |e . u|
 *   vb[12] Ya >= |Yb|, |Yt|, the detector columns term of every event
 *            (below); 1e300 (no bound) where K is 1
 *   vb[13] delta >= |u - (1, 0, 0)|
 * All extremes are over the rotation angles the scorer visits, so they hold
 * at every event.  Corners are the detector corners 2 pixels outside the
 * pixel area (g->corner, frame of SamposW).
 *
 * Spot geometry (forward_comp.m:40-50).  center - grainpos = L2 u
 * (L2 = (Lsd - SW1)/u0) and dety22/detz22 add diffvec e, e = (0, Gt2, Gt3)
 * / konst, so in the frame of grainpos the triangle (voxel, center, spot)
 * has the angle 2 theta at the voxel: phix = acos(e . u) and
 * phiy = phix - 2 theta are its other angles, and diffvec =
 * L2 sin(2 theta) / sin(phiy).  K_out (:49) takes the voxel as SamposW and
 * the spot as (Lsd, dety22, detz22), which differ from that frame by
 * o = (0, RotAxisOffset - P0y, -P0z):
 *   K_out ~ L2 u + diffvec e + o.
 * The tilted-detector spot (:51-55) lies on the ray SamposW + t K_out.
 * Cone: |L2 u + diffvec e| >= L2 sqrt(1 - a^2), a = e . u, |a| <=
 * |(u1, u2)|, so K_out is within eps = asin(|o| / (L2 sqrt(1 - a^2))) of
 * the triangle's side and 2 theta <= gamma + eps, gamma the largest angle
 * between u and the corner rays (the detector is convex, so the corners
 * bound it).  K = max sin^2((gamma + eps) / 2).
 * Rows: the z/x slope of K_out is u2/u0 + (diffvec/L2) e_z / u0 + o_z /
 * (L2 u0), and a spot on the detector has a slope between the smallest and
 * largest corner slope (all corners in front of the voxel).  So
 * (diffvec/L2) e_z lies in [s_min u0 - u2 - o_z/L2, s_max u0 - u2 - o_z/L2],
 * whose extremes over omega are Zb, Zt.
 * Columns: likewise with the y/x slopes, (diffvec/L2) e_y lies in
 * [t_min u0 - u1 - o_y/L2, t_max u0 - u1 - o_y/L2] (t the corner y/x slopes),
 * whose extremes over omega are Yb, Yt. */
__device__ __forceinline__ double wave_max_d(double v) {
  for (int off = 32; off >= 1; off >>= 1) {
    const double o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}

__device__ __forceinline__ double wave_min_d(double v) {
  for (int off = 32; off >= 1; off >>= 1) {
    const double o = __shfl_xor(v, off, 64);
    v = o < v ? o : v;
  }
  return v;
}

/* The running extremes of the voxel bounds over the rotation angles. */
struct vb_acc {
  double d2max, kmax, e0, e1, u2lo, u2hi, ayz, zt, zb, yt, yb;
  bool front, rows;
};

__device__ __forceinline__ void vb_start(vb_acc &A) {
  A.d2max = 0.0, A.kmax = 0.0, A.e0 = 0.0, A.e1 = 0.0, A.u2lo = 2.0, A.u2hi = -2.0, A.ayz = 0.0;
  A.zt = -1e300, A.zb = 1e300, A.yt = -1e300, A.yb = 1e300;
  A.front = true, A.rows = true;
}

/* sqrt(x) for x >= 0 from the refined reciprocal square root (0 below) */
__device__ __forceinline__ double fast_sqrt(double x) { return x > 0.0 ? x * fast_rsq(x) : x * 0.0; }

/* One rotation angle's terms of the voxel bounds (P = S*pos of the voxel,
 * al, be, ga, oy, oz, on as in the kernels below).  Quotients and roots come
 * from the refined hardware reciprocals (relative error below 5e-15; the
 * margins that vb_write adds are 1e-9 relative): IEEE divisions and roots
 * took 10.9 ms for 3.2M voxels x 181 angles, these 5.6 ms. */
__device__ __forceinline__ void vb_omega(const grs_dgeo *g, const double *P, double c, double s, double al, double be,
                                         double ga, double oy, double oz, double on, vb_acc &A) {
  double sw[3], u[3];
  beam_terms(g, P, c, s, sw, u);
  const double u0 = u[0], u1 = u[1], u2 = u[2];
  const double sw0 = sw[0], sw1 = sw[1], sw2 = sw[2];
  const double d2 = (1.0 - u0) * (1.0 - u0) + u1 * u1 + u2 * u2;
  A.d2max = d2 > A.d2max ? d2 : A.d2max;
  const double a0 = __builtin_fabs(u0 - 1.0), a1 = __builtin_fabs(u1 - ((al * s + be * c) + ga));
  A.e0 = a0 > A.e0 ? a0 : A.e0;
  A.e1 = a1 > A.e1 ? a1 : A.e1;
  A.u2lo = u2 < A.u2lo ? u2 : A.u2lo;
  A.u2hi = u2 > A.u2hi ? u2 : A.u2hi;
  const double ay = fast_sqrt(__builtin_fma(u1, u1, u2 * u2)) * (1.0 + 1e-9) + 1e-12;
  A.ayz = ay > A.ayz ? ay : A.ayz;
  double cmin = 1.0, smin = 1e300, smax = -1e300, tmin = 1e300, tmax = -1e300;
  for (int j = 0; j < 4; j++) {
    const double dx = g->corner[3 * j] - sw0, dy = g->corner[3 * j + 1] - sw1, dz = g->corner[3 * j + 2] - sw2;
    const double cj = __builtin_fma(u0, dx, __builtin_fma(u1, dy, u2 * dz)) *
                      fast_rsq(__builtin_fma(dx, dx, __builtin_fma(dy, dy, dz * dz)));
    A.front = A.front && (cj > 1e-3);
    cmin = __builtin_fmin(cj, cmin);
    A.rows = A.rows && (dx > 0.0);
    const double ix = fast_rcp(dx);
    const double sl = dz * ix, ty = dy * ix;
    smin = __builtin_fmin(sl, smin);
    smax = __builtin_fmax(sl, smax);
    tmin = __builtin_fmin(ty, tmin);
    tmax = __builtin_fmax(ty, tmax);
  }
  const double L2 = (g->Lsd - sw0) * fast_rcp(u0), iL2 = fast_rcp(L2);
  A.front = A.front && (L2 > 0.0) && (ay < 1.0);
  /* sin and cos of gamma + eps, gamma = acos(cmin) */
  double se = (on * iL2) * fast_rsq(1.0 - (ay < 1.0 ? ay * ay : 0.0));
  se = se * (1.0 + 1e-9) + 1e-12;
  A.front = A.front && (se < 1.0);
  se = se < 1.0 ? se : 1.0;
  const double ce = fast_sqrt(1.0 - se * se);
  const double cm = cmin < 1.0 ? cmin : 1.0;
  const double sg = fast_sqrt(1.0 - cm * cm);
  const double k = (1.0 - (cm * ce - sg * se)) * 0.5;
  A.kmax = k > A.kmax ? k : A.kmax;
  const double ozl = oz * iL2;
  const double t1 = (smax * u0 - u2) - ozl, t0 = (smin * u0 - u2) - ozl;
  A.zt = t1 > A.zt ? t1 : A.zt;
  A.zb = t0 < A.zb ? t0 : A.zb;
  const double oyl = oy * iL2;
  const double y1 = (tmax * u0 - u1) - oyl, y0 = (tmin * u0 - u1) - oyl;
  A.yt = y1 > A.yt ? y1 : A.yt;
  A.yb = y0 < A.yb ? y0 : A.yb;
}

/* a NaN anywhere turns the bound off: the comparisons above skip NaNs */
__device__ __forceinline__ bool vb_nan(const vb_acc &A) {
  return !(A.d2max == A.d2max && A.kmax == A.kmax && A.zt == A.zt && A.zb == A.zb && A.yt == A.yt && A.yb == A.yb);
}

/* The GRS_VB values of a voxel from the extremes over every rotation angle. */
__device__ __forceinline__ void vb_write(const grs_dgeo *g, double al, double be, double ga, const vb_acc &A,
                                         bool nan_any, double *o) {
  const double delta = __builtin_sqrt(A.d2max) * (1.0 + 1e-9) + 1e-12;
  const double alpha = 2.0 * grs_asin(delta * 0.5 < 1.0 ? delta * 0.5 : 1.0) + 1e-9;
  double K = 1.0;
  const bool ok = A.front && !nan_any && 2.0 * g->theta_win + alpha < g->pio2 - 1e-3;
  if (ok) {
    K = A.kmax * (1.0 + 1e-6) + 1e-9;
    K = K < 1.0 ? K : 1.0;
  }
  const bool use_rows = ok && A.rows && A.ayz < 1.0;
  o[0] = ((__builtin_sqrt(al * al + be * be) * 0.5 + A.e0) + A.e1) * (1.0 + 1e-9) + 1e-12;
  o[1] = A.u2lo - 1e-12;
  o[2] = A.u2hi + 1e-12;
  o[3] = K;
  o[4] = al;
  o[5] = be;
  o[6] = ga;
  o[7] = use_rows ? A.zt + (__builtin_fabs(A.zt) * 1e-9 + 1e-12) : 1e300;
  o[8] = use_rows ? A.zb - (__builtin_fabs(A.zb) * 1e-9 + 1e-12) : -1e300;
  const double sn = A.ayz < 1.0 ? A.ayz : 1.0;
  o[9] = sn;
  o[10] = __builtin_sqrt(1.0 - sn * sn);
  o[11] = o[10] > 0.0 ? sn / o[10] : 1e300;
  const double ya = __builtin_fabs(A.yt) > __builtin_fabs(A.yb) ? __builtin_fabs(A.yt) : __builtin_fabs(A.yb);
  o[12] = use_rows ? ya * (1.0 + 1e-9) + 1e-12 : 1e300;
  o[13] = delta;
}

/* One 256-thread block per voxel: thread t takes the rotation angles t,
 * t + 256, ... (one each for up to 256 angles, which keeps the latency of a
 * one-voxel call short), and the extremes are reduced across each wave and
 * then across the four waves; maxima, minima and flags are exact, so the
 * result does not depend on the partition. */
__device__ __forceinline__ void voxel_bounds_block(const grs_dgeo *g, const double *pos, const double *cs,
                                                   int32_t nrot, double *vb) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  double P[3];
  voxel_P(g, pos, P);
  const double al = P[0] / g->Lss, be = P[1] / g->Lss, ga = (g->RAO - g->P0y) / g->Lss;
  const double oy = g->RAO - g->P0y, oz = -g->P0z;
  const double on = __builtin_sqrt(oy * oy + oz * oz);
  vb_acc A;
  vb_start(A);
  for (int32_t om = tid; om < nrot; om += 256) vb_omega(g, P, cs[2 * om], cs[2 * om + 1], al, be, ga, oy, oz, on, A);
  const bool nan_seen = __ballot(vb_nan(A)) != 0;
  A.front = __ballot(!A.front) == 0;
  A.rows = __ballot(!A.rows) == 0;
  A.d2max = wave_max_d(A.d2max);
  A.kmax = wave_max_d(A.kmax);
  A.e0 = wave_max_d(A.e0);
  A.e1 = wave_max_d(A.e1);
  A.u2lo = wave_min_d(A.u2lo);
  A.u2hi = wave_max_d(A.u2hi);
  A.ayz = wave_max_d(A.ayz);
  A.zt = wave_max_d(A.zt);
  A.zb = wave_min_d(A.zb);
  A.yt = wave_max_d(A.yt);
  A.yb = wave_min_d(A.yb);
  /* the four waves' maxima, minima and flags (exact, so order-free) */
  __shared__ double red[4][14];
  if (lane == 0) {
    double *r = red[wv];
    r[0] = A.d2max, r[1] = A.kmax, r[2] = A.e0, r[3] = A.e1, r[4] = A.u2lo, r[5] = A.u2hi, r[6] = A.ayz;
    r[7] = A.zt, r[8] = A.zb, r[9] = A.front ? 1.0 : 0.0, r[10] = A.rows ? 1.0 : 0.0, r[11] = nan_seen ? 1.0 : 0.0;
    r[12] = A.yt, r[13] = A.yb;
  }
  __syncthreads();
  if (tid != 0) return;
  bool nan_any = false;
  for (int k = 0; k < 4; k++) {
    const double *r = red[k];
    A.d2max = r[0] > A.d2max ? r[0] : A.d2max;
    A.kmax = r[1] > A.kmax ? r[1] : A.kmax;
    A.e0 = r[2] > A.e0 ? r[2] : A.e0;
    A.e1 = r[3] > A.e1 ? r[3] : A.e1;
    A.u2lo = r[4] < A.u2lo ? r[4] : A.u2lo;
    A.u2hi = r[5] > A.u2hi ? r[5] : A.u2hi;
    A.ayz = r[6] > A.ayz ? r[6] : A.ayz;
    A.zt = r[7] > A.zt ? r[7] : A.zt;
    A.zb = r[8] < A.zb ? r[8] : A.zb;
    A.yt = r[12] > A.yt ? r[12] : A.yt;
    A.yb = r[13] < A.yb ? r[13] : A.yb;
    A.front = A.front && r[9] != 0.0;
    A.rows = A.rows && r[10] != 0.0;
    nan_any = nan_any || r[11] != 0.0;
  }
  vb_write(g, al, be, ga, A, nan_any, vb);
}

__global__ __launch_bounds__(256) void k_voxel_bounds(const grs_dgeo *g, const double *pos, const double *cs,
                                                      int32_t nrot, double *vb) {
  const int64_t v = blockIdx.x;
  voxel_bounds_block(g, pos + 3 * v, cs, nrot, vb + GRS_VB * v);
}

/* The same bounds with L lanes per voxel (a power of two), lane l taking the
 * angles l, l + L, ...: one lane for millions of voxels, where a block per
 * voxel spends most of its time in the reductions (3.2M voxels: about 34 ms
 * as blocks), more lanes while a lane each would leave the chip without waves
 * (45,000 voxels x 361 angles: 511 us with one lane, 177 us with four).
 * Maxima, minima and flags are exact, so every form writes the same values. */
template <int L>
__global__ __launch_bounds__(256) void k_voxel_bounds_lanes(const grs_dgeo *g, const double *pos, int64_t V,
                                                            const double *cs, int32_t nrot, double *vb) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t v0 = t / L;
  const int64_t v = v0 < V ? v0 : V - 1; /* the lanes past the end repeat the last voxel: whole groups reduce */
  double P[3];
  voxel_P(g, pos + 3 * v, P);
  const double al = P[0] / g->Lss, be = P[1] / g->Lss, ga = (g->RAO - g->P0y) / g->Lss;
  const double oy = g->RAO - g->P0y, oz = -g->P0z;
  const double on = __builtin_sqrt(oy * oy + oz * oz);
  vb_acc A;
  vb_start(A);
  for (int32_t om = (int32_t)(t % L); om < nrot; om += L)
    vb_omega(g, P, cs[2 * om], cs[2 * om + 1], al, be, ga, oy, oz, on, A);
  int nan_any = vb_nan(A) ? 1 : 0, front = A.front ? 1 : 0, rows = A.rows ? 1 : 0;
  for (int off = L / 2; off >= 1; off >>= 1) {
    A.d2max = __builtin_fmax(A.d2max, __shfl_xor(A.d2max, off, 64));
    A.kmax = __builtin_fmax(A.kmax, __shfl_xor(A.kmax, off, 64));
    A.e0 = __builtin_fmax(A.e0, __shfl_xor(A.e0, off, 64));
    A.e1 = __builtin_fmax(A.e1, __shfl_xor(A.e1, off, 64));
    A.u2lo = __builtin_fmin(A.u2lo, __shfl_xor(A.u2lo, off, 64));
    A.u2hi = __builtin_fmax(A.u2hi, __shfl_xor(A.u2hi, off, 64));
    A.ayz = __builtin_fmax(A.ayz, __shfl_xor(A.ayz, off, 64));
    A.zt = __builtin_fmax(A.zt, __shfl_xor(A.zt, off, 64));
    A.zb = __builtin_fmin(A.zb, __shfl_xor(A.zb, off, 64));
    A.yt = __builtin_fmax(A.yt, __shfl_xor(A.yt, off, 64));
    A.yb = __builtin_fmin(A.yb, __shfl_xor(A.yb, off, 64));
    nan_any |= __shfl_xor(nan_any, off, 64);
    front &= __shfl_xor(front, off, 64);
    rows &= __shfl_xor(rows, off, 64);
  }
  A.front = front != 0;
  A.rows = rows != 0;
  if (t % L == 0 && v0 < V) vb_write(g, al, be, ga, A, nan_any != 0, vb + GRS_VB * v);
}

/* Largest sin(theta) = -cos(beta) of an event that can reach the detector,
 * from the voxel bounds.  With F = diffvec / L2 = sin(2 theta) / sin(phiy)
 * and the unit vector e = (0, Gt2, Gt3) / konst, F e_z lies in [Zb, Zt]
 * (rows) and F e_y in [Yb, Yt] (columns), so F |e_y| <= Ya.
 *   Rows: for Gz > 0 (Gz < 0 likewise with -Zb) e_z >= Gz/|G| = gz, as
 *   konst <= |G|, so F <= T = Zt / gz.
 *   Columns: Gt1/|G| differs from cos(beta) = u . G/|G| by at most
 *   |u - (1, 0, 0)| <= delta, so |Gt1|/|G| <= s1 + delta for an event in the
 *   window (s1 >= -cos(beta), the caller's bound before this one), konst^2
 *   >= |G|^2 (1 - (s1 + delta)^2), e_z^2 <= gz^2 / (1 - (s1 + delta)^2) and
 *   |e_y| = sqrt(1 - e_z^2) gives F <= T = Ya / sqrt(1 - that bound).
 * With T the smaller of the two: phiy = pi/2 - asin(a) - 2 theta with
 * |asin a| <= eta gives F >= sin(2 theta) / cos(2 theta - eta) when
 * 2 theta >= eta, so sin(2 theta) (1 - T sin eta) <= T cos eta cos(2 theta),
 * i.e. tan(2 theta) <= T' = T cos(eta) / (1 - T sin(eta)), or 2 theta < eta.
 * Then sin(theta)^2 = T'^2 / (2 q (q + 1)), q = sqrt(1 + T'^2), with T'
 * raised to tan(eta).  Returns 1 (no bound) where neither bound applies. */
__device__ __forceinline__ double det_sin_theta(double gz, double s1, double zt, double zb, double ya, double dl,
                                                double sn, double cn, double te) {
  double T = 1e300;
  const double Z = gz > 0.0 ? zt : -zb;
  if (gz != 0.0 && Z > 0.0 && Z < 1e299) T = Z * fast_rcp(__builtin_fabs(gz));
  if (ya < 1e299) {
    const double gx = (s1 + 1e-12) + dl;
    if (gx < 0.99) {
      const double ez2 = (gz * gz) * fast_rcp(1.0 - gx * gx) * (1.0 + 1e-12);
      if (ez2 < 0.98) {
        const double Tc = ya * fast_rsq(1.0 - ez2);
        T = Tc < T ? Tc : T;
      }
    }
  }
  if (!(T < 1e299)) return 1.0;
  const double den = 1.0 - T * sn;
  if (!(den > 0.0) || !(cn > 0.0)) return 1.0;
  double Tp = T * cn * fast_rcp(den);
  Tp = Tp > te ? Tp : te;
  const double q2 = 1.0 + Tp * Tp;
  const double q = q2 * fast_rsq(q2);
  const double st = Tp * fast_rsq((2.0 * q) * (q + 1.0));
  return st * (1.0 + 1e-9) + 1e-12;
}

/* grs_filt_acos and grs_filt_atan2 (grs_math.h: the same polynomials and
 * reductions) with the square root and the quotient taken from the refined
 * hardware reciprocals, which adds about 1e-14 to their error bounds (5e-12
 * and 2e-12 rad); NaN outside [-1, 1] as there. */
__device__ __forceinline__ double acos_core(double x) {
  const double R[8] = GRS_FILT_ASIN_R;
  const double ax = __builtin_fabs(x);
  const bool small = ax <= 0.5;
  const double zb = (1.0 - ax) * 0.5;
  const double u = small ? x : (zb == 0.0 ? 0.0 : zb * fast_rsq(zb));
  const double z = small ? x * x : zb;
  double p = R[7];
  p = __builtin_fma(p, z, R[6]);
  p = __builtin_fma(p, z, R[5]);
  p = __builtin_fma(p, z, R[4]);
  p = __builtin_fma(p, z, R[3]);
  p = __builtin_fma(p, z, R[2]);
  p = __builtin_fma(p, z, R[1]);
  p = __builtin_fma(p, z, R[0]);
  const double as = __builtin_fma(u * z, p, u);
  if (small) return GRS_PIO2_HI - as;
  return x > 0.0 ? 2.0 * as : GRS_PI_HI - 2.0 * as;
}
__device__ __forceinline__ double atan2_core(double y, double x) {
  const double S[7] = GRS_FILT_ATAN_S;
  const double ax = __builtin_fabs(x), ay = __builtin_fabs(y);
  const double mx = ax > ay ? ax : ay, mn = ax > ay ? ay : ax;
  if (!(mx > 0.0)) return mx == 0.0 ? 0.0 : mx;
  const bool big = mn > GRS_TAN_PI_8 * mx;
  const double w = big ? (mn - mx) * fast_rcp(mn + mx) : mn * fast_rcp(mx);
  const double z = w * w;
  double p = S[6];
  p = __builtin_fma(p, z, S[5]);
  p = __builtin_fma(p, z, S[4]);
  p = __builtin_fma(p, z, S[3]);
  p = __builtin_fma(p, z, S[2]);
  p = __builtin_fma(p, z, S[1]);
  p = __builtin_fma(p, z, S[0]);
  double a = __builtin_fma(w * z, p, w);
  if (big) a = a + 0.5 * GRS_PIO2_HI;
  if (ay > ax) a = GRS_PIO2_HI - a;
  if (x < 0.0) a = GRS_PI_HI - a;
  return y < 0.0 ? -a : a;
}
/* the device math test's entries (fn 10, 11) */
__device__ __noinline__ double filt_acos(double x) { return acos_core(x); }
__device__ __noinline__ double filt_atan2(double y, double x) { return atan2_core(y, x); }

/* The omega solve's three angles in one out-of-line call: acos(a) (pi at
 * a <= -1), acos(b) (0 at b >= 1) and atan2(y, x), the two polynomial
 * chains of acos side by side.  Inlined, they raise the register pressure
 * of the whole kernel (spills in the candidate loop); three calls cost 2%
 * of the seeding launch more than one. */
struct arc_angles {
  double pa, pb, phi;
};
__device__ __noinline__ arc_angles arc_ends(double a, double b, double y, double x) {
  arc_angles r;
  r.pa = acos_core(a);
  r.pb = acos_core(b);
  r.phi = atan2_core(y, x);
  if (a <= -1.0) r.pa = GRS_PI;
  if (b >= 1.0) r.pb = 0.0;
  return r;
}

__global__ void k_sub_from_q(const grs_dgeo *g, const double *q, int64_t N, double *SUB, int32_t *valid) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  double U[9];
  int ok = grs_U_from_q(q[4 * i + 1], q[4 * i + 2], q[4 * i + 3], U);
  valid[i] = ok;
  if (ok) grs_SUB(g, U, SUB + 9 * i);
  else
    for (int k = 0; k < 9; k++) SUB[9 * i + k] = 0.0;
}

/* One row of the beam table: every term of the spot construction that depends
 * on (voxel, omega) alone. */
__device__ __forceinline__ void beam_row(const grs_dgeo *g, const double *P, double c, double s, double *r) {
  om_terms w;
  omega_terms(g, P, c, s, &w);
  r[0] = w.u0;
  r[1] = w.u1;
  r[2] = w.u2;
  r[3] = w.k0;
  r[4] = w.d1;
  r[5] = w.d2;
  r[6] = w.L2;
  r[7] = w.tnum;
  r[8] = w.ov1;
  r[9] = w.ov2;
  r[10] = c;
  r[11] = s;
}

/* The beam table of V voxels in device memory, for launches whose voxels have
 * many evaluations each and whose tables stay in cache: the scoring kernel then loads the terms of a
 * candidate (six 16-byte loads from L1/L2) instead of 45 operations with two
 * reciprocals.  262,144 orientations and 500 groups of 729 at two voxels: 13.0 -> 12.3 ms;
 * 24 orientation fits: 1.47 -> 1.39 ms. */
__global__ __launch_bounds__(256) void k_beam(const grs_dgeo *g, const double *pos, int64_t V, const double *cs,
                                              int32_t nrot, double *beam) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= V * nrot) return;
  const int64_t v = t / nrot;
  const int32_t om = (int32_t)(t - v * nrot);
  double P[3];
  voxel_P(g, pos + 3 * v, P);
  beam_row(g, P, cs[2 * om], cs[2 * om + 1], beam + GRS_BT * t);
}

/* What a one-voxel launch needs beside the stack, in one kernel: block 0
 * writes the position (which comes with the launch) and its bounds, the
 * others S*U*B of 256 orientations each. */
struct one_pos {
  double x[3];
};
__global__ __launch_bounds__(256) void k_one_voxel(const grs_dgeo *g, one_pos at, const double *cs, int32_t nrot,
                                                   const double *q, int64_t N, double *pos, double *vb, double *SUB,
                                                   int32_t *valid) {
  if (blockIdx.x == 0) {
    if (threadIdx.x < 3) pos[threadIdx.x] = at.x[threadIdx.x];
    voxel_bounds_block(g, at.x, cs, nrot, vb);
    return;
  }
  const int64_t i = (int64_t)(blockIdx.x - 1) * 256 + threadIdx.x;
  if (i >= N) return;
  double U[9];
  const int ok = grs_U_from_q(q[4 * i + 1], q[4 * i + 2], q[4 * i + 3], U);
  valid[i] = ok;
  if (ok) grs_SUB(g, U, SUB + 9 * i);
  else
    for (int k = 0; k < 9; k++) SUB[9 * i + k] = 0.0;
}

__global__ void k_sub_from_U(const grs_dgeo *g, const double *U, int64_t N, double *SUB, int32_t *valid) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  grs_SUB(g, U + 9 * i, SUB + 9 * i);
  valid[i] = 1;
}

__global__ void k_sub_from_euler(const grs_dgeo *g, const double *eu, int64_t N, double *SUB, int32_t *valid) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  double U[9];
  grs_U_from_euler_deg(eu[3 * i], eu[3 * i + 1], eu[3 * i + 2], U);
  grs_SUB(g, U, SUB + 9 * i);
  valid[i] = 1;
}

__global__ void k_math_eval(int fn, const double *x, double *y, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double v = x[i], r;
  switch (fn) {
    case 0: r = grs_sin(v); break;
    case 1: r = grs_cos(v); break;
    case 2: r = grs_acos(v); break;
    case 3: r = grs_atan(v); break;
    case 4: r = grs_round(v); break;
    case 5: r = grs_sqrt(v); break;
    case 7: r = grs_asin(v); break;
    case 8: r = grs_filt_acos(v); break;
    case 9: r = grs_filt_atan2(grs_sin(v), grs_cos(v)); break;
    case 10: r = filt_acos(v); break;
    case 11: r = filt_atan2(grs_sin(v), grs_cos(v)); break;
    case 12: r = fast_rcp(v); break;
    case 13: r = fast_rsq(v); break;
    default: r = 1.0 / v; break;
  }
  y[i] = r;
}

/* Plain device copy (calibrates memory counters: reads and writes n words). */
__global__ void k_copy_u32(const uint32_t *src, uint32_t *dst, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) dst[i] = src[i];
}

/* Flags keys that are not non-negative, non-NaN floats. */
__global__ void k_check_keys(const uint32_t *keys, int64_t n, uint32_t *bad) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  uint32_t b = 0;
  for (; i < n; i += stride) b |= (keys[i] > 0x7F800000u) ? 1u : 0u;
  if (b) atomicOr(bad, 1u);
}

/* ---------------------------------------------------------------------- */
/* mapping of evaluations                                                   */

__device__ __forceinline__ void eval_slots(const grs_eval_args &a, int64_t e, int64_t *vi, int64_t *ui) {
  if (a.map == GRS_MAP_ONE_VOXEL) {
    *vi = 0;
    *ui = e;
  } else if (a.map == GRS_MAP_ONE_U) {
    *vi = e;
    *ui = 0;
  } else if (a.map == GRS_MAP_GRID) {
    const int64_t v = e / a.n_u;
    *vi = v;
    *ui = (e - v * a.n_u) + v * a.u_stride;
  } else {
    *vi = a.eval_vox[e];
    *ui = a.eval_u[e];
  }
}

/* ---------------------------------------------------------------------- */
/* wave-level median over a key list in global memory                      */

/* number of keys < x among list[0..n) */
__device__ __forceinline__ int32_t wave_count_lt_global(const uint32_t *list, int32_t n, uint32_t x, int lane) {
  int32_t c = 0;
  for (int32_t b = 0; b < n; b += 64) {
    int32_t j = b + lane;
    bool p = j < n && list[j] < x;
    c += __popcll(__ballot(p));
  }
  return c;
}

__device__ uint32_t wave_select_global(const uint32_t *list, int32_t n, int32_t k, int lane) {
  uint32_t res = 0;
  for (int bit = 31; bit >= 0; --bit) {
    uint32_t cand = res | (1u << bit);
    if (wave_count_lt_global(list, n, cand, lane) <= k) res = cand;
  }
  return res;
}

/* Median of n <= 64*R keys held R per lane in registers: the k-th smallest
 * key by bisection on its bits (count of keys below a candidate by ballot). */
template <int R>
__device__ float wave_median_reg(const uint32_t *list, int32_t n, int lane) {
  const int32_t k1 = (n & 1) ? (n >> 1) : (n >> 1) - 1;
  uint32_t r[R];
#pragma unroll
  for (int j = 0; j < R; j++) {
    int32_t idx = j * 64 + lane;
    r[j] = idx < n ? list[idx] : 0xFFFFFFFFu;
  }
  uint32_t res = 0;
  /* keys are non-negative floats: bit 31 is clear */
  for (int bit = 30; bit >= 0; --bit) {
    uint32_t cand = res | (1u << bit);
    int32_t c = 0;
#pragma unroll
    for (int j = 0; j < R; j++) c += __popcll(__ballot(r[j] < cand));
    if (c <= k1) res = cand;
  }
  const uint32_t v1 = res;
  if (n & 1) return key_to_float(v1);
  int32_t cle = 0;
  uint32_t mn = 0xFFFFFFFFu;
#pragma unroll
  for (int j = 0; j < R; j++) {
    cle += __popcll(__ballot(r[j] <= v1));
    if (r[j] > v1 && r[j] < mn) mn = r[j];
  }
  const uint32_t v2 = cle > k1 + 1 ? v1 : wave_min_u32(mn);
  float a = key_to_float(v1), b = key_to_float(v2);
  return a + (b - a) / 2.0f;
}

__device__ float wave_median(const uint32_t *list, int32_t n, int lane) {
  if (n <= 128) return wave_median_reg<2>(list, n, lane);
  if (n <= 256) return wave_median_reg<4>(list, n, lane);
  if (n <= 512) return wave_median_reg<8>(list, n, lane);
  if (n <= 64 * GRS_REG_KEYS) return wave_median_reg<GRS_REG_KEYS>(list, n, lane);
  const int32_t k1 = (n & 1) ? (n >> 1) : (n >> 1) - 1;
  uint32_t v1 = wave_select_global(list, n, k1, lane), v2;
  if (n & 1) return key_to_float(v1);
  int32_t cle = 0;
  uint32_t mn = 0xFFFFFFFFu;
  for (int32_t b = 0; b < n; b += 64) {
    int32_t j = b + lane;
    uint32_t kv = j < n ? list[j] : 0xFFFFFFFFu;
    cle += __popcll(__ballot(j < n && kv <= v1));
    if (j < n && kv > v1 && kv < mn) mn = kv;
  }
  v2 = cle > k1 + 1 ? v1 : wave_min_u32(mn);
  float a = key_to_float(v1), b = key_to_float(v2);
  return a + (b - a) / 2.0f;
}

/* ---------------------------------------------------------------------- */
/* orientation of an evaluation                                            */

/* Fills sub (S*U*B) for evaluation e and the voxel slot; returns 1 when the
 * orientation is valid, 0 when its row is skipped (|q_vec| > 1), -1 when the
 * evaluation is an empty CSR row (GRS_MAP_CSR_LIST).  row/jloc receive the CSR
 * row and the index inside the row's expanded list. */
template <int MAP>
__device__ __forceinline__ int eval_setup(const grs_eval_args &a, int64_t e, int64_t *vi, double *sub, int64_t *row,
                                          int64_t *jloc, int64_t *hint = nullptr) {
  if (MAP == GRS_MAP_CSR || MAP == GRS_MAP_CSR_LIST) {
    const grs_csr &c = a.csr;
    int64_t ge = e;
    if (MAP == GRS_MAP_CSR_LIST) {
      ge = c.elist[e];
      if (ge < 0) return -1;
    }
    /* the row of the previous evaluation of this wave, or the next one,
     * usually holds ge (a wave's evaluations ascend); else a binary search */
    int64_t lo = -1;
    if (hint && *hint >= 0) {
      const int64_t h = *hint;
      if (c.row_eoff[h] <= ge) {
        if (h + 1 >= c.nrows || c.row_eoff[h + 1] > ge) lo = h;
        else if (h + 2 >= c.nrows || c.row_eoff[h + 2] > ge) lo = h + 1;
      }
    }
    if (lo < 0) {
      int64_t hi = c.nrows;
      lo = 0;
      while (hi - lo > 1) {
        int64_t mid = (lo + hi) >> 1;
        if (c.row_eoff[mid] <= ge) lo = mid;
        else hi = mid;
      }
    }
    if (hint) *hint = lo;
    int64_t j = ge - c.row_eoff[lo];
    int64_t cand = c.row_ptr[lo] + j / c.S;
    int32_t smp = (int32_t)(j % c.S);
    int32_t n1 = c.nr + 1;
    int32_t k1 = smp / (n1 * n1), k2 = (smp / n1) % n1, k3 = smp % n1;
    const double *q = c.cand_q + 4 * cand;
    const double half = (c.gridsize * (double)c.nr) / 2.0;
    double q1 = (q[1] - half) + (double)k1 * c.gridsize;
    double q2 = (q[2] - half) + (double)k2 * c.gridsize;
    double q3 = (q[3] - half) + (double)k3 * c.gridsize;
    double U[9];
    *vi = lo;
    *row = lo;
    *jloc = j;
    if (!grs_U_from_q(q1, q2, q3, U)) return 0;
    grs_SUB(a.g, U, sub);
    return 1;
  } else {
    int64_t ui;
    eval_slots(a, e, vi, &ui);
    *row = e;
    *jloc = 0;
    if (!a.valid[ui]) return 0;
#pragma unroll
    for (int k = 0; k < 9; k++) sub[k] = a.SUB[ui * 9 + k];
    return 1;
  }
}

/* ---------------------------------------------------------------------- */
/* k_fast                                                                  */

/* Counts-only output of a grid evaluation: the counts and the key
 * (class << 32) | (2^32 - 1 - i) of orientation i of its voxel, where class
 * orders C = ni/ns as MATLAB's sortrows(...,'descend') does: NaN (ns = 0)
 * first as 2^31, else floor(C * 2^30) + 1, which separates every two distinct
 * ratios of counts up to GRS_KEY_MAX_EVENTS; a skipped orientation has C = 0
 * (class 1).  Equal classes order by ascending i (a stable sort). */
__device__ __forceinline__ void grid_counts_out(const grs_eval_args &a, int64_t e, int32_t ns, int32_t ni,
                                                bool valid) {
  if (a.out_ns) {
    a.out_ns[e] = ns;
    a.out_ni[e] = ni;
  }
  if (a.out_key) {
    uint64_t cls = 1;
    if (valid) {
      if (ns > 0) cls = (uint64_t)__builtin_floor(((double)ni / (double)ns) * 1073741824.0) + 1ull;
      else cls = 1ull << 31;
    }
    const uint64_t i = (uint64_t)(e % a.n_u);
    a.out_key[e] = (unsigned long long)((cls << 32) | (0xFFFFFFFFull - i));
  }
}

/* The exact forward_comp.m:28-65 pipeline of one event (omega index om,
 * reflection h): returns 1 and the stack index when the event is selected;
 * yz receives the unrounded pixel coordinates of a selected event.  The
 * per (voxel, omega) terms are recomputed here with the function of the
 * exact pipeline (grs_vw_terms).  Kept out of line: it runs for about 1e-4 of the events, and inlining it would raise
 * the register pressure of the whole kernel. */
__device__ __noinline__ int exact_event(const grs_dgeo *g, const double *pos, const double *cs, const double *gwt,
                                        uint32_t ev, uint32_t *idx, double *yz) {
  const int32_t om = (int32_t)(ev >> 8), h = (int32_t)(ev & 255u);
  grs_vw v;
  grs_vw_terms(g, pos, cs[2 * om], cs[2 * om + 1], &v);
  const double *t = gwt + h * GRS_GWT;
  double Gt[3];
  grs_Gt(v.c, v.s, t[0], t[1], t[2], Gt);
  double Glen;
  double beta = grs_event_beta(&v, Gt, &Glen);
  int32_t dy = 0, dz = 0;
  double w[2] = {0.0, 0.0};
  if (!grs_event_finish_yz(g, &v, Gt, Glen, beta, &dy, &dz, w)) return 0;
  *idx = (uint32_t)((int64_t)(dz - 1) + (int64_t)(dy - 1) * g->nz + (int64_t)om * g->nz * g->ny);
  yz[0] = w[0];
  yz[1] = w[1];
  return 1;
}

/* Omega solve of one reflection.  With (g0, g1) the in-plane part of a
 * vector that rotates with omega, |G| = gn and r = |(g0, g1)|, the term
 * r cos(omega + phi) / gn, phi = atan2(g1, g0), must lie in [lo_cb, hi_cb]
 * (the caller folds every other part of cos(beta), forward_comp.m:31, and its
 * bounds into the window), so omega + phi must lie in the arcs where
 * cos(psi) is in [lo_cb gn / r, hi_cb gn / r] (gn / r from a refined
 * reciprocal square root).  The arc angles come from one call of
 * arc_ends (errors below 5e-12 rad); the arcs are widened by 1e-6 rad and
 * the index bounds by 1e-6 steps.  The ranges of rotation indices [i0, i1]
 * land in four fixed slots (two arcs x two periods) and are disjoint, in
 * no particular order.  Returns the bit mask of the slots in use or -1 when
 * more would be needed (the caller then scans every event). */
__device__ __forceinline__ int om_ranges(const grs_dgeo *g, double g0, double g1, double gn, double lo_cb,
                                         double hi_cb, int32_t nrot, double idom, int32_t *i0, int32_t *i1) {
  const double twopi = 2.0 * GRS_PI, eps = 1e-6;
  const double r2 = g0 * g0 + g1 * g1;
  const double ir = r2 > 0.0 ? fast_rsq(r2) : 0.0;
  const double r = r2 > 0.0 ? r2 * ir : r2 * 0.0; /* NaN stays NaN */
  if (lo_cb != lo_cb || hi_cb != hi_cb || r != r || !(gn > 0.0)) return -1;
  if (!(hi_cb > lo_cb)) return 0;
  double lo[2], hi[2];
  int niv = 0;
  bool whole = false;
  if (!(r > 1e-12 * gn)) {
    /* |cos(beta) x component| <= r / gn <= 1e-12 at every omega */
    whole = lo_cb <= 1e-12 && hi_cb >= -1e-12;
    if (!whole) return 0;
  } else {
    const double gr = gn * ir;
    const double a = lo_cb * gr, b = hi_cb * gr;
    if (!(a < 1.0) || !(b > -1.0)) return 0;
    const arc_angles an = arc_ends(a, b, g1, g0);
    const double pa = an.pa, pb = an.pb, phi = an.phi;
    /* the gaps between the two arcs, around psi = 0 and psi = pi: one of at
     * most 1e-5 rotation steps is closed (its events join the candidates),
     * so that the index ranges of different arcs and periods never share
     * an index */
    const bool gap0 = (2.0 * (pb - eps)) * idom <= 1e-5;
    const bool gap_pi = (twopi - 2.0 * (pa + eps)) * idom <= 1e-5;
    if (gap0 && gap_pi) {
      whole = true;
    } else if (gap0) {
      lo[0] = (-pa - eps) - phi;
      hi[0] = (pa + eps) - phi;
      niv = 1;
    } else if (gap_pi) {
      lo[0] = (pb - eps) - phi;
      hi[0] = (twopi - pb + eps) - phi;
      niv = 1;
    } else {
      lo[0] = (pb - eps) - phi;
      hi[0] = (pa + eps) - phi;
      lo[1] = (-pa - eps) - phi;
      hi[1] = (-pb + eps) - phi;
      niv = 2;
    }
  }
  if (whole) {
    i0[0] = 0;
    i1[0] = nrot - 1;
    return 1;
  }
  /* slot 2 k + j: arc k in its first period that ends at or after om0 and in
   * the next.  The arcs and their periods are more than 1e-5 steps apart, so
   * the ranges are disjoint as they come; their order does not matter to the
   * caller.  The subtraction of 1e-9 keeps a period whose arc ends next to
   * om0 (its range may be empty); an arc that would reach into a third period
   * makes the caller scan every event. */
  uint32_t mask = 0;
#pragma unroll
  for (int k = 0; k < 2; k++) {
    if (k >= niv) break;
    const double m = __builtin_ceil((g->om0 - hi[k]) * (1.0 / twopi) - 1e-9);
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const double L = lo[k] + twopi * (m + (double)j), U = hi[k] + twopi * (m + (double)j);
      double f0 = __builtin_ceil((L - g->om0) * idom - 1e-6);
      double f1 = __builtin_floor((U - g->om0) * idom + 1e-6);
      f0 = f0 > 0.0 ? f0 : 0.0;
      f1 = f1 < (double)(nrot - 1) ? f1 : (double)(nrot - 1);
      const bool ok = L <= g->om_last + 1e-9 && U >= g->om0 - 1e-9 && f0 <= f1;
      i0[2 * k + j] = (int32_t)f0;
      i1[2 * k + j] = (int32_t)f1;
      mask |= (ok ? 1u : 0u) << (2 * k + j);
    }
    if (lo[k] + twopi * (m + 2.0) <= g->om_last + 1e-9) return -1;
  }
  return (int)mask;
}

/* LDS regions of one wave of k_fast / k_fit_nm */
struct fast_lds_regions {
  double *gwt;      /* per reflection: G, 1/|G|, |G|^2 (indexed by the reflection) */
  uint32_t *ring1;  /* phase-A survivors (omega << 8 | hkl) */
  uint32_t *ring2;  /* events for the exact pipeline */
  uint32_t *ring3;  /* selected events: stack index */
  uint32_t *rstart; /* omega-solve ranges: (i0 << 8 | hkl) */
  uint32_t *rcum;   /* exclusive prefix of range lengths */
  double *Pw;       /* S*pos of the voxel */
  /* S*U*B of the evaluation: the omega solve reads it from LDS, which keeps
   * its 18 registers free for the candidate loop */
  double *sbuf;
};

/* the regions of wave wib when every wave holds reflections hlo .. hlo + Hn - 1 at most */
__device__ __forceinline__ fast_lds_regions fast_regions(double *smem, int wib, int32_t hlo, int32_t Hn) {
  fast_lds_regions L;
  double *w = smem + wib * fast_wave_doubles(Hn);
  L.gwt = w - (int64_t)hlo * GRS_GWT;
  L.ring1 = (uint32_t *)(w + (int64_t)Hn * GRS_GWT);
  L.ring2 = L.ring1 + GRS_QCAP;
  L.ring3 = L.ring2 + GRS_QCAP;
  L.rstart = L.ring3 + GRS_QCAP;
  L.rcum = L.rstart + 4 * Hn;
  L.Pw = w + (int64_t)Hn * GRS_GWT + GRS_RING_DOUBLES + GRS_RANGE_DOUBLES(Hn);
  L.sbuf = L.Pw + 4;
  return L;
}

/* One wave scores the events of reflections hlo .. hend - 1 of the evaluation
 * (voxel vi, orientation sub): the counts and, with MEDIAN, the keys of the
 * selected events in wlist.  TEAM: the waves of a block share the
 * evaluation, each with its own reflections, and append their keys to one
 * list through the block's counter tcount. */
template <bool MEDIAN, bool AUDIT, bool TEAM>
__device__ __forceinline__ void score_events(const grs_eval_args &a, const grs_dgeo *g, const double *b1thr,
                                             const double *btab, const fast_lds_regions &L, const double *sub,
                                             int64_t vi, int32_t hlo, int32_t hend, uint32_t *wlist, int32_t *tcount,
                                             int32_t *ns_out, int32_t *ni_out) {
  const int lane = threadIdx.x & 63;
  double *gwt = L.gwt;
  uint32_t *ring1 = L.ring1, *ring2 = L.ring2, *ring3 = L.ring3, *rstart = L.rstart, *rcum = L.rcum;
  double *Pw = L.Pw, *sbuf = L.sbuf;
  const int32_t nrot = g->nrot;
  const int64_t nz = g->nz, nzny = g->nz * g->ny;
  const uint32_t nz32 = (uint32_t)nz, nzny32 = (uint32_t)nzny; /* the stack holds fewer than 2^32 entries */
  /* counts-only on the tiled mask: the selected events carry tiled bit numbers */
  const bool tiled = !MEDIAN && a.bits_tiled && !a.count_keys;
  const uint32_t ntz = (uint32_t)((nz + 31) >> 5), nty = (uint32_t)((g->ny + 31) >> 5);
  const uint32_t *hbits = tiled ? a.hit_tbits : a.hit_bits;
  const double m4pi = -4.0 * GRS_PI;
  /* phase A margins: see the header comment */
  const double dcb = 1e-12;
  const double cbm = g->cos_beta_max - dcb;
  const double lmin = g->lambda_min, lmax = g->lambda_max;
  const double lrel = 1e-9 * lmax;
  const double inv4pi = 1.0 / (4.0 * GRS_PI);
  const double idom = g->om_solve ? 1.0 / g->dom : 0.0;
  /* per-reflection terms; with the omega solve also the candidate ranges */
  const bool solve = g->om_solve != 0;
  if (lane == 0) {
    voxel_P(g, a.pos + 3 * vi, Pw);
#pragma unroll
    for (int k = 0; k < 9; k++) sbuf[k] = sub[k];
  }
  wave_sync();
  double vW = 0.0, vu2lo = 0.0, vu2hi = 0.0, sK = 1.0, val = 0.0, vbe = 0.0, vga = 0.0;
  double vzt = 1e300, vzb = -1e300, vsn = 1.0, vcn = 0.0, vte = 0.0, vya = 1e300, vdl = 0.0;
  if (solve) {
    const double *b = a.vb + GRS_VB * vi;
    vW = b[0];
    vu2lo = b[1];
    vu2hi = b[2];
    sK = __builtin_sqrt(b[3]);
    val = b[4];
    vbe = b[5];
    vga = b[6];
    vzt = b[7];
    vzb = b[8];
    vsn = b[9];
    vcn = b[10];
    vte = b[11];
    vya = b[12];
    vdl = b[13];
  }
  uint32_t R = 0;
  bool overflow = false;
  for (int hb = hlo; hb < hend; hb += 64) {
    const int h = hb + lane;
    int nr_h = 0; /* bit mask of the valid slots of ri0/ri1, or -1 */
    int32_t ri0[4], ri1[4];
    if (h < hend) {
      double gw[3];
      grs_Gw(sbuf, a.hkl + 3 * h, gw);
      double n2 = (gw[0] * gw[0] + gw[1] * gw[1]) + gw[2] * gw[2];
      const double ign = fast_rsq(n2);
      const double gn = n2 * ign;
      double *t = gwt + h * GRS_GWT;
      t[0] = gw[0];
      t[1] = gw[1];
      t[2] = gw[2];
      t[3] = ign;
      t[4] = n2;
      double ml = lrel + (1e-12 * (4.0 * GRS_PI)) * ign; /* absolute lambda margin */
      if (solve) {
        /* cos(beta) window: beta and lambda bounds with the phase-A margins,
         * the detector cone and the detector rows and columns.  cos(beta) = u . G/gn lies within rg W
         * of r' cos(omega + phi') / gn + c0 + u2 g2 / gn, where
         * (g0', g1') = (g0 + ga g1, g1 - ga g0) has modulus r' and angle
         * phi' and u2 spans [vb[1], vb[2]] (the voxel bounds), so the
         * window moves onto the first term. */
        double lo_cb = cbm;
        double lw = -(lmax + ml) * gn * inv4pi;
        lo_cb = lw > lo_cb ? lw : lo_cb;
        lo_cb = -sK > lo_cb ? -sK : lo_cb;
        const double z = gw[2] * ign;
        const double st = det_sin_theta(z, -lo_cb, vzt, vzb, vya, vdl, vsn, vcn, vte);
        lo_cb = -st > lo_cb ? -st : lo_cb;
        double hi_cb = dcb;
        double hw = -(lmin - ml) * gn * inv4pi;
        hi_cb = hw < hi_cb ? hw : hi_cb;
        const double q2 = gw[0] * gw[0] + gw[1] * gw[1];
        const double rg = q2 > 0.0 ? q2 * fast_rsq(q2) * ign : 0.0;
        const double c0 = (val * gw[0] + vbe * gw[1]) * (0.5 * ign);
        const double sa = z * vu2lo, sb = z * vu2hi;
        const double slo = sa < sb ? sa : sb, shi = sa < sb ? sb : sa;
        const double w = rg * vW;
        nr_h = om_ranges(g, gw[0] + vga * gw[1], gw[1] - vga * gw[0], gn, ((lo_cb - c0) - shi) - w - 1e-12,
                         ((hi_cb - c0) - slo) + w + 1e-12, nrot, idom, ri0, ri1);
      }
    }
    if (solve) {
      overflow = overflow || (__ballot(nr_h < 0) != 0);
      const uint32_t msk = nr_h > 0 ? (uint32_t)nr_h : 0u;
      const int cnt = __popc(msk);
      int incl = cnt;
      for (int off = 1; off < 64; off <<= 1) {
        int v = __shfl_up(incl, off, 64);
        if (lane >= off) incl += v;
      }
      uint32_t pos = R + (uint32_t)(incl - cnt);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        if ((msk >> k) & 1u) {
          rstart[pos] = ((uint32_t)ri0[k] << 8) | (uint32_t)h;
          rcum[pos] = (uint32_t)(ri1[k] - ri0[k] + 1);
          pos++;
        }
      }
      R += (uint32_t)__shfl(incl, 63, 64);
    }
  }
  wave_sync();
  uint32_t total = 0;
  if (solve && !overflow) {
    /* lengths -> exclusive prefix sums; the first candidate of each range
     * sets its bit in ring1, a bitmap of the first GRS_QCAP * 32 candidates
     * (unused otherwise on this path) */
    for (int k = lane; k < GRS_QCAP; k += 64) ring1[k] = 0u;
    for (uint32_t cb = 0; cb < R; cb += 64) {
      const uint32_t r = cb + lane;
      const uint32_t len = r < R ? rcum[r] : 0u;
      uint32_t incl = len;
      for (int off = 1; off < 64; off <<= 1) {
        uint32_t v = (uint32_t)__shfl_up((int)incl, off, 64);
        if (lane >= off) incl += v;
      }
      wave_sync();
      const uint32_t first = total + incl - len;
      if (r < R) {
        rcum[r] = first;
        if (first < GRS_QCAP * 32u) atomicOr(&ring1[first >> 5], 1u << (first & 31u));
      }
      total += (uint32_t)__shfl((int)incl, 63, 64);
      wave_sync();
    }
    if (lane == 0) rcum[R] = total;
    wave_sync();
  }

  const double *vpos = a.pos + 3 * vi;
  uint32_t head1 = 0, tail1 = 0, head2 = 0, tail2 = 0, head3 = 0, tail3 = 0;
  int32_t ns = 0, ni = 0;
  /* the gather of the previous batch is consumed one batch later */
  bool p_sel = false, p_hit = false;
  uint32_t p_key = 0;

  auto consume = [&]() {
    uint64_t ms = __ballot(p_sel);
    if (MEDIAN) {
      int32_t at = ns;
      if (TEAM && ms) {
        /* the team's waves append to one list */
        if (lane == 0) at = atomicAdd(tcount, (int32_t)__popcll(ms));
        at = __builtin_amdgcn_readfirstlane(at);
      }
      if (p_sel) wlist[at + (int32_t)lane_prefix(ms)] = p_key;
    }
    ns += (int32_t)__popcll(ms);
    bool hit;
    if (MEDIAN) hit = p_sel && g->has_hit && p_key <= g->hit_key;
    else hit = p_hit;
    ni += (int32_t)__popcll(__ballot(hit));
    p_sel = false;
    p_hit = false;
  };

  /* gather: distance key (or hit bit) of n selected events of ring3 */
  auto gather = [&](uint32_t n) {
    consume();
    if ((uint32_t)lane < n) {
      uint32_t idx = ring3[(head3 + lane) & (GRS_QCAP - 1)];
      p_sel = true;
      if (MEDIAN) p_key = a.keys[idx];
      else if (a.count_keys) p_hit = g->has_hit && a.keys[idx] <= g->hit_key;
      else p_hit = (hbits[idx >> 5] >> (idx & 31u)) & 1u;
    }
    head3 += n;
  };

  auto push3 = [&](bool sel, uint32_t idx) {
    uint64_t m = __ballot(sel);
    if (sel) ring3[(tail3 + lane_prefix(m)) & (GRS_QCAP - 1)] = idx;
    tail3 += (uint32_t)__popcll(m);
    if (tail3 - head3 >= 64) {
      wave_sync();
      gather(64);
      wave_sync();
    }
  };

  /* phase B2: exact pipeline on n events of ring2 */
  auto b2 = [&](uint32_t n) {
    bool sel = false;
    uint32_t idx = 0;
    if ((uint32_t)lane < n) {
      double yz[2];
      sel = exact_event(a.g, vpos, a.cs, gwt, ring2[(head2 + lane) & (GRS_QCAP - 1)], &idx, yz) != 0;
      if (sel && tiled) {
        const uint32_t omx = idx / nzny32, rem = idx - omx * nzny32, y0 = rem / nz32;
        idx = grs_tiled_bit(omx, y0 + 1u, rem - y0 * nz32 + 1u, ntz, nty);
      }
    }
    head2 += n;
    push3(sel, idx);
  };

  /* phase B1: resolve n events of ring1 or queue them for the exact pipeline */
  auto b1_core = [&](bool valid, uint32_t ev, uint32_t n) {
    int st = 0;
    uint32_t idx = 0;
    bool bad = false, inwin = false;
    double dev = 0.0;
    if (valid) {
      int32_t om = (int32_t)(ev >> 8), h = (int32_t)(ev & 255u);
      const double *t = gwt + h * GRS_GWT;
      b1_out o;
      o.ry = o.rz = 0.0;
      o.dy = o.dz = 0;
      o.win = 0;
      const double *brow = btab ? btab + GRS_BT * om : nullptr;
      const double cc = brow ? brow[10] : a.cs[2 * om], ss = brow ? brow[11] : a.cs[2 * om + 1];
      st = b1_classify<true>(g, cc, ss, Pw, brow, t, b1thr, &o);
      if (st == 1)
        idx = tiled ? grs_tiled_bit((uint32_t)om, (uint32_t)o.dy, (uint32_t)o.dz, ntz, nty)
                    : (uint32_t)(o.dz - 1) + (uint32_t)(o.dy - 1) * nz32 + (uint32_t)om * nzny32;
      inwin = o.win != 0;
      if (AUDIT) {
        double yz[2] = {0.0, 0.0};
        uint32_t eidx = 0;
        const int es = exact_event(a.g, vpos, a.cs, gwt, ev, &eidx, yz);
        bad = (st == 0 && es) || (st == 1 && (!es || eidx != idx));
        if (st == 1 && es) dev = __builtin_fmax(__builtin_fabs(o.ry - yz[0]), __builtin_fabs(o.rz - yz[1]));
      }
    }
    if (AUDIT) {
      /* whole-wave reductions, outside the divergent block */
      uint64_t mb = __ballot(bad), m1 = __ballot(st == 1), m0 = __ballot(valid && st == 0);
      uint64_t m2 = __ballot(st == 2), mw = __ballot(inwin);
      for (int off = 32; off >= 1; off >>= 1) dev = __builtin_fmax(dev, __shfl_xor(dev, off, 64));
      if (lane == 0) {
        atomicAdd(a.audit + 0, (unsigned long long)n);
        atomicAdd(a.audit + 1, (unsigned long long)__popcll(m1));
        atomicAdd(a.audit + 2, (unsigned long long)__popcll(m0));
        atomicAdd(a.audit + 3, (unsigned long long)__popcll(m2));
        atomicAdd(a.audit + 4, (unsigned long long)__popcll(mb));
        atomicMax(a.audit + 5, (unsigned long long)__double_as_longlong(dev));
        atomicAdd(a.audit + 6, (unsigned long long)__popcll(mw));
      }
    }
    uint64_t m2 = __ballot(st == 2);
    if (st == 2) ring2[(tail2 + lane_prefix(m2)) & (GRS_QCAP - 1)] = ev;
    tail2 += (uint32_t)__popcll(m2);
    push3(st == 1, idx);
    if (tail2 - head2 >= 64) {
      wave_sync();
      b2(64);
      wave_sync();
    }
  };

  auto b1 = [&](uint32_t n) {
    const bool valid = (uint32_t)lane < n;
    const uint32_t ev = valid ? ring1[(head1 + lane) & (GRS_QCAP - 1)] : 0u;
    head1 += n;
    b1_core(valid, ev, n);
  };

  if (solve && !overflow) {
    /* candidates of the omega solve, 64 per step, straight to phase B1.
     * Ranges are non-empty and rcum is their exclusive prefix, so the range
     * of a candidate is the number of set bits up to its own in the bitmap
     * of first candidates, less one.  (Marks written and read back on every
     * step: 27.0 instead of 26.7 ms for 1,024 voxels x 343 x 7.9 samples; the
     * range looked up one step ahead: 27.0.) */
    uint32_t rb = 0xFFFFFFFFu; /* set bits before base, less one */
    for (uint32_t base = 0; base < total; base += 64) {
      const uint32_t at = base & (GRS_QCAP * 32u - 1u);
      if (base > 0 && at == 0) {
        /* the next GRS_QCAP * 32 candidates */
        wave_sync();
        for (int k = lane; k < GRS_QCAP; k += 64) ring1[k] = 0u;
        wave_sync();
        for (uint32_t r = lane; r < R; r += 64) {
          const uint32_t p = rcum[r] - base;
          if (p < GRS_QCAP * 32u) atomicOr(&ring1[p >> 5], 1u << (p & 31u));
        }
        wave_sync();
      }
      const uint32_t idx = base + (uint32_t)lane;
      const bool valid = idx < total;
      const uint32_t m0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)ring1[at >> 5]);
      const uint32_t m1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)ring1[(at >> 5) + 1]);
      const uint64_t starts = ((uint64_t)m1 << 32) | m0;
      const uint32_t r = rb + lane_prefix(starts) + (uint32_t)((starts >> lane) & 1ull);
      rb += (uint32_t)__popcll(starts);
      uint32_t ev = 0;
      if (valid) {
        const uint32_t st0 = rstart[r];
        ev = (((st0 >> 8) + (idx - rcum[r])) << 8) | (st0 & 255u);
      }
      b1_core(valid, ev, total - base < 64u ? total - base : 64u);
    }
  }
  /* phase A (no omega solve): wave-uniform steps of 64 consecutive events;
   * lane l owns event l + 64*k, tracked as (omega, hkl) without divisions */
  const int32_t Hn = hend - hlo;
  int32_t om = 0, h = hlo;
  int32_t nsteps = 0;
  if (!(solve && !overflow) && Hn > 0) {
    nsteps = (nrot * Hn + 63) / 64;
    om = lane / Hn;
    h = hlo + (lane - om * Hn);
  }
  for (int32_t k = 0; k < nsteps; ++k) {
    bool pass = false;
    if (om < nrot) {
      const double c = a.cs[2 * om], s = a.cs[2 * om + 1];
      double swv[3], uv[3];
      beam_terms(g, Pw, c, s, swv, uv);
      const double u0 = uv[0], u1 = uv[1], u2 = uv[2];
      const double *t = gwt + h * GRS_GWT;
      double Gt0 = c * t[0] - s * t[1];
      double Gt1 = s * t[0] + c * t[1];
      double dot = __builtin_fma(u2, t[2], __builtin_fma(u1, Gt1, u0 * Gt0));
      double l4 = m4pi * dot;
      /* the phase-A thresholds of the reflection (margins: see the header comment) */
      const double gn = __builtin_sqrt(t[4]);
      const double ml = lrel + (1e-12 * (4.0 * GRS_PI)) * t[3];
      pass = (dot < dcb * gn) && (dot > cbm * gn) && (l4 > (lmin - ml) * t[4]) && (l4 < (lmax + ml) * t[4]);
    }
    uint64_t m = __ballot(pass);
    if (pass) ring1[(tail1 + lane_prefix(m)) & (GRS_QCAP - 1)] = ((uint32_t)om << 8) | (uint32_t)h;
    tail1 += (uint32_t)__popcll(m);
    if (tail1 - head1 >= 64) {
      wave_sync();
      b1(64);
      wave_sync();
    }
    h += 64;
    while (h >= hend) {
      h -= Hn;
      om++;
    }
  }
  while (tail1 != head1) {
    uint32_t n = tail1 - head1;
    if (n > 64) n = 64;
    wave_sync();
    b1(n);
    wave_sync();
  }
  while (tail2 != head2) {
    uint32_t n = tail2 - head2;
    if (n > 64) n = 64;
    wave_sync();
    b2(n);
    wave_sync();
  }
  while (tail3 != head3) {
    uint32_t n = tail3 - head3;
    if (n > 64) n = 64;
    wave_sync();
    gather(n);
    wave_sync();
  }
  consume();
  *ns_out = ns;
  *ni_out = ni;
}

template <bool MEDIAN, int MAP, bool AUDIT, bool TEAM>
__global__ __launch_bounds__(64 * GRS_WPB, GRS_FAST_MIN_WAVES) void k_fast(grs_eval_args a, int32_t H) {
  extern __shared__ double smem[];
  const int lane = threadIdx.x & 63;
  const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); /* uniform: a wave's addresses and bounds stay scalar */
  /* a team's waves split the reflections evenly */
  const int32_t Hn = TEAM ? (H + (int)(blockDim.x >> 6) - 1) / (int)(blockDim.x >> 6) : H;
  const int32_t hlo = TEAM ? (wib * Hn < H ? wib * Hn : H) : 0, hend = hlo + Hn < H ? hlo + Hn : H;
  const int64_t per_wave = fast_wave_doubles(Hn);
  const fast_lds_regions L = fast_regions(smem, wib, hlo, Hn);
  /* the geometry constants live in LDS: the loop bodies read ~30 of them per
   * batch, and neither scalar registers (spilled) nor vector loads (the
   * compiler cannot prove them unchanged across the loop's stores) serve */
  __shared__ grs_dgeo sg;
  __shared__ double b1thr[12]; /* b1_thresholds */
  __shared__ int32_t team[3];  /* TEAM: ns, ni and the keys listed so far */
  if (threadIdx.x == 0) {
    sg = *a.g;
    b1_thresholds(&sg, b1thr);
  }
  __syncthreads();
  const grs_dgeo *g = &sg;
  const int wpb = (int)(blockDim.x >> 6);
  /* one voxel for every evaluation: its per-omega beam terms are computed
   * once per block into LDS behind the per-wave regions (the launch sizes
   * the allocation with the same rule) */
  const double *btab = nullptr;
  if (!TEAM && MAP == GRS_MAP_ONE_VOXEL && a.nrot == g->nrot && fast_tab_doubles(MAP, a.nrot, H, wpb) > 0 &&
      a.e0 < a.n_eval) {
    double *bt = smem + (int64_t)wpb * per_wave;
    double P[3];
    voxel_P(g, a.pos, P);
    for (int32_t om = (int32_t)threadIdx.x; om < g->nrot; om += (int32_t)blockDim.x) {
      beam_row(g, P, a.cs[2 * om], a.cs[2 * om + 1], bt + GRS_BT * om);
    }
    __syncthreads();
    btab = bt;
  }
  /* blocks are dealt to the 8 XCDs in turn (block b on XCD b mod 8): with
   * xcd_map, block b takes the place b / 8 + (b mod 8) * gridDim.x / 8 in
   * the evaluation order, so that each XCD's L2 sees a contiguous run of
   * evaluations (neighbouring samples of a CSR row share detector tiles) */
  int64_t vblock = blockIdx.x;
  if (a.xcd_map && (gridDim.x & 7u) == 0u) vblock = (int64_t)(blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  /* an evaluation per wave, or per block of a team */
  const int64_t gwave = TEAM ? vblock : vblock * wpb + wib;
  const int64_t nwaves = TEAM ? gridDim.x : (int64_t)gridDim.x * wpb;
  uint32_t *wlist = MEDIAN ? a.scratch + gwave * a.scratch_stride : nullptr;
  int64_t row_hint = -1;
  for (int64_t e = a.e0 + gwave; e < a.n_eval; e += nwaves) {
    int64_t vi, row, jloc;
    double sub[9];
    int ok = eval_setup<MAP>(a, e, &vi, sub, &row, &jloc, &row_hint);
    if (ok <= 0) {
      if (!MEDIAN) {
        /* a skipped orientation counts as C = NaN for the argmax; in a grid
         * it has C = 0 */
        if (MAP == GRS_MAP_GRID) {
          if (lane == 0) grid_counts_out(a, e, 0, 0, false);
        } else if (lane == 0 && ok == 0) {
          atomicMax(a.csr.row_best + row, (unsigned long long)(((1ull << GRS_KEY_JBITS) - 1) - (uint64_t)jloc));
        }
      } else if (lane == 0 && (!TEAM || wib == 0)) {
        a.out_ns[e] = 0;
        a.out_ni[e] = 0;
        a.out_C[e] = 0.0;
        a.out_med[e] = 0.0f;
      }
      continue;
    }
    int32_t ns, ni;
    if (TEAM) {
      if (threadIdx.x == 0) team[0] = team[1] = team[2] = 0;
      __syncthreads();
    }
    if (MAP == GRS_MAP_GRID)
      btab = a.beam ? a.beam + (int64_t)GRS_BT * a.nrot * vi : nullptr;
    score_events<MEDIAN, AUDIT, TEAM>(a, g, b1thr, btab, L, sub, vi, hlo, hend, wlist, &team[2], &ns, &ni);
    if (TEAM) {
      if (lane == 0) {
        atomicAdd(&team[0], ns);
        atomicAdd(&team[1], ni);
      }
      __threadfence_block();
      __syncthreads();
      /* the first wave closes the evaluation; the others wait for it where
       * the counters are cleared */
      if (wib != 0) continue;
      ns = team[0];
      ni = team[1];
    }
    if (MEDIAN) {
      __threadfence_block();
      float med = 2000.0f;
      if (ns > 0) med = wave_median(wlist, ns, lane);
      if (lane == 0) {
        a.out_ns[e] = ns;
        a.out_ni[e] = ni;
        a.out_C[e] = (double)ni / (double)ns;
        a.out_med[e] = med;
      }
    } else if (MAP == GRS_MAP_GRID) {
      if (lane == 0) grid_counts_out(a, e, ns, ni, true);
    } else if (lane == 0) {
      uint64_t jpart = ((1ull << GRS_KEY_JBITS) - 1) - (uint64_t)jloc;
      uint64_t cpart = 0;
      if (ns > 0) {
        double C = (double)ni / (double)ns;
        cpart = (uint64_t)__builtin_floor(C * 1073741824.0) + 1ull;
      }
      atomicMax(a.csr.row_best + row, (unsigned long long)((cpart << GRS_KEY_JBITS) | jpart));
    }
    wave_sync();
  }
}

/* ---------------------------------------------------------------------- */
/* orientation fits                                                        */

/* One block per fit of 1 - Nr_intersect/Nr_simu over (q1, q2, q3)
 * (fit_OR_constrain_with_local_comp_cuda.m:116-126): the whole
 * fminsearchbnd on the device.  The block's 16 waves are four teams of four
 * (score_events with the reflections split four ways), one team per point: a
 * requested reflection is scored together with the three points that its
 * value can lead to (grs_nm::points), the initial simplex and a shrink
 * have at most four points.  The first wave steps the method
 * (nm_lanes).  The points, values and counts are the sequential method's.
 * Bound: one iteration's chain (a wave's events of 22 of 86 reflections, the step
 * of the simplex and the barriers between).  A launch, two copies and a
 * synchronisation per iteration took 3.3 ms for 24 fits of 64 iterations
 * (52 us each, 36 of them one wave's walk through all events); this takes
 * 1.3 ms.  GRS_FIT_SLICE requests end a launch, so that it ends whatever max_iter
 * is; the host launches again while fits are left. */
#define GRS_FIT_TEAM 4
#define GRS_FIT_PTS 4
#define GRS_FIT_SLICE 4096

__global__ __launch_bounds__(64 * GRS_FIT_TEAM * GRS_FIT_PTS, GRS_FAST_MIN_WAVES) void k_fit_nm(
    grs_eval_args a, int32_t H, const double *x0, double half_width, int32_t max_fe, int32_t max_it, double tol_f,
    double tol_x, int32_t first, grs_nm *nms, double *res, int32_t *left) {
  GRS_NO_CONTRACT
  extern __shared__ double smem[];
  __shared__ __align__(16) unsigned char nm_buf[sizeof(grs_nm)];
  __shared__ double xs[GRS_FIT_PTS][3];
  __shared__ grs_dgeo sg;
  __shared__ double b1thr[12];
  __shared__ int32_t cnt[GRS_FIT_PTS][2];
  __shared__ double fs[GRS_FIT_PTS];
  __shared__ int npts;
  grs_nm *nm = reinterpret_cast<grs_nm *>(nm_buf);
  const int t = threadIdx.x, lane = t & 63, wib = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t m = blockIdx.x;
  const int p = wib / GRS_FIT_TEAM, w = wib % GRS_FIT_TEAM;
  const int32_t Hn = (H + GRS_FIT_TEAM - 1) / GRS_FIT_TEAM;
  const int32_t hlo = w * Hn < H ? w * Hn : H, hend = hlo + Hn < H ? hlo + Hn : H;
  const fast_lds_regions L = fast_regions(smem, wib, hlo, Hn);
  if (t == 0) {
    sg = *a.g;
    b1_thresholds(&sg, b1thr);
    if (first) {
      double lo[3], hi[3], xm[3];
      for (int k = 0; k < 3; k++) {
        /* fit_OR_constrain_with_local_comp_cuda.m:124-125 */
        xm[k] = x0[3 * m + k];
        const double u = xm[k] - half_width, v = xm[k] + half_width;
        lo[k] = grs_nm_max(u, -1.0);
        hi[k] = (v != v) ? 1.0 : (v < 1.0 ? v : 1.0);
      }
      nm->max_fe = max_fe;
      nm->max_it = max_it;
      nm->tol_f = tol_f;
      nm->tol_x = tol_x;
      nm->nf = 0;
      nm->it = 0;
      nm->start(3, xm, lo, hi);
    } else {
      *nm = nms[m];
    }
  }
  __syncthreads();
  int32_t step = 0;
  for (; step < GRS_FIT_SLICE; step++) {
    if (t == 0) npts = nm->points();
    if (t < 2 * GRS_FIT_PTS) cnt[t >> 1][t & 1] = 0;
    __syncthreads();
    const int np = npts;
    if (np == 0) break;
    if (t < 3 * np) {
      const int q = t / 3, k = t - 3 * q;
      double u = nm->pend[q][k];
      if (nm->st == grs_nm::REFLECT && q > 0) {
        const double xb = nm->xbar[k], vn = nm->v[nm->n][k];
        u = GRS_NM_FOLLOW_UP(q, xb, vn);
      }
      double u3[3];
      u3[k] = u;
      nm->xform1(u3, k, &xs[q][k]);
    }
    __syncthreads();
    double U[9], sub[9];
    if (p < np && grs_U_from_q(xs[p][0], xs[p][1], xs[p][2], U)) {
      grs_SUB(a.g, U, sub);
      int32_t ns, ni;
      score_events<false, false, true>(a, &sg, b1thr, a.beam + (int64_t)GRS_BT * a.nrot * m, L, sub, m, hlo, hend, nullptr, nullptr, &ns, &ni);
      if (lane == 0) {
        atomicAdd(&cnt[p][0], ns);
        atomicAdd(&cnt[p][1], ni);
      }
    }
    __syncthreads();
    if (wib == 0) {
      /* fit_OR_fun_local.m:98; 0/0 (no event, or |q_vec| > 1) is NaN */
      if (t < GRS_FIT_PTS) fs[t] = 1.0 - (double)cnt[t][1] / (double)cnt[t][0];
      wave_sync();
      nm_lanes<3> S(nm, t);
      S.step(fs);
      S.store();
    }
    __syncthreads();
  }
  if (t == 0) {
    nms[m] = *nm;
    if (!nm->done()) atomicAdd(left, 1);
    double *r = res + 6 * m;
    nm->result(r, r + 3);
    r[4] = (double)nm->nf;
    r[5] = (double)nm->it;
  }
}

/* ---------------------------------------------------------------------- */
/* batched compete: device-side steps between and after the two launches   */

__global__ void k_fill_u32(uint32_t *p, int64_t n, uint32_t v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_fill_u64(unsigned long long *p, int64_t n, unsigned long long v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

/* winner of each CSR row from its packed argmax key: the index of the
 * first maximum in the expanded list (-1 for an empty row) */
__global__ void k_winner_list(const unsigned long long *row_best, const int64_t *row_eoff, int64_t m, int64_t *elist) {
  int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= m) return;
  if (row_eoff[r + 1] == row_eoff[r]) {
    elist[r] = -1;
    return;
  }
  const unsigned long long jmask = (1ull << GRS_KEY_JBITS) - 1;
  elist[r] = row_eoff[r] + (int64_t)(jmask - (row_best[r] & jmask));
}

/* best index in the row's expanded list and its quaternion (the local
 * sample of the grid, q0 from the vector part, 0 when |q_vec| > 1) */
__global__ void k_winner_out(const int64_t *elist, const int64_t *row_eoff, const int64_t *row_ptr,
                             const double *cand_q, int32_t nr, double gridsize, int64_t m, int64_t *best,
                             double *best_q) {
  GRS_NO_CONTRACT
  int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= m) return;
  double *bq = best_q + 4 * r;
  if (elist[r] < 0) {
    best[r] = -1;
    bq[0] = bq[1] = bq[2] = bq[3] = 0.0;
    return;
  }
  const int64_t n1 = nr + 1, S = n1 * n1 * n1;
  const int64_t j = elist[r] - row_eoff[r];
  const int64_t cand = row_ptr[r] + j / S;
  const int64_t smp = j % S;
  const int64_t k[3] = {smp / (n1 * n1), (smp / n1) % n1, smp % n1};
  const double *q = cand_q + 4 * cand;
  const double half = (gridsize * (double)nr) / 2.0;
  double v[3];
  for (int t = 0; t < 3; t++) v[t] = (q[1 + t] - half) + (double)k[t] * gridsize;
  const double ss = (v[0] * v[0] + v[1] * v[1]) + v[2] * v[2];
  bq[0] = ss <= 1.0 ? __builtin_sqrt(1.0 - ss) : 0.0;
  bq[1] = v[0];
  bq[2] = v[1];
  bq[3] = v[2];
  best[r] = j;
}

/* bit i of the hit mask = (keys[i] <= hit_key) */
__global__ void k_pack_hits(const uint32_t *keys, int64_t n, uint32_t hit_key, int32_t has_hit, uint32_t *bits) {
  int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t nw = (n + 31) >> 5;
  if (w >= nw) return;
  uint32_t b = 0;
  if (has_hit) {
    for (int k = 0; k < 32; k++) {
      int64_t i = (w << 5) + k;
      if (i < n && keys[i] <= hit_key) b |= 1u << k;
    }
  }
  bits[w] = b;
}

/* the same mask in 32 x 32 pixel tiles (grs_tiled_bit): thread per 32-bit
 * word, word = tile * 32 + (dy - 1) mod 32, bit = (dz - 1) mod 32; pixels
 * outside the stack are 0 */
__global__ void k_pack_hits_tiled(const uint32_t *keys, int64_t nz, int64_t ny, int64_t nw, uint32_t ntz,
                                  uint32_t nty, uint32_t hit_key, int32_t has_hit, uint32_t *tbits) {
  const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= nw) return;
  const int64_t tile = w >> 5;
  const int64_t tz = tile % ntz, rest = tile / ntz;
  const int64_t ty = rest % nty, om = rest / nty;
  const int64_t y = ty * 32 + (w & 31);
  uint32_t b = 0;
  if (has_hit && y < ny) {
    const uint32_t *col = keys + (om * ny + y) * nz;
    for (int k = 0; k < 32; k++) {
      const int64_t z = tz * 32 + k;
      if (z < nz && col[z] <= hit_key) b |= 1u << k;
    }
  }
  tbits[w] = b;
}

/* ---------------------------------------------------------------------- */
/* k_plain                                                                 */

__device__ uint32_t plain_select(uint32_t *A, int64_t T, int32_t n, int32_t k) {
  int32_t lo = 0, hi = n - 1;
  while (lo < hi) {
    uint32_t pivot = A[(int64_t)((lo + hi) >> 1) * T];
    int32_t i = lo, j = hi;
    while (i <= j) {
      while (A[(int64_t)i * T] < pivot) i++;
      while (A[(int64_t)j * T] > pivot) j--;
      if (i <= j) {
        uint32_t tmp = A[(int64_t)i * T];
        A[(int64_t)i * T] = A[(int64_t)j * T];
        A[(int64_t)j * T] = tmp;
        i++;
        j--;
      }
    }
    if (k <= j) hi = j;
    else if (k >= i) lo = i;
    else break;
  }
  return A[(int64_t)k * T];
}

__global__ __launch_bounds__(256) void k_plain(grs_eval_args a, int64_t T) {
  int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= T) return;
  const grs_dgeo *g = a.g;
  const int32_t nrot = g->nrot, H = g->H;
  uint32_t *buf = a.scratch + tid; /* element j at buf[j*T] */
  for (int64_t e = tid; e < a.n_eval; e += T) {
    int64_t vi, ui;
    eval_slots(a, e, &vi, &ui);
    if (!a.valid[ui]) {
      a.out_ns[e] = 0;
      a.out_ni[e] = 0;
      a.out_C[e] = 0.0;
      a.out_med[e] = 0.0f;
      continue;
    }
    const double *SUB = a.SUB + ui * 9;
    const double *pos = a.pos + vi * 3;
    int32_t ns = 0, ni = 0;
    for (int32_t om = 0; om < nrot; om++) {
      grs_vw v;
      grs_vw_terms(g, pos, a.cs[2 * om], a.cs[2 * om + 1], &v);
      for (int32_t h = 0; h < H; h++) {
        double gw[3], Gt[3], Glen;
        grs_Gw(SUB, a.hkl + 3 * h, gw);
        grs_Gt(v.c, v.s, gw[0], gw[1], gw[2], Gt);
        double beta = grs_event_beta(&v, Gt, &Glen);
        int32_t dy, dz;
        if (grs_event_finish(g, &v, Gt, Glen, beta, &dy, &dz)) {
          uint32_t key = a.keys[(int64_t)(dz - 1) + (int64_t)(dy - 1) * g->nz + (int64_t)om * g->nz * g->ny];
          buf[(int64_t)ns * T] = key;
          ns++;
          if (g->has_hit && key <= g->hit_key) ni++;
        }
      }
    }
    float med = 2000.0f;
    if (ns > 0) {
      int32_t k1 = (ns & 1) ? (ns >> 1) : (ns >> 1) - 1;
      uint32_t v1 = plain_select(buf, T, ns, k1);
      if (ns & 1) {
        med = key_to_float(v1);
      } else {
        uint32_t v2 = 0xFFFFFFFFu;
        for (int32_t j = k1 + 1; j < ns; j++) {
          uint32_t x = buf[(int64_t)j * T];
          v2 = x < v2 ? x : v2;
        }
        float fa = key_to_float(v1), fb = key_to_float(v2);
        med = fa + (fb - fa) / 2.0f;
      }
    }
    a.out_ns[e] = ns;
    a.out_ni[e] = ni;
    a.out_C[e] = (double)ni / (double)ns;
    a.out_med[e] = med;
  }
}

/* ---------------------------------------------------------------------- */
/* voxel rows of cuda_grow_indexed_region                                  */

/* The rows [x y z C mask DisMedian] stay on the device as they came: block b
 * of GROW_T rows counts its rows inside the mask, k_grow_list gives row i its
 * place among the scored ones (slot, -1 outside the mask) and writes the
 * position there, k_grow_out forms the 7 output values and the growth flag.
 * Bound: 48 bytes in and 56 out per row; on the host the same loops and their
 * copies took about 40 ms for 3.2M rows, the three kernels take 0.28 ms.
 * They stand in this file because a process loads each file's kernels at the
 * first launch of one of them, 0.8 ms of its first growth call. */
#define GROW_T 256

__device__ __forceinline__ int64_t grow_block_sum(int32_t v, int32_t *part) {
  const uint64_t lanes = 64;
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, (int)lanes);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  int64_t s = 0;
  for (int k = 0; k < GROW_T / 64; k++) s += part[k];
  __syncthreads();
  return s;
}

__global__ __launch_bounds__(GROW_T) void k_grow_count(const double *rows, int64_t M, int32_t *count) {
  __shared__ int32_t part[GROW_T / 64];
  const int64_t i = (int64_t)blockIdx.x * GROW_T + threadIdx.x;
  const int64_t n = grow_block_sum(i < M && rows[6 * i + 4] > 0.0 ? 1 : 0, part);
  if (threadIdx.x == 0) count[blockIdx.x] = (int32_t)n;
}

/* count: rows inside the mask per block, or nullptr when every row is inside;
 * total receives their sum */
__global__ __launch_bounds__(GROW_T) void k_grow_list(const double *rows, int64_t M, const double *p1,
                                                      const int32_t *count, double *pos, int32_t *slot,
                                                      int64_t *total) {
  __shared__ int32_t part[GROW_T / 64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t b = blockIdx.x, i = b * GROW_T + threadIdx.x;
  int64_t k = i;
  bool in = i < M;
  if (count) {
    int32_t before = 0;
    for (int64_t j = threadIdx.x; j < b; j += GROW_T) before += count[j];
    const int64_t base = grow_block_sum(before, part);
    in = in && rows[6 * i + 4] > 0.0;
    const uint64_t m = __ballot(in);
    if (lane == 0) part[wv] = (int32_t)__popcll(m);
    __syncthreads();
    k = base + __popcll(lane == 0 ? 0ull : m & (~0ull >> (64 - lane)));
    for (int w = 0; w < wv; w++) k += part[w];
    if (total && b == (int64_t)gridDim.x - 1 && threadIdx.x == 0) *total = base + count[b];
  }
  if (i < M) slot[i] = in ? (int32_t)k : -1;
  if (in) grs_voxel_pos(rows[6 * i], rows[6 * i + 1], rows[6 * i + 2], p1, pos + 3 * k);
}

__global__ __launch_bounds__(GROW_T) void k_grow_out(const double *rows, int64_t M, const double *p1,
                                                     const int32_t *slot, const int32_t *ns, const int32_t *ni,
                                                     const double *C, const float *med, double *out) {
  GRS_NO_CONTRACT
  const int64_t i = (int64_t)blockIdx.x * GROW_T + threadIdx.x;
  if (i >= M) return;
  const double *v = rows + 6 * i;
  double *o = out + 7 * i;
  o[0] = v[0];
  o[1] = v[1];
  o[2] = v[2];
  const int32_t k = slot[i];
  if (k < 0) {
    o[3] = o[4] = o[5] = o[6] = 0.0;
    return;
  }
  const double Cn = C[k], dm = (double)med[k];
  /* min([DisMedian maxDmedian]) with MATLAB's NaN rule */
  const double a = v[5], b = p1[13];
  const double lim = a != a ? b : (b != b ? a : (b < a ? b : a));
  const bool flag = (Cn > v[3] && dm <= lim) && (Cn >= p1[11] * (1.0 - p1[12]));
  o[3] = (double)ns[k];
  o[4] = (double)ni[k];
  o[5] = dm;
  o[6] = flag ? 1.0 : 0.0;
}

/* ---------------------------------------------------------------------- */
/* compete: first maximum of C per voxel row, NaN never wins              */

__global__ __launch_bounds__(256) void k_compete_ids(const double *ids, int64_t n_id, int64_t G,
                                                     unsigned long long *bad) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (j >= n_id) return;
  const double g = ids[j];
  if (!(g >= 1.0 && g <= (double)G && g == __builtin_floor(g))) atomicMin(bad, (unsigned long long)j);
}

/* one wave per row: its position and its evaluations */
__global__ __launch_bounds__(256) void k_compete_list(const double *vox, int64_t M, const int64_t *rs,
                                                      const double *ids, int64_t G, const double *p1, double *pos,
                                                      int32_t *evox, int32_t *eu) {
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= M) return;
  const double *v = vox + 5 * r;
  if (lane == 0) grs_voxel_pos(v[0], v[1], v[2], p1, pos + 3 * r);
  const int64_t e0 = rs[r], n = rs[r + 1] - e0, lo = (int64_t)v[3] - 1;
  for (int64_t k = lane; k < n; k += 64) {
    const double g = ids[lo + k];
    evox[e0 + k] = (int32_t)r;
    eu[e0 + k] = g >= 1.0 && g <= (double)G ? (int32_t)g - 1 : 0;
  }
}

__global__ void k_compete_out(const int64_t *rs, int64_t M, int64_t row0, const int32_t *eu, const double *euler,
                              const int32_t *ni, const double *C, const float *med, double *out) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= M) return;
  const int64_t a = rs[r], b = rs[r + 1];
  int64_t bi = -1;
  double bc = 0.0;
  for (int64_t j = a; j < b; j++) {
    const double c = C[j];
    if (c == c && (bi < 0 || c > bc)) {
      bi = j;
      bc = c;
    }
  }
  if (bi < 0 && b > a) bi = a;
  double *o = out + 8 * r;
  o[0] = (double)(row0 + r + 1);
  if (bi < 0) {
    for (int t = 1; t < 8; t++) o[t] = 0.0;
    return;
  }
  const int32_t g = eu[bi];
  o[1] = euler[3 * (int64_t)g];
  o[2] = euler[3 * (int64_t)g + 1];
  o[3] = euler[3 * (int64_t)g + 2];
  o[4] = (double)(g + 1);
  o[5] = C[bi];
  o[6] = (double)ni[bi];
  o[7] = (double)med[bi];
}

/* ---------------------------------------------------------------------- */
/* launchers                                                               */

static inline unsigned blocks_for(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

hipError_t grs_launch_omega_cs(const double *d_rot, int32_t nrot, double *d_cs, hipStream_t st) {
  if (nrot <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_omega_cs, dim3(blocks_for(nrot, 256)), dim3(256), 0, st, d_rot, nrot, d_cs);
  return hipGetLastError();
}

hipError_t grs_launch_voxel_pos(const double *d_rows, int64_t M, int32_t stride, const double *d_p1, double *d_pos,
                                hipStream_t st) {
  if (M <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_voxel_pos, dim3(blocks_for(M, 256)), dim3(256), 0, st, d_rows, M, stride, d_p1, d_pos);
  return hipGetLastError();
}

hipError_t grs_launch_beam(const grs_dgeo *d_g, const double *d_pos, int64_t V, const double *d_cs, int32_t nrot,
                           double *d_beam, hipStream_t st) {
  if (V <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_beam, dim3(blocks_for(V * nrot, 256)), dim3(256), 0, st, d_g, d_pos, V, d_cs, nrot, d_beam);
  return hipGetLastError();
}

hipError_t grs_launch_voxel_bounds(const grs_dgeo *d_g, const double *d_pos, int64_t V, const double *d_cs,
                                   int32_t nrot, double *d_vb, hipStream_t st) {
  if (V <= 0) return hipSuccess;
  if (V > 0x7fffffff) return hipErrorInvalidValue;
  /* a block per voxel below a thousand (the latency of a walk over the angles
   * counts: 6 us for one voxel), else enough lanes per voxel for about eight
   * waves per SIMD of 256 CUs */
  if (V < 1024)
    hipLaunchKernelGGL(k_voxel_bounds, dim3((unsigned)V), dim3(256), 0, st, d_g, d_pos, d_cs, nrot, d_vb);
  else if (V < 32768)
    hipLaunchKernelGGL(k_voxel_bounds_lanes<16>, dim3((unsigned)((V * 16 + 255) / 256)), dim3(256), 0, st, d_g, d_pos,
                       V, d_cs, nrot, d_vb);
  else if (V < 262144)
    hipLaunchKernelGGL(k_voxel_bounds_lanes<4>, dim3((unsigned)((V * 4 + 255) / 256)), dim3(256), 0, st, d_g, d_pos,
                       V, d_cs, nrot, d_vb);
  else
    hipLaunchKernelGGL(k_voxel_bounds_lanes<1>, dim3((unsigned)((V + 255) / 256)), dim3(256), 0, st, d_g, d_pos, V,
                       d_cs, nrot, d_vb);
  return hipGetLastError();
}

hipError_t grs_launch_one_voxel(const grs_dgeo *d_g, const double *pos, const double *d_cs, int32_t nrot,
                                const double *d_q, int64_t N, double *d_pos, double *d_vb, double *d_SUB,
                                int32_t *d_valid, hipStream_t st) {
  one_pos at = {{pos[0], pos[1], pos[2]}};
  hipLaunchKernelGGL(k_one_voxel, dim3((unsigned)(1 + (N + 255) / 256)), dim3(256), 0, st, d_g, at, d_cs, nrot, d_q, N,
                     d_pos, d_vb, d_SUB, d_valid);
  return hipGetLastError();
}

hipError_t grs_launch_sub_from_q(const grs_dgeo *d_g, const double *d_q, int64_t N, double *d_SUB, int32_t *d_valid,
                                 hipStream_t st) {
  if (N <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sub_from_q, dim3(blocks_for(N, 256)), dim3(256), 0, st, d_g, d_q, N, d_SUB, d_valid);
  return hipGetLastError();
}

hipError_t grs_launch_sub_from_U(const grs_dgeo *d_g, const double *d_U, int64_t N, double *d_SUB, int32_t *d_valid,
                                 hipStream_t st) {
  if (N <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sub_from_U, dim3(blocks_for(N, 256)), dim3(256), 0, st, d_g, d_U, N, d_SUB, d_valid);
  return hipGetLastError();
}

hipError_t grs_launch_sub_from_euler(const grs_dgeo *d_g, const double *d_eu, int64_t N, double *d_SUB,
                                     int32_t *d_valid, hipStream_t st) {
  if (N <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sub_from_euler, dim3(blocks_for(N, 256)), dim3(256), 0, st, d_g, d_eu, N, d_SUB, d_valid);
  return hipGetLastError();
}

static size_t fast_lds(int32_t H, int wpb, const grs_eval_args *a) {
  return (size_t)((int64_t)wpb * fast_wave_doubles(H) + fast_tab_doubles(a->map, a->nrot, H, wpb)) * sizeof(double);
}

/* Resident blocks per CU of one k_fast instantiation at wpb waves per block
 * (cached per wpb). */
template <bool MEDIAN, int MAP, bool AUDIT, bool TEAM>
static int fast_blocks_per_cu(size_t lds, int wpb) {
  static int cached[GRS_WPB + 1] = {0};
  static size_t cached_lds[GRS_WPB + 1] = {0};
  if (cached[wpb] == 0 || cached_lds[wpb] != lds) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_fast<MEDIAN, MAP, AUDIT, TEAM>, 64 * wpb, lds) != hipSuccess ||
        nb <= 0)
      nb = 1;
    cached[wpb] = nb;
    cached_lds[wpb] = lds;
  }
  return cached[wpb];
}

static int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    cus = 256;
  return cus;
}

/* Persistent launch: at most as many waves as can be resident at once.
 * TEAM: the block's waves share each evaluation. */
template <bool MEDIAN, int MAP, bool AUDIT = false, bool TEAM = false>
static hipError_t launch_fast_impl(const grs_eval_args *a, int32_t H, int64_t n_waves, int wpb, hipStream_t st) {
  if (wpb != 1 && wpb != 2 && wpb != 4 && wpb != 8) return hipErrorInvalidValue;
  /* every wave (team) of the launch needs a scratch slot: fewer slots than a
   * block has waves take smaller blocks */
  while (!TEAM && wpb > 1 && n_waves < wpb) wpb >>= 1;
  size_t lds = TEAM ? (size_t)wpb * (size_t)fast_wave_doubles((H + wpb - 1) / wpb) * sizeof(double) : fast_lds(H, wpb, a);
  if (lds > 65536) {
    /* above the default dynamic LDS limit of a launch */
    hipError_t e = hipFuncSetAttribute((const void *)k_fast<MEDIAN, MAP, AUDIT, TEAM>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  int64_t resident = (int64_t)device_cus() * fast_blocks_per_cu<MEDIAN, MAP, AUDIT, TEAM>(lds, wpb);
  int64_t blocks = TEAM ? a->n_eval - a->e0 : n_waves / wpb; /* n_waves is a multiple of 4: no wave beyond the scratch slots */
  if (TEAM && blocks > n_waves) blocks = n_waves;
  if (blocks > resident) blocks = resident;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL((k_fast<MEDIAN, MAP, AUDIT, TEAM>), dim3((unsigned)blocks), dim3(64 * wpb), lds, st, *a, H);
  return hipGetLastError();
}

/* Waves that share an evaluation in a launch of n evaluations (1: none).
 * While the chip has more SIMDs than evaluations the call takes as long as
 * one wave's walk through an evaluation's events, and splitting the
 * reflections shortens it; the set-up is repeated by every wave, so larger launches
 * lose.  A one-voxel call of 100, 300, 729, 1500, 2187, 4000 orientations (86
 * reflections, 181 angles; whole call on resident buffers, us): a wave each
 * 44, 73, 69, 78, 75, 71; two 37, 40, 44, 54, 70, 86; four 35, 38, 44, 66, 81,
 * 118; eight 34, 41, 58, 86, 112, 179.  The order is the same with 64 x 361.
 * Growth, compete pairs and CSR winners, which have no beam table in LDS,
 * cross near 2,000: calls of 1,500 take 139, 152 and 271 with two waves, 145,
 * 165 and 293 with a wave each, of 2,560 160, 182 and 313 against 148, 169
 * and 295. */
static int fast_team(int64_t n) { return n <= 512 ? 4 : n <= 2560 ? 2 : 1; }

template <int MAP>
static hipError_t launch_fast_median(const grs_eval_args *a, int32_t H, int64_t n_waves, int wpb, hipStream_t st) {
  const int team = fast_team(a->n_eval - a->e0);
  if (team > 1) return launch_fast_impl<true, MAP, false, true>(a, H, n_waves, team, st);
  return launch_fast_impl<true, MAP>(a, H, n_waves, wpb, st);
}

size_t grs_fit_nm_bytes(void) { return sizeof(grs_nm); }

hipError_t grs_launch_fit_nm(const grs_eval_args *a, int32_t H, int64_t M, const double *d_x0, double half_width,
                             int32_t max_fe, int32_t max_it, double tol_f, double tol_x, int32_t first, void *d_nm,
                             double *d_res, int32_t *d_left, hipStream_t st) {
  if (M <= 0) return hipSuccess;
  const int waves = GRS_FIT_TEAM * GRS_FIT_PTS;
  const size_t lds = (size_t)waves * (size_t)fast_wave_doubles((H + GRS_FIT_TEAM - 1) / GRS_FIT_TEAM) * sizeof(double);
  hipError_t e = hipFuncSetAttribute((const void *)k_fit_nm, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_fit_nm, dim3((unsigned)M), dim3(64 * waves), lds, st, *a, H, d_x0, half_width, max_fe, max_it,
                     tol_f, tol_x, first, static_cast<grs_nm *>(d_nm), d_res, d_left);
  return hipGetLastError();
}

hipError_t grs_launch_fast(const grs_eval_args *a, int32_t H, int64_t n_waves, int32_t wpb, hipStream_t st) {
  if (a->n_eval <= a->e0) return hipSuccess;
  switch (a->map) {
    case GRS_MAP_ONE_VOXEL: return launch_fast_median<GRS_MAP_ONE_VOXEL>(a, H, n_waves, wpb, st);
    case GRS_MAP_ONE_U: return launch_fast_median<GRS_MAP_ONE_U>(a, H, n_waves, wpb, st);
    case GRS_MAP_PAIRS: return launch_fast_median<GRS_MAP_PAIRS>(a, H, n_waves, wpb, st);
    case GRS_MAP_CSR_LIST: return launch_fast_median<GRS_MAP_CSR_LIST>(a, H, n_waves, wpb, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t grs_launch_fast_counts(const grs_eval_args *a, int32_t H, int64_t n_waves, int32_t wpb, hipStream_t st) {
  if (a->n_eval <= a->e0) return hipSuccess;
  if (a->map == GRS_MAP_CSR) return launch_fast_impl<false, GRS_MAP_CSR>(a, H, n_waves, wpb, st);
  if (a->map == GRS_MAP_GRID && a->n_u > 0) return launch_fast_impl<false, GRS_MAP_GRID>(a, H, n_waves, wpb, st);
  return hipErrorInvalidValue;
}

/* One-voxel evaluation that also runs the exact pipeline on every event of
 * phase B1 and counts disagreements (a->audit). */
hipError_t grs_launch_fast_audit(const grs_eval_args *a, int32_t H, int64_t n_waves, hipStream_t st) {
  if (a->n_eval <= a->e0) return hipSuccess;
  if (a->map != GRS_MAP_ONE_VOXEL || !a->audit) return hipErrorInvalidValue;
  return launch_fast_impl<true, GRS_MAP_ONE_VOXEL, true>(a, H, n_waves, GRS_WPB, st);
}

hipError_t grs_launch_pack_hits(const uint32_t *d_keys, int64_t n, uint32_t hit_key, int32_t has_hit,
                                uint32_t *d_bits, hipStream_t st) {
  int64_t nw = (n + 31) >> 5;
  if (nw <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pack_hits, dim3(blocks_for(nw, 256)), dim3(256), 0, st, d_keys, n, hit_key, has_hit, d_bits);
  return hipGetLastError();
}

hipError_t grs_launch_pack_hits_tiled(const uint32_t *d_keys, int64_t nz, int64_t ny, int64_t nrot, uint32_t hit_key,
                                      int32_t has_hit, uint32_t *d_tbits, hipStream_t st) {
  const int64_t ntz = (nz + 31) >> 5, nty = (ny + 31) >> 5;
  const int64_t nw = ntz * nty * nrot * 32;
  if (nw <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pack_hits_tiled, dim3(blocks_for(nw, 256)), dim3(256), 0, st, d_keys, nz, ny, nw,
                     (uint32_t)ntz, (uint32_t)nty, hit_key, has_hit, d_tbits);
  return hipGetLastError();
}

hipError_t grs_launch_plain(const grs_eval_args *a, int64_t T, hipStream_t st) {
  if (a->n_eval <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_plain, dim3(blocks_for(T, 256)), dim3(256), 0, st, *a, T);
  return hipGetLastError();
}

int64_t grs_grow_blocks(int64_t M) { return (M + GROW_T - 1) / GROW_T; }

hipError_t grs_launch_grow_list(const double *d_rows, int64_t M, const double *d_p1, int32_t *d_count, double *d_pos,
                                int32_t *d_slot, int64_t *d_total, hipStream_t st) {
  if (M <= 0) return hipSuccess;
  const dim3 grid((unsigned)grs_grow_blocks(M));
  if (d_count) hipLaunchKernelGGL(k_grow_count, grid, dim3(GROW_T), 0, st, d_rows, M, d_count);
  hipLaunchKernelGGL(k_grow_list, grid, dim3(GROW_T), 0, st, d_rows, M, d_p1, d_count, d_pos, d_slot, d_total);
  return hipGetLastError();
}

hipError_t grs_launch_grow_out(const double *d_rows, int64_t M, const double *d_p1, const int32_t *d_slot,
                               const int32_t *d_ns, const int32_t *d_ni, const double *d_C, const float *d_med,
                               double *d_out, hipStream_t st) {
  if (M <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_grow_out, dim3((unsigned)grs_grow_blocks(M)), dim3(GROW_T), 0, st, d_rows, M, d_p1, d_slot,
                     d_ns, d_ni, d_C, d_med, d_out);
  return hipGetLastError();
}

hipError_t grs_launch_compete_list(const double *d_vox, int64_t M, const int64_t *d_rs, const double *d_ids,
                                   int64_t n_id, int64_t G, const double *d_p1, double *d_pos, int32_t *d_evox,
                                   int32_t *d_eu, unsigned long long *d_bad, hipStream_t st) {
  if (M <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, st, d_bad, (int64_t)1, ~0ull);
  if (n_id > 0)
    hipLaunchKernelGGL(k_compete_ids, dim3(blocks_for(n_id, 256)), dim3(256), 0, st, d_ids, n_id, G, d_bad);
  hipLaunchKernelGGL(k_compete_list, dim3(blocks_for(M, 4)), dim3(256), 0, st, d_vox, M, d_rs, d_ids, G, d_p1, d_pos,
                     d_evox, d_eu);
  return hipGetLastError();
}

hipError_t grs_launch_compete_out(const int64_t *d_rs, int64_t M, int64_t row0, const int32_t *d_eu,
                                  const double *d_euler, const int32_t *d_ni, const double *d_C, const float *d_med,
                                  double *d_out, hipStream_t st) {
  if (M <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_compete_out, dim3(blocks_for(M, 64)), dim3(64), 0, st, d_rs, M, row0, d_eu, d_euler, d_ni, d_C,
                     d_med, d_out);
  return hipGetLastError();
}

hipError_t grs_launch_math_eval(int fn, const double *d_x, double *d_y, int64_t n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_math_eval, dim3(blocks_for(n, 256)), dim3(256), 0, st, fn, d_x, d_y, n);
  return hipGetLastError();
}

hipError_t grs_launch_copy_u32(const uint32_t *d_src, uint32_t *d_dst, int64_t n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  int64_t b = blocks_for(n, 256);
  if (b > 65536) b = 65536;
  hipLaunchKernelGGL(k_copy_u32, dim3((unsigned)b), dim3(256), 0, st, d_src, d_dst, n);
  return hipGetLastError();
}

hipError_t grs_launch_check_keys(const uint32_t *d_keys, int64_t n, uint32_t *d_bad, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  int64_t b = blocks_for(n, 256);
  if (b > 4096) b = 4096;
  hipLaunchKernelGGL(k_check_keys, dim3((unsigned)b), dim3(256), 0, st, d_keys, n, d_bad);
  return hipGetLastError();
}

int64_t grs_fast_wave_slots(int device) {
  (void)device;
  /* the scratch is indexed by wave: no launch has more than this, twice the
   * waves that a CU can hold (16 at 128 VGPRs) */
  return (int64_t)device_cus() * 64;
}

hipError_t grs_launch_fill_u32(uint32_t *d_p, int64_t n, uint32_t v, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u32, dim3(blocks_for(n, 256)), dim3(256), 0, st, d_p, n, v);
  return hipGetLastError();
}

hipError_t grs_launch_fill_u64(unsigned long long *d_p, int64_t n, unsigned long long v, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u64, dim3(blocks_for(n, 256)), dim3(256), 0, st, d_p, n, v);
  return hipGetLastError();
}

hipError_t grs_launch_winner_list(const unsigned long long *d_row_best, const int64_t *d_row_eoff, int64_t m,
                                  int64_t *d_elist, hipStream_t st) {
  if (m <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_winner_list, dim3(blocks_for(m, 256)), dim3(256), 0, st, d_row_best, d_row_eoff, m, d_elist);
  return hipGetLastError();
}

hipError_t grs_launch_winner_out(const int64_t *d_elist, const int64_t *d_row_eoff, const int64_t *d_row_ptr,
                                 const double *d_cand_q, int32_t nr, double gridsize, int64_t m, int64_t *d_best,
                                 double *d_best_q, hipStream_t st) {
  if (m <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_winner_out, dim3(blocks_for(m, 256)), dim3(256), 0, st, d_elist, d_row_eoff, d_row_ptr, d_cand_q,
                     nr, gridsize, m, d_best, d_best_q);
  return hipGetLastError();
}
