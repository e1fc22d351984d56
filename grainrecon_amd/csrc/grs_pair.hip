/*
 * grs_pair.hip -- spot pairing of forward_comp_pair_spots.m on the GPU.
 *
 * forward_comp_pair_spots.m:3-93 repeats forward_comp.m for one (U, pos) and,
 * for every selected event that hits the distance stack (dis <= minEucDis /
 * mean pixel size, :70), looks for the nearest experimental spot of the same
 * projection (Spots{i}(:,9:10), Euclidean distance in pixels to the rounded
 * event pixel, first minimum, :73-74); the pair is kept when that distance is
 * below min(sqrt(Spots{i}(id,11)), 15) (:75).  The kept rows are
 *   [reshape(U,1,9) pos hkl' Energy_hkl rot_angle Spots{i}(id,9:10)
 *    Spots{i}(id,11) dety detz dis]                       (:78-79)
 * in (projection, reflection) order, where pos already has RotAxisOffset
 * subtracted from its second component (:16) and the whole row is single
 * precision because dis is (MATLAB concatenation of double and single).
 *
 * k_pair_events   one thread per (orientation, projection, reflection): the
 *                 event, the hit test on the ordered keys, the list of hits.
 * k_pair_spots    one wave per hit: the nearest-spot search over the
 *                 projection's spots (CSR by projection, resident on the
 *                 device).
 * k_pair_scan     one block per orientation: exclusive scan of the pair flags
 *                 (the row order) and the pair count.
 * k_pair_rows     the 23 values of every pair, rounded to single precision.
 */
#include <hip/hip_runtime.h>

#include "grs_internal.h"
#include "grs_resolve.h"

/* One thread per event: those that are selected and hit go to the list hits
 * (in any order; everything is stored at the event's own place).  b1_classify
 * decides nearly every event; the exact pipeline runs for what it leaves
 * open and, for the wavelength, for the hits (2.6% of the events). */
__global__ __launch_bounds__(256) void k_pair_events(const grs_dgeo *g, const double *hkl, const double *cs,
                                                     const uint32_t *keys, const double *pos, const double *SUB,
                                                     int64_t M, int32_t *flag, double *lam, int32_t *dyz, float *dis,
                                                     int64_t *hits, uint32_t *n_hits) {
  GRS_NO_CONTRACT
  __shared__ double thr[12];
  if (threadIdx.x == 0) b1_thresholds(g, thr);
  __syncthreads();
  const int32_t H = g->H, nrot = g->nrot;
  const int64_t E = (int64_t)nrot * H;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= M * E) return;
  const int64_t m = t / E, rem = t - m * E;
  const int32_t om = (int32_t)(rem / H), h = (int32_t)(rem - (int64_t)om * H);
  flag[t] = 0;
  const double c = cs[2 * om], s = cs[2 * om + 1];
  double gw[3], P[3];
  grs_Gw(SUB + 9 * m, hkl + 3 * h, gw);
  voxel_P(g, pos + 3 * m, P);
  const double g2 = (gw[0] * gw[0] + gw[1] * gw[1]) + gw[2] * gw[2];
  const double t5[5] = {gw[0], gw[1], gw[2], fast_rsq(g2), g2};
  b1_out bo;
  const int st = b1_classify<true>(g, c, s, P, nullptr, t5, thr, &bo);
  if (st == 0) return;
  grs_vw v;
  double Gt[3], Glen, beta;
  int32_t dy = bo.dy, dz = bo.dz;
  auto exact = [&]() {
    grs_vw_terms(g, pos + 3 * m, c, s, &v);
    grs_Gt(v.c, v.s, gw[0], gw[1], gw[2], Gt);
    beta = grs_event_beta(&v, Gt, &Glen);
  };
  if (st == 2) {
    exact();
    if (!grs_event_finish(g, &v, Gt, Glen, beta, &dy, &dz)) return;
  }
  const uint32_t key = keys[(int64_t)(dz - 1) + (int64_t)(dy - 1) * g->nz + (int64_t)om * g->nz * g->ny];
  if (!(g->has_hit && key <= g->hit_key)) return;
  if (st == 1) exact();
  /* lambdahkl with the operations of forward_comp.m:33-37 */
  const double theta = beta - g->pio2;
  const double d = ((1.0 / Glen) * 2.0) * GRS_PI;
  lam[t] = (2.0 * d) * grs_sin(theta);
  dyz[2 * t] = dy;
  dyz[2 * t + 1] = dz;
  dis[t] = __uint_as_float(key);
  hits[atomicAdd(n_hits, 1u)] = t;
}

/* One wave per hit: the nearest spot of its projection (the first one on a
 * tie), and the flag of the pair when it is within min(sqrt(area), 15).  A
 * thread per event walking its projection's 690 spots with a root for each
 * held every wave for one or two lanes: 230 us for three orientations with the
 * events, 22 us now.  A larger sum of squares cannot have a smaller root, so
 * only a smaller one is rooted. */
__global__ __launch_bounds__(256) void k_pair_spots(const grs_dgeo *g, const int64_t *fptr, const double *fsp,
                                                    const int32_t *dyz, const int64_t *hits, const uint32_t *n_hits,
                                                    int32_t *flag, int64_t *sid) {
  GRS_NO_CONTRACT
  const int lane = threadIdx.x & 63;
  const int64_t E = (int64_t)g->nrot * g->H, n = *n_hits;
  for (int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); w < n; w += (int64_t)gridDim.x * 4) {
    const int64_t t = hits[w];
    const int32_t om = (int32_t)((t % E) / g->H);
    const double dy = (double)dyz[2 * t], dz = (double)dyz[2 * t + 1];
    double best = __builtin_inf(), s2 = __builtin_inf();
    int64_t bi = INT64_MAX;
    for (int64_t k = fptr[om] + lane; k < fptr[om + 1]; k += 64) {
      const double ey = fsp[3 * k] - dy, ez = fsp[3 * k + 1] - dz;
      const double q = ey * ey + ez * ez;
      if (q < s2 || (bi == INT64_MAX && q == q)) {
        const double d = grs_sqrt(q);
        if (bi == INT64_MAX || d < best) {
          best = d;
          s2 = q;
          bi = k;
        }
      }
    }
    for (int off = 32; off >= 1; off >>= 1) {
      const double ob = __shfl_xor(best, off, 64);
      const int64_t oi = (int64_t)__shfl_xor((long long)bi, off, 64);
      if (oi != INT64_MAX && (bi == INT64_MAX || ob < best || (ob == best && oi < bi))) {
        best = ob;
        bi = oi;
      }
    }
    if (lane == 0 && bi != INT64_MAX) {
      const double sa = grs_sqrt(fsp[3 * bi + 2]);
      const double lim = (sa == sa && sa < 15.0) ? sa : 15.0;
      if (best < lim) {
        flag[t] = 1;
        sid[t] = bi;
      }
    }
  }
}

__global__ __launch_bounds__(1024) void k_pair_scan(const int32_t *flag, int64_t E, int32_t *off, int64_t *count) {
  __shared__ int32_t part[1024];
  const int tid = threadIdx.x, bd = blockDim.x;
  const int64_t m = blockIdx.x;
  const int32_t *f = flag + m * E;
  const int64_t per = (E + bd - 1) / bd;
  const int64_t lo = (int64_t)tid * per, hi = lo + per < E ? lo + per : E;
  int32_t c = 0;
  for (int64_t i = lo; i < hi; i++) c += f[i];
  part[tid] = c;
  __syncthreads();
  for (int o = 1; o < bd; o <<= 1) {
    const int32_t v = tid >= o ? part[tid - o] : 0;
    __syncthreads();
    part[tid] += v;
    __syncthreads();
  }
  int32_t run = part[tid] - c;
  for (int64_t i = lo; i < hi; i++) {
    off[m * E + i] = run;
    run += f[i];
  }
  if (tid == bd - 1) count[m] = part[tid];
}

__global__ __launch_bounds__(256) void k_pair_rows(const grs_dgeo *g, const double *hkl, const double *rot,
                                                   const double *pos, const double *U, int64_t M, const double *fsp,
                                                   const int32_t *flag, const int64_t *sid, const double *lam,
                                                   const int32_t *dyz, const float *dis, const int32_t *off,
                                                   const int64_t *row_ptr, double *rows) {
  GRS_NO_CONTRACT
  const int32_t H = g->H, nrot = g->nrot;
  const int64_t E = (int64_t)nrot * H;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= M * E || !flag[t]) return;
  const int64_t m = t / E, rem = t - m * E;
  const int32_t om = (int32_t)(rem / H), h = (int32_t)(rem - (int64_t)om * H);
  double *r = rows + (row_ptr[m] + off[t]) * 23;
  const double *u = U + 9 * m;
  /* reshape(U,1,9): column-major */
  for (int c = 0; c < 3; c++)
    for (int k = 0; k < 3; k++) r[3 * c + k] = (double)(float)u[3 * k + c];
  r[9] = (double)(float)pos[3 * m];
  r[10] = (double)(float)(pos[3 * m + 1] - g->RAO);
  r[11] = (double)(float)pos[3 * m + 2];
  for (int k = 0; k < 3; k++) r[12 + k] = (double)(float)hkl[3 * h + k];
  r[15] = (double)(float)(12.398 / lam[t]);
  r[16] = (double)(float)rot[om];
  const int64_t s = sid[t];
  r[17] = (double)(float)fsp[3 * s];
  r[18] = (double)(float)fsp[3 * s + 1];
  r[19] = (double)(float)fsp[3 * s + 2];
  r[20] = (double)(float)dyz[2 * t];
  r[21] = (double)(float)dyz[2 * t + 1];
  r[22] = (double)dis[t];
}

static unsigned pair_grid(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

hipError_t grs_launch_pair_events(const grs_dgeo *d_g, const double *d_hkl, const double *d_cs,
                                  const uint32_t *d_keys, const double *d_pos, const double *d_SUB, int64_t M,
                                  int64_t E, const int64_t *d_fptr, const double *d_fsp, int32_t *d_flag,
                                  int64_t *d_sid, double *d_lam, int32_t *d_dyz, float *d_dis, int64_t *d_hits,
                                  uint32_t *d_nhits, hipStream_t st) {
  if (M <= 0 || E <= 0) return hipSuccess;
  hipError_t e = grs_launch_fill_u32(d_nhits, 1, 0u, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_pair_events, dim3(pair_grid(M * E, 256)), dim3(256), 0, st, d_g, d_hkl, d_cs, d_keys, d_pos,
                     d_SUB, M, d_flag, d_lam, d_dyz, d_dis, d_hits, d_nhits);
  /* waves for a few hundred hits an orientation; more are taken in turn */
  const int64_t blocks = 128 * M < 2048 ? 128 * M : 2048;
  hipLaunchKernelGGL(k_pair_spots, dim3((unsigned)blocks), dim3(256), 0, st, d_g, d_fptr, d_fsp, d_dyz, d_hits,
                     d_nhits, d_flag, d_sid);
  return hipGetLastError();
}

hipError_t grs_launch_pair_scan(const int32_t *d_flag, int64_t M, int64_t E, int32_t *d_off, int64_t *d_count,
                                hipStream_t st) {
  if (M <= 0 || E <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pair_scan, dim3((unsigned)M), dim3(1024), 0, st, d_flag, E, d_off, d_count);
  return hipGetLastError();
}

hipError_t grs_launch_pair_rows(const grs_dgeo *d_g, const double *d_hkl, const double *d_rot, const double *d_pos,
                                const double *d_U, int64_t M, int64_t E, const double *d_fsp, const int32_t *d_flag,
                                const int64_t *d_sid, const double *d_lam, const int32_t *d_dyz, const float *d_dis,
                                const int32_t *d_off, const int64_t *d_row_ptr, double *d_rows, hipStream_t st) {
  if (M <= 0 || E <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pair_rows, dim3(pair_grid(M * E, 256)), dim3(256), 0, st, d_g, d_hkl, d_rot, d_pos, d_U, M,
                     d_fsp, d_flag, d_sid, d_lam, d_dyz, d_dis, d_off, d_row_ptr, d_rows);
  return hipGetLastError();
}
