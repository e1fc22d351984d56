/*
 * grs_prep.hip -- device-side input preparation for the scoring engine.
 *
 * k_render_spots   forward simulation of binary spot masks with the
 *                  forward_comp.m geometry: every selected (omega, hkl) event
 *                  of every (voxel, grain orientation) sets its pixel.  Used to
 *                  build synthetic data sets whose spots are the projections of
 *                  the grains.
 * k_edt_cols/rows  exact Euclidean distance transform of each binary
 *                  projection, the bwdist of GrainMapping_fun.m:73-75: the
 *                  distance from every pixel to the nearest spot pixel, stored
 *                  as single(sqrt(d^2)).  Separable algorithm of P. Felzenszwalb
 *                  and D. Huttenlocher, "Distance Transforms of Sampled
 *                  Functions", Theory of Computing 8 (2012): a 1-D distance
 *                  along detz, then the lower envelope of parabolas along dety.
 *                  Envelope intersections are rationals with denominators
 *                  below 2*ny, evaluated in double, so every decision and every
 *                  d^2 is exact.  A projection without any spot pixel gives
 *                  +Inf everywhere, as bwdist does.  Used beyond the sizes of
 * k_edt_lines/tile the same transform for sides up to 4096 x about 9600
 *                  (every detector in use): the distance along detz from bit
 *                  masks of the lines, then the minimum along dety in LDS by
 *                  divide and conquer over the rows, all in whole numbers.
 * Layout of masks and stacks: MATLAB column-major (detz fastest, then dety,
 * then omega).
 */
#include <hip/hip_runtime.h>

#include "grs_internal.h"

#define GRS_EDT_INF 0x3FFFFFFF

__global__ void k_render_spots(const grs_dgeo *g, const double *pos, const int32_t *grain, int64_t M,
                               const double *SUB, const double *hkl, const double *cs, uint8_t *mask) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int32_t nrot = g->nrot, H = g->H;
  if (i >= M * nrot) return;
  int64_t v = i / nrot;
  int32_t om = (int32_t)(i - v * nrot);
  const double *sub = SUB + 9 * (int64_t)grain[v];
  grs_vw t;
  grs_vw_terms(g, pos + 3 * v, cs[2 * om], cs[2 * om + 1], &t);
  const int64_t nz = g->nz, nzny = g->nz * g->ny;
  for (int32_t h = 0; h < H; h++) {
    double gw[3], Gt[3], Glen;
    grs_Gw(sub, hkl + 3 * h, gw);
    grs_Gt(t.c, t.s, gw[0], gw[1], gw[2], Gt);
    double beta = grs_event_beta(&t, Gt, &Glen);
    int32_t dy, dz;
    if (grs_event_finish(g, &t, Gt, Glen, beta, &dy, &dz))
      mask[(int64_t)(dz - 1) + (int64_t)(dy - 1) * nz + (int64_t)om * nzny] = 1;
  }
}

/* Every selected event of voxel v (orientation SUB[grain[v]]): the omega and
 * hkl indices and the unrounded pixel coordinates -dety22/py + dety0,
 * -detz22/pz + detz0.  Slots come from an atomic counter; the host sorts. */
__global__ void k_sim_events(const grs_dgeo *g, const double *pos, const int32_t *grain, int64_t M,
                             const double *SUB, const double *hkl, const double *cs, int64_t cap,
                             unsigned long long *counter, int32_t *ev_vox, int32_t *ev_om, int32_t *ev_h,
                             double *ev_yz) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int32_t nrot = g->nrot, H = g->H;
  if (i >= M * nrot) return;
  int64_t v = i / nrot;
  int32_t om = (int32_t)(i - v * nrot);
  const double *sub = SUB + 9 * (int64_t)grain[v];
  grs_vw t;
  grs_vw_terms(g, pos + 3 * v, cs[2 * om], cs[2 * om + 1], &t);
  for (int32_t h = 0; h < H; h++) {
    double gw[3], Gt[3], Glen;
    grs_Gw(sub, hkl + 3 * h, gw);
    grs_Gt(t.c, t.s, gw[0], gw[1], gw[2], Gt);
    double beta = grs_event_beta(&t, Gt, &Glen);
    int32_t dy, dz;
    double yz[2];
    if (grs_event_finish_yz(g, &t, Gt, Glen, beta, &dy, &dz, yz)) {
      unsigned long long slot = atomicAdd(counter, 1ull);
      if (slot < (unsigned long long)cap) {
        ev_vox[slot] = (int32_t)v;
        ev_om[slot] = om;
        ev_h[slot] = h;
        ev_yz[2 * slot] = yz[0];
        ev_yz[2 * slot + 1] = yz[1];
      }
    }
  }
}

/* ---- distance transform, one pass over the mask and one over the stack -------
 *
 * k_edt_lines: one wave per (dety, omega) line of nz pixels.  Every 64 pixels
 * become a 64-bit mask by ballot; per mask also the last set pixel before it
 * and the first after it (0xFFFF: none), by a scan across the lanes (lane k
 * holds mask k, so nz <= 4096).  12 bytes per 64 pixels, and a word per
 * projection that says whether it has a spot pixel.
 *
 * k_edt_tile: one block per TZ consecutive detz positions of a projection.
 * g(y) = distance along detz to the nearest spot pixel of line y comes from
 * the masks into LDS (16 bits; GRS_EDT_NONE when the line has none), and
 * d^2(y) = min over p of g(p)^2 + (y - p)^2 is found in whole numbers.  For
 * p < p' the difference of the two terms grows with y, so a minimiser of row
 * y bounds the minimisers of the rows after it from below and of the rows
 * before it from above.  Every 64th row (and the last) is searched outwards
 * from itself until (y - p)^2 reaches the minimum; the rows between, at
 * steps 32, 16 and so on to 1, only between the minimisers of their two
 * neighbours: about 2 candidates a row and level whatever the distances are,
 * where a search outwards from every row costs its distance (1,000 and more
 * in a projection with few spots).  The steps below 16 stay in a thread's
 * registers: it writes 16 rows of one detz position, TZ lanes side by side.
 *
 * Bound: the 1 byte read and 4 bytes written per pixel, and about as long in
 * LDS reads and arithmetic.  The two kernels it replaces at these sizes
 * (k_edt_cols, one thread walking a line byte by byte with lines nz apart, and
 * k_edt_rows, one thread per detz row with its envelope in HBM) took
 * 8.8 + 12.8 ms for 1024 x 1024 x 181; these take 0.2 + 1.5 ms. */
#define GRS_EDT_NONE 32767u /* its square exceeds every d^2, and the sums stay below 2^31 */

__global__ __launch_bounds__(256) void k_edt_lines(const uint8_t *mask, int32_t nz, int64_t nlines, int32_t nch,
                                                   int32_t ny, uint64_t *words, uint32_t *near, uint32_t *any) {
  const int lane = threadIdx.x & 63;
  const int64_t line = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (line >= nlines) return;
  const uint8_t *m = mask + line * nz;
  uint64_t mine = 0;
  for (int32_t c0 = 0; c0 < nch; c0 += 8) {
    uint8_t b[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int32_t z = (c0 + k) * 64 + lane;
      b[k] = z < nz ? m[z] : (uint8_t)0;
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const uint64_t w = __ballot(b[k] != 0);
      if (lane == c0 + k) mine = w;
    }
  }
  if (__ballot(mine != 0) && lane == 0) any[line / ny] = 1u;
  /* inclusive scans, then shifted by one lane */
  int32_t last = mine ? lane * 64 + 63 - __clzll((long long)mine) : -1;
  int32_t next = mine ? lane * 64 + __ffsll((unsigned long long)mine) - 1 : 0xFFFF;
  for (int off = 1; off < 64; off <<= 1) {
    const int32_t a = __shfl_up(last, off, 64), b = __shfl_down(next, off, 64);
    if (lane >= off) last = a > last ? a : last;
    if (lane + off < 64) next = b < next ? b : next;
  }
  last = __shfl_up(last, 1, 64);
  next = __shfl_down(next, 1, 64);
  if (lane == 0) last = -1;
  if (lane == 63) next = 0xFFFF;
  if (lane < nch) {
    words[line * nch + lane] = mine;
    near[line * nch + lane] = ((uint32_t)last & 0xFFFFu) | ((uint32_t)next << 16);
  }
}

/* the smallest g(p)^2 + (y - p)^2 over p = lo..hi of one detz position (col:
 * its g values, TZ apart), and a p that gives it */
template <int TZ>
__device__ __forceinline__ uint32_t edt_min(const uint16_t *col, int32_t y, int32_t lo, int32_t hi, int32_t *at) {
  uint32_t best = 0xFFFFFFFFu;
  int32_t bp = lo;
  for (int32_t p = lo; p <= hi; p += 4) {
    uint32_t g[4];
#pragma unroll
    for (int k = 0; k < 4; k++) g[k] = col[(p + k < hi ? p + k : hi) * TZ];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int32_t q = p + k < hi ? p + k : hi;
      const int32_t d = y - q;
      const uint32_t f = __umul24(g[k], g[k]) + (uint32_t)__mul24(d, d);
      if (f < best) {
        best = f;
        bp = q;
      }
    }
  }
  *at = bp;
  return best;
}

__device__ __forceinline__ float edt_root(uint32_t f) {
  if (f >= GRS_EDT_NONE * GRS_EDT_NONE) return __int_as_float(0x7F800000);
  /* below 2^24 f is a float, and the correctly rounded root of it is the
   * double root rounded to single */
  return f < (1u << 24) ? __builtin_sqrtf((float)f) : (float)__builtin_sqrt((double)f);
}

template <int TZ>
__global__ __launch_bounds__(1024) void k_edt_tile(const uint64_t *words, const uint32_t *near, const uint32_t *any,
                                                   int32_t nz, int32_t ny, int32_t nch, int32_t ntz, float *out) {
  extern __shared__ uint16_t lds[];
  uint16_t *g = lds;           /* [ny][TZ] */
  uint16_t *pr = lds + ny * TZ; /* minimisers of the rows 0, 16, 32, ... and ny - 1: [nr + 1][TZ] */
  const int64_t sl = blockIdx.x / ntz;
  const int32_t z0 = (int32_t)(blockIdx.x - sl * ntz) * TZ;
  const int32_t iz = (int32_t)threadIdx.x % TZ, item = (int32_t)threadIdx.x / TZ, items = (int32_t)blockDim.x / TZ;
  const int32_t z = z0 + iz;
  const bool in = z < nz;
  float *o = out + sl * (int64_t)nz * ny + z;
  if (any[sl] == 0u) {
    /* every row's search would walk all rows (1024 x 1024 x 181 empty: 3.36 ms, 0.36 like this) */
    for (int32_t y = item; y < ny; y += items)
      if (in) o[(int64_t)y * nz] = __int_as_float(0x7F800000);
    return;
  }
  const int bit = z & 63;
  const uint64_t below = ~0ull >> (63 - bit), above = ~0ull << bit;
  const int64_t w0 = sl * ny * nch + (z0 >> 6);
#pragma unroll 4
  for (int32_t y = item; y < ny; y += items) {
    const uint64_t w = words[w0 + (int64_t)y * nch];
    const uint32_t nr = near[w0 + (int64_t)y * nch];
    const int32_t base = z0 & ~63;
    const uint64_t wb = w & below, wa = w & above;
    const int32_t l = wb ? base + 63 - __clzll((long long)wb) : (int32_t)(int16_t)(nr & 0xFFFFu);
    const int32_t n = wa ? base + __ffsll((unsigned long long)wa) - 1 : (int32_t)(nr >> 16);
    uint32_t d = GRS_EDT_NONE;
    if (l >= 0) d = (uint32_t)(z - l);
    if (n != 0xFFFF && (uint32_t)(n - z) < d) d = (uint32_t)(n - z);
    g[y * TZ + iz] = (uint16_t)d;
  }
  __syncthreads();
  const uint16_t *col = g + iz;
  const int32_t nr = (ny - 1 + 15) / 16;
  /* every 64th row and the last: outwards from the row */
  const int32_t na = (nr + 3) / 4;
  for (int32_t t = item; t <= na; t += items) {
    const int32_t r = 4 * t < nr ? 4 * t : nr;
    const int32_t y = 16 * r < ny - 1 ? 16 * r : ny - 1;
    uint32_t best = __umul24(col[y * TZ], col[y * TZ]);
    int32_t bp = y;
    for (int32_t k = 1; k < ny; k++) {
      const uint32_t kk = (uint32_t)__mul24(k, k);
      if (kk >= best) break;
      const int32_t a = y - k > 0 ? y - k : 0, b = y + k < ny - 1 ? y + k : ny - 1;
      const uint32_t ga = col[a * TZ], gb = col[b * TZ];
      /* a clamped row counts with a larger distance than its own: never wrongly best */
      const uint32_t fa = __umul24(ga, ga) + kk, fb = __umul24(gb, gb) + kk;
      if (fa < best) {
        best = fa;
        bp = a;
      }
      if (fb < best) {
        best = fb;
        bp = b;
      }
    }
    pr[r * TZ + iz] = (uint16_t)bp;
  }
  __syncthreads();
  for (int32_t half = 2; half >= 1; half >>= 1) {
    for (int32_t r = half + 2 * half * item; r < nr; r += 2 * half * items) {
      const int32_t e = r + half < nr ? r + half : nr;
      int32_t at;
      edt_min<TZ>(col, 16 * r, pr[(r - half) * TZ + iz], pr[e * TZ + iz], &at);
      pr[r * TZ + iz] = (uint16_t)at;
    }
    __syncthreads();
  }
  /* 16 rows at a time over the candidates between their two neighbours' minimisers: with d = y0 - p the
   * term of row y0 + k is (g(p)^2 + d^2) + k (2 d) + k^2, so a row takes one multiply-add and half a
   * three-way minimum per candidate */
  for (int32_t s = item; s < (nr > 0 ? nr : 1); s += items) {
    const int32_t y0 = 16 * s, lo = pr[s * TZ + iz], hi = nr > 0 ? pr[(s + 1) * TZ + iz] : lo;
    int32_t m[17];
#pragma unroll
    for (int k = 0; k < 17; k++) m[k] = INT32_MAX;
    for (int32_t p = lo; p <= hi; p += 2) {
      const int32_t q = p + 1 < hi ? p + 1 : hi;
      const uint32_t ga = col[p * TZ], gb = col[q * TZ];
      const int32_t da = y0 - p, db = y0 - q;
      const int32_t ca = (int32_t)__umul24(ga, ga) + __mul24(da, da), cb = (int32_t)__umul24(gb, gb) + __mul24(db, db);
#pragma unroll
      for (int k = 0; k < 17; k++) {
        const int32_t fa = ca + __mul24(k, 2 * da), fb = cb + __mul24(k, 2 * db);
        const int32_t f = fa < fb ? fa : fb;
        m[k] = f < m[k] ? f : m[k];
      }
    }
    const int32_t rows = s + 1 < nr ? 16 : ny - y0; /* the last 16 rows end with row ny - 1, up to 17 of them */
#pragma unroll
    for (int k = 0; k < 17; k++)
      if (in && k < rows) o[(int64_t)(y0 + k) * nz] = edt_root((uint32_t)(m[k] + k * k));
  }
}

/* 1-D distance along detz within each (dety, omega) column. */
__global__ void k_edt_cols(const uint8_t *mask, int64_t nz, int64_t ncols, int32_t *g1) {
  int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncols) return;
  const uint8_t *m = mask + c * nz;
  int32_t *o = g1 + c * nz;
  int32_t d = GRS_EDT_INF;
  for (int64_t z = 0; z < nz; z++) {
    if (m[z]) d = 0;
    else if (d < GRS_EDT_INF) d++;
    o[z] = d;
  }
  d = GRS_EDT_INF;
  for (int64_t z = nz - 1; z >= 0; z--) {
    if (m[z]) d = 0;
    else if (d < GRS_EDT_INF) d++;
    if (d < o[z]) o[z] = d;
  }
}

/* Lower envelope along dety for each (detz row, omega) of a chunk of slices;
 * v/zb are per-thread work arrays, element k at [k*T + tid]. */
__global__ void k_edt_rows(const int32_t *g1, int64_t nz, int64_t ny, int64_t slice0, int64_t nslices,
                           int32_t *v, double *zb, float *out) {
  int64_t T = nz * nslices;
  int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= T) return;
  int64_t iz = tid % nz;
  int64_t sl = slice0 + tid / nz;
  const int32_t *col = g1 + sl * nz * ny + iz; /* f(q) = col[q*nz]^2 */
  float *o = out + sl * nz * ny + iz;
  int64_t k = -1;
  for (int64_t q = 0; q < ny; q++) {
    int32_t gq = col[q * nz];
    if (gq >= GRS_EDT_INF) continue;
    double fq = (double)gq * (double)gq;
    double s = 0.0;
    while (k >= 0) {
      int32_t p = v[k * T + tid];
      int32_t gp = col[(int64_t)p * nz];
      double fp = (double)gp * (double)gp;
      s = ((fq + (double)q * (double)q) - (fp + (double)p * (double)p)) / (2.0 * (double)q - 2.0 * (double)p);
      if (s <= zb[k * T + tid]) k--;
      else break;
    }
    k++;
    v[k * T + tid] = (int32_t)q;
    zb[k * T + tid] = k == 0 ? -1.0e300 : s;
  }
  if (k < 0) {
    for (int64_t q = 0; q < ny; q++) o[q * nz] = __int_as_float(0x7F800000);
    return;
  }
  int64_t j = 0;
  for (int64_t q = 0; q < ny; q++) {
    while (j < k && zb[(j + 1) * T + tid] < (double)q) j++;
    int32_t p = v[j * T + tid];
    int32_t gp = col[(int64_t)p * nz];
    double d2 = ((double)q - (double)p) * ((double)q - (double)p) + (double)gp * (double)gp;
    o[q * nz] = (float)__builtin_sqrt(d2);
  }
}

static inline unsigned nblk(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

hipError_t grs_launch_render(const grs_dgeo *d_g, const double *d_pos, const int32_t *d_grain, int64_t M,
                             int32_t nrot, const double *d_SUB, const double *d_hkl, const double *d_cs,
                             uint8_t *d_mask, hipStream_t st) {
  int64_t n = M * nrot;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_render_spots, dim3(nblk(n, 128)), dim3(128), 0, st, d_g, d_pos, d_grain, M, d_SUB, d_hkl,
                     d_cs, d_mask);
  return hipGetLastError();
}

hipError_t grs_launch_sim_events(const grs_dgeo *d_g, const double *d_pos, const int32_t *d_grain, int64_t M,
                                 int32_t nrot, const double *d_SUB, const double *d_hkl, const double *d_cs, int64_t cap,
                                 unsigned long long *d_counter, int32_t *d_vox, int32_t *d_om, int32_t *d_h,
                                 double *d_yz, hipStream_t st) {
  int64_t n = M * nrot;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sim_events, dim3(nblk(n, 128)), dim3(128), 0, st, d_g, d_pos, d_grain, M, d_SUB, d_hkl, d_cs,
                     cap, d_counter, d_vox, d_om, d_h, d_yz);
  return hipGetLastError();
}

/* LDS of a k_edt_tile block */
static size_t edt_tile_bytes(int64_t ny, int tz) { return (size_t)(2 * tz) * (size_t)(ny + (ny - 1 + 15) / 16 + 1); }

/* the widest tile whose g values fit a CU's 160 KB of LDS (64 lines up to
 * ny = 1203, 32 up to 2408, ...).  Wider tiles write longer runs of detz, but
 * have a CU to themselves: tiles of which two fit take 1.27 instead of 1.47 ms
 * for 1024 x 1024 x 181 with 690 spots a projection, 1.76 and 1.97 with 50, the
 * same at 512 rows, 3.52 instead of 3.35 for 2048 x 2048 x 60 with 50; 0
 * beyond the sides and the launch sizes (below 2^32 threads) the two kernels
 * take */
int grs_edt_tile_width(int64_t nz, int64_t ny, int64_t nslices) {
  if (nz > 4096 || ny * nslices >= (int64_t)1 << 25) return 0;
  for (int tz = 64; tz >= 8; tz >>= 1)
    if (edt_tile_bytes(ny, tz) <= 163840) return nslices * ((nz + tz - 1) / tz) < (int64_t)1 << 22 ? tz : 0;
  return 0;
}

int64_t grs_edt_work_bytes(int64_t nz, int64_t ny, int64_t nslices) {
  return ny * nslices * ((nz + 63) / 64) * 12 + nslices * 4;
}

template <int TZ>
static hipError_t launch_edt_tile(const uint64_t *words, const uint32_t *near, const uint32_t *any, int64_t nz,
                                  int64_t ny, int64_t nslices, float *d_out, hipStream_t st) {
  const int32_t ntz = (int32_t)((nz + TZ - 1) / TZ);
  const size_t lds = edt_tile_bytes(ny, TZ);
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_edt_tile<TZ>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, 163840);
  if (e != hipSuccess) return e;
  /* a thread for every 16 rows of a detz position, up to 1024 */
  int64_t threads = (int64_t)TZ * ((ny + 15) / 16);
  threads = threads < 64 ? 64 : threads > 1024 ? 1024 : (threads + 63) / 64 * 64;
  hipLaunchKernelGGL(k_edt_tile<TZ>, dim3((unsigned)(nslices * ntz)), dim3((unsigned)threads), lds, st, words, near, any,
                     (int32_t)nz, (int32_t)ny, (int32_t)((nz + 63) / 64), ntz, d_out);
  return hipGetLastError();
}

hipError_t grs_launch_edt(const uint8_t *d_mask, int64_t nz, int64_t ny, int64_t nslices, void *d_work, float *d_out,
                          hipStream_t st) {
  const int64_t nlines = ny * nslices, nch = (nz + 63) / 64;
  uint64_t *words = static_cast<uint64_t *>(d_work);
  uint32_t *near = reinterpret_cast<uint32_t *>(words + nlines * nch);
  uint32_t *any = near + nlines * nch;
  hipError_t e = grs_launch_fill_u32(any, nslices, 0u, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_edt_lines, dim3(nblk(nlines, 4)), dim3(256), 0, st, d_mask, (int32_t)nz, nlines, (int32_t)nch,
                     (int32_t)ny, words, near, any);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  switch (grs_edt_tile_width(nz, ny, nslices)) {
    case 64: return launch_edt_tile<64>(words, near, any, nz, ny, nslices, d_out, st);
    case 32: return launch_edt_tile<32>(words, near, any, nz, ny, nslices, d_out, st);
    case 16: return launch_edt_tile<16>(words, near, any, nz, ny, nslices, d_out, st);
    case 8: return launch_edt_tile<8>(words, near, any, nz, ny, nslices, d_out, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t grs_launch_edt_cols(const uint8_t *d_mask, int64_t nz, int64_t ncols, int32_t *d_g1, hipStream_t st) {
  if (ncols <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_edt_cols, dim3(nblk(ncols, 256)), dim3(256), 0, st, d_mask, nz, ncols, d_g1);
  return hipGetLastError();
}

hipError_t grs_launch_edt_rows(const int32_t *d_g1, int64_t nz, int64_t ny, int64_t slice0, int64_t nslices,
                               int32_t *d_v, double *d_z, float *d_out, hipStream_t st) {
  int64_t T = nz * nslices;
  if (T <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_edt_rows, dim3(nblk(T, 256)), dim3(256), 0, st, d_g1, nz, ny, slice0, nslices, d_v, d_z,
                     d_out);
  return hipGetLastError();
}
