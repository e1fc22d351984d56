/*
 * grs_region.hip -- region growth around an indexed seed with the volumes
 * resident on the device (grow_indexed_region_cuda.m:29-151).
 *
 * k_region_list    :44-77: the voxels of the bounding box within Box_L of
 *                  its centre point, with their completeness (the seed's
 *                  replaced by the indexed completeness), mask and median
 *                  distance gathered from the volumes; only voxels inside the
 *                  mask are listed (the operator scores no others,
 *                  grow_indexed_region_parallel.m:61-90).
 * k_region_accept  the growth rule of cuda_grow_indexed_region
 *                  (grow_indexed_region_parallel.m:78-81) on the scores of
 *                  the listed voxels, and the write-back of :117-128
 *                  (completeness = Nr_intersect/Nr_simu, median distance,
 *                  Nr_intersect) into the volumes; the accepted voxels and
 *                  their completeness are appended to a list for the
 *                  weighted centre, which the host sums in MATLAB's find()
 *                  order.
 * k_grow_count, k_grow_list, k_grow_out  the voxel rows of
 *                  cuda_grow_indexed_region: the rows inside the mask listed in
 *                  order with their positions, and the operator's output rows.
 * Volumes are nx x ny x nz doubles with x fastest (MATLAB's I(x,y,z)).
 */
#include <hip/hip_runtime.h>

#include "grs_internal.h"

__global__ void k_region_list(const double *I, const double *mask, const double *dm, int64_t nx, int64_t ny,
                              int64_t lo0, int64_t lo1, int64_t lo2, int64_t bx, int64_t by, int64_t bz, double cp0,
                              double cp1, double cp2, double boxL, int64_t seed_lin, double seed_comp, double *rows,
                              uint32_t *counts) {
  GRS_NO_CONTRACT
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= bx * by * bz) return;
  const int64_t ix = t % bx, iy = (t / bx) % by, iz = t / (bx * by);
  const double x = (double)(lo0 + ix), y = (double)(lo1 + iy), z = (double)(lo2 + iz);
  const double dx = x - cp0, dy = y - cp1, dz = z - cp2;
  const double d = grs_sqrt((dx * dx + dy * dy) + dz * dz);
  if (!(d <= boxL)) return;
  atomicAdd(counts + 1, 1u);
  const int64_t lin = (lo0 + ix - 1) + nx * ((lo1 + iy - 1) + ny * (lo2 + iz - 1));
  if (!(mask[lin] > 0.0)) return;
  const uint32_t k = atomicAdd(counts, 1u);
  double *r = rows + 6 * (int64_t)k;
  r[0] = x;
  r[1] = y;
  r[2] = z;
  r[3] = lin == seed_lin ? seed_comp : I[lin];
  r[4] = mask[lin];
  r[5] = dm[lin];
}

__global__ void k_region_accept(const double *rows, int64_t M, const int32_t *ns, const int32_t *ni, const double *C,
                                const float *med, const double *p1, int64_t nx, int64_t ny, double *vC, double *vDM,
                                double *vNI, int64_t *acc_lin, double *acc_C, uint32_t *count) {
  GRS_NO_CONTRACT
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  const double *v = rows + 6 * i;
  const double Cn = C[i], dmv = (double)med[i];
  /* min([DisMedian maxDmedian]) with MATLAB's NaN rule */
  const double a = v[5], b = p1[13];
  const double lim = a != a ? b : (b != b ? a : (a < b ? a : b));
  if (!((Cn > v[3] && dmv <= lim) && (Cn >= p1[11] * (1.0 - p1[12])))) return;
  const int64_t lin = ((int64_t)v[0] - 1) + nx * (((int64_t)v[1] - 1) + ny * ((int64_t)v[2] - 1));
  const double Cw = (double)ni[i] / (double)ns[i];
  vC[lin] = Cw;
  vDM[lin] = dmv;
  vNI[lin] = (double)ni[i];
  const uint32_t k = atomicAdd(count, 1u);
  acc_lin[k] = lin;
  acc_C[k] = Cw;
}

/* ---- voxel rows of cuda_grow_indexed_region ---------------------------------
 *
 * The rows [x y z C mask DisMedian] stay on the device as they came: block b
 * of GROW_T rows counts its rows inside the mask, k_grow_list gives row i its
 * place among the scored ones (slot, -1 outside the mask) and writes the
 * position there, k_grow_out forms the 7 output values and the growth flag.
 * Bound: 48 bytes in and 56 out per row; on the host the same loops and their
 * copies took about 40 ms for 3.2M rows, the three kernels take 0.28 ms. */
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

hipError_t grs_launch_region_list(const double *d_I, const double *d_mask, const double *d_dm, int64_t nx, int64_t ny,
                                  const int64_t *lo, const int64_t *bdim, const double *cp, double boxL,
                                  int64_t seed_lin, double seed_comp, double *d_rows, uint32_t *d_counts,
                                  hipStream_t st) {
  const int64_t n = bdim[0] * bdim[1] * bdim[2];
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_region_list, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, d_I, d_mask, d_dm, nx, ny,
                     lo[0], lo[1], lo[2], bdim[0], bdim[1], bdim[2], cp[0], cp[1], cp[2], boxL, seed_lin, seed_comp,
                     d_rows, d_counts);
  return hipGetLastError();
}

hipError_t grs_launch_region_accept(const double *d_rows, int64_t M, const int32_t *d_ns, const int32_t *d_ni,
                                    const double *d_C, const float *d_med, const double *d_p1, int64_t nx, int64_t ny,
                                    double *d_vC, double *d_vDM, double *d_vNI, int64_t *d_acc_lin, double *d_acc_C,
                                    uint32_t *d_count, hipStream_t st) {
  if (M <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_region_accept, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, st, d_rows, M, d_ns, d_ni,
                     d_C, d_med, d_p1, nx, ny, d_vC, d_vDM, d_vNI, d_acc_lin, d_acc_C, d_count);
  return hipGetLastError();
}

/* out[i] = v[lin[i]] (lin checked by the caller) */
__global__ void k_gather_f64(const double *v, const int64_t *lin, int64_t n, double *out) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) out[i] = v[lin[i]];
}

hipError_t grs_launch_gather_f64(const double *d_v, const int64_t *d_lin, int64_t n, double *d_out, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  const int64_t blocks = (n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536;
  hipLaunchKernelGGL(k_gather_f64, dim3((unsigned)blocks), dim3(256), 0, st, d_v, d_lin, n, d_out);
  return hipGetLastError();
}

/* v[lin[i]] = val[i] (lin checked by the caller, no index repeated) */
__global__ void k_scatter_f64(double *v, const int64_t *lin, const double *val, int64_t n) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) v[lin[i]] = val[i];
}

hipError_t grs_launch_scatter_f64(double *d_v, const int64_t *d_lin, const double *d_val, int64_t n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  const int64_t blocks = (n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536;
  hipLaunchKernelGGL(k_scatter_f64, dim3((unsigned)blocks), dim3(256), 0, st, d_v, d_lin, d_val, n);
  return hipGetLastError();
}
