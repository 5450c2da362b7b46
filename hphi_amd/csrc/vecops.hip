// Streaming vector kernels used by the host C drivers (Lanczos, TPQ, LOBPCG).
// All reductions are two-stage with a fixed grid and a fixed summation order,
// so a result depends only on the data, never on scheduling.
#include <hip/hip_runtime.h>

#include <cstring>

#include "engine_internal.h"
#include "hphi_amd.h"

#define HIPCHK(x)                                                                  \
  do {                                                                             \
    hipError_t e_ = (x);                                                           \
    if (e_ != hipSuccess) return hphi_set_error("%s failed: %s", #x, hipGetErrorString(e_)); \
  } while (0)

#define VO_TPB 256
#define VO_GRID 2048

__device__ __forceinline__ double block_sum(double v, double *sh) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < VO_TPB / 64; w++) s += sh[w];
  __syncthreads();
  return s;
}

// beta^2 = sum |v0 - alpha v1|^2   (Lanczos_EigenValue.c:170-177)
__global__ __launch_bounds__(VO_TPB) void k_lanczos_beta(const double2 *v0, const double2 *v1, uint64_t n,
                                                         double alpha, double *partial) {
  __shared__ double sh[VO_TPB / 64];
  double s = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * VO_TPB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * VO_TPB) {
    double2 a = v0[i], b = v1[i];
    double r = a.x - alpha * b.x, m = a.y - alpha * b.y;
    s += r * r + m * m;
  }
  s = block_sum(s, sh);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// Lanczos residual with the normalisation deferred: r <- r - f w (f = alpha_m
// s_m, w the unnormalised Lanczos vector of step m), |r|^2 per block; with vg
// also vg += cg w (the eigenvector sum).  One pass of 48 bytes per state.
// With lz (the state of a run, see k_lz_step) f comes from it and prdct.
__global__ __launch_bounds__(VO_TPB) void k_lz_resid(double2 *r, const double2 *w, double2 *vg, uint64_t n, double f,
                                                     double cg, double *partial, double *lz, const double2 *prdct) {
  __shared__ double sh[VO_TPB / 64];
  if (lz) {
    f = lz[1] * lz[1] * prdct->x * lz[1];
    if (blockIdx.x == 0 && threadIdx.x == 0) lz[2] = (double)wall_clock64();
  }
  double s = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * VO_TPB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * VO_TPB) {
    const double2 a = r[i], b = w[i];
    const double2 t = make_double2(a.x - f * b.x, a.y - f * b.y);
    r[i] = t;
    s += t.x * t.x + t.y * t.y;
    if (vg) {
      const double2 g = vg[i];
      vg[i] = make_double2(g.x + cg * b.x, g.y + cg * b.y);
    }
  }
  s = block_sum(s, sh);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// temp1 = v1; temp2 = (v0 - alpha v1)/beta; v0 = -beta temp1; v1 = temp2
// (Lanczos_EigenValue.c:154-160)
__global__ __launch_bounds__(VO_TPB) void k_lanczos_update(double2 *v0, double2 *v1, uint64_t n, double alpha,
                                                           double beta) {
  for (uint64_t i = (uint64_t)blockIdx.x * VO_TPB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * VO_TPB) {
    double2 a = v0[i], b = v1[i];
    double2 t2 = make_double2((a.x - alpha * b.x) / beta, (a.y - alpha * b.y) / beta);
    v0[i] = make_double2(-beta * b.x, -beta * b.y);
    v1[i] = t2;
  }
}

// Per-column sums of a [n][K] block, one read of the block.  Column c of
// workgroup b is the sum over 256 "rows" t of the terms i = b 256 + t + m 256
// grid, each row in ascending m, the rows by block_sum's tree.  Thread t holds
// column t % K of the K rows r (256/K) + t / K, so a wave reads consecutive
// amplitudes; the rows pass through LDS to that tree.  (One column after
// another, each strided by 16 K bytes, read the block K times: 148 us for the
// norms and 322 us for the dots of 8 columns of 2^20 states; now 33 and 71, a
// read at 3.8-4.1 TB/s.)
template <int K, int NV, class F>
__device__ __forceinline__ void col_sums(uint64_t n, double *partial, F term) {
  __shared__ double sh[VO_TPB / 64];
  __shared__ double rows[VO_TPB][K + (K > 1)];  // padded against bank conflicts
  const int c = threadIdx.x % K, g = threadIdx.x / K;
  double s[NV][K];
#pragma unroll
  for (int q = 0; q < NV; q++)
#pragma unroll
    for (int r = 0; r < K; r++) s[q][r] = 0.0;
  for (uint64_t i0 = (uint64_t)blockIdx.x * VO_TPB; i0 < n; i0 += (uint64_t)gridDim.x * VO_TPB) {
#pragma unroll
    for (int r = 0; r < K; r++) {
      const uint64_t i = i0 + r * (VO_TPB / K) + g;
      if (i < n) {
        double v[NV];
        term(i * K + c, v);
#pragma unroll
        for (int q = 0; q < NV; q++) s[q][r] += v[q];
      }
    }
  }
#pragma unroll
  for (int q = 0; q < NV; q++) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < K; r++) rows[r * (VO_TPB / K) + g][c] = s[q][r];
    __syncthreads();
    for (int cc = 0; cc < K; cc++) {
      const double t = block_sum(rows[threadIdx.x][cc], sh);
      if (threadIdx.x == 0) partial[NV * ((uint64_t)blockIdx.x * K + cc) + q] = t;
    }
  }
}

// squared norms: partial[blk*K + c]
template <int K>
__global__ __launch_bounds__(VO_TPB) void k_norm2(const double2 *v, uint64_t n, double *partial) {
  col_sums<K, 1>(n, partial, [&](uint64_t e, double *s) {
    const double2 a = v[e];
    s[0] = a.x * a.x + a.y * a.y;
  });
}

// <x_c|y_c>: partial[2*(blk*K + c)] (re, im)
template <int K>
__global__ __launch_bounds__(VO_TPB) void k_dot(const double2 *x, const double2 *y, uint64_t n, double *partial) {
  col_sums<K, 2>(n, partial, [&](uint64_t e, double *s) {
    const double2 a = x[e], b = y[e];
    s[0] = a.x * b.x + a.y * b.y;
    s[1] = a.x * b.y - a.y * b.x;
  });
}

// the same sums for a number of columns with no kernel of its own, a column at a time
__global__ __launch_bounds__(VO_TPB) void k_norm2_any(const double2 *v, uint64_t n, int k, double *partial) {
  __shared__ double sh[VO_TPB / 64];
  for (int c = 0; c < k; c++) {
    double s = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * VO_TPB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * VO_TPB) {
      double2 a = v[i * k + c];
      s += a.x * a.x + a.y * a.y;
    }
    s = block_sum(s, sh);
    if (threadIdx.x == 0) partial[(uint64_t)blockIdx.x * k + c] = s;
  }
}

__global__ __launch_bounds__(VO_TPB) void k_dot_any(const double2 *x, const double2 *y, uint64_t n, int k,
                                                    double *partial) {
  __shared__ double sh[VO_TPB / 64];
  for (int c = 0; c < k; c++) {
    double sr = 0.0, si = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * VO_TPB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * VO_TPB) {
      double2 a = x[i * k + c], b = y[i * k + c];
      sr += a.x * b.x + a.y * b.y;
      si += a.x * b.y - a.y * b.x;
    }
    sr = block_sum(sr, sh);
    si = block_sum(si, sh);
    if (threadIdx.x == 0) {
      partial[2 * ((uint64_t)blockIdx.x * k + c)] = sr;
      partial[2 * ((uint64_t)blockIdx.x * k + c) + 1] = si;
    }
  }
}

#define VO_DISPATCH(KK, CALL, OTHER) \
  switch (KK) {                      \
    case 1: CALL(1); break;          \
    case 2: CALL(2); break;          \
    case 4: CALL(4); break;          \
    case 8: CALL(8); break;          \
    case 16: CALL(16); break;        \
    default: OTHER;                  \
  }

// y_c = a_c x_c + b_c y_c  (complex a, b per column)
__global__ __launch_bounds__(VO_TPB) void k_axpby(const double2 *x, double2 *y, uint64_t n, int k,
                                                  const double2 *ab) {
  for (uint64_t i = (uint64_t)blockIdx.x * VO_TPB + threadIdx.x; i < n * k; i += (uint64_t)gridDim.x * VO_TPB) {
    int c = (int)(i % k);
    double2 a = ab[2 * c], b = ab[2 * c + 1], xv = x[i], yv = y[i];
    y[i] = make_double2(a.x * xv.x - a.y * xv.y + b.x * yv.x - b.y * yv.y,
                        a.x * xv.y + a.y * xv.x + b.x * yv.y + b.y * yv.x);
  }
}

// out[c] = sum_b partial[b*m + c]: one workgroup per c, strided per-thread
// sums then a tree, the same order on every call
__global__ __launch_bounds__(VO_TPB) void k_sum_partials(const double *partial, int nblk, int m, double *out) {
  __shared__ double sh[VO_TPB];
  const int c = blockIdx.x;
  double s = 0.0;
  for (int b = threadIdx.x; b < nblk; b += VO_TPB) s += partial[(uint64_t)b * m + c];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int st = VO_TPB / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[c] = sh[0];
}

static int vo_grid(uint64_t n) {
  uint64_t g = (n + VO_TPB - 1) / VO_TPB;
  if (g > VO_GRID) g = VO_GRID;
  if (g < 1) g = 1;
  return (int)g;
}

// scratch: e->d_partial holds HV_MAX_GRID*16 double2 = enough for VO_GRID*32 doubles
static int finish_sum(hphi_engine *e, int g, int m, double *host_out) {
  double *part = (double *)e->d_partial;
  hipLaunchKernelGGL(k_sum_partials, dim3(m), dim3(VO_TPB), 0, e->stream, part, g, m, (double *)e->hd_prdct);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(e->stream));
  memcpy(host_out, e->h_prdct, sizeof(double) * m);
  return 0;
}

extern "C" int hphi_vec_lanczos_resid(hphi_engine *e, double *r, const double *w, double *vg, double f, double cg,
                                      double *r2) {
  if (!e || !r || !w || !r2) return hphi_set_error("hphi_vec_lanczos_resid: NULL argument");
  int g = vo_grid(e->dim);
  hipLaunchKernelGGL(k_lz_resid, dim3(g), dim3(VO_TPB), 0, e->stream, (double2 *)r, (const double2 *)w,
                     (double2 *)vg, e->dim, f, cg, (double *)e->d_partial, (double *)nullptr, (const double2 *)nullptr);
  return finish_sum(e, g, 1, r2);
}

// ---- Lanczos steps without the host: lz = (c0, c1 = s_m) of the next H·v and
// the clock at the start of its residual pass
__global__ void k_lz_set(double *lz, double c0, double c1) {
  lz[0] = c0;
  lz[1] = c1;
}

// Ends a step: |r|^2 (summed as k_sum_partials does), alpha_m and beta_m, the
// scale factors of the next step, and (alpha, beta, ticks of the residual
// pass) to the host's ring.  The same operations as the host's, so a run gives
// the same bits either way.
__global__ __launch_bounds__(VO_TPB) void k_lz_step(const double *partial, int nblk, const double2 *prdct, double *lz,
                                                    double *ring) {
  __shared__ double sh[VO_TPB];
  double t = 0.0;
  for (int b = threadIdx.x; b < nblk; b += VO_TPB) t += partial[b];
  sh[threadIdx.x] = t;
  __syncthreads();
  for (int st = VO_TPB / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double s = lz[1], beta = sqrt(sh[0]);
    ring[0] = s * s * prdct->x;
    ring[1] = beta;
    ring[2] = (double)wall_clock64() - lz[2];
    lz[0] = -beta * s;
    lz[1] = 1.0 / beta;
  }
}

static double *lz_state_dev(hphi_engine *e) { return (double *)e->d_prdct + 32; }
static double *lz_ring(void *base) { return (double *)base + 2 * HV_HOST_PARTIALS; }

// the next step's H·v will be v0 <- c0 v0 + c1 H v1
extern "C" int hphi_lz_set(hphi_engine *e, double c0, double c1) {
  if (hphi_build_tables(e) || hphi_build_diag(e)) return -1;  // a restarted run comes here first
  for (int i = 0; i < 2; i++)
    if (!e->lz_ev[i]) HIPCHK(hipEventCreateWithFlags(&e->lz_ev[i], hipEventDisableTiming));
  hipLaunchKernelGGL(k_lz_set, dim3(1), dim3(1), 0, e->stream, lz_state_dev(e), c0, c1);
  HIPCHK(hipGetLastError());
  return 0;
}

// Queues one step: r <- c0 r + c1 H w, then the residual pass r <- r - alpha s w;
// slot: the ring entry of its results.  Waits for nothing.
extern "C" int hphi_lz_step(hphi_engine *e, double *r, const double *w, int slot) {
  double *lz = lz_state_dev(e);
  const double2 *prdct = (const double2 *)e->d_prdct;
  if (hphi_hv_launch_cdev(e, r, w, lz)) return -1;
  const int g = vo_grid(e->dim);
  hipLaunchKernelGGL(k_lz_resid, dim3(g), dim3(VO_TPB), 0, e->stream, (double2 *)r, (const double2 *)w,
                     (double2 *)nullptr, e->dim, 0.0, 0.0, (double *)e->d_partial, lz, prdct);
  hipLaunchKernelGGL(k_lz_step, dim3(1), dim3(VO_TPB), 0, e->stream, (const double *)e->d_partial, g, prdct, lz,
                     lz_ring(e->hd_prdct) + 4 * (slot % LZ_RING));
  HIPCHK(hipGetLastError());
  return 0;
}

extern "C" int hphi_lz_mark(hphi_engine *e, int i) {
  HIPCHK(hipEventRecord(e->lz_ev[i & 1], e->stream));
  return 0;
}
extern "C" int hphi_lz_wait(hphi_engine *e, int i) {
  HIPCHK(hipEventSynchronize(e->lz_ev[i & 1]));
  return 0;
}

// a waited step's alpha, beta and the seconds of its residual pass
extern "C" void hphi_lz_read(const hphi_engine *e, int slot, double *out) {
  const double *p = lz_ring(e->h_prdct) + 4 * (slot % LZ_RING);
  out[0] = p[0];
  out[1] = p[1];
  out[2] = 1e-8 * p[2];  // 100 MHz
}

extern "C" int hphi_vec_lanczos_beta(hphi_engine *e, const double *v0, const double *v1, double alpha,
                                     double *beta2) {
  if (!e || !v0 || !v1 || !beta2) return hphi_set_error("hphi_vec_lanczos_beta: NULL argument");
  int g = vo_grid(e->dim);
  hipLaunchKernelGGL(k_lanczos_beta, dim3(g), dim3(VO_TPB), 0, e->stream, (const double2 *)v0,
                     (const double2 *)v1, e->dim, alpha, (double *)e->d_partial);
  return finish_sum(e, g, 1, beta2);
}

// the update above plus vg += c * v1_new (eigenvector accumulation)
__global__ __launch_bounds__(VO_TPB) void k_lanczos_update_acc(double2 *v0, double2 *v1, double2 *vg, uint64_t n,
                                                               double alpha, double beta, double c) {
  for (uint64_t i = (uint64_t)blockIdx.x * VO_TPB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * VO_TPB) {
    double2 a = v0[i], b = v1[i], g = vg[i];
    double2 t2 = make_double2((a.x - alpha * b.x) / beta, (a.y - alpha * b.y) / beta);
    v0[i] = make_double2(-beta * b.x, -beta * b.y);
    v1[i] = t2;
    vg[i] = make_double2(g.x + c * t2.x, g.y + c * t2.y);
  }
}
extern "C" int hphi_vec_lanczos_update_acc(hphi_engine *e, double *v0, double *v1, double *vg, double alpha,
                                           double beta, double c) {
  if (!e || !v0 || !v1 || !vg) return hphi_set_error("hphi_vec_lanczos_update_acc: NULL argument");
  hipLaunchKernelGGL(k_lanczos_update_acc, dim3(vo_grid(e->dim)), dim3(VO_TPB), 0, e->stream, (double2 *)v0,
                     (double2 *)v1, (double2 *)vg, e->dim, alpha, beta, c);
  HIPCHK(hipGetLastError());
  // the copy / zero / fill helpers run on the null stream, which is not ordered
  // against the engine's non-blocking stream: finish before returning
  HIPCHK(hipStreamSynchronize(e->stream));
  return 0;
}
extern "C" int hphi_vec_lanczos_update(hphi_engine *e, double *v0, double *v1, double alpha, double beta) {
  if (!e || !v0 || !v1) return hphi_set_error("hphi_vec_lanczos_update: NULL argument");
  hipLaunchKernelGGL(k_lanczos_update, dim3(vo_grid(e->dim)), dim3(VO_TPB), 0, e->stream, (double2 *)v0,
                     (double2 *)v1, e->dim, alpha, beta);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(e->stream));
  return 0;
}

extern "C" int hphi_vec_norm2(hphi_engine *e, const double *v, int k, double *out) {
  if (!e || !v || !out || k < 1 || k > 16) return hphi_set_error("hphi_vec_norm2: bad argument");
  int g = vo_grid(e->dim);
#define VO_CALL(K) \
  hipLaunchKernelGGL(k_norm2<K>, dim3(g), dim3(VO_TPB), 0, e->stream, (const double2 *)v, e->dim, (double *)e->d_partial)
  VO_DISPATCH(k, VO_CALL,
              hipLaunchKernelGGL(k_norm2_any, dim3(g), dim3(VO_TPB), 0, e->stream, (const double2 *)v, e->dim, k,
                                 (double *)e->d_partial))
#undef VO_CALL
  return finish_sum(e, g, k, out);
}

extern "C" int hphi_vec_dot(hphi_engine *e, const double *x, const double *y, int k, double *out) {
  if (!e || !x || !y || !out || k < 1 || k > 16) return hphi_set_error("hphi_vec_dot: bad argument");
  int g = vo_grid(e->dim);
#define VO_CALL(K)                                                                                          \
  hipLaunchKernelGGL(k_dot<K>, dim3(g), dim3(VO_TPB), 0, e->stream, (const double2 *)x, (const double2 *)y, \
                     e->dim, (double *)e->d_partial)
  VO_DISPATCH(k, VO_CALL,
              hipLaunchKernelGGL(k_dot_any, dim3(g), dim3(VO_TPB), 0, e->stream, (const double2 *)x,
                                 (const double2 *)y, e->dim, k, (double *)e->d_partial))
#undef VO_CALL
  return finish_sum(e, g, 2 * k, out);
}

extern "C" int hphi_vec_axpby(hphi_engine *e, const double *x, double *y, int k, const double *ab) {
  if (!e || !x || !y || !ab || k < 1 || k > 16) return hphi_set_error("hphi_vec_axpby: bad argument");
  double2 *d_ab = (double2 *)e->d_coef;
  HIPCHK(hipMemcpyAsync(d_ab, ab, sizeof(double2) * 2 * k, hipMemcpyHostToDevice, e->stream));
  hipLaunchKernelGGL(k_axpby, dim3(vo_grid(e->dim * k)), dim3(VO_TPB), 0, e->stream, (const double2 *)x,
                     (double2 *)y, e->dim, k, (const double2 *)d_ab);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(e->stream));
  return 0;
}

extern "C" int hphi_engine_sync(hphi_engine *e) {
  if (!e) return hphi_set_error("NULL engine");
  HIPCHK(hipStreamSynchronize(e->stream));
  return 0;
}
