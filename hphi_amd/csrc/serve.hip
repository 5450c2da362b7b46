// Continuous-batching Lanczos service: many small diagonalisation jobs share
// every kernel launch.
//
// Each job is a canonical Hamiltonian (Spin or Hubbard) whose lowest n
// eigenvalues are wanted.  Jobs whose basis and term structure agree (same
// lattice and sector; couplings may differ) share a slab: one copy of the
// basis tables, and SL_K interleaved columns (element j*SL_K + c) for the
// Lanczos vectors, the diagonal and the couplings.  One lane per basis state
// decodes the state's bits, predicates, Jordan-Wigner signs and target
// indices once and applies them to every running column of its slab, so up
// to SL_K jobs pay for one index decode and read one 64-byte row per term;
// large sectors with a class layout run by classes (hphi_slab_cls_pays).
//
// A tick
//   1. admits waiting jobs: first, free columns of running slabs go to arrived
//      jobs of the same structure among the first ADMIT_WINDOW waiting (slab
//      steps cost about the same however many columns run); then jobs are
//      admitted in arrival order (the largest first among jobs that arrive
//      together), into a free column of a slab of the same
//      structure, or into a new slab while its HBM footprint (tables, SL_K
//      columns of diagonal and two Lanczos vectors, alpha/beta histories) fits
//      the arena; a new column gets its couplings, its diagonal and its start
//      vector on the device;
//   2. advances every running job by S steps (S = the convergence-check
//      interval, at most SL_SMAX; fewer when a job reaches its dimension or
//      the step limit) of the reference's plain Lanczos recurrence
//      (src/Lanczos_EigenValue.c:153-177): per step four packed launches over
//      all slabs (residual + norm, beta, H·v, alpha), then one launch of the
//      batched eigenvalue check, with no host round trip between the steps
//      (a workgroup takes one tile of SV_TPB states, XCD-contiguous);
//   3. copies the (alpha, beta) of every step and the check results of all
//      jobs to the host in one transfer each, tests convergence of the lowest
//      n distinct Ritz values (Cullum-Willoughby filtered) and retires
//      converged jobs, freeing a slab's arena memory when its last job leaves.
//
// The recurrence is rearranged so that every vector is touched by two passes
// per step.  A slab keeps two arrays, R and Q.  At step m of a column, R
// holds r = v0 after the previous H·v and Q holds w_{m-1}, the previous
// Lanczos vector before normalisation (v_{m-1} = s_{m-1} w_{m-1}):
//   pass 1: w_m = r - alpha_{m-1} s_{m-1} w_{m-1}, written over R, and |w_m|^2;
//   beta_{m-1} = |w_m|, s_m = 1/beta_{m-1};
//   pass 2: Q <- -beta_{m-1} s_{m-1} Q + s_m (H w_m)  (= -beta v_{m-1} + H v_m)
//           and alpha_m = s_m^2 <w_m|H w_m>;
// then R and Q swap roles for the whole slab (every column steps every tick;
// a new column is started in the slab's current R).  This is the
// reference's v1 <- (v0 - alpha v1)/beta, v0 <- -beta v1 + H v1 with the
// division by beta folded into the H·v.
//
// Tiles map to slabs through a prefix table.  A job's reductions run over its
// slab's tiles in a fixed order and its column's arithmetic does not depend
// on the other columns, so its result is bit-identical alone and in any mix.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <deque>
#include <map>
#include <time.h>
#include <vector>

#include "engine_internal.h"
#include "hv_class.h"
#include "hphi_amd.h"

#define HIPCHK(x)                                                                  \
  do {                                                                             \
    hipError_t e_ = (x);                                                           \
    if (e_ != hipSuccess) return hphi_set_error("%s failed: %s", #x, hipGetErrorString(e_)); \
  } while (0)

#define SV_TPB 256  // one tile = SV_TPB states of one slab
#define SL_K 4      // columns (jobs) per slab (8 with one lane per state: 2-3 waves per SIMD, slower per column)
#define SL_U 2      // terms per gather batch (SL_U * SL_K gathers in flight)
#define SL_SMAX 16  // Lanczos steps per tick at most
#define SL_TPW 1    // tiles per workgroup (a chunk): 1, 2, 4, 8 measured, 1 fastest at every job size

struct SlabDev {
  uint64_t dim;
  const uint64_t *list1;
  const uint4 *l21p;  // list_2_1 as uint16, zero-padded to a multiple of 8 entries
  const uint64_t *l22;
  const GTerm *terms;   // term structure of the slab (couplings in coef)
  const double2 *coef;  // [n_terms][SL_K]
  const double *diag;   // [dim][SL_K]
  double2 *R, *Q;       // [dim][SL_K]
  uint64_t irght, size21;
  int n_low, n_high, n_mixed, nlow;
  int mask;   // columns with a running job
  int realc;  // columns whose couplings are all real
  int slot[SL_K];
  const ClsArgs *cls;  // class layout of the slab, or null
  int sgn;             // terms carry Jordan-Wigner signs
};
struct ColDev {  // one running job in one step of a tick
  int slab, col, slot;
  int step, check;  // Lanczos step computed (1-based); run the eigenvalue check after it
  int job;          // index of the job in the tick (rows of the outputs)
  double *ahist, *bhist;
};
typedef const SlabDev __attribute__((address_space(4))) *CSlab;
typedef const ColDev __attribute__((address_space(4))) *CCol;
typedef const ClsArgs __attribute__((address_space(4))) *CCls;
typedef const uint64_t __attribute__((address_space(4))) *CU64;
typedef const double __attribute__((address_space(4))) *CD2;  // couplings as (re, im) doubles

// job state per slot (device): [0] alpha_{m-1}, [1] s_{m-1}, [2] beta_{m-1}, [3] s_m
#define JS_STRIDE 4

__device__ __forceinline__ int find_slab(CU64 prefix, int n, uint64_t tile) {
  int lo = 0, hi = n;  // prefix[lo] <= tile < prefix[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (prefix[mid] <= tile) lo = mid;
    else hi = mid;
  }
  return lo;
}

// XCD-contiguous chunk order.  Workgroups are dealt to the 8 XCDs round-robin
// by blockIdx, so workgroup b of a grid of G (a multiple of 8) takes logical
// chunk (b % 8) G/8 + b / 8: each XCD sweeps one contiguous range of chunks,
// and the gathers of neighbouring states meet in that XCD's own L2.  Logical
// chunks at or past the launch's total (the rounding) have no work.
__device__ __forceinline__ uint64_t sl_chunk() {
  return (uint64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
}

// Pass 2 costs a workgroup more or less by its slab's terms, so each XCD takes
// an eighth of every slab, not of the launch: slab sb has prefix[sb + 1] - prefix[sb]
// chunks, a multiple of 8; workgroup b takes chunk (b % 8) of its slab's eight ranges.
__device__ __forceinline__ uint64_t sl_chunk8(CU64 prefix, int ns, int *sb) {
  const uint64_t slot = blockIdx.x >> 3, p0 = prefix[0];
  *sb = find_slab(prefix, ns, p0 + 8 * slot);
  const uint64_t at = prefix[*sb], m = prefix[*sb + 1] - at;
  return at + (uint64_t)(blockIdx.x & 7) * (m >> 3) + (slot - ((at - p0) >> 3));
}

// pass 1: w = r - alpha_{m-1} s_{m-1} q over R per running column, |w|^2 per
// chunk of SL_TPW tiles.  Lane (state, column) = (base + t / SL_K, t % SL_K), so
// every load and store of a wave covers one contiguous range of rows.
__global__ __launch_bounds__(SV_TPB) void k_sl_resid(const SlabDev *slabs, const uint64_t *prefix, int ns,
                                                     const double *js, double *partial) {
  const uint64_t chunk = sl_chunk();
  if (chunk >= ((CU64)prefix)[ns]) return;
  const int sb = find_slab((CU64)prefix, ns, chunk);
  CSlab S = (CSlab)slabs + sb;
  const int c = threadIdx.x % SL_K;
  const bool run = (S->mask >> c) & 1;
  const int sl = S->slot[c];
  const double f = js[sl * JS_STRIDE + 0] * js[sl * JS_STRIDE + 1];
  const uint64_t e0 = (chunk - ((CU64)prefix)[sb]) * SL_TPW * SV_TPB * SL_K + threadIdx.x;
  const uint64_t n = S->dim * SL_K, cend = e0 - threadIdx.x + (uint64_t)SL_TPW * SV_TPB * SL_K;
  const uint64_t eend = n < cend ? n : cend;
  double2 *__restrict__ R = S->R;
  const double2 *__restrict__ Q = S->Q;
  double acc = 0.0;
  if (run) {
    for (uint64_t e = e0; e < eend; e += SV_TPB) {
      double2 w = R[e];
      if (f != 0.0) {
        const double2 q = Q[e];
        w = make_double2(w.x - f * q.x, w.y - f * q.y);
        R[e] = w;
      }
      acc += w.x * w.x + w.y * w.y;
    }
  }
  // lanes with equal t % SL_K hold one column
  for (int off = 32; off >= SL_K; off >>= 1) acc += __shfl_xor(acc, off, 64);
  __shared__ double red[SV_TPB / 64][SL_K];
  if ((threadIdx.x & 63) < SL_K) red[threadIdx.x >> 6][threadIdx.x & 63] = acc;
  __syncthreads();
  if (threadIdx.x < SL_K) {
    double t = 0.0;
    for (int w = 0; w < SV_TPB / 64; w++) t += red[w][threadIdx.x];
    partial[chunk * SL_K + threadIdx.x] = t;
  }
}

__device__ __forceinline__ bool sl_pred(int kind, uint32_t tmask, uint32_t tval, uint32_t x) {
  const uint32_t ym = x & tmask;
  const int pc = __popc(ym);
  return (kind == P_EQ) ? (ym == tval) : ((kind == P_DIFF) ? (pc == 1) : (pc != 1));
}

__device__ __forceinline__ double sl_sign(uint32_t sgn, uint32_t x) {
  return (sgn != 0u && (__popc(x & sgn) & 1)) ? -1.0 : 1.0;
}

// acc_c += coef[t][c] * s * g_c for every column of the slab.  Columns without
// a running job are computed too (their results are never stored), so the
// term loop carries no per-column tests.  REAL: the couplings of every
// running column are real.  The complex form applies the imaginary part in
// separate fused steps after the real one, so a real column gets the same
// values on either path: a fused step with a zero factor adds a zero.
template <bool REAL>
__device__ __forceinline__ void sl_mac(double *ar, double *ai, CD2 cf, double s, const double2 *g) {
#pragma unroll
  for (int c = 0; c < SL_K; c++) {
    const double cr = s * cf[2 * c];
    ar[c] = __builtin_fma(cr, g[c].x, ar[c]);
    ai[c] = __builtin_fma(cr, g[c].y, ai[c]);
    if (!REAL) {
      const double ci = s * cf[2 * c + 1];
      ar[c] = __builtin_fma(-ci, g[c].y, ar[c]);
      ai[c] = __builtin_fma(ci, g[c].x, ai[c]);
    }
  }
}

__device__ __forceinline__ void sl_load(const double2 *__restrict__ row, bool act, double2 *g) {
#pragma unroll
  for (int c = 0; c < SL_K; c++) g[c] = make_double2(0.0, 0.0);
  if (act) {
#pragma unroll
    for (int c = 0; c < SL_K; c++) g[c] = row[c];
  }
}

// (H w)_c of one state j of slab S for the running columns, then
// Q_c <- cc_c Q_c + s_c (H w)_c and <w_c|H w_c> accumulated into (pre, pim).
// Gather form of the reference's per-term scatter (mltplySpinCore.c:273-307,
// mltplyHubbardCore.c:305-347); list_2_1 is read from the LDS copy s21.
template <bool REAL>
__device__ __forceinline__ void sl_hv_state(CSlab S, uint64_t j, const uint16_t *s21, const double *js, double *pre,
                                            double *pim) {
  const uint64_t dim = S->dim;
  const bool valid = j < dim;
  const uint64_t jj = valid ? j : dim - 1;
  const int mask = S->mask;
  const double2 *__restrict__ R = S->R;
  const uint64_t *__restrict__ l22 = S->l22;
  const uint32_t irght = (uint32_t)S->irght;
  const int nlow = S->nlow;
  const CTerm tl = (CTerm)S->terms;
  const CTerm th = tl + S->n_low;
  const CTerm tm = th + S->n_high;
  const CD2 cl = (CD2)S->coef;
  const CD2 ch = cl + (uint64_t)S->n_low * SL_K * 2;
  const CD2 cm = ch + (uint64_t)S->n_high * SL_K * 2;
  const uint32_t x = (uint32_t)S->list1[jj];
  double ar[SL_K], ai[SL_K];
  double2 own[SL_K];
#pragma unroll
  for (int c = 0; c < SL_K; c++) {
    own[c] = R[jj * SL_K + c];
    const double d = S->diag[jj * SL_K + c];
    ar[c] = d * own[c].x;
    ai[c] = d * own[c].y;
  }
  const uint32_t ia = x & irght, ib = x >> nlow;
  const int64_t b21 = (int64_t)s21[ia];
  // ---- low-half terms: same block
  for (int t = 0; t < S->n_low; t += SL_U) {
    uint64_t idx[SL_U];
    bool act[SL_U];
#pragma unroll
    for (int u = 0; u < SL_U; u++) {
      const GTerm T = load_term(tl + t + u);
      const uint32_t y = x ^ (uint32_t)T.flip;
      const int64_t l = (int64_t)s21[y & irght];
      idx[u] = (uint64_t)((int64_t)j + l - b21);
      act[u] = valid & sl_pred(T.kind, (uint32_t)T.tmask, (uint32_t)T.tval, x) & (l != 0) & (idx[u] < dim);
    }
    double2 g[SL_U][SL_K];
#pragma unroll
    for (int u = 0; u < SL_U; u++) sl_load(R + idx[u] * SL_K, act[u], g[u]);
#pragma unroll
    for (int u = 0; u < SL_U; u++) {
      const GTerm T = load_term(tl + t + u);
      sl_mac<REAL>(ar, ai, cl + (uint64_t)(t + u) * SL_K * 2, sl_sign((uint32_t)T.sgn, x), g[u]);
    }
  }
  // ---- high-half and mixed terms
  const uint32_t ib0 = __builtin_amdgcn_readfirstlane(ib);
  const bool uni = (__ballot(ib != ib0) == 0ull);
  if (uni) {  // the wave's states share one high block: high-term work is scalar
    const uint32_t xh = ib0 << nlow;
    const int64_t l22_0 = (int64_t)l22[ib0];
    for (int t = 0; t < S->n_high; t += SL_U) {
      uint64_t idx[SL_U];
      bool act[SL_U];
#pragma unroll
      for (int u = 0; u < SL_U; u++) {
        const GTerm T = load_term(th + t + u);
        const bool a = sl_pred(T.kind, (uint32_t)T.tmask, (uint32_t)T.tval, xh);
        int64_t l = 0;
        if (a) l = (int64_t)l22[(xh ^ (uint32_t)T.flip) >> nlow];
        idx[u] = (uint64_t)((int64_t)j + l - l22_0);
        act[u] = a & valid & (l != 0) & (idx[u] < dim);
      }
      double2 g[SL_U][SL_K];
#pragma unroll
      for (int u = 0; u < SL_U; u++) sl_load(R + idx[u] * SL_K, act[u], g[u]);
#pragma unroll
      for (int u = 0; u < SL_U; u++) {
        const GTerm T = load_term(th + t + u);
        sl_mac<REAL>(ar, ai, ch + (uint64_t)(t + u) * SL_K * 2, sl_sign((uint32_t)T.sgn, xh), g[u]);
      }
    }
    for (int t = 0; t < S->n_mixed; t += SL_U) {
      uint64_t idx[SL_U];
      bool act[SL_U];
#pragma unroll
      for (int u = 0; u < SL_U; u++) {
        const GTerm T = load_term(tm + t + u);
        const uint32_t y = x ^ (uint32_t)T.flip;
        const int64_t lb = (int64_t)l22[(xh ^ (uint32_t)T.flip) >> nlow];
        const int64_t la = (int64_t)s21[y & irght];
        idx[u] = (uint64_t)(la + lb - 3);
        act[u] = valid & sl_pred(T.kind, (uint32_t)T.tmask, (uint32_t)T.tval, x) & (la != 0) & (lb != 0) &
                 (idx[u] < dim);
      }
      double2 g[SL_U][SL_K];
#pragma unroll
      for (int u = 0; u < SL_U; u++) sl_load(R + idx[u] * SL_K, act[u], g[u]);
#pragma unroll
      for (int u = 0; u < SL_U; u++) {
        const GTerm T = load_term(tm + t + u);
        sl_mac<REAL>(ar, ai, cm + (uint64_t)(t + u) * SL_K * 2, sl_sign((uint32_t)T.sgn, x), g[u]);
      }
    }
  } else {  // lanes span several blocks: per-lane list_2_2 lookups
    for (int t = 0; t < S->n_high + S->n_mixed; t += SL_U) {
      uint64_t idx[SL_U];
      bool act[SL_U];
#pragma unroll
      for (int u = 0; u < SL_U; u++) {
        const GTerm T = load_term(th + t + u);
        const uint32_t y = x ^ (uint32_t)T.flip;
        bool a = valid & sl_pred(T.kind, (uint32_t)T.tmask, (uint32_t)T.tval, x);
        int64_t la = b21, lb = 0;
        if (a) {
          lb = (int64_t)l22[y >> nlow];
          if ((y & irght) != ia) la = (int64_t)s21[y & irght];
        }
        idx[u] = (uint64_t)(la + lb - 3);
        act[u] = a & (la != 0) & (lb != 0) & (idx[u] < dim);
      }
      double2 g[SL_U][SL_K];
#pragma unroll
      for (int u = 0; u < SL_U; u++) sl_load(R + idx[u] * SL_K, act[u], g[u]);
#pragma unroll
      for (int u = 0; u < SL_U; u++) {
        const GTerm T = load_term(th + t + u);
        sl_mac<REAL>(ar, ai, ch + (uint64_t)(t + u) * SL_K * 2, sl_sign((uint32_t)T.sgn, x), g[u]);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < SL_K; c++) {
    if (!((mask >> c) & 1) || !valid) continue;
    const int sl = S->slot[c];
    const double sc = js[sl * JS_STRIDE + 3], cc = -js[sl * JS_STRIDE + 2] * js[sl * JS_STRIDE + 1];
    double2 *q = S->Q + j * SL_K + c;
    const double2 p = *q;
    *q = make_double2(cc * p.x + sc * ar[c], cc * p.y + sc * ai[c]);
    pre[c] += own[c].x * ar[c] + own[c].y * ai[c];
    pim[c] += own[c].x * ai[c] - own[c].y * ar[c];
  }
}

// pass 2 by states, one chunk of SL_TPW tiles of a slab: Q_c <- cc_c Q_c + s_c (H w)_c
// for the running columns; <w_c|H w_c> per wave and column into red.  s21v: list_2_1 in LDS
__device__ __forceinline__ void sl_by_state(CSlab S, uint64_t chunk, const uint4 *s21v, const double *js,
                                            double2 (*red)[SL_K]) {
  const uint16_t *s21 = (const uint16_t *)s21v;
  __syncthreads();
  double pre[SL_K], pim[SL_K];
#pragma unroll
  for (int c = 0; c < SL_K; c++) pre[c] = pim[c] = 0.0;
  const uint64_t t0 = chunk * SL_TPW;
  const int full = (1 << SL_K) - 1;
  const bool real = ((S->realc | ~S->mask) & full) == full;  // every running column has real couplings
  const uint64_t dim = S->dim;
  for (int t = 0; t < SL_TPW; t++) {
    const uint64_t j = (t0 + t) * SV_TPB + threadIdx.x;
    if ((t0 + t) * SV_TPB >= dim) break;  // uniform: the chunk's last tiles may lie past the slab
    if (real) sl_hv_state<true>(S, j, s21, js, pre, pim);
    else sl_hv_state<false>(S, j, s21, js, pre, pim);
  }
#pragma unroll
  for (int c = 0; c < SL_K; c++) {
    for (int off = 32; off > 0; off >>= 1) {
      pre[c] += __shfl_xor(pre[c], off, 64);
      pim[c] += __shfl_xor(pim[c], off, 64);
    }
  }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int c = 0; c < SL_K; c++) red[threadIdx.x >> 6][c] = make_double2(pre[c], pim[c]);
}

// ---- pass 2 by classes (the layout of hv_class.hip): a wave takes 64 / SL_K ranks
// of one class in SC_B blocks of it, one column per lane, so a load instruction
// covers whole rows; low-half targets come once for all blocks, the blocks of
// high-half and mixed targets from the slab's table, couplings from LDS.
//
// A burst of 40 jobs (24-site sectors and smaller), microseconds per launch:
// by states 1,126; by classes with an eighth of the launch per XCD 1,023 (XCDs
// with the heavier slabs last), an eighth of every slab 803, units dealt so that
// workgroups running together stay neighbours 733.  It misses L2 for 4.0 GB per
// launch, 5.5 TB/s, the rate of a large copy; one or four blocks per wave cost 8 %.
#define SL_LDS (40 << 10)         // of one workgroup, for four per CU
#define SC_B 2                    // blocks per wave
#define SC_RPT (64 / SL_K)        // ranks per tile
#define SC_W (SV_TPB / 64)        // waves per workgroup
#define SC_U 8                    // terms per batch (4 the same, 2 slower)
#define SC_G 128                  // workgroups of an XCD taken to run together (64 and 256 2 % slower)
#define SC_UPW 4                  // units per wave: 1 and 2 fill LDS more often (1 %), 16 leave a tail (9 %)

template <bool REAL>
__device__ __forceinline__ void sc_mac(double2 &a, const double *cf, bool neg, double2 g) {
  const double cr = neg ? -cf[0] : cf[0];
  a.x = __builtin_fma(cr, g.x, a.x);
  a.y = __builtin_fma(cr, g.y, a.y);
  if (!REAL) {  // as sl_mac: a zero imaginary part adds zeros
    const double ci = neg ? -cf[1] : cf[1];
    a.x = __builtin_fma(-ci, g.y, a.x);
    a.y = __builtin_fma(ci, g.x, a.y);
  }
}

// sco: the terms' couplings, [term][SL_K] of (REAL ? 1 : 2) doubles; sla: row
// offsets of the mixed terms' low-half flips, [flip][ranks of the workgroup]
template <bool REAL, bool SGN>
__device__ __forceinline__ void sc_units(CSlab S, CCls C, uint32_t u0, uint32_t u1, uint32_t step,
                                         const uint16_t *s21, uint32_t *sla, const double *sco, const double *js,
                                         double *pre, double *pim) {
  constexpr int CW = REAL ? 1 : 2;
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t col = lane % SL_K, coff = col * 16u, irght = (uint32_t)S->irght;
  const CU32 bstart = (CU32)C->bstart, bxh = (CU32)C->bxh, tgt = (CU32)C->tgt;
  const int n_low = C->n_low, n_high = C->n_high, n_mixed = C->n_mixed, nt = C->nt;
  const int n_lowp = C->n_lowp, n_mixp = C->n_mixp;
  const CClsTerm TL = (CClsTerm)C->terms, TH = TL + n_low, TM = TH + n_high;
  const double2 *__restrict__ R = S->R;
  const bool run = (S->mask >> col) & 1;
  const int sl = S->slot[col];
  const double sc = js[sl * JS_STRIDE + 3], cc = -js[sl * JS_STRIDE + 2] * js[sl * JS_STRIDE + 1];
  const double *cfl = sco + col * CW, *cfh = cfl + n_low * SL_K * CW, *cfm = cfh + n_high * SL_K * CW;
  uint32_t *la = sla + wave * SC_RPT + lane / SL_K;
  for (uint32_t u = u0 + wave; u < u1; u += step) {
    int c = 0, hi = C->ncls;  // upre[c] <= u < upre[hi]
    while (hi - c > 1) {
      const int mid = (c + hi) >> 1;
      if (C->upre[mid] <= u) c = mid;
      else hi = mid;
    }
    const uint32_t loc = u - C->upre[c], ntile = C->ntile[c], size = C->size[c];
    const uint32_t grp = loc / ntile, r = (loc % ntile) * SC_RPT + lane / SL_K;
    const uint32_t p0 = C->start[c] + grp * SC_B, nb = C->start[c] + C->nblk[c] - p0;  // blocks from here on
    if (r >= size) continue;
    const uint32_t own = r * (16u * SL_K) + coff;
    uint32_t base[SC_B], xh[SC_B], row[SC_B];
    double2 acc[SC_B];
#pragma unroll
    for (int b = 0; b < SC_B; b++) {
      const uint32_t p = p0 + (b < (int)nb ? b : 0);  // past the class's last block: the first again, not stored
      base[b] = bstart[p];
      xh[b] = bxh[p];
      row[b] = p * (uint32_t)nt;
    }
    const uint32_t ia = (uint32_t)S->list1[base[0] + r] & irght;
#pragma unroll
    for (int b = 0; b < SC_B; b++) {
      const double2 w = cl_at(R + (uint64_t)base[b] * SL_K, own);
      const double d = S->diag[((uint64_t)base[b] + r) * SL_K + col];
      acc[b] = make_double2(d * w.x, d * w.y);
    }
    // ---- low-half terms
    for (int t = 0; t < n_low; t += SC_U) {
      double2 g[SC_U][SC_B];
      bool neg[SC_U];
#pragma unroll
      for (int q = 0; q < SC_U; q++) {
        const ClsTerm T = cl_term(TL + t + q);
        const uint32_t m = ia & T.tmask;
        const bool act = t < n_lowp ? (__popc(m) & 1) != 0 : m == T.tval;
        const uint32_t off = ((uint32_t)s21[ia ^ T.flip] - 2u) * (16u * SL_K) + coff;
        neg[q] = SGN && (__popc(ia & T.sgn) & 1);
#pragma unroll
        for (int b = 0; b < SC_B; b++) g[q][b] = make_double2(0.0, 0.0);
        if (act) {
#pragma unroll
          for (int b = 0; b < SC_B; b++) g[q][b] = cl_at(R + (uint64_t)base[b] * SL_K, off);
        }
      }
#pragma unroll
      for (int q = 0; q < SC_U; q++)
#pragma unroll
        for (int b = 0; b < SC_B; b++) sc_mac<REAL>(acc[b], cfl + (t + q) * SL_K * CW, neg[q], g[q][b]);
    }
    // ---- high-half terms: the same rank of another block
    for (int t = 0; t < n_high; t += SC_U) {
      double2 g[SC_U][SC_B];
      uint32_t to[SC_U][SC_B];
#pragma unroll
      for (int b = 0; b < SC_B; b++)
#pragma unroll
        for (int q = 0; q < SC_U; q++) to[q][b] = tgt[row[b] + t + q];
#pragma unroll
      for (int q = 0; q < SC_U; q++)
#pragma unroll
        for (int b = 0; b < SC_B; b++) {
          g[q][b] = make_double2(0.0, 0.0);
          if (to[q][b] != CL_NONE) g[q][b] = cl_at(R + (uint64_t)to[q][b] * SL_K, own);
        }
#pragma unroll
      for (int q = 0; q < SC_U; q++) {
        const ClsTerm T = cl_term(TH + t + q);
#pragma unroll
        for (int b = 0; b < SC_B; b++)
          sc_mac<REAL>(acc[b], cfh + (t + q) * SL_K * CW, SGN && (__popc(xh[b] & T.sgn) & 1), g[q][b]);
      }
    }
    // ---- mixed terms: the lanes of a state share its row offsets
    for (int q = (int)col; q < C->nlo; q += SL_K) la[q * (SC_W * SC_RPT)] = ((uint32_t)s21[ia ^ C->lo[q]] - 2u) * (16u * SL_K);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int t = 0; t < n_mixed; t += SC_U) {
      const bool par = t < n_mixp;
      double2 g[SC_U][SC_B];
      uint32_t to[SC_U][SC_B];
      uint32_t ls[SC_U];
#pragma unroll
      for (int b = 0; b < SC_B; b++)
#pragma unroll
        for (int q = 0; q < SC_U; q++) to[q][b] = tgt[row[b] + n_high + t + q];
#pragma unroll
      for (int q = 0; q < SC_U; q++) {
        const ClsTerm T = cl_term(TM + t + q);
        const uint32_t off = la[T.lo * (SC_W * SC_RPT)] + coff;
        const uint32_t m = ia & T.tmask, lp = par ? (uint32_t)__popc(m) & 1u : (m == T.tlo ? 1u : 0u);
        ls[q] = SGN ? (uint32_t)__popc(ia & T.sgn) : 0u;
#pragma unroll
        for (int b = 0; b < SC_B; b++) {
          // scalar: what lp must be in this block (2: never)
          const uint32_t ok = par ? ((uint32_t)__popc(xh[b] & T.tmask) & 1u) ^ 1u : 1u;
          const uint32_t want = to[q][b] == CL_NONE ? 2u : ok;
          g[q][b] = make_double2(0.0, 0.0);
          if (lp == want) g[q][b] = cl_at(R + (uint64_t)to[q][b] * SL_K, off);
        }
      }
#pragma unroll
      for (int q = 0; q < SC_U; q++) {
        const ClsTerm T = cl_term(TM + t + q);
#pragma unroll
        for (int b = 0; b < SC_B; b++)
          sc_mac<REAL>(acc[b], cfm + (t + q) * SL_K * CW, SGN && ((ls[q] + (uint32_t)__popc(xh[b] & T.sgn)) & 1u),
                       g[q][b]);
      }
    }
    if (run) {
#pragma unroll
      for (int b = 0; b < SC_B; b++) {
        if (b < (int)nb) {
          const double2 w = cl_at(R + (uint64_t)base[b] * SL_K, own);
          double2 *q = (double2 *)((char *)(S->Q + (uint64_t)base[b] * SL_K) + own);
          const double2 p = *q;
          *q = make_double2(cc * p.x + sc * acc[b].x, cc * p.y + sc * acc[b].y);
          *pre += w.x * acc[b].x + w.y * acc[b].y;
          *pim += w.x * acc[b].y - w.y * acc[b].x;
        }
      }
    }
  }
}

// couplings in class order into LDS; a padding term's are zero
template <bool REAL>
__device__ __forceinline__ void sc_coef(CSlab S, CCls C, double *sco) {
  const ClsTerm *T = C->terms;
  const int n = (C->n_low + C->nt) * SL_K;
  for (int i = threadIdx.x; i < n; i += SV_TPB) {
    const int src = T[i / SL_K].src;
    const double2 v = src < 0 ? make_double2(0.0, 0.0) : S->coef[src * SL_K + i % SL_K];
    if (REAL) sco[i] = v.x;
    else ((double2 *)sco)[i] = v;
  }
}

// pass 2 by classes, workgroup i of the slab's 8 m; LDS: list_2_1, row offsets, couplings
__device__ __forceinline__ void sl_by_class(CSlab S, CCls C, uint32_t i, uint32_t m, const uint4 *s21v, uint32_t *sla,
                                            double *sco, const double *js, double2 (*red)[SL_K]) {
  const uint16_t *s21 = (const uint16_t *)s21v;
  const int full = (1 << SL_K) - 1;
  const bool real = ((S->realc | ~S->mask) & full) == full;  // every running column has real couplings
  if (real) sc_coef<true>(S, C, sco);
  else sc_coef<false>(S, C, sco);
  __syncthreads();
  // an eighth of the units per XCD, dealt to groups of SC_G workgroups, whose
  // waves take every (4 x group)-th unit: workgroups that run together work on
  // neighbouring units, whose gathers meet in L2
  const uint32_t x = i / m, g0 = i % m / SC_G * SC_G;
  const uint32_t gn = g0 + SC_G < m ? SC_G : m - g0;
  const uint64_t X0 = (uint64_t)C->units * x / 8, XN = (uint64_t)C->units * (x + 1) / 8 - X0;
  const uint32_t u0 = (uint32_t)(X0 + XN * g0 / m) + (i % m - g0) * SC_W, u1 = (uint32_t)(X0 + XN * (g0 + gn) / m);
  double pre = 0.0, pim = 0.0;
  if (S->sgn) {
    if (real) sc_units<true, true>(S, C, u0, u1, gn * SC_W, s21, sla, sco, js, &pre, &pim);
    else sc_units<false, true>(S, C, u0, u1, gn * SC_W, s21, sla, sco, js, &pre, &pim);
  } else {
    if (real) sc_units<true, false>(S, C, u0, u1, gn * SC_W, s21, sla, sco, js, &pre, &pim);
    else sc_units<false, false>(S, C, u0, u1, gn * SC_W, s21, sla, sco, js, &pre, &pim);
  }
  for (int off = 32; off >= SL_K; off >>= 1) {
    pre += __shfl_xor(pre, off, 64);
    pim += __shfl_xor(pim, off, 64);
  }
  if ((threadIdx.x & 63) < SL_K) red[threadIdx.x >> 6][threadIdx.x & 63] = make_double2(pre, pim);
}

// Pass 2 of all slabs: by classes or by states, the slab decides.  One kernel for
// both, so that slabs of either kind fill the device together (as two launches, one
// after the other, a burst of 40 jobs takes 2 % longer); either path's registers
// allow 16 waves per CU, four workgroups, and so do 40 KB of LDS.  Dynamic LDS:
// list_2_1; by classes the row offsets (nla uint32) from the n21-th 16 bytes on, then the couplings.
__global__ __launch_bounds__(SV_TPB) void k_sl_hv(const SlabDev *slabs, const uint64_t *prefix, int ns,
                                                  const double *js, double2 *partial, uint32_t n21, uint32_t nla) {
  extern __shared__ uint4 s21v[];
  __shared__ double2 red[SC_W][SL_K];
  int sb;
  const uint64_t chunk = sl_chunk8((CU64)prefix, ns, &sb);
  CSlab S = (CSlab)slabs + sb;
  const uint32_t n8 = (uint32_t)((S->size21 + 7) / 8);  // 16-byte rows of the packed table
  for (uint32_t i = threadIdx.x; i < n8; i += SV_TPB) s21v[i] = S->l21p[i];
  const uint64_t at = ((CU64)prefix)[sb];
  if (S->cls)
    sl_by_class(S, (CCls)S->cls, (uint32_t)(chunk - at), (uint32_t)(((CU64)prefix)[sb + 1] - at) / 8, s21v,
                (uint32_t *)(s21v + n21), (double *)((uint32_t *)(s21v + n21) + nla), js, red);
  else
    sl_by_state(S, chunk - at, s21v, js, red);
  __syncthreads();
  if (threadIdx.x < SL_K) {
    double2 s = red[0][threadIdx.x];
    for (int w = 1; w < SC_W; w++) {
      s.x += red[w][threadIdx.x].x;
      s.y += red[w][threadIdx.x].y;
    }
    partial[chunk * SL_K + threadIdx.x] = s;
  }
}

// per job (one workgroup each): fixed-order sum over the slab's tiles of one
// column.  Latency-bound: up to 10,600 partial sums of a 24-site slab, eight loads
// in flight on 1,024 threads (256 threads, one each: 19.1 and 13.7 us per launch for
// beta and alpha in a burst of 40 jobs; now 8.0 and 8.4).
#define CS_TPB 1024
#define CS_U 8
__device__ double col_sum(const double *part, int stride, uint64_t t0, uint64_t t1) {
  __shared__ double s[CS_TPB / 64];
  double a[CS_U];
#pragma unroll
  for (int u = 0; u < CS_U; u++) a[u] = 0.0;
  for (uint64_t t = t0 + threadIdx.x; t < t1; t += CS_TPB * CS_U) {
#pragma unroll
    for (int u = 0; u < CS_U; u++)
      if (t + u * CS_TPB < t1) a[u] += part[(t + u * CS_TPB) * stride];
  }
#pragma unroll
  for (int u = 1; u < CS_U; u++) a[0] += a[u];
  for (int o = 32; o > 0; o >>= 1) a[0] += __shfl_xor(a[0], o, 64);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = a[0];
  __syncthreads();
  double r = 0.0;
  for (int w = 0; w < CS_TPB / 64; w++) r += s[w];
  return r;
}

// beta_{m-1} = |w_m| and s_m = 1/beta_{m-1}; a beta below 1e-14 ends the
// recurrence (the Krylov space is exhausted) and s_m = 0 keeps pass 2 finite
__global__ __launch_bounds__(CS_TPB) void k_sl_norm(const ColDev *cols, const uint64_t *prefix, const double *partial,
                                                 double *js) {
  CCol J = (CCol)cols + blockIdx.x;
  const double b2 = col_sum(partial + J->col, SL_K, ((CU64)prefix)[J->slab], ((CU64)prefix)[J->slab + 1]);
  if (threadIdx.x == 0) {
    const double b = sqrt(b2);
    double *st = js + J->slot * JS_STRIDE;
    st[2] = b;
    st[3] = (b > 0.0 && (J->step == 1 || b >= 1e-14)) ? 1.0 / b : 0.0;
    if (J->step >= 2) J->bhist[J->step - 1] = b;
  }
}

// alpha_m = s_m^2 Re <w|H w>; out = (alpha_m, beta_{m-1}) per job
__global__ __launch_bounds__(CS_TPB) void k_sl_alpha(const ColDev *cols, const uint64_t *prefix, const double2 *partial,
                                                  double *js, double *out) {
  CCol J = (CCol)cols + blockIdx.x;
  const double a = col_sum((const double *)partial + 2 * J->col, 2 * SL_K, ((CU64)prefix)[J->slab],
                           ((CU64)prefix)[J->slab + 1]);
  if (threadIdx.x == 0) {
    double *st = js + J->slot * JS_STRIDE;
    const double sc = st[3];
    const double al = a * sc * sc;
    st[0] = al;
    st[1] = sc;
    J->ahist[J->step] = al;
    out[2 * J->job] = al;
    out[2 * J->job + 1] = st[2];
  }
}

// Lowest good eigenvalues of each checking job's tridiagonal T_m (alpha[1..m],
// beta[1..m-1]) and of T_m without its first row and column, by Sturm counts;
// then the Cullum-Willoughby test and the merging of ghost copies (the rules of
// hphi_lanczos_good_eigenvalues).  out: [16 values, count] per job.
//
// One workgroup per job, and a Sturm count is a chain of m dependent divisions:
// the time is that chain times the rounds of the search.  CK_S lanes therefore
// evaluate CK_S points of an eigenvalue's interval per round (its middle and
// CK_S - 1 others): some 14 rounds of 17 sections instead of 55 halvings down to
// the same two adjacent numbers.  alpha and beta are staged in LDS (CK_LDS of
// them; longer histories are read from memory), bounds and the ghost test use all lanes.
// A burst of 40 jobs: 1,466 us per check with one lane per eigenvalue, 360-400 now.
#define CK_EXTRA 6
#define CK_TPB 512
#define CK_S 16       // lanes, i.e. points per round, of one eigenvalue's search
#define CK_LDS 2048   // rows of T_m staged in LDS
#define CK_LMAX 256   // largest window of T_m eigenvalues examined
__device__ __forceinline__ int ck_sturm(const double *a, const double *b, int n, double x) {
  int c = 0;
  double q = a[0] - x;
  for (int i = 1; i < n; i++) {
    if (fabs(q) < 1e-300) q = -1e-300;  // a vanishing pivot, and counted as such
    if (q < 0) c++;
    q = (a[i] - x) - b[i - 1] * b[i - 1] / q;
  }
  return c + (q < 0);
}

__global__ __launch_bounds__(CK_TPB) void k_sl_check(const ColDev *cols, int want, double *out) {
  CCol J = (CCol)cols + blockIdx.x;
  if (!J->check) return;
  const int m = J->step;
  const double *ga = J->ahist + 1, *gb = J->bhist + 1;
  __shared__ double sa[CK_LDS], sb[CK_LDS];
  __shared__ double ev[CK_LMAX], evh[CK_LMAX];
  __shared__ double red[3][CK_TPB / 64];
  __shared__ int next_s, bad[CK_LMAX];
  const int cap = m < CK_LMAX ? m : CK_LMAX;
  const int t = threadIdx.x;
  // Gershgorin bounds and the scale
  double lo = ga[0], hi = ga[0], scale = 0.0;
  for (int i = t; i < m; i += CK_TPB) {
    const double ai = ga[i], bi = i < m - 1 ? gb[i] : 0.0;
    if (i < CK_LDS) {
      sa[i] = ai;
      sb[i] = bi;
    }
    const double r = (i > 0 ? fabs(gb[i - 1]) : 0.0) + fabs(bi);
    lo = fmin(lo, ai - r);
    hi = fmax(hi, ai + r);
    scale = fmax(scale, fabs(ai) + r);
  }
  for (int o = 32; o > 0; o >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, o, 64));
    hi = fmax(hi, __shfl_xor(hi, o, 64));
    scale = fmax(scale, __shfl_xor(scale, o, 64));
  }
  if ((t & 63) == 0) {
    red[0][t >> 6] = lo;
    red[1][t >> 6] = hi;
    red[2][t >> 6] = scale;
  }
  __syncthreads();
  for (int w = 0; w < CK_TPB / 64; w++) {
    lo = fmin(lo, red[0][w]);
    hi = fmax(hi, red[1][w]);
    scale = fmax(scale, red[2][w]);
  }
  const double span = hi - lo;
  lo = lo - 1e-12 * span - 1e-300;
  hi = hi + 1e-12 * span + 1e-300;
  const bool staged = m <= CK_LDS;
  const int lane = t % CK_S, grp = t / CK_S, sh = (t & 63) / CK_S * CK_S;
  // Without reorthogonalisation converged eigenvalues keep gaining ghost copies,
  // which fill a fixed window of T_m's lowest eigenvalues as m grows: the window
  // starts at want + CK_EXTRA and doubles until it holds `want` good values or
  // reaches min(m, CK_LMAX).  Each round searches only the new indices.
  int L0 = 0, L = want + CK_EXTRA < cap ? want + CK_EXTRA : cap;
  for (;;) {
    const int Lh = L < m - 1 ? L : m - 1, Lh0 = L0 < m - 1 ? L0 : m - 1;
    const int nf = L - L0, ns = nf + Lh - Lh0;
    for (int s0 = 0; s0 < ns; s0 += CK_TPB / CK_S) {
      const int s = s0 + grp;
      const bool on = s < ns, hat = s >= nf;
      const int idx = !on ? 0 : hat ? Lh0 + s - nf : L0 + s, n = hat ? m - 1 : m;
      double l = lo, h = hi;
      bool work = on;
      for (int it = 0; it < 200; it++) {
        const double mid = 0.5 * (l + h);
        work = work && mid > l && mid < h;
        if (__ballot(work) == 0ull) break;
        auto point = [&](int i) { return i == CK_S / 2 - 1 ? mid : l + (h - l) * ((i + 1) * (1.0 / (CK_S + 1))); };
        bool above = false;
        if (work) {
          const double x = point(lane);
          above = (staged ? ck_sturm(sa + hat, sb + hat, n, x) : ck_sturm(ga + hat, gb + hat, n, x)) > idx;
        }
        const uint32_t mask = (uint32_t)(__ballot(above) >> sh) & ((1u << CK_S) - 1);
        if (work) {
          const int f = mask ? __ffs(mask) - 1 : CK_S;  // the first point above the eigenvalue
          const double nl = f > 0 ? fmax(l, point(f - 1)) : l, nh = f < CK_S ? fmin(h, point(f)) : h;
          l = nl;
          h = nh;
        }
      }
      if (on && lane == 0) (hat ? evh : ev)[idx] = 0.5 * (l + h);
    }
    __syncthreads();
    const double tol = 1e-11 * (scale > 1.0 ? scale : 1.0);
    for (int i = t; i < L; i += CK_TPB) {  // spurious: simple in T_m and an eigenvalue of the reduced matrix
      int mult = 0, hits = 0;
      for (int j = 0; j < L; j++) mult += fabs(ev[j] - ev[i]) <= tol;
      if (mult == 1 && i < L - 1)
        for (int j = 0; j < Lh; j++) hits += fabs(evh[j] - ev[i]) <= tol;
      bad[i] = hits;
    }
    __syncthreads();
    if (t == 0) {
      double *o = out + (uint64_t)J->job * 17;
      int got = 0;
      double last = 0.0;
      if (m == 1) {
        o[0] = ga[0];
        got = 1;
      }
      for (int i = 0; i < L && got < want && m > 1; i++) {
        if (bad[i]) continue;
        if (got > 0 && fabs(ev[i] - last) <= tol) continue;
        last = ev[i];
        o[got++] = last;
      }
      o[16] = (double)got;
      next_s = (got >= want || L >= cap) ? 0 : (2 * L < cap ? 2 * L : cap);
    }
    __syncthreads();
    const int nx = next_s;
    if (nx == 0) break;
    L0 = L;
    L = nx;
    __syncthreads();  // next_s is read by every thread before thread 0 writes it again
  }
}

// start vector of a new column: R_c = SplitMix64 uniform complex (normalised
// by the first pass), Q_c = 0, slot state zero
__global__ void k_sl_start(double2 *R, double2 *Q, int col, uint64_t dim, uint64_t seed, double *js, int slot) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < JS_STRIDE) js[slot * JS_STRIDE + i] = 0.0;
  if (i >= dim) return;
  auto mix = [](uint64_t x) {
    uint64_t y = x + 0x9E3779B97F4A7C15ull;
    y = (y ^ (y >> 30)) * 0xBF58476D1CE4E5B9ull;
    y = (y ^ (y >> 27)) * 0x94D049BB133111EBull;
    return y ^ (y >> 31);
  };
  const uint64_t s0 = seed * 0x9E3779B97F4A7C15ull;
  const double u1 = (double)(mix(s0 ^ (2 * i)) >> 11) * (1.0 / 9007199254740992.0);
  const double u2 = (double)(mix(s0 ^ (2 * i + 1)) >> 11) * (1.0 / 9007199254740992.0);
  R[i * SL_K + col] = make_double2(2.0 * u1 - 1.0, 2.0 * u2 - 1.0);
  Q[i * SL_K + col] = make_double2(0.0, 0.0);
}

// ==================================================================== host
// Which slabs run by classes (mode -1; 1: every one the layout fits).  By classes
// a wave covers 16 ranks of two blocks with four lanes per state that all test the
// term, where by states a lane tests it for its state's columns at once; it pays
// where the gathers, not those tests, are the time.  Microseconds per launch, by
// states / by classes, one slab and four:
//   Spin   20 sites, 10 up (184,756)       43 / 48     120 / 106 (rings of 40 to 64 terms from 5 x 2^15
//          23 sites, 7 up (245,157)        47 / 50     159 / 136  states on: the fuller launches count)
//          24 sites, 6 up (134,596)        43 / 50     118 / 101
//          20 sites, 190 terms (184,756)  140 / 171    452 / 437
//          22 sites, 8 up (319,770)        67 / 56     196 / 160
//          4x4 J1-J2 (12,870)              34 / 43     45 / 46
//          6x4, 6 up (134,596)             73 / 101    194 / 208
//          6x4, 7 up (346,104)            141 / 109    413 / 353
//          6x4, 12 up (2.7e6)             870 / 673
//   Hubbard 12 sites, 3 + 3 (48,400)       19 / 33     31 / 42
//          5 + 6 (731,808)                 89 / 91     261 / 250 (three slabs, as below)
//          6 + 6 (853,776)                104 / 97     306 / 301
//          13 sites, 6 + 6 (2.9e6)        386 / 347   1085 / 980
//          12 sites, 6 + 6, with 4 four-orbital InterAll pairs (a term acts on 0.39 of the
//          states, not half): 117 / 120, 341 / 353; complex hops (0.25) 140 / 139, 384 / 380
// LDS: four workgroups per CU.  All-to-all exchange on 26 sites, 7 up (657,800; 325
// terms, 42 KB): 664 / 663, 1829 / 2032; on 24 (735,471; 276 terms, 30 KB) 634 / 530, 1785 / 1413.
bool hphi_slab_cls_pays(const hphi_engine &h) {
  const bool hub = h.model == HPHI_MODEL_HUBBARD;
  double share = 0.0;
  size_t n = 0;
  std::vector<uint64_t> lo;  // low-half flips of the mixed terms
  for (const GTerm &t : h.h_terms_dev) {
    if (t.kind == P_EQ && t.tmask == 0 && t.tval != 0) continue;
    n++;
    share += t.kind != P_EQ ? 0.5 : 1.0 / (double)((uint64_t)1 << __builtin_popcountll(t.tmask));
    const uint64_t all = t.flip | t.tmask | t.sgn, f = t.flip & h.irght;
    if ((all & h.irght) && (all & ~h.irght) && std::find(lo.begin(), lo.end(), f) == lo.end()) lo.push_back(f);
  }
  if (h.dim < (hub ? (uint64_t)3 << 18 : n <= 64 ? (uint64_t)5 << 15 : (uint64_t)1 << 18)) return false;
  const size_t lds = 2 * h.size21 + sizeof(uint32_t) * SC_W * SC_RPT * lo.size() + 16 * SL_K * (n + 14) +  // padding
                     sizeof(double2) * SC_W * SL_K;
  return lds <= SL_LDS && (!hub || share >= 0.4 * (double)n);
}

namespace {

struct Arena {
  char *base = nullptr;
  size_t size = 0;
  std::map<size_t, size_t> fre;  // offset -> length
  void init(char *b, size_t n) {
    base = b;
    size = n;
    fre.clear();
    fre[0] = n;
  }
  bool alloc(size_t n, size_t *off) {
    n = (n + 255) & ~(size_t)255;
    for (auto it = fre.begin(); it != fre.end(); ++it) {
      if (it->second >= n) {
        *off = it->first;
        const size_t rest = it->second - n, o = it->first;
        fre.erase(it);
        if (rest) fre[o + n] = rest;
        return true;
      }
    }
    return false;
  }
  void release(size_t off, size_t n) {
    n = (n + 255) & ~(size_t)255;
    auto it = fre.emplace(off, n).first;
    auto nx = std::next(it);
    if (nx != fre.end() && it->first + it->second == nx->first) {
      it->second += nx->second;
      fre.erase(nx);
    }
    if (it != fre.begin()) {
      auto pv = std::prev(it);
      if (pv->first + pv->second == it->first) {
        pv->second += it->second;
        fre.erase(it);
      }
    }
  }
};

size_t al256(size_t n) { return (n + 255) & ~(size_t)255; }

struct Slab;

struct Job {
  int id = 0;
  uint64_t seed = 0;
  double t_arrival = 0, t_admit = 0, t_done = 0;
  hphi_engine h;  // host-side preparation only (no device members used)
  uint64_t shash = 0;  // structure_hash(h)
  Slab *slab = nullptr;
  int col = -1, slot = -1;
  int realc = 1;
  bool cls = false;  // its slab has the class layout
  std::vector<double> alpha, beta;
  int step = 0, nprev = 0, tick_steps = 0;
  double prev[16];
  hphi_job_result res{};
};

// The engine pads each term group (low, high, mixed) to the plain kernels'
// batch; the slab kernel reads SL_U terms per batch, so its groups keep only
// the padding that batch needs.  A padding term never matches (P_EQ with an
// empty mask and a nonzero value); no compiled term has that form.
void slab_repad(hphi_engine &h) {
  const int n[3] = {h.n_low, h.n_high, h.n_mixed};
  std::vector<GTerm> out;
  int m[3], at = 0;
  for (int g = 0; g < 3; g++) {
    const size_t start = out.size();
    for (int t = at; t < at + n[g]; t++) {
      const GTerm &x = h.h_terms_dev[t];
      if (!(x.kind == P_EQ && x.tmask == 0 && x.tval != 0)) out.push_back(x);
    }
    GTerm z{};
    z.kind = P_EQ;
    z.tmask = 0;
    z.tval = 1;
    while ((out.size() - start) % SL_U) out.push_back(z);
    m[g] = (int)(out.size() - start);
    at += n[g];
  }
  h.h_terms_dev.swap(out);
  h.n_low = m[0];
  h.n_high = m[1];
  h.n_mixed = m[2];
}

// FNV-1a over what same_structure compares: equal structures hash equally
uint64_t structure_hash(const hphi_engine &h) {
  uint64_t x = 1469598103934665603ull;
  auto mix = [&x](uint64_t v) {
    for (int b = 0; b < 8; b++) {
      x ^= (v >> (8 * b)) & 0xffu;
      x *= 1099511628211ull;
    }
  };
  mix((uint64_t)h.model);
  mix((uint64_t)h.nsite);
  mix((uint64_t)h.nup);
  mix((uint64_t)h.ndown);
  mix(h.dim);
  mix((uint64_t)h.n_low);
  mix((uint64_t)h.n_high);
  mix((uint64_t)h.n_mixed);
  mix((uint64_t)h.h_terms_dev.size());
  mix((uint64_t)h.h_dterms.size());
  for (const GTerm &t : h.h_terms_dev) {
    mix(t.flip);
    mix(t.tmask);
    mix(t.tval);
    mix(t.sgn);
    mix((uint64_t)t.kind);
  }
  return x;
}

// Jobs share a slab when basis and term structure agree (couplings may differ).
bool same_structure(const hphi_engine &a, const hphi_engine &b) {
  if (a.model != b.model || a.nsite != b.nsite || a.nup != b.nup || a.ndown != b.ndown || a.dim != b.dim ||
      a.n_low != b.n_low || a.n_high != b.n_high || a.n_mixed != b.n_mixed ||
      a.h_terms_dev.size() != b.h_terms_dev.size() || a.h_dterms.size() != b.h_dterms.size())
    return false;
  for (size_t t = 0; t < a.h_terms_dev.size(); t++) {
    const GTerm &x = a.h_terms_dev[t], &y = b.h_terms_dev[t];
    if (x.flip != y.flip || x.tmask != y.tmask || x.tval != y.tval || x.sgn != y.sgn || x.kind != y.kind)
      return false;
  }
  return true;
}

struct Slab {
  hphi_engine proto;  // structure: the first job's preparation (host side)
  uint64_t shash = 0;  // structure_hash(proto)
  size_t off = 0, bytes = 0;
  uint64_t *list1 = nullptr, *l22 = nullptr, *jb = nullptr;
  uint32_t *l21 = nullptr;
  uint16_t *l21p = nullptr;  // list_2_1 packed for the LDS copy of every workgroup
  GTerm *terms = nullptr;
  double2 *coef = nullptr;
  double *diag = nullptr;
  double2 *R = nullptr, *Q = nullptr;
  DTerm *dterms = nullptr;  // [SL_K][nd]
  double *hist = nullptr;   // [SL_K][2][max_iter + 2]
  std::vector<double2> coef_host;
  ClsArgs cls{};             // class layout (plan with device addresses)
  ClsArgs *d_cls = nullptr;  // its copy on the device; null: by states
  uint64_t hv_chunks = 0;    // workgroups of its H·v
  uint64_t nnz = 0;  // off-diagonal elements of one column's H (hphi_term_nnz)
  Job *col[SL_K] = {};
  int used() const {
    int n = 0;
    for (int c = 0; c < SL_K; c++) n += col[c] != nullptr;
    return n;
  }
};

// arena bytes of a slab; cls: with the class layout
size_t slab_footprint(const hphi_engine &h, int max_iter, bool cls) {
  const size_t nt = std::max<size_t>(h.h_terms_dev.size(), 1), nd = std::max<size_t>(h.h_dterms.size(), 1);
  return al256(8 * h.dim) + al256(4 * h.size21) + al256(16 * ((h.size21 + 7) / 8)) + al256(8 * h.size22) + al256(8 * (h.sdim + 1)) +
         al256(sizeof(GTerm) * nt) + al256(16 * SL_K * nt) + al256(8 * SL_K * h.dim) + 2 * al256(16 * SL_K * h.dim) +
         al256(sizeof(DTerm) * SL_K * nd) + al256(8 * SL_K * 2 * (size_t)(max_iter + 2)) +
         (cls ? al256(sizeof(ClsArgs)) + al256(hphi_cls_bytes_bound(&h)) : 0);
}

// The class layout, if the sector and its terms fit it, its tables leave the
// slab within the arena and list_2_1 (32 KB), row offsets (16 KB) and couplings
// (64 KB) fit LDS; the answer depends on the structure and the arena alone, so
// every slab of a structure runs the same kernel.
bool slab_cls(const hphi_engine &h, int max_iter, size_t arena, int mode) {
  return mode != 0 && (mode == 1 || hphi_slab_cls_pays(h)) && h.size21 <= 16384 && h.h_terms_dev.size() + 5 * 7 <= 1024 &&
         hphi_cls_bytes_bound(&h) && slab_footprint(h, max_iter, true) <= arena;
}

double mono_now() {
  struct timespec ts;
  clock_gettime(CLOCK_MONOTONIC, &ts);
  return ts.tv_sec + 1e-9 * ts.tv_nsec;
}

}  // namespace

struct hphi_server {
  hphi_server_params p{};
  hipStream_t stream = nullptr;
  Arena arena;
  char *d_arena = nullptr;
  double *d_js = nullptr, *d_out = nullptr, *h_out = nullptr, *d_part = nullptr;
  double *d_ev = nullptr, *h_ev = nullptr;  // per-job check results [17]
  SlabDev *d_slabs = nullptr;
  ColDev *d_cols = nullptr;
  uint64_t *d_prefix = nullptr;
  char *h_stage = nullptr;  // pinned staging for uploads
  size_t stage_size = 0, stage_used = 0;
  std::deque<Job *> waiting;
  std::vector<Job *> active;
  std::vector<Slab *> slabs;
  std::vector<int> free_slots;
  std::vector<hphi_job_result> done;
  int next_id = 0;
  double t0 = 0;
  size_t max_tiles = 0;
  double st_admit = 0, st_gpu = 0, st_check = 0;  // seconds spent per phase
  uint64_t st_ticks = 0, st_job_steps = 0, st_slab_steps = 0;
  // slab H·v launches: HIP-event time, algorithmic bytes, launches
  hipEvent_t ev_hv[2 * SL_SMAX] = {};
  double st_hv_s = 0, st_hv_bytes = 0;
  uint64_t st_hv_launches = 0;
  uint64_t st_moves = 0;  // columns moved between slabs (compact)
  int cls = -1;           // slabs by classes: -1 where it is the faster one, 0 none, 1 every one the layout fits
};

extern "C" double hphi_server_now(const hphi_server *s) { return s ? mono_now() - s->t0 : 0.0; }

extern "C" int hphi_server_create(const hphi_server_params *p, hphi_server **out) {
  if (!p || !out) return hphi_set_error("hphi_server_create: NULL argument");
  *out = nullptr;
  if (hphi_ensure_binom_table()) return -1;
  hphi_server *s = new hphi_server();
  s->p = *p;
  if (s->p.max_jobs <= 0) s->p.max_jobs = 64;
  if (s->p.max_jobs > 4096) s->p.max_jobs = 4096;
  if (s->p.n_eigen <= 0) s->p.n_eigen = 4;
  if (s->p.n_eigen > 16) s->p.n_eigen = 16;
  if (s->p.eps <= 0) s->p.eps = 1e-12;
  if (s->p.max_iter <= 0) s->p.max_iter = 2000;
  if (s->p.check_every <= 0) s->p.check_every = 5;
  const size_t budget = s->p.hbm_budget ? s->p.hbm_budget : ((size_t)16 << 30);
  s->max_tiles = (size_t)1 << 22;  // 4M tiles x 256 states = 1.07e9 states in flight
  int rc = 0;
  const int mj = s->p.max_jobs;
  if (hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking) != hipSuccess ||
      hipMalloc(&s->d_arena, budget) != hipSuccess ||
      hipMalloc(&s->d_js, sizeof(double) * JS_STRIDE * mj) != hipSuccess ||
      hipMalloc(&s->d_out, sizeof(double) * 2 * mj * SL_SMAX) != hipSuccess ||
      hipMalloc(&s->d_slabs, sizeof(SlabDev) * mj * SL_SMAX) != hipSuccess ||
      hipMalloc(&s->d_cols, sizeof(ColDev) * mj * SL_SMAX) != hipSuccess ||
      hipMalloc(&s->d_prefix, sizeof(uint64_t) * 2 * (mj + 1) * SL_SMAX) != hipSuccess ||
      hipMalloc(&s->d_part, sizeof(double2) * SL_K * (s->max_tiles + 8 * (size_t)mj)) != hipSuccess ||
      hipHostMalloc(&s->h_out, sizeof(double) * 2 * mj * SL_SMAX, hipHostMallocDefault) != hipSuccess ||
      hipMalloc(&s->d_ev, sizeof(double) * 17 * mj) != hipSuccess ||
      hipHostMalloc(&s->h_ev, sizeof(double) * 17 * mj, hipHostMallocDefault) != hipSuccess)
    rc = hphi_set_error("hphi_server_create: device allocation failed");
  s->stage_size = (size_t)16 << 20;
  if (!rc && hipHostMalloc(&s->h_stage, s->stage_size, hipHostMallocDefault) != hipSuccess)
    rc = hphi_set_error("hphi_server_create: pinned staging allocation failed");
  for (int i = 0; i < 2 * SL_SMAX && !rc; i++)
    if (hipEventCreate(&s->ev_hv[i]) != hipSuccess) rc = hphi_set_error("hphi_server_create: hipEventCreate failed");
  if (rc) {
    hphi_server_destroy(s);
    return -1;
  }
  s->arena.init(s->d_arena, budget);
  for (int i = mj - 1; i >= 0; i--) s->free_slots.push_back(i);
  s->t0 = mono_now();
  *out = s;
  return 0;
}

extern "C" void hphi_server_destroy(hphi_server *s) {
  if (!s) return;
  if (s->stream) (void)hipStreamSynchronize(s->stream);
  for (Job *j : s->active) delete j;
  for (Job *j : s->waiting) delete j;
  for (Slab *b : s->slabs) delete b;
  (void)hipFree(s->d_arena);
  (void)hipFree(s->d_js);
  (void)hipFree(s->d_out);
  (void)hipFree(s->d_slabs);
  (void)hipFree(s->d_cols);
  (void)hipFree(s->d_prefix);
  (void)hipFree(s->d_part);
  if (s->h_out) (void)hipHostFree(s->h_out);
  (void)hipFree(s->d_ev);
  if (s->h_ev) (void)hipHostFree(s->h_ev);
  if (s->h_stage) (void)hipHostFree(s->h_stage);
  for (int i = 0; i < 2 * SL_SMAX; i++)
    if (s->ev_hv[i]) (void)hipEventDestroy(s->ev_hv[i]);
  if (s->stream) (void)hipStreamDestroy(s->stream);
  delete s;
}

extern "C" int hphi_server_submit(hphi_server *s, const hphi_model_desc *d, uint64_t seed, double t_arrival,
                                  int *id) {
  if (!s || !d) return hphi_set_error("hphi_server_submit: NULL argument");
  if (d->model != HPHI_MODEL_SPIN && d->model != HPHI_MODEL_HUBBARD)
    return hphi_set_error("the service runs canonical Spin and Hubbard models");
  Job *j = new Job();
  if (hphi_engine_prepare(d, &j->h)) {
    delete j;
    return -1;
  }
  if (j->h.nbits > 32) {
    delete j;
    return hphi_set_error("the service runs states of at most 32 bits");
  }
  slab_repad(j->h);
  j->shash = structure_hash(j->h);
  for (const GTerm &t : j->h.h_terms_dev)
    if (t.cim != 0.0) j->realc = 0;
  j->cls = slab_cls(j->h, s->p.max_iter, s->arena.size, s->cls);
  const size_t fp = slab_footprint(j->h, s->p.max_iter, j->cls);
  if (fp > s->arena.size) {
    delete j;
    return hphi_set_error("job footprint %zu exceeds the HBM budget", fp);
  }
  j->id = s->next_id++;
  j->seed = seed;
  j->t_arrival = t_arrival;
  // the queue is ordered by arrival; among jobs that arrive together the
  // largest goes first, so the last jobs to run are small ones (1,000-request
  // stream back-to-back: 171.2 -> 172.6 solves/s)
  auto before = [](const Job *a, const Job *b) {
    return a->t_arrival < b->t_arrival || (a->t_arrival == b->t_arrival && a->h.dim > b->h.dim);
  };
  s->waiting.insert(std::upper_bound(s->waiting.begin(), s->waiting.end(), j, before), j);
  if (id) *id = j->id;
  return 0;
}

// copy into pinned staging (valid until the tick's synchronisation)
static void *stage(hphi_server *s, const void *src, size_t n) {
  if (s->stage_used + n > s->stage_size) return nullptr;
  char *p = s->h_stage + s->stage_used;
  memcpy(p, src, n);
  s->stage_used += al256(n);
  return p;
}

// list_2_1 as uint16 (rank + 2 < 2^16 for <= 16 low bits), zero-padded to n entries
__global__ void k_pack21(const uint32_t *l21, uint64_t size21, uint64_t n, uint16_t *out) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = i < size21 ? (uint16_t)l21[i] : (uint16_t)0;
}

// a new slab with the job's structure: tables on the device, terms uploaded;
// returns 1 when the staging buffer is full (retry next tick)
static int slab_create(hphi_server *s, const Job *j, size_t off, size_t bytes, Slab **out) {
  const hphi_engine &h = j->h;
  const size_t nt = std::max<size_t>(h.h_terms_dev.size(), 1), nd = std::max<size_t>(h.h_dterms.size(), 1);
  const size_t tb = sizeof(GTerm) * h.h_terms_dev.size();
  ClsArgs plan{};
  std::vector<char> up;
  const bool cls = j->cls && hphi_cls_plan(&h, plan, up);
  if (s->stage_used + al256(tb) + al256(up.size()) + al256(sizeof plan) > s->stage_size) return 1;
  Slab *b = new Slab();
  b->proto = h;
  b->nnz = hphi_term_nnz(&h);
  b->shash = j->shash;
  b->off = off;
  b->bytes = bytes;
  char *p = s->d_arena + off;
  b->list1 = (uint64_t *)p, p += al256(8 * h.dim);
  b->l21 = (uint32_t *)p, p += al256(4 * h.size21);
  b->l21p = (uint16_t *)p, p += al256(16 * ((h.size21 + 7) / 8));
  b->l22 = (uint64_t *)p, p += al256(8 * h.size22);
  b->jb = (uint64_t *)p, p += al256(8 * (h.sdim + 1));
  b->terms = (GTerm *)p, p += al256(sizeof(GTerm) * nt);
  b->coef = (double2 *)p, p += al256(16 * SL_K * nt);
  b->diag = (double *)p, p += al256(8 * SL_K * h.dim);
  b->R = (double2 *)p, p += al256(16 * SL_K * h.dim);
  b->Q = (double2 *)p, p += al256(16 * SL_K * h.dim);
  b->dterms = (DTerm *)p, p += al256(sizeof(DTerm) * SL_K * nd);
  b->hist = (double *)p, p += al256(8 * SL_K * 2 * (size_t)(s->p.max_iter + 2));
  b->coef_host.assign(SL_K * nt, make_double2(0.0, 0.0));
  int rc = 0;
  if (tb) {
    void *st = stage(s, h.h_terms_dev.data(), tb);
    if (hipMemcpyAsync(b->terms, st, tb, hipMemcpyHostToDevice, s->stream) != hipSuccess)
      rc = hphi_set_error("slab term upload failed");
  }
  const SzParams P = hphi_sz_params(&h);
  if (!rc && hphi_launch_tables(P, h.sdim, h.size21, b->jb, b->l21, b->l22, b->list1, s->stream)) rc = -1;
  if (!rc) {
    const uint64_t n = (h.size21 + 7) / 8 * 8;
    hipLaunchKernelGGL(k_pack21, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s->stream, b->l21, h.size21, n,
                       b->l21p);
    if (hipGetLastError() != hipSuccess) rc = hphi_set_error("slab table packing failed");
  }
  b->hv_chunks = (h.dim + (uint64_t)SL_TPW * SV_TPB - 1) / ((uint64_t)SL_TPW * SV_TPB);
  if (!rc && cls) {
    b->cls = plan;
    hphi_cls_units(b->cls, SC_B, SC_RPT);
    // SC_UPW units per wave, fewer while that leaves CUs idle; no more workgroups than by states
    const uint64_t w = (b->cls.units + SC_W - 1) / SC_W;
    b->hv_chunks = std::min<uint64_t>(b->hv_chunks, std::max<uint64_t>(w / SC_UPW, std::min<uint64_t>(w, 256)));
    b->d_cls = (ClsArgs *)p, p += al256(sizeof(ClsArgs));
    if (hphi_cls_upload(&h, b->cls, p, stage(s, up.data(), up.size()), b->l22, s->stream)) rc = -1;
    if (!rc && hipMemcpyAsync(b->d_cls, stage(s, &b->cls, sizeof plan), sizeof plan, hipMemcpyHostToDevice,
                              s->stream) != hipSuccess)
      rc = hphi_set_error("slab class layout upload failed");
  }
  if (rc) {
    delete b;
    return -1;
  }
  *out = b;
  return 0;
}

// the job takes column c of slab b: couplings, diagonal, start vector;
// returns 1 when the staging buffer is full (retry next tick)
static int column_start(hphi_server *s, Slab *b, int c, Job *j) {
  const hphi_engine &h = j->h;
  const size_t nt = h.h_terms_dev.size(), nd = h.h_dterms.size();
  const size_t cb = sizeof(double2) * b->coef_host.size(), db = sizeof(DTerm) * nd;
  if (s->stage_used + al256(cb) + al256(db) > s->stage_size) return 1;
  for (size_t t = 0; t < nt; t++)
    b->coef_host[t * SL_K + c] = make_double2(h.h_terms_dev[t].cre, h.h_terms_dev[t].cim);
  HIPCHK(hipMemcpyAsync(b->coef, stage(s, b->coef_host.data(), cb), cb, hipMemcpyHostToDevice, s->stream));
  DTerm *dt = b->dterms + (size_t)c * std::max<size_t>(nd, 1);
  if (db) HIPCHK(hipMemcpyAsync(dt, stage(s, h.h_dterms.data(), db), db, hipMemcpyHostToDevice, s->stream));
  if (hphi_launch_diag(h, b->list1, dt, b->diag, s->stream, SL_K, c)) return -1;
  const unsigned g = (unsigned)((h.dim + 255) / 256);
  hipLaunchKernelGGL(k_sl_start, dim3(g), dim3(256), 0, s->stream, b->R, b->Q, c, h.dim, j->seed, s->d_js, j->slot);
  HIPCHK(hipGetLastError());
  b->col[c] = j;
  j->slab = b;
  j->col = c;
  j->step = 0;
  j->alpha.assign(1, 0.0);
  j->beta.assign(1, 0.0);
  return 0;
}

// moves column cs of one slab into column cd of another slab of the same
// structure: the Lanczos vectors R and Q, the diagonal, the couplings and the
// alpha/beta history (nh doubles per column)
__global__ void k_sl_move(const double2 *R0, const double2 *Q0, const double *d0, const double2 *c0, const double *h0,
                          double2 *R1, double2 *Q1, double *d1, double2 *c1, double *h1, int cs, int cd,
                          uint64_t dim, uint64_t nt, uint64_t nh) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < dim) {
    R1[i * SL_K + cd] = R0[i * SL_K + cs];
    Q1[i * SL_K + cd] = Q0[i * SL_K + cs];
    d1[i * SL_K + cd] = d0[i * SL_K + cs];
  }
  if (i < nt) c1[i * SL_K + cd] = c0[i * SL_K + cs];
  if (i < nh) h1[(uint64_t)cd * nh + i] = h0[(uint64_t)cs * nh + i];
}

static void retire(hphi_server *s, Job *j, double now, int converged, const double *ev, int n) {
  j->res.id = j->id;
  j->res.iterations = j->step;
  j->res.converged = converged;
  j->res.n_found = n;
  for (int i = 0; i < n && i < 16; i++) j->res.eigenvalues[i] = ev[i];
  j->res.t_arrival = j->t_arrival;
  j->res.t_admit = j->t_admit;
  j->res.t_done = now;
  j->res.dim = j->h.dim;
  s->done.push_back(j->res);
  s->free_slots.push_back(j->slot);
  j->slab->col[j->col] = nullptr;
}

// admission in arrival order: a free column of a slab of the same structure,
// else a new slab while the arena has room
// The job takes column c of running slab b (slot and bookkeeping); 1: retry
// next tick (staging full)
static int admit_into(hphi_server *s, Job *j, Slab *b, int c, double now) {
  j->slot = s->free_slots.back();
  const int rc = column_start(s, b, c, j);
  if (rc) return rc;
  s->free_slots.pop_back();
  j->t_admit = now;
  s->active.push_back(j);
  return 0;
}

// Free columns of running slabs go first to arrived jobs of their structure
// among the first ADMIT_WINDOW waiting jobs, ahead of queue order: a slab step
// costs about the same however many of its columns run, so full slabs advance
// more jobs per launch.  The rest is admitted in arrival order (admit).
#define ADMIT_WINDOW 256
static int admit_fill(hphi_server *s, double now) {
  for (Slab *b : s->slabs) {
    while (b->used() < SL_K && !s->free_slots.empty()) {
      int c = -1;
      for (int q = SL_K - 1; q >= 0; q--)
        if (!b->col[q]) c = q;
      auto it = s->waiting.begin();
      int seen = 0;
      for (; it != s->waiting.end() && seen < ADMIT_WINDOW; ++it, ++seen) {
        const Job *w = *it;
        if (w->t_arrival <= now && w->shash == b->shash && same_structure(b->proto, w->h)) break;
      }
      if (it == s->waiting.end() || seen == ADMIT_WINDOW) break;
      Job *j = *it;
      const int rc = admit_into(s, j, b, c, now);
      if (rc == 1) return 0;
      if (rc) return -1;
      s->waiting.erase(it);
    }
  }
  return 0;
}

static int admit(hphi_server *s, double now) {
  if (admit_fill(s, now)) return -1;
  while (!s->waiting.empty() && !s->free_slots.empty()) {
    Job *j = s->waiting.front();
    if (j->t_arrival > now) break;
    Slab *b = nullptr;
    int c = -1;
    for (Slab *x : s->slabs) {
      if (x->used() == SL_K || x->shash != j->shash || !same_structure(x->proto, j->h)) continue;
      b = x;
      for (int q = SL_K - 1; q >= 0; q--)
        if (!x->col[q]) c = q;
      break;
    }
    bool fresh = false;
    if (!b) {
      const size_t bytes = slab_footprint(j->h, s->p.max_iter, j->cls);
      size_t off;
      if (!s->arena.alloc(bytes, &off)) break;
      const int rc = slab_create(s, j, off, bytes, &b);
      if (rc) {
        s->arena.release(off, bytes);
        if (rc == 1) break;
        return -1;
      }
      s->slabs.push_back(b);
      c = 0;
      fresh = true;
    }
    j->slot = s->free_slots.back();
    const int rc = column_start(s, b, c, j);
    if (rc) {
      if (fresh) {  // nothing was launched on the new slab's columns: release it
        s->slabs.pop_back();
        s->arena.release(b->off, b->bytes);
        delete b;
      }
      if (rc == 1) break;
      return -1;
    }
    s->free_slots.pop_back();
    s->waiting.pop_front();
    j->t_admit = now;
    s->active.push_back(j);
  }
  return 0;
}

// Slabs of one structure whose running columns fit in fewer slabs are packed:
// columns move from the emptiest slabs into the fullest ones with free
// columns, so a structure whose queue has drained runs ceil(columns / SL_K)
// slab steps per step instead of one per slab.  Structures with arrived
// waiting jobs are left alone (admission fills their free columns).  A moved
// column keeps its arithmetic (same tiles, same per-column reductions, and a
// real column computes the same values on the complex path), so its results do
// not change.
static int compact(hphi_server *s, double now) {
  std::vector<uint64_t> busy;  // structures with arrived waiting jobs in the admission window
  int seen = 0;
  for (const Job *w : s->waiting) {
    if (seen++ == ADMIT_WINDOW) break;
    if (w->t_arrival <= now) busy.push_back(w->shash);
  }
  std::map<uint64_t, std::vector<Slab *>> groups;
  for (Slab *b : s->slabs) {
    const int u = b->used();
    if (u > 0 && u < SL_K && std::find(busy.begin(), busy.end(), b->shash) == busy.end())
      groups[b->shash].push_back(b);
  }
  const uint64_t nh = 2 * ((uint64_t)s->p.max_iter + 2);
  for (auto &g : groups) {
    std::vector<Slab *> &L = g.second;
    int cols = 0;
    for (const Slab *b : L) cols += b->used();
    if ((size_t)((cols + SL_K - 1) / SL_K) >= L.size()) continue;  // no slab to free
    std::sort(L.begin(), L.end(), [](const Slab *a, const Slab *b) { return a->used() > b->used(); });
    size_t i = 0, k = L.size() - 1;
    while (i < k) {
      Slab *A = L[i], *B = L[k];
      if (A->used() == SL_K) { i++; continue; }
      if (B->used() == 0 || !same_structure(A->proto, B->proto)) { k--; continue; }
      int cs = 0, cd = 0;
      while (!B->col[cs]) cs++;
      while (A->col[cd]) cd++;
      const hphi_engine &h = A->proto;
      const uint64_t nt = h.h_terms_dev.size();
      const uint64_t n = std::max<uint64_t>(std::max<uint64_t>(h.dim, nt), nh);
      hipLaunchKernelGGL(k_sl_move, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s->stream, B->R, B->Q,
                         B->diag, B->coef, B->hist, A->R, A->Q, A->diag, A->coef, A->hist, cs, cd, h.dim, nt, nh);
      HIPCHK(hipGetLastError());
      for (uint64_t t = 0; t < nt; t++) A->coef_host[t * SL_K + cd] = B->coef_host[t * SL_K + cs];
      Job *j = B->col[cs];
      B->col[cs] = nullptr;
      A->col[cd] = j;
      j->slab = A;
      j->col = cd;
      s->st_moves++;
    }
  }
  return 0;
}

extern "C" int hphi_server_tick(hphi_server *s, int *n_active, int *n_waiting) {
  if (!s) return hphi_set_error("hphi_server_tick: NULL argument");
  double now = hphi_server_now(s);
  const double ta = now;
  s->stage_used = 0;
  if (admit(s, now)) return -1;
  s->st_admit += hphi_server_now(s) - ta;
  if (!s->active.empty()) {
    const double tg = hphi_server_now(s);
    // 2. S Lanczos steps for every running job, packed launches over the slabs
    const int S = std::min(s->p.check_every, SL_SMAX);
    const int n = (int)s->active.size();
    std::vector<int> nst(n);  // steps of each job this tick
    for (int i = 0; i < n; i++) {
      Job *j = s->active[i];
      const uint64_t lim = std::min<uint64_t>(j->h.dim, (uint64_t)s->p.max_iter);
      nst[i] = (int)std::min<uint64_t>((uint64_t)S, lim - (uint64_t)j->step);
      j->tick_steps = nst[i];
    }
    std::vector<int> s_chk(S, 0);  // jobs whose last step of the tick is step st
    for (int i = 0; i < n; i++) s_chk[nst[i] - 1]++;
    std::vector<SlabDev> sd;
    std::vector<ColDev> cd;
    std::vector<uint64_t> prefix;  // per step: tiles of pass 1 by slab, then workgroups of pass 2 by slab
    std::vector<int> s_nk(S), s_pv0(S);  // slabs with a class layout (the first ones); start of pass 2's prefix
    std::vector<int> s_ns(S), s_nc(S), s_sd0(S), s_cd0(S), s_pf0(S);
    // algorithmic bytes of each step's slab H·v: per slab 8 dim (list_1), per
    // running column 56 dim (own row, diagonal, Q read and write) + 16 per
    // off-diagonal element (the gathered row entry)
    std::vector<double> s_bytes(S, 0.0);
    std::map<const Slab *, int> index;
    const size_t hl = (size_t)s->p.max_iter + 2;
    uint64_t tiles = 0, max21 = 0, maxk21 = 0, maxla = 0, maxco = 0;
    std::vector<Slab *> order(s->slabs);
    std::stable_sort(order.begin(), order.end(), [](const Slab *a, const Slab *b) {  // the largest slabs start first
      return (a->d_cls != nullptr) > (b->d_cls != nullptr) ||
             ((a->d_cls != nullptr) == (b->d_cls != nullptr) && a->nnz > b->nnz);
    });
    std::vector<uint64_t> pv;
    for (int st = 0; st < S; st++) {
      s_sd0[st] = (int)sd.size();
      s_cd0[st] = (int)cd.size();
      s_pf0[st] = (int)prefix.size();
      prefix.push_back(0);
      pv.assign(1, 0);
      index.clear();
      for (Slab *b : order) {
        const hphi_engine &h = b->proto;
        SlabDev d{};
        for (int c = 0; c < SL_K; c++) {
          const Job *j = b->col[c];
          d.slot[c] = j ? j->slot : 0;
          if (j && j->tick_steps > st) {
            d.mask |= 1 << c;
            d.realc |= j->realc << c;
          }
        }
        if (!d.mask) continue;
        d.dim = h.dim;
        d.list1 = b->list1;
        d.l21p = (const uint4 *)b->l21p;
        d.l22 = b->l22;
        d.terms = b->terms;
        d.coef = b->coef;
        d.diag = b->diag;
        d.R = b->R;
        d.Q = b->Q;
        d.irght = h.irght;
        d.size21 = h.size21;
        d.n_low = h.n_low;
        d.n_high = h.n_high;
        d.n_mixed = h.n_mixed;
        d.nlow = h.nlow;
        d.cls = b->d_cls;
        d.sgn = h.model == HPHI_MODEL_HUBBARD;
        index[b] = (int)sd.size() - s_sd0[st];
        s_bytes[st] += 8.0 * (double)h.dim +
                       (double)__builtin_popcount(d.mask) * (56.0 * (double)h.dim + 16.0 * (double)b->nnz);
        sd.push_back(d);
        prefix.push_back(prefix.back() + (h.dim + (uint64_t)SL_TPW * SV_TPB - 1) / ((uint64_t)SL_TPW * SV_TPB));
        pv.push_back(pv.back() + (b->hv_chunks + 7) / 8 * 8);
        if (b->d_cls) {
          s_nk[st]++;
          maxk21 = std::max<uint64_t>(maxk21, h.size21);
          maxla = std::max<uint64_t>(maxla, (uint64_t)b->cls.nlo * SC_W * SC_RPT);
          maxco = std::max<uint64_t>(maxco, (uint64_t)(b->cls.n_low + b->cls.nt) * SL_K * 16);
        } else {
          max21 = std::max<uint64_t>(max21, h.size21);
        }
        std::swap(b->R, b->Q);  // roles after this step
      }
      for (int i = 0; i < n; i++) {
        if (nst[i] <= st) continue;
        Job *j = s->active[i];
        double *hb = j->slab->hist + (size_t)j->col * 2 * hl;
        cd.push_back(ColDev{index[j->slab], j->col, j->slot, j->step + st + 1, st == nst[i] - 1, i, hb, hb + hl});
      }
      s_ns[st] = (int)sd.size() - s_sd0[st];
      s_nc[st] = (int)cd.size() - s_cd0[st];
      tiles = std::max<uint64_t>(tiles, prefix.back());
      s_pv0[st] = (int)prefix.size();
      prefix.insert(prefix.end(), pv.begin(), pv.end());
    }
    if (tiles > s->max_tiles) return hphi_set_error("too many tiles in flight");
    const size_t lds = 16 * (size_t)((max21 + 7) / 8);  // list_2_1 as uint16 (rank + 2 < 2^16 for <= 16 low bits)
    const uint32_t n21 = (uint32_t)((maxk21 + 7) / 8), nla = (uint32_t)((maxla + 3) / 4 * 4);
    const size_t ldsk = 16 * (size_t)n21 + 4 * (size_t)nla + maxco;
    // one launch of pass 2, unless list_2_1 of a slab without class layout would
    // leave the others fewer workgroups per CU
    const size_t ldsm = std::max(lds, ldsk);
    const bool split = ldsm > SL_LDS;
    if (ldsm > 65536)
      (void)hipFuncSetAttribute((const void *)k_sl_hv, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ldsm);
    HIPCHK(hipMemcpyAsync(s->d_slabs, sd.data(), sizeof(SlabDev) * sd.size(), hipMemcpyHostToDevice, s->stream));
    HIPCHK(hipMemcpyAsync(s->d_cols, cd.data(), sizeof(ColDev) * cd.size(), hipMemcpyHostToDevice, s->stream));
    HIPCHK(hipMemcpyAsync(s->d_prefix, prefix.data(), sizeof(uint64_t) * prefix.size(), hipMemcpyHostToDevice,
                          s->stream));
    for (int st = 0; st < S; st++) {
      const int ns = s_ns[st], nc = s_nc[st];
      if (!nc) continue;
      const SlabDev *dsl = s->d_slabs + s_sd0[st];
      const ColDev *dcl = s->d_cols + s_cd0[st];
      const uint64_t *dpf = s->d_prefix + s_pf0[st];
      const unsigned T = (unsigned)((prefix[s_pf0[st] + ns] + 7) / 8 * 8);  // grid of sl_chunk()
      double *out = s->d_out + (size_t)st * 2 * n;
      hipLaunchKernelGGL(k_sl_resid, dim3(T), dim3(SV_TPB), 0, s->stream, dsl, dpf, ns, (const double *)s->d_js,
                         s->d_part);
      hipLaunchKernelGGL(k_sl_norm, dim3(nc), dim3(CS_TPB), 0, s->stream, dcl, dpf, (const double *)s->d_part,
                         s->d_js);
      HIPCHK(hipEventRecord(s->ev_hv[2 * st], s->stream));
      const uint64_t *dpv = s->d_prefix + s_pv0[st], *pvh = prefix.data() + s_pv0[st];
      const int nk = s_nk[st];
      for (int a = 0, b; a < ns; a = b) {  // slabs a .. b-1
        b = split && a < nk ? nk : ns;
        hipLaunchKernelGGL(k_sl_hv, dim3((unsigned)(pvh[b] - pvh[a])), dim3(SV_TPB), !split ? ldsm : a < nk ? ldsk : lds,
                           s->stream, dsl + a, dpv + a, b - a, (const double *)s->d_js, (double2 *)s->d_part, n21, nla);
      }
      HIPCHK(hipEventRecord(s->ev_hv[2 * st + 1], s->stream));
      hipLaunchKernelGGL(k_sl_alpha, dim3(nc), dim3(CS_TPB), 0, s->stream, dcl, dpv, (const double2 *)s->d_part,
                         s->d_js, out);
      if (s_chk[st]) hipLaunchKernelGGL(k_sl_check, dim3(nc), dim3(CK_TPB), 0, s->stream, dcl, s->p.n_eigen, s->d_ev);
      HIPCHK(hipGetLastError());
      s->st_slab_steps += ns;
    }
    HIPCHK(hipMemcpyAsync(s->h_out, s->d_out, sizeof(double) * 2 * n * S, hipMemcpyDeviceToHost, s->stream));
    HIPCHK(hipMemcpyAsync(s->h_ev, s->d_ev, sizeof(double) * 17 * n, hipMemcpyDeviceToHost, s->stream));
    HIPCHK(hipStreamSynchronize(s->stream));
    now = hphi_server_now(s);
    s->st_gpu += now - tg;
    for (int st = 0; st < S; st++) {
      if (!s_nc[st]) continue;
      float ms = 0.f;
      HIPCHK(hipEventElapsedTime(&ms, s->ev_hv[2 * st], s->ev_hv[2 * st + 1]));
      s->st_hv_s += 1e-3 * ms;
      s->st_hv_bytes += s_bytes[st];
      s->st_hv_launches++;
    }
    s->st_ticks++;
    // 3. convergence and retirement
    std::vector<Job *> keep;
    keep.reserve(n);
    for (int i = 0; i < n; i++) {
      Job *j = s->active[i];
      s->st_job_steps += nst[i];
      bool broken = false;
      for (int st = 0; st < nst[i]; st++) {
        const double *o = s->h_out + ((size_t)st * n + i) * 2;
        const int m = j->step + 1;
        j->alpha.push_back(o[0]);                  // alpha[m]
        if (m >= 2) j->beta.push_back(o[1]);      // beta[m-1]
        j->step = m;
        // beta[m-1] ~ 0: the recurrence ended at step m-1 (alpha[m] and later are void)
        if (m >= 2 && j->beta[m - 1] < 1e-14) {
          broken = true;
          j->step = m - 1;
          break;
        }
      }
      const int m = j->step;
      const bool exhausted = broken || (uint64_t)m >= j->h.dim;
      double cur[16];
      int nc;
      if (broken) {
        nc = hphi_lanczos_good_eigenvalues(j->alpha.data() + 1, j->beta.data() + 1, m, s->p.n_eigen, cur);
      } else {  // the check after the job's last step of the tick ran on the device
        const double *o = s->h_ev + 17 * (size_t)i;
        nc = (int)o[16];
        for (int q = 0; q < nc; q++) cur[q] = o[q];
        // the device window stops at CK_LMAX values of T_m; with more ghost copies
        // than that below the wanted values the host filter widens it up to m
        if (nc < (int)std::min<uint64_t>((uint64_t)s->p.n_eigen, j->h.dim) && m > CK_LMAX)
          nc = hphi_lanczos_good_eigenvalues(j->alpha.data() + 1, j->beta.data() + 1, m, s->p.n_eigen, cur);
      }
      const int want = (int)std::min<uint64_t>((uint64_t)s->p.n_eigen, j->h.dim);
      // converged: the values stopped moving and their Ritz residuals are small
      // (T_{m-1} with beta_{m-1}: beta_m comes with the next step)
      bool conv = (exhausted && nc >= 1);
      if (!conv && hphi_lanczos_converged(j->prev, j->nprev, cur, nc, want, s->p.eps))
        conv = m < 2 || hphi_lanczos_residuals_small(j->alpha.data() + 1, j->beta.data() + 1, m - 1, j->beta[m - 1],
                                                     cur, want, s->p.eps);
      if (conv || m >= s->p.max_iter) {
        retire(s, j, now, conv ? 1 : 0, cur, nc);
        delete j;
        continue;
      }
      memcpy(j->prev, cur, sizeof cur);
      j->nprev = nc;
      keep.push_back(j);
    }
    s->active.swap(keep);
    if (compact(s, now)) return -1;
    // slabs whose last job left give their memory back
    std::vector<Slab *> live;
    for (Slab *b : s->slabs) {
      if (b->used()) {
        live.push_back(b);
      } else {
        s->arena.release(b->off, b->bytes);
        delete b;
      }
    }
    s->slabs.swap(live);
    s->st_check += hphi_server_now(s) - now;
  }
  if (n_active) *n_active = (int)s->active.size();
  if (n_waiting) *n_waiting = (int)s->waiting.size();
  return 0;
}

extern "C" int hphi_server_tune(hphi_server *s, const char *knob, int value) {
  if (!s || !knob) return hphi_set_error("hphi_server_tune: NULL argument");
  if (strcmp(knob, "cls")) return hphi_set_error("unknown tuning knob %s", knob);
  if (value < -1 || value > 1) return hphi_set_error("cls must be -1, 0 or 1");
  s->cls = value;
  return 0;
}

extern "C" int hphi_server_stats(const hphi_server *s, double *out) {
  if (!s || !out) return hphi_set_error("hphi_server_stats: NULL argument");
  out[0] = s->st_admit;
  out[1] = s->st_gpu;
  out[2] = s->st_check;
  out[3] = (double)s->st_ticks;
  out[4] = (double)s->st_job_steps;
  out[5] = (double)s->st_slab_steps;
  out[6] = s->st_hv_s;
  out[7] = s->st_hv_bytes;
  out[8] = (double)s->st_hv_launches;
  out[9] = (double)s->st_moves;
  return 0;
}

extern "C" int hphi_server_results(hphi_server *s, hphi_job_result *out, int max, int *n) {
  if (!s || !n) return hphi_set_error("hphi_server_results: NULL argument");
  const int k = (int)std::min<size_t>(s->done.size(), (size_t)std::max(max, 0));
  for (int i = 0; i < k; i++) out[i] = s->done[i];
  s->done.erase(s->done.begin(), s->done.begin() + k);
  *n = k;
  return 0;
}
