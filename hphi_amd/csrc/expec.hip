// Expectation values of a device vector v (normalised by the caller):
//
//   hphi_expec_energy_flct   <- expec_energy_flct (src/expec_energy_flct.c:40-160,186-660):
//                               <v|H|v>, <Hv|Hv> and the doublon / electron-number / Sz moments
//   hphi_expec_cisajs        <- expec_cisajs (src/expec_cisajs.c:69-650): <v|c+_{i s1} c_{j s2}|v>
//   hphi_expec_cisajscktalt  <- expec_cisajscktaltdc (src/expec_cisajscktaltdc.c:87-1647):
//                               <v|c+_{i s1} c_{j s2} c+_{k s3} c_{l s4}|v>
//
// Every Green's function entry is compiled on the host into gather terms (the
// same forms the Hamiltonian uses).  A term without its factor is an item; terms
// of several entries that agree share one (densities and exchanges of (i, k) and
// (k, i)).  One workgroup evaluates EX_CW items: lane j holds target state x = list_1[j]
// (or j) and adds sign * conj(v[j]) * v[idx(x ^ flip)] of each item that acts,
// <v|O|v> = sum_x conj(v_x) (O v)_x; an entry is the sum of factor times item.
// Reductions run in a fixed order (waves, then blocks), so results are
// reproducible run to run.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <utility>
#include <vector>

#include "engine_internal.h"

#define EX_TPB 256
#define EX_GRID 512
#define EX_CW 8  // items per workgroup

namespace {

template <typename W>
struct CorrTerm {
  W flip, tmask, tval, sgn;
};

__device__ __forceinline__ double wave_sum(double s) {
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  return s;
}

// per state: w = |v_j|^2; kind 1 (SpinGC): S = 2 popcount(x) - N;
// kind 2 (Hubbard models): D doublons, N electrons, S = N_up - N_down
__global__ __launch_bounds__(EX_TPB) void k_moments(const double2 *v, const uint64_t *list1, uint64_t dim, int kind,
                                                     int nsite, double *partial) {
  double r[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  const uint64_t EVEN = 0x5555555555555555ull;
  for (uint64_t j = (uint64_t)blockIdx.x * EX_TPB + threadIdx.x; j < dim; j += (uint64_t)gridDim.x * EX_TPB) {
    const double2 a = v[j];
    const double w = a.x * a.x + a.y * a.y;
    const uint64_t x = list1 ? list1[j] : j;
    if (kind == 1) {
      const double S = (double)(2 * (int)__popcll(x) - nsite);
      r[4] += w * S;
      r[5] += w * S * S;
    } else {
      const double D = (double)(int)__popcll(x & (x >> 1) & EVEN);
      const int up = (int)__popcll(x & EVEN), dn = (int)__popcll(x & (EVEN << 1));
      const double N = (double)(up + dn), S = (double)(up - dn);
      r[0] += w * D;
      r[1] += w * D * D;
      r[2] += w * N;
      r[3] += w * N * N;
      r[4] += w * S;
      r[5] += w * S * S;
    }
  }
  __shared__ double sh[EX_TPB / 64][6];
#pragma unroll
  for (int q = 0; q < 6; q++) {
    const double s = wave_sum(r[q]);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][q] = s;
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    double s = 0.0;
    for (int w = 0; w < EX_TPB / 64; w++) s += sh[w][threadIdx.x];
    partial[(uint64_t)blockIdx.x * 6 + threadIdx.x] = s;
  }
}

__device__ __forceinline__ uint32_t ex_popc(uint32_t x) { return (uint32_t)__popc(x); }
__device__ __forceinline__ uint32_t ex_popc(uint64_t x) { return (uint32_t)__popcll(x); }

// One state against EX_CW items.  PROJ: items without flip and sign, |v_j|^2 alone.
template <typename W, bool CANON, bool PROJ>
__device__ __forceinline__ void corr_state(const double2 *v, const uint32_t *l21, const uint64_t *l22, uint64_t dim,
                                           W irght, int nlow, const CorrTerm<W> (&T)[EX_CW], W x, double2 a,
                                           double (&ar)[EX_CW], double (&ai)[EX_CW]) {
  if (PROJ) {
    const double w = a.x * a.x + a.y * a.y;
#pragma unroll
    for (int q = 0; q < EX_CW; q++)
      if ((x & T[q].tmask) == T[q].tval) ar[q] += w;
    return;
  }
  bool act[EX_CW];
  uint64_t idx[EX_CW];
#pragma unroll
  for (int q = 0; q < EX_CW; q++) {
    act[q] = (x & T[q].tmask) == T[q].tval;
    idx[q] = (uint64_t)(x ^ T[q].flip);
  }
  if (CANON) {  // rank tables, 0 = not in the sector
    uint32_t la[EX_CW];
    uint64_t lb[EX_CW];
#pragma unroll
    for (int q = 0; q < EX_CW; q++) {
      la[q] = 0;
      lb[q] = 0;
      if (act[q]) {
        la[q] = l21[(W)idx[q] & irght];
        lb[q] = l22[(W)idx[q] >> nlow];
      }
    }
#pragma unroll
    for (int q = 0; q < EX_CW; q++) {
      idx[q] = la[q] + lb[q] - 3;
      act[q] = la[q] != 0 && lb[q] != 0;
    }
  }
  double2 u[EX_CW];
#pragma unroll
  for (int q = 0; q < EX_CW; q++) {
    act[q] = act[q] && idx[q] < dim;
    u[q] = make_double2(0.0, 0.0);
    if (act[q]) u[q] = v[idx[q]];
  }
#pragma unroll
  for (int q = 0; q < EX_CW; q++) {
    if (!act[q]) continue;
    const bool neg = ex_popc((W)(x & T[q].sgn)) & 1u;
    const double ux = neg ? -u[q].x : u[q].x, uy = neg ? -u[q].y : u[q].y;
    ar[q] += a.x * ux + a.y * uy;
    ai[q] += a.x * uy - a.y * ux;
  }
}

// block (bx, c): items c*EX_CW .. c*EX_CW+EX_CW-1, the first np chunks projectors.
// Their masks stay in scalar registers over all the workgroup's states, eight
// items' table lookups and gathers are in flight together, and the grid gives
// each lane several states, so that the sums over the workgroup cost little.
// (One slot after another per state, one state per lane, 64-bit: 1,330 us for the 2,360
// entries of a 20-site chain; now 135, with 1,180 items left of them.)
template <typename W, bool CANON>
__global__ __launch_bounds__(EX_TPB) void k_corr(const double2 *v, const uint64_t *list1, const uint32_t *l21,
                                                 const uint64_t *l22, uint64_t dim, W irght, int nlow,
                                                 const CorrTerm<W> *terms, int np, double2 *partial) {
  typedef const CorrTerm<W> __attribute__((address_space(4))) *CT;
  CorrTerm<W> T[EX_CW];
  const CT t = (CT)terms + (size_t)blockIdx.y * EX_CW;
#pragma unroll
  for (int q = 0; q < EX_CW; q++) {
    T[q].flip = t[q].flip;
    T[q].tmask = t[q].tmask;
    T[q].tval = t[q].tval;
    T[q].sgn = t[q].sgn;
  }
  double ar[EX_CW], ai[EX_CW];
#pragma unroll
  for (int q = 0; q < EX_CW; q++) ar[q] = ai[q] = 0.0;
  const uint64_t j0 = (uint64_t)blockIdx.x * EX_TPB + threadIdx.x, dj = (uint64_t)gridDim.x * EX_TPB;
  if ((int)blockIdx.y < np) {
    for (uint64_t j = j0; j < dim; j += dj)
      corr_state<W, CANON, true>(v, l21, l22, dim, irght, nlow, T, CANON ? (W)list1[j] : (W)j, v[j], ar, ai);
  } else {
    for (uint64_t j = j0; j < dim; j += dj)
      corr_state<W, CANON, false>(v, l21, l22, dim, irght, nlow, T, CANON ? (W)list1[j] : (W)j, v[j], ar, ai);
  }
  __shared__ double sh[EX_TPB / 64][EX_CW][2];
#pragma unroll
  for (int q = 0; q < EX_CW; q++) {
    const double sr = wave_sum(ar[q]), si = wave_sum(ai[q]);
    if ((threadIdx.x & 63) == 0) {
      sh[threadIdx.x >> 6][q][0] = sr;
      sh[threadIdx.x >> 6][q][1] = si;
    }
  }
  __syncthreads();
  if (threadIdx.x < EX_CW) {
    double sr = 0.0, si = 0.0;
    for (int w = 0; w < EX_TPB / 64; w++) {
      sr += sh[w][threadIdx.x][0];
      si += sh[w][threadIdx.x][1];
    }
    partial[((uint64_t)blockIdx.y * gridDim.x + blockIdx.x) * EX_CW + threadIdx.x] = make_double2(sr, si);
  }
}

// item s: sum over the blocks of its chunk, a wave per item (one thread took 128 us)
__global__ __launch_bounds__(EX_TPB) void k_corr_final(const double2 *partial, int nblk, int n, double2 *out) {
  const int s = blockIdx.x * (EX_TPB / 64) + (threadIdx.x >> 6);
  if (s >= n) return;
  const int c = s / EX_CW, q = s % EX_CW;
  double sr = 0.0, si = 0.0;
  for (int b = threadIdx.x & 63; b < nblk; b += 64) {
    const double2 p = partial[((uint64_t)c * nblk + b) * EX_CW + q];
    sr += p.x;
    si += p.y;
  }
  sr = wave_sum(sr);
  si = wave_sum(si);
  if ((threadIdx.x & 63) == 0) out[s] = make_double2(sr, si);
}

int ex_grid(uint64_t dim) {
  uint64_t g = (dim + EX_TPB - 1) / EX_TPB;
  return (int)(g < EX_GRID ? (g ? g : 1) : EX_GRID);
}

// density-like projector: target (and source) has (x & mask) == val
void push_proj(std::vector<GTerm> &out, uint64_t mask, uint64_t val) {
  GTerm g{};
  g.kind = P_EQ;
  g.tmask = mask;
  g.tval = val;
  g.cre = 1.0;
  out.push_back(g);
}

// Items of the compiled slots: distinct terms without their factors, projectors
// first, both kinds padded to EX_CW with items that never act.
struct Items {
  std::vector<CorrTerm<uint64_t>> t;
  std::vector<int> of;  // item of every term, slot after slot
  size_t nproj = 0;     // projectors with their padding
  explicit Items(const std::vector<std::vector<GTerm>> &slots) {
    size_t n = 0, cap = 64;
    for (const auto &sl : slots) n += sl.size();
    while (cap < 2 * n) cap *= 2;
    std::vector<int> table(cap, -1), kind[2];
    std::vector<CorrTerm<uint64_t>> uniq;
    of.reserve(n);
    for (const auto &sl : slots)
      for (const GTerm &g : sl) {
        uint64_t h = (g.flip * 0x9E3779B97F4A7C15ull) ^ (g.tmask * 0xBF58476D1CE4E5B9ull) ^
                     (g.tval * 0x94D049BB133111EBull) ^ (g.sgn * 0xD6E8FEB86659FD93ull);
        h ^= h >> 31;
        for (;; h++) {
          int &k = table[h & (cap - 1)];
          if (k < 0) {
            k = (int)uniq.size();
            uniq.push_back(CorrTerm<uint64_t>{g.flip, g.tmask, g.tval, g.sgn});
            kind[g.flip || g.sgn ? 1 : 0].push_back(k);
          }
          const CorrTerm<uint64_t> &u = uniq[k];
          if (u.flip == g.flip && u.tmask == g.tmask && u.tval == g.tval && u.sgn == g.sgn) {
            of.push_back(k);
            break;
          }
        }
      }
    std::vector<int> at(uniq.size());
    for (int c = 0; c < 2; c++) {
      for (int k : kind[c]) {
        at[k] = (int)t.size();
        t.push_back(uniq[k]);
      }
      while (t.size() % EX_CW) t.push_back(CorrTerm<uint64_t>{0, 0, 1, 0});
      if (c == 0) nproj = t.size();
    }
    for (int &k : of) k = at[k];
  }
};

template <typename W, bool CANON>
int corr_launch(hphi_engine *e, const double2 *v, const CorrTerm<W> *terms, int g, int nchunk, int np, double2 *part) {
  for (int c0 = 0; c0 < nchunk; c0 += 65535) {  // grid.y limit
    const int nc = nchunk - c0 < 65535 ? nchunk - c0 : 65535;
    hipLaunchKernelGGL((k_corr<W, CANON>), dim3(g, nc), dim3(EX_TPB), 0, e->stream, v, e->d_list1, e->d_l21, e->d_l22,
                       e->dim, (W)e->irght, e->nlow, terms + (size_t)c0 * EX_CW, np - c0,
                       part + (size_t)c0 * g * EX_CW);
    if (hipGetLastError() != hipSuccess) return hphi_set_error("hphi_expec: k_corr launch failed");
  }
  return 0;
}

// evaluate the compiled slots on v; out[2*s], out[2*s+1] = re, im
int run_corr(hphi_engine *e, const double *v, const std::vector<std::vector<GTerm>> &slots, double *out) {
  const int nslot = (int)slots.size();
  if (nslot == 0) return 0;
  if (hphi_build_tables(e)) return -1;
  const Items I(slots);
  std::vector<double> val(2 * I.t.size());
  if (!I.t.empty()) {
    const int n = (int)I.t.size(), nchunk = n / EX_CW, np = (int)(I.nproj / EX_CW);
    // some 16 workgroups per CU over all chunks, and up to EX_GRID for one
    int g = ex_grid(e->dim);
    g = std::max(1, std::min(g, (16 * std::max(e->num_cu, 1) + nchunk - 1) / nchunk));
    const bool narrow = e->nbits <= 32, gc = hphi_model_gc(e->model);
    std::vector<CorrTerm<uint32_t>> t32;
    const void *src = I.t.data();
    size_t tb = sizeof(I.t[0]) * n;
    if (narrow) {
      for (const auto &t : I.t)
        t32.push_back(CorrTerm<uint32_t>{(uint32_t)t.flip, (uint32_t)t.tmask, (uint32_t)t.tval, (uint32_t)t.sgn});
      src = t32.data();
      tb = sizeof(t32[0]) * n;
    }
    const size_t at = (tb + 255) / 256 * 256, ao = at + sizeof(double2) * (size_t)nchunk * g * EX_CW;
    char *d = nullptr;
    if (hphi_dev_alloc(ao + sizeof(double2) * n, (void **)&d)) return -1;
    double2 *part = (double2 *)(d + at), *res = (double2 *)(d + ao);
    const double2 *vv = (const double2 *)v;
    int rc = -1;
    if (hipMemcpyAsync(d, src, tb, hipMemcpyHostToDevice, e->stream) != hipSuccess)
      hphi_set_error("hphi_expec: term upload failed");
    else if (narrow)
      rc = gc ? corr_launch<uint32_t, false>(e, vv, (const CorrTerm<uint32_t> *)d, g, nchunk, np, part)
              : corr_launch<uint32_t, true>(e, vv, (const CorrTerm<uint32_t> *)d, g, nchunk, np, part);
    else
      rc = gc ? corr_launch<uint64_t, false>(e, vv, (const CorrTerm<uint64_t> *)d, g, nchunk, np, part)
              : corr_launch<uint64_t, true>(e, vv, (const CorrTerm<uint64_t> *)d, g, nchunk, np, part);
    if (!rc) {
      hipLaunchKernelGGL(k_corr_final, dim3((n + EX_TPB / 64 - 1) / (EX_TPB / 64)), dim3(EX_TPB), 0, e->stream,
                         (const double2 *)part, g, n, res);
      if (hipGetLastError() != hipSuccess ||
          hipMemcpyAsync(val.data(), res, sizeof(double2) * n, hipMemcpyDeviceToHost, e->stream) != hipSuccess)
        rc = hphi_set_error("hphi_expec: correlator pass failed");
    }
    if (hipStreamSynchronize(e->stream) != hipSuccess) rc = hphi_set_error("hphi_expec: correlator pass failed");
    hphi_dev_free(d);
    if (rc) return -1;
  }
  size_t k = 0;
  for (int s = 0; s < nslot; s++) {
    double re = 0.0, im = 0.0;
    for (const GTerm &g : slots[s]) {
      const double *p = &val[2 * I.of[k++]];
      re += g.cre * p[0] - g.cim * p[1];
      im += g.cre * p[1] + g.cim * p[0];
    }
    out[2 * s] = re;
    out[2 * s + 1] = im;
  }
  return 0;
}

}  // namespace

extern "C" int hphi_expec_energy_flct(hphi_engine *e, const double *v, hphi_phys *out) {
  if (!e || !v || !out) return hphi_set_error("hphi_expec_energy_flct: NULL argument");
  memset(out, 0, sizeof *out);
  if (hphi_build_tables(e)) return -1;
  // moments (expec_energy_flct_HalfSpinGC / _Hubbard / _HubbardGC)
  const int kind = e->model == HPHI_MODEL_SPINGC ? 1 : hphi_model_hubbard(e->model) ? 2 : 0;
  if (kind) {
    const int g = ex_grid(e->dim);
    double *d_part = nullptr;
    std::vector<double> part((size_t)g * 6);
    if (hphi_dev_alloc(sizeof(double) * part.size(), (void **)&d_part)) return -1;
    hipLaunchKernelGGL(k_moments, dim3(g), dim3(EX_TPB), 0, e->stream, (const double2 *)v,
                       hphi_model_gc(e->model) ? (const uint64_t *)nullptr : e->d_list1, e->dim, kind, e->nsite,
                       d_part);
    const bool ok = hipGetLastError() == hipSuccess &&
                    hipMemcpyAsync(part.data(), d_part, sizeof(double) * part.size(), hipMemcpyDeviceToHost,
                                   e->stream) == hipSuccess &&
                    hipStreamSynchronize(e->stream) == hipSuccess;
    hphi_dev_free(d_part);
    if (!ok) return hphi_set_error("hphi_expec_energy_flct: moment pass failed");
    double m[6] = {0, 0, 0, 0, 0, 0};
    for (int b = 0; b < g; b++)
      for (int q = 0; q < 6; q++) m[q] += part[(size_t)b * 6 + q];
    if (kind == 1) {  // expec_energy_flct.c:484-491
      out->num = e->nsite;
      out->num2 = (double)e->nsite * e->nsite;
    } else {  // :290-297, :414-421
      out->doublon = m[0];
      out->doublon2 = m[1];
      out->num = m[2];
      out->num2 = m[3];
    }
    out->sz = 0.5 * m[4];
    out->sz2 = 0.25 * m[5];
  } else {  // canonical Spin: constants (expec_energy_flct.c:104-118)
    const double sz = 0.5 * (double)(e->nup - e->ndown);
    out->num = e->nsite;
    out->num2 = (double)e->nsite * e->nsite;
    out->sz = sz;
    out->sz2 = sz * sz;
  }
  // energy <v|H|v> (the H·v's prdct) and variance <Hv|Hv> (:141-158)
  double *hv = nullptr, pr[2], n2;
  if (hphi_dev_alloc(16 * e->dim, (void **)&hv)) return -1;
  int rc = -1;
  if (!hphi_dev_zero(hv, 16 * e->dim) && !hphi_mltply_dev(e, hv, v, pr) && !hphi_vec_norm2(e, hv, 1, &n2)) {
    out->energy = pr[0];
    out->var = n2;
    rc = 0;
  }
  hphi_dev_free(hv);
  return rc;
}

extern "C" int hphi_expec_cisajs(hphi_engine *e, const double *v, int n, const int *idx, double *out) {
  if (!e || !v || (n > 0 && (!idx || !out))) return hphi_set_error("hphi_expec_cisajs: NULL argument");
  const int N = e->nsite;
  const bool hub = hphi_model_hubbard(e->model), gc = hphi_model_gc(e->model);
  std::vector<std::vector<GTerm>> slots(n);
  for (int t = 0; t < n; t++) {
    const int i = idx[4 * t], s1 = idx[4 * t + 1], j = idx[4 * t + 2], s2 = idx[4 * t + 3];
    if (i < 0 || j < 0 || i >= N || j >= N || s1 < 0 || s1 > 1 || s2 < 0 || s2 > 1)
      return hphi_set_error("OneBodyG entry %d (%d %d %d %d) out of range", t, i, s1, j, s2);
    std::vector<GTerm> &sl = slots[t];
    if (hub) {
      if (!gc && s1 != s2) continue;  // Sz-conserving sector (expec_cisajs.c:276-282)
      const int a = 2 * i + s1, b = 2 * j + s2;
      if (a == b) {  // n_a (:330-338)
        push_proj(sl, 1ull << a, 1ull << a);
      } else {  // c+_a c_b with its Jordan-Wigner sign (general_hopp / GC_general_hopp)
        GTerm g{};
        g.kind = P_EQ;
        g.flip = (1ull << a) | (1ull << b);
        g.tmask = g.flip;
        g.tval = 1ull << a;
        g.sgn = hphi_between_mask(a, b);
        g.cre = 1.0;
        sl.push_back(g);
      }
    } else {
      if (i != j) continue;  // no hopping between localized spins (:406-408, :571-574)
      if (s1 == s2) {        // [bit_i == s1] (:389-403, :546-552)
        push_proj(sl, 1ull << i, s1 ? 1ull << i : 0ull);
      } else if (gc) {  // transverse: target bit s1, source bit s2 (:553-566)
        GTerm g{};
        g.kind = P_EQ;
        g.flip = 1ull << i;
        g.tmask = g.flip;
        g.tval = s1 ? g.flip : 0ull;
        g.cre = 1.0;
        sl.push_back(g);
      }  // canonical Spin: s1 != s2 changes Sz, 0 (:409-412)
    }
  }
  return run_corr(e, v, slots, out);
}

extern "C" int hphi_expec_cisajscktalt(hphi_engine *e, const double *v, int n, const int *idx, double *out) {
  if (!e || !v || (n > 0 && (!idx || !out))) return hphi_set_error("hphi_expec_cisajscktalt: NULL argument");
  const int N = e->nsite;
  const bool hub = hphi_model_hubbard(e->model), gc = hphi_model_gc(e->model);
  std::vector<std::vector<GTerm>> slots(n);
  for (int t = 0; t < n; t++) {
    const int *q = idx + 8 * t;
    for (int u = 0; u < 8; u += 2)
      if (q[u] < 0 || q[u] >= N || q[u + 1] < 0 || q[u + 1] > 1)
        return hphi_set_error("TwoBodyG entry %d out of range", t);
    std::vector<GTerm> &sl = slots[t];
    if (hub) {
      if (!gc && q[1] + q[5] != q[3] + q[7]) continue;  // expec_cisajscktaltdc.c:535-541
      hphi_compile_two_hops(2 * q[0] + q[1], 2 * q[2] + q[3], 2 * q[4] + q[5], 2 * q[6] + q[7], 1.0, 0.0, sl);
      continue;
    }
    // spin entries are (i s1 i s2 k s3 k s4) (readdef.c:1497-1503); the pair
    // with the smaller site comes first (Rearray_Interactions, :274-381)
    if (q[0] != q[2] || q[4] != q[6])
      return hphi_set_error("spin TwoBodyG entry %d needs i == j and k == l", t);
    int A = q[0], s1 = q[1], s2 = q[3], B = q[4], s3 = q[5], s4 = q[7];
    if (A > B) {
      std::swap(A, B);
      std::swap(s1, s3);
      std::swap(s2, s4);
    }
    if (!gc) {  // canonical branches (:736-772): diagonal, one-site, exchange; others 0
      const bool keep = (s1 == s2 && s3 == s4) || (A == B && s1 == s4 && s3 == s2) || (s1 == s4 && s2 == s3);
      if (!keep) continue;
    }
    hphi_compile_spin_pair(A, s1, s2, B, s3, s4, 1.0, 0.0, sl);
  }
  return run_corr(e, v, slots, out);
}

// SpinGC three-, four- and six-body Green's functions
// (expec_Threebody_SpinGCHalf / expec_Fourbody_SpinGCHalf /
// expec_Sixbody_SpinGCHalf, src/expec_cisajscktaltdc.c:901-1420).  An entry
// holds nbody pairs (site, sigma)(site, sigma); pair p is O_p = |s><s'| on its
// site when both sites agree.  The value is <v| O_1 O_2 O_3 ... O_nbody |v>:
//  * pairs 3 .. nbody are applied to v right to left (mltplyHalfSpinGC_mini,
//    src/mltplySpin.c:416-490); one on two different sites leaves zero;
//  * the first two follow Rearray_Interactions (:274-381): (i,i)(k,k) as given,
//    the cross form (i,k)(k,i) as -|s1><s4|_i |s3><s2|_k; any other first two
//    pairs are not evaluated (ok = 0; the reference prints the first eight
//    indices and zeros).
// The product of on-site projectors and flips is one gather term: per site the
// composed operator |a><b| (|a><b| after |c><d| is delta(b, c) |a><d|), the
// target x has bits a, the source is x with bits b.
extern "C" int hphi_expec_spin_nbody(hphi_engine *e, const double *v, int nbody, int n, const int *idx, double *out,
                                     int *ok) {
  if (!e || !v || (n > 0 && (!idx || !out || !ok))) return hphi_set_error("hphi_expec_spin_nbody: NULL argument");
  if (nbody != 3 && nbody != 4 && nbody != 6) return hphi_set_error("hphi_expec_spin_nbody: nbody must be 3, 4 or 6");
  if (e->model != HPHI_MODEL_SPINGC)
    return hphi_set_error("hphi_expec_spin_nbody: the reference defines these for SpinGC (spin 1/2) only");
  const int N = e->nsite;
  std::vector<std::vector<GTerm>> slots(n);
  for (int t = 0; t < n; t++) {
    const int *q = idx + 4 * nbody * t;
    for (int u = 0; u < 4 * nbody; u += 2)
      if (q[u] < 0 || q[u] >= N || q[u + 1] < 0 || q[u + 1] > 1)
        return hphi_set_error("%d-body Green's function entry %d out of range", nbody, t);
    ok[t] = 1;
    // the first two pairs after Rearray_Interactions: (site, s, s') x 2 and the sign
    int A, a1, a2, B, b1, b2;
    double sign = 1.0;
    if (q[0] == q[2] && q[4] == q[6]) {
      A = q[0], a1 = q[1], a2 = q[3], B = q[4], b1 = q[5], b2 = q[7];
    } else if (q[0] == q[6] && q[4] == q[2]) {
      A = q[0], a1 = q[1], a2 = q[7], B = q[4], b1 = q[5], b2 = q[3];
      sign = -1.0;
    } else {
      ok[t] = 0;
      continue;
    }
    if (A > B) {  // the pair with the smaller site first
      std::swap(A, B);
      std::swap(a1, b1);
      std::swap(a2, b2);
    }
    // compose, in the order the operators act on the ket
    int ca[64], cb[64];
    for (int s = 0; s < N; s++) ca[s] = cb[s] = -1;
    bool zero = false;
    auto apply = [&](int site, int s_to, int s_from) {
      if (ca[site] < 0) {
        ca[site] = s_to;
        cb[site] = s_from;
      } else if (s_from == ca[site]) {
        ca[site] = s_to;
      } else {
        zero = true;
      }
    };
    for (int p = nbody - 1; p >= 2 && !zero; p--) {
      const int *r = q + 4 * p;
      if (r[0] != r[2]) zero = true;  // mltplyHalfSpinGC_mini adds nothing for two sites
      else apply(r[0], r[1], r[3]);
    }
    if (!zero) apply(B, b1, b2);
    if (!zero) apply(A, a1, a2);
    if (zero) continue;
    GTerm g{};
    g.kind = P_EQ;
    for (int s = 0; s < N; s++) {
      if (ca[s] < 0) continue;
      const uint64_t bit = 1ull << s;
      g.tmask |= bit;
      if (ca[s]) g.tval |= bit;
      if (ca[s] != cb[s]) g.flip |= bit;
    }
    g.cre = sign;
    slots[t].push_back(g);
  }
  return run_corr(e, v, slots, out);
}
