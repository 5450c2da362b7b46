// Gather-form H·v of canonical sectors (Spin, Hubbard), a tile of low-half ranks
// for several blocks at once.
//
// A state is (block = its high-half bits, rank of its low-half bits among
// those of its class), at index start[block] + rank; blocks of one class (equal
// particle numbers in the high half) have the same low halves in the same
// order.  k_hv_canon decodes every state of its own: predicate, rank lookup and
// 64-bit address of every term, some 28 vector instructions per term and state,
// which is half its time on sectors whose vectors stay in the caches.  Here
// a wave takes 64 consecutive ranks of one class and CB blocks of that class:
//  * low-half terms: predicate and target rank are the same in every block, so
//    they are computed once; the gather's address is the block's scalar base
//    plus the rank's 32-bit offset, with no vector arithmetic per block;
//  * high-half terms: the target block's base comes from a table of every
//    block and term (no base: the term does not act there); the offset is the
//    state's own rank;
//  * mixed terms: the base from the same table, the target rank from LDS, where
//    each lane keeps one rank per low-half flip that occurs (16 for the 48 mixed
//    terms of the 8x4 sector).
// Same sums in the same order as k_hv_canon (value predicates after parity
// ones within a group).  Microseconds per H·v, k_hv_canon / this kernel:
//   16-site J1-J2 chain (12,870 states)  15.6 / 10.8    6x4 J1-J2 (2.7e6)    292 / 151
//   20-site ladder (184,756)             20.9 / 16.8    12-site Hubbard      55.3 / 34.4
//   23-site chain (1.35e6)               90.2 / 50.5    7x4 J1-J2 (4.0e7)    5657 / 3070
//   4x4 Hubbard (1.7e8)                14,350 / 11,400  8x4 J1-J2 (6.0e8, with the
//   high-half pass)                    90,000 / 67,400
// The small ones are a chain of latencies, the middle ones were bound by that
// arithmetic and are now by the L1's 64 bytes per cycle and L2; the first pass of 8x4
// fetches 240 GB from beyond L2 in 46.8 ms, 5.1 TB/s.
//
// Blocks of K columns: LPS = K / CPL lanes share a state and a wave takes 64 / LPS
// ranks.  k_hv_blk / this kernel, microseconds: 6x4 J1-J2 k = 2 492 / 302, k = 4 880 /
// 600, k = 8 1,795 / 1,338, k = 16 3,926 / 3,266; 23-site chain k = 8 496 / 334;
// 16-site chain k = 8 20.7 / 11.3; 12-site Hubbard k = 8 215 / 145; 7x4 k = 4 19,285 /
// 14,658.  6x4 with k = 8 misses L2 for 9.1 GB, 7.1 TB/s: a state's columns fill a
// 128-byte line, so nothing of a gather is shared by neighbours, and the gathers
// of 32 CUs reach further than their 4 MB.  Rank-slice order of the units (2 to
// 64 tiles of every block before the next slice) gave nothing there and cost 10-25 %
// on 8x4.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <vector>

#include "engine_internal.h"
#include "hv_class.h"

#define HIPCHK(x)                                                                  \
  do {                                                                             \
    hipError_t e_ = (x);                                                           \
    if (e_ != hipSuccess) return hphi_set_error("%s failed: %s", #x, hipGetErrorString(e_)); \
  } while (0)

#define CL_U 8  // gathers in flight per lane: CL_U / CB terms per batch (4 and 16 within 3 % or slower)

// rank of low-half value y within its class
template <int RK>
__device__ __forceinline__ uint32_t cl_rank(const uint16_t *t, uint32_t y) {
  if (RK == 3)
    return (uint32_t)t[y & 255u] + (uint32_t)t[256u + 25u * (y >> 8) + 5u * (uint32_t)__popc(y & 0x55u) +
                                                (uint32_t)__popc(y & 0xAAu)];
  return (uint32_t)t[y & 255u] + (uint32_t)t[256u + 9u * (y >> 8) + (uint32_t)__popc(y & 255u)];
}

template <bool REALC>
__device__ __forceinline__ void cl_mac(double2 &a, double cr, double ci, double2 g) {
  a.x += cr * g.x;
  a.y += cr * g.y;
  if (!REALC) {
    a.x -= ci * g.y;
    a.y += ci * g.x;
  }
}

// terms per batch: eight gathers in flight
constexpr int cl_batch(int per_term) { return per_term >= CL_U ? 1 : CL_U / per_term; }

// n low-half terms of one predicate kind (PAR: the parity of the masked bits is
// odd; else the masked bits have a value) on CB blocks
template <int K, int CPL, int CB, bool PAR, bool REALC, int RK>
__device__ __forceinline__ void cl_low(CClsTerm TL, int n, uint32_t ia, uint32_t coff, const double2 *v1,
                                       const uint32_t *base, const uint16_t *s21, double2 (&acc)[CB][CPL]) {
  constexpr int U = cl_batch(CB * CPL);
#pragma unroll 1
  for (int t = 0; t < n; t += U) {
    double2 g[U][CB][CPL];
    uint32_t off[U];
    bool act[U];
#pragma unroll
    for (int q = 0; q < U; q++) {
      const ClsTerm T = cl_term(TL + t + q);
      act[q] = PAR ? (__popc(ia & T.tmask) & 1) != 0 : (ia & T.tmask) == T.tval;
      off[q] = cl_rank<RK>(s21, ia ^ T.flip) * (16u * K) + coff;
    }
#pragma unroll
    for (int q = 0; q < U; q++) {
#pragma unroll
      for (int b = 0; b < CB; b++)
#pragma unroll
        for (int i = 0; i < CPL; i++) g[q][b][i] = make_double2(0.0, 0.0);
      if (act[q]) {
#pragma unroll
        for (int b = 0; b < CB; b++)
#pragma unroll
          for (int i = 0; i < CPL; i++) g[q][b][i] = cl_at(v1 + (uint64_t)base[b] * K, off[q] + 16 * (K / CPL) * i);
      }
    }
#pragma unroll
    for (int q = 0; q < U; q++) {
      const ClsTerm T = cl_term(TL + t + q);
      const bool neg = RK == 3 && (__popc(ia & T.sgn) & 1);
      const double cr = neg ? -T.cre : T.cre, ci = neg ? -T.cim : T.cim;
#pragma unroll
      for (int b = 0; b < CB; b++)
#pragma unroll
        for (int i = 0; i < CPL; i++) cl_mac<REALC>(acc[b][i], cr, ci, g[q][b][i]);
    }
  }
}

// n mixed terms of one predicate kind: the low half's part of the predicate per
// lane, the high half's per block; tgt: the terms' first column of the table
template <int K, int CPL, int CB, bool PAR, bool REALC, int RK>
__device__ __forceinline__ void cl_mixed(CClsTerm TM, int n, uint32_t ia, const double2 *v1, const uint32_t *xh,
                                         CU32 tgt, const uint32_t *row, const uint32_t *sla,
                                         double2 (&acc)[CB][CPL]) {
  constexpr int U = cl_batch(CB * CPL);
#pragma unroll 1
  for (int t = 0; t < n; t += U) {
    double2 g[U][CB][CPL];
    uint32_t off[U], lp[U], to[U][CB];
#pragma unroll
    for (int b = 0; b < CB; b++)
#pragma unroll
      for (int q = 0; q < U; q++) to[q][b] = tgt[row[b] + t + q];
#pragma unroll
    for (int q = 0; q < U; q++) {
      const ClsTerm T = cl_term(TM + t + q);
      off[q] = sla[T.lo * CL_TPB + threadIdx.x];
      lp[q] = PAR ? (uint32_t)__popc(ia & T.tmask) & 1u : ((ia & T.tmask) == T.tlo ? 1u : 0u);
    }
#pragma unroll
    for (int q = 0; q < U; q++) {
      const ClsTerm T = cl_term(TM + t + q);
#pragma unroll
      for (int b = 0; b < CB; b++) {
        // scalar: what lp must be in this block (2: never)
        const uint32_t ok = PAR ? ((uint32_t)__popc(xh[b] & T.tmask) & 1u) ^ 1u : 1u;
        const uint32_t want = to[q][b] == CL_NONE ? 2u : ok;
#pragma unroll
        for (int i = 0; i < CPL; i++) g[q][b][i] = make_double2(0.0, 0.0);
        if (lp[q] == want) {
#pragma unroll
          for (int i = 0; i < CPL; i++) g[q][b][i] = cl_at(v1 + (uint64_t)to[q][b] * K, off[q] + 16 * (K / CPL) * i);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < U; q++) {
      const ClsTerm T = cl_term(TM + t + q);
      const uint32_t ls = RK == 3 ? (uint32_t)__popc(ia & T.sgn) : 0u;
#pragma unroll
      for (int b = 0; b < CB; b++) {
        const bool neg = RK == 3 && ((ls + (uint32_t)__popc(xh[b] & T.sgn)) & 1u);
#pragma unroll
        for (int i = 0; i < CPL; i++) cl_mac<REALC>(acc[b][i], neg ? -T.cre : T.cre, neg ? -T.cim : T.cim, g[q][b][i]);
      }
    }
  }
}

template <int K, int CPL, int CB, bool REALC, int RK>
__global__ __launch_bounds__(CL_TPB) void k_hv_cls(const HvArgs A, const ClsArgs C) {
  constexpr int U = cl_batch(CB * CPL);  // terms per batch
  constexpr int LPS = K / CPL;           // lanes per state
  constexpr int RPT = 64 / LPS;          // ranks per tile
  constexpr bool SGN = RK == 3;
  constexpr int NT = RK == 3 ? HRANK_N : CRANK_N;
  __shared__ uint16_t s21[NT];
  extern __shared__ uint32_t sla[];  // [nlo][CL_TPB]: offsets of the low-half flips of the mixed terms
  const uint32_t tid = threadIdx.x;
  for (uint32_t i = tid; i < NT / 4; i += CL_TPB) ((uint2 *)s21)[i] = ((const uint2 *)A.crank)[i];
  __syncthreads();
  const uint32_t lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const CU32 bstart = (CU32)C.bstart, bxh = (CU32)C.bxh, tgt = (CU32)C.tgt;
  const CClsTerm TL = (CClsTerm)C.terms, TH = TL + C.n_low, TM = TH + C.n_high;
  const double2 *v1 = (const double2 *)A.v1;
  double2 *v0 = (double2 *)A.v0;
  // an XCD takes a contiguous range of units
  const uint32_t xcd = blockIdx.x & 7u, slot = (blockIdx.x >> 3) * (CL_TPB / 64) + wave;
  const uint32_t nslot = (gridDim.x >> 3) * (CL_TPB / 64);
  const uint32_t U1 = (uint32_t)((uint64_t)C.units * (xcd + 1) / 8);
  const double2 cs = hv_scale(A.c0, A.c1, A.cdev);
  const uint32_t coff = (lane % LPS) * 16u;  // this lane's first column; the others at steps of LPS
  double pre[CPL], pim[CPL];
#pragma unroll
  for (int i = 0; i < CPL; i++) pre[i] = pim[i] = 0.0;
  for (uint32_t u = (uint32_t)((uint64_t)C.units * xcd / 8) + slot; u < U1; u += nslot) {
    uint32_t p0, nb, size, tile;  // first block, blocks from there on in its class, ranks of the class, tile of ranks
    if (C.sblk) {
      const CU32 G = (CU32)C.grp + 4 * ((CU32)C.sblk)[u / LPS];
      p0 = G[1];
      nb = G[2];
      size = G[3];
      tile = u - G[0] * LPS;
    } else {
      int c = 0, hi = C.ncls;  // upre[c] <= u < upre[hi]
      while (hi - c > 1) {
        const int mid = (c + hi) >> 1;
        if (C.upre[mid] <= u) c = mid;
        else hi = mid;
      }
      const uint32_t loc = u - C.upre[c], ntile = C.ntile[c], grp = loc / ntile;
      tile = loc % ntile;
      size = C.size[c];
      p0 = C.start[c] + grp * CB;
      nb = C.start[c] + C.nblk[c] - p0;
    }
    const uint32_t r = tile * RPT + lane / LPS;
    if (r >= size) continue;
    const uint32_t own_off = r * (16u * K) + coff;
    uint32_t base[CB], xh[CB], row[CB];
    double2 acc[CB][CPL];
#pragma unroll
    for (int b = 0; b < CB; b++) {
      const uint32_t p = p0 + (b < (int)nb ? b : 0);  // past the class's last block: the first again, not stored
      base[b] = bstart[p];
      xh[b] = bxh[p];
      row[b] = p * (uint32_t)C.nt;
    }
    const uint32_t ia = (uint32_t)A.list1[base[0] + r] & (uint32_t)A.irght;
#pragma unroll
    for (int b = 0; b < CB; b++)
#pragma unroll
      for (int i = 0; i < CPL; i++) acc[b][i] = cl_at(v1 + (uint64_t)base[b] * K, own_off + 16 * (K / CPL) * i);
    if (K == 1 && A.v1t) {  // tile-major copy for the high-half pass
#pragma unroll
      for (int b = 0; b < CB; b++)
        if (b < (int)nb) {
          const ulonglong2 ts = A.tofs[xh[b] >> A.nlow];
          A.v1t[ts.x + (uint64_t)(r / HI_RT) * ts.y + r % HI_RT] = acc[b][0];
        }
    }
#pragma unroll
    for (int b = 0; b < CB; b++) {
      const double d = *(const double *)((const char *)(A.diag + base[b]) + (r << 3));
#pragma unroll
      for (int i = 0; i < CPL; i++) {
        acc[b][i].x *= d;
        acc[b][i].y *= d;
      }
    }
    // ---- low-half terms: one predicate and one target rank for all blocks
    cl_low<K, CPL, CB, true, REALC, RK>(TL, C.n_lowp, ia, coff, v1, base, s21, acc);
    cl_low<K, CPL, CB, false, REALC, RK>(TL + C.n_lowp, C.n_low - C.n_lowp, ia, coff, v1, base, s21, acc);
    // ---- high-half terms: the same rank of another block
    for (int t = C.skip; t < C.n_high; t += U) {
      double2 g[U][CB][CPL];
      uint32_t to[U][CB];
#pragma unroll
      for (int b = 0; b < CB; b++)
#pragma unroll
        for (int q = 0; q < U; q++) to[q][b] = tgt[row[b] + t + q];
#pragma unroll
      for (int q = 0; q < U; q++)
#pragma unroll
        for (int b = 0; b < CB; b++) {
#pragma unroll
          for (int i = 0; i < CPL; i++) g[q][b][i] = make_double2(0.0, 0.0);
          if (to[q][b] != CL_NONE) {
#pragma unroll
            for (int i = 0; i < CPL; i++) g[q][b][i] = cl_at(v1 + (uint64_t)to[q][b] * K, own_off + 16 * (K / CPL) * i);
          }
        }
#pragma unroll
      for (int q = 0; q < U; q++) {
        const ClsTerm T = cl_term(TH + t + q);
#pragma unroll
        for (int b = 0; b < CB; b++) {
          const bool neg = SGN && (__popc(xh[b] & T.sgn) & 1);
#pragma unroll
          for (int i = 0; i < CPL; i++)
            cl_mac<REALC>(acc[b][i], neg ? -T.cre : T.cre, neg ? -T.cim : T.cim, g[q][b][i]);
        }
      }
    }
    // ---- mixed terms: another rank of another block
    for (int q = 0; q < C.nlo; q++) sla[q * CL_TPB + tid] = cl_rank<RK>(s21, ia ^ C.lo[q]) * (16u * K) + coff;
    cl_mixed<K, CPL, CB, true, REALC, RK>(TM, C.n_mixp, ia, v1, xh, tgt + C.n_high, row, sla, acc);
    cl_mixed<K, CPL, CB, false, REALC, RK>(TM + C.n_mixp, C.n_mixed - C.n_mixp, ia, v1, xh, tgt + C.n_high + C.n_mixp, row, sla,
                                   acc);
#pragma unroll
    for (int b = 0; b < CB; b++) {
      if (b < (int)nb) {
#pragma unroll
        for (int i = 0; i < CPL; i++) {
          const double2 a = cl_at(v1 + (uint64_t)base[b] * K, own_off + 16 * (K / CPL) * i);
          double2 *out = (double2 *)((char *)(v0 + (uint64_t)base[b] * K) + own_off + 16 * (K / CPL) * i);
          double2 o = make_double2(cs.y * acc[b][i].x, cs.y * acc[b][i].y);
          if (!A.overwrite) {
            const double2 p = *out;
            o.x += cs.x * p.x;
            o.y += cs.x * p.y;
          }
          *out = o;
          pre[i] += a.x * acc[b][i].x + a.y * acc[b][i].y;
          pim[i] += a.x * acc[b][i].y - a.y * acc[b][i].x;
        }
      }
    }
  }
  // prdct per column: lanes with equal lane % LPS hold the same columns
  __shared__ double2 red[CL_TPB / 64][K];
#pragma unroll
  for (int i = 0; i < CPL; i++) {
#pragma unroll
    for (int off = 32; off >= LPS; off >>= 1) {
      pre[i] += __shfl_xor(pre[i], off, 64);
      pim[i] += __shfl_xor(pim[i], off, 64);
    }
    if (lane < (uint32_t)LPS) red[wave][lane + LPS * i] = make_double2(pre[i], pim[i]);
  }
  __syncthreads();
  if (tid < (uint32_t)K) {
    double2 s = red[0][tid];
    for (int w = 1; w < CL_TPB / 64; w++) {
      s.x += red[w][tid].x;
      s.y += red[w][tid].y;
    }
    A.partial[(uint64_t)blockIdx.x * K + tid] = s;
  }
}

// tgt[p][t]: the first index of the block that high or mixed term t reads from
// block p, or CL_NONE where the high half fails its predicate or has no target
__global__ __launch_bounds__(256) void k_cls_targets(const uint32_t *bxh, const uint64_t *l22, uint32_t np, int nlow,
                                                     const ClsTerm *terms, int n_low, int nt, int n_high, uint32_t irght,
                                                     uint32_t *tgt) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (uint64_t)np * nt) return;
  const uint32_t p = (uint32_t)(i / nt), t = (uint32_t)(i % nt);
  const ClsTerm T = terms[n_low + t];
  const uint32_t xh = bxh[p], hm = T.tmask & ~irght;
  bool ok;
  if (T.src < 0) ok = false;
  else if (T.parity) ok = (int)t >= n_high || (__popc(xh & hm) & 1);  // a mixed one: either value, the low half decides
  else ok = (xh & hm) == (T.tval & ~irght);
  const uint64_t s = ok ? l22[((xh ^ T.flip) & ~irght) >> nlow] : 0;
  tgt[i] = s ? (uint32_t)(s - 1) : CL_NONE;
}

// group of every slot
__global__ __launch_bounds__(256) void k_cls_slots(const uint4 *grp, uint32_t n, uint32_t *sblk) {
  const uint32_t g = blockIdx.x;
  const uint32_t s0 = grp[g].x, m = (grp[g].w + 63) / 64;
  for (uint32_t i = threadIdx.x; i < m; i += 256) sblk[s0 + i] = g;
}

// ---------------------------------------------------------------- host ----

// the particle numbers a term changes, per species; false: not known from its masks
static bool conserves(const GTerm &t, uint64_t up) {
  if (t.kind != P_EQ) {  // two bits that differ, both flipped: of one species
    const int nb = __builtin_popcountll(t.tmask), nu = __builtin_popcountll(t.tmask & up);
    return t.kind == P_DIFF && nb == 2 && t.flip == t.tmask && (nu == 0 || nu == 2);
  }
  if (t.flip & ~t.tmask) return false;
  const uint64_t y = t.tval ^ t.flip;
  return __builtin_popcountll(t.tval & up) == __builtin_popcountll(y & up) &&
         __builtin_popcountll(t.tval & ~up) == __builtin_popcountll(y & ~up);
}

// Does the layout fit this sector and these terms?
static bool cls_possible(const hphi_engine *e) {
  const int nhigh = e->nbits - e->nlow;
  if (hphi_model_gc(e->model) || !(e->model == HPHI_MODEL_SPIN || e->model == HPHI_MODEL_HUBBARD)) return false;
  if (e->nbits > 32 || e->nlow > 16 || nhigh < 1 || nhigh > 16 || e->dim >= CL_NONE) return false;
  const uint64_t up = e->model == HPHI_MODEL_HUBBARD ? 0x5555555555555555ull : ~0ull;
  for (const GTerm &t : e->h_terms_dev)
    if (!(t.kind == P_EQ && t.tmask == 0 && t.tval != 0) && !conserves(t, up)) return false;
  return true;
}

// Blocks per wave, one column.  Few states: one, for more waves (12,870 states:
// 10.8 us with one, 13.1 with two, 18.1 with four; 184,756: 16.8, 17.5, 22.3).
// Where the vectors sit in the caches and arithmetic counts: two for Spin
// (1.35e6: 56.9, 50.5, 56.4; 2.7e6: 168, 151, 169), four for Hubbard, whose rank
// lookup costs more (8.5e5: 43.0, 37.8, 34.4).  Beyond the caches: one, whose rank
// tiles follow closest on each other in a block (Spin 4.0e7: 3,070, 3,197, 3,527; 6.0e8:
// 69,733, 72,963 with two; Hubbard 1.7e8: 11,393, 11,407, 11,573).
static int cls_blocks(const hphi_engine *e) {
  const uint64_t d = e->dim;
  if (d >= (uint64_t)1 << 24) return 1;
  if (e->model == HPHI_MODEL_HUBBARD) return d < ((uint64_t)1 << 17) ? 1 : d < ((uint64_t)1 << 19) ? 2 : 4;
  return d < ((uint64_t)1 << 18) ? 1 : 2;
}

// Blocks per wave and columns per lane of a block of k columns.  One column per
// lane: a load instruction then covers whole states (Spin 2.7e6, k = 8, two
// blocks: 1,338 us with one column per lane, 1,459 with two, 1,668 with four).
// Hubbard's rank lookup is worth sharing by two (8.5e5, k = 8: 170, 145, 187).
// Blocks: one while k columns still leave few waves (12,870 states, k = 8: 11.3,
// 13.0, 17.6 us with one, two, four), then two (2.7e6: 1,384, 1,338, 1,364), four
// beyond the caches (4.0e7, k = 4: 15,032, 14,865, 14,658).
void hphi_cls_shape(const hphi_engine *e, int k, int *cb, int *cpl) {
  const int slot = hphi_block_slot(k), own = slot < 0 ? -2 : e->cls_blocks_k[slot];
  const int set = own != -2 ? own : e->cls_blocks;
  *cb = set > 0 ? set : cls_blocks(e);
  *cpl = 1;
  if (k == 1) return;
  const uint64_t n = e->dim * (uint64_t)k;
  if (set == 0) *cb = n < ((uint64_t)1 << 18) ? 1 : e->dim < ((uint64_t)1 << 24) ? 2 : 4;
  if (e->model == HPHI_MODEL_HUBBARD && n >= ((uint64_t)1 << 18)) *cpl = 2;
}

// Where the gather kernels are as fast or faster, by two things.
//
// Row offsets: one KB of LDS per low-half flip of the mixed terms.  Exchange and
// hops have 16 at most; four-orbital InterAll entries of 16 Hubbard sites up to 72.
// Up to 26, four workgroups share a CU; up to 36, three, which pays where the tiles
// are full; beyond, two.  Microseconds, k_hv_canon / this kernel for k = 1, k_hv_blk /
// this one for k = 8:
//   16 sites, 4 + 4 electrons (3.3e6)   24 flips 299 / 207, 1370 / 1029; 36 378 / 314, 1679 / 1449;
//                                       40 406 / 465, 1782 / 2036
//   14 sites, 7 + 7 (1.2e7)             36 1411 / 868, 6389 / 5092; 40 1510 / 1221, 6794 / 7075
//   13 sites, 4 + 4 (5.1e5, fill 0.70)  34 91 / 101, 274 / 330
//
// Fill of the tiles: a class of few ranks leaves lanes of its tiles idle.  Below 2^17
// states the device has room for the idle ones, from 2^19 on no sector is that
// dilute; between them (k = 1 unless noted):
//   Spin of 30, 32 sites, 5 up (fill 0.34, 0.35)     23.4 / 25.5, 27.3 / 30.3; k = 2 32.6 / 27.8
//   24, 28 sites, 6 up (fill 0.49, 0.53)             19.9 / 17.5, 35.9 / 32.7
//   Hubbard 16 sites, 3 + 3 (0.42)                   26.1 / 28.7; k = 2 31.7 / 44.4, k = 4 93 / 75
//   Hubbard 7x2, 3 + 4 (0.55)                        33.2 / 38.1
//   Hubbard 16 sites, 2 + 5 (0.61)                   41.0 / 35.4; k = 2 50.3 / 48.4
//   Hubbard 5x3, 3 + 3 (0.41), k = 4                 57.5 / 67.0; 143,325 states (0.44) 49.1 / 42.3
//
// Hubbard sectors of a few workgroups: a chain of latencies either way, and the
// gather kernels' is the shorter (k_hv_canon has one rank lookup less in front of a
// term).  225 states: 11.5 / 12.5, k = 2 10.3 / 12.1, k = 4 12.4 / 11.5; 36: k = 4 9.8 / 10.8;
// 784: 11.6 / 12.7, k = 2 12.8 / 12.5; 3,136: 11.9 / 12.3; 4,900: 12.0 / 11.7.
static bool cls_pays(const hphi_engine *e, int k) {
  const ClsArgs &A = e->cls_args;
  if (A.nlo > 36) return false;
  const bool hub = e->model == HPHI_MODEL_HUBBARD;
  if (hub && k <= 4 && e->dim < (k == 1 ? 4096u : k == 2 ? 512u : 128u)) return false;
  if (A.nlo <= 26 && (e->dim < (uint64_t)1 << 17 || e->dim >= (uint64_t)1 << 19 || k > (hub ? 4 : 1))) return true;
  uint64_t lanes = 0;
  for (int c = 0; c < A.ncls; c++) lanes += (uint64_t)A.nblk[c] * ((A.size[c] + 63) / 64 * 64);
  const double fill = (double)e->dim / (double)lanes;
  if (A.nlo > 26) return fill >= 0.75;
  if (k == 4) return fill >= 0.45 || e->dim < (uint64_t)3 << 16 || e->dim >= (uint64_t)1 << 18;
  return fill >= (hub ? 0.56 : 0.45);
}

// a launch shape of the other kernel for k columns set by hand keeps that kernel
int hphi_cls_wanted(const hphi_engine *e, int k) {
  const int slot = hphi_block_slot(k);
  if (slot < 0 || !e->d_cls) return 0;
  const int on = e->cls_k[slot] != -2 ? e->cls_k[slot] : e->cls;
  if (on == 0 || !(k == 1 ? e->use_c2 : hphi_use_blk(e, slot))) return 0;
  return on == 1 || (cls_pays(e, k) && !(e->hand & (k == 1 ? HAND_C2 : HAND_BLK_TPB | HAND_BLK_WGS | HAND_BLK_CPL(slot))));
}

// Sums bit-equal to the gather kernels': real couplings (a complex product is
// three roundings there, two fused steps here), no group with both kinds of
// predicate, whose terms stand in another order here, and no term filed under
// mixed here and under low there (a flip within the low half with a mask or
// sign that reaches into the high one).
int hphi_cls_same_order(const hphi_engine *e) {
  const ClsArgs &A = e->cls_args;
  if (!e->c2_realc) return 0;
  for (int t = 0; t < e->n_low; t++) {
    const GTerm &x = e->h_terms_dev[t];
    if ((x.flip | x.tmask | x.sgn) & ~e->irght) return 0;
  }
  return (A.n_lowp == 0 || A.n_lowp == A.n_low) && (A.n_mixp == 0 || A.n_mixp == A.n_mixed);
}

// Blocks by class, their first indices and high halves, and the terms in three
// groups (padded with terms that never act): counts into A, terms, first
// indices and high halves into up.  false: the layout does not fit.
bool hphi_cls_plan(const hphi_engine *e, ClsArgs &A, std::vector<char> &up) {
  if (!cls_possible(e)) return false;
  const int nhigh = e->nbits - e->nlow;
  const bool hub = e->model == HPHI_MODEL_HUBBARD;
  const SzParams S = hphi_sz_params(e);
  const uint64_t even = 0x5555555555555555ull;
  auto C = [](int n, int k) -> uint64_t {
    if (k < 0 || k > n) return 0;
    uint64_t r = 1;
    for (int i = 1; i <= k; i++) r = r * (uint64_t)(n - k + i) / (uint64_t)i;
    return r;
  };
  uint64_t cu[33], cd[33];  // low-half values by the particles left for them
  for (int k = 0; k <= 32; k++) {
    cu[k] = hub ? C(S.nlu, k) : C(e->nlow, k);
    cd[k] = hub ? C(S.nld, k) : 1;
  }
  struct Cls {
    uint64_t size;
    std::vector<uint32_t> xh, at;
  };
  std::map<uint32_t, Cls> cls;
  uint64_t pos = 0;
  for (uint32_t ib = 0; ib < (1u << nhigh); ib++) {
    const uint64_t x = (uint64_t)ib << e->nlow;
    const int u = hub ? __builtin_popcountll(x & even) : __builtin_popcountll(x);
    const int d = hub ? __builtin_popcountll(x & ~even) : 0;
    if (u > e->nup || (hub && d > e->ndown) || e->nup - u > 32 || (hub && e->ndown - d > 32)) continue;
    const uint64_t n = cu[e->nup - u] * (hub ? cd[e->ndown - d] : 1);
    if (!n) continue;
    Cls &k = cls[(uint32_t)(u * 64 + d)];
    k.size = n;
    k.xh.push_back((uint32_t)x);
    k.at.push_back((uint32_t)pos);
    pos += n;
  }
  if (pos != e->dim || cls.size() > CL_MAXC) return false;
  std::vector<uint32_t> at, xh;
  A = ClsArgs{};
  for (const auto &k : cls) {
    A.start[A.ncls] = (uint32_t)at.size();
    A.nblk[A.ncls] = (uint32_t)k.second.at.size();
    A.size[A.ncls] = (uint32_t)k.second.size;
    A.ncls++;
    at.insert(at.end(), k.second.at.begin(), k.second.at.end());
    xh.insert(xh.end(), k.second.xh.begin(), k.second.xh.end());
  }
  // terms by group: pure low; those that leave the high half for another block
  // and touch no low bit, the same ones the engine files under high, so that
  // the high-half pass applies exactly what this kernel then skips (a term
  // without a flip whose mask lies in the high half is none of them); the others
  std::vector<ClsTerm> grp[5];  // low by parity, low by value, high, mixed by parity, mixed by value
  std::vector<uint32_t> lo;
  for (size_t i = 0; i < e->h_terms_dev.size(); i++) {
    const GTerm &t = e->h_terms_dev[i];
    if (t.kind == P_EQ && t.tmask == 0 && t.tval != 0) continue;
    const uint64_t all = t.flip | t.tmask | t.sgn, hm = ~e->irght;
    ClsTerm c{};
    c.cre = t.cre;
    c.cim = t.cim;
    c.flip = (uint32_t)t.flip;
    c.tmask = (uint32_t)t.tmask;
    c.tval = (uint32_t)t.tval;
    c.tlo = (uint32_t)(t.tval & e->irght);
    c.sgn = (uint32_t)t.sgn;
    c.parity = t.kind == P_DIFF;
    c.src = (int)i;
    const int g = (all & hm) == 0 ? 0 : (all & e->irght) == 0 && (t.flip & hm) ? 1 : 2;
    if (g == 2) {
      const uint32_t f = (uint32_t)(t.flip & e->irght);
      size_t q = std::find(lo.begin(), lo.end(), f) - lo.begin();
      if (q == lo.size()) lo.push_back(f);
      c.lo = (int)q;
    }
    grp[g == 1 ? 2 : g == 0 ? (c.parity ? 0 : 1) : (c.parity ? 3 : 4)].push_back(c);
  }
  if (lo.size() > CL_MAXLO) return false;
  ClsTerm never{};  // an empty mask has neither odd parity nor this value
  never.tval = never.tlo = 1;
  never.src = -1;
  for (auto &g : grp)
    while (g.size() % 8) g.push_back(never);
  A.n_lowp = (int)grp[0].size();
  A.n_low = A.n_lowp + (int)grp[1].size();
  A.n_high = (int)grp[2].size();
  A.n_mixp = (int)grp[3].size();
  A.n_mixed = A.n_mixp + (int)grp[4].size();
  A.nt = A.n_high + A.n_mixed;
  A.nlo = (int)lo.size();
  std::copy(lo.begin(), lo.end(), A.lo);
  std::vector<ClsTerm> terms;
  for (auto &g : grp) terms.insert(terms.end(), g.begin(), g.end());
  A.np = (uint32_t)at.size();
  // the target table, 4 bytes per block and term: a vector's bytes or 128 MB at most (8x4 J1-J2 takes
  // 27 MB; thousands of density-assisted hops on 16 sites would take gigabytes), rows addressed in 32 bits
  const uint64_t entries = (uint64_t)A.np * (uint64_t)A.nt;
  if (entries > 0xffffffffull || 4 * entries > std::max<uint64_t>(16 * e->dim, (uint64_t)128 << 20)) return false;
  const size_t tb = sizeof(ClsTerm) * terms.size();
  up.resize(tb + 8 * (size_t)A.np);
  std::copy(terms.begin(), terms.end(), (ClsTerm *)up.data());
  std::copy(at.begin(), at.end(), (uint32_t *)(up.data() + tb));
  std::copy(xh.begin(), xh.end(), (uint32_t *)(up.data() + tb) + A.np);
  return true;
}

// device bytes of a plan: up, then the target table
size_t hphi_cls_bytes(const ClsArgs &A) {
  return sizeof(ClsTerm) * (size_t)(A.n_low + A.nt) + 4 * (size_t)A.np * (2 + (size_t)A.nt);
}

// at most hphi_cls_bytes of the plan, without building it; 0: none
size_t hphi_cls_bytes_bound(const hphi_engine *e) {
  if (!cls_possible(e)) return 0;
  size_t n[3] = {0, 0, 0};
  for (const GTerm &t : e->h_terms_dev) {
    const uint64_t all = t.flip | t.tmask | t.sgn;
    n[(all & ~e->irght) == 0 ? 0 : (all & e->irght) == 0 ? 1 : 2]++;
  }
  for (auto &x : n) x += 14;  // padding of two predicate kinds
  const size_t np = std::min<size_t>((size_t)1 << (e->nbits - e->nlow), e->dim);
  return sizeof(ClsTerm) * (n[0] + n[1] + n[2]) + 4 * np * (2 + n[1] + n[2]);
}

// the plan on the device at dev: up is copied on st (and has to live until the
// copy is done), then the target table computed from list_2_2
int hphi_cls_upload(const hphi_engine *e, ClsArgs &A, char *dev, const void *up, const uint64_t *l22, hipStream_t st) {
  const size_t tb = sizeof(ClsTerm) * (size_t)(A.n_low + A.nt);
  A.terms = (const ClsTerm *)dev;
  A.bstart = (const uint32_t *)(dev + tb);
  A.bxh = A.bstart + A.np;
  uint32_t *tgt = (uint32_t *)(A.bxh + A.np);
  A.tgt = tgt;
  HIPCHK(hipMemcpyAsync(dev, up, tb + 8 * (size_t)A.np, hipMemcpyHostToDevice, st));
  const uint64_t n = (uint64_t)A.np * A.nt;
  if (n)
    hipLaunchKernelGGL(k_cls_targets, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, A.bxh, l22, A.np, e->nlow,
                       A.terms, A.n_low, A.nt, A.n_high, (uint32_t)e->irght, tgt);
  HIPCHK(hipGetLastError());
  return 0;
}

// The order of the units.  Class after class, an XCD the next eighth of them after
// the other: each XCD's gathers stay near its own part and meet in its L2, and
// what misses finds the 256 MB memory-side cache.  From 2^24 states on: groups follow
// the first index of their first block and are dealt to the XCDs one by one, to the
// one with the fewest slots, so that all XCDs work in one neighbourhood of the
// vector instead of eight and gathers that miss L2 have a chance in that cache.
// By class / by index, k = 1: rings of 24, 25, 26, 27 sites (2.7e6 to 2.0e7 states)
// 90 / 104, 157 / 190, 382 / 410, 870 / 875 us; Hubbard 14 sites, 6 + 6 (9.0e6) 261 / 274, 7x2
// (1.2e7) 463 / 520; 7x4 (4.0e7) 3,380 / 3,070; 4x4 Hubbard (1.7e8) 12,880 / 11,400; 8x4 75,300 /
// 69,700 (with an eighth per XCD by index 72,700, 13,667 on 4x4 Hubbard; dealt four by four
// 70,500, 11,634).  Blocks cross over earlier, at some 600 MB: ring of 25, k = 4 763 / 777, k = 8
// 1,595 / 1,550, k = 16 4,084 / 3,667; 7x2 k = 4 1,992 / 1,979, k = 8 4,463 / 4,079; an
// engine keeps one order, the single column's.
static int cls_by_index(const hphi_engine *e) {
  if (e->cls_order >= 0) return e->cls_order;
  return e->dim >= (uint64_t)1 << 24;
}

// Groups of cb blocks of a class in the order of a vector beyond the caches.
static uint32_t cls_groups(const hphi_engine *e, const ClsArgs &A, const uint32_t *xh, uint32_t cb,
                           std::vector<uint4> &out) {
  std::vector<uint32_t> at((size_t)1 << (e->nbits - e->nlow), CL_NONE);  // class and first block by high half
  std::vector<uint32_t> cls(at.size());
  for (int c = 0; c < A.ncls; c++)
    for (uint32_t i = 0; i < A.nblk[c]; i += cb) {
      const uint32_t h = xh[A.start[c] + i] >> e->nlow;
      at[h] = A.start[c] + i;
      cls[h] = c;
    }
  std::vector<uint4> q[8];
  uint32_t load[8] = {};
  for (size_t h = 0; h < at.size(); h++) {
    if (at[h] == CL_NONE) continue;
    const int c = cls[h], x = (int)(std::min_element(load, load + 8) - load);
    q[x].push_back(make_uint4(0, at[h], std::min(cb, A.start[c] + A.nblk[c] - at[h]), A.size[c]));
    load[x] += (A.size[c] + 63) / 64;
  }
  uint32_t slot = 0;
  for (const auto &v : q)
    for (uint4 g : v) {
      g.x = slot;
      slot += (g.w + 63) / 64;
      out.push_back(g);
    }
  return slot;
}

// One device allocation, written on e->stream, which the caller waits for before it
// frees up.  Sectors or terms the layout does not fit keep k_hv_canon.
int hphi_cls_build(hphi_engine *e, std::vector<char> &up) {
  ClsArgs &A = e->cls_args;
  if (e->d_cls || e->cls == 0 || !e->c2_ok || !e->c2_crank_ok || !hphi_cls_plan(e, A, up)) return 0;
  const size_t plan = (hphi_cls_bytes(A) + 255) / 256 * 256;
  std::vector<uint4> grp;
  const uint32_t *xh = (const uint32_t *)(up.data() + sizeof(ClsTerm) * (size_t)(A.n_low + A.nt)) + A.np;
  uint64_t slots = 0;
  for (int i = 0; i < 3 && cls_by_index(e); i++) {
    const size_t n = grp.size();
    A.nslot[i] = cls_groups(e, A, xh, 1u << i, grp);
    A.ngroup[i] = (uint32_t)(grp.size() - n);
    slots += A.nslot[i];
  }
  const size_t gb = sizeof(uint4) * grp.size(), bytes = plan + gb + 4 * slots;
  char *p = nullptr;
  if (hipMalloc((void **)&p, std::max<size_t>(bytes, 1)) != hipSuccess) {
    (void)hipGetLastError();
    return 0;  // no room: k_hv_canon serves this engine
  }
  e->d_cls = p;
  e->bytes += bytes;
  const size_t at = (up.size() + 15) / 16 * 16;  // the groups follow the plan's upload
  up.resize(at + gb);
  if (gb) memcpy(up.data() + at, grp.data(), gb);
  if (hphi_cls_upload(e, A, p, up.data(), e->d_l22, e->stream)) return -1;
  if (!gb) return 0;
  HIPCHK(hipMemcpyAsync(p + plan, up.data() + at, gb, hipMemcpyHostToDevice, e->stream));
  const uint4 *dg = (const uint4 *)(p + plan);
  uint32_t *ds = (uint32_t *)(p + plan + gb);
  for (int i = 0; i < 3; i++) {
    A.groups[i] = dg;
    A.gslot[i] = ds;
    hipLaunchKernelGGL(k_cls_slots, dim3(A.ngroup[i]), dim3(256), 0, e->stream, dg, A.ngroup[i], ds);
    dg += A.ngroup[i];
    ds += A.nslot[i];
  }
  HIPCHK(hipGetLastError());
  return 0;
}

// groups and units (a tile of 64 / lps ranks of a group) of a launch with cb blocks per wave
static void cls_launch_units(ClsArgs &A, int cb, int lps) {
  const int i = cb == 4 ? 2 : cb - 1;
  if (!A.groups[i]) {
    hphi_cls_units(A, cb, 64 / lps);
    return;
  }
  A.grp = A.groups[i];
  A.sblk = A.gslot[i];
  A.units = A.nslot[i] * (uint32_t)lps;
}

// units (a rank tile of a group of blocks) of a launch with cb blocks per wave
// and rpt ranks per tile
void hphi_cls_units(ClsArgs &A, int cb, int rpt) {
  uint32_t u = 0;
  for (int c = 0; c < A.ncls; c++) {
    A.upre[c] = u;
    A.ntile[c] = (A.size[c] + rpt - 1) / rpt;
    u += (A.nblk[c] + cb - 1) / cb * A.ntile[c];
  }
  A.upre[A.ncls] = u;
  A.units = u;
}

int hphi_cls_grid(const hphi_engine *e, int k) {
  ClsArgs A = e->cls_args;
  int cb, cpl;
  hphi_cls_shape(e, k, &cb, &cpl);
  cls_launch_units(A, cb, k / cpl);
  const uint64_t want = (A.units + CL_TPB / 64 - 1) / (CL_TPB / 64);
  uint64_t g = std::min<uint64_t>(want, (uint64_t)e->cls_wgs_per_cu * std::max(e->num_cu, 1));
  g = std::max<uint64_t>((g + 7) / 8 * 8, 8);
  // HV_NOALLOC_PARTIALS / k partial sums per column
  return (int)std::min<uint64_t>(g, k > 4 ? HV_NOALLOC_PARTIALS / k : HV_MAX_GRID);
}

template <int K, int CPL, int CB>
static int cls_launch(hphi_engine *e, const HvArgs &H, const ClsArgs &A, int g) {
  const size_t lds = sizeof(uint32_t) * CL_TPB * std::max(A.nlo, 1);
  const bool hub = e->model == HPHI_MODEL_HUBBARD;
#define CL_GO(R, RK) hipLaunchKernelGGL((k_hv_cls<K, CPL, CB, R, RK>), dim3(g), dim3(CL_TPB), lds, e->stream, H, A)
  if (hub) {
    if (e->c2_realc) CL_GO(true, 3);
    else CL_GO(false, 3);
  } else if constexpr (CPL == 1) {  // two columns per lane: Hubbard alone (hphi_cls_shape)
    if (e->c2_realc) CL_GO(true, 2);
    else CL_GO(false, 2);
  }
#undef CL_GO
  HIPCHK(hipGetLastError());
  return 0;
}

int hphi_hv_launch_cls(hphi_engine *e, const HvArgs &H, int k, int g, int skip_high) {
  ClsArgs A = e->cls_args;
  int cb, cpl;
  hphi_cls_shape(e, k, &cb, &cpl);
  cls_launch_units(A, cb, k / cpl);
  if (skip_high) A.skip = A.n_high;  // the high terms have a pass of their own
#define CASE(KK, CC, BB) \
  if (k == KK && cpl == CC && cb == BB) return cls_launch<KK, CC, BB>(e, H, A, g);
#define CASES(KK, CC) CASE(KK, CC, 1) CASE(KK, CC, 2) CASE(KK, CC, 4)
  CASES(1, 1)
  CASES(2, 1)
  CASES(4, 1)
  CASES(8, 1)
  CASES(16, 1)
  CASES(2, 2)
  CASES(4, 2)
  CASES(8, 2)
  CASES(16, 2)
#undef CASES
#undef CASE
  return hphi_set_error("no class kernel for k=%d, %d columns per lane, %d blocks", k, cpl, cb);
}
