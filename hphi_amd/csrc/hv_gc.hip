// H·v of grand-canonical sectors (SpinGC, HubbardGC) in LDS tiles.
//
// A grand-canonical state is its own index, so a term maps state x to
// x ^ flip.  The block kernel (hv_block.hip) gathers every source from the
// memory system: on the 13x2 triangular strip 65 exchange and 26 field terms
// read each amplitude about 45 times, and the gathers' rate through the
// fabric (about 8 TB/s) is what bounds it.  Here a workgroup takes the 2^s
// states that differ only in a set S of s bits (and KC of the K columns),
// reads them once into LDS, and applies every term whose flip lies inside S
// from there.  The sets are chosen on the host (gc_plan) so that a few passes
// over the vector cover the terms; what no worthwhile pass covers is gathered
// from memory in the first pass.  Each pass streams 16 (v1) + 16 or 32 (v0)
// bytes per amplitude.
//
// Within a tile thread t owns the elements t + TPB e (e < E): the top bits of
// the tile's local state index are e, so a term's predicate and sign split
// into one test per thread and a part known per element.  The loops over the
// terms are sorted by that part, which leaves per element one LDS read with an
// immediate offset and two FMAs (one test per element instead: 46 ps per
// amplitude against 37 on the 11x2 strip at k = 16).
//
// 11x2 triangular strip, k = 16 (6.7e7 amplitudes): 6.45 ms in the block kernel,
// 2.67 ms here in three passes (0.61 ms for 32 bytes per amplitude, 3.6 TB/s, then
// 1.03 ms each for 48 bytes, 3.2 TB/s; a device copy of that size reaches 4.4, a
// read-modify-write stream 5.5); k = 1: 442 -> 146 us; HubbardGC ring of 11 sites
// with complex spin flips, k = 2: 308 -> 262 us (95 and 2 x 84: 4.6 and 4.8 TB/s of a
// vector that the memory-side cache holds).  Reading the next tile's rows while the
// terms run (spills), and tiles of 1024 threads with 4 elements each, were no faster
// (2.98 and 3.16 ms, this form 2.50 beside them).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <utility>
#include <vector>

#include "engine_internal.h"

#define HIPCHK(x)                                                                  \
  do {                                                                             \
    hipError_t e_ = (x);                                                           \
    if (e_ != hipSuccess) return hphi_set_error("%s failed: %s", #x, hipGetErrorString(e_)); \
  } while (0)

#define GC_TPB 512  // threads per tile: 4096 elements, 64 KB of LDS, two tiles per CU

// one pass: its terms and bit sets (host-made, passed by value)
struct GcArgs {
  const double2 *v1;
  double2 *v0;
  const double *diag;
  // in the tile: parity terms (by case), parity terms with a sign (by case),
  // nother of any form; then nrem gathered from memory
  const GcTerm *terms;
  uint32_t count[2][GC_CASES];
  int nother, nrem;
  int K, overwrite;
  double c0, c1;
  const double *cdev;
  uint64_t nouter;            // tiles per column group: 2^(n - s)
  uint32_t xe[GC_E];          // state bits of element e
  uint32_t sb[16];            // state bit of each local bit
  uint32_t omask[17], oshl[17];  // runs of tile-number bits and their shifts into the state
  int nrun;
  double2 *partial;
};

typedef const GcTerm __attribute__((address_space(4))) *CGcTerm;

// acc += c g
template <bool REALC>
__device__ __forceinline__ void gc_mac(double2 &acc, double cr, double ci, double2 g) {
  acc.x += cr * g.x;
  acc.y += cr * g.y;
  if (!REALC) {
    acc.x -= ci * g.y;
    acc.y += ci * g.x;
  }
}

// element E of a parity term (see gc_parity): its LDS read and its product
template <int E, int M, int F, int HALF, int TPB>
__device__ __forceinline__ void gc_read(const double2 *src, double2 (&g)[GC_E]) {
  if constexpr ((__builtin_popcount(E & M) & 1) == HALF) g[E] = src[(E ^ F) * TPB];
}
template <int E, int M, int HALF, bool SGN, bool REALC>
__device__ __forceinline__ void gc_use(double cr, double ci, uint32_t es, const double2 (&g)[GC_E], double2 (&acc)[GC_E]) {
  if constexpr ((__builtin_popcount(E & M) & 1) == HALF) {
    if (SGN)
      gc_mac<REALC>(acc[E], (es >> E) & 1u ? -cr : cr, (es >> (8 + E)) & 1u ? -ci : ci, g[E]);
    else
      gc_mac<REALC>(acc[E], cr, ci, g[E]);
  }
}
template <int M, int F, int HALF, bool SGN, bool REALC, int TPB, int... E>
__device__ __forceinline__ void gc_half(const double2 *src, double cr, double ci, uint32_t es, double2 (&acc)[GC_E],
                                        std::integer_sequence<int, E...>) {
  double2 g[GC_E];
  (gc_read<E, M, F, HALF, TPB>(src, g), ...);
  (gc_use<E, M, HALF, SGN, REALC>(cr, ci, es, g, acc), ...);
  asm volatile("; case %0" ::"i"(2 * M + HALF));  // keeps the cases apart: merged, their stores to acc become indexed
}

// One parity term on this thread's elements.  M: the element bits its
// predicate tests, F: the element bits its flip changes; the elements with
// an even number of M's bits are acted on where lp holds, the others where it
// does not.  es: the scalar sign of every element (real part, imaginary << 8).
// Element numbers are template arguments: as loop counters they would still
// be variables when the switch's cases are merged, and acc would go to memory.
template <int M, int F, bool SGN, bool REALC, int TPB>
__device__ __forceinline__ void gc_parity(const double2 *src, bool lp, double cr, double ci, uint32_t es,
                                          double2 (&acc)[GC_E]) {
  using seq = std::make_integer_sequence<int, GC_E>;
  if (lp) gc_half<M, F, 0, SGN, REALC, TPB>(src, cr, ci, es, acc, seq{});
  if constexpr (M != 0) {
    if (!lp) gc_half<M, F, 1, SGN, REALC, TPB>(src, cr, ci, es, acc, seq{});
  }
}

// The parity terms inside the tile from term t on, in the plan's order of
// their case (the element bits of predicate and flip): a loop of its own per
// case, so that the LDS reads are one base address with immediate offsets,
// with no test per element.  Returns the term after the last.
template <bool SGN, bool REALC, int TPB>
__device__ __forceinline__ int gc_parity_terms(const GcArgs &A, int t, uint32_t x0, const double2 *tile,
                                               double2 (&acc)[GC_E]) {
#define GC_CASE(C, M, F)                                                                      \
  _Pragma("unroll 1") for (const int t1 = t + (int)A.count[SGN][C]; t < t1; t++) {            \
    const CGcTerm T = (CGcTerm)A.terms + t;                                                   \
    const bool lp = (((uint32_t)__popc(x0 & T->tmask) ^ T->tval) & 1u) != 0u;                 \
    double cr = T->cre, ci = T->cim;                                                          \
    if (SGN) {                                                                                \
      if (__popc(x0 & T->sgn) & 1) cr = -cr;                                                  \
      if (__popc(x0 & T->sgi) & 1) ci = -ci;                                                  \
    }                                                                                         \
    gc_parity<M, F, SGN, REALC, TPB>(tile + (threadIdx.x ^ T->flow), lp, cr, ci, T->es, acc); \
  }
  GC_CASE(0, 0, 0) GC_CASE(1, 1, 1) GC_CASE(2, 2, 2) GC_CASE(3, 3, 3)
  GC_CASE(4, 4, 4) GC_CASE(5, 5, 5) GC_CASE(6, 6, 6) GC_CASE(7, 7, 7)
  GC_CASE(8, 0, 1) GC_CASE(9, 0, 2) GC_CASE(10, 0, 3) GC_CASE(11, 0, 4)
  GC_CASE(12, 0, 5) GC_CASE(13, 0, 6) GC_CASE(14, 0, 7)
#undef GC_CASE
  return t;
}

// the other terms inside the tile, any predicate
template <int E, bool REALC, int TPB>
__device__ __forceinline__ void gc_other(const GcArgs &A, CGcTerm T, uint32_t x0, const double2 *src,
                                         double2 (&acc)[GC_E]) {
  const uint32_t x = x0 | A.xe[E];
  if (T->parity ? (((uint32_t)__popc(x & T->tmask) ^ T->tval) & 1u) != 0u : (x & T->tmask) == T->tval)
    gc_mac<REALC>(acc[E], __popc(x & T->sgn) & 1 ? -T->cre : T->cre, __popc(x & T->sgi) & 1 ? -T->cim : T->cim,
                  src[(E ^ T->fe) * TPB]);
}
template <bool REALC, int TPB, int... E>
__device__ __forceinline__ void gc_other_terms(const GcArgs &A, int t0, int t1, uint32_t x0, const double2 *tile,
                                               double2 (&acc)[GC_E], std::integer_sequence<int, E...>) {
#pragma unroll 1
  for (int t = t0; t < t1; t++) {
    const CGcTerm T = (CGcTerm)A.terms + t;
    (gc_other<E, REALC, TPB>(A, T, x0, tile + (threadIdx.x ^ T->flow), acc), ...);
  }
}

template <int... E>
__device__ __forceinline__ void gc_copy(const double2 (&from)[GC_E], double2 (&to)[GC_E],
                                        std::integer_sequence<int, E...>) {
  ((to[E] = from[E]), ...);
}

template <int KC, int TPB, bool REALC, bool FIRST, bool REM>
__global__ __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_hv_gc(const GcArgs A) {
  extern __shared__ double2 tile[];
  constexpr int LB = __builtin_ctz(TPB / KC);  // local state bits of the thread index
  const uint32_t tid = threadIdx.x;
  const uint32_t c = tid % KC, l0 = tid / KC;
  const int K = A.K, ncg = K / KC;
  uint32_t xl = 0;
#pragma unroll
  for (int i = 0; i < LB; i++) xl |= ((l0 >> i) & 1u) << A.sb[i];
  // an XCD takes a contiguous range of tiles; the column groups of one tile
  // run on neighbouring workgroups (they share cache lines when KC < 8)
  const uint32_t xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, nslot = (gridDim.x >> 3) / ncg;
  const uint32_t cg = slot % ncg;
  const uint64_t o1 = A.nouter * (xcd + 1) / 8;
  const uint64_t lane = (uint64_t)xl * K + cg * KC + c;  // this thread's part of an element's index
  double pre = 0.0, pim = 0.0;
  for (uint64_t o = slot < nslot * ncg ? A.nouter * xcd / 8 + slot / ncg : o1; o < o1; o += nslot) {
    uint32_t xo = 0;
    for (int i = 0; i < A.nrun; i++) xo |= ((uint32_t)o & A.omask[i]) << A.oshl[i];
    const uint32_t x0 = xo | xl;
    double2 row[GC_E];
#pragma unroll
    for (int e = 0; e < GC_E; e++) row[e] = (A.v1 + (uint64_t)(xo | A.xe[e]) * K)[lane];
#pragma unroll
    for (int e = 0; e < GC_E; e++) tile[tid + e * TPB] = row[e];
#pragma unroll
    for (int e = 0; e < GC_E; e++) {
      if (FIRST) {
        const double d = (A.diag + (xo | A.xe[e]))[xl];
        row[e].x *= d;
        row[e].y *= d;
      } else {
        row[e] = make_double2(0.0, 0.0);
      }
    }
    using seq = std::make_integer_sequence<int, GC_E>;
    double2 acc[GC_E];  // only constant subscripts: stays in registers through the terms' switches
    gc_copy(row, acc, seq{});
    __syncthreads();
    int t = gc_parity_terms<false, REALC, TPB>(A, 0, x0, tile, acc);
    t = gc_parity_terms<true, REALC, TPB>(A, t, x0, tile, acc);
    gc_other_terms<REALC, TPB>(A, t, t + A.nother, x0, tile, acc, seq{});
    t += A.nother;
    gc_copy(acc, row, seq{});
    if (REM) {
      const double2 *v = A.v1 + cg * KC + c;
#pragma unroll 1
      for (const int t1 = t + A.nrem; t < t1; t++) {
        const CGcTerm T = (CGcTerm)A.terms + t;
        const uint32_t tmask = T->tmask, tval = T->tval, sgn = T->sgn, sgi = T->sgi, flip = T->flip;
        const bool par = T->parity != 0;
        const double cr = T->cre, ci = T->cim;
#pragma unroll
        for (int h = 0; h < GC_E; h += 4) {
          double2 g[4];
          bool act[4];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const uint32_t x = x0 | A.xe[h + e];
            act[e] = par ? (((uint32_t)__popc(x & tmask) ^ tval) & 1u) != 0u : (x & tmask) == tval;
            if (act[e]) g[e] = v[(uint64_t)(x ^ flip) * K];
          }
#pragma unroll
          for (int e = 0; e < 4; e++) {
            if (act[e]) {
              const uint32_t x = x0 | A.xe[h + e];
              gc_mac<REALC>(row[h + e], __popc(x & sgn) & 1 ? -cr : cr, __popc(x & sgi) & 1 ? -ci : ci, g[e]);
            }
          }
        }
      }
    }
#pragma unroll
    for (int e = 0; e < GC_E; e++) {
      const double2 a = tile[tid + e * TPB];
      pre += a.x * row[e].x + a.y * row[e].y;
      pim += a.x * row[e].y - a.y * row[e].x;
    }
    __syncthreads();  // the next tile overwrites this one
    const bool add = !FIRST || !A.overwrite;
    const double2 cs = hv_scale(A.c0, A.c1, A.cdev);
    const double c0 = add ? (FIRST ? cs.x : 1.0) : 0.0, c1 = cs.y;
#pragma unroll
    for (int h = 0; h < GC_E; h += 4) {
      double2 old[4];
#pragma unroll
      for (int e = 0; e < 4; e++)
        old[e] = add ? (A.v0 + (uint64_t)(xo | A.xe[h + e]) * K)[lane] : make_double2(0.0, 0.0);
#pragma unroll
      for (int e = 0; e < 4; e++)
        (A.v0 + (uint64_t)(xo | A.xe[h + e]) * K)[lane] =
            make_double2(c0 * old[e].x + c1 * row[h + e].x, c0 * old[e].y + c1 * row[h + e].y);
    }
  }
  // prdct partials of this workgroup's columns; zeros for the others
#pragma unroll
  for (int off = 32; off >= KC; off >>= 1) {
    pre += __shfl_xor(pre, off, 64);
    pim += __shfl_xor(pim, off, 64);
  }
  __shared__ double2 red[TPB / 64][KC];
  if ((tid & 63) < KC) red[tid >> 6][tid & 63] = make_double2(pre, pim);
  __syncthreads();
  if (tid < (uint32_t)K) {
    double2 s = make_double2(0.0, 0.0);
    if (tid / KC == cg)
      for (int w = 0; w < TPB / 64; w++) {
        s.x += red[w][tid % KC].x;
        s.y += red[w][tid % KC].y;
      }
    A.partial[(uint64_t)blockIdx.x * K + tid] = s;
  }
}

// ---------------------------------------------------------------- host ----

// Relative costs of one amplitude: a further pass moves 48 bytes; a gathered
// term moves 16 bytes for the share of states it acts on.  They only decide
// which terms get a pass of their own (10x2 strip, k = 16: eight exchange terms
// gathered 742 us, in a third pass 635).
#define GC_COST_PASS 6.5
#define GC_COST_GATHER 2.0

// a term of the plan: a compiled term, or two that act on complementary states
// with conjugate couplings (sgi: the sign mask of the imaginary part)
struct GcSrc {
  GTerm t;
  uint32_t sgi;
};

static double gc_weight(const GcSrc &s) {
  if (s.t.kind != P_EQ) return s.t.tmask == 0 ? GC_COST_GATHER : 0.5 * GC_COST_GATHER;
  return GC_COST_GATHER / (double)(1u << std::min(__builtin_popcountll(s.t.tmask), 20));
}

// The plan's terms.  A transverse field's two directions (one bit, both
// values, the same coupling) act on every state: a parity term of no bits.  A
// complex hop and its Hermitian partner (complementary values of two bits,
// conjugate couplings) act where the two bits differ, and the imaginary part
// changes sign with the first one's bit: a parity term with its own sign mask.
static bool gc_sources(const hphi_engine *e, std::vector<GcSrc> &out) {
  std::map<uint64_t, std::vector<size_t>> open;  // value terms of one or two bits without their partner, by flip
  for (const GTerm &t : e->h_terms_dev) {
    if (t.kind == P_EQ && t.tmask == 0 && t.tval != 0) continue;  // padding
    if (t.kind != P_EQ && __builtin_popcountll(t.tmask) != 2) return false;
    const int nb = __builtin_popcountll(t.tmask);
    bool merged = false;
    if (t.kind == P_EQ && t.flip == t.tmask && (nb == 1 || (nb == 2 && __builtin_popcountll(t.tval) == 1))) {
      std::vector<size_t> &same = open[t.flip];
      for (size_t i : same) {
        GTerm &u = out[i].t;
        if (u.kind != P_EQ || u.tval != (t.tval ^ t.tmask) || u.sgn != t.sgn || u.cre != t.cre) continue;
        if (nb == 1 && u.cim == t.cim) {
          u.kind = P_SAME;
          u.tmask = u.tval = 0;
          merged = true;
        } else if (nb == 2 && u.cim == -t.cim) {
          out[i].sgi = (uint32_t)(u.sgn ^ u.tval);
          u.kind = P_DIFF;
          u.tval = 0;
          u.cim = -u.cim;
          merged = true;
        }
        if (merged) break;
      }
      if (!merged) same.push_back(out.size());
    }
    if (!merged) out.push_back(GcSrc{t, (uint32_t)t.sgn});
  }
  return true;
}

// The s bits (low `keep` bits included) that cover the most weight of the open
// terms: grown from every starting bit, each time by the bit that completes
// the most weight, and among equals the one that shares most with open terms.
// One- and two-bit flips go through a weight matrix (their gains are updated
// as bits join); wider ones count once per flip, for the bit that completes them.
// All plans of a 22-site strip: 0.15 ms of one core; of HubbardGC 10 with 200
// four-orbital pairs: 1.26 ms with every term looked up for every bit and every block
// size's plan made anew, 0.15 so.
static uint32_t gc_pick(const std::vector<GcSrc> &terms, const std::vector<char> &open, int n, int s, int keep,
                        double *weight) {
  double one[32] = {}, two[32][32] = {}, touch[32] = {};
  std::vector<std::pair<uint32_t, double>> wide;
  for (size_t t = 0; t < terms.size(); t++) {
    if (!open[t]) continue;
    const uint32_t f = (uint32_t)terms[t].t.flip;
    const double w = gc_weight(terms[t]);
    const int nb = __builtin_popcount(f), a = f ? __builtin_ctz(f) : 0;
    for (uint32_t r = f; r; r &= r - 1) touch[__builtin_ctz(r)] += 1e-3 * w;
    if (nb == 1) one[a] += w;
    else if (nb == 2) two[a][31 - __builtin_clz(f)] += w, two[31 - __builtin_clz(f)][a] += w;
    else if (nb > 2) wide.emplace_back(f, w);
  }
  std::sort(wide.begin(), wide.end());  // terms of one flip count together (the weights are powers of two: exact)
  size_t nw = 0;
  for (const auto &f : wide)
    if (nw > 0 && wide[nw - 1].first == f.first) wide[nw - 1].second += f.second;
    else wide[nw++] = f;
  wide.resize(nw);
  uint32_t best = 0;
  double bw = -1.0;
  for (int start = 0; start < n; start++) {
    uint32_t S = 0;
    double gain[32], w = 0.0;
    std::copy(one, one + n, gain);
    auto add = [&](int b) {
      S |= 1u << b;
      w += gain[b];
      for (int q = 0; q < n; q++) gain[q] += two[b][q];
    };
    for (int b = 0; b < keep; b++) add(b);
    if (!((S >> start) & 1)) add(start);
    if (__builtin_popcount(S) > s) continue;
    while (__builtin_popcount(S) < s) {
      int bb = -1;
      double bs = -1.0, sc[32];
      for (int b = 0; b < n; b++) sc[b] = gain[b] + touch[b];
      for (const auto &f : wide) {
        const uint32_t missing = f.first & ~S;
        if (missing && !(missing & (missing - 1))) sc[__builtin_ctz(missing)] += f.second;
      }
      for (int b = 0; b < n; b++)
        if (!((S >> b) & 1) && sc[b] > bs) bs = sc[b], bb = b;
      add(bb);
    }
    for (const auto &f : wide)
      if ((f.first & ~S) == 0) w += f.second;
    if (w > bw) bw = w, best = S;
  }
  *weight = bw;
  return best;
}

// Which grand-canonical engines take this path: 32-bit states, two-bit parity
// predicates, and tiles enough to give every CU one.  Per H·v, block
// kernel / tiles: 64 tiles (9x2 strip, k = 1) 32.3 / 31.9 us, 128 (9x2, k = 2)
// 48.9 / 47.1 and (HubbardGC 9, k = 2) 28.6 / 37.6, 256 (9x2, k = 4) 72 / 60 and
// (HubbardGC 9, k = 4) 44.1 / 44.4, 256 (10x2, k = 1) 115 / 57.  gc_pays says which of them.
#define GC_MIN_TILES 256

static int gc_kc(int k) { return k >= 4 ? 4 : k; }

int hphi_gc_wanted(const hphi_engine *e, int k) {
  const int sl = hphi_block_slot(k);
  if (sl < 0 || !hphi_model_gc(e->model)) return 0;
  const int on = e->gc_tile_k[sl] != -2 ? e->gc_tile_k[sl] : e->gc_tile;
  if (on == 0) return 0;
  // a block-kernel shape set by hand keeps that kernel
  if (on < 0 && k > 1 && (e->hand & (HAND_BLK_TPB | HAND_BLK_WGS | HAND_BLK_CPL(sl)))) return 0;
  if (k > 1 && !hphi_use_blk(e, sl)) return 0;
  return e->gc_plan[sl].npass > 0;
}

// Where the tiles are the faster ones, by default, among sectors with tiles
// enough.  W: the gathers an amplitude needs in the block kernel, wrem: those
// the first pass still makes.  Two things cost what the tiles save; per H·v,
// block kernel / tiles:
//  * terms of no case of gc_parity (a test per element) and gathered ones.  With
//    fewer than 512 tiles, one per workgroup, up to 0.3 of the terms (a ring of 18
//    sites, k = 4, with 10 InterAll pairs, 0.53: 58 / 71 us; 20 sites, k = 1, 5 pairs,
//    0.33: 57 / 60; HubbardGC 10, k = 1, 0.05: 50 / 48); with more, k = 2 two thirds (20
//    sites, 0.88: 202 / 215, 0.68: 111 / 111; HubbardGC 11, 0.69: 318 / 330), k = 4 half, and a
//    quarter where there are three passes (21 sites, 0.78: 431 / 458; HubbardGC 11, 0.67: 585 / 667,
//    three passes at 0.35: 689 / 799; 20 sites, 0.50: 163 / 149); any share for k = 1
//    (22 sites, 0.67: 294 / 209) and for k >= 8, where the block kernel's rows no
//    longer share cache lines (20 sites, 0.92: 1897 / 1169).
//  * blocks of 512 MB on, k >= 8, with few terms, of which some are gathered:
//    HubbardGC 11 (W 11, wrem 2) k = 16 1937 / 2247, a ring of 24 sites (12, 3) k = 8
//    3885 / 4542; HubbardGC 11 with 20 more pairs (13, 4) k = 16 3594 / 3120; the ring of
//    25 in three passes (12.5, 0) k = 8 9406 / 8958; HubbardGC 10 (10, 0, 256 MB) 487 / 434.
static bool gc_pays(const hphi_engine *e, int k, const GcPlan &P, double W, double wrem) {
  int fast = 0, slow = 0;
  for (int q = 0; q < P.npass; q++) {
    fast += P.pass[q].nloc - P.pass[q].nother;
    slow += P.pass[q].nother + P.pass[q].nrem;
  }
  const double share = (double)slow / std::max(fast + slow, 1);
  const uint64_t tiles = ((uint64_t)1 << P.pass[0].nob) * (uint64_t)(k / gc_kc(k));
  if (k <= 4 && tiles < 512) return share <= 0.3;
  if (k == 2) return share <= 2.0 / 3.0;
  if (k == 4) return share <= (P.npass >= 3 ? 0.25 : 0.5);
  return k < 8 || e->dim * (uint64_t)k < (uint64_t)1 << 25 || W >= 13.0 || wrem < 2.0;
}

// The passes of every block size, and their term tables on the device; called
// once the engine's diagonal is built, so that launches allocate nothing.
int hphi_gc_plan_build(hphi_engine *e) {
  if (!hphi_model_gc(e->model) || e->nbits > 32) return 0;
  std::vector<GcSrc> terms;
  if (!gc_sources(e, terms)) return 0;
  const int n = e->nbits, nt = (int)terms.size();
  std::vector<GcTerm> all;
  GcPlan made;  // the last plan made, its columns per tile and what it gathers
  int made_kc = 0;
  double W = 0.0, made_wrem = 0.0;
  for (const GcSrc &t : terms) W += gc_weight(t) / GC_COST_GATHER;
  for (int k = 1; k <= 16; k *= 2) {
    const int kc = gc_kc(k);
    const int s = __builtin_ctz(GC_TPB * GC_E / kc);
    GcPlan &P = e->gc_plan[hphi_block_slot(k)];
    P = GcPlan{};
    if (n < s + 3 || (e->gc_tile != 1 && ((uint64_t)1 << (n - s)) * (uint64_t)(k / kc) < GC_MIN_TILES)) continue;
    if (made_kc == kc) {  // the same tiles, more of them
      P = made;
      if (e->gc_tile != 1 && !gc_pays(e, k, P, W, made_wrem)) P = GcPlan{};
      continue;
    }
    const int keep = kc == 1 ? 3 : kc == 2 ? 2 : 0;  // runs of 128 bytes, 64 with KC = 4
    std::vector<char> open(nt, 1);
    uint32_t S[GC_MAXPASS];
    while (P.npass < GC_MAXPASS) {
      double w = 0.0;
      const uint32_t pick = gc_pick(terms, open, n, s, keep, &w);
      if (P.npass > 0 && w < GC_COST_PASS) break;
      S[P.npass++] = pick;
      for (int t = 0; t < nt; t++)
        if (((uint32_t)terms[t].t.flip & ~pick) == 0) open[t] = 0;
    }
    // a term that several passes cover goes to the one with the fewest terms
    // (the first pass also gathers and reads the diagonal: it counts those)
    int nrem = 0;
    double wrem = 0.0;
    for (int t = 0; t < nt; t++)
      if (open[t]) nrem++, wrem += gc_weight(terms[t]) / GC_COST_GATHER;
    std::vector<int> pass(nt, -1);
    int load[GC_MAXPASS] = {4 * nrem + 4};
    for (int many = 0; many < 2; many++)
      for (int t = 0; t < nt; t++) {
        int opts = 0, at = -1;
        for (int q = 0; q < P.npass; q++)
          if (((uint32_t)terms[t].t.flip & ~S[q]) == 0) {
            opts++;
            if (at < 0 || load[q] < load[at]) at = q;
          }
        if (opts == 0 || (opts > 1) != (many > 0)) continue;
        pass[t] = at;
        load[at]++;
      }
    for (int q = 0; q < P.npass; q++) {
      GcPass &Q = P.pass[q];
      Q.at = (int)all.size();
      int nb = 0;
      uint8_t pos[32];
      for (int b = 0; b < n; b++)
        if ((S[q] >> b) & 1) pos[b] = (uint8_t)nb, Q.sb[nb++] = (uint32_t)b;
      for (int b = 0; b < n; b++) {
        if ((S[q] >> b) & 1) continue;
        // tile-number bit nob goes to state bit b: a run shares one shift
        const uint32_t sh = (uint32_t)(b - Q.nob);
        if (Q.nrun == 0 || Q.oshl[Q.nrun - 1] != sh) Q.oshl[Q.nrun++] = sh;
        Q.omask[Q.nrun - 1] |= 1u << Q.nob++;
      }
      const int lb = s - 3;  // GC_E = 8: the top three local bits are the element number
      for (int x = 0; x < GC_E; x++)
        for (int b = 0; b < 3; b++)
          if ((x >> b) & 1) Q.xe[x] |= 1u << Q.sb[lb + b];
      std::vector<GcTerm> in[2 * GC_CASES + 1];  // by sign and case, then the others
      for (int t = 0; t < nt; t++) {
        if (pass[t] != q) continue;
        const GTerm &u = terms[t].t;
        const uint32_t f = (uint32_t)u.flip;
        uint32_t fl = 0, fm = 0;
        for (int b = 0; b < n; b++) {
          if ((f >> b) & 1) fl |= 1u << pos[b];
          if (((S[q] & (uint32_t)u.tmask) >> b) & 1) fm |= 1u << pos[b];
        }
        GcTerm g{};
        g.flow = (fl & ((1u << lb) - 1)) * (uint32_t)kc;
        g.fe = fl >> lb;
        for (int x = 0; x < GC_E; x++) {
          if (__builtin_popcount(Q.xe[x] & (uint32_t)u.sgn) & 1) g.es |= 1u << x;
          if (__builtin_popcount(Q.xe[x] & terms[t].sgi) & 1) g.es |= 1u << (8 + x);
        }
        g.flip = f;
        g.src = t;
        const uint32_t me = fm >> lb;
        const int sign = u.sgn || terms[t].sgi ? 1 : 0;
        if (u.kind != P_EQ && (me == g.fe || me == 0))
          in[sign * GC_CASES + (int)(me == g.fe ? me : 7 + g.fe)].push_back(g);
        else
          in[2 * GC_CASES].push_back(g);
      }
      for (int c = 0; c <= 2 * GC_CASES; c++) {
        if (c < 2 * GC_CASES) Q.count[c / GC_CASES][c % GC_CASES] = (uint32_t)in[c].size();
        else Q.nother = (int)in[c].size();
        Q.nloc += (int)in[c].size();
        all.insert(all.end(), in[c].begin(), in[c].end());
      }
      if (q == 0) {  // what no pass covers is gathered from memory in the first one
        for (int t = 0; t < nt; t++)
          if (pass[t] < 0) {
            GcTerm g{};
            g.flip = (uint32_t)terms[t].t.flip;
            g.src = t;
            all.push_back(g);
          }
        Q.nrem = nrem;
      }
    }
    made = P;
    made_kc = kc;
    made_wrem = wrem;
    if (e->gc_tile != 1 && !gc_pays(e, k, P, W, wrem)) P = GcPlan{};
  }
  for (GcTerm &g : all) {
    const GTerm &t = terms[g.src].t;
    g.tmask = (uint32_t)t.tmask;
    g.sgn = (uint32_t)t.sgn;
    g.sgi = terms[g.src].sgi;
    g.parity = t.kind != P_EQ;
    g.tval = t.kind == P_EQ ? (uint32_t)t.tval : (t.kind == P_SAME ? 1u : 0u);  // parity inverted for "agree"
    g.cre = t.cre;
    g.cim = t.cim;
  }
  if (std::all_of(e->gc_plan, e->gc_plan + 5, [](const GcPlan &P) { return P.npass == 0; })) return 0;
  if (hipMalloc((void **)&e->d_gcterms, sizeof(GcTerm) * all.size()) != hipSuccess) {
    (void)hipGetLastError();
    e->d_gcterms = nullptr;
    for (GcPlan &P : e->gc_plan) P.npass = 0;  // no room: the gather kernels serve this engine
    return 0;
  }
  HIPCHK(hipMemcpy(e->d_gcterms, all.data(), sizeof(GcTerm) * all.size(), hipMemcpyHostToDevice));
  e->bytes += sizeof(GcTerm) * all.size();
  return 0;
}

// workgroups of one pass: two per CU (their tiles fill the LDS), whole column
// groups on every XCD
static int gc_grid(const hphi_engine *e, int k) {
  const GcPlan &P = e->gc_plan[hphi_block_slot(k)];
  const int ncg = k / gc_kc(k);
  const uint64_t per_xcd = std::max<uint64_t>((((uint64_t)1 << P.pass[0].nob) + 7) / 8, 1) * (uint64_t)ncg;
  const uint64_t want = (uint64_t)std::max(e->num_cu, 8) * 2 / 8;
  uint64_t g = std::min(per_xcd, std::max<uint64_t>(want / ncg * ncg, ncg));
  return (int)(8 * g);
}

int hphi_gc_partials(const hphi_engine *e, int k) { return gc_grid(e, k) * e->gc_plan[hphi_block_slot(k)].npass; }

template <int KC>
static int gc_launch(hphi_engine *e, const GcArgs &G, int g, bool first) {
  constexpr size_t lds = sizeof(double2) * GC_TPB * GC_E;
#define GC_GO(R, F, M) hipLaunchKernelGGL((k_hv_gc<KC, GC_TPB, R, F, M>), dim3(g), dim3(GC_TPB), lds, e->stream, G)
#define GC_SEL(R)                     \
  if (!first) GC_GO(R, false, false); \
  else if (G.nrem) GC_GO(R, true, true); \
  else GC_GO(R, true, false);
  if (e->c2_realc) {
    GC_SEL(true)
  } else {
    GC_SEL(false)
  }
#undef GC_SEL
#undef GC_GO
  HIPCHK(hipGetLastError());
  return 0;
}

// every pass in stream order; partials at A.partial[0 .. *grid * k)
int hphi_hv_launch_gc(hphi_engine *e, const HvArgs &A, int k, int *grid) {
  const GcPlan &P = e->gc_plan[hphi_block_slot(k)];
  const int g = gc_grid(e, k), kc = gc_kc(k);
  for (int p = 0; p < P.npass; p++) {
    const GcPass &Q = P.pass[p];
    GcArgs G{};
    G.v1 = (const double2 *)A.v1;
    G.v0 = (double2 *)A.v0;
    G.diag = A.diag;
    G.terms = e->d_gcterms + Q.at;
    for (int c = 0; c < GC_CASES; c++) G.count[0][c] = Q.count[0][c], G.count[1][c] = Q.count[1][c];
    G.nother = Q.nother;
    G.nrem = Q.nrem;
    G.K = k;
    G.overwrite = A.overwrite;
    G.c0 = A.c0;
    G.c1 = A.c1;
    G.cdev = A.cdev;
    G.nrun = Q.nrun;
    G.nouter = (uint64_t)1 << Q.nob;
    std::copy(Q.sb, Q.sb + 16, G.sb);
    std::copy(Q.omask, Q.omask + 17, G.omask);
    std::copy(Q.oshl, Q.oshl + 17, G.oshl);
    std::copy(Q.xe, Q.xe + GC_E, G.xe);
    G.partial = A.partial + (uint64_t)p * g * k;
    const int rc = kc == 1 ? gc_launch<1>(e, G, g, p == 0) : kc == 2 ? gc_launch<2>(e, G, g, p == 0)
                                                                   : gc_launch<4>(e, G, g, p == 0);
    if (rc) return -1;
  }
  *grid = g * P.npass;
  return 0;
}
