// Internal types of the hphi_amd engine (device term tables, kernel argument
// blocks, engine state).  Not part of the C ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "hphi_amd.h"

#define HV_TPB 256        // threads per workgroup of the H·v kernels
#define HV_UNROLL 8       // terms per unrolled gather batch of the generic kernels
#define HV_TERM_PAD 16    // term groups are padded with never-active terms to a multiple of
                          // this, so every batch size in use (8, 16) reads whole groups
#define HV_NOALLOC_PARTIALS (1 << 18)  // k x workgroups of an allocation-free H·v (4 MiB of partial sums)
#define LZ_RING 64             // Lanczos steps in flight at most, 4 doubles each after the host partials
#define HV_HOST_PARTIALS 256  // partial sums of prdct a call adds up on the host
#define HV_MAX_GRID 65536 // upper bound of H·v workgroups (sizes the partial-sum buffer)

// predicate kinds of a gather term, evaluated on the TARGET state x
// grand-canonical models index the vector by the state's bits (no tables)
static inline bool hphi_model_gc(int m) { return m == HPHI_MODEL_SPINGC || m == HPHI_MODEL_HUBBARDGC; }
// Hubbard models: site i's orbitals are bits 2i (up) and 2i+1 (down)
static inline bool hphi_model_hubbard(int m) { return m == HPHI_MODEL_HUBBARD || m == HPHI_MODEL_HUBBARDGC; }

enum { P_EQ = 0,    // (x & tmask) == tval            (hopping, transverse field)
       P_DIFF = 1,  // popcount(x & tmask) == 1       (exchange: the two spins differ)
       P_SAME = 2   // popcount(x & tmask) != 1       (pair lift: the two spins agree)
};

// one off-diagonal term in gather form: source = x ^ flip, weight
// (cre + i cim) * (-1)^popcount(x & sgn) when the predicate holds
struct GTerm {
  uint64_t flip, tmask, tval, sgn;
  double cre, cim;
  int kind, pad;
};

// Term tables are read through the constant address space: the loads are
// known invariant, so uniform accesses become scalar (SMEM) loads instead of
// per-lane vector loads that would queue behind the gathers.
typedef const GTerm __attribute__((address_space(4))) *CTerm;

__device__ __forceinline__ GTerm load_term(CTerm p) {
  GTerm t;
  t.flip = p->flip;
  t.tmask = p->tmask;
  t.tval = p->tval;
  t.sgn = p->sgn;
  t.cre = p->cre;
  t.cim = p->cim;
  t.kind = p->kind;
  t.pad = 0;
  return t;
}

// host-side term compilers shared by the Hamiltonian and the Green's functions:
// bits strictly between orbitals a and b; V c+_{a1} c_{b1} c+_{a2} c_{b2}
// (fermions, Jordan-Wigner sign); V (|s1><s2|)_A (|s3><s4|)_B (spin-1/2)
uint64_t hphi_between_mask(int a, int b);
void hphi_compile_two_hops(int a1, int b1, int a2, int b2, double vre, double vim, std::vector<GTerm> &out);
void hphi_compile_spin_pair(int A, int s1, int s2, int B, int s3, int s4, double vre, double vim,
                            std::vector<GTerm> &out);

// diagonal term kinds (diagonalcalc.c set functions, per model)
enum { D_INTRA = 0, D_CHEMI_H, D_CHEMI_S, D_INTER_H, D_INTER_S, D_HUND_H, D_HUND_S, D_NN, D_SS };

struct DTerm {
  int kind, pad;
  uint64_t m1, m2, m3, m4;
  double V;
};

// runs of one kind in a diagonal's terms, after the skip leading constants (sum
// d0): the term compiler lists at most five kinds, each together
#define DIAG_RUNS 8
struct DRuns {
  double d0;
  int skip, n, kind[DIAG_RUNS], len[DIAG_RUNS];
};

struct SzParams {
  int hubbard, nlow, nhigh, nup, ndn;
  int nlu, nld, nhu, nhd;  // Hubbard: up/down positions in the low / high half
  uint64_t sdim, ihfbit, size21, dim;
};

struct HvArgs {
  uint64_t dim;
  const uint64_t *list1;
  const uint32_t *l21;
  const uint64_t *l22;
  const double *diag;
  const GTerm *terms;
  int n_low, n_high, n_mixed;  // group sizes (padded): the groups' offsets
  int e_low, e_high, e_mixed;  // loop extents: terms up to the launch's batch (<= the group sizes)
  int nlow;
  uint64_t irght;
  double *v0;
  const double *v1;
  double2 *partial;
  int xcd_map;
  uint64_t size21;
  int overwrite;  // 1: v0 = c1 H v1 (v0 not read); 0: v0 = c0 v0 + c1 H v1 (reference: c0 = c1 = 1)
  double c0, c1;  // scale factors of the output (prdct stays <v1|H v1>)
  const double *cdev;  // (c0, c1) on the device instead, where the caller has them there (k = 1)
  // canonical Spin: list_2_1[ia] = rank of ia among the values of its popcount
  // + 2, from two byte tables (hphi_crank_tables)
  const uint16_t *crank;
  // k_hv_canon also writes the tile-major copy of v1 for the high-half pass
  // when v1t is set: state (block ib, rank r) at tofs[ib].x + (r / HI_RT) tofs[ib].y + r % HI_RT
  double2 *v1t;
  const ulonglong2 *tofs;
};

// scale factors of the output
__device__ __forceinline__ double2 hv_scale(double c0, double c1, const double *cdev) {
  if (!cdev) return make_double2(c0, c1);
  const double __attribute__((address_space(4))) *c = (const double __attribute__((address_space(4))) *)cdev;
  return make_double2(c[0], c[1]);
}

// byte tables of the combinatorial rank (spin, nlow <= 16): rank(ia) =
// t[ia & 255] + t[256 + 9 * ((ia >> 8) & 255) + popcount(ia & 255)]
#define CRANK_N (256 + 256 * 9)

// list_2_1[ia] (rank + 2) of a canonical spin sector from the byte tables t
// staged in LDS (hphi_crank_tables)
__device__ __forceinline__ int64_t crank_l21(const uint16_t *t, uint32_t ia) {
  return (int64_t)t[ia & 255u] + (int64_t)t[256u + 9u * ((ia >> 8) & 255u) + (uint32_t)__popc(ia & 255u)] + 2;
}

// canonical Hubbard (up orbitals even bits, down odd): the rank of ia among the
// values with its up and down counts, t[ia & 255] + t[256 + 25 h + 5 u + d]
// with u, d the up / down counts of the low byte (hphi_hrank_tables)
#define HRANK_N (256 + 256 * 25)
__device__ __forceinline__ int64_t hrank_l21(const uint16_t *t, uint32_t ia) {
  return (int64_t)t[ia & 255u] +
         (int64_t)t[256u + 25u * ((ia >> 8) & 255u) + 5u * (uint32_t)__popc(ia & 0x55u) + (uint32_t)__popc(ia & 0xAAu)] +
         2;
}

// Canonical Spin and Hubbard, high-half terms by rank tiles (hv_canon.hip):
// for each class c (blocks whose high half holds the same number of up
// spins, or of up and of down electrons) its blocks (high-half values,
// ascending), the block size, the block groups of HI_BPG blocks, the
// workgroups before the class, and where the class's rank tiles start in the
// tile-major copy of v1 (tile R of block position p at base[c] + (R nblk[c] + p) HI_RT)
#define HI_MAXC 96
#define HI_RT 32              // ranks per tile (8x4 J1-J2: 89.8 ms at 32, 90.5 at 16, 92.8 at 8; 64 no better)
#define HI_BPG (256 / HI_RT)  // blocks per workgroup
struct HiPlan {
  int ncls;
  uint32_t start[HI_MAXC], nblk[HI_MAXC], size[HI_MAXC], ngrp[HI_MAXC];
  uint64_t wgp[HI_MAXC + 1], base[HI_MAXC + 1];
};

// Canonical H·v by classes (hv_class.hip)
struct ClsTerm {
  double cre, cim;
  uint32_t flip, tmask, tval, sgn;
  uint32_t tlo;            // the low half's part of tval
  int parity, src, lo;     // parity predicate (else value); compiled term (-1: padding); low-half flip of a mixed term
};
#define CL_TPB 256
#define CL_MAXC 96
#define CL_MAXLO 64               // distinct low-half flips of the mixed terms
struct ClsArgs {
  int ncls, n_low, n_high, n_mixed, nt, nlo, skip;
  int n_lowp, n_mixp;  // of the low and mixed terms, those with a parity predicate (first)
  uint32_t units, np;  // np: blocks
  uint32_t start[CL_MAXC], nblk[CL_MAXC], size[CL_MAXC], ntile[CL_MAXC], upre[CL_MAXC + 1];
  uint32_t lo[CL_MAXLO];
  const ClsTerm *terms;
  // groups of 1, 2 and 4 blocks in launch order, (first slot, first block, blocks, ranks) each, and the group of
  // every slot of 64 ranks; the launch's own in grp, sblk
  const uint4 *groups[3], *grp;
  const uint32_t *gslot[3], *sblk;
  uint32_t ngroup[3], nslot[3];
  const uint32_t *bstart, *bxh, *tgt;  // per block in class order; tgt [block][high and mixed terms]
};

// Grand-canonical H·v in LDS tiles (hv_gc.hip): a pass applies the terms whose
// flips lie inside its bit set S to the tiles of 2^|S| states.
struct GcTerm {
  double cre, cim;
  uint32_t flow, fe, flip;  // flip in the tile's element index: thread part, element part; in the state
  uint32_t tmask, tval;     // predicate (tval: the value, or 1 when an even parity passes)
  uint32_t sgn, sgi, es;    // sign masks of the real and imaginary part; their parities per element
  int parity, src;
};
#define GC_E 8       // elements per thread of k_hv_gc
#define GC_CASES 15  // parity terms by the element bits of predicate and flip: both m (0..7), or none and f (7 + f)
#define GC_MAXPASS 8
struct GcPass {
  int at = 0, nloc = 0, nother = 0, nrem = 0;  // first term; terms in the tile, those of no case; terms gathered
  uint32_t count[2][GC_CASES] = {};             // parity terms without and with a sign, by case
  int nob = 0, nrun = 0;                 // state bits outside S, and the runs they form
  uint32_t sb[16] = {}, omask[17] = {}, oshl[17] = {}, xe[GC_E] = {};
};
struct GcPlan {
  int npass = 0;
  GcPass pass[GC_MAXPASS];
};

// launch shapes set by hand: of k_hv_canon; of k_hv_blk for every block size; its
// columns per lane of one (slot 1..4: k = 2, 4, 8, 16)
#define HAND_C2 1
#define HAND_BLK_TPB 2
#define HAND_BLK_WGS 4
#define HAND_BLK_CPL(slot) (4 << (slot))

// place of a block size in per-size arrays; -1: no kernel for it
static inline int hphi_block_slot(int k) {
  return k == 1 ? 0 : k == 2 ? 1 : k == 4 ? 2 : k == 8 ? 3 : k == 16 ? 4 : -1;
}

struct hphi_engine {
  int model = 0, nsite = 0, nup = 0, ndown = 0, nbits = 0, nlow = 0;
  uint64_t dim = 0, sdim = 0, size21 = 0, size22 = 0, irght = 0, ilft = 0, ihfbit = 0;
  hipStream_t stream = nullptr;
  int num_cu = 256;
  int grid_per_cu = 8;  // H·v workgroups per CU (tunable)
  int xcd_map = 1;      // contiguous tile ranges per XCD (tunable)
  int xcd_tuned = 0;    // xcd_map was set through hphi_engine_tune
  bool tables_ready = false, diag_ready = false;
  uint64_t *d_list1 = nullptr, *d_l22 = nullptr, *d_jb = nullptr;
  uint32_t *d_l21 = nullptr;
  double *d_diag = nullptr;
  GTerm *d_terms = nullptr;
  DTerm *d_dterms = nullptr;
  std::vector<GTerm> h_terms, h_terms_dev;
  std::vector<DTerm> h_dterms;
  int n_low = 0, n_high = 0, n_mixed = 0;
  int r_low = 0, r_high = 0, r_mixed = 0;  // compiled terms per group, before padding
  void *d_partial = nullptr, *d_prdct = nullptr, *h_prdct = nullptr, *d_coef = nullptr;
  hipEvent_t lz_ev[2] = {};
  void *hd_prdct = nullptr;  // h_prdct (pinned) as the device addresses it
  double *d_stage0 = nullptr, *d_stage1 = nullptr;
  // host-pointer calls: per worker thread a stream and two pinned bounce
  // buffers of HOST_CHUNK bytes, with the events that free them
  int n_host = 0;
  hipStream_t h_stream[16] = {};
  char *h_bounce[16][2] = {};
  hipEvent_t h_ev[16][2] = {};
  uint64_t bytes = 0;
  // canonical single-vector kernel (hv_canon.hip) configuration
  int c2_ok = 0, c2_realc = 1, c2_lds21 = 0, c2_max_lds = 0;
  int c2_tpb = 1024, c2_wgs_per_cu = 1, use_c2 = 1;
  int c2_crank = 0, c2_crank_ok = 0, c2_unroll = 8;
  uint16_t *d_crank = nullptr;
  // block kernel (hv_block.hip): columns per lane for k = 2, 4, 8, 16 (0: default),
  // workgroup size (0: by table size), workgroups per CU (0: by workgroup size)
  int bk_cpl[4] = {0, 0, 0, 0};
  int bk_tpb = 0, bk_wgs_per_cu = 0, use_blk = 1;
  int device = 0;  // the device current when the engine was created
  int lb_mfma = 1;  // LOBPCG block-8 Gram on the FP64 matrix cores
  // canonical Spin and Hubbard: high-half terms in their own pass over a tile-major copy of v1
  int hi_split = -1;      // -1: by sector size, 0: off, 1: on when the sector allows it
  int hi_ok = -1;         // -1: not checked yet, 0: the sector does not allow it
  int hi_wgs_per_cu = 6;  // workgroups per CU of that pass (8x4 J1-J2: 6 best of 4-16)
  int hi_fuse_copy = 1;   // the first pass writes the tile-major copy (0: a copy kernel does)
  int hi_p1_wgs_per_cu = 256;  // workgroups per CU of that first pass (8x4 J1-J2: 90.4 ms at 256, 93.6 at 48)
  uint32_t *d_hb = nullptr;      // blocks of each class (hi_plan)
  uint32_t *d_hitgt = nullptr;  // targets of the high-half pass
  double2 *d_v1t = nullptr;      // tile-major copy of v1, hi_plan.base[ncls] elements
  ulonglong2 *d_tofs = nullptr;  // per block: its first tile-major element, and the stride between its tiles
  HiPlan hi_plan{};
  // canonical H·v by classes: -1 unless a shape of k_hv_canon is set, 0 off, 1 on where the sector allows it
  int cls = -1, cls_blocks = 0, cls_order = -1;
  int cls_wgs_per_cu = 256;  // by class: 8x4 J1-J2 77.3 ms at 64, 75.1 at 256; 7x4 3.67, 3.37; no effect below
  // launch shapes set by hand (HAND_*), which keep k_hv_canon or k_hv_blk where the knobs above are -1
  int hand = 0;
  void *d_cls = nullptr;
  ClsArgs cls_args{};
  // grand-canonical H·v in LDS tiles: -1 by size, 0 off, 1 also with a hand-set block shape
  int gc_tile = -1;
  // the same for one block size (1, 2, 4, 8, 16), the autotuner's choice; -2: as for the engine
  int cls_k[5] = {-2, -2, -2, -2, -2}, cls_blocks_k[5] = {-2, -2, -2, -2, -2}, gc_tile_k[5] = {-2, -2, -2, -2, -2};
  int use_blk_k[5] = {-2, -2, -2, -2, -2};
  GcPlan gc_plan[5];  // block sizes 1, 2, 4, 8, 16
  GcTerm *d_gcterms = nullptr;
};

// may blocks of the size in this place leave the generic kernel?
static inline int hphi_use_blk(const hphi_engine *e, int slot) {
  return e->use_blk_k[slot] != -2 ? e->use_blk_k[slot] : e->use_blk;
}

extern "C" int hphi_set_error(const char *fmt, ...);
extern "C" int hphi_block_size_ok(const char *entry, int k);
int hphi_build_tables(hphi_engine *e);
int hphi_build_diag(hphi_engine *e);
int hphi_hv_launch(hphi_engine *e, int k, double *v0, const double *v1);
int hphi_hv_launch_ex(hphi_engine *e, int k, double *v0, const double *v1, int overwrite);
// v0 <- c0 v0 + c1 H v1 with (c0, c1) read from cdev; prdct in d_prdct
int hphi_hv_launch_cdev(hphi_engine *e, double *v0, const double *v1, const double *cdev);
int hphi_hv_launch_gather(hphi_engine *e, int k, double *v0, const double *v1);
int hphi_hv_grid(const hphi_engine *e, int k);
int hphi_canon_config(hphi_engine *e);
void hphi_crank_tables(uint16_t *t);
void hphi_hrank_tables(uint16_t *t);
int hphi_engine_prepare(const hphi_model_desc *d, hphi_engine *e);
int hphi_ensure_binom_table();
// off-diagonal elements of H in a canonical sector (0 for grand-canonical models)
uint64_t hphi_term_nnz(const hphi_engine *e);
SzParams hphi_sz_params(const hphi_engine *e);
int hphi_launch_tables(const SzParams &P, uint64_t sdim, uint64_t size21, uint64_t *jb, uint32_t *l21, uint64_t *l22, uint64_t *list1, hipStream_t st);
// diag[j * stride + col] for the states j of h's sector, dterms its diagonal terms on the device
int hphi_launch_diag(const hphi_engine &h, const uint64_t *list1, const DTerm *dterms, double *diag, hipStream_t st,
                     int stride = 1, int col = 0);
int hphi_hv_launch_canon(hphi_engine *e, const HvArgs &A, int g, int skip_high = 0);
// canonical Spin: is the high-half pass usable and wanted for this engine (host check only)
int hphi_hi_wanted(const hphi_engine *e);
// the same, building its plan and buffers on first use (-1: error)
int hphi_hi_split_on(hphi_engine *e);
// launches the high-half pass: accumulates into A.v0, partials at partial[0..*grid)
int hphi_hv_launch_high(hphi_engine *e, const HvArgs &A, double2 *partial, int *grid);
int hphi_cls_build(hphi_engine *e, std::vector<char> &up);
bool hphi_cls_plan(const hphi_engine *e, ClsArgs &A, std::vector<char> &up);
size_t hphi_cls_bytes(const ClsArgs &A);
size_t hphi_cls_bytes_bound(const hphi_engine *e);
int hphi_cls_upload(const hphi_engine *e, ClsArgs &A, char *dev, const void *up, const uint64_t *l22, hipStream_t st);
void hphi_cls_units(ClsArgs &A, int cb, int rpt);
int hphi_cls_wanted(const hphi_engine *e, int k);
int hphi_cls_same_order(const hphi_engine *e);
int hphi_cls_grid(const hphi_engine *e, int k);
void hphi_cls_shape(const hphi_engine *e, int k, int *cb, int *cpl);
int hphi_hv_launch_cls(hphi_engine *e, const HvArgs &H, int k, int g, int skip_high);
int hphi_gc_wanted(const hphi_engine *e, int k);
int hphi_gc_plan_build(hphi_engine *e);
int hphi_gc_partials(const hphi_engine *e, int k);  // workgroups of all passes of one H·v
int hphi_hv_launch_gc(hphi_engine *e, const HvArgs &A, int k, int *grid);
int hphi_blk_ok(const hphi_engine *e);
int hphi_blk_cpl_ok(int k, int cpl);
void hphi_blk_shape(const hphi_engine *e, int k, int *cpl, int *tpb, int *wgs_per_cu);
int hphi_blk_grid(const hphi_engine *e, int k);
// records the device address of the allocation-free entry point's scratch array
int hphi_noalloc_setup(int device);
int hphi_hv_launch_blk(hphi_engine *e, const HvArgs &A, int k, int *grid);
