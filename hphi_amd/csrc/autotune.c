/*
 * Launch-shape autotuner for the H·v kernels (host C over the hphi_amd C ABI).
 *
 * For the single-vector canonical kernels it sweeps blocks per wave of the one by
 * classes, and of the other workgroup size, workgroups per CU, list_2_1 in LDS
 * or L2, and the XCD-contiguous tile mapping; for the block kernel (k > 1) it
 * sweeps columns per lane, workgroup size, workgroups per CU and the XCD
 * mapping; the per-column kernel is always a candidate, and the grand-canonical
 * tiles where the sector has them for k columns.  Each candidate is timed with
 * HIP events over `reps` H·v calls on the caller's vectors (v0 accumulates: the
 * caller re-initialises it).  The fastest is left set for block size k, and
 * under it the fastest of the gather kernels, which callers that need their
 * order of summation (LOBPCG) run whatever won.  The choice between kernels is
 * kept per block size, and shapes that the sweep sets do not count as set by
 * hand, so no other block size loses its kernel.  A one-line report per
 * candidate is written to `report` when it is non-NULL.
 */
#include <stdio.h>
#include <string.h>

#include "hphi_amd.h"

int hphi_set_error(const char *fmt, ...);
int hphi_block_size_ok(const char *entry, int k);
int hphi_tune_hand(const hphi_engine *e);
void hphi_tune_hand_restore(hphi_engine *e, int hand);

typedef struct {
  int n, gather; /* gather: one of the gather kernels */
  const char *knob[7];
  int val[7];
} cand_t;

static void add(cand_t *c, const char *knob, int val) {
  c->knob[c->n] = knob;
  c->val[c->n] = val;
  c->n++;
}

static int apply(hphi_engine *e, const cand_t *c) {
  for (int i = 0; i < c->n; i++)
    if (hphi_engine_tune(e, c->knob[i], c->val[i])) return -1;
  return 0;
}

/* the candidates for block size k, in the order they are timed */
typedef struct {
  char cls[24], cls_blocks[24], gc_tile[24], blk_cpl[24]; /* knobs of this k */
  char use[24];                                           /* 0: the per-column kernel */
  int has_cls, has_gc, n;
  cand_t c[96];
} sweep_t;

static cand_t *gather(sweep_t *s, int fast) {
  cand_t *c = &s->c[s->n++];
  c->gather = 1;
  add(c, s->use, fast);
  if (s->has_cls) add(c, s->cls, 0);
  if (s->has_gc) add(c, s->gc_tile, 0);
  return c;
}

static void candidates(hphi_engine *e, int k, sweep_t *s) {
  int on = 0;
  snprintf(s->cls, sizeof s->cls, "cls_k%d", k);
  snprintf(s->cls_blocks, sizeof s->cls_blocks, "cls_blocks_k%d", k);
  snprintf(s->gc_tile, sizeof s->gc_tile, "gc_tile_k%d", k);
  snprintf(s->blk_cpl, sizeof s->blk_cpl, "blk_cpl%d", k);
  if (k == 1) strcpy(s->use, "use_c2");
  else snprintf(s->use, sizeof s->use, "use_blk_k%d", k);
  /* an earlier choice for this k does not decide what is offered now */
  if (k > 1) hphi_engine_tune(e, s->use, -2);
  hphi_engine_tune(e, s->cls, -2);
  hphi_engine_tune(e, s->cls_blocks, -2);
  hphi_engine_tune(e, s->gc_tile, -2);
  hphi_engine_get_tune(e, s->cls, &s->has_cls);
  hphi_engine_get_tune(e, s->gc_tile, &s->has_gc);
  for (int cb = 1; s->has_cls && cb <= 4; cb *= 2) { /* by classes */
    cand_t *c = &s->c[s->n++];
    add(c, s->use, 1), add(c, s->cls, 1), add(c, s->cls_blocks, cb);
  }
  if (s->has_gc) { /* grand-canonical tiles: one shape */
    cand_t *c = &s->c[s->n++];
    add(c, s->use, 1), add(c, s->gc_tile, 1);
  }
  if (k == 1 && hphi_engine_get_tune(e, s->use, &on) == 0 && on) {
    /* is list_2_1 allowed in LDS for this model, are there rank tables? */
    int saved = 0;
    hphi_engine_get_tune(e, "lds21", &saved);
    const int lds_ok = hphi_engine_tune(e, "lds21", 1) == 0;
    hphi_engine_tune(e, "lds21", saved);
    hphi_engine_get_tune(e, "c2_crank", &saved);
    const int crank_ok = hphi_engine_tune(e, "c2_crank", 1) == 0;
    hphi_engine_tune(e, "c2_crank", saved);
    for (int xcd = 1; xcd >= 0; xcd--) {
      int tpbs[3] = {256, 512, 1024};
      if (lds_ok) {
        for (int a = 1; a < 3; a++) {
          cand_t *c = gather(s, 1);
          add(c, "xcd_map", xcd), add(c, "tpb", tpbs[a]);
          add(c, "wgs_per_cu", 1), add(c, "lds21", 1), add(c, "c2_crank", 0);
        }
      }
      for (int a = 0; a < 3; a++)
        for (int w = 2; w <= 8; w *= 2)
          if (tpbs[a] * w <= 4096) {
            cand_t *c = gather(s, 1);
            add(c, "xcd_map", xcd), add(c, "tpb", tpbs[a]);
            add(c, "wgs_per_cu", w), add(c, "lds21", 0), add(c, "c2_crank", 0);
          }
      if (crank_ok) { /* rank tables: large grids of small workgroups */
        const int ws[4] = {14, 21, 40, 48};
        for (int a = 0; a < 4; a++) {
          cand_t *c = gather(s, 1);
          add(c, "xcd_map", xcd), add(c, "tpb", 256);
          add(c, "wgs_per_cu", ws[a]), add(c, "c2_crank", 1);
        }
      }
    }
  }
  if (k > 1 && hphi_engine_get_tune(e, s->use, &on) == 0 && on) {
    /* block kernel: columns per lane x workgroup size x workgroups per CU x XCD map */
    int cpls[3] = {1, 4, k}, ncpl = k > 4 ? 3 : 2;
    if (k <= 4) cpls[1] = k;
    for (int xcd = 1; xcd >= 0; xcd--)
      for (int a = 0; a < ncpl; a++) {
        /* wide lanes hold 2*cpl accumulators: keep them on 256-thread groups */
        for (int w = 2; w <= 8; w *= 2) {
          cand_t *c = gather(s, 1);
          add(c, "xcd_map", xcd), add(c, s->blk_cpl, cpls[a]);
          add(c, "blk_tpb", 256), add(c, "blk_wgs_per_cu", w);
        }
        if (cpls[a] <= 4) {
          cand_t *c = gather(s, 1);
          add(c, "xcd_map", xcd), add(c, s->blk_cpl, cpls[a]);
          add(c, "blk_tpb", 1024), add(c, "blk_wgs_per_cu", 1);
        }
      }
  }
  for (int xcd = 1; xcd >= 0; xcd--)
    for (int g = 2; g <= 16; g *= 2) {
      cand_t *c = gather(s, 0);
      add(c, "xcd_map", xcd), add(c, "grid_per_cu", g);
    }
}

int hphi_autotune(hphi_engine *e, int k, double *v0, const double *v1, int reps, char *report,
                  size_t report_len) {
  if (!e || !v0 || !v1) return hphi_set_error("hphi_autotune: NULL argument");
  if (hphi_block_size_ok("hphi_autotune", k)) return -1;
  if (hphi_diagonalcalc(e, NULL)) return -1; /* tables and plans: which kernels there are to choose from */
  if (reps < 1) reps = 2;
  const int hand = hphi_tune_hand(e);
  sweep_t s;
  memset(&s, 0, sizeof s);
  candidates(e, k, &s);

  double best = 1e300, best_gather = 1e300;
  int bi = -1, gi = -1, rc = 0;
  size_t used = 0;
  if (report && report_len) report[0] = 0;
  for (int i = 0; i < s.n && !rc; i++) {
    const cand_t *c = &s.c[i];
    double ms = 0.0;
    if (apply(e, c)) continue;
    if ((rc = hphi_time_mltply_dev(e, k, v0, v1, 1, reps, &ms))) break;
    if (report && used + 160 < report_len) {
      for (int q = 0; q < c->n; q++)
        used += (size_t)snprintf(report + used, report_len - used, "%s=%d ", c->knob[q], c->val[q]);
      used += (size_t)snprintf(report + used, report_len - used, ": %.3f ms\n", ms);
    }
    if (ms < best) best = ms, bi = i;
    if (c->gather && ms < best_gather) best_gather = ms, gi = i;
  }
  if (!rc && bi < 0) rc = hphi_set_error("hphi_autotune: no candidate ran");
  /* the gather kernels' shape, then the winner's settings over it */
  if (!rc && gi >= 0) rc = apply(e, &s.c[gi]);
  if (!rc) rc = apply(e, &s.c[bi]);
  hphi_tune_hand_restore(e, hand);
  return rc ? -1 : 0;
}
