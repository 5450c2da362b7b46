// Host-side plans of the H·v kernels, without a device: prints one "name value"
// line per check for tests/test_host_plans.py.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "engine_internal.h"
#include "hphi_amd.h"

int hphi_engine_prepare(const hphi_model_desc *d, hphi_engine *e);
bool hphi_slab_cls_pays(const hphi_engine &h);

// a canonical engine as hphi_engine_create leaves it, with its class layout planned
static bool plan(const hphi_model_desc &d, hphi_engine &e, std::vector<char> &up) {
  if (hphi_engine_prepare(&d, &e)) return false;
  hphi_canon_config(&e);
  e.num_cu = 256;
  e.c2_crank = 1;
  if (!hphi_cls_plan(&e, e.cls_args, up)) return false;
  e.d_cls = up.data();
  return true;
}

static void block_sizes() {
  const int ij[] = {0, 1, 1, 2, 2, 3, 6, 7};
  const double J[] = {1, 1, 1, 1};
  hphi_model_desc d{};
  d.model = HPHI_MODEL_SPIN, d.nsite = 8, d.nup = 4;
  d.n_exchange = 4, d.exchange_ij = ij, d.exchange_J = J;
  hphi_engine e;
  std::vector<char> up;
  if (!plan(d, e, up)) return;
  for (int k : {1, 2, 4, 8, 16, 0, -1, 3, 32, 64, 65, 128, 1024, 1028})
    printf("cls_wanted_%d %d\n", k, hphi_cls_wanted(&e, k));
}

// Hubbard ring of 6 sites with hops re + i im and the InterAll entries ia, planned
static bool ring(double re, double im, const std::vector<int> &ia, const std::vector<double> &iv, hphi_engine &e,
                 std::vector<char> &up) {
  const int n = 6;
  std::vector<int> idx;
  std::vector<double> t;
  for (int i = 0; i < n; i++)
    for (int s = 0; s < 2; s++) {
      const int j = (i + 1) % n, a[8] = {i, s, j, s, j, s, i, s};
      idx.insert(idx.end(), a, a + 8);
      for (int q = 0; q < 2; q++) t.push_back(re), t.push_back(q ? -im : im);
    }
  hphi_model_desc d{};
  d.model = HPHI_MODEL_HUBBARD, d.nsite = n, d.nup = 3, d.ndown = 3;
  d.n_transfer = (int)idx.size() / 4, d.transfer_idx = idx.data(), d.transfer_t = t.data();
  d.n_interall = (int)iv.size() / 2, d.interall_idx = ia.data(), d.interall_V = iv.data();
  return plan(d, e, up);
}
static const std::vector<int> NN_HIGH = {4, 0, 4, 0, 5, 1, 5, 1};  // n n on two sites of the high half
static const std::vector<int> ASSISTED = {5, 0, 5, 0, 0, 0, 1, 0, 1, 0, 0, 0, 5, 0, 5, 0};  // n in the high half, hop in the low one

// terms whose flip leaves the high half: the engine's group against the class
// layout's, for hops, a density product in the high half and a density-assisted hop
static void high_terms() {
  std::vector<int> ia = NN_HIGH;
  ia.insert(ia.end(), ASSISTED.begin(), ASSISTED.end());
  hphi_engine e;
  std::vector<char> up;
  if (!ring(1.0, 0.0, ia, {0.7, 0.0, 0.2, 0.1, 0.2, -0.1}, e, up)) return;
  e.hi_split = 1;
  const ClsTerm *T = (const ClsTerm *)up.data();
  int differ = 0, high = 0;
  for (int i = 0; i < e.cls_args.n_low + e.cls_args.nt; i++) {
    if (T[i].src < 0) continue;
    const bool here = i >= e.cls_args.n_low && i < e.cls_args.n_low + e.cls_args.n_high;
    differ += here != (T[i].src >= e.n_low && T[i].src < e.n_low + e.n_high);
    high += here;
  }
  printf("hi_wanted %d\nhigh_terms %d\nhigh_filed_differently %d\n", hphi_hi_wanted(&e), high, differ);
}

// may LOBPCG's H·v, which needs the gather kernels' order of summation, run by classes?
static void same_order() {
  std::vector<char> up;
  hphi_engine real, cplx, nn, assisted;
  if (ring(1.0, 0.0, {}, {}, real, up)) printf("same_order_real_hops %d\n", hphi_cls_same_order(&real));
  if (ring(1.0, 0.3, {}, {}, cplx, up)) printf("same_order_complex_hops %d\n", hphi_cls_same_order(&cplx));
  if (ring(0.0, 0.0, NN_HIGH, {0.7, 0.0}, nn, up)) printf("same_order_nn_high %d\n", hphi_cls_same_order(&nn));
  if (ring(0.0, 0.0, ASSISTED, {0.2, 0.0, 0.2, 0.0}, assisted, up))
    printf("same_order_assisted %d\n", hphi_cls_same_order(&assisted));
}

// Which kernel by default: a J1-J2 ring, and a Hubbard chain with `pairs` InterAll
// entries that move two electrons, one within each half
static void by_default(const char *name, hphi_model_desc &d) {
  hphi_engine e;
  std::vector<char> up;
  if (!plan(d, e, up)) return;
  printf("default_%s", name);
  for (int k = 1; k <= 16; k *= 2) printf(" %d", hphi_cls_wanted(&e, k));
  printf(" %d", hphi_slab_cls_pays(e));
  e.cls = 1;
  printf(" %d %d\n", hphi_cls_wanted(&e, 1), e.cls_args.nlo);
}
static void ring_default(int n, int nup) {
  std::vector<int> ij;
  for (int q = 1; q <= 2; q++)
    for (int i = 0; i < n; i++) ij.push_back(i), ij.push_back((i + q) % n);
  std::vector<double> J(2 * n, 1.0);
  hphi_model_desc d{};
  d.model = HPHI_MODEL_SPIN, d.nsite = n, d.nup = nup;
  d.n_exchange = 2 * n, d.exchange_ij = ij.data(), d.exchange_J = J.data();
  by_default(("spin_" + std::to_string(n) + "_" + std::to_string(nup)).c_str(), d);
}
// all-to-all exchange: many terms, whose couplings take LDS in a served slab
static void all_to_all_default(int n, int nup) {
  std::vector<int> ij;
  for (int i = 0; i < n; i++)
    for (int j = i + 1; j < n; j++) ij.push_back(i), ij.push_back(j);
  std::vector<double> J(ij.size() / 2, 1.0);
  hphi_model_desc d{};
  d.model = HPHI_MODEL_SPIN, d.nsite = n, d.nup = nup;
  d.n_exchange = (int)J.size(), d.exchange_ij = ij.data(), d.exchange_J = J.data();
  by_default(("all_" + std::to_string(n) + "_" + std::to_string(nup)).c_str(), d);
}
static void hubbard_default(int n, int u, int w, int pairs) {
  std::vector<int> idx, ia;
  std::vector<double> t, iv;
  for (int i = 0; i < n; i++)
    for (int s = 0; s < 2; s++) {
      const int j = (i + 1) % n, a[8] = {i, s, j, s, j, s, i, s};
      idx.insert(idx.end(), a, a + 8);
      t.insert(t.end(), {1.0, 0.0, 1.0, 0.0});
    }
  for (int s = 0; s < 2; s++)
    for (int i = 0; i < n / 2; i++)
      for (int j = i + 1; j < n / 2 && pairs > 0; j++, pairs--) {
        const int k = n / 2 + i, l = n / 2 + j, a[16] = {i, s, j, s, k, s, l, s, l, s, k, s, j, s, i, s};
        ia.insert(ia.end(), a, a + 16);
        iv.insert(iv.end(), {0.1, 0.0, 0.1, 0.0});
      }
  hphi_model_desc d{};
  d.model = HPHI_MODEL_HUBBARD, d.nsite = n, d.nup = u, d.ndown = w;
  d.n_transfer = (int)idx.size() / 4, d.transfer_idx = idx.data(), d.transfer_t = t.data();
  d.n_interall = (int)iv.size() / 2, d.interall_idx = ia.data(), d.interall_V = iv.data();
  by_default(("hubbard_" + std::to_string(n) + "_" + std::to_string(u) + "_" + std::to_string(w) + "_" +
              std::to_string(iv.size() / 4)).c_str(), d);
}
static void defaults() {
  all_to_all_default(24, 8), all_to_all_default(26, 7);
  ring_default(22, 8), ring_default(20, 10), all_to_all_default(20, 10), hubbard_default(12, 5, 6, 0), hubbard_default(12, 6, 6, 4);
  ring_default(20, 2), ring_default(28, 5), ring_default(30, 5), ring_default(32, 27), ring_default(24, 6);
  ring_default(32, 6), ring_default(24, 12);
  hubbard_default(4, 1, 1, 0), hubbard_default(6, 2, 2, 0), hubbard_default(8, 3, 3, 0), hubbard_default(8, 4, 4, 0);
  hubbard_default(8, 1, 1, 0), hubbard_default(14, 3, 3, 0), hubbard_default(16, 3, 3, 0), hubbard_default(15, 3, 3, 0);
  hubbard_default(16, 2, 5, 0), hubbard_default(12, 6, 6, 0), hubbard_default(12, 6, 6, 30), hubbard_default(16, 4, 4, 20);
  hubbard_default(16, 4, 4, 32), hubbard_default(16, 4, 4, 36), hubbard_default(12, 3, 3, 30);
}

// n sites, u + w electrons, `extra` more terms on a ring of hops: each hop assisted by
// the densities of other orbitals; is there a class layout?
static void many_terms(int n, int u, int w, int extra) {
  std::vector<int> ia, idx;
  std::vector<double> iv, t;
  for (int i = 0; i < n; i++)
    for (int s = 0; s < 2; s++) {
      const int j = (i + 1) % n, a[8] = {i, s, j, s, j, s, i, s};
      idx.insert(idx.end(), a, a + 8);
      t.insert(t.end(), {1.0, 0.0, 1.0, 0.0});
    }
  for (int i = 0; i < n; i++)
    for (int j = 0; j < n; j++)
      for (int m = 0; m < n; m++)
        for (int s = 0; s < 4 && extra > 0; s++) {
          if (i == j || m == i || m == j || i > j) continue;
          const int a[16] = {m, s / 2, m, s / 2, i, s % 2, j, s % 2, j, s % 2, i, s % 2, m, s / 2, m, s / 2};
          ia.insert(ia.end(), a, a + 16);
          iv.insert(iv.end(), {0.1, 0.0, 0.1, 0.0});
          extra -= 2;
        }
  hphi_model_desc d{};
  d.model = HPHI_MODEL_HUBBARD, d.nsite = n, d.nup = u, d.ndown = w;
  d.n_transfer = (int)idx.size() / 4, d.transfer_idx = idx.data(), d.transfer_t = t.data();
  d.n_interall = (int)iv.size() / 2, d.interall_idx = ia.data(), d.interall_V = iv.data();
  hphi_engine e;
  std::vector<char> up;
  const bool ok = plan(d, e, up);
  printf("many_terms_%d_%d_%d %d\n", n, u, (int)iv.size() / 2, ok);
}

// The autotuner's device calls, in place of the library's: building makes the
// class layout of a fresh engine available, and a timed call costs what `cost` says.
static void *layout;
static double (*cost)(const hphi_engine *e, int k);
extern "C" int hphi_diagonalcalc(hphi_engine *e, double *) {
  if (hphi_model_gc(e->model))
    for (GcPlan &P : e->gc_plan) P.npass = 1;
  else
    e->d_cls = layout;
  return 0;
}
extern "C" int hphi_time_mltply_dev(hphi_engine *e, int k, double *, const double *, int, int, double *ms) {
  *ms = cost(e, k);
  return 0;
}

static bool has(const char *report, const char *a) { return strstr(report, a) != nullptr; }

// a chain of 20 sites that no call has built yet
static bool fresh(hphi_engine &e, std::vector<char> &up) {
  static std::vector<int> ij;
  static std::vector<double> J;
  ij.clear(), J.clear();
  for (int i = 0; i < 20; i++) ij.push_back(i), ij.push_back((i + 1) % 20), J.push_back(1.0);
  hphi_model_desc d{};
  d.model = HPHI_MODEL_SPIN, d.nsite = 20, d.nup = 10;
  d.n_exchange = 20, d.exchange_ij = ij.data(), d.exchange_J = J.data();
  if (!plan(d, e, up)) return false;
  layout = e.d_cls;
  e.d_cls = nullptr;
  return true;
}

static void autotune_fresh() {
  cost = [](const hphi_engine *, int) { return 1.0; };
  for (int k : {1, 8}) {
    hphi_engine e;
    std::vector<char> up, rep(8192);
    double v = 0;
    if (fresh(e, up) && hphi_autotune(&e, k, &v, &v, 1, rep.data(), rep.size()) == 0)
      printf("autotune_fresh_%d %d\n", k, has(rep.data(), "cls"));
  }
}

static int knob(const hphi_engine *e, const char *name, int k) {
  int v = -1;
  if (hphi_engine_get_tune(e, (std::string(name) + "_k" + std::to_string(k)).c_str(), &v)) hphi_engine_get_tune(e, name, &v);
  return v;
}
static bool generic(const hphi_engine *e, int k) { return !(k == 1 ? e->use_c2 : knob(e, "use_blk", k)); }

// "<name> <class kernel or tiles in use>,<blocks per wave or 0>..." for k = 1, 2, 4, 8, 16
static void state(const char *name, const hphi_engine &e) {
  printf("%s", name);
  for (int k = 1; k <= 16; k *= 2) {
    int cb = 0, cpl = 0;
    if (!hphi_model_gc(e.model)) hphi_cls_shape(&e, k, &cb, &cpl);
    printf(" %d,%d", hphi_cls_wanted(&e, k) || hphi_gc_wanted(&e, k), cb);
  }
  printf("\n");
}

// what the autotuner leaves for every block size, by who wins the sweep for one of them
static void autotune_sizes() {
  struct Run {
    const char *name;
    int k;
    double (*cost)(const hphi_engine *e, int k);
  };
  const Run spin[] = {
      {"tuned_none", 0, nullptr},
      {"tuned_1_canon", 1, [](const hphi_engine *e, int k) { return hphi_cls_wanted(e, k) ? 2.0 : generic(e, k) ? 3.0 : 1.0; }},
      {"tuned_1_lds", 1, [](const hphi_engine *e, int k) { return hphi_cls_wanted(e, k) || generic(e, k) ? 2.0 : 1.0 + e->c2_crank; }},
      {"tuned_1_class4", 1, [](const hphi_engine *e, int k) {
         int cb, cpl;
         hphi_cls_shape(e, k, &cb, &cpl);
         return hphi_cls_wanted(e, k) && cb == 4 ? 1.0 : e->c2_tpb == 512 ? 2.0 : 3.0;
       }},
      {"tuned_1_generic", 1, [](const hphi_engine *e, int k) { return generic(e, k) ? 1.0 : 2.0; }},
      {"tuned_8_block", 8, [](const hphi_engine *e, int k) { return hphi_cls_wanted(e, k) || generic(e, k) ? 2.0 : 1.0; }},
      {"tuned_8_generic", 8, [](const hphi_engine *e, int k) { return generic(e, k) ? 1.0 : 2.0; }}};
  double v = 0;
  for (const Run &r : spin) {
    hphi_engine e;
    std::vector<char> up;
    if (!fresh(e, up)) return;
    hphi_diagonalcalc(&e, nullptr);
    cost = r.cost;
    if (r.k && hphi_autotune(&e, r.k, &v, &v, 1, nullptr, 0)) continue;
    state(r.name, e);
    if (!strcmp(r.name, "tuned_1_class4")) printf("tuned_1_class4_tpb %d\n", e.c2_tpb);  // under it: the best gather shape
  }
  const Run gc[] = {
      {"gc_none", 0, nullptr},
      {"gc_1_generic", 1, [](const hphi_engine *e, int k) { return hphi_gc_wanted(e, k) ? 2.0 : 1.0; }},
      {"gc_2_block", 2, [](const hphi_engine *e, int k) { return hphi_gc_wanted(e, k) || generic(e, k) ? 2.0 : 1.0; }},
      {"gc_8_generic", 8, [](const hphi_engine *e, int k) { return generic(e, k) ? 1.0 : 2.0; }}};
  for (const Run &r : gc) {
    hphi_engine e;
    e.model = HPHI_MODEL_SPINGC;
    hphi_diagonalcalc(&e, nullptr);
    cost = r.cost;
    if (r.k && hphi_autotune(&e, r.k, &v, &v, 1, nullptr, 0)) continue;
    state(r.name, e);
  }
  // a shape set by hand stays one
  hphi_engine e;
  std::vector<char> up;
  if (!fresh(e, up)) return;
  hphi_diagonalcalc(&e, nullptr);
  hphi_engine_tune(&e, "blk_tpb", 256);
  cost = [](const hphi_engine *, int) { return 1.0; };
  if (!hphi_autotune(&e, 1, &v, &v, 1, nullptr, 0)) state("tuned_1_by_hand", e);
}

// device memory, with room or without
static bool room = false;
extern "C" hipError_t hipMalloc(void **p, size_t n) {
  *p = room ? malloc(n) : nullptr;
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
extern "C" hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind) {
  memcpy(to, from, n);
  return hipSuccess;
}

static void tiles_without_memory() {
  std::vector<int> ij;
  std::vector<double> J(20, 1.0);
  for (int i = 0; i < 20; i++) ij.push_back(i), ij.push_back((i + 1) % 20);
  hphi_model_desc d{};
  d.model = HPHI_MODEL_SPINGC, d.nsite = 20;
  d.n_exchange = 20, d.exchange_ij = ij.data(), d.exchange_J = J.data();
  hphi_engine e;
  if (hphi_engine_prepare(&d, &e)) return;
  const int rc = hphi_gc_plan_build(&e);
  printf("tiles_without_memory %d %d\n", rc, hphi_gc_wanted(&e, 1) || hphi_gc_wanted(&e, 16));
}

// Which block sizes of a grand-canonical ring run in tiles by default: SpinGC with
// bonds to `far` neighbours and `pairs` InterAll terms, a projector times a flip; HubbardGC with hops
static void gc_default(const char *name, int n, int far, int pairs, bool hubbard) {
  std::vector<int> ij, ia, idx;
  std::vector<double> J, iv, t;
  for (int q = 1; q <= far; q++)
    for (int i = 0; i < n; i++) ij.push_back(i), ij.push_back((i + q) % n), J.push_back(1.0 / q);
  for (int q = 0; q < pairs; q++) {
    const int a = q % n, b = (q + 1 + q / n) % n;
    const int e[16] = {a, 1, a, 0, b, 1, b, 1, b, 1, b, 1, a, 0, a, 1};
    ia.insert(ia.end(), e, e + 16);
    iv.insert(iv.end(), {0.1, 0.05, 0.1, -0.05});
  }
  for (int i = 0; i < n && hubbard; i++)
    for (int s = 0; s < 2; s++) {
      const int j = (i + 1) % n, a[8] = {i, s, j, s, j, s, i, s};
      idx.insert(idx.end(), a, a + 8);
      t.insert(t.end(), {1.0, 0.0, 1.0, 0.0});
    }
  hphi_model_desc d{};
  d.model = hubbard ? HPHI_MODEL_HUBBARDGC : HPHI_MODEL_SPINGC, d.nsite = n;
  d.n_exchange = hubbard ? 0 : (int)J.size(), d.exchange_ij = ij.data(), d.exchange_J = J.data();
  d.n_interall = (int)iv.size() / 2, d.interall_idx = ia.data(), d.interall_V = iv.data();
  d.n_transfer = (int)idx.size() / 4, d.transfer_idx = idx.data(), d.transfer_t = t.data();
  printf("gc_%s", name);
  for (int forced = 0; forced < 2; forced++) {
    hphi_engine e;
    if (hphi_engine_prepare(&d, &e)) break;
    if (forced) e.gc_tile = 1;
    room = true;
    hphi_gc_plan_build(&e);
    room = false;
    for (int k = 1; k <= 16; k *= 2) printf(" %d", hphi_gc_wanted(&e, k));
    free(e.d_gcterms);
  }
  printf("\n");
}
static void gc_defaults() {
  gc_default("j1j2_18", 18, 2, 0, false), gc_default("j1j2_22", 22, 2, 0, false), gc_default("ring_24", 24, 1, 0, false);
  gc_default("pairs_18", 18, 1, 10, false), gc_default("pairs_20", 20, 1, 30, false), gc_default("pairs_22", 22, 1, 30, false);
  gc_default("hubbard_10", 10, 0, 0, true), gc_default("hubbard_11", 11, 0, 0, true);
}

int main() {
  gc_defaults();
  defaults();
  many_terms(16, 3, 3, 200), many_terms(16, 3, 3, 6000), many_terms(16, 8, 8, 6000);
  tiles_without_memory();
  autotune_fresh();
  autotune_sizes();
  block_sizes();
  high_terms();
  same_order();
  return 0;
}
