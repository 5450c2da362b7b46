// Host-side plans of the H·v kernels, without a device: prints one "name value"
// line per check for tests/test_host_plans.py.
#include <cstdio>
#include <cstring>
#include <vector>

#include "engine_internal.h"
#include "hphi_amd.h"

int hphi_engine_prepare(const hphi_model_desc *d, hphi_engine *e);

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

// The autotuner's device calls, in place of the library's: building makes the
// class layout of a fresh engine available, and a timed call costs what `cost` says.
static void *layout;
static double (*cost)(const hphi_engine *e, int k);
extern "C" int hphi_diagonalcalc(hphi_engine *e, double *) {
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

int main() {
  autotune_fresh();
  block_sizes();
  high_terms();
  same_order();
  return 0;
}
