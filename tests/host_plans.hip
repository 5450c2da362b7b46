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

int main() {
  block_sizes();
  return 0;
}
