// Chunk depths that the autotuner times (cpml_internal.h) over random grids: the
// default of cpml_gpu_set_time_block is among them, each once, in ascending order.
#include <cstdio>
#include <random>

#include "../../seismic_cpml_amd/csrc/cpml_internal.h"

int main() {
  std::mt19937 rng(3);
  auto pick = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
  int below = 0, above = 0;
  for (int q = 0; q < 20000; ++q) {
    const int ndim = pick(2, 3), es = 4 * pick(1, 2), order = ndim == 3 ? 2 : 2 << pick(0, 2);
    const int nx = pick(2, 900), ny = pick(2, 900), nz = pick(2, 900);
    const int nt = pick(1, ndim == 3 ? 2 : cpml::tb2d_max_nt(order, es));
    const int ow = cpml::tb_default_strip(nt * (order - 1), es);
    const int def = cpml::tb_default_chunk(ndim, nx, ny, nz, es, nt, ow);
    const std::vector<int> c = cpml::tb_autotune_chunks(ndim, nx, ny, nz, es, order, nt);
    bool found = false, ascending = true;
    for (size_t k = 0; k < c.size(); ++k) {
      found |= c[k] == def;
      ascending &= c[k] > 0 && (k == 0 || c[k] > c[k - 1]);
    }
    if (ow < 1 || ow > 64 - 2 * nt * (order - 1) || !found || !ascending) {
      std::printf("%dD %d x %d x %d, %d bytes, order %d, %d steps\n", ndim, nx, ny, nz, es, order, nt);
      return 1;
    }
    if (ndim == 3) ++(def < 32 ? below : above);
  }
  std::printf("%d %d\n", below, above);
  return below && above ? 0 : 1;
}
