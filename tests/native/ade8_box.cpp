// Prints the pair box of the ADE-RK4 step (cpml_ade8_split.h): nx ny npml bytes.
#include <cstdio>
#include <cstdlib>

#include "../../seismic_cpml_amd/csrc/cpml_ade8_split.h"

int main(int, char **a) {
  const int nx = std::atoi(a[1]), ny = std::atoi(a[2]), npml = std::atoi(a[3]);
  const cpml::AdeBox b = std::atoi(a[4]) == 4 ? cpml::ade_pair_box<float>(nx, ny, npml)
                                              : cpml::ade_pair_box<double>(nx, ny, npml);
  std::printf("%d %d %d %d\n", b.x0, b.x1, b.y0, b.y1);
}
