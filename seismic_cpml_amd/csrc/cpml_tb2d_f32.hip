// Time-blocked 2D step on one grid, float.
#include "cpml_tb2d_grid.h"

namespace cpml {
template hipError_t launch_tb2d<float>(int, int, const TB2D<float> &, hipStream_t);
template hipError_t launch_tb2d_energy<float>(const Energy<float> &, const double *, int, int,
                                            hipStream_t);
}  // namespace cpml
