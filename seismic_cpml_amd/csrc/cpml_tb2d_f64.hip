// Time-blocked 2D step on one grid, double.
#include "cpml_tb2d_grid.h"

namespace cpml {
template hipError_t launch_tb2d<double>(int, int, const TB2D<double> &, hipStream_t);
template hipError_t launch_tb2d_energy<double>(const Energy<double> &, const double *, int, int,
                                            hipStream_t);
}  // namespace cpml
