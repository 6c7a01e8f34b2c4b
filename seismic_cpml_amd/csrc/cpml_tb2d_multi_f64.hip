// Time-blocked 2D step on many grids, double.
#include "cpml_tb2d_multi.h"

namespace cpml {
template hipError_t launch_tb2d_multi<double>(int, int, const TB2D<double> *, const int4 *,
                                           const int (&)[4], int, int, hipStream_t);
}  // namespace cpml
