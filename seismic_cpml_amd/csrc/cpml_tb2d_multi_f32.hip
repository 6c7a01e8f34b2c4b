// Time-blocked 2D step on many grids, float.
#include "cpml_tb2d_multi.h"

namespace cpml {
template hipError_t launch_tb2d_multi<float>(int, int, const TB2D<float> *, const int4 *,
                                           const int (&)[4], int, int, hipStream_t);
}  // namespace cpml
