// The 2D kernels of degrees 11 to 12.
#include "launchers.hpp"

namespace exw {
void fill_2d_k11_12(DimKernels &t) { fill_dim_kernels<2, MAX_DEGREE, 11>(t); }
}  // namespace exw
