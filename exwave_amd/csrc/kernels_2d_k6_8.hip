// The 2D kernels of degrees 6 to 8.
#include "launchers.hpp"

namespace exw {
void fill_2d_k6_8(DimKernels &t) { fill_dim_kernels<2, 8, 6>(t); }
}  // namespace exw
