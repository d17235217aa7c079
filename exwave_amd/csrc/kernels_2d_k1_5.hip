// The 2D kernels of degrees 1 to 5.
#include "launchers.hpp"

namespace exw {
void fill_2d_k1_5(DimKernels &t) { fill_dim_kernels<2, 5, 1>(t); }
}  // namespace exw
