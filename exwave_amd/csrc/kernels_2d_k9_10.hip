// The 2D kernels of degrees 9 to 10.
#include "launchers.hpp"

namespace exw {
void fill_2d_k9_10(DimKernels &t) { fill_dim_kernels<2, 10, 9>(t); }
}  // namespace exw
