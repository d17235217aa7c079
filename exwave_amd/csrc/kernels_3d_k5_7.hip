// The 3D kernels of degrees 5 to 7.
#include "launchers.hpp"

namespace exw {
void fill_3d_k5_7(DimKernels &t) { fill_dim_kernels<3, 7, 5>(t); }
}  // namespace exw
