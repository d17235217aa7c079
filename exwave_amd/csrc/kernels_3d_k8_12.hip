// The 3D kernels of degrees 8 to 12.
#include "launchers.hpp"

namespace exw {
void fill_3d_k8_12(DimKernels &t) { fill_dim_kernels<3, MAX_DEGREE_3D, 8>(t); }
}  // namespace exw
