// The 3D kernels of degrees 1 to 4.
#include "launchers.hpp"

namespace exw {
void fill_3d_k1_4(DimKernels &t) { fill_dim_kernels<3, 4, 1>(t); }
}  // namespace exw
