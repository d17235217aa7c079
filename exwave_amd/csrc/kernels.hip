// kernels.hip -- the kernel tables of both dimensions (degrees 1..MAX_DEGREE,
// FP64/FP32 operator arithmetic, Cartesian/general geometry).
#include "launchers.hpp"

namespace exw {
const DimKernels &kernels_2d() {
  static const DimKernels table = [] {
    DimKernels t{};
    t.coef = launch_cart_coef<2>;
    fill_2d_k1_5(t);
    fill_2d_k6_8(t);
    fill_2d_k9_10(t);
    fill_2d_k11_12(t);
    return t;
  }();
  return table;
}
const DimKernels &kernels_3d() {
  static const DimKernels table = [] {
    DimKernels t{};
    t.coef = launch_cart_coef<3>;
    fill_3d_k1_4(t);
    fill_3d_k5_7(t);
    fill_3d_k8_12(t);
    return t;
  }();
  return table;
}
}  // namespace exw
