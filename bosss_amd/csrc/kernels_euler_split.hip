// Cell-split forms of the Euler (Rusanov and HLLC) 3D p = 3 kernels, compiled in their own
// translation unit (scheduling flags of the other p = 3 kernels; built in parallel with them).
#include <vector>

#include "registry.hpp"

namespace bosss {
#define BOSSS_EULER_SPLIT(H)                                                                                   \
  template __global__ void kt_forward<FormEuler<3, H>, 3, 3, 5, double, MODE_RES, true>(TArgs<double>);       \
  template __global__ void kt_forward<FormEuler<3, H>, 3, 3, 5, float, MODE_RES, true>(TArgs<float>);         \
  template __global__ void kt_jvp_euler<FormEuler<3, H>, 3, 3, 5, double, true>(TArgs<double>);               \
  template __global__ void kt_jvp_euler<FormEuler<3, H>, 3, 3, 5, float, true>(TArgs<float>);                 \
  template __global__ void kt_vjp_euler<FormEuler<3, H>, 3, 3, 5, double, false, true>(TArgs<double>);        \
  template __global__ void kt_vjp_euler<FormEuler<3, H>, 3, 3, 5, float, false, true>(TArgs<float>);          \
  template __global__ void kt_vjp_euler<FormEuler<3, H>, 3, 3, 5, double, true, true>(TArgs<double>);         \
  template __global__ void kt_vjp_euler<FormEuler<3, H>, 3, 3, 5, float, true, true>(TArgs<float>);
BOSSS_EULER_SPLIT(false)
BOSSS_EULER_SPLIT(true)
#undef BOSSS_EULER_SPLIT
}  // namespace bosss
