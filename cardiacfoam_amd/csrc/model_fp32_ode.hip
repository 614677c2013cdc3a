// FP32 instantiations of the adaptive solvers' kernels (RKF45, OpenFOAM's Euler), compiled
// with the approximate functions of model_fp32.hip.
#include "batch_kernels.hpp"

namespace cg {
CG_DEFINE_MODEL_ENTRIES(float, true, fp32_ode)
CG_DEFINE_BATCH_ENTRY(float, true, fp32_ode)
} // namespace cg
