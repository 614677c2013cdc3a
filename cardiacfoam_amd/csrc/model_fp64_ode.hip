// FP64 instantiations of the adaptive solvers' kernels (RKF45, OpenFOAM's Euler).
#include "batch_kernels.hpp"

namespace cg {
CG_DEFINE_MODEL_ENTRIES(double, true, fp64_ode)
CG_DEFINE_BATCH_ENTRY(double, true, fp64_ode)
} // namespace cg
