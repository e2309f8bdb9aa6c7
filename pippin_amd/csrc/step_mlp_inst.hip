// The step kernel with the learned warm start, one instance per object file
// (see step_inst.hip).
#include <hip/hip_runtime.h>

#include "kstep.hpp"
#include "spec_models.hpp"
#include "step_kernels.hpp"

#define PH_CAT_(a, b) a##b
#define PH_CAT(a, b) PH_CAT_(a, b)

namespace phk {
const void* PH_CAT(mlp_kernel_, PH_TAG)() { return (const void*)k_step_mlp<PH_K, PH_MT>; }
}  // namespace phk
