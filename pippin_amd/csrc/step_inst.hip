// One instance of the step kernels per object file, so that the build compiles
// them side by side: PH_K envs per wavefront, PH_MT the model type (DModel, or
// a model-specialised struct), PH_TAG the suffix of the functions below.
#include <hip/hip_runtime.h>

#include "kstep.hpp"
#include "spec_models.hpp"
#include "step_kernels.hpp"

#define PH_CAT_(a, b) a##b
#define PH_CAT(a, b) PH_CAT_(a, b)

namespace phk {
const void* PH_CAT(step_kernel_, PH_TAG)() { return (const void*)k_step<PH_K, PH_MT>; }
const void* PH_CAT(ws_kernel_, PH_TAG)() { return (const void*)k_step_ws<PH_K, PH_MT>; }
}  // namespace phk
