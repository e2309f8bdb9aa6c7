// The front and back of the split PGS step, one instance per object file (see
// step_inst.hip).
#include <hip/hip_runtime.h>

#include "kstep.hpp"
#include "step_kernels.hpp"

#define PH_CAT_(a, b) a##b
#define PH_CAT(a, b) PH_CAT_(a, b)

namespace phk {
const void* PH_CAT(pgs_front_, PH_TAG)() { return (const void*)k_pgs_front<PH_K>; }
const void* PH_CAT(pgs_back_, PH_TAG)() { return (const void*)k_pgs_back<PH_K>; }
}  // namespace phk
