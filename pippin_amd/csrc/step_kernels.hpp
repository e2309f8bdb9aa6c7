// The step kernels' instances (step_inst.hip, step_mlp_inst.hip, pgs_inst.hip), each compiled
// in an object file of its own: K = 1, 2 or 4 envs per wavefront with run-time
// sizes, and K = 4 with the Ant's compile-time sizes.
#pragma once

namespace phk {

#define PH_INST(tag)                  \
  const void* step_kernel_##tag();    \
  const void* ws_kernel_##tag();      \
  const void* mlp_kernel_##tag();
PH_INST(k1)
PH_INST(k2)
PH_INST(k4)
PH_INST(ant)
#undef PH_INST
#define PH_INST(tag)              \
  const void* pgs_front_##tag();  \
  const void* pgs_back_##tag();
PH_INST(k1)
PH_INST(k2)
PH_INST(k4)
#undef PH_INST

inline const void* pgs_front_kernel(int K) { return K == 4 ? pgs_front_k4() : K == 2 ? pgs_front_k2() : pgs_front_k1(); }
inline const void* pgs_back_kernel(int K) { return K == 4 ? pgs_back_k4() : K == 2 ? pgs_back_k2() : pgs_back_k1(); }

inline const void* step_kernel(int K, int spec) {
  if (spec == 1 && K == 4) return step_kernel_ant();
  return K == 4 ? step_kernel_k4() : K == 2 ? step_kernel_k2() : step_kernel_k1();
}
inline const void* ws_kernel(int K, int spec) {
  if (spec == 1 && K == 4) return ws_kernel_ant();
  return K == 4 ? ws_kernel_k4() : K == 2 ? ws_kernel_k2() : ws_kernel_k1();
}
inline const void* mlp_kernel(int K, int spec) {
  if (spec == 1 && K == 4) return mlp_kernel_ant();
  return K == 4 ? mlp_kernel_k4() : K == 2 ? mlp_kernel_k2() : mlp_kernel_k1();
}

}  // namespace phk
