// Rules by which the host sizes and picks launches, apart from the runtime so
// that they can be checked without a device.
#pragma once
#include <stdint.h>

#include <algorithm>

namespace phk {

// Workgroups of the PGS sweeps over rows that are not packed (k_pgs_sweeps),
// which follow the packed sweeps: as many as the device holds of them. Usually
// few envs or none are left to them, and their wavefronts end after reading row
// counts; but in a batch of dense scenes most envs can have more rows than the
// packed sweeps' LDS holds, and then it takes several wavefronts per SIMD to
// cover each one's dependent chain (4096 Ants pressed into the floor, 2 steps:
// 14.0 ms with one per SIMD, 6.6 ms with all that fit; where every env is
// packed, 4096 Ants walking, 1.80 ms either way).
inline unsigned general_sweep_blocks(int64_t envs, int per_cu, int cus) {
  return (unsigned)std::min<int64_t>(envs, (int64_t)std::max(per_cu, 4) * std::max(cus, 1));
}

}  // namespace phk
