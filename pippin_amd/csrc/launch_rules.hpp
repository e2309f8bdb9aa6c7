// Rules by which the host sizes and picks launches, apart from the runtime so
// that they can be checked without a device.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <cstdlib>
#include <vector>

#include "../../include/pippin_hip.h"

namespace phk {

// The shape a sim starts with: as many envs per wavefront as fit 64 KiB of LDS
// (lds_bytes each), on the grid schedule. PGS models whose rows pack and can meet
// on the same dofs (split) start with the split step: fused, the sweeps of several
// envs wait for each other at every row (Ant, 4096 envs, 4 steps: 9.9 ms fused,
// 1.84 ms split; six-body pile, 8192 envs: 125 and 11.0 ms). Where each dof block
// has one row at most, a sweep or two is all there is, and four launches a step
// are more than one (1024 envs, 20 steps: cartpole 530 us fused, 907 split; a
// hinge with a limit 485 and 892). envs_per_wave (PIPPIN_HIP_ENVS_PER_WG; null: not set)
// asks for 1, 2 or 4 envs on the grid schedule and is ignored where it is another
// value or more than the device's LDS per workgroup, lds_max, holds.
struct StartShape {
  int envs_per_wave, schedule;
};
inline StartShape start_shape(int64_t lds_bytes, bool split, int64_t lds_max, const char* envs_per_wave) {
  if (envs_per_wave) {
    const int k = std::atoi(envs_per_wave);
    if ((k == 1 || k == 2 || k == 4) && k * lds_bytes <= lds_max) return {k, PH_SCHED_GRID};
  }
  if (split) return {1, PH_SCHED_PGS_SPLIT};
  for (int k : {4, 2})
    if (k * lds_bytes <= 64 * 1024) return {k, PH_SCHED_GRID};
  return {1, PH_SCHED_GRID};
}

// Envs per wavefront of the split PGS step's front and back and of the pose
// kernel, for envs of lds_bytes each. A round of wavefronts takes about
// 1 : 1.2 : 1.5 for 1, 2 and 4 envs (the generic Ant kernel: 344, 410 and 520 us
// per 4-step round), so the fewest rounds win once the device is full, and one
// env per wavefront while it is not.
inline int envs_per_wave_by_rounds(int64_t lds_bytes, int cus, int64_t envs) {
  const double weight[] = {1.0, 1.2, 1.5};
  int best = 1;
  double cost = 0.0;
  for (int i = 0; i < 3; i++) {
    const int K = 1 << i;
    const int64_t lds = K * lds_bytes;
    if (lds > 64 * 1024) break;
    const int64_t resident = (int64_t)cus * std::min<int64_t>(4, 160 * 1024 / lds), waves = (envs + K - 1) / K;
    const double c = weight[i] * (double)((waves + resident - 1) / resident);
    if (i == 0 || c < cost) {
      best = K;
      cost = c;
    }
  }
  return best;
}

// Envs per wavefront of the step with the learned warm start: the launch
// shape's, except that the split PGS step's has none to give (its front and back
// pick theirs by the range) and the learned step runs fused. Several envs of a
// wavefront wait for each other at every row there, so with several dof blocks
// one env is the best throughout (six-body pile, 4096 envs, 4 steps: 11.4 ms with
// 1, 37 with 2, 46 with 4; three boxes 3.7, 6.4, 6.9). A single tree has few rows,
// and the rounds decide (Ant, 1024 envs: 2.2, 3.7, 4.0 ms; 4096: 8.5, 7.9, 5.3).
inline int learned_envs_per_wave(int shape_envs, bool split, int nblock, int64_t lds_bytes, int cus, int64_t envs) {
  if (!split) return shape_envs;
  return nblock > 1 ? 1 : envs_per_wave_by_rounds(lds_bytes, cus, envs);
}

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

// Whether a launch carries its own time stamps. A grid launch of the plain step
// is a single dispatch and can, which saves two event records (cartpole, one
// env: 30 us by the dispatch, 33 to 39 us between records). An autotuning's trials
// do not: other schedules are sequences that are timed between records, and on
// launches of some tens of microseconds the two clocks differ by more than the
// candidates.
inline bool timed_by_dispatch(bool plain, bool trial, bool grid) { return plain && !trial && grid; }

// Which of an autotuning's candidates to keep, by the times of their timed
// launches (one entry per round; none: not timed): the lowest median. prefer
// names a candidate to take instead of another, -1 for none: it is taken where
// the trials do not tell the two apart, that is where its fastest launch was no
// slower than the median of the lowest. Returns -1 when nothing was timed.
inline int tune_choice(const std::vector<std::vector<double>>& ms, const std::vector<int>& prefer) {
  int best = -1;
  double least = 0.0;
  for (size_t c = 0; c < ms.size(); c++) {
    if (ms[c].empty()) continue;
    std::vector<double> v = ms[c];
    std::sort(v.begin(), v.end());
    const double med = v[v.size() / 2];
    if (best < 0 || med < least) {
      least = med;
      best = (int)c;
    }
  }
  if (best < 0 || prefer[best] < 0) return best;
  const std::vector<double>& v = ms[prefer[best]];
  return !v.empty() && *std::min_element(v.begin(), v.end()) <= least ? prefer[best] : best;
}

}  // namespace phk
