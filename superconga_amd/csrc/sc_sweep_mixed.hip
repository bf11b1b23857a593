// sc_sweep_mixed.hip -- the sweep kernels with FP32 stepping.
#include "sc_sweep.hpp"

namespace scamd {

bool launchSweepMixed(int el, int waves, const SweepArgs &a, int slots, hipStream_t stream,
                     bool keldysh) {
  return launchSweepOf<float>(el, waves, a, slots, stream, keldysh);
}

} // namespace scamd
