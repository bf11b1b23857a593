// sc_sweep_fp64.hip -- the sweep kernels with FP64 stepping.
#include "sc_sweep.hpp"

namespace scamd {

bool launchSweepFp64(int el, int waves, const SweepArgs &a, int slots, hipStream_t stream,
                     bool keldysh) {
  return launchSweepOf<double>(el, waves, a, slots, stream, keldysh);
}

} // namespace scamd
