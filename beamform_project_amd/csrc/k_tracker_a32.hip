// k_tracker_a32.hip -- instantiations of the tracker for 32 antennas (one
// translation unit per antenna count keeps builds parallel).
#include "tracker_wave.hpp"

namespace bfhip {
BF_DEFINE_TRACKER_FOR_A(32)
}  // namespace bfhip
