// k_tracker_a128.hip -- instantiations of the tracker for 128 antennas (one
// translation unit per antenna count keeps builds parallel).
#include "tracker_wave.hpp"

namespace bfhip {
BF_DEFINE_TRACKER_FOR_A(128)
}  // namespace bfhip
