// k_tracker_a256.hip -- instantiations of the tracker for 256 antennas (one
// translation unit per antenna count keeps builds parallel).
#include "tracker_wave.hpp"

namespace bfhip {
BF_DEFINE_TRACKER_FOR_A(256)
}  // namespace bfhip
