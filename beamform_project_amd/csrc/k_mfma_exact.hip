// k_mfma_exact.hip -- the MFMA fixed-grid beamformer with float weights:
// every weight as three bfloat16 slices that add up to it exactly (PARTS = 3
// of mfma_fused.hpp), for the FP32, DIRECT and TILED selectors.
//
// Bound by the matrix cores: 12 MFMAs of 16 cycles per 16 spectra, 8 beams
// and 64 antennas, against 8 for the fp16 split.  The FP32 FMA kernel it
// replaces was bound by its FMAs (A = 64, T = 15360, B = 64, S = 10, tiled:
// 1.88 ms, 90 TFLOP/s; here 0.34 ms, 500 TFLOP/s, 0.6 of the error).
#include "mfma_fused.hpp"

namespace bfhip {
namespace {

// Three slices of A / 16 k-steps cost 3 A / 4 registers per 8-beam N-tile:
// two N-tiles per wave up to 64 antennas, one above.
template <int A>
void launch_a(hipStream_t stream, const MfmaLaunch& L) {
    MfmaConfig cfg;
    cfg.waves = 4;
    cfg.db = 0;
    cfg.nt = A <= 64 && L.B > 32 ? 2 : 1;
    cfg.resident = A == 256 ? 512 : 768;
    if constexpr (A <= 64) {
        if (cfg.nt == 2) {
            mfma_detail::launch_shape<A, 2, 4, 3, false>(stream, L, cfg);
            return;
        }
    }
    mfma_detail::launch_shape<A, 1, 4, 3, false>(stream, L, cfg);
}

}  // namespace

void launch_mfma_exact(hipStream_t stream, const MfmaLaunch& L, int A) {
    switch (A) {
    case 32: launch_a<32>(stream, L); break;
    case 64: launch_a<64>(stream, L); break;
    case 128: launch_a<128>(stream, L); break;
    case 256: launch_a<256>(stream, L); break;
    default: invalid("n_ant must be 32, 64, 128, or 256");
    }
    hip_check(hipGetLastError(), "mfma_fused_kernel launch");
}

}  // namespace bfhip
