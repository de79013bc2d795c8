// Launch shapes that are plain arithmetic (no HIP): shared by the launchers and checked on the host.
#pragma once

#include <cstdint>

namespace bf16n {
namespace dev {

// Wavefronts per block of a launch of `waves` wavefronts (at most sixteen per CU) whose blocks have `full` of them where they
// fill the device.  Where blocks of `full` would put more on one CU than an even split does, the launch is one block per
// CU of as many as that split takes, four at least (as in every wave64 product: each block stages the table for itself).
// k_w64_mmv_lds, us with blocks of 8 or 16 everywhere / with this rule: 66048 x 2048 (2,064 wavefronts), 2 / 5 / 7 BF16
// columns 53.5 / 69.4 / 81.3 -> 48.4 / 59.6 / 69.6; 98304 x 2048, 4: 67.4 -> 63.4; 10240 x 2048, 8: 17.9 -> 15.1; 4112 x 4096,
// 4 FP32 columns: 14.2 -> 12.1; 16448 x 4096, 2 / 8 BF16 columns: 29.4 / 50.7 -> 25.7 / 38.3; 66048 x 4096, 8: 183 -> 133.
inline int spread_waves(int64_t waves, int cus, int full) {
    const auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
    const int64_t even = up(waves, cus) < 4 ? 4 : up(waves, cus);
    return even < full * up(up(waves, full), cus) ? (int) even : full;
}

} // namespace dev
} // namespace bf16n
