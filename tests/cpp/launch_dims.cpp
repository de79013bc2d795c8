// spread_waves (csrc/launch_dims.h): prints, for every launch of 1 .. 16 * cus wavefronts, how far the fullest CU is from an
// even split (worst case over the launches), the largest block, and the block size of a launch that fills the device.
#include "launch_dims.h"

#include <algorithm>
#include <cstdio>

int main() {
    for (int cus : {256, 64, 1}) {
        for (int full : {8, 16}) {
            int64_t over = 0;
            int largest = 0;
            for (int64_t waves = 1; waves <= 16 * (int64_t) cus; waves++) {
                const int b = bf16n::dev::spread_waves(waves, cus, full);
                const int64_t blocks = (waves + b - 1) / b, fullest = b * ((blocks + cus - 1) / cus);
                const int64_t even = std::max<int64_t>(4, (waves + cus - 1) / cus);
                over = std::max(over, fullest - even);
                largest = std::max(largest, b);
            }
            std::printf("%d %d: %lld %d %d\n", cus, full, (long long) over, largest, bf16n::dev::spread_waves(16 * cus, cus, full));
        }
    }
    // just above the sizes that the device takes in blocks of eight, one per CU: 2,064 wavefronts are 230 blocks of nine, not
    // 129 of sixteen nor 258 of eight (two on two CUs); 3,880 fill the device either way
    std::printf("%d %d %d\n", bf16n::dev::spread_waves(2064, 256, 16), bf16n::dev::spread_waves(2064, 256, 8), bf16n::dev::spread_waves(3880, 256, 8));
    return 0;
}
