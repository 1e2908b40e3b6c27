// conv_mix2.hip -- convolution passes (conv_mix.hpp) for every eighth even edge
// N = 2^a 3^b 5^c 7^d from 48 to 512, counted from the third.
#include "conv_mix.hpp"

namespace fi {
ConvFn conv_part2(int n, bool fp64) {
    return conv_mix_lookup<54, 90, 128, 192, 252, 324, 420, 504>(n, fp64);
}
}  // namespace fi
