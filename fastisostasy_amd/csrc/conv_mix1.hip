// conv_mix1.hip -- convolution passes (conv_mix.hpp) for every eighth even edge
// N = 2^a 3^b 5^c 7^d from 48 to 512, counted from the second.
#include "conv_mix.hpp"

namespace fi {
ConvFn conv_part1(int n, bool fp64) {
    return conv_mix_lookup<50, 84, 126, 180, 250, 320, 400, 500>(n, fp64);
}
}  // namespace fi
