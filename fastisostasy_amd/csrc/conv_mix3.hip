// conv_mix3.hip -- convolution passes (conv_mix.hpp) for every eighth even edge
// N = 2^a 3^b 5^c 7^d from 48 to 512, counted from the fourth.
#include "conv_mix.hpp"

namespace fi {
ConvFn conv_part3(int n, bool fp64) {
    return conv_mix_lookup<56, 96, 140, 196, 256, 336, 432, 512>(n, fp64);
}
}  // namespace fi
