// conv_mix0.hip -- convolution passes (conv_mix.hpp) for every eighth even edge
// N = 2^a 3^b 5^c 7^d from 48 to 512, counted from the first.
#include "conv_mix.hpp"

namespace fi {
ConvFn conv_part0(int n, bool fp64) {
    return conv_mix_lookup<48, 80, 120, 168, 240, 300, 392, 490>(n, fp64);
}
}  // namespace fi
