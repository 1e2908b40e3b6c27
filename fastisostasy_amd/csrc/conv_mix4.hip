// conv_mix4.hip -- convolution passes (conv_mix.hpp) for every eighth even edge
// N = 2^a 3^b 5^c 7^d from 48 to 512, counted from the fifth.
#include "conv_mix.hpp"

namespace fi {
ConvFn conv_part4(int n, bool fp64) {
    return conv_mix_lookup<60, 98, 144, 200, 270, 350, 448>(n, fp64);
}
}  // namespace fi
