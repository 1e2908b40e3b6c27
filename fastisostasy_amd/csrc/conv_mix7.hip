// conv_mix7.hip -- convolution passes (conv_mix.hpp) for every eighth even edge
// N = 2^a 3^b 5^c 7^d from 48 to 512, counted from the eighth.
#include "conv_mix.hpp"

namespace fi {
ConvFn conv_part7(int n, bool fp64) {
    return conv_mix_lookup<72, 112, 162, 224, 294, 384, 486>(n, fp64);
}
}  // namespace fi
