// conv_mix6.hip -- convolution passes (conv_mix.hpp) for every eighth even edge
// N = 2^a 3^b 5^c 7^d from 48 to 512, counted from the seventh.
#include "conv_mix.hpp"

namespace fi {
ConvFn conv_part6(int n, bool fp64) {
    return conv_mix_lookup<70, 108, 160, 216, 288, 378, 480>(n, fp64);
}
}  // namespace fi
