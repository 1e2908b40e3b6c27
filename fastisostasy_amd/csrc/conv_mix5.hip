// conv_mix5.hip -- convolution passes (conv_mix.hpp) for every eighth even edge
// N = 2^a 3^b 5^c 7^d from 48 to 512, counted from the sixth.
#include "conv_mix.hpp"

namespace fi {
ConvFn conv_part5(int n, bool fp64) {
    return conv_mix_lookup<64, 100, 150, 210, 280, 360, 450>(n, fp64);
}
}  // namespace fi
