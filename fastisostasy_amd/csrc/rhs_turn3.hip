// rhs_turn3.hip -- two-launch attempt kernels (rhs_turn.hpp) for every eighth
// even length 2^a 3^b 5^c 7^d from 48 to 512, counted from the fourth.
#include "rhs_turn.hpp"

namespace fi {
TurnFn turn_part3(int n, bool fp64) {
    return turn_lookup<56, 96, 140, 196, 256, 336, 432, 512>(n, fp64);
}
}  // namespace fi
