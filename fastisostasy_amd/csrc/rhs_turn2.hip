// rhs_turn2.hip -- two-launch attempt kernels (rhs_turn.hpp) for every eighth
// even length 2^a 3^b 5^c 7^d from 48 to 512, counted from the third.
#include "rhs_turn.hpp"

namespace fi {
TurnFn turn_part2(int n, bool fp64) {
    return turn_lookup<54, 90, 128, 192, 252, 324, 420, 504>(n, fp64);
}
}  // namespace fi
