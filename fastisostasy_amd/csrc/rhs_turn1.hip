// rhs_turn1.hip -- two-launch attempt kernels (rhs_turn.hpp) for every eighth
// even length 2^a 3^b 5^c 7^d from 48 to 512, counted from the second.
#include "rhs_turn.hpp"

namespace fi {
TurnFn turn_part1(int n, bool fp64) {
    return turn_lookup<50, 84, 126, 180, 250, 320, 400, 500>(n, fp64);
}
}  // namespace fi
