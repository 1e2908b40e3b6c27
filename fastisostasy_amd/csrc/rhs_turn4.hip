// rhs_turn4.hip -- two-launch attempt kernels (rhs_turn.hpp) for every eighth
// even length 2^a 3^b 5^c 7^d from 48 to 512, counted from the fifth.
#include "rhs_turn.hpp"

namespace fi {
TurnFn turn_part4(int n, bool fp64) {
    return turn_lookup<60, 98, 144, 200, 270, 350, 448>(n, fp64);
}
}  // namespace fi
