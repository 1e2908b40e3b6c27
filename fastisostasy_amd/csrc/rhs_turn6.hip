// rhs_turn6.hip -- two-launch attempt kernels (rhs_turn.hpp) for every eighth
// even length 2^a 3^b 5^c 7^d from 48 to 512, counted from the seventh.
#include "rhs_turn.hpp"

namespace fi {
TurnFn turn_part6(int n, bool fp64) {
    return turn_lookup<70, 108, 160, 216, 288, 378, 480>(n, fp64);
}
}  // namespace fi
