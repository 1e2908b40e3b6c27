// rhs_turn7.hip -- two-launch attempt kernels (rhs_turn.hpp) for every eighth
// even length 2^a 3^b 5^c 7^d from 48 to 512, counted from the eighth.
#include "rhs_turn.hpp"

namespace fi {
TurnFn turn_part7(int n, bool fp64) {
    return turn_lookup<72, 112, 162, 224, 294, 384, 486>(n, fp64);
}
}  // namespace fi
