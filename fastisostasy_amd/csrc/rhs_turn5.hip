// rhs_turn5.hip -- two-launch attempt kernels (rhs_turn.hpp) for every eighth
// even length 2^a 3^b 5^c 7^d from 48 to 512, counted from the sixth.
#include "rhs_turn.hpp"

namespace fi {
TurnFn turn_part5(int n, bool fp64) {
    return turn_lookup<64, 100, 150, 210, 280, 360, 450>(n, fp64);
}
}  // namespace fi
