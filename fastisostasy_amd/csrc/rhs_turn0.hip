// rhs_turn0.hip -- two-launch attempt kernels (rhs_turn.hpp) for every eighth
// even length 2^a 3^b 5^c 7^d from 48 to 512, counted from the first.
#include "rhs_turn.hpp"

namespace fi {
TurnFn turn_part0(int n, bool fp64) {
    return turn_lookup<48, 80, 120, 168, 240, 300, 392, 490>(n, fp64);
}
}  // namespace fi
