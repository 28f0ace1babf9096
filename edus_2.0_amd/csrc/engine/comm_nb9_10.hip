// Instantiation of the commutator kernel (comm_kernel.hpp), nb = 9 .. 10.
#include "comm_kernel.hpp"

namespace edus {

void launch_comm_nb9_10(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s)
{
    switch (nb) {
        case 9: launch_nb<9>(a, layout, kind, tile, s); break;
        case 10: launch_nb<10>(a, layout, kind, tile, s); break;
        default: break;
    }
}

}  // namespace edus
