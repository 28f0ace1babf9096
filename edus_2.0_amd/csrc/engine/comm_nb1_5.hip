// Instantiation of the commutator kernel (comm_kernel.hpp), nb = 1 .. 5.
#include "comm_kernel.hpp"

namespace edus {

void launch_comm_nb1_5(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s)
{
    switch (nb) {
        case 1: launch_nb<1>(a, layout, kind, tile, s); break;
        case 2: launch_nb<2>(a, layout, kind, tile, s); break;
        case 3: launch_nb<3>(a, layout, kind, tile, s); break;
        case 4: launch_nb<4>(a, layout, kind, tile, s); break;
        case 5: launch_nb<5>(a, layout, kind, tile, s); break;
        default: break;
    }
}

}  // namespace edus
