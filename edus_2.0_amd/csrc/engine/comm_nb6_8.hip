// Instantiation of the commutator kernel (comm_kernel.hpp), nb = 6 .. 8.
#include "comm_kernel.hpp"

namespace edus {

void launch_comm_nb6_8(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s)
{
    switch (nb) {
        case 6: launch_nb<6>(a, layout, kind, tile, s); break;
        case 7: launch_nb<7>(a, layout, kind, tile, s); break;
        case 8: launch_nb<8>(a, layout, kind, tile, s); break;
        default: break;
    }
}

}  // namespace edus
