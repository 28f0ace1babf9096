// Instantiation of the commutator kernel (comm_kernel.hpp), nb = 16.
#include "comm_kernel.hpp"

namespace edus {

void launch_comm_nb16(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s)
{
    switch (nb) {
        case 16: launch_nb<16>(a, layout, kind, tile, s); break;
        default: break;
    }
}

}  // namespace edus
