// Instantiation of the commutator kernel (comm_kernel.hpp), nb = 15.
#include "comm_kernel.hpp"

namespace edus {

void launch_comm_nb15(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s)
{
    switch (nb) {
        case 15: launch_nb<15>(a, layout, kind, tile, s); break;
        default: break;
    }
}

}  // namespace edus
