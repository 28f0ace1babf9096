// Instantiation of the commutator kernel (comm_kernel.hpp), nb = 14.
#include "comm_kernel.hpp"

namespace edus {

void launch_comm_nb14(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s)
{
    switch (nb) {
        case 14: launch_nb<14>(a, layout, kind, tile, s); break;
        default: break;
    }
}

}  // namespace edus
