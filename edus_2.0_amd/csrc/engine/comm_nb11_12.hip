// Instantiation of the commutator kernel (comm_kernel.hpp), nb = 11 .. 12.
#include "comm_kernel.hpp"

namespace edus {

void launch_comm_nb11_12(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s)
{
    switch (nb) {
        case 11: launch_nb<11>(a, layout, kind, tile, s); break;
        case 12: launch_nb<12>(a, layout, kind, tile, s); break;
        default: break;
    }
}

}  // namespace edus
