// Launch of the fused commutator kernel (comm_kernel.hpp).
#include <stdexcept>

#include "common.hpp"
#include "kernels.hpp"

namespace edus {

// instantiated by the comm_nb*.hip files
void launch_comm_nb1_5(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s);
void launch_comm_nb6_8(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s);
void launch_comm_nb9_10(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s);
void launch_comm_nb11_12(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s);
void launch_comm_nb13(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s);
void launch_comm_nb14(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s);
void launch_comm_nb15(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s);
void launch_comm_nb16(const CommArgs& a, int nb, int layout, int kind, int tile, hipStream_t s);

void launch_comm(int nb, int layout, int kind, int tile, const CommArgs& args, hipStream_t s)
{
    CommArgs a = args;
    a.n_add = 0;
    a.n_addf = 0;
    for (int r = 0; r < 4; ++r) {
        a.add[r] = nullptr;
        a.add_dd[r] = -1;
        a.addf[r] = nullptr;
        a.addf_dd[r] = -1;
    }
    if (args.tri && (layout != kFull || args.sigma || args.hsum || kind == kCommScalar))
        throw std::runtime_error("upper-triangle H0 and xi: FULL layout without exchange, MFMA engines only");
    if (args.nst > 0 && (args.up.ab_order > 0 || args.up.out1 == args.rho || args.up.out2 == args.rho))
        throw std::runtime_error("the stencil reads the stage input at other k-points: it must not be overwritten");
    if (args.D2 && !args.D) throw std::runtime_error("a second derivative array needs the first");
    if (args.hsum && !args.hart) throw std::runtime_error("the Hartree shift needs V with the plane sums");
    if (kind == kCommMfma32 && args.H0f) {
        if (args.sigma) throw std::runtime_error("FP32 H0 with exchange: H0 holds -Sigma[rho0] and stays FP64");
        a.addf[a.n_addf++] = args.H0f;
        for (int d = 0; d < 3; ++d)
            if (args.xif[d]) {
                a.addf[a.n_addf] = args.xif[d];
                a.addf_dd[a.n_addf++] = d;
            }
    } else {
        for (int d = 0; d < 3; ++d)
            if (args.xi[d]) {
                a.add[a.n_add] = args.xi[d];
                a.add_dd[a.n_add++] = d;
            }
        if (args.sigma) a.add[a.n_add++] = args.sigma;
    }
    switch (nb) {
        case 1: case 2: case 3: case 4: case 5: launch_comm_nb1_5(a, nb, layout, kind, tile, s); break;
        case 6: case 7: case 8: launch_comm_nb6_8(a, nb, layout, kind, tile, s); break;
        case 9: case 10: launch_comm_nb9_10(a, nb, layout, kind, tile, s); break;
        case 11: case 12: launch_comm_nb11_12(a, nb, layout, kind, tile, s); break;
        case 13: launch_comm_nb13(a, nb, layout, kind, tile, s); break;
        case 14: launch_comm_nb14(a, nb, layout, kind, tile, s); break;
        case 15: launch_comm_nb15(a, nb, layout, kind, tile, s); break;
        case 16: launch_comm_nb16(a, nb, layout, kind, tile, s); break;
        default: break;  // rejected at context creation
    }
}

}  // namespace edus
