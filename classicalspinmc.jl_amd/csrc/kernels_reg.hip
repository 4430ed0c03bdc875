// kernels_reg.hip -- picks the register-table sweep kernel (reg_kernel.h,
// compiled per neighbour count).
#include "kernels.h"

namespace csmc {

template <int K2C>
hipError_t launch_reg_s(int spt, bool diag, int two_colour, int nsys, size_t lds_bytes, const WGArgs &a,
                        hipStream_t st);

hipError_t launch_wg_reg(int k2c, int spt, bool diag, int two_colour, int nsys, size_t lds_bytes,
                         const WGArgs &a, hipStream_t st) {
    if (k2c == 3) return launch_reg_s<3>(spt, diag, two_colour, nsys, lds_bytes, a, st);
    if (k2c == 4) return launch_reg_s<4>(spt, diag, two_colour, nsys, lds_bytes, a, st);
    if (k2c == 6) return launch_reg_s<6>(spt, diag, two_colour, nsys, lds_bytes, a, st);
    return hipErrorInvalidValue;
}

}  // namespace csmc
