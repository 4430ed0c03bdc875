// kernels_reg6.hip -- the register-table sweep kernels (reg_kernel.h) of
// lattices with 6 bilinear neighbours per site.
#include "reg_kernel.h"

namespace csmc {

template hipError_t launch_reg_s<6>(int spt, bool diag, int two_colour, int nsys, size_t lds_bytes,
                                     const WGArgs &a, hipStream_t st);

}  // namespace csmc
