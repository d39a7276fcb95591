// The FP64 instantiations of the x faces with the update (k_xlast).
#include "fvg_kernels_impl.hpp"

namespace fvg {

#define FVG_XLAST(M, WHAT)                                                                                             \
    template __global__ void k_xlast<M, WHAT, true, double>(KP, int, const double*, const double*, double*);  \
    template __global__ void k_xlast<M, WHAT, false, double>(KP, int, const double*, const double*, double*);
FVG_XLAST(MODE_PLAIN, 1)
FVG_XLAST(MODE_PLAIN, 2)
FVG_XLAST(MODE_PLAIN, 3)
FVG_XLAST(MODE_LEARNED, LF_STORE)
FVG_XLAST(MODE_LEARNED, LF_KEPT)

}   // namespace fvg
