// The FP32-flux instantiations of the residual kernels (float reconstruction and fluxes, FP64 state).
#include "fvg_kernels_impl.hpp"

namespace fvg {

#define FVG_UPDATE(NV, UPD) template __global__ void k_update<NV, UPD, float>(KP, const double*, const double*, double*);
#define FVG_INST(NV)                     \
    template __global__ void k_cells<NV, true, float>(KP);  \
    template __global__ void k_cells<NV, false, float>(KP); \
    FVG_UPDATE(NV, UPD_RESIDUAL)         \
    FVG_UPDATE(NV, UPD_AXPY)             \
    FVG_UPDATE(NV, UPD_RK2_2)            \
    FVG_UPDATE(NV, UPD_RK3_2)            \
    FVG_UPDATE(NV, UPD_RK3_3)
FVG_INST(4)
FVG_INST(5)
template __global__ void k_cells_march<float>(KP);
#define FVG_FACES(NV, D, PER)                                            \
    template __global__ void k_faces<NV, D, MODE_PLAIN, 1, PER, float>(KP); \
    template __global__ void k_faces<NV, D, MODE_PLAIN, 2, PER, float>(KP); \
    template __global__ void k_faces<NV, D, MODE_PLAIN, 3, PER, float>(KP);
#define FVG_AXIS(NV, D)   \
    FVG_FACES(NV, D, true)  \
    FVG_FACES(NV, D, false) \
    template __global__ void k_faces<NV, D, MODE_FIRST_ORDER, 0, false, float>(KP);
FVG_AXIS(4, 0)
FVG_AXIS(4, 1)
template __global__ void k_faces<5, 0, MODE_FIRST_ORDER, 0, false, float>(KP);   // k_xlast takes the others
FVG_AXIS(5, 1)
FVG_AXIS(5, 2)

}   // namespace fvg
