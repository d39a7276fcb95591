// The FP64 instantiations of the residual kernels (the reference's arithmetic, bit for bit).
#include "fvg_kernels_impl.hpp"

namespace fvg {

#define FVG_UPDATE(NV, UPD) template __global__ void k_update<NV, UPD, double>(KP, const double*, const double*, double*);
#define FVG_INST(NV)                     \
    template __global__ void k_cells<NV, true, double>(KP);  \
    template __global__ void k_cells<NV, false, double>(KP); \
    FVG_UPDATE(NV, UPD_RESIDUAL)         \
    FVG_UPDATE(NV, UPD_AXPY)             \
    FVG_UPDATE(NV, UPD_RK2_2)            \
    FVG_UPDATE(NV, UPD_RK3_2)            \
    FVG_UPDATE(NV, UPD_RK3_3)
FVG_INST(4)
FVG_INST(5)
template __global__ void k_cells_march<double>(KP);
#define FVG_FACES(NV, D, PER)                                            \
    template __global__ void k_faces<NV, D, MODE_PLAIN, 1, PER, double>(KP); \
    template __global__ void k_faces<NV, D, MODE_PLAIN, 2, PER, double>(KP); \
    template __global__ void k_faces<NV, D, MODE_PLAIN, 3, PER, double>(KP);
#define FVG_AXIS(NV, D)   \
    FVG_FACES(NV, D, true)  \
    FVG_FACES(NV, D, false) \
    template __global__ void k_faces<NV, D, MODE_FIRST_ORDER, 0, false, double>(KP);
FVG_AXIS(4, 0)
FVG_AXIS(4, 1)
// x faces of a 3-D mesh: first order and the seed of a MUSCL-Hancock run (k_xlast takes the others)
template __global__ void k_faces<5, 0, MODE_PLAIN, 1, true, double>(KP);
template __global__ void k_faces<5, 0, MODE_PLAIN, 1, false, double>(KP);
template __global__ void k_faces<5, 0, MODE_FIRST_ORDER, 0, false, double>(KP);
FVG_AXIS(5, 1)
FVG_AXIS(5, 2)

#define FVG_HANCOCK(NV, D)                                                      \
    template __global__ void k_faces<NV, D, MODE_HANCOCK, 0, true, double>(KP); \
    template __global__ void k_faces<NV, D, MODE_HANCOCK, 0, false, double>(KP);
FVG_HANCOCK(4, 0)
FVG_HANCOCK(4, 1)
FVG_HANCOCK(5, 0)
FVG_HANCOCK(5, 1)
FVG_HANCOCK(5, 2)

}   // namespace fvg
