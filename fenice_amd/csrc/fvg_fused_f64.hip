// The FP64 instantiations of the fused residual passes (k_xacc, k_lacc) of every mode and stage the host launches.
#include "fvg_kernels_impl.hpp"

namespace fvg {

#define FVG_FUSED_MODE(NV, M, USE, T) template __global__ void k_xacc<NV, M, USE, T>(KP);
#define FVG_YPASS(M, USE, T) template __global__ void k_lacc<5, 1, M, USE, -1, T>(KP, const double*, const double*, double*);
#define FVG_LAST(NV, M, USE, UPD, T) \
    template __global__ void k_lacc<NV, (NV == 5 ? 2 : 1), M, USE, UPD, T>(KP, const double*, const double*, double*);
#define FVG_LAST_ALL(NV, M, T)                  \
    FVG_LAST(NV, M, 0, UPD_RESIDUAL, T)         \
    FVG_LAST(NV, M, 0, UPD_RK2_2, T)            \
    FVG_LAST(NV, M, 0, UPD_RK3_2, T)            \
    FVG_LAST(NV, M, 0, UPD_RK3_3, T)
#define FVG_FUSED(NV, T)                                      \
    FVG_FUSED_MODE(NV, MODE_PLAIN, 0, T)                      \
    FVG_FUSED_MODE(NV, MODE_FIRST_ORDER, 0, T)                \
    FVG_FUSED_MODE(NV, MODE_LEARNED, LF_STORE, T)             \
    FVG_FUSED_MODE(NV, MODE_LEARNED, LF_KEPT, T)              \
    FVG_LAST_ALL(NV, MODE_PLAIN, T)                           \
    FVG_LAST_ALL(NV, MODE_FIRST_ORDER, T)                     \
    FVG_LAST(NV, MODE_LEARNED, LF_STORE, UPD_RESIDUAL, T)     \
    FVG_LAST(NV, MODE_LEARNED, LF_KEPT, UPD_RK2_2, T)         \
    FVG_LAST(NV, MODE_LEARNED, LF_KEPT, UPD_RK3_2, T)         \
    FVG_LAST(NV, MODE_LEARNED, LF_KEPT, UPD_RK3_3, T)
FVG_FUSED(4, double)
FVG_FUSED(5, double)
FVG_YPASS(MODE_PLAIN, 0, double)
FVG_YPASS(MODE_FIRST_ORDER, 0, double)
FVG_YPASS(MODE_LEARNED, LF_STORE, double)
FVG_YPASS(MODE_LEARNED, LF_KEPT, double)
FVG_FUSED_MODE(4, MODE_HANCOCK, 0, double)
FVG_FUSED_MODE(5, MODE_HANCOCK, 0, double)
FVG_YPASS(MODE_HANCOCK, 0, double)
FVG_LAST(4, MODE_HANCOCK, 0, UPD_RESIDUAL, double)
FVG_LAST(5, MODE_HANCOCK, 0, UPD_RESIDUAL, double)
template __global__ void k_axpy<4>(KP, const double*, const double*, double*);
template __global__ void k_axpy<5>(KP, const double*, const double*, double*);

}   // namespace fvg
