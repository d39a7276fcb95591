// The FP32-flux instantiations of the learned indicator's kernels.
#include "fvg_kernels_impl.hpp"

namespace fvg {

#define FVG_LEARNED(NV, D)                                                  \
    template __global__ void k_faces_learned<NV, D, LF_STORE, true, float>(KP);  \
    template __global__ void k_faces_learned<NV, D, LF_STORE, false, float>(KP); \
    template __global__ void k_faces_learned<NV, D, LF_KEPT, true, float>(KP);   \
    template __global__ void k_faces_learned<NV, D, LF_KEPT, false, float>(KP);  \
    template __global__ void k_audit<NV, D, float>(KP);                          \
    template __global__ void k_samples<NV, D, float>(KP, float*, float*);
FVG_LEARNED(4, 0)
FVG_LEARNED(4, 1)
FVG_LEARNED(5, 0)
FVG_LEARNED(5, 1)
FVG_LEARNED(5, 2)

}   // namespace fvg
