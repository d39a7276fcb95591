// The FP32-flux instantiations of the learned indicator's kernels.
#include "fvg_kernels_impl.hpp"

namespace fvg {

#define FVG_FACES(NV, D)                                                    \
    template __global__ void k_faces_learned<NV, D, LF_STORE, true, float>(KP);  \
    template __global__ void k_faces_learned<NV, D, LF_STORE, false, float>(KP); \
    template __global__ void k_faces_learned<NV, D, LF_KEPT, true, float>(KP);   \
    template __global__ void k_faces_learned<NV, D, LF_KEPT, false, float>(KP);
#define FVG_AUDIT(NV, D)                             \
    template __global__ void k_audit<NV, D, float>(KP); \
    template __global__ void k_samples<NV, D, float>(KP, float*, float*);
FVG_FACES(4, 0)
FVG_FACES(4, 1)
FVG_FACES(5, 1)
FVG_FACES(5, 2)
FVG_AUDIT(4, 0)
FVG_AUDIT(4, 1)
FVG_AUDIT(5, 0)
FVG_AUDIT(5, 1)
FVG_AUDIT(5, 2)

}   // namespace fvg
