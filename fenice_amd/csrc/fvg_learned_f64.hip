// The FP64 instantiations of the learned indicator's kernels.
#include "fvg_kernels_impl.hpp"

namespace fvg {

#define FVG_FACES(NV, D)                                                    \
    template __global__ void k_faces_learned<NV, D, LF_STORE, true, double>(KP);  \
    template __global__ void k_faces_learned<NV, D, LF_STORE, false, double>(KP); \
    template __global__ void k_faces_learned<NV, D, LF_KEPT, true, double>(KP);   \
    template __global__ void k_faces_learned<NV, D, LF_KEPT, false, double>(KP);
#define FVG_AUDIT(NV, D)                             \
    template __global__ void k_audit<NV, D, double>(KP); \
    template __global__ void k_samples<NV, D, double>(KP, float*, float*);
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
