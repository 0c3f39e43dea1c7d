// Folded step kernels with four lanes per bead of the H3, OH3, BrH2 and O3
// surfaces (the kernels are in fold.hpp).  Compiled without machine-level
// loop-invariant code motion, as every translation unit with binary32 H3 step
// kernels.
#include "fold.hpp"

namespace cam {

step_fn fold_kernel_quad(int surface, int precision, int nbeads, int ensemble, int *tpb)
{
    if (surface == CAM_SURFACE_H3)
        return precision == CAM_PREC_FP64 ? fold::pick_fold_w<SurfH3Q, double, 3, 1>(nbeads, ensemble, tpb)
                                          : fold::pick_fold_w<SurfH3Q, float, 3, 1>(nbeads, ensemble, tpb);
    if (surface == CAM_SURFACE_OH3) return fold::pick_fold_w<SurfOH3Q, double, 3, 1>(nbeads, ensemble, tpb);
    if (surface == CAM_SURFACE_BRH2) return fold::pick_fold_w<SurfBrH2Q, double, 2, 1>(nbeads, ensemble, tpb);
    if (surface == CAM_SURFACE_O3) return fold::pick_fold_w<SurfO3Q, double, 3, 1>(nbeads, ensemble, tpb);
    return nullptr;
}

}  // namespace cam
