// MFMA SpMM instances: real matrices, FP64 (rg_mfma.h).
#include "rg_mfma.h"

namespace rg {

hipError_t launch_mfma_f64(const MfmaShape &s, const BsrDev &A, bool cv, const void *X, void *Y, int W, int R,
                           const EpiArgs &e, int grid, hipStream_t st, int *grid_out) {
    return cv ? by_shape<double, true, false>(s, A, X, Y, W, R, e, grid, st, grid_out)
              : by_shape<double, false, false>(s, A, X, Y, W, R, e, grid, st, grid_out);
}

} // namespace rg
