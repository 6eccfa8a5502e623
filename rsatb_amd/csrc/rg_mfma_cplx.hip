// MFMA SpMM instances: complex matrices (k-points), both precisions (rg_mfma.h).
#include "rg_mfma.h"

namespace rg {

hipError_t launch_mfma_cplx(const MfmaShape &s, const BsrDev &A, bool fp32, const void *X, void *Y, int W, int R,
                            const EpiArgs &e, int grid, hipStream_t st, int *grid_out) {
    return fp32 ? by_shape<float, true, true>(s, A, X, Y, W, R, e, grid, st, grid_out)
                : by_shape<double, true, true>(s, A, X, Y, W, R, e, grid, st, grid_out);
}

} // namespace rg
