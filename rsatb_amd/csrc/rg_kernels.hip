// gfx950 kernels of the KPM moment loop.
//
// k_spmm: block-row-gather BSR SpMM Y = epi(A X) over a block of R sample
// columns, fused with the Chebyshev recurrence and the per-column moment
// dots (the three passes rsatb runs separately: mult_dense, axpby, dot;
// rsatb/calc/cheby.hpp:555-606, rsatb/calc/dos.hpp:150-173).
//
// Mapping. A wavefront (64 lanes) owns G = 64/LPR block rows; within a row,
// lane q owns sample columns q*UPL .. q*UPL+UPL-1. With LPR = 64 (R > 32) a
// wave owns exactly one block row, so the block row, its CSR range and every
// matrix entry are wave-uniform and are fetched by scalar loads and fed to
// the FMAs as SGPR operands: the matrix is streamed from HBM once per apply
// and never occupies VGPRs. Each lane keeps b x UPL accumulators; per matrix
// entry it issues UPL (real vectors) or 2 UPL (complex vectors) FMAs, with
// one coalesced vector load per block column (64 lanes x UPL x 8/16 B
// contiguous). With R <= 32 (LPR = R rounded up to 8/16/32) several block
// rows share a wave and entries come through vector loads.
//
// Dots. Every lane accumulates its columns' dot products in FP64 over all
// rows it visits (grid-stride over block rows), then the workgroup reduces
// over sub-rows (xor shuffles) and waves (LDS) and writes one partial per
// column; k_reduce sums the partials of all workgroups in a fixed order, so
// results are deterministic run to run.
#include "rg_internal.h"

#include <atomic>

#include <algorithm>
#include <numeric>
#include <type_traits>

namespace rg {

MfmaKnobs g_mfma;
thread_local bool t_mfma_grid_query = false;

namespace {

constexpr int kWaves = 4;   // waves per workgroup
constexpr int kMaxGrid = 2048;
// Waves below which an MFMA launch halves its tiles per wave (1.5 a SIMD).
// Measured with R = 64 / 128 complex, FP64, us a step, whole against halved
// once and twice: 640 rows (b = 9) 22.4, 22.3, 22.3 / 34.9, 34.7, 31.5; 1,200
// rows 34.2, 31.0 / 68.3, 56.5, 50.0; 1,680 rows (b = 13) 50.4, 57.3 / 104,
// 98, 101.
constexpr int64_t kMfmaSplitWaves = 1536;

// b = 1 SpMM over real vectors with 2 columns per lane: 1 always, 0 never,
// 2 by precision and row length.
int g_b1_wide = 2;
// The VALU SpMM computes the entry range of uniform rows (1) or loads it (0).
int g_uniform_rows = 1;
// Bytes of a row one lane owns in the b = 1 slab SpMM (16, 32 or 64; 0: the
// column-per-lane layout of k_spmm), and the fewest workgroups a slab launch
// may have (below it the rows go to k_spmm, whose layouts spread them over
// more waves). Measured on graphene p_z, R = 16 real, FP64 / FP32 step at
// 1,048,576 rows: k_spmm 134.1 / 69.7 us, slabs of 16 bytes 92.3 / 42.3 us
// (0.63 / 0.72 of the HBM peak), 32 bytes 99.2 / 45.0, 64 bytes 117.7 / 65.8;
// the 16,384-row graphene run (FP64 / FP32) 2.90 / 2.73 ms with k_spmm,
// 2.61 / 2.86 ms with 16-byte slabs: the FP32 slab launch there has 256
// workgroups, one wave per SIMD.
// Automatic (-1): 16 bytes, 32 for complex FP64 vectors (two columns a lane:
// the C4-shaped adjoint, 65,536 rows x 13 entries, R = 32 complex, forward
// 25.1 -> 23.7 ms and backward 70.4 -> 69.5 ms against 16 bytes).
int g_b1v_bytes = -1;
int g_b1v_min_grid = 512;
// The same for the slab layout of other widths; long rows (eight entries on
// average) gain from it down to 256 workgroups. Measured, FP64, column-per-lane
// against slabs: 16,384 rows of four, R = 10 complex (655 workgroups) 7.1 / 7.7
// us, R = 24 real (780) 7.4 / 8.0; 65,536 rows, R = 24 15.4 / 11.5; 9,000 rows
// of thirteen, R = 10 complex (360) 10.0 / 8.0, R = 24 (428) 9.3 / 8.2.
int g_b1g_min_grid = 1024;
constexpr int kLongRow = 8, kLongRowMinGrid = 256;
// Vector bytes up to which the slab SpMMs walk XCD-contiguous row ranges.
// Measured (round robin / contiguous): 479,596 rows of thirteen, FP32 R = 32
// (61 MB) 71.9 / 69.0 us, FP64 R = 4 46.2 / 34.3, R = 10 56.7 / 49.2, R = 32
// complex (245 MB) 302 / 318; 59,212 rows, R = 32 complex (30 MB) 33.7 / 30.8;
// 1,048,576 rows of four, R = 16 (134 MB) 93.1 / 99.0.
constexpr int64_t kXcdVectorBytes = (int64_t)64 << 20;
template <typename S> struct V2;
template <> struct V2<double> { using T = double2; };
template <> struct V2<float> { using T = float2; };

// ---------------------------------------------------------------- algebra
__device__ __forceinline__ void mac(double &acc, double a, double x) { acc = __builtin_fma(a, x, acc); }
__device__ __forceinline__ void mac(float &acc, float a, float x) { acc = __builtin_fmaf(a, x, acc); }
__device__ __forceinline__ void mac(double2 &acc, double a, double2 x) {
    acc.x = __builtin_fma(a, x.x, acc.x);
    acc.y = __builtin_fma(a, x.y, acc.y);
}
__device__ __forceinline__ void mac(float2 &acc, float a, float2 x) {
    acc.x = __builtin_fmaf(a, x.x, acc.x);
    acc.y = __builtin_fmaf(a, x.y, acc.y);
}
__device__ __forceinline__ void mac(double2 &acc, double2 a, double2 x) {
    acc.x = __builtin_fma(a.x, x.x, __builtin_fma(-a.y, x.y, acc.x));
    acc.y = __builtin_fma(a.x, x.y, __builtin_fma(a.y, x.x, acc.y));
}
__device__ __forceinline__ void mac(float2 &acc, float2 a, float2 x) {
    acc.x = __builtin_fmaf(a.x, x.x, __builtin_fmaf(-a.y, x.y, acc.x));
    acc.y = __builtin_fmaf(a.x, x.y, __builtin_fmaf(a.y, x.x, acc.y));
}

template <typename T> __device__ __forceinline__ T vzero() { return T{}; }

// y = alpha v + beta s (- p)
__device__ __forceinline__ double affine(double v, double alpha, double beta, double s) {
    return __builtin_fma(alpha, v, beta * s);
}
__device__ __forceinline__ double2 affine(double2 v, double alpha, double beta, double2 s) {
    return double2{__builtin_fma(alpha, v.x, beta * s.x), __builtin_fma(alpha, v.y, beta * s.y)};
}
__device__ __forceinline__ float affine(float v, double alpha, double beta, float s) {
    return (float)__builtin_fma(alpha, (double)v, beta * (double)s);
}
__device__ __forceinline__ float2 affine(float2 v, double alpha, double beta, float2 s) {
    return float2{(float)__builtin_fma(alpha, (double)v.x, beta * (double)s.x),
                  (float)__builtin_fma(alpha, (double)v.y, beta * (double)s.y)};
}
__device__ __forceinline__ double sub(double a, double b) { return a - b; }
__device__ __forceinline__ float sub(float a, float b) { return a - b; }
__device__ __forceinline__ double2 sub(double2 a, double2 b) { return double2{a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ float2 sub(float2 a, float2 b) { return float2{a.x - b.x, a.y - b.y}; }

// d += conj(a) b in FP64. Products of two floats are exact in FP64.
__device__ __forceinline__ void dotacc(double2 &d, double a, double b) { d.x = __builtin_fma(a, b, d.x); }
__device__ __forceinline__ void dotacc(double2 &d, float a, float b) { d.x = __builtin_fma((double)a, (double)b, d.x); }
__device__ __forceinline__ void dotacc(double2 &d, double2 a, double2 b) {
    d.x = __builtin_fma(a.x, b.x, __builtin_fma(a.y, b.y, d.x));
    d.y = __builtin_fma(a.x, b.y, __builtin_fma(-a.y, b.x, d.y));
}
__device__ __forceinline__ void dotacc(double2 &d, float2 a, float2 b) {
    dotacc(d, double2{(double)a.x, (double)a.y}, double2{(double)b.x, (double)b.y});
}

__device__ __forceinline__ int dev_ndot(int mode) {
    return mode == EPI_FIRST ? 3 : mode == EPI_STEP ? 2 : mode == EPI_PLAINSTEP ? 1 : 0;
}

// ------------------------------------------------------------------ SpMM
template <typename S, bool CM, bool CV, int BS, int LPR, int UPL>
__global__ __launch_bounds__(256) void k_spmm(int64_t nbr, int bs_rt, int ulen,
                                              const int64_t *__restrict__ row_ptr,
                                              const int32_t *__restrict__ col_ind,
                                              const void *__restrict__ vals_v,
                                              const void *__restrict__ x_v, void *__restrict__ y_v,
                                              int R, EpiArgs e) {
    using VT = std::conditional_t<CV, typename V2<S>::T, S>;
    using MT = std::conditional_t<CM, typename V2<S>::T, S>;
    constexpr int G = 64 / LPR;
    constexpr int MAXB = BS > 0 ? BS : 16;
    constexpr int COLS = LPR * UPL; // columns one sub-row covers

    const MT *__restrict__ vals = static_cast<const MT *>(vals_v);
    const VT *__restrict__ X = static_cast<const VT *>(x_v);
    VT *__restrict__ Y = static_cast<VT *>(y_v);
    const VT *__restrict__ XS = static_cast<const VT *>(e.xs);
    const VT *__restrict__ XP = static_cast<const VT *>(e.xp);
    const VT *__restrict__ PSI = static_cast<const VT *>(e.psi);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = (G > 1) ? (lane / LPR) : 0;
    const int q = (G > 1) ? (lane % LPR) : lane;
    const int bs = BS > 0 ? BS : bs_rt;
    const int mode = e.mode;
    const int ndot = dev_ndot(mode);

    double2 dacc[3][UPL];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int j = 0; j < UPL; ++j) dacc[d][j] = double2{0.0, 0.0};

    const int64_t rows_per_wg = (int64_t)kWaves * G;
    for (int64_t base = (int64_t)blockIdx.x * rows_per_wg; base < nbr;
         base += (int64_t)gridDim.x * rows_per_wg) {
        const int64_t br = base + (int64_t)wave * G + g;
        if (br >= nbr) continue;

        VT acc[MAXB][UPL];
#pragma unroll
        for (int r = 0; r < MAXB; ++r)
#pragma unroll
            for (int j = 0; j < UPL; ++j) acc[r][j] = vzero<VT>();

        // uniform rows: the range follows from br, and the column index
        // loads wait on nothing (one dependent load fewer per row)
        const int64_t s0 = ulen > 0 ? br * ulen : row_ptr[br];
        const int64_t s1 = ulen > 0 ? s0 + ulen : row_ptr[br + 1];
        int64_t s = s0;
        if constexpr (BS == 1) {
            // Scalar entries: the gather of each entry's X row waits on its
            // column index, so U entries' indices and values are loaded
            // first and their U row loads issued back to back (the
            // accumulation order is unchanged). U = 4 measured best: 4-entry
            // graphene rows take it whole (FP64 step 161 -> 137 us at
            // 1,048,576 rows), 22-entry rows gain over U = 8 (74 -> 67 us),
            // and complex vectors stay at 8 waves per SIMD.
            constexpr int U = 4;
            for (; s + U <= s1; s += U) {
                int64_t bc[U];
                MT a[U];
#pragma unroll
                for (int t = 0; t < U; ++t) {
                    bc[t] = col_ind[s + t];
                    a[t] = vals[s + t];
                }
                VT xk[U][UPL];
#pragma unroll
                for (int t = 0; t < U; ++t)
#pragma unroll
                    for (int j = 0; j < UPL; ++j) {
                        const int u = q * UPL + j;
                        xk[t][j] = (u < R) ? X[bc[t] * R + u] : vzero<VT>();
                    }
#pragma unroll
                for (int t = 0; t < U; ++t)
#pragma unroll
                    for (int j = 0; j < UPL; ++j) mac(acc[0][j], a[t], xk[t][j]);
            }
        }
        for (; s < s1; ++s) {
            const int64_t bc = col_ind[s];
            const MT *__restrict__ blk = vals + s * (int64_t)(bs * bs);
            const VT *__restrict__ xb = X + bc * (int64_t)bs * R;
#pragma unroll
            for (int k = 0; k < MAXB; ++k) {
                if (BS == 0 && k >= bs) continue;
                VT xk[UPL];
#pragma unroll
                for (int j = 0; j < UPL; ++j) {
                    const int u = q * UPL + j;
                    xk[j] = (u < R) ? xb[(int64_t)k * R + u] : vzero<VT>();
                }
#pragma unroll
                for (int r = 0; r < MAXB; ++r) {
                    if (BS == 0 && r >= bs) continue;
                    const MT a = blk[k * bs + r]; // blocks are stored column-major on the device
#pragma unroll
                    for (int j = 0; j < UPL; ++j) mac(acc[r][j], a, xk[j]);
                }
            }
        }

#pragma unroll
        for (int r = 0; r < MAXB; ++r) {
            if (BS == 0 && r >= bs) continue;
            const int64_t row = br * bs + r;
#pragma unroll
            for (int j = 0; j < UPL; ++j) {
                const int u = q * UPL + j;
                if (u >= R) continue;
                const int64_t idx = row * R + u;
                VT y = acc[r][j];
                if (mode == EPI_FIRST) {
                    const VT xs = XS[idx];
                    y = affine(y, e.alpha, e.beta, xs);
                    dotacc(dacc[0][j], xs, xs);
                    dotacc(dacc[1][j], xs, y);
                    dotacc(dacc[2][j], y, y);
                } else if (mode == EPI_STEP) {
                    const VT xs = XS[idx];
                    y = sub(affine(y, e.alpha, e.beta, xs), XP[idx]);
                    dotacc(dacc[0][j], y, y);
                    dotacc(dacc[1][j], y, xs);
                } else if (mode == EPI_PLAINSTEP) {
                    y = sub(affine(y, e.alpha, e.beta, XS[idx]), XP[idx]);
                    dotacc(dacc[0][j], PSI[idx], y);
                } else if (mode == EPI_ADJ) {
                    y = sub(affine(y, e.alpha, e.beta, XS[idx]), XP[idx]);
                    y = affine(y, 1.0, e.cm, static_cast<const VT *>(e.qm)[idx]);
                    y = affine(y, 1.0, e.cz, static_cast<const VT *>(e.qz)[idx]);
                    y = affine(y, 1.0, e.cp, static_cast<const VT *>(e.qp)[idx]);
                }
                Y[idx] = y;
            }
        }
    }

    if (ndot == 0) return;

    // sub-rows of one wave hold the same columns: fold them (xor tree)
    if (G > 1) {
#pragma unroll
        for (int off = LPR; off < 64; off <<= 1)
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int j = 0; j < UPL; ++j) {
                    dacc[d][j].x += __shfl_xor(dacc[d][j].x, off);
                    dacc[d][j].y += __shfl_xor(dacc[d][j].y, off);
                }
    }
    __shared__ double2 sm[kWaves][COLS];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= ndot) break;
        if (g == 0) {
#pragma unroll
            for (int j = 0; j < UPL; ++j) sm[wave][q * UPL + j] = dacc[d][j];
        }
        __syncthreads();
        for (int u = threadIdx.x; u < COLS && u < R; u += blockDim.x) {
            double2 acc2 = sm[0][u];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) {
                acc2.x += sm[w][u].x;
                acc2.y += sm[w][u].y;
            }
            e.partials[((int64_t)blockIdx.x * ndot + d) * R + u] = acc2;
        }
        __syncthreads();
    }
}

int lpr_for(int R) { return R <= 8 ? 8 : R <= 16 ? 16 : R <= 32 ? 32 : 64; }

int upl_for(int R) { return R <= 64 ? 1 : R <= 128 ? 2 : 4; }

// The wide b = 1 layout (half the lanes per row, two columns per lane) for
// scalar entries and real vectors, 8 < R <= 32: FP32, or rows of >= 8
// entries (g_b1_wide 2), always (1) or never (0).
bool b1_wide(const BsrDev &A, bool fp32, bool cv, int R) {
    if (A.b != 1 || cv || R <= 8 || R > 32) return false;
    return g_b1_wide == 1 || (g_b1_wide == 2 && (fp32 || A.nnzb >= 8 * A.nbr));
}

// Lanes per block row of the VALU SpMM launch for this operand.
int b1v_lpr(const BsrDev &A, bool fp32, bool cv, int R);
int valu_lpr(const BsrDev &A, bool fp32, bool cv, int R) {
    if (const int l = b1v_lpr(A, fp32, cv, R)) return l;
    if (b1_wide(A, fp32, cv, R)) return R <= 16 ? 8 : 16;
    return lpr_for(R);
}

template <typename S, bool CM, bool CV, int BS, int LPR, int UPL>
hipError_t go(const BsrDev &A, const void *X, void *Y, int R, const EpiArgs &e, int grid,
              hipStream_t st) {
    hipLaunchKernelGGL((k_spmm<S, CM, CV, BS, LPR, UPL>), dim3(grid), dim3(64 * kWaves), 0, st,
                       A.nbr, (int)A.b, g_uniform_rows ? A.ulen : 0, A.row_ptr, A.col_ind, A.vals, X, Y, R, e);
    return hipGetLastError();
}

template <typename S, bool CM, bool CV, int BS>
hipError_t by_layout(const BsrDev &A, const void *X, void *Y, int R, const EpiArgs &e, int grid,
                     hipStream_t st) {
    if constexpr (BS == 1 && !CV) {
        // Scalar entries, real vectors: half the lanes per row and two
        // columns per lane, twice the rows (and independent gathers) per
        // wave. Measured on graphene p_z with R = 16: FP32 step 103 -> 76 us
        // at 1,048,576 rows of 4 entries, FP64 86 -> 75 us at 190,528 rows of
        // 22 entries, but FP64 163 -> 193 us at 4 entries a row; complex
        // vectors (R = 32) slower. Automatic: FP32, or rows of >= 8 entries.
        const bool wide = b1_wide(A, sizeof(S) == 4, CV, R);
        if (wide && R <= 16) return go<S, CM, CV, BS, 8, 2>(A, X, Y, R, e, grid, st);
        if (wide) return go<S, CM, CV, BS, 16, 2>(A, X, Y, R, e, grid, st);
    }
    switch (lpr_for(R)) {
    case 8: return go<S, CM, CV, BS, 8, 1>(A, X, Y, R, e, grid, st);
    case 16: return go<S, CM, CV, BS, 16, 1>(A, X, Y, R, e, grid, st);
    case 32: return go<S, CM, CV, BS, 32, 1>(A, X, Y, R, e, grid, st);
    default: break;
    }
    switch (upl_for(R)) {
    case 1: return go<S, CM, CV, BS, 64, 1>(A, X, Y, R, e, grid, st);
    case 2: return go<S, CM, CV, BS, 64, 2>(A, X, Y, R, e, grid, st);
    default: return go<S, CM, CV, BS, 64, 4>(A, X, Y, R, e, grid, st);
    }
}

template <typename S, bool CM, bool CV>
hipError_t by_block(const BsrDev &A, const void *X, void *Y, int R, const EpiArgs &e, int grid,
                    hipStream_t st) {
    if (A.b == 1) return by_layout<S, CM, CV, 1>(A, X, Y, R, e, grid, st);
    if (A.b == 13) return by_layout<S, CM, CV, 13>(A, X, Y, R, e, grid, st);
    return by_layout<S, CM, CV, 0>(A, X, Y, R, e, grid, st);
}

// The rows of a workgroup of a grid-stride launch, `per` rows a stride. With
// xcd (the grid a multiple of 8) every XCD walks its own contiguous eighth:
// workgroups go to the XCDs in turn, and neighbouring rows gather the same
// rows of X through one L2.
struct RowWalk {
    int64_t lo, hi, step;
    __device__ __forceinline__ RowWalk(int64_t n, int per, int xcd) {
        if (xcd) {
            const int64_t eighth = ((n + per - 1) / per + 7) / 8 * per;
            const int64_t x0 = (int64_t)(blockIdx.x & 7) * eighth;
            lo = x0 + (int64_t)(blockIdx.x >> 3) * per;
            hi = min(n, x0 + eighth);
            step = (int64_t)(gridDim.x >> 3) * per;
        } else {
            lo = (int64_t)blockIdx.x * per;
            hi = n;
            step = (int64_t)gridDim.x * per;
        }
    }
};

// ------------------------------------------------------- b = 1 slab SpMM
// Scalar entries, real matrix, R = LPR * CPL exactly: lane q of a row's LPR
// lanes owns the contiguous slab of columns q * CPL .. q * CPL + CPL - 1 and
// moves it as 16-byte loads and stores (CPL values of 8 or 16 bytes: 16, 32
// or 64 bytes a lane). Fewer lanes per row put more rows, and more
// independent gathers, in one wave than the column-per-lane layout of
// k_spmm; every product and epilogue value is formed by the same operations
// in the same order as there (the dots differ only in their summation
// order). Vector operands must be 16-byte aligned.
template <typename S, bool CV, int LPR, int CPL>
__global__ __launch_bounds__(256) void k_spmm_b1v(int64_t nbr, int ulen, int xcd, const int64_t *__restrict__ row_ptr,
                                                  const int32_t *__restrict__ col_ind,
                                                  const S *__restrict__ vals, const S *__restrict__ X,
                                                  S *__restrict__ Y, EpiArgs e) {
    using VT = std::conditional_t<CV, typename V2<S>::T, S>;
    constexpr int G = 64 / LPR;
    constexpr int NS = CPL * (CV ? 2 : 1);    // scalars a lane owns in a row
    constexpr int EPC = 16 / (int)sizeof(S);  // scalars a 16-byte chunk holds
    constexpr int NCH = NS / EPC;             // chunks a lane moves per row
    static_assert(NS % EPC == 0 && 64 % LPR == 0, "slab of whole 16-byte chunks");
    typedef S C16 __attribute__((ext_vector_type(EPC)));
    constexpr int64_t W = (int64_t)LPR * NS;  // scalars a row holds

    const S *__restrict__ XS = static_cast<const S *>(e.xs);
    const S *__restrict__ XP = static_cast<const S *>(e.xp);
    const S *__restrict__ PSI = static_cast<const S *>(e.psi);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane / LPR;
    const int q = lane % LPR;
    const int mode = e.mode;
    const int ndot = dev_ndot(mode);

    auto ld = [](const S *p, S (&v)[NS]) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const C16 t = *reinterpret_cast<const C16 *>(p + c * EPC);
#pragma unroll
            for (int k = 0; k < EPC; ++k) v[c * EPC + k] = t[k];
        }
    };
    auto vt = [](const S (&v)[NS], int j) -> VT {
        if constexpr (CV) return VT{v[2 * j], v[2 * j + 1]};
        else return v[j];
    };

    double2 dacc[3][CPL];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int j = 0; j < CPL; ++j) dacc[d][j] = double2{0.0, 0.0};

    const RowWalk walk(nbr, kWaves * G, xcd);
    for (int64_t base = walk.lo; base < walk.hi; base += walk.step) {
        const int64_t br = base + (int64_t)wave * G + g;
        if (br >= walk.hi) continue;
        S acc[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) acc[i] = S(0);
        const int64_t s0 = ulen > 0 ? br * ulen : row_ptr[br];
        const int64_t s1 = ulen > 0 ? s0 + ulen : row_ptr[br + 1];
        const int64_t lo = (int64_t)q * NS;
        int64_t s = s0;
        constexpr int U = 4;
        for (; s + U <= s1; s += U) {
            int32_t bc[U];
            S a[U];
#pragma unroll
            for (int t = 0; t < U; ++t) {
                bc[t] = col_ind[s + t];
                a[t] = vals[s + t];
            }
            S xk[U][NS];
#pragma unroll
            for (int t = 0; t < U; ++t) ld(X + bc[t] * W + lo, xk[t]);
#pragma unroll
            for (int t = 0; t < U; ++t)
#pragma unroll
                for (int i = 0; i < NS; ++i) mac(acc[i], a[t], xk[t][i]);
        }
        for (; s < s1; ++s) {
            const int64_t bc = col_ind[s];
            const S a = vals[s];
            S xk[NS];
            ld(X + bc * W + lo, xk);
#pragma unroll
            for (int i = 0; i < NS; ++i) mac(acc[i], a, xk[i]);
        }

        const int64_t idx = br * W + lo;
        S y[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) y[i] = acc[i];
        if (mode == EPI_FIRST) {
            S xs[NS];
            ld(XS + idx, xs);
#pragma unroll
            for (int i = 0; i < NS; ++i) y[i] = affine(y[i], e.alpha, e.beta, xs[i]);
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                dotacc(dacc[0][j], vt(xs, j), vt(xs, j));
                dotacc(dacc[1][j], vt(xs, j), vt(y, j));
                dotacc(dacc[2][j], vt(y, j), vt(y, j));
            }
        } else if (mode == EPI_STEP) {
            S xs[NS], xp[NS];
            ld(XS + idx, xs);
            ld(XP + idx, xp);
#pragma unroll
            for (int i = 0; i < NS; ++i) y[i] = sub(affine(y[i], e.alpha, e.beta, xs[i]), xp[i]);
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                dotacc(dacc[0][j], vt(y, j), vt(y, j));
                dotacc(dacc[1][j], vt(y, j), vt(xs, j));
            }
        } else if (mode == EPI_PLAINSTEP) {
            S xs[NS], xp[NS], ps[NS];
            ld(XS + idx, xs);
            ld(XP + idx, xp);
            ld(PSI + idx, ps);
#pragma unroll
            for (int i = 0; i < NS; ++i) y[i] = sub(affine(y[i], e.alpha, e.beta, xs[i]), xp[i]);
#pragma unroll
            for (int j = 0; j < CPL; ++j) dotacc(dacc[0][j], vt(ps, j), vt(y, j));
        } else if (mode == EPI_ADJ) {
            S xs[NS], xp[NS], t[NS];
            ld(XS + idx, xs);
            ld(XP + idx, xp);
#pragma unroll
            for (int i = 0; i < NS; ++i) y[i] = sub(affine(y[i], e.alpha, e.beta, xs[i]), xp[i]);
            ld(static_cast<const S *>(e.qm) + idx, t);
#pragma unroll
            for (int i = 0; i < NS; ++i) y[i] = affine(y[i], 1.0, e.cm, t[i]);
            ld(static_cast<const S *>(e.qz) + idx, t);
#pragma unroll
            for (int i = 0; i < NS; ++i) y[i] = affine(y[i], 1.0, e.cz, t[i]);
            ld(static_cast<const S *>(e.qp) + idx, t);
#pragma unroll
            for (int i = 0; i < NS; ++i) y[i] = affine(y[i], 1.0, e.cp, t[i]);
        }
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            C16 t;
#pragma unroll
            for (int k = 0; k < EPC; ++k) t[k] = y[c * EPC + k];
            *reinterpret_cast<C16 *>(Y + idx + c * EPC) = t;
        }
    }

    if (ndot == 0) return;
    // the rows of one wave hold the same columns: fold them (xor tree)
    if (G > 1) {
#pragma unroll
        for (int off = LPR; off < 64; off <<= 1)
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int j = 0; j < CPL; ++j) {
                    dacc[d][j].x += __shfl_xor(dacc[d][j].x, off);
                    dacc[d][j].y += __shfl_xor(dacc[d][j].y, off);
                }
    }
    constexpr int COLS = LPR * CPL;
    __shared__ double2 sm[kWaves][COLS];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= ndot) break;
        if (g == 0) {
#pragma unroll
            for (int j = 0; j < CPL; ++j) sm[wave][q * CPL + j] = dacc[d][j];
        }
        __syncthreads();
        for (int u = threadIdx.x; u < COLS; u += blockDim.x) {
            double2 acc2 = sm[0][u];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) {
                acc2.x += sm[w][u].x;
                acc2.y += sm[w][u].y;
            }
            e.partials[((int64_t)blockIdx.x * ndot + d) * COLS + u] = acc2;
        }
        __syncthreads();
    }
}

// The slab layout for any row of whole 16-byte pieces: cpr lanes a row (a
// piece each), as many whole rows in a workgroup as fit its 256 lanes, the
// products and epilogues as in k_spmm_b1v. The dots of a column are summed
// over the workgroup's rows through LDS, `parts` lanes a column. Bound by the
// gathers: one row's entry is one wide load a lane, where a column per lane
// leaves R mod 64 lanes idle and loads 4 to 16 bytes a lane. Measured (a moment
// step, column-per-lane / slabs): 1,048,576 rows of four entries, FP64 R = 10
// 120 / 70 us, one phase column 48 / 19; 479,596 rows of thirteen, R = 10 85 /
// 49, R = 10 complex 141 / 108, R = 24 204 / 128; 59,212 rows of thirteen, R =
// 10 complex 19.5 / 14.8, R = 64 51 / 31. Loading a group's indices and values
// with wide loads changed nothing; folding the one to three last entries into
// a masked group of four cost 10 % at thirteen entries.
template <typename S, bool CV>
__global__ __launch_bounds__(256) void k_spmm_b1g(int64_t nbr, int cpr, int ulen, int xcd,
                                                  const int64_t *__restrict__ row_ptr,
                                                  const int32_t *__restrict__ col_ind, const S *__restrict__ vals,
                                                  const S *__restrict__ X, S *__restrict__ Y, EpiArgs e) {
    using VT = std::conditional_t<CV, typename V2<S>::T, S>;
    constexpr int NS = 16 / (int)sizeof(S);   // scalars a lane owns in a row
    constexpr int CPL = NS / (CV ? 2 : 1);    // columns
    typedef S C16 __attribute__((ext_vector_type(NS)));
    const int rpb = 256 / cpr;
    const int lr = (int)threadIdx.x / cpr, q = (int)threadIdx.x - lr * cpr;
    const int64_t W = (int64_t)cpr * NS, lo = (int64_t)q * NS;
    const int mode = e.mode;
    const int ndot = dev_ndot(mode);
    const S *__restrict__ XS = static_cast<const S *>(e.xs);
    const S *__restrict__ XP = static_cast<const S *>(e.xp);
    const S *__restrict__ PSI = static_cast<const S *>(e.psi);
    auto ld = [](const S *p) { return *reinterpret_cast<const C16 *>(p); };
    auto vt = [](C16 v, int j) -> VT {
        if constexpr (CV) return VT{v[2 * j], v[2 * j + 1]};
        else return v[j];
    };
    auto aff = [](C16 v, double a, double b, C16 s) -> C16 {
        C16 o;
#pragma unroll
        for (int i = 0; i < NS; ++i) o[i] = affine(v[i], a, b, s[i]);
        return o;
    };
    double2 dacc[3][CPL];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int j = 0; j < CPL; ++j) dacc[d][j] = double2{0.0, 0.0};

    const RowWalk walk(nbr, rpb, xcd);
    for (int64_t base = walk.lo; base < walk.hi; base += walk.step) {
        const int64_t br = base + lr;
        if (lr >= rpb || br >= walk.hi) continue;
        const int64_t s0 = ulen > 0 ? br * ulen : row_ptr[br];
        const int64_t s1 = ulen > 0 ? s0 + ulen : row_ptr[br + 1];
        C16 y = C16(S(0));
        int64_t s = s0;
        constexpr int U = 4;
        for (; s + U <= s1; s += U) {
            int32_t c[U];
            S a[U];
            C16 g[U];
#pragma unroll
            for (int t = 0; t < U; ++t) {
                c[t] = col_ind[s + t];
                a[t] = vals[s + t];
            }
#pragma unroll
            for (int t = 0; t < U; ++t) g[t] = ld(X + c[t] * W + lo);
#pragma unroll
            for (int t = 0; t < U; ++t)
#pragma unroll
                for (int i = 0; i < NS; ++i) {
                    S yi = y[i];
                    mac(yi, a[t], (S)g[t][i]);
                    y[i] = yi;
                }
        }
        for (; s < s1; ++s) {
            const C16 g = ld(X + (int64_t)col_ind[s] * W + lo);
            const S a = vals[s];
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                S yi = y[i];
                mac(yi, a, (S)g[i]);
                y[i] = yi;
            }
        }
        const int64_t idx = br * W + lo;
        if (mode == EPI_FIRST) {
            const C16 xs = ld(XS + idx);
            y = aff(y, e.alpha, e.beta, xs);
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                dotacc(dacc[0][j], vt(xs, j), vt(xs, j));
                dotacc(dacc[1][j], vt(xs, j), vt(y, j));
                dotacc(dacc[2][j], vt(y, j), vt(y, j));
            }
        } else if (mode != EPI_PLAIN) {
            const C16 xs = ld(XS + idx), xp = ld(XP + idx);
            y = aff(y, e.alpha, e.beta, xs) - xp;
            if (mode == EPI_STEP) {
#pragma unroll
                for (int j = 0; j < CPL; ++j) {
                    dotacc(dacc[0][j], vt(y, j), vt(y, j));
                    dotacc(dacc[1][j], vt(y, j), vt(xs, j));
                }
            } else if (mode == EPI_PLAINSTEP) {
                const C16 ps = ld(PSI + idx);
#pragma unroll
                for (int j = 0; j < CPL; ++j) dotacc(dacc[0][j], vt(ps, j), vt(y, j));
            } else {
                y = aff(y, 1.0, e.cm, ld(static_cast<const S *>(e.qm) + idx));
                y = aff(y, 1.0, e.cz, ld(static_cast<const S *>(e.qz) + idx));
                y = aff(y, 1.0, e.cp, ld(static_cast<const S *>(e.qp) + idx));
            }
        }
        *reinterpret_cast<C16 *>(Y + idx) = y;
    }
    if (ndot == 0) return;
    const int ncol = cpr * CPL, parts = min(min(rpb, 16), max(1, 256 / ncol));
    __shared__ double2 sm[256 * CPL], sp[256];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d >= ndot) break;
        if (lr < rpb)
#pragma unroll
            for (int j = 0; j < CPL; ++j) sm[lr * ncol + q * CPL + j] = dacc[d][j];
        __syncthreads();
        for (int t = threadIdx.x; t < ncol * parts; t += 256) {
            const int u = t % ncol, p = t / ncol;
            double2 v{0.0, 0.0};
            for (int r = p; r < rpb; r += parts) {
                v.x += sm[r * ncol + u].x;
                v.y += sm[r * ncol + u].y;
            }
            if (parts == 1) e.partials[((int64_t)blockIdx.x * ndot + d) * ncol + u] = v;
            else sp[t] = v;
        }
        __syncthreads();
        if (parts > 1 && (int)threadIdx.x < ncol) {
            double2 v = sp[threadIdx.x];
            for (int p = 1; p < parts; ++p) {
                v.x += sp[p * ncol + threadIdx.x].x;
                v.y += sp[p * ncol + threadIdx.x].y;
            }
            e.partials[((int64_t)blockIdx.x * ndot + d) * ncol + threadIdx.x] = v;
        }
    }
}

int xcd_walk(const BsrDev &A, int grid, int64_t row_bytes) {
    return g_mfma.xcd_map && grid % 8 == 0 && A.nbr * row_bytes <= kXcdVectorBytes;
}

// Lanes per row (16-byte pieces) of k_spmm_b1g for this launch shape, or 0
// when it does not apply.
int b1g_cpr(const BsrDev &A, bool fp32, bool cv, int R) {
    if (A.b != 1 || A.is_complex || g_b1v_bytes == 0) return 0;
    const int bytes = R * (fp32 ? 4 : 8) * (cv ? 2 : 1);
    if (bytes % 16 != 0 || bytes / 16 > 256) return 0;
    const int cpr = bytes / 16;
    // One or two lanes a row read their own long stretches of entries, a cache line a
    // lane, where a column per lane reads a row's entries once for all its lanes.
    // Measured at 200,000 rows, column per lane / slab: one lane, FP64, thirteen
    // entries 26.3 / 15.4 us, seventeen 32.5 / 33.7, twenty-three 42.2 / 60.4; FP32
    // seventeen 23.9 / 15.8, twenty-three 31.8 / 35.3; two lanes, FP64, seventeen 33.8 /
    // 26.3, twenty-three 43.5 / 46.0, FP32 twenty-three 34.2 / 31.0, thirty-three 48.2 /
    // 61.8. The fewer rows in flight, the longer they may be (59,000 rows, two lanes,
    // forty-nine entries 0.55 to 0.7 of the time; 130,000 rows, one lane, thirty-three
    // 1.1 to 1.2).
    const int64_t most = cpr == 1 ? (fp32 ? 19 : 15) : cpr == 2 ? (fp32 ? 27 : 19) : INT32_MAX;
    if (A.nbr > 100000 && A.nnzb > most * A.nbr) return 0;
    const int64_t g = (A.nbr + 256 / cpr - 1) / (256 / cpr);
    const bool longrow = g_b1g_min_grid > 0 && A.nnzb >= kLongRow * A.nbr;
    return g >= (longrow ? std::min(g_b1g_min_grid, kLongRowMinGrid) : g_b1g_min_grid) ? cpr : 0;
}

template <typename S, bool CV>
hipError_t go_b1g(int cpr, const BsrDev &A, const void *X, void *Y, const EpiArgs &e, int grid, hipStream_t st) {
    hipLaunchKernelGGL((k_spmm_b1g<S, CV>), dim3(grid), dim3(256), 0, st, A.nbr, cpr, g_uniform_rows ? A.ulen : 0,
                       xcd_walk(A, grid, (int64_t)cpr * 16), A.row_ptr, A.col_ind, static_cast<const S *>(A.vals),
                       static_cast<const S *>(X), static_cast<S *>(Y), e);
    return hipGetLastError();
}

// Lanes per row of the slab layout for this launch shape, or 0 when it does
// not apply: b = 1, real matrix, R of 16 or 32, g_b1v_bytes a lane.
int b1v_lpr(const BsrDev &A, bool fp32, bool cv, int R) {
    if (A.b != 1 || A.is_complex || g_b1v_bytes == 0 || (R != 16 && R != 32)) return 0;
    const int vt = (fp32 ? 4 : 8) * (cv ? 2 : 1);
    const int bytes = g_b1v_bytes > 0 ? g_b1v_bytes : (vt == 16 ? 32 : 16);
    const int cpl = bytes / vt;
    if (cpl < 1 || R % cpl != 0) return 0;
    const int lpr = R / cpl;
    const int64_t rows_per_wg = (int64_t)kWaves * (64 / lpr);
    if ((A.nbr + rows_per_wg - 1) / rows_per_wg < g_b1v_min_grid) return 0;
    return lpr;
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

template <typename S, bool CV, int LPR, int CPL>
hipError_t go_b1v(const BsrDev &A, const void *X, void *Y, const EpiArgs &e, int grid, hipStream_t st) {
    hipLaunchKernelGGL((k_spmm_b1v<S, CV, LPR, CPL>), dim3(grid), dim3(64 * kWaves), 0, st, A.nbr,
                       g_uniform_rows ? A.ulen : 0, xcd_walk(A, grid, (int64_t)LPR * CPL * (CV ? 2 : 1) * sizeof(S)),
                       A.row_ptr, A.col_ind, static_cast<const S *>(A.vals), static_cast<const S *>(X),
                       static_cast<S *>(Y), e);
    return hipGetLastError();
}

// The slab launch for lpr = b1v_lpr(...) (nonzero).
template <typename S, bool CV>
hipError_t by_b1v(int lpr, const BsrDev &A, const void *X, void *Y, int R, const EpiArgs &e, int grid,
                  hipStream_t st) {
    constexpr int VT = (int)sizeof(S) * (CV ? 2 : 1);
    auto pick = [&](auto bytes_c) -> hipError_t {
        constexpr int CPL = decltype(bytes_c)::value / VT;
        if constexpr (CPL < 1 || 16 % CPL != 0 || (CPL * VT) % 16 != 0) {
            return hipErrorInvalidValue;
        } else {
            if (R == 16) return go_b1v<S, CV, 16 / CPL, CPL>(A, X, Y, e, grid, st);
            if constexpr (32 / CPL <= 64) return go_b1v<S, CV, 32 / CPL, CPL>(A, X, Y, e, grid, st);
            return hipErrorInvalidValue;
        }
    };
    const int bytes = R / lpr * VT;
    if (bytes == 16) return pick(std::integral_constant<int, 16>{});
    if (bytes == 32) return pick(std::integral_constant<int, 32>{});
    if (bytes == 64) return pick(std::integral_constant<int, 64>{});
    return hipErrorInvalidValue;
}


// ------------------------------------------------------------ reduction
// Neumaier-compensated sum of a and b into (s, c): s + c carries the exact
// sum to twice the working precision (Neumaier 1974, "improved Kahan").
__device__ __forceinline__ void two_sum_acc(double &s, double &c, double x) {
    const double t = s + x;
    c += (fabs(s) >= fabs(x)) ? ((s - t) + x) : ((x - t) + s);
    s = t;
}

// One (dot, column) pair per wave; blockIdx.y selects a step of a batched
// reduction (partials and out advance by their step strides).
__global__ __launch_bounds__(256) void k_reduce(const double2 *__restrict__ partials, int ngroups,
                                                int ndot, int R, double2 *__restrict__ out, int64_t pstride,
                                                int64_t ostride) {
    partials += (int64_t)blockIdx.y * pstride;
    out += (int64_t)blockIdx.y * ostride;
    const int lane = threadIdx.x & 63;
    const int pair = blockIdx.x * (int)(blockDim.x >> 6) + (threadIdx.x >> 6);
    const int npairs = ndot * R;
    if (pair >= npairs) return;
    const int d = pair / R;
    const int u = pair - d * R;
    // compensated FP64 sums over the workgroup partials, then a fixed xor tree
    double sx = 0.0, cx = 0.0, sy = 0.0, cy = 0.0;
    // 32 loads in flight per lane (all of a 2048-workgroup launch's partials
    // in one round trip) before they are summed in order
    constexpr int B = 32;
    for (int g0 = lane; g0 < ngroups; g0 += 64 * B) {
        double2 p[B];
#pragma unroll
        for (int q = 0; q < B; ++q) {
            const int gi = g0 + 64 * q;
            p[q] = gi < ngroups ? partials[((int64_t)gi * ndot + d) * R + u] : double2{0.0, 0.0};
        }
#pragma unroll
        for (int q = 0; q < B; ++q) {
            two_sum_acc(sx, cx, p[q].x);
            two_sum_acc(sy, cy, p[q].y);
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double ox = __shfl_xor(sx, off), ocx = __shfl_xor(cx, off);
        const double oy = __shfl_xor(sy, off), ocy = __shfl_xor(cy, off);
        cx += ocx;
        cy += ocy;
        two_sum_acc(sx, cx, ox);
        two_sum_acc(sy, cy, oy);
    }
    if (lane == 0) out[pair] = double2{sx + cx, sy + cy};
}

// --------------------------------------------------------------- samples
__device__ __forceinline__ uint64_t mix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__global__ __launch_bounds__(256) void k_samples(int kind, uint64_t seed, int64_t rows, int R,
                                                 double scale, int complex_vec, void *out) {
    const int64_t n = rows * (int64_t)R;
    const uint64_t ms = mix64(seed);
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = t / R;
        const int64_t c = t - i * R;
        const uint64_t h = mix64(mix64(ms ^ (uint64_t)i) ^ (uint64_t)c);
        if (kind == 0) { // RademacherSign (rsatb/calc/rs_ldos.hpp:256-264)
            const double v = (h & 1ull) ? scale : -scale;
            if (complex_vec) static_cast<double2 *>(out)[t] = double2{v, 0.0};
            else static_cast<double *>(out)[t] = v;
        } else { // phase 2 pi u, u = top 53 bits * 2^-53
            const double u = (double)(h >> 11) * (1.0 / 9007199254740992.0);
            double sn, cs;
            sincos(6.283185307179586476925286766559 * u, &sn, &cs);
            static_cast<double2 *>(out)[t] = double2{cs * scale, sn * scale};
        }
    }
}

__global__ __launch_bounds__(256) void k_f64_to_f32(const double *__restrict__ in,
                                                    float *__restrict__ out, int64_t n) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (int64_t)gridDim.x * blockDim.x)
        out[t] = (float)in[t];
}

// Block gather: one block of m scalars per row of threads' grid-stride walk.
__global__ __launch_bounds__(256) void k_block_perm(const double *__restrict__ in,
                                                    const int32_t *__restrict__ perm,
                                                    double *__restrict__ out, int64_t nblk, int64_t m) {
    const int64_t n = nblk * m;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t p = t / m;
        out[t] = in[(int64_t)perm[p] * m + (t - p * m)];
    }
}

__global__ __launch_bounds__(256) void k_stage(const double *__restrict__ in, int in_complex,
                                               void *__restrict__ out, int out_complex,
                                               int out_fp32, int64_t n) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (int64_t)gridDim.x * blockDim.x) {
        const double re = in_complex ? in[2 * t] : in[t];
        const double im = in_complex ? in[2 * t + 1] : 0.0;
        if (out_fp32) {
            float *o = static_cast<float *>(out);
            if (out_complex) {
                o[2 * t] = (float)re;
                o[2 * t + 1] = (float)im;
            } else {
                o[t] = (float)re;
            }
        } else {
            double *o = static_cast<double *>(out);
            if (out_complex) {
                o[2 * t] = re;
                o[2 * t + 1] = im;
            } else {
                o[t] = re;
            }
        }
    }
}

// Row-major -> column-major within every b x b block (real or complex).
__global__ __launch_bounds__(256) void k_block_transpose(const double *__restrict__ in,
                                                         double *__restrict__ out, int64_t nnzb,
                                                         int b, int cplx) {
    const int64_t per = (int64_t)b * b;
    const int64_t n = nnzb * per;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t s = t / per;
        const int e = (int)(t - s * per);
        const int r = e / b, c = e - (e / b) * b; // source (r, c) row-major
        const int64_t dst = s * per + (int64_t)c * b + r;
        if (cplx) {
            out[2 * dst] = in[2 * t];
            out[2 * dst + 1] = in[2 * t + 1];
        } else {
            out[dst] = in[t];
        }
    }
}

int grid_1d(int64_t n) {
    int64_t g = (n + 255) / 256;
    if (g > 8192) g = 8192;
    if (g < 1) g = 1;
    return (int)g;
}

} // namespace

namespace {
// Workgroups of the VALU SpMM: kWaves waves of 64 / lpr block rows each.
int valu_grid(int64_t nbr, int lpr) {
    const int G = 64 / lpr;
    const int64_t rows_per_wg = (int64_t)kWaves * G;
    int64_t g = (nbr + rows_per_wg - 1) / rows_per_wg;
    if (g > kMaxGrid) g = kMaxGrid;
    if (g < 1) g = 1;
    return (int)g;
}
} // namespace

// Workgroups of the VALU SpMM for this operand, by the layout the launch takes.
static int valu_launch_grid(const BsrDev &A, VecMode vm, int R) {
    if (b1v_lpr(A, vm.fp32, vm.complex_vec, R) == 0)
        if (const int cpr = b1g_cpr(A, vm.fp32, vm.complex_vec, R)) {
            const int64_t rpb = 256 / cpr, g = ((A.nbr + rpb - 1) / rpb + 7) / 8 * 8; // whole XCD rounds
            return (int)(g > kMaxGrid ? kMaxGrid : g);
        }
    const int g = valu_grid(A.nbr, valu_lpr(A, vm.fp32, vm.complex_vec, R));
    return b1v_lpr(A, vm.fp32, vm.complex_vec, R) ? (g + 7) / 8 * 8 : g;
}

// Whether few columns on many short rows stay with the VALU kernel, whose waves take
// eight rows where an MFMA wave (4,096 fit the chip) takes one and pays a row's
// chain of loads for little. Measured, us a step, MFMA / VALU: FP32, a block of 13 a
// row, R = 4: 4,000 rows 8.4 / 7.8, 8,000 11.9 / 8.2, 20,000 25.6 / 16.6; five blocks of
// 13, 8,000 rows 19.6 / 16.4, 20,000 39.9 / 33.8, seventeen, 14,000 rows 68 / 59 (FP64 no
// slower; a lane sums the dots of a row or two, where compensation gains nothing); a
// block of 8, 20,000 rows 19.5 / 14.1, 6,000 8.9 / 11.5, of 9 21.1 / 17.5, of 12 20.3 /
// 21.6; FP64, a block of 13, 8,000 rows 13.5 / 11.9, complex vectors 13.4 / 14.0; a
// block of 8, 60,000 rows 54.8 / 43.8.
static bool valu_rows(const BsrDev &A, bool fp32, bool cv, int R) {
    if (A.nbr < 3500 || R > 16) return false;
    const int64_t k = A.nnzb * A.b / A.nbr; // columns of an average row's panel
    const bool one = k <= 13;               // about a block a row
    if (A.is_complex) return fp32 && one && R <= 8 && (A.b == 13 ? A.nbr >= 6000 : A.b == 8 && A.nbr >= 12000);
    if (!fp32) return one && !cv && R <= 8 && (A.b == 13 ? A.nbr >= 6000 : A.b == 8 && A.nbr >= 12000);
    if (A.b == 13) return one || (R <= 8 && A.nbr >= 6000);
    if (A.nbr < 12000) return false;
    if (A.b == 8) return one || (k <= 24 && R <= 8);
    return one && R <= (A.nbr >= 40000 ? 8 : 4) && (A.b <= 10 || (cv && A.b <= 12));
}

// The MFMA launch shape for this operand, or nt = 0 when it takes the VALU
// kernel: b >= 8 with a gather table (below, an MFMA's 16 rows are mostly
// padding). One chunk of the fewest tiles that hold the W columns (two chunks
// past 256), then halved into more chunks while the launch has too few waves. e: columns a lane moves per access, 16 bytes
// where W is a multiple.
// The VALU kernel these widths took before feeds the matrix through scalar
// loads and waits on them: 13-orbital diamond with vacancies, 1,596 rows, W =
// 40: 63.9 us a product there; W = 16 60.8 us.
static MfmaShape mfma_shape(const BsrDev &A, bool fp32, bool cv, int R) {
    MfmaShape s;
    const int W = R * (cv ? 2 : 1);
    if (A.b < 8 || !A.mrow || (A.is_complex && !cv) || W > 512 || valu_rows(A, fp32, cv, R)) return s;
    s.nchunks = W > 256 ? 2 : 1;
    const int per = (W + s.nchunks - 1) / s.nchunks; // columns a chunk must hold
    static const int even64[] = {2, 4, 6, 8, 12, 16}, even32[] = {2, 4, 8, 12, 16}, half32[] = {2, 4, 8, 16};
    static const int odd[] = {1, 4};
    const int *set = odd;
    int n = 2;
    s.e = 1;
    if (W % 2 == 0 && (cv || W > 16)) {
        s.e = fp32 && W % 4 == 0 ? 4 : 2;
        set = !fp32 ? even64 : s.e == 4 ? even32 : half32;
        n = !fp32 ? 6 : s.e == 4 ? 5 : 4;
    }
    int k = 0;
    while (k + 1 < n && 16 * set[k] < per) ++k;
    s.nt = set[k];
    if (s.e == 1) // odd widths past 64: two or four waves of four tiles, not sixteen tiles mostly empty
        while (64 * s.nchunks < W && s.nchunks < kWaves) s.nchunks *= 2;
    if (s.nt == 2) s.e = 2; // two tiles hold one 8-byte (FP32) or 16-byte (FP64) access a lane
    if (16 * s.nt * s.nchunks < W) return MfmaShape{};
    const bool pow2 = (s.nt & (s.nt - 1)) == 0;
    s.mask = !pow2 || 16 * s.nt * s.nchunks != W || (s.e == 1 && s.nt > 1) || (fp32 && s.e == 2 && s.nt > 2);
    while (!s.mask && s.nt > 2 && s.nchunks < kWaves &&
           (s.nt > g_mfma.ntcap || A.nbr * s.nchunks < kMfmaSplitWaves)) {
        s.nt /= 2;
        s.nchunks *= 2;
        if (s.nt == 2) s.e = 2;
    }
    return s;
}

// Workgroups a shape's launch asks for (capped further by what is resident).
static int mfma_grid_req(const BsrDev &A, const MfmaShape &s) {
    int64_t g = (A.nbr * s.nchunks + kWaves - 1) / kWaves;
    if (g > kMaxGrid) g = kMaxGrid;
    return (int)(((g + 7) / 8) * 8); // whole XCD rounds (kMaxGrid is a multiple of 8)
}

int spmm_launch_grid(const BsrDev &A, VecMode vm, int R) {
    if (mfma_shape(A, vm.fp32, vm.complex_vec, R).nt > 0) {
        // the grid the step launch of this operand takes (kernels differ in
        // their resident capacity)
        EpiArgs e;
        e.mode = EPI_STEP;
        int g = 0;
        t_mfma_grid_query = true;
        const hipError_t he = launch_spmm(A, vm, nullptr, nullptr, R, e, nullptr, &g);
        t_mfma_grid_query = false;
        return he == hipSuccess ? g : kMaxGrid;
    }
    return valu_launch_grid(A, vm, R);
}

hipError_t launch_spmm(const BsrDev &A, VecMode vm, const void *X, void *Y, int R,
                       const EpiArgs &e, hipStream_t stream, int *grid_out) {
    if (R < 1 || R > 256 || A.b < 1 || A.b > 16) return hipErrorInvalidValue;
    if (A.is_complex && !vm.complex_vec) return hipErrorInvalidValue;
    const MfmaShape ms = mfma_shape(A, vm.fp32, vm.complex_vec, R);
    if (ms.nt > 0) {
        const int W = R * (vm.complex_vec ? 2 : 1), grid = mfma_grid_req(A, ms);
        if (A.is_complex) return launch_mfma_cplx(ms, A, vm.fp32, X, Y, W, R, e, grid, stream, grid_out);
        return vm.fp32 ? launch_mfma_f32(ms, A, vm.complex_vec, X, Y, W, R, e, grid, stream, grid_out)
                       : launch_mfma_f64(ms, A, vm.complex_vec, X, Y, W, R, e, grid, stream, grid_out);
    }
    // sized by the layout the launch takes (the wide b = 1 layout covers twice
    // the rows per workgroup)
    const int grid = valu_launch_grid(A, vm, R);
    if (grid_out) *grid_out = grid;
    const void *ops[] = {X, Y, e.xs, e.xp, e.psi, e.qm, e.qz, e.qp};
    bool ok = true;
    for (const void *o : ops) ok = ok && aligned16(o);
    if (ok) {
        if (const int lpr = b1v_lpr(A, vm.fp32, vm.complex_vec, R)) {
            if (vm.fp32) return vm.complex_vec ? by_b1v<float, true>(lpr, A, X, Y, R, e, grid, stream)
                                               : by_b1v<float, false>(lpr, A, X, Y, R, e, grid, stream);
            return vm.complex_vec ? by_b1v<double, true>(lpr, A, X, Y, R, e, grid, stream)
                                  : by_b1v<double, false>(lpr, A, X, Y, R, e, grid, stream);
        }
        if (const int cpr = b1g_cpr(A, vm.fp32, vm.complex_vec, R)) {
            if (vm.fp32) return vm.complex_vec ? go_b1g<float, true>(cpr, A, X, Y, e, grid, stream)
                                               : go_b1g<float, false>(cpr, A, X, Y, e, grid, stream);
            return vm.complex_vec ? go_b1g<double, true>(cpr, A, X, Y, e, grid, stream)
                                  : go_b1g<double, false>(cpr, A, X, Y, e, grid, stream);
        }
    }
    if (!vm.fp32) {
        if (A.is_complex) return by_block<double, true, true>(A, X, Y, R, e, grid, stream);
        if (vm.complex_vec) return by_block<double, false, true>(A, X, Y, R, e, grid, stream);
        return by_block<double, false, false>(A, X, Y, R, e, grid, stream);
    }
    if (A.is_complex) return by_block<float, true, true>(A, X, Y, R, e, grid, stream);
    if (vm.complex_vec) return by_block<float, false, true>(A, X, Y, R, e, grid, stream);
    return by_block<float, false, false>(A, X, Y, R, e, grid, stream);
}

int spmm_max_grid() { return kMaxGrid; }

void set_xcd_map(int on) { g_mfma.xcd_map = on ? 1 : 0; }
void set_mfma_ntcap(int nt) { g_mfma.ntcap = nt; }
void set_mfma_grid_cap(int g) { g_mfma.grid_cap = g >= 8 && g <= kMaxGrid ? (g / 8) * 8 : 0; }
void set_b1_wide(int mode) { g_b1_wide = mode == 0 || mode == 1 ? mode : 2; }
void set_uniform_rows(int on) { g_uniform_rows = on != 0; }
void set_b1_slab(int bytes) { g_b1v_bytes = bytes == 0 || bytes == 16 || bytes == 32 || bytes == 64 ? bytes : -1; }
void set_b1_slab_min_grid(int g) {
    g_b1v_min_grid = g >= 0 ? g : 512;
    g_b1g_min_grid = g >= 0 ? g : 1024;
}
hipError_t launch_block_transpose(const double *in, double *out, int64_t nnzb, int b, bool cplx,
                                  hipStream_t stream) {
    hipLaunchKernelGGL(k_block_transpose, dim3(grid_1d(nnzb * b * b)), dim3(256), 0, stream, in,
                       out, nnzb, b, cplx ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_reduce(const double2 *partials, int ngroups, int ndot, int R, double2 *out,
                         hipStream_t stream) {
    return launch_reduce_steps(partials, 0, ngroups, ndot, R, out, 0, 1, stream);
}

hipError_t launch_reduce_steps(const double2 *partials, int64_t pstride, int ngroups, int ndot, int R,
                               double2 *out, int64_t ostride, int nsteps, hipStream_t stream) {
    if (nsteps < 1) return hipSuccess;
    // one wave (one dot and column) a workgroup: the strided partial loads
    // spread over as many compute units as there are sums
    const int npairs = ndot * R;
    for (int s0 = 0; s0 < nsteps; s0 += 65535) // grid.y holds at most 65535
        hipLaunchKernelGGL(k_reduce, dim3(npairs, (unsigned)std::min(nsteps - s0, 65535)), dim3(64), 0, stream,
                           partials + (int64_t)s0 * pstride, ngroups, ndot, R, out + (int64_t)s0 * ostride, pstride,
                           ostride);
    return hipGetLastError();
}

hipError_t launch_samples(int kind, uint64_t seed, int64_t rows, int R, double scale,
                          bool complex_vec, void *out, hipStream_t stream) {
    hipLaunchKernelGGL(k_samples, dim3(grid_1d(rows * R)), dim3(256), 0, stream, kind, seed, rows,
                       R, scale, complex_vec ? 1 : 0, out);
    return hipGetLastError();
}

hipError_t launch_f64_to_f32(const double *in, float *out, int64_t n, hipStream_t stream) {
    hipLaunchKernelGGL(k_f64_to_f32, dim3(grid_1d(n)), dim3(256), 0, stream, in, out, n);
    return hipGetLastError();
}

hipError_t launch_block_perm(const double *in, const int32_t *perm, double *out, int64_t nblk, int64_t m,
                             hipStream_t stream) {
    if (nblk <= 0 || m <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_block_perm, dim3(grid_1d(nblk * m)), dim3(256), 0, stream, in, perm, out, nblk, m);
    return hipGetLastError();
}

hipError_t launch_stage(const double *in, bool in_complex, void *out, bool out_complex,
                        bool out_fp32, int64_t n, hipStream_t stream) {
    hipLaunchKernelGGL(k_stage, dim3(grid_1d(n)), dim3(256), 0, stream, in, in_complex ? 1 : 0,
                       out, out_complex ? 1 : 0, out_fp32 ? 1 : 0, n);
    return hipGetLastError();
}

} // namespace rg
