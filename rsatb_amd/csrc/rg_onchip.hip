// The moment loop of a small scalar operator, one sample column per workgroup.
//
// An operator of a few thousand rows (b = 1, real matrix, orthogonal form)
// spends its moment loop in launches: 4 us a step at 336 rows, most of it the
// chain launch, index load, gather, dot fold. The columns of the sample block
// never meet, and a column of 4096 complex numbers is 64 KB: here one
// workgroup keeps its column's t_n in LDS (twice, so that one barrier a step is
// enough), t_{n-1} in registers, and runs thousands of steps in one launch.
// What bounds a step is the chain barrier, LDS gather, FMAs, LDS write; rows of
// at most ENT entries keep them in registers, longer ones read them from L2,
// whose 64 bytes a clock and CU then bound it (12 bytes an entry), so the
// launch rule caps the entries.
// Measured, R = 16 real (complex), FP64, a step of a 1,024-moment run against
// one launch a step: four entries a row, 336 rows 0.5 us (0.7) against 4.0
// (4.4), 1,024 rows 0.7 (1.1) against 4.1 (4.5), 4,096 rows 1.1 (1.9) against 4.1
// (4.4), 8,000 rows 3.3 against 5.0 (entries read every step); thirteen entries,
// 336 rows 0.6 against 5.4, 1,600 rows 3.7 against 6.1.
//
// Every row's products and its epilogue are the operations of the launched
// kernels (k_spmm, k_spmm_b1v) in their order, so the vectors are the same bit
// for bit; a step's dots are summed in another fixed order (lanes of a wave,
// then waves), and leave as the step's sums, with no partials to reduce.
#include "rg_internal.h"

#include <algorithm>
#include <type_traits>

namespace rg {
namespace {

constexpr int kMaxThreads = 1024;
constexpr int kRing = 64; // steps whose wave sums wait in LDS

template <typename S> struct V2;
// native vectors (held in registers where HIP's own struct types go to memory)
typedef double dv2 __attribute__((ext_vector_type(2)));
typedef float fv2 __attribute__((ext_vector_type(2)));
template <> struct V2<double> { using T = dv2; };
template <> struct V2<float> { using T = fv2; };

__device__ __forceinline__ void mac(double &acc, double a, double x) { acc = __builtin_fma(a, x, acc); }
__device__ __forceinline__ void mac(float &acc, float a, float x) { acc = __builtin_fmaf(a, x, acc); }
__device__ __forceinline__ void mac(dv2 &acc, double a, dv2 x) {
    acc.x = __builtin_fma(a, x.x, acc.x);
    acc.y = __builtin_fma(a, x.y, acc.y);
}
__device__ __forceinline__ void mac(fv2 &acc, float a, fv2 x) {
    acc.x = __builtin_fmaf(a, x.x, acc.x);
    acc.y = __builtin_fmaf(a, x.y, acc.y);
}
// alpha v + beta s
__device__ __forceinline__ double affine(double v, double alpha, double beta, double s) {
    return __builtin_fma(alpha, v, beta * s);
}
__device__ __forceinline__ float affine(float v, double alpha, double beta, float s) {
    return (float)__builtin_fma(alpha, (double)v, beta * (double)s);
}
__device__ __forceinline__ dv2 affine(dv2 v, double alpha, double beta, dv2 s) {
    return dv2{affine(v.x, alpha, beta, s.x), affine(v.y, alpha, beta, s.y)};
}
__device__ __forceinline__ fv2 affine(fv2 v, double alpha, double beta, fv2 s) {
    return fv2{affine(v.x, alpha, beta, s.x), affine(v.y, alpha, beta, s.y)};
}
__device__ __forceinline__ double sub(double a, double b) { return a - b; }
__device__ __forceinline__ float sub(float a, float b) { return a - b; }
__device__ __forceinline__ dv2 sub(dv2 a, dv2 b) { return dv2{a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ fv2 sub(fv2 a, fv2 b) { return fv2{a.x - b.x, a.y - b.y}; }
// (re, im) += conj(a) b in FP64; a self-dot is real
__device__ __forceinline__ void dot(double &re, double &, double a, double b, bool) { re = __builtin_fma(a, b, re); }
__device__ __forceinline__ void dot(double &re, double &im, dv2 a, dv2 b, bool self) {
    re = __builtin_fma(a.x, b.x, __builtin_fma(a.y, b.y, re));
    if (!self) im = __builtin_fma(a.x, b.y, __builtin_fma(-a.y, b.x, im));
}
__device__ __forceinline__ double wide(float v) { return (double)v; }
__device__ __forceinline__ double wide(double v) { return v; }
__device__ __forceinline__ dv2 wide(fv2 v) { return dv2{(double)v.x, (double)v.y}; }
__device__ __forceinline__ dv2 wide(dv2 v) { return v; }

template <int CTRL, int ROWS> __device__ __forceinline__ double dpp_add(double v) {
    int lo, hi;
    __builtin_memcpy(&lo, &v, 4);
    __builtin_memcpy(&hi, reinterpret_cast<const char *>(&v) + 4, 4);
    lo = __builtin_amdgcn_update_dpp(0, lo, CTRL, ROWS, 0xf, false);
    hi = __builtin_amdgcn_update_dpp(0, hi, CTRL, ROWS, 0xf, false);
    double o;
    __builtin_memcpy(&o, &lo, 4);
    __builtin_memcpy(reinterpret_cast<char *>(&o) + 4, &hi, 4);
    return v + o;
}
// the wave's sum, in lane 63: row shifts by 1, 2, 4, 8, then broadcasts of the
// rows' last lanes (data parallel primitives: no LDS round trips)
__device__ __forceinline__ double wave_sum63(double v) {
    v = dpp_add<0x111, 0xf>(v);
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);
    v = dpp_add<0x143, 0xc>(v);
    return v;
}

// RPT rows a thread (rows tid + k blockDim), ENT register entries a row (0:
// read every step). t0, t1: [n][R] state; first: t0 holds the samples and the
// launch starts with step 0 (t1 = A~ t0 and its three dots), else it goes on
// from t0, t1; `steps` doubled steps; raw: dots of the launch's first step on,
// [step][3][R].
template <typename S, bool CV, int RPT, int ENT>
__global__ __launch_bounds__(kMaxThreads) void k_onchip(int n, const int64_t *__restrict__ row_ptr,
                                                        const int32_t *__restrict__ col_ind,
                                                        const S *__restrict__ vals, void *t0v, void *t1v, int R,
                                                        int first, int steps, OnchipWindow w,
                                                        double2 *__restrict__ raw) {
    using V = std::conditional_t<CV, typename V2<S>::T, S>;
    constexpr int NV = CV ? 3 : 2; // sums a step keeps: <2|2>, Re and Im <2|1>
    extern __shared__ __align__(16) unsigned char lds[];
    V *xl = reinterpret_cast<V *>(lds); // two vectors of n
    double *ring = reinterpret_cast<double *>(lds + (((size_t)2 * n * sizeof(V) + 15) & ~(size_t)15));
    V *T0 = static_cast<V *>(t0v), *T1 = static_cast<V *>(t1v);
    const int u = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
    const int lane = tid & 63, wave = tid >> 6, nw = nt >> 6;

    V xp[RPT], xs[RPT];
    int s0[RPT], cnt[RPT];
    int32_t ec[RPT][ENT > 0 ? ENT : 1];
    S ev[RPT][ENT > 0 ? ENT : 1];
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int r = tid + k * nt;
        const bool in = r < n;
        xp[k] = in ? T0[(int64_t)r * R + u] : V{};
        xs[k] = in && !first ? T1[(int64_t)r * R + u] : V{};
        s0[k] = in ? (int)row_ptr[r] : 0;
        cnt[k] = in ? (int)(row_ptr[r + 1] - row_ptr[r]) : 0;
#pragma unroll
        for (int e = 0; e < (ENT > 0 ? ENT : 0); ++e) {
            const bool have = e < cnt[k];
            ec[k][e] = have ? col_ind[s0[k] + e] : (in ? r : 0);
            ev[k][e] = have ? vals[s0[k] + e] : S(0);
        }
        if (in) xl[r] = first ? xp[k] : xs[k];
    }
    __syncthreads();

    auto row = [&](int k, const V *x) -> V {
        V acc{};
        if constexpr (ENT > 0) {
            V g[ENT];
#pragma unroll
            for (int e = 0; e < ENT; ++e) g[e] = x[ec[k][e]];
#pragma unroll
            for (int e = 0; e < ENT; ++e) mac(acc, ev[k][e], g[e]);
        } else {
            int e = 0;
            for (; e + 4 <= cnt[k]; e += 4) {
                int32_t c[4];
                S a[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    c[q] = col_ind[s0[k] + e + q];
                    a[q] = vals[s0[k] + e + q];
                }
                V g[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) g[q] = x[c[q]];
#pragma unroll
                for (int q = 0; q < 4; ++q) mac(acc, a[q], g[q]);
            }
            for (; e < cnt[k]; ++e) mac(acc, vals[s0[k] + e], x[col_ind[s0[k] + e]]);
        }
        return acc;
    };

    int cur = 0;
    if (first) {
        double d[5] = {0, 0, 0, 0, 0}; // <0|0>, <0|1> (re, im), <1|1>
        double none = 0.0;
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const int r = tid + k * nt;
            xs[k] = affine(row(k, xl), w.alpha1, w.beta1, xp[k]);
            if (r >= n) xs[k] = V{};
            dot(d[0], none, wide(xp[k]), wide(xp[k]), true);
            dot(d[1], d[2], wide(xp[k]), wide(xs[k]), false);
            dot(d[3], none, wide(xs[k]), wide(xs[k]), true);
            if (r < n) xl[n + r] = xs[k];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = wave_sum63(d[q]);
        if (lane == 63)
#pragma unroll
            for (int q = 0; q < 4; ++q) ring[wave * 4 + q] = d[q];
        __syncthreads();
        if (tid == 0) {
            double s[4] = {0, 0, 0, 0};
            for (int q = 0; q < nw; ++q)
                for (int j = 0; j < 4; ++j) s[j] += ring[q * 4 + j];
            raw[u] = double2{s[0], 0.0};
            raw[R + u] = double2{s[1], s[2]};
            raw[2 * R + u] = double2{s[3], 0.0};
        }
        raw += 3 * R;
        cur = 1;
        __syncthreads(); // ring is free again
    }

    for (int st = 0; st < steps; ++st) {
        const V *x = xl + cur * n;
        V *y = xl + (cur ^ 1) * n;
        double d0 = 0.0, d1 = 0.0, d2 = 0.0, none = 0.0;
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            const int r = tid + k * nt;
            V t = sub(affine(row(k, x), w.alpha, w.beta, xs[k]), xp[k]);
            if (r < n) y[r] = t;
            else t = V{};
            dot(d0, none, wide(t), wide(t), true);
            dot(d1, d2, wide(t), wide(xs[k]), false);
            xp[k] = xs[k];
            xs[k] = t;
        }
        d0 = wave_sum63(d0);
        d1 = wave_sum63(d1);
        if (CV) d2 = wave_sum63(d2);
        const int slot = st % kRing;
        if (lane == 63) {
            double *o = ring + (slot * nw + wave) * NV;
            o[0] = d0;
            o[1] = d1;
            if (CV) o[2] = d2;
        }
        cur ^= 1;
        __syncthreads();
        // a full ring (or the last steps): one thread a step sums its waves
        if (slot == kRing - 1 || st == steps - 1) {
            if (tid <= slot) {
                double s[3] = {0, 0, 0};
                for (int q = 0; q < nw; ++q)
                    for (int j = 0; j < NV; ++j) s[j] += ring[(tid * nw + q) * NV + j];
                double2 *o = raw + (int64_t)(st - slot + tid) * 3 * R;
                o[u] = double2{s[0], 0.0};
                o[R + u] = double2{s[1], s[2]};
            }
            __syncthreads();
        }
    }

#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int r = tid + k * nt;
        if (r < n) {
            T0[(int64_t)r * R + u] = xp[k];
            T1[(int64_t)r * R + u] = xs[k];
        }
    }
}

template <typename S, bool CV, int RPT, int ENT>
hipError_t go(const BsrDev &A, int nt, size_t lds, void *t0, void *t1, int R, bool first, int steps,
              const OnchipWindow &w, double2 *raw, hipStream_t st) {
    auto *kernel = &k_onchip<S, CV, RPT, ENT>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_onchip<S, CV, RPT, ENT>), dim3(R), dim3(nt), lds, st, (int)A.nbr, A.row_ptr, A.col_ind,
                       static_cast<const S *>(A.vals), t0, t1, R, first ? 1 : 0, steps, w, raw);
    return hipGetLastError();
}

template <typename S, bool CV>
hipError_t by_rows(const BsrDev &A, int rpt, int nt, size_t lds, void *t0, void *t1, int R, bool first, int steps,
                   const OnchipWindow &w, double2 *raw, hipStream_t st) {
    const bool few = A.maxlen <= 4;
    if (rpt == 1) {
        if (few) return go<S, CV, 1, 4>(A, nt, lds, t0, t1, R, first, steps, w, raw, st);
        if (A.maxlen <= 16) return go<S, CV, 1, 16>(A, nt, lds, t0, t1, R, first, steps, w, raw, st);
        return go<S, CV, 1, 0>(A, nt, lds, t0, t1, R, first, steps, w, raw, st);
    }
    if (rpt == 2)
        return few ? go<S, CV, 2, 4>(A, nt, lds, t0, t1, R, first, steps, w, raw, st)
                   : go<S, CV, 2, 0>(A, nt, lds, t0, t1, R, first, steps, w, raw, st);
    if (rpt == 4)
        return few ? go<S, CV, 4, 4>(A, nt, lds, t0, t1, R, first, steps, w, raw, st)
                   : go<S, CV, 4, 0>(A, nt, lds, t0, t1, R, first, steps, w, raw, st);
    return go<S, CV, 8, 0>(A, nt, lds, t0, t1, R, first, steps, w, raw, st);
}

// LDS: two copies of a column and the ring of sums.
size_t onchip_lds(int n, VecMode vm, int nt) {
    const size_t elem = (size_t)(vm.complex_vec ? 2 : 1) * (vm.fp32 ? 4 : 8);
    return (((size_t)2 * n * elem + 15) & ~(size_t)15) + (size_t)kRing * (nt / 64) * 3 * 8;
}

void onchip_shape(int n, int *rpt, int *nt) {
    *rpt = n <= 1024 ? 1 : n <= 2048 ? 2 : n <= 4096 ? 4 : 8;
    *nt = ((n + *rpt - 1) / *rpt + 63) / 64 * 64;
}

} // namespace

// Two columns in LDS (at most 8192 rows, about 4,900 of complex FP64). Rows in
// registers have no other bound. Entries read every step are bound to 384 KB (R =
// 16, FP64, 20,800 entries 3.7 us a step, launched 6.1; 39,900 on rows of thirteen
// 7.3, launched 6.0), and cost a step about as much for one column as for 256, where
// a launched step is 3.6 us for one. Measured, on the chip / launched, us a step: 2,500
// rows of seven 3.6 / 3.9 (R = 1), 3.8 / 4.8 (16); of thirteen, FP64 5.7 / 4.4, 6.0 / 5.8,
// FP32 3.5 / 4.3; past 4,096 rows (eight a thread) 4,097 of three 4.1 / 3.6, ragged
// 4.5 / 4.8 (16), 7,000 of three 5.3 / 3.6, 5.4 / 4.6 (16), 10.9 / 44 (256).
bool onchip_fits(const BsrDev &A, VecMode vm, int R) {
    if (A.b != 1 || A.is_complex || A.nbr < 1 || A.nbr > 8192 || A.maxlen < 0) return false;
    int rpt, nt;
    onchip_shape((int)A.nbr, &rpt, &nt);
    if (onchip_lds((int)A.nbr, vm, nt) > (size_t)156 << 10) return false;
    const bool held = (A.maxlen <= 4 && rpt <= 4) || (A.maxlen <= 16 && rpt == 1);
    if (held) return true;
    if (A.nnzb * (vm.fp32 ? 8 : 12) > 384 << 10) return false;
    const int row_bytes = R * (vm.complex_vec ? 2 : 1) * (vm.fp32 ? 4 : 8);
    if (A.nbr > 4096) // FP32 to 6,000 rows of four and five, read together: 4.0 / 4.7 (16)
        return row_bytes >= 512 || (R >= 16 && ((A.nbr <= 5000 && A.nnzb <= 24000) ||
                                                (vm.fp32 && A.nbr <= 6000 && A.nnzb >= 4 * A.nbr && A.nnzb <= 5 * A.nbr)));
    return A.nbr <= 2048 || vm.fp32 || R >= 16 || A.nnzb <= 24000;
}

hipError_t launch_onchip(const BsrDev &A, VecMode vm, void *t0, void *t1, int R, bool first, int steps,
                         const OnchipWindow &w, double2 *raw, hipStream_t st) {
    if (R < 1 || steps < 0 || !onchip_fits(A, vm, R)) return hipErrorInvalidValue;
    int rpt, nt;
    onchip_shape((int)A.nbr, &rpt, &nt);
    const size_t lds = onchip_lds((int)A.nbr, vm, nt);
    if (vm.fp32)
        return vm.complex_vec ? by_rows<float, true>(A, rpt, nt, lds, t0, t1, R, first, steps, w, raw, st)
                              : by_rows<float, false>(A, rpt, nt, lds, t0, t1, R, first, steps, w, raw, st);
    return vm.complex_vec ? by_rows<double, true>(A, rpt, nt, lds, t0, t1, R, first, steps, w, raw, st)
                          : by_rows<double, false>(A, rpt, nt, lds, t0, t1, R, first, steps, w, raw, st);
}

} // namespace rg
