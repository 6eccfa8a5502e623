// The MFMA SpMM: dense-block products Y = epi(A X) on the matrix cores.
//
// Block rows with b >= 8. The block row's stored blocks are concatenated
// along K, so a row of 17 blocks of 13 x 13 is one 13 x 221 panel times a
// gathered 221 x W panel of X (W real columns: R, or 2R for complex vectors),
// tiled as 16 x 16 x 4 MFMAs: only the 13 -> 16 row padding is wasted (81 % of
// issued MFMA work is useful), K is padded once per block row (221 -> 224).
//
// Operand layouts of v_mfma_{f64,f32}_16x16x4 (lane l, i = l % 16, g = l / 16):
//   A[i][k = g], B[k = g][j = i]; accumulator element v holds D[4 g + v][i]
//   for f32 and D[4 v + g][i] for f64 (both measured on gfx950).
// N is relabelled (col_of below) so that X, Y and the recurrence operands
// move as coalesced 16-byte loads/stores, and the (re, im) halves of a
// complex column sit in the same lane (tiles t, t + 1, t even), so the complex
// dots need no shuffles.
// Blocks are stored column-major on the device, so the 13 rows of one A
// column are contiguous and the A fragment load is coalesced.
//
// Widths. NT tiles of 16 columns per wave and nchunks waves side by side cover
// 16 NT nchunks >= W columns; when that is more than W (MASK) the lanes past
// the last column load the last columns again, compute on them and store
// nothing: no vector is padded in memory, only MFMA slots are spent.
//
// Complex matrices (CM): A's (re, im) come as one pair per lane and every pair
// of tiles takes four real products, re += ar xr - ai xi, im += ar xi + ai xr.
//
// Each translation unit that includes this file instantiates one family
// (launch_mfma_f64, launch_mfma_f32, launch_mfma_cplx), so they compile side
// by side.
#pragma once

#include "rg_internal.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace rg {

namespace {

constexpr int kMfmaWaves = 4; // waves per workgroup

template <typename S> struct Acc4;
template <> struct Acc4<double> { typedef double T __attribute__((ext_vector_type(4))); };
template <> struct Acc4<float> { typedef float T __attribute__((ext_vector_type(4))); };

__device__ __forceinline__ Acc4<double>::T mfma16(double a, double b, Acc4<double>::T c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ Acc4<float>::T mfma16(float a, float b, Acc4<float>::T c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// s += x with the rounding error carried in c (TwoSum, Knuth 1969: exact
// for any s and x; s + c is the sum to about twice the working precision).
__device__ __forceinline__ void two_sum_add(double &s, double &c, double x) {
    const double t = s + x;
    const double bp = t - s;
    c += (s - (t - bp)) + (x - bp);
    s = t;
}

// Column mapping: tile t of lane i holds real column
//   col(t, i) = (t / E) 16 E + i E + t % E,   E | NT,
// so every load of E elements (16 bytes where W allows it) of a row's 16 lanes
// covers 16 E contiguous columns, and with E even the (re, im) halves of a
// complex column stay in one lane, next to each other in t. With MASK, `w`
// columns are left in the chunk (a multiple of E): the accesses past them go
// to the last E columns instead, and are not stored.
template <int NT, int E, bool MASK> struct ColMap {
    int off[MASK ? NT / E : 1];
    int i, w;
    __device__ __forceinline__ ColMap(int i_, int w_) : i(i_), w(w_) {
        if constexpr (MASK) {
#pragma unroll
            for (int q = 0; q < NT / E; ++q) off[q] = min(q * 16 * E + i * E, w - E);
        }
    }
    __device__ __forceinline__ int at(int q) const {
        if constexpr (MASK) return off[q];
        else return q * 16 * E + i * E;
    }
    __device__ __forceinline__ bool live(int q) const {
        if constexpr (MASK) return q * 16 * E + i * E < w;
        else return true;
    }
    __device__ __forceinline__ int col(int t) const { return (t / E) * 16 * E + i * E + t % E; }
};

// native vectors of the non-temporal builtins
typedef float f4nt __attribute__((ext_vector_type(4)));
typedef float f2nt __attribute__((ext_vector_type(2)));

// v[t] = row[col(t)]; NTL: a non-temporal load (data read once, kept out of the
// way of the gathered rows in L2)
template <typename S, int NT, int E, bool MASK, bool NTL = false>
__device__ __forceinline__ void load_cols(const S *__restrict__ row, const ColMap<NT, E, MASK> &cm, S (&v)[NT]) {
    constexpr int B = E * (int)sizeof(S);
#pragma unroll
    for (int q = 0; q < NT / E; ++q) {
        const S *p = row + cm.at(q);
        if constexpr (B == 16) {
            f4nt w;
            if constexpr (NTL) w = __builtin_nontemporal_load(reinterpret_cast<const f4nt *>(p));
            else w = *reinterpret_cast<const f4nt *>(p);
            __builtin_memcpy(&v[q * E], &w, 16);
        } else if constexpr (B == 8 && E == 2) {
            f2nt w;
            if constexpr (NTL) w = __builtin_nontemporal_load(reinterpret_cast<const f2nt *>(p));
            else w = *reinterpret_cast<const f2nt *>(p);
            __builtin_memcpy(&v[q * E], &w, 8);
        } else {
            static_assert(E == 1, "one column, or 8 or 16 bytes");
            v[q] = NTL ? __builtin_nontemporal_load(p) : *p;
        }
    }
}

// row[col(t)] = v[t] for the live columns, non-temporal (an output row is not
// read again in the launch)
template <typename S, int NT, int E, bool MASK>
__device__ __forceinline__ void store_cols(S *__restrict__ row, const ColMap<NT, E, MASK> &cm, const S (&v)[NT]) {
    constexpr int B = E * (int)sizeof(S);
#pragma unroll
    for (int q = 0; q < NT / E; ++q) {
        if (!cm.live(q)) continue;
        S *p = row + cm.at(q);
        if constexpr (B == 16) {
            f4nt w;
            __builtin_memcpy(&w, &v[q * E], 16);
            __builtin_nontemporal_store(w, reinterpret_cast<f4nt *>(p));
        } else if constexpr (B == 8 && E == 2) {
            f2nt w;
            __builtin_memcpy(&w, &v[q * E], 8);
            __builtin_nontemporal_store(w, reinterpret_cast<f2nt *>(p));
        } else {
            __builtin_nontemporal_store(v[q], p);
        }
    }
}

// Per-lane FP64 dot sums of the MFMA SpMM, ND dots x NT tiles. The
// precision form (S = float) keeps a compensation term beside every sum:
// its terms are products of two FP32 values, exact in FP64, so summing them
// with TwoSum is the compensated dot product Dot2 (Ogita, Rump and Oishi
// 2005) with an exact product step. The compensation terms live in LDS (a
// slot per lane, dot and tile; cl points at this lane's first), not in
// registers, so the kernel keeps its occupancy. The FP64 form sums with
// FMAs, as the reference's own dots do.
template <typename S, int ND, int NT> struct DotAcc {
    static constexpr bool kComp = sizeof(S) == 4;
    double s[ND][NT];
    double *cl = nullptr;
    __device__ __forceinline__ double &comp(int d, int t) { return cl[(d * NT + t) * 64]; }
    // comp(d, t) += x without reading it back (each lane owns its slots)
    __device__ __forceinline__ void comp_add(int d, int t, double x) {
        __hip_atomic_fetch_add(&cl[(d * NT + t) * 64], x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                s[d][t] = 0.0;
                if constexpr (kComp) {
                    if (cl) comp(d, t) = 0.0;
                }
            }
    }
    // s[d][t] += a1 b1 + a2 b2, in that order
    __device__ __forceinline__ void add2(int d, int t, double a1, double b1, double a2, double b2) {
        if constexpr (kComp) {
            double err = 0.0;
            two_sum_add(s[d][t], err, a1 * b1);
            two_sum_add(s[d][t], err, a2 * b2);
            comp_add(d, t, err);
        } else {
            s[d][t] = __builtin_fma(a2, b2, __builtin_fma(a1, b1, s[d][t]));
        }
    }
    __device__ __forceinline__ void add(int d, int t, double a, double b) {
        if constexpr (kComp) {
            double err = 0.0;
            two_sum_add(s[d][t], err, a * b);
            comp_add(d, t, err);
        } else {
            s[d][t] = __builtin_fma(a, b, s[d][t]);
        }
    }
    // the lane groups (lanes i, i + 16, i + 32, i + 48) of every tile folded
    // into one sum, its compensation included
    __device__ __forceinline__ double fold4(int d, int t) {
        double v = s[d][t];
        if constexpr (kComp) {
            double c = comp(d, t);
#pragma unroll
            for (int off = 16; off < 64; off <<= 1) {
                const double o = __shfl_xor(v, off), oc = __shfl_xor(c, off);
                two_sum_add(v, c, o);
                c += oc;
            }
            return v + c;
        } else {
            v += __shfl_xor(v, 16);
            v += __shfl_xor(v, 32);
            return v;
        }
    }
};

template <typename S, int NT, int MODE>
using MfmaDots = DotAcc<S, (epi_ndot(MODE) > 0 ? epi_ndot(MODE) : 1), NT>;

// With PRE (the FP64 step), pxs and pxp arrive holding the Xs and Xp values
// of the first output rows (loaded by the kernel before the row's K loop), and
// each pass loads the next pass's values into them as soon as its own are
// consumed, so the epilogue's reads overlap its compute instead of stalling.
template <typename S, int NT, int E, bool MASK, int MODE, bool CV, bool PRE>
__device__ __forceinline__ void mfma_epilogue(const typename Acc4<S>::T (&acc)[NT], int64_t br,
                                              int b, int W, int col0, const ColMap<NT, E, MASK> &cm, int g,
                                              const EpiArgs &e, MfmaDots<S, NT, MODE> &dacc,
                                              S *__restrict__ Y, S (&pxs)[NT], S (&pxp)[NT]) {
    const S *__restrict__ XS = static_cast<const S *>(e.xs);
    const S *__restrict__ XP = static_cast<const S *>(e.xp);
    const S *__restrict__ PSI = static_cast<const S *>(e.psi);
    // one output row per pass keeps the epilogue's registers low: the barrier
    // holds the next passes' loads back. Written out: picking a pass's
    // accumulator element in a loop took a tree of branches per tile
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        __builtin_amdgcn_sched_barrier(0);
        // accumulator element v holds row 4 v + g (f64) or 4 g + v (f32)
        const int r = sizeof(S) == 8 ? 4 * v + g : 4 * g + v;
        if (r >= b) continue;
        const int64_t base = (br * b + r) * (int64_t)W + col0;
        S y[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) y[t] = acc[t][v];
        // the next pass's output row of this lane (PRE loads it early)
        const int rn = sizeof(S) == 8 ? 4 * (v + 1) + g : 4 * g + v + 1;
        const bool next = PRE && v < 3 && rn < b;
        const int64_t base_n = (br * b + rn) * (int64_t)W + col0;
        if constexpr (MODE != EPI_PLAIN) {
            S xs[NT];
            if constexpr (PRE) {
#pragma unroll
                for (int t = 0; t < NT; ++t) xs[t] = pxs[t];
            } else {
                load_cols<S, NT, E, MASK, true>(XS + base, cm, xs);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t)
                y[t] = (S)__builtin_fma(e.alpha, (double)y[t], e.beta * (double)xs[t]);
            if constexpr (MODE == EPI_STEP || MODE == EPI_PLAINSTEP || MODE == EPI_ADJ) {
                if constexpr (PRE) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) y[t] = y[t] - pxp[t];
                    if (next) load_cols<S, NT, E, MASK, true>(XP + base_n, cm, pxp);
                } else {
                    S xp[NT];
                    load_cols<S, NT, E, MASK, true>(XP + base, cm, xp);
#pragma unroll
                    for (int t = 0; t < NT; ++t) y[t] = y[t] - xp[t];
                }
            }
            if constexpr (MODE == EPI_ADJ) {
                const S *qs[3] = {static_cast<const S *>(e.qm), static_cast<const S *>(e.qz),
                                  static_cast<const S *>(e.qp)};
                const double cs[3] = {e.cm, e.cz, e.cp};
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    S qv[NT];
                    load_cols<S, NT, E, MASK, true>(qs[q] + base, cm, qv);
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        y[t] = (S)__builtin_fma(cs[q], (double)qv[t], (double)y[t]);
                }
            }
            // dots (FP64): conj(a) b per complex column (t, t+1) or per
            // real column; a self-dot is real and keeps no imaginary part
            auto dot = [&](int d, const S (&a)[NT], const S (&bb)[NT], bool self) {
                if constexpr (CV) {
#pragma unroll
                    for (int t = 0; t < NT; t += 2) {
                        const double ar = a[t], ai = a[t + 1], br_ = bb[t], bi = bb[t + 1];
                        dacc.add2(d, t, ai, bi, ar, br_);
                        if (!self) dacc.add2(d, t + 1, -ai, br_, ar, bi);
                    }
                } else {
#pragma unroll
                    for (int t = 0; t < NT; ++t) dacc.add(d, t, (double)a[t], (double)bb[t]);
                }
            };
            if constexpr (MODE == EPI_FIRST) {
                dot(0, xs, xs, true);
                dot(1, xs, y, false);
                dot(2, y, y, true);
            } else if constexpr (MODE == EPI_STEP) {
                dot(0, y, y, true);
                dot(1, y, xs, false);
                if constexpr (PRE) {
                    if (next) load_cols<S, NT, E, MASK, true>(XS + base_n, cm, pxs);
                }
            } else if constexpr (MODE == EPI_PLAINSTEP) {
                S ps[NT];
                load_cols<S, NT, E, MASK, true>(PSI + base, cm, ps);
                dot(0, ps, y, false);
            }
        }
        store_cols<S, NT, E, MASK>(Y + base, cm, y);
    }
}

// Per-workgroup dot partials of the MFMA SpMMs: the lane groups of every
// column are folded, then the waves sharing a column chunk, into
// e.partials[(blockIdx.x * NDOT + d) * R + u].
template <typename S, int NT, int E, bool MASK, int MODE, bool CV>
__device__ __forceinline__ void mfma_dot_partials(MfmaDots<S, NT, MODE> &dacc, int wave,
                                                  const ColMap<NT, E, MASK> &cm, int g, int nchunks, int R,
                                                  const EpiArgs &e) {
    constexpr int NDOT = epi_ndot(MODE);
    constexpr int CW = 16 * NT;
    if constexpr (NDOT > 0) {
        // per wave: CW real columns -> CW/2 complex (or CW real) units
        constexpr int UPC = CV ? CW / 2 : CW;
        __shared__ double2 sm[kMfmaWaves][UPC];
        // unrolled: the sums stay in registers (a loop over d would index them)
#pragma unroll
        for (int d = 0; d < NDOT; ++d) {
            // fold the four lane groups (rows of the 16-row tile) of every column
            double f[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) f[t] = dacc.fold4(d, t);
            if (g == 0) {
#pragma unroll
                for (int t = 0; t < NT; t += (CV ? 2 : 1)) {
                    const int uu = CV ? cm.col(t) / 2 : cm.col(t);
                    sm[wave][uu] = CV ? double2{f[t], f[t + 1]} : double2{f[t], 0.0};
                }
            }
            __syncthreads();
            for (int u = threadIdx.x; u < R; u += blockDim.x) {
                const int ch = (u * (CV ? 2 : 1)) / CW;
                const int uu = u - ch * UPC;
                double2 acc2 = double2{0.0, 0.0};
                for (int w = ch; w < kMfmaWaves; w += nchunks) {
                    acc2.x += sm[w][uu].x;
                    acc2.y += sm[w][uu].y;
                }
                e.partials[((int64_t)blockIdx.x * NDOT + d) * R + u] = acc2;
            }
            __syncthreads();
        }
    }
}

// Register prefetch depth: PD buffers, PD - 1 K steps in flight per wave.
// Narrow kernels (few tiles a step) need more steps in flight to cover a
// gather's latency and have the registers; at sixteen FP64 tiles the kernels
// hold one wave per SIMD and the rows in flight already fill an XCD's L2.
// Measured at the diamond 24^3 sandwich, R = 128 complex, depth 2 / 3 / 4:
// FP64 plain 4727 / 4522 / 4583 us, FP64 step 5348 / 5474 / 5510 us; FP32
// (plain, step) at 2: 2329, 2699 us, at 3: 2414, 2749 us, at 4: 2450, 3421
// us; at the diamond 8^3 sandwich, R = 64: FP64 plain 107.4 us at 2, 105.6 at 3,
// FP64 step 114.9 / 116.4 us, FP32 plain 54.0 us at 3, 70.8 at 4.
template <typename S, int NT, int MODE, bool CV, bool CM> constexpr int prefetch_depth() {
    if (NT == 1) return 8;
    if (NT == 2) return 6;
    if (NT == 4) return 4;
    if (sizeof(S) == 8) return MODE == EPI_PLAIN ? 3 : 2;
    return NT == 16 && (MODE == EPI_STEP || (CV && MODE == EPI_PLAIN)) ? 2 : 3;
}

// What bounds it, at 4,096 rows of 17 blocks of 13 x 13, FP64, W = 128 (103 us;
// parts of the kernel taken out one at a time): the MFMAs alone are 51 us (a
// fifth of it padding 13 rows to 16), operands from L2 add 20, their misses 12,
// and the epilogue's streams 25. Waves of a SIMD in step, a start or a priority
// apart, deeper buffers, and fetching the next row's first steps during the
// epilogue all left the time where it was or raised it. Two waves a SIMD as launch
// bounds keep the accumulators in VGPRs (at sixteen FP64 tiles they need the
// AGPRs and one wave): with the written-out epilogue and the masked row pick,
// FP64 W = 128 107.5 -> 102.5 us plain and 109.6 -> 103.1 step; 8,000 rows, FP32
// W = 256 216 -> 205, 236 -> 223 and 290 -> 253 us (first).
template <typename S, int NT, int E, bool MASK, int MODE, bool CV, bool CM>
__global__ __launch_bounds__(256, (sizeof(S) == 8 && NT > 8) ? 1 : 2) void k_spmm_mfma(int64_t nbr, int b,
                                                   const MfmaRow *__restrict__ rows,
                                                   const int32_t *__restrict__ xrow,
                                                   const S *__restrict__ vals,
                                                   const S *__restrict__ zero,
                                                   const S *__restrict__ X, S *__restrict__ Y,
                                                   int W, int R, int nchunks, int xcd_map,
                                                   EpiArgs e) {
    using A4 = typename Acc4<S>::T;
    typedef S A2 __attribute__((ext_vector_type(2)));
    using AT = std::conditional_t<CM, A2, S>;
    constexpr int PD = prefetch_depth<S, NT, MODE, CV, CM>();
    static_assert(8 * PD - 4 <= kXrowSpare, "the gather table's spare entries cover the fetches past a row");
    static_assert(!CV || E % 2 == 0, "a complex column's halves share a lane");
    static_assert(!CM || CV, "complex matrices act on complex vectors");
    constexpr int NDOT = epi_ndot(MODE);
    constexpr int CW = 16 * NT; // real columns per chunk
    // the FP64 step at sixteen tiles (one wave per SIMD, registers to spare)
    // loads its epilogue's inputs ahead
    constexpr bool PRE = sizeof(S) == 8 && NT == 16 && MODE == EPI_STEP && !CM && !MASK;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15;
    const int g = lane >> 4;
    // nchunks divides kMfmaWaves: a wave keeps chunk wave % nchunks
    const int col0 = (wave % nchunks) * CW;
    const ColMap<NT, E, MASK> cm(i, W - col0);
    // Workgroups are dispatched round-robin over the 8 XCDs; with xcd_map each
    // XCD walks its own contiguous eighth of the block rows, so the rows in
    // flight on one XCD (and their gathered neighbours) stay close together
    // in its L2.
    // Position p computes block row rows[p].br; the eighths are cut by rows, not
    // by whole regions: an operator of ten regions gave two XCDs twice the
    // rows of the others.
    int64_t r_lo = 0, r_hi = nbr;
    int64_t kq = blockIdx.x, nk = gridDim.x;
    if (xcd_map) {
        const int x = blockIdx.x & 7;
        kq = blockIdx.x >> 3;
        nk = gridDim.x >> 3;
        r_lo = nbr * x / 8;
        r_hi = nbr * (x + 1) / 8;
    }
    const int64_t total = (r_hi - r_lo) * nchunks;

    MfmaDots<S, NT, MODE> dacc;
    if constexpr (MfmaDots<S, NT, MODE>::kComp && NDOT > 0) {
        __shared__ double comp_lds[kMfmaWaves * NDOT * NT * 64];
        dacc.cl = comp_lds + wave * NDOT * NT * 64 + lane;
    }
    dacc.zero();

    const int32_t m0 = g == 0 ? -1 : 0, m1 = g == 1 ? -1 : 0, m2 = g == 2 ? -1 : 0, m3 = g == 3 ? -1 : 0;
    for (int64_t it = kq * kMfmaWaves + wave; it < total; it += nk * kMfmaWaves) {
        const int64_t pos = r_lo + it / nchunks;
        // one 16-byte scalar load: a row's chain is this, the table, the gathers
        const MfmaRow row = rows[pos];
        const int64_t br = row.br, s0 = row.s0;
        const int nblk = row.nblk;
        int64_t kb = (int64_t)row.at4 * 4;
        const int nsteps = (nblk * b + 3) >> 2;
        // the first output rows' Xs, Xp values, in flight during the K loop
        S pxs[NT], pxp[NT];
        if constexpr (PRE) {
            const int64_t base0 = (br * b + g) * (int64_t)W + col0; // FP64 pass 0: row g < 8 <= b
            load_cols<S, NT, E, MASK, true>(static_cast<const S *>(e.xs) + base0, cm, pxs);
            load_cols<S, NT, E, MASK, true>(static_cast<const S *>(e.xp) + base0, cm, pxp);
        }

        A4 acc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = A4{0, 0, 0, 0};

        // Step st covers K columns 4 st .. 4 st + 3 of the row's column-major
        // b x K panel (element (i, k) at s0 b^2 + k b + i); lane group g takes
        // column k = 4 st + g, its X row from the gather table (wave-uniform
        // scalar loads, so no vector load sits between the steps' loads). PD
        // register buffers: steps st + 1 .. st + PD - 1 are in flight while
        // step st's MFMAs run. Past the row's K the table still names a valid row
        // (the row's own to the end of its last step); a = 0 there.
        // Lanes outside the panel (i >= b, or k >= K) load their A element from
        // `zero` (one element, 0) instead of selecting on loaded data, which
        // would hold up the next loads.
        const int K = nblk * b;
        const AT *__restrict__ panel = reinterpret_cast<const AT *>(vals) + s0 * (int64_t)b * b;
        int fst = 0; // next step to fetch
        int32_t nx0 = xrow[kb], nx1 = xrow[kb + 1], nx2 = xrow[kb + 2], nx3 = xrow[kb + 3];
        auto fetch = [&](AT &a, S (&bv)[NT]) {
            // masks, not a select: the compiler branched over the lane groups
            const int64_t xr = (nx0 & m0) | (nx1 & m1) | (nx2 & m2) | (nx3 & m3);
            const int k = 4 * fst + g;
            a = __builtin_nontemporal_load((i < b && k < K) ? panel + (int64_t)k * b + i
                                                            : reinterpret_cast<const AT *>(zero));
            load_cols<S, NT, E, MASK>(X + xr * W + col0, cm, bv);
            // the next step's table entries (in range: the table keeps 8 PD - 4 <= 64 spare entries)
            kb += 4;
            nx0 = xrow[kb];
            nx1 = xrow[kb + 1];
            nx2 = xrow[kb + 2];
            nx3 = xrow[kb + 3];
            ++fst;
        };
        auto mma = [&](AT a, const S (&bv)[NT]) {
            if constexpr (CM) {
                // the four real products of (ar + i ai)(xr + i xi); the two
                // tiles' chains alternate
#pragma unroll
                for (int t = 0; t < NT; t += 2) {
                    acc[t] = mfma16(a.x, bv[t], acc[t]);
                    acc[t + 1] = mfma16(a.x, bv[t + 1], acc[t + 1]);
                }
#pragma unroll
                for (int t = 0; t < NT; t += 2) {
                    acc[t] = mfma16(-a.y, bv[t + 1], acc[t]);
                    acc[t + 1] = mfma16(a.y, bv[t], acc[t + 1]);
                }
            } else {
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[t] = mfma16(a, bv[t], acc[t]);
            }
        };
        // PD register buffers, PD - 1 steps in flight. The fetches are
        // unconditional (up to 2 PD - 2 steps past the row: their A lanes read
        // the zero word and their X rows are valid), so the wait before each
        // MFMA group counts only the later buffers' loads on every path.
        if constexpr (PD >= 4) {
            // Deep buffers stop at the row's end: running on, as below, would fetch
            // up to 2 PD - 2 steps of nothing, four times the loads of a row of one
            // block (20,000 rows of a block of 9, one column, FP64, 28.9 -> 17.0 us; 640
            // rows of seventeen, W = 16, 9.2 -> 8.5; W = 48 13.2 -> 12.3; W = 40, 1,596
            // rows of 13, 24.0 -> 24.6).
            AT ab[PD];
            S bb[PD][NT];
            if (nsteps >= PD) {
#pragma unroll
                for (int q = 0; q < PD - 1; ++q) fetch(ab[q], bb[q]);
                int st = 0;
                for (; st + 2 * PD - 1 <= nsteps; st += PD) {
#pragma unroll
                    for (int q = 0; q < PD; ++q) {
                        fetch(ab[(q + PD - 1) % PD], bb[(q + PD - 1) % PD]);
                        mma(ab[q], bb[q]);
                    }
                }
                // PD - 1 steps are in flight, up to PD - 1 more to come
#pragma unroll
                for (int q = 0; q < PD; ++q) {
                    if (st + q + PD - 1 < nsteps) fetch(ab[(q + PD - 1) % PD], bb[(q + PD - 1) % PD]);
                    if (q < PD - 1 || st + q < nsteps) mma(ab[q], bb[q]);
                }
#pragma unroll
                for (int q = 0; q < PD - 2; ++q)
                    if (st + PD + q < nsteps) mma(ab[q], bb[q]);
            } else {
#pragma unroll
                for (int q = 0; q < PD - 1; ++q)
                    if (q < nsteps) fetch(ab[q], bb[q]);
#pragma unroll
                for (int q = 0; q < PD - 1; ++q)
                    if (q < nsteps) mma(ab[q], bb[q]);
            }
        } else if (nsteps > 0) {
            AT ab[PD];
            S bb[PD][NT];
#pragma unroll
            for (int q = 0; q < PD - 1; ++q) fetch(ab[q], bb[q]);
            for (int st = 0; st < nsteps; st += PD) {
#pragma unroll
                for (int q = 0; q < PD; ++q) {
                    fetch(ab[(q + PD - 1) % PD], bb[(q + PD - 1) % PD]);
                    if (st + q < nsteps) mma(ab[q], bb[q]);
                }
            }
        }

        mfma_epilogue<S, NT, E, MASK, MODE, CV, PRE>(acc, br, b, W, col0, cm, g, e, dacc, Y, pxs, pxp);
    }

    mfma_dot_partials<S, NT, E, MASK, MODE, CV>(dacc, wave, cm, g, nchunks, R, e);
}

// Workgroups of one MFMA SpMM kernel that are resident at once, at most
// per_cu_cap per compute unit, a multiple of 8 (whole XCD rounds), at most
// spmm_max_grid(). With no queued workgroups the grid-stride loop walks the
// schedule's regions in order on every XCD. The cap is two for eight tiles and
// more (their rows in flight fill the L2; diamond 24^3, R = 128 complex, grids
// of 2048 / resident / 512 / 256: FP64 plain 4994 / 4807 / 4638 / 4808 us,
// FP32 2886 / 2870 / 2560 / 2709 us) and four below, whose waves hide less
// latency each (FP64 step at two against four: 1,200 rows of b = 9, W = 128 at
// four tiles 36.9 / 31.0 us; 4,096 rows of b = 13, W = 32 48.8 / 45.8 us).
int mfma_resident_grid(const void *kernel, int per_cu_cap) {
    int dev = 0, ncu = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu < 1 ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64 * kMfmaWaves, 0) != hipSuccess || per_cu < 1)
        return 512;
    const int64_t g = ((int64_t)std::min(per_cu, per_cu_cap) * ncu / 8) * 8;
    return (int)std::max<int64_t>(8, std::min<int64_t>(g, spmm_max_grid()));
}

template <typename S, int NT, int E, bool MASK, int MODE, bool CV, bool CM>
hipError_t go_mfma(const MfmaShape &s, const BsrDev &A, const void *X, void *Y, int W, int R, const EpiArgs &e,
                   int grid_req, hipStream_t st, int *grid_out) {
    auto *kernel = &k_spmm_mfma<S, NT, E, MASK, MODE, CV, CM>;
    static std::atomic<int> resident{0};
    int res = resident.load(std::memory_order_relaxed);
    if (res == 0) {
        res = mfma_resident_grid(reinterpret_cast<const void *>(kernel), NT <= 4 ? 4 : 2);
        resident.store(res, std::memory_order_relaxed);
    }
    const int grid = std::min(grid_req, g_mfma.grid_cap > 0 ? g_mfma.grid_cap : res);
    if (grid_out) *grid_out = grid;
    if (t_mfma_grid_query) return hipSuccess;
    // the zero element of lanes outside a panel: 16 aligned zero bytes of the
    // gather table's spare entries
    const int32_t *xrow = reinterpret_cast<const int32_t *>(A.mrow + A.nbr);
    const void *zero = xrow + A.xlen;
    hipLaunchKernelGGL((k_spmm_mfma<S, NT, E, MASK, MODE, CV, CM>), dim3(grid), dim3(64 * kMfmaWaves), 0, st, A.nbr,
                       (int)A.b, A.mrow, xrow, static_cast<const S *>(A.vals), static_cast<const S *>(zero),
                       static_cast<const S *>(X), static_cast<S *>(Y), W, R, s.nchunks, g_mfma.xcd_map, e);
    return hipGetLastError();
}

template <typename S, int NT, int E, bool MASK, bool CV, bool CM>
hipError_t by_mode(const MfmaShape &s, const BsrDev &A, const void *X, void *Y, int W, int R, const EpiArgs &e,
                   int grid, hipStream_t st, int *grid_out) {
    switch (e.mode) {
    case EPI_PLAIN: return go_mfma<S, NT, E, MASK, EPI_PLAIN, CV, CM>(s, A, X, Y, W, R, e, grid, st, grid_out);
    case EPI_FIRST: return go_mfma<S, NT, E, MASK, EPI_FIRST, CV, CM>(s, A, X, Y, W, R, e, grid, st, grid_out);
    case EPI_STEP: return go_mfma<S, NT, E, MASK, EPI_STEP, CV, CM>(s, A, X, Y, W, R, e, grid, st, grid_out);
    case EPI_PLAINSTEP: return go_mfma<S, NT, E, MASK, EPI_PLAINSTEP, CV, CM>(s, A, X, Y, W, R, e, grid, st, grid_out);
    default: return go_mfma<S, NT, E, MASK, EPI_ADJ, CV, CM>(s, A, X, Y, W, R, e, grid, st, grid_out);
    }
}

// The instance of a shape (mfma_shape makes no others).
template <typename S, bool CV, bool CM>
hipError_t by_shape(const MfmaShape &s, const BsrDev &A, const void *X, void *Y, int W, int R, const EpiArgs &e,
                    int grid, hipStream_t st, int *grid_out) {
    constexpr int EF = 16 / (int)sizeof(S); // columns of a 16-byte access
#define RG_MFMA_CASE(NT_, E_, MASK_)                                                                             \
    if (s.nt == NT_ && s.e == E_ && s.mask == MASK_)                                                             \
        return by_mode<S, NT_, E_, MASK_, CV, CM>(s, A, X, Y, W, R, e, grid, st, grid_out);
    RG_MFMA_CASE(2, 2, false)
    RG_MFMA_CASE(4, EF, false)
    RG_MFMA_CASE(8, EF, false)
    RG_MFMA_CASE(16, EF, false)
    RG_MFMA_CASE(2, 2, true)
    RG_MFMA_CASE(4, EF, true)
    RG_MFMA_CASE(8, EF, true)
    RG_MFMA_CASE(12, EF, true)
    RG_MFMA_CASE(16, EF, true)
    if constexpr (EF == 2) {
        RG_MFMA_CASE(6, 2, true)
    } else {
        RG_MFMA_CASE(4, 2, true)
        RG_MFMA_CASE(8, 2, true)
        RG_MFMA_CASE(16, 2, true)
    }
    if constexpr (!CV) {
        RG_MFMA_CASE(1, 1, false)
        RG_MFMA_CASE(1, 1, true)
        RG_MFMA_CASE(4, 1, true)
    }
#undef RG_MFMA_CASE
    return hipErrorInvalidValue;
}

} // namespace
} // namespace rg
