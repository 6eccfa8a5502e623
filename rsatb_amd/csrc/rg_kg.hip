// Kubo-Greenwood sequences of a scalar (b = 1, real) operator, and the node
// sums of the spectrum.
//
// One launch a moment in place of seven. The base vector x = T_m r is gathered
// once for four products, H x (the recurrence) and B_a x (the left vectors),
// whose matrices share H's pattern, and blockIdx.y adds the three right
// recurrences, which never meet the base. No dots are formed. A lane owns 16
// contiguous bytes of a row and a workgroup holds as many whole rows
// as fit 256 lanes, so any width of whole 16-byte pieces is taken. Every
// product and recurrence is the launched kernels' operations in their order.
// Bound: the six vectors a moment that are stored (HBM), and the gather.
// Measured at graphene 128 x 128 (65,536 rows of four, R = 16, FP64): seven
// launches 7.5 us each, 52 us a moment; 23 us a moment here (126 MB, 5.5 TB/s).
#include "rg_internal.h"

#include <algorithm>
#include <type_traits>

namespace rg {
namespace {

template <typename S> __device__ __forceinline__ S fmas(S a, S b, S c);
template <> __device__ __forceinline__ double fmas(double a, double b, double c) { return __builtin_fma(a, b, c); }
template <> __device__ __forceinline__ float fmas(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double affine(double v, double alpha, double beta, double s) {
    return __builtin_fma(alpha, v, beta * s);
}
__device__ __forceinline__ float affine(float v, double alpha, double beta, float s) {
    return (float)__builtin_fma(alpha, (double)v, beta * (double)s);
}

template <typename S>
__global__ __launch_bounds__(256) void k_kg_moment(int64_t n, int ulen, const int64_t *__restrict__ row_ptr,
                                                   const int32_t *__restrict__ col_ind, KgMoment a) {
    constexpr int E = 16 / (int)sizeof(S); // scalars a lane owns
    typedef S C16 __attribute__((ext_vector_type(E)));
    const int cpr = a.cpr, rpb = 256 / cpr;
    const int lr = (int)threadIdx.x / cpr, q = (int)threadIdx.x - lr * cpr;
    const int64_t br = (int64_t)blockIdx.x * rpb + lr;
    if (lr >= rpb || br >= n) return;
    const int64_t W = (int64_t)cpr * E, idx = br * W + (int64_t)q * E;
    const int64_t s0 = ulen > 0 ? br * ulen : row_ptr[br], s1 = ulen > 0 ? s0 + ulen : row_ptr[br + 1];
    const S *__restrict__ h = static_cast<const S *>(a.h);
    auto at = [&](const void *p, int64_t off) -> C16 { return *reinterpret_cast<const C16 *>(static_cast<const S *>(p) + off); };
    auto put = [&](void *p, C16 v) { *reinterpret_cast<C16 *>(static_cast<S *>(p) + idx) = v; };
    auto recur = [&](C16 y, const void *x, const void *xp) -> C16 {
        const C16 xs = at(x, idx);
        const bool first = xp == nullptr;
        C16 o;
#pragma unroll
        for (int i = 0; i < E; ++i) o[i] = affine(y[i], first ? a.alpha1 : a.alpha, first ? a.beta1 : a.beta, xs[i]);
        if (!first) {
            const C16 p = at(xp, idx);
#pragma unroll
            for (int i = 0; i < E; ++i) o[i] = o[i] - p[i];
        }
        return o;
    };
    constexpr int U = 4; // entries whose indices and gathers are in flight together
    if (blockIdx.y > 0) {
        // R_m = 2 A~ R_{m-1} - R_{m-2} of one axis
        const int64_t off = (int64_t)(blockIdx.y - 1) * a.right_stride;
        const S *x = static_cast<const S *>(a.rx) + off;
        const S *xp = a.rxp ? static_cast<const S *>(a.rxp) + off : nullptr;
        C16 y = C16(S(0));
        int64_t s = s0;
        for (; s + U <= s1; s += U) {
            int64_t c[U];
            S v[U];
            C16 g[U];
#pragma unroll
            for (int t = 0; t < U; ++t) {
                c[t] = col_ind[s + t];
                v[t] = h[s + t];
            }
#pragma unroll
            for (int t = 0; t < U; ++t) g[t] = at(x, c[t] * W + (int64_t)q * E);
#pragma unroll
            for (int t = 0; t < U; ++t)
#pragma unroll
                for (int i = 0; i < E; ++i) y[i] = fmas<S>(v[t], g[t][i], y[i]);
        }
        for (; s < s1; ++s) {
            const C16 g = at(x, (int64_t)col_ind[s] * W + (int64_t)q * E);
#pragma unroll
            for (int i = 0; i < E; ++i) y[i] = fmas<S>(h[s], g[i], y[i]);
        }
        put(static_cast<S *>(a.ry) + off, recur(y, x, xp));
        return;
    }
    const S *__restrict__ b0 = static_cast<const S *>(a.b[0]), *__restrict__ b1 = static_cast<const S *>(a.b[1]),
                         *__restrict__ b2 = static_cast<const S *>(a.b[2]);
    C16 y = C16(S(0)), l0 = y, l1 = y, l2 = y;
    auto add = [&](C16 g, S vh, S v0, S v1, S v2) {
#pragma unroll
        for (int i = 0; i < E; ++i) {
            y[i] = fmas<S>(vh, g[i], y[i]);
            l0[i] = fmas<S>(v0, g[i], l0[i]);
            l1[i] = fmas<S>(v1, g[i], l1[i]);
            l2[i] = fmas<S>(v2, g[i], l2[i]);
        }
    };
    int64_t s = s0;
    for (; s + U <= s1; s += U) {
        int64_t c[U];
        S v[U][4];
        C16 g[U];
#pragma unroll
        for (int t = 0; t < U; ++t) {
            c[t] = col_ind[s + t];
            v[t][0] = h[s + t];
            v[t][1] = b0[s + t];
            v[t][2] = b1[s + t];
            v[t][3] = b2[s + t];
        }
#pragma unroll
        for (int t = 0; t < U; ++t) g[t] = at(a.x, c[t] * W + (int64_t)q * E);
#pragma unroll
        for (int t = 0; t < U; ++t) add(g[t], v[t][0], v[t][1], v[t][2], v[t][3]);
    }
    for (; s < s1; ++s) add(at(a.x, (int64_t)col_ind[s] * W + (int64_t)q * E), h[s], b0[s], b1[s], b2[s]);
    const C16 l[3] = {l0, l1, l2};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        put(static_cast<S *>(a.left) + d * a.left_stride, l[d]);
        if (a.right0) put(static_cast<S *>(a.right0) + d * a.left_stride, l[d]);
    }
    if (a.y) put(a.y, recur(y, a.x, a.xp));
}

// ------------------------------------------------------- moment products
// mu^{ab} = alpha L_a^T R_b of real sequences: M x M outputs over K = rows R,
// each sequence M vectors of K contiguous elements. The chip is filled by cutting
// K: a workgroup of 2 x 2 waves owns a T x T tile (T = 32 A) of one chunk of K,
// and k_kg_sum adds the chunks in order. A lane of an MFMA operand takes four
// K elements in 16-byte accesses, so a row's four lane groups load 64 contiguous
// bytes each time (FP32 is widened in registers: products of two FP32 values
// are exact), and four MFMAs take one element each; no LDS. Rows lie ld
// apart and have at least sixteen elements of memory. An XCD takes a contiguous
// eighth of a product's (chunk, tile) list, so that its L2 holds the rows of few
// chunks, or of a strip of tiles, and no XCD idles when there are fewer chunks than
// XCDs (a chunk to an XCD: M = 1,024 33 TF/s, M = 1,500 and above 8). Bound by the
// MFMAs (M^2 K / 36.6 TF/s) above M of about 100, by reading the sequences below.
// Measured, three products, against rocBLAS, which cuts K only for some sizes:
// M = 64, K = 4,096 0.67 -> 0.014 ms; M = 90, K = 409,600 2.35 -> 0.52; M = 128, K =
// 120,000 58 -> 0.25; M = 200, K = 262,144 1.72 -> 1.68; M = 256 1.80 -> 1.71; M = 512,
// K = 131,072 63 -> 3.6; M = 1,024, K = 73,728 36 -> 8.0; M = 1,500, K = 65,536 32 ->
// 16.1; M = 2,048, K = 32,768 16.7 -> 13.9; M = 4,096, K = 16,384 26.2 -> 26.6, K =
// 2,048 3.3 -> 4.0 (one chunk's parts are written and read again; storing the
// results from here instead moved the accumulators between the register files
// and took 46 in place of 58 TF/s at every size). Vectors a power of two apart took
// 10.6 instead of 9.6 ms (M = 256, K = 1,048,576), a masked tail of scalar loads in
// the loop 9.6 instead of 7.0. Error of the moments against 80-bit sums (rel. 2-norm),
// library / here: K = 36,000, M = 128 5.1e-15 / 2.9e-16; K = 96,000, M = 96
// 8.7e-15 / 2.0e-16: shorter chains of additions.
typedef double d4 __attribute__((ext_vector_type(4)));

template <typename S, int A>
__global__ __launch_bounds__(256, 1) void k_kg_gemm(KgGemm p, int64_t K, int64_t ld, int64_t kc, int M, int nt, int nchunk,
                                                    double *__restrict__ part) {
    constexpr int T = 32 * A;
    constexpr int E = 16 / (int)sizeof(S), P = 4 / E; // elements of an access, accesses a row
    typedef S SE __attribute__((ext_vector_type(E), aligned(sizeof(S))));
    // a product's items in the order (chunk, tile); every XCD takes a contiguous
    // eighth, another one in each product, as the eighths differ by an item
    const int tiles = nt * nt, items = tiles * nchunk, pair = (int)blockIdx.y;
    const int xcd = ((int)blockIdx.x + pair) & 7;
    const int item = (int)((int64_t)items * xcd / 8) + ((int)blockIdx.x >> 3);
    if (item >= (int)((int64_t)items * (xcd + 1) / 8)) return;
    const int chunk = item / tiles, tile = item - chunk * tiles;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, g = lane >> 4;
    // rows of the product are right vectors n, columns left vectors m, so that
    // the parts and mu (column-major) lie alike
    // tiles go down strips of four rows: 32 in flight on an XCD read 12 panels
    const int strip = tile / (4 * nt), high = min(4, nt - 4 * strip), along = tile - strip * 4 * nt;
    const int n0 = (4 * strip + along % high) * T + (wave >> 1) * 16 * A, m0 = (along / high) * T + (wave & 1) * 16 * A;
    const S *__restrict__ rp[A], *__restrict__ lp[A];
#pragma unroll
    for (int r = 0; r < A; ++r) { // vectors past M load the last one and are not stored
        rp[r] = static_cast<const S *>(p.r[pair]) + (int64_t)min(n0 + 16 * r + i, M - 1) * ld;
        lp[r] = static_cast<const S *>(p.l[pair]) + (int64_t)min(m0 + 16 * r + i, M - 1) * ld;
    }
    const int64_t k0 = chunk * kc, k1 = min(K, k0 + kc);
    d4 acc[A][A];
#pragma unroll
    for (int r = 0; r < A; ++r)
#pragma unroll
        for (int c = 0; c < A; ++c) acc[r][c] = d4(0.0);
    // The last block of K starts at klast: a ragged one repeats elements, which
    // are zeroed when it is used (as is what lies past a K below 16).
    const int64_t klast = max(K - 16, (int64_t)0);
    auto load = [&](int64_t k, d4 (&a)[A], d4 (&b)[A]) {
        const int64_t kk = min(k, klast) + E * g;
#pragma unroll
        for (int r = 0; r < A; ++r)
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const SE x = *reinterpret_cast<const SE *>(rp[r] + kk + 4 * E * q);
                const SE y = *reinterpret_cast<const SE *>(lp[r] + kk + 4 * E * q);
#pragma unroll
                for (int j = 0; j < E; ++j) {
                    a[r][E * q + j] = (double)x[j];
                    b[r][E * q + j] = (double)y[j];
                }
            }
    };
    d4 a0[A], b0[A], a1[A], b1[A];
    load(k0, a0, b0);
    for (int64_t k = k0; k < k1; k += 16) {
        load(k + 16 < k1 ? k + 16 : k0, a1, b1);
        __builtin_amdgcn_sched_barrier(0); // in flight during the products
        if (k > klast || K < 16) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t e = min(k, klast) + E * g + 4 * E * (j / E) + j % E;
                if (e < k || e >= K) {
#pragma unroll
                    for (int r = 0; r < A; ++r) a0[r][j] = b0[r][j] = 0.0;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < A; ++r)
#pragma unroll
                for (int c = 0; c < A; ++c)
                    acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[r][j], b0[c][j], acc[r][c], 0, 0, 0);
        // moved, not taken in turn: unrolling by two moved the accumulators
        // between the register files on each turn (7.0 -> 7.5 ms)
#pragma unroll
        for (int r = 0; r < A; ++r) {
            a0[r] = a1[r];
            b0[r] = b1[r];
        }
    }
    const int64_t Mp = (int64_t)nt * T;
    double *__restrict__ out = part + ((int64_t)pair * nchunk + chunk) * Mp * Mp;
#pragma unroll
    for (int r = 0; r < A; ++r)
#pragma unroll
        for (int c = 0; c < A; ++c)
#pragma unroll
            for (int v = 0; v < 4; ++v) out[(int64_t)(n0 + 16 * r + 4 * v + g) * Mp + m0 + 16 * c + i] = acc[r][c][v];
}

// out[n M + m] = alpha sum over the chunks of part[n][m] + beta out[n M + m]:
// 64 elements a workgroup, four threads each taking every fourth chunk.
__global__ __launch_bounds__(256) void k_kg_sum(const double *__restrict__ part, int nchunk, int Mp, int M,
                                                double alpha, double beta, double *__restrict__ out,
                                                int64_t out_stride) {
    __shared__ double sm[4][64];
    const int u = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t e = (int64_t)blockIdx.x * 64 + u, mat = (int64_t)Mp * Mp;
    const int n = (int)(e / M), m = (int)(e - (int64_t)n * M);
    double s = 0.0;
    if (n < M) {
        const double *q = part + (int64_t)blockIdx.y * nchunk * mat + (int64_t)n * Mp + m;
#pragma unroll 8
        for (int c = w; c < nchunk; c += 4) s += q[c * mat];
    }
    sm[w][u] = s;
    __syncthreads();
    if (w == 0 && n < M) {
        double *o = out + blockIdx.y * out_stride + e;
        const double v = alpha * (sm[0][u] + sm[1][u] + sm[2][u] + sm[3][u]);
        *o = beta == 0.0 ? v : v + beta * *o;
    }
}

// *flag = 1 unless the two patterns are the same (their row counts are)
__global__ __launch_bounds__(256) void k_same_pattern(int64_t n, int64_t nnz, const int64_t *__restrict__ rp,
                                                      const int64_t *__restrict__ rq, const int32_t *__restrict__ cp,
                                                      const int32_t *__restrict__ cq, int *__restrict__ flag) {
    bool same = true;
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < nnz + n + 1; t += (int64_t)gridDim.x * 256)
        same = same && (t < nnz ? cp[t] == cq[t] : rp[t - nnz] == rq[t - nnz]);
    if (!same) *flag = 1;
}

// Node weights, complex column-major [m + k M], theta_k = pi (k + 1/2) / M:
// GC = g cos(m theta), GE = g e^{i m theta}, GNE = m GE
__global__ __launch_bounds__(256) void k_kg_weights(int M, const double *__restrict__ g, double2 *__restrict__ W) {
    const int64_t mm = (int64_t)M * M;
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < mm; t += (int64_t)gridDim.x * 256) {
        const int m = (int)(t % M), k = (int)(t / M);
        const double th = 3.14159265358979323846 * (k + 0.5) / M;
        double sn, cs;
        sincos(m * th, &sn, &cs);
        W[t] = double2{g[m] * cs, 0.0};
        W[mm + t] = double2{g[m] * cs, g[m] * sn};
        W[2 * mm + t] = double2{m * g[m] * cs, m * g[m] * sn};
    }
}

__global__ __launch_bounds__(256) void k_kg_widen(const double *__restrict__ in, int cplx, double2 *__restrict__ out,
                                                  int64_t n) {
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < n; t += (int64_t)gridDim.x * 256)
        out[t] = cplx ? double2{in[2 * t], in[2 * t + 1]} : double2{in[t], 0.0};
}

// One wave a node k and pair: the sums over m of (weight column k) x (column k
// of Q_t). out[(pair * 4 + j) * M + k]: Greenwood j = 0: GC Q_0; Bastin
// GC Q_0, conj(GE) Q_1, conj(GNE) Q_1, GC Q_2.
__global__ __launch_bounds__(256) void k_kg_nodes(int M, int bastin, const double2 *__restrict__ W,
                                                  const double2 *__restrict__ Q, double2 *__restrict__ out) {
    const int k = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (k >= M) return;
    const int64_t mm = (int64_t)M * M;
    const double2 *w = W + (int64_t)k * M, *q = Q + (int64_t)blockIdx.y * 3 * mm + (int64_t)k * M;
    double2 *o = out + (int64_t)blockIdx.y * 4 * M + k;
    auto sum = [&](int wsel, bool conj, int t) -> double2 {
        double2 s{0.0, 0.0};
        for (int m = lane; m < M; m += 64) {
            const double2 a = w[wsel * mm + m], b = q[t * mm + m];
            const double ai = conj ? -a.y : a.y;
            s.x += a.x * b.x - ai * b.y;
            s.y += a.x * b.y + ai * b.x;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            s.x += __shfl_xor(s.x, off);
            s.y += __shfl_xor(s.y, off);
        }
        return s;
    };
    const double2 a = sum(0, false, 0);
    if (lane == 0) o[0] = a;
    if (!bastin) return;
    const double2 b = sum(1, true, 1), c = sum(2, true, 1), d = sum(0, false, 2);
    if (lane == 0) {
        o[M] = b;
        o[2 * M] = c;
        o[3 * M] = d;
    }
}

unsigned grid_for(int64_t n) {
    const int64_t g = (n + 255) / 256;
    return (unsigned)(g < 1 ? 1 : g > 8192 ? 8192 : g);
}

} // namespace

int kg_lanes(VecMode vm, int R) {
    const int64_t bytes = (int64_t)R * (vm.complex_vec ? 2 : 1) * (vm.fp32 ? 4 : 8);
    return bytes % 16 == 0 && bytes <= 16 * 256 ? (int)(bytes / 16) : 0;
}

hipError_t launch_kg_moment(const BsrDev &H, VecMode vm, const KgMoment &a, int right, hipStream_t st) {
    if (H.b != 1 || H.is_complex || a.cpr < 1 || a.cpr > 256) return hipErrorInvalidValue;
    const int rpb = 256 / a.cpr;
    const dim3 grid((unsigned)((H.nbr + rpb - 1) / rpb), right ? 4 : 1);
    if (vm.fp32)
        hipLaunchKernelGGL((k_kg_moment<float>), grid, dim3(256), 0, st, H.nbr, H.ulen, H.row_ptr, H.col_ind, a);
    else
        hipLaunchKernelGGL((k_kg_moment<double>), grid, dim3(256), 0, st, H.nbr, H.ulen, H.row_ptr, H.col_ind, a);
    return hipGetLastError();
}

hipError_t launch_same_pattern(const BsrDev &A, const BsrDev &B, int *flag, hipStream_t st) {
    hipLaunchKernelGGL(k_same_pattern, dim3(grid_for(A.nnzb + A.nbr + 1)), dim3(256), 0, st, A.nbr, A.nnzb, A.row_ptr,
                       B.row_ptr, A.col_ind, B.col_ind, flag);
    return hipGetLastError();
}

// Tile side: the fewest padded outputs, wider on a tie. Chunks of K: at least 64
// elements each, one workgroup a CU of every product while that gives eight or
// more (two where the tiles are narrow). With fewer the last round of workgroups
// counts: the fewest chunks within 5 % of the least time, in K elements, where a
// workgroup takes kc + 24 (its first loads wait), the rounds of workgroups end a
// quarter of one late (one round of 243 on 256 CUs took two), and a workgroup's
// part of the output, written and summed, is a round of 96. Measured, three
// products, K = 65,536: M = 1,100 one chunk 28 TF/s, three 51.
KgGemmPlan kg_gemm_plan(int M, int64_t K, int npairs) {
    KgGemmPlan p;
    int64_t best = 0;
    for (int a = 4; a >= 2; --a) {
        const int64_t side = (M + 32 * a - 1) / (32 * a) * (32 * a);
        if (best == 0 || side < best) {
            best = side;
            p.a = a;
        }
    }
    p.nt = (int)(best / (32 * p.a));
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu < 1)
        ncu = 256;
    const int64_t tiles = (int64_t)p.nt * p.nt, slots = p.a == 4 ? ncu : 2 * ncu, most = (K + 63) / 64;
    int64_t want = std::max<int64_t>(1, std::min<int64_t>(slots / tiles, most));
    if (slots / tiles < 8) {
        auto time = [&](int64_t c) {
            const int64_t wgs = c * tiles * npairs, rounds = (wgs + slots - 1) / slots;
            return ((double)rounds + 0.25) * ((double)K / c + 24.0) + 96.0 * wgs / slots;
        };
        const int64_t top = std::min<int64_t>(8, most);
        double least = time(1);
        for (int64_t c = 2; c <= top; ++c) least = std::min(least, time(c));
        for (want = 1; time(want) > 1.05 * least;) ++want;
    }
    kg_gemm_chunks(p, K, want);
    return p;
}

// K in at most `want` chunks of whole blocks of sixteen
void kg_gemm_chunks(KgGemmPlan &p, int64_t K, int64_t want) {
    p.kc = ((K + want - 1) / want + 15) / 16 * 16;
    p.nchunk = (int)((K + p.kc - 1) / p.kc);
}

hipError_t launch_kg_gemm(const KgGemmPlan &pl, const KgGemm &p, int npairs, bool fp32, int64_t K, int64_t ld, int M,
                          double alpha, double beta, double *part, size_t part_bytes, double *out, int64_t out_stride,
                          hipStream_t st) {
    if (M < 1 || K < 1 || npairs < 1 || npairs > 6 || part_bytes < kg_gemm_bytes(pl, npairs)) return hipErrorInvalidValue;
    const int Mp = pl.nt * 32 * pl.a;
    const dim3 grid((unsigned)((pl.nchunk * pl.nt * pl.nt + 7) / 8 * 8), (unsigned)npairs);
#define RG_KG_CASE(S_, A_)                                                                                          \
    hipLaunchKernelGGL((k_kg_gemm<S_, A_>), grid, dim3(256), 0, st, p, K, ld, pl.kc, M, pl.nt, pl.nchunk, part)
    if (fp32) {
        if (pl.a == 2) RG_KG_CASE(float, 2);
        else if (pl.a == 3) RG_KG_CASE(float, 3);
        else RG_KG_CASE(float, 4);
    } else {
        if (pl.a == 2) RG_KG_CASE(double, 2);
        else if (pl.a == 3) RG_KG_CASE(double, 3);
        else RG_KG_CASE(double, 4);
    }
#undef RG_KG_CASE
    hipError_t he = hipGetLastError();
    if (he != hipSuccess) return he;
    hipLaunchKernelGGL(k_kg_sum, dim3((unsigned)(((int64_t)M * M + 63) / 64), (unsigned)npairs), dim3(256), 0, st, part,
                       pl.nchunk, Mp, M, alpha, beta, out, out_stride);
    return hipGetLastError();
}

hipError_t launch_kg_weights(int M, const double *g, double2 *W, hipStream_t st) {
    hipLaunchKernelGGL(k_kg_weights, dim3(grid_for((int64_t)M * M)), dim3(256), 0, st, M, g, W);
    return hipGetLastError();
}

hipError_t launch_kg_widen(const double *in, bool cplx, double2 *out, int64_t n, hipStream_t st) {
    hipLaunchKernelGGL(k_kg_widen, dim3(grid_for(n)), dim3(256), 0, st, in, cplx ? 1 : 0, out, n);
    return hipGetLastError();
}

hipError_t launch_kg_nodes(int M, bool bastin, int npairs, const double2 *W, const double2 *Q, double2 *out,
                           hipStream_t st) {
    hipLaunchKernelGGL(k_kg_nodes, dim3((unsigned)((M + 3) / 4), (unsigned)npairs), dim3(256), 0, st, M, bastin ? 1 : 0,
                       W, Q, out);
    return hipGetLastError();
}

} // namespace rg
