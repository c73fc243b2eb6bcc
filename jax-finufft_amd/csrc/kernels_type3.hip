// Type-3 kernels: extents of the point sets, pre-phasing of the strengths,
// per-target deconvolution factors and post-phasing.  Replaces the type-3
// stages of cuFINUFFT's setpts/execute (called at lib/kernels.cc.cu:66-75;
// source absent from the reference).  The method is the published FINUFFT
// type-3 scheme: with source centre C and target centre D per dimension,
//   f_k = e^{i iflag s_k.C} / prod_d psi_hat(h_d g_d (s_dk - D_d))
//         * sum_l b_l e^{i iflag h g (s_k - D) . l},
//   b   = spread of c_j e^{i iflag D.(x_j - C)} at x'_j = (x_j - C) / g.
#include <cfloat>

#include "jfa_device.hpp"

namespace jfa {
namespace {

struct V3 {
    double v[3];
};

constexpr int kMinmaxBlocks = 1024;

template <typename T>
__global__ void __launch_bounds__(256) minmax_partial_kernel(int64_t n, const T *__restrict__ a,
                                                             double *part) {
    __shared__ double smin[256], smax[256];
    double mn = DBL_MAX, mx = -DBL_MAX;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * 256) {
        double v = (double)a[i];
        mn = v < mn ? v : mn;
        mx = v > mx ? v : mx;
    }
    smin[threadIdx.x] = mn;
    smax[threadIdx.x] = mx;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
            smin[threadIdx.x] = fmin(smin[threadIdx.x], smin[threadIdx.x + off]);
            smax[threadIdx.x] = fmax(smax[threadIdx.x], smax[threadIdx.x + off]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = smin[0];
        part[2 * blockIdx.x + 1] = smax[0];
    }
}

__global__ void __launch_bounds__(256) minmax_final_kernel(int nparts, const double *part,
                                                           double *out) {
    __shared__ double smin[256], smax[256];
    double mn = DBL_MAX, mx = -DBL_MAX;
    for (int i = threadIdx.x; i < nparts; i += 256) {
        mn = fmin(mn, part[2 * i]);
        mx = fmax(mx, part[2 * i + 1]);
    }
    smin[threadIdx.x] = mn;
    smax[threadIdx.x] = mx;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
            smin[threadIdx.x] = fmin(smin[threadIdx.x], smin[threadIdx.x + off]);
            smax[threadIdx.x] = fmax(smax[threadIdx.x], smax[threadIdx.x + off]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = smin[0];
        out[1] = smax[0];
    }
}

template <typename T, int DIM>
__global__ void __launch_bounds__(256)
    t3_prephase_kernel(int64_t M, int ntr, const T *__restrict__ x, const T *__restrict__ y,
                       const T *__restrict__ z, V3 C, V3 D, int iflag, const T *__restrict__ c,
                       T *__restrict__ cp) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= M) return;
    double ph = D.v[0] * ((double)x[j] - C.v[0]);
    if constexpr (DIM > 1) ph += D.v[1] * ((double)y[j] - C.v[1]);
    if constexpr (DIM > 2) ph += D.v[2] * ((double)z[j] - C.v[2]);
    double sn, cs;
    sincos((double)iflag * ph, &sn, &cs);
    for (int t = 0; t < ntr; ++t) {
        const int64_t q = (int64_t)t * M + j;
        const double a = (double)c[2 * q], b = (double)c[2 * q + 1];
        cp[2 * q] = (T)(a * cs - b * sn);
        cp[2 * q + 1] = (T)(a * sn + b * cs);
    }
}

template <typename T, int DIM>
__global__ void __launch_bounds__(256)
    t3_deconv_kernel(int64_t N, const T *__restrict__ s, const T *__restrict__ t,
                     const T *__restrict__ u, V3 D, V3 hg, int ns, int nq,
                     const double *__restrict__ quad, T *__restrict__ dec) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= N) return;
    const T *ss[3] = {s, t, u};
    double prod = 1.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const double w = hg.v[d] * ((double)ss[d][k] - D.v[d]);
        const double a = 0.5 * w * ns;
        double acc = 0.0;
        for (int q = 0; q < nq; ++q) acc += quad[q] * cos(a * quad[nq + q]);
        prod *= ns * acc;
    }
    dec[k] = (T)(1.0 / prod);
}

// The same in fp32, from the Chebyshev series of psi_hat / ns over |w| <= 1 / inv_range:
// two fp64 operations per term and axis instead of a cosine per node, so that the
// factors cost little more than reading the targets.  ns = 8, three axes, 2^20
// targets: 56 cosines an axis 352 us, 28 terms 16 us.  (An fp64 plan keeps the
// quadrature: the series' last digits are no better, see kernel_fourier_series.)
template <int DIM>
__global__ void __launch_bounds__(256)
    t3_deconv_series_kernel(int64_t N, const float *__restrict__ s, const float *__restrict__ t,
                            const float *__restrict__ u, V3 D, V3 hg, int ns, int nt,
                            double inv_range, const double *__restrict__ coef,
                            float *__restrict__ dec) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= N) return;
    const float *ss[3] = {s, t, u};
    double v2[DIM], b1[DIM], b2[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const double r = hg.v[d] * ((double)ss[d][k] - D.v[d]) * inv_range;
        v2[d] = 4.0 * r * r - 2.0;  // 2 v
        b1[d] = b2[d] = 0.0;
    }
    for (int j = nt - 1; j > 0; --j)
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const double b = fma(v2[d], b1[d], coef[j] - b2[d]);
            b2[d] = b1[d];
            b1[d] = b;
        }
    double prod = 1.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) prod *= ns * fma(0.5 * v2[d], b1[d], coef[0] - b2[d]);
    dec[k] = (float)(1.0 / prod);
}

template <typename T, int DIM>
__global__ void __launch_bounds__(256)
    t3_postphase_kernel(int64_t N, int ntr, const T *__restrict__ s, const T *__restrict__ t,
                        const T *__restrict__ u, V3 C, int iflag, const T *__restrict__ dec,
                        T *__restrict__ f) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= N) return;
    double ph = (double)s[k] * C.v[0];
    if constexpr (DIM > 1) ph += (double)t[k] * C.v[1];
    if constexpr (DIM > 2) ph += (double)u[k] * C.v[2];
    double sn, cs;
    sincos((double)iflag * ph, &sn, &cs);
    const double sc = (double)dec[k];
    cs *= sc;
    sn *= sc;
    for (int tr = 0; tr < ntr; ++tr) {
        const int64_t q = (int64_t)tr * N + k;
        const double a = (double)f[2 * q], b = (double)f[2 * q + 1];
        f[2 * q] = (T)(a * cs - b * sn);
        f[2 * q + 1] = (T)(a * sn + b * cs);
    }
}

// Target boxes (type 3 over a partition of the targets): box of target k
// along each axis, b_d = floor((s_dk - lo_d) / width_d) clamped to [0, k_d).
template <typename T, int DIM>
__device__ __forceinline__ int box_of(const T *const *ss, int64_t k, const BoxGrid &bg) {
    int b = 0;
#pragma unroll
    for (int d = DIM - 1; d >= 0; --d) {
        int bd = bg.width[d] > 0 ? (int)floor(((double)ss[d][k] - bg.lo[d]) / bg.width[d]) : 0;
        bd = bd < 0 ? 0 : (bd >= bg.k[d] ? bg.k[d] - 1 : bd);
        b = b * bg.k[d] + bd;
    }
    return b;
}

template <typename T, int DIM>
__global__ void __launch_bounds__(256)
    t3_box_count_kernel(int64_t N, const T *__restrict__ s, const T *__restrict__ t,
                        const T *__restrict__ u, BoxGrid bg, int *__restrict__ count) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= N) return;
    const T *ss[3] = {s, t, u};
    atomicAdd(&count[box_of<T, DIM>(ss, k, bg)], 1);
}

// start[b] = sum of count[< b] (nbox + 1 entries), one workgroup
__global__ void __launch_bounds__(1024)
    t3_box_scan_kernel(int nbox, const int *__restrict__ count, int64_t *__restrict__ start) {
    __shared__ int64_t sa[1024];
    const int tid = threadIdx.x;
    const int per = (nbox + 1023) / 1024;
    const int lo = min(tid * per, nbox), hi = min(lo + per, nbox);
    int64_t a = 0;
    for (int b = lo; b < hi; ++b) a += count[b];
    sa[tid] = a;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int64_t v = tid >= off ? sa[tid - off] : 0;
        __syncthreads();
        sa[tid] += v;
        __syncthreads();
    }
    int64_t e = sa[tid] - a;
    for (int b = lo; b < hi; ++b) {
        start[b] = e;
        e += count[b];
    }
    if (tid == 1023) start[nbox] = sa[1023];
}

// Targets in box order: perm[q] = original index and the coordinates at
// q, for q in [start[b], start[b + 1]) the targets of box b.  The order
// within a box is that of the atomic slot claims; no result depends on it
// (every target is interpolated on its own).
__global__ void __launch_bounds__(256)
    t3_box_next_kernel(int nbox, const int64_t *__restrict__ start, int *__restrict__ next) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b < nbox) next[b] = (int)start[b];
}

template <typename T, int DIM>
__global__ void __launch_bounds__(256)
    t3_box_place_kernel(int64_t N, const T *__restrict__ s, const T *__restrict__ t,
                        const T *__restrict__ u, BoxGrid bg, int *__restrict__ next,
                        int *__restrict__ perm, T *__restrict__ sorted) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= N) return;
    const T *ss[3] = {s, t, u};
    const int q = atomicAdd(&next[box_of<T, DIM>(ss, k, bg)], 1);
    perm[q] = (int)k;
#pragma unroll
    for (int d = 0; d < DIM; ++d) sorted[(int64_t)d * N + q] = ss[d][k];
}

// f[t][perm[q]] = out[t][q] for the box-ordered outputs of every box (box b's
// transforms stored as [t][N_b] at out + 2 nb start[b])
template <typename T>
__global__ void __launch_bounds__(256)
    t3_unsort_kernel(int64_t N, int nb, int nbox, const int64_t *__restrict__ start,
                     const int *__restrict__ perm, const T *__restrict__ out, T *__restrict__ f) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= N) return;
    int lo = 0, hi = nbox;  // the box b with start[b] <= q < start[b + 1]
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (start[mid] <= q) lo = mid;
        else hi = mid;
    }
    const int64_t s0 = start[lo], nbx = start[lo + 1] - s0;
    const int64_t k = perm[q];
    for (int t = 0; t < nb; ++t) {
        const int64_t src = (int64_t)nb * s0 + (int64_t)t * nbx + (q - s0);
        f[2 * ((int64_t)t * N + k)] = out[2 * src];
        f[2 * ((int64_t)t * N + k) + 1] = out[2 * src + 1];
    }
}

V3 v3(const double *a, int dim) {
    V3 r{{0, 0, 0}};
    for (int d = 0; d < dim; ++d) r.v[d] = a[d];
    return r;
}

}  // namespace

template <typename T>
int launch_minmax(int64_t n, const T *a, double *out2, hipStream_t s) {
    // out2 points at [min, max]; the partials live right after it
    return launch_minmax_to<T>(n, a, out2, out2 + 2, s);
}

template <typename T>
int launch_minmax_to(int64_t n, const T *a, double *out2, double *part, hipStream_t s) {
    int64_t nb = (n + 255) / 256;
    int blocks = (int)(nb < kMinmaxBlocks ? (nb > 0 ? nb : 1) : kMinmaxBlocks);
    minmax_partial_kernel<T><<<blocks, 256, 0, s>>>(n, a, part);
    minmax_final_kernel<<<1, 256, 0, s>>>(blocks, part, out2);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int launch_t3_prephase(int dim, int64_t M, int ntr, const T *x, const T *y, const T *z,
                       const double *C, const double *D, int iflag, const T *c, T *cp,
                       hipStream_t stream) {
    if (M == 0 || ntr == 0) return JFA_OK;
    unsigned blocks = (unsigned)((M + 255) / 256);
    JFA_DISPATCH_DIM(dim, t3_prephase_kernel<T, DIM_><<<blocks, 256, 0, stream>>>(
                              M, ntr, x, y, z, v3(C, dim), v3(D, dim), iflag, c, cp));
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int launch_t3_deconv_factors(int dim, int64_t N, const T *s, const T *t, const T *u,
                             const double *D, const double *hg, int ns, double range,
                             const double *table, T *dec, hipStream_t stream) {
    if (N == 0) return JFA_OK;
    unsigned blocks = (unsigned)((N + 255) / 256);
    if constexpr (sizeof(T) == 4) {
        JFA_DISPATCH_DIM(dim, t3_deconv_series_kernel<DIM_><<<blocks, 256, 0, stream>>>(
                                  N, s, t, u, v3(D, dim), v3(hg, dim), ns, ns + 20, 1.0 / range,
                                  table, dec));
    } else {
        JFA_DISPATCH_DIM(dim, t3_deconv_kernel<T, DIM_><<<blocks, 256, 0, stream>>>(
                                  N, s, t, u, v3(D, dim), v3(hg, dim), ns, 2 * ns + 40, table,
                                  dec));
    }
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int launch_t3_postphase(int dim, int64_t N, int ntr, const T *s, const T *t, const T *u,
                        const double *C, int iflag, const T *dec, T *f, hipStream_t stream) {
    if (N == 0 || ntr == 0) return JFA_OK;
    unsigned blocks = (unsigned)((N + 255) / 256);
    JFA_DISPATCH_DIM(dim, t3_postphase_kernel<T, DIM_><<<blocks, 256, 0, stream>>>(
                              N, ntr, s, t, u, v3(C, dim), iflag, dec, f));
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int launch_t3_box_sort(int dim, int64_t N, const T *s, const T *t, const T *u,
                       const BoxGrid &bg, int nbox, int *count, int64_t *start, int *perm,
                       T *sorted, hipStream_t stream) {
    if (N == 0) return JFA_OK;
    if (int rc = launch_fill_zero(count, sizeof(int) * 2 * nbox, stream)) return rc;
    const unsigned blocks = (unsigned)((N + 255) / 256);
    JFA_DISPATCH_DIM(dim, t3_box_count_kernel<T, DIM_><<<blocks, 256, 0, stream>>>(
                              N, s, t, u, bg, count));
    t3_box_scan_kernel<<<1, 1024, 0, stream>>>(nbox, count, start);
    // next[b] = start[b], as ints (N < 2^31)
    int *next = count + nbox;
    t3_box_next_kernel<<<(unsigned)((nbox + 255) / 256), 256, 0, stream>>>(nbox, start, next);
    JFA_DISPATCH_DIM(dim, t3_box_place_kernel<T, DIM_><<<blocks, 256, 0, stream>>>(
                              N, s, t, u, bg, next, perm, sorted));
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int launch_t3_unsort(int64_t N, int nb, int nbox, const int64_t *start, const int *perm,
                     const T *out, T *f, hipStream_t stream) {
    if (N == 0 || nb == 0) return JFA_OK;
    t3_unsort_kernel<T><<<(unsigned)((N + 255) / 256), 256, 0, stream>>>(N, nb, nbox, start,
                                                                         perm, out, f);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

#define JFA_INST(T)                                                                            \
    template int launch_t3_box_sort<T>(int, int64_t, const T *, const T *, const T *,         \
                                       const BoxGrid &, int, int *, int64_t *, int *, T *,    \
                                       hipStream_t);                                           \
    template int launch_t3_unsort<T>(int64_t, int, int, const int64_t *, const int *,        \
                                     const T *, T *, hipStream_t);                             \
    template int launch_minmax_to<T>(int64_t, const T *, double *, double *, hipStream_t);    \
    template int launch_minmax<T>(int64_t, const T *, double *, hipStream_t);                  \
    template int launch_t3_prephase<T>(int, int64_t, int, const T *, const T *, const T *,     \
                                       const double *, const double *, int, const T *, T *,   \
                                       hipStream_t);                                           \
    template int launch_t3_deconv_factors<T>(int, int64_t, const T *, const T *, const T *,    \
                                             const double *, const double *, int, double,        \
                                             const double *, T *, hipStream_t);                \
    template int launch_t3_postphase<T>(int, int64_t, int, const T *, const T *, const T *,    \
                                        const double *, int, const T *, T *, hipStream_t);
JFA_INST(float)
JFA_INST(double)
#undef JFA_INST

}  // namespace jfa
