// Device helpers shared by the setpts / spread / interp kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "jfa_internal.hpp"

namespace jfa {

// Fold a coordinate to the periodic fine grid and locate its tap window.
// u = (x - shift) * scale mod nf in [0, nf); the ns taps are l0 .. l0+ns-1 with
// l0 = ceil(u - ns/2); frac = l0 - (u - ns/2) in [0, 1).  Everything is done in
// double so that the integer first tap is the same wherever it is computed
// (bin counting and the sorted scatter both call this one function).
struct Folded {
    int l0w;     // first tap wrapped into [0, nf)
    double t;    // Horner variable 2*frac - 1 in [-1, 1)
};

__device__ __forceinline__ Folded fold_point(double x, int64_t nf, double scale, double shift,
                                             int ns) {
    const double dnf = (double)nf;
    double u = (x - shift) * scale;
    // On [-nf, 0) and [0, nf) the reduction u - nf floor(u / nf) and the two
    // corrections after it give u + nf and u, up to the sign of a zero and a
    // result of nf in place of 0, which yield the same taps and t; so points
    // of [-pi, pi) skip its division.
    if (u < 0.0 && u >= -dnf)
        u += dnf;
    else if (!(u >= 0.0 && u < dnf))
        u -= dnf * floor(u / dnf);
    if (u >= dnf) u -= dnf;
    if (u < 0.0) u += dnf;
    const double v = u - 0.5 * ns;
    const double l0 = ceil(v);
    Folded f;
    int li = (int)l0;
    f.l0w = li < 0 ? li + (int)nf : li;
    f.t = 2.0 * (l0 - v) - 1.0;
    return f;
}

// ns kernel values for one point along one dimension.  Tap i sits at offset
// r_i = -ns/2 + i + (t+1)/2 cells from the point; its weight is
// phi(2 r_i / ns).  HORNER: evaluate the plan-time fitted polynomials
// (coef[p*NS + i] multiplies t^p); otherwise exp/sqrt directly.
//
// phi is even and r_{ns-1-i}(-t) = -r_i(t), so tap ns-1-i at t is tap i's
// polynomial P_i at -t.  Writing P_i(t) = E(t^2) + t O(t^2) (its even and odd
// coefficients), both taps come from one Horner pass over E and O in t^2:
// about NC + 2 FMAs per pair instead of 2 (NC - 1).
template <typename T, int NS, bool HORNER, typename Coef>
__device__ __forceinline__ void eval_kernel(Coef coef, T beta, T t, T *ker) {
    if constexpr (HORNER) {
        constexpr int NC = horner_nc(NS);
        constexpr int NE = (NC + 1) / 2, NO = NC / 2;  // even / odd coefficient counts
        const T s = t * t;
#pragma unroll
        for (int i = 0; i < (NS + 1) / 2; ++i) {
            T e = coef[2 * (NE - 1) * NS + i];
#pragma unroll
            for (int k = NE - 2; k >= 0; --k) e = fma(e, s, coef[2 * k * NS + i]);
            T o = coef[(2 * NO - 1) * NS + i];
#pragma unroll
            for (int k = NO - 2; k >= 0; --k) o = fma(o, s, coef[(2 * k + 1) * NS + i]);
            ker[i] = fma(t, o, e);
            if (NS - 1 - i != i) ker[NS - 1 - i] = fma(-t, o, e);
        }
    } else {
        const T inv = T(2) / T(NS);
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            T z = (T(-0.5 * NS) + T(i) + T(0.5) * (t + T(1))) * inv;
            T a = T(1) - z * z;
            ker[i] = a < T(0) ? T(0) : exp(beta * (sqrt(a) - T(1)));
        }
    }
}

__device__ __forceinline__ void atomic_add_global(float *p, float v) { unsafeAtomicAdd(p, v); }
__device__ __forceinline__ void atomic_add_global(double *p, double v) { unsafeAtomicAdd(p, v); }

}  // namespace jfa

// Expand BODY for the runtime width `ns` as a compile-time constant NS_.
#define JFA_DISPATCH_NS(ns, ...)                                   \
    switch (ns) {                                                  \
        case 2: { constexpr int NS_ = 2; __VA_ARGS__; } break;     \
        case 3: { constexpr int NS_ = 3; __VA_ARGS__; } break;     \
        case 4: { constexpr int NS_ = 4; __VA_ARGS__; } break;     \
        case 5: { constexpr int NS_ = 5; __VA_ARGS__; } break;     \
        case 6: { constexpr int NS_ = 6; __VA_ARGS__; } break;     \
        case 7: { constexpr int NS_ = 7; __VA_ARGS__; } break;     \
        case 8: { constexpr int NS_ = 8; __VA_ARGS__; } break;     \
        case 9: { constexpr int NS_ = 9; __VA_ARGS__; } break;     \
        case 10: { constexpr int NS_ = 10; __VA_ARGS__; } break;   \
        case 11: { constexpr int NS_ = 11; __VA_ARGS__; } break;   \
        case 12: { constexpr int NS_ = 12; __VA_ARGS__; } break;   \
        case 13: { constexpr int NS_ = 13; __VA_ARGS__; } break;   \
        case 14: { constexpr int NS_ = 14; __VA_ARGS__; } break;   \
        case 15: { constexpr int NS_ = 15; __VA_ARGS__; } break;   \
        case 16: { constexpr int NS_ = 16; __VA_ARGS__; } break;   \
        default: ::jfa::set_error("unsupported kernel width %d", ns); return JFA_ERR_BAD_ARG; \
    }

#define JFA_DISPATCH_DIM(dim, ...)                                 \
    switch (dim) {                                                 \
        case 1: { constexpr int DIM_ = 1; __VA_ARGS__; } break;    \
        case 2: { constexpr int DIM_ = 2; __VA_ARGS__; } break;    \
        case 3: { constexpr int DIM_ = 3; __VA_ARGS__; } break;    \
        default: ::jfa::set_error("unsupported dimension %d", dim); return JFA_ERR_BAD_ARG; \
    }
