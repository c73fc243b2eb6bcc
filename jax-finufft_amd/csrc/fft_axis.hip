// Pruned FFT passes between the fine grid and the modes, one kernel per axis.
// Replaces the full nf0 x nf1 (x nf2) FFT cuFINUFFT runs inside execute
// (called at lib/kernels.cc.cu:75; source absent from the reference).
//
// Of the nf_d fine-grid frequencies along an axis only the n_d mode
// frequencies k in [-n_d/2, (n_d-1)/2] are kept.  Type 1 transforms x, then y
// (then z), each pass writing its mode frequencies only; type 2 runs z, y, x,
// each pass reading its modes and taking the other inputs as zero.  Arrays
// keep x fastest throughout, and a mode axis is stored in the caller's mode
// order, so that no pass transposes:
//
//   2D   modes [n1][n0] <-> W [nf1][n0] <-> grid [nf1][nf0]
//   3D   modes [n2][n1][n0] <-> V [nf2][n1][n0] <-> W [nf2][nf1][n0] <-> grid
//
// The 1/psi_hat factors (deconvolution / amplification) ride on the pass that
// touches the modes.  A pass moves its input once and its output once: what
// bounds them is HBM on grids beyond the caches (x pass of 512^3 from 256 modes:
// 1.6 GB in 0.35 ms) and latency below.  The rocFFT 1D passes with separate
// transposes and scaling kernels they replace move each intermediate two or
// three times: modes -> 512^3 grid, 256^3 modes, 1.36 -> 0.73 ms; 360^3 modes ->
// the kept 720 x 375 x 375 cells of a type-3 inner grid, 1.85 -> 1.13 ms; 2048^2
// grid -> 1024^2 modes, 46 -> 37 us (fp32).  Those stay for plans with an axis these
// passes do not run (axis_fft): beyond 4096 cells, or of a length whose smallest radix
// leaves more threads for 32 bytes of columns than a workgroup has (of the even lengths
// in fp32 1458, 1944, 2000, 2430, 2500, 2592, 2916, 3000, 3200, 3240, 3456, 3750, 3888,
// 4000, 4050; in fp64 2700, 3000, 3200, 3240, 3456, 3600, 3750, 3840, 3888, 4000, 4050).
//
// One workgroup transforms a tile in LDS: one (or a few) contiguous rows along
// x, or TC neighbouring columns along y / z (TC complex values are 128 bytes
// where LDS and the thread limit allow, so a wave reads whole cache lines).
// Stockham autosort, radices up to 16, one butterfly per thread and stage: the
// first stage reads global memory and the last writes it, so an FFT of three
// stages crosses LDS twice; each stage reads all its inputs into registers
// before the barrier that lets it overwrite them.
#include <algorithm>
#include <type_traits>

#include "jfa_device.hpp"
#include "plan_state.hpp"

namespace jfa {
namespace {

template <typename T>
struct alignas(2 * sizeof(T)) Cx {
    T x, y;
};

// ---------------------------------------------------------------- constants
// cos / sin of 2 pi k / n at compile time: the angle is reduced to the first
// octant exactly (in integers), where the Taylor series converges to rounding.
constexpr double taylor_cos(double a) {
    double s = 1, t = 1;
    for (int i = 1; i < 12; ++i) {
        t *= -a * a / ((2 * i - 1) * (2 * i));
        s += t;
    }
    return s;
}
constexpr double taylor_sin(double a) {
    double s = a, t = a;
    for (int i = 1; i < 12; ++i) {
        t *= -a * a / ((2 * i) * (2 * i + 1));
        s += t;
    }
    return s;
}
constexpr double kTwoPi = 6.283185307179586476925286766559;
constexpr double cos2pi(int k, int n) {
    k %= n;
    if (2 * k > n) k = n - k;                              // cos(2 pi - a) = cos a
    if (4 * k > n) return -cos2pi(n - 2 * k, 2 * n);       // cos(pi - a) = -cos a
    if (8 * k > n) return taylor_sin(kTwoPi * (n - 4 * k) / (4.0 * n));
    return taylor_cos(kTwoPi * k / n);
}
constexpr double sin2pi(int k, int n) {
    k %= n;
    if (2 * k > n) return -sin2pi(n - k, n);
    if (4 * k > n) return sin2pi(n - 2 * k, 2 * n);        // sin(pi - a) = sin a
    if (8 * k > n) return taylor_cos(kTwoPi * (n - 4 * k) / (4.0 * n));
    return taylor_sin(kTwoPi * k / n);
}

// v * exp(-2 pi i K / N)
template <typename T, int K, int N>
__device__ __forceinline__ Cx<T> rot(Cx<T> v) {
    constexpr int k = K % N;
    if constexpr (k == 0) return v;
    else if constexpr (4 * k == N) return {v.y, -v.x};
    else if constexpr (2 * k == N) return {-v.x, -v.y};
    else if constexpr (4 * k == 3 * N) return {-v.y, v.x};
    else if constexpr (8 * k == N) {
        constexpr T h = (T)cos2pi(1, 8);
        return {h * (v.x + v.y), h * (v.y - v.x)};
    } else if constexpr (8 * k == 3 * N) {
        constexpr T h = (T)cos2pi(1, 8);
        return {h * (v.y - v.x), -h * (v.x + v.y)};
    } else {
        constexpr T c = (T)cos2pi(k, N), s = (T)sin2pi(k, N);
        return {v.x * c + v.y * s, v.y * c - v.x * s};
    }
}

template <typename T>
__device__ __forceinline__ Cx<T> add(Cx<T> a, Cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> sub(Cx<T> a, Cx<T> b) { return {a.x - b.x, a.y - b.y}; }

// In-place DFT v[k] = sum_n v[n] exp(-2 pi i n k / N) in registers: 2, 3, 4
// and 5 directly, the others split N = A B.
constexpr int split_of(int n) {
    return n == 6 ? 2 : n == 8 ? 4 : n == 9 ? 3 : n == 10 ? 5 : n == 12 ? 4 : n == 15 ? 5
           : n == 16 ? 4 : 0;
}
template <typename T, int A, int B, int N2, int K1>
__device__ __forceinline__ void twist(Cx<T> (&u)[A]) {
    if constexpr (K1 < A) {
        u[K1] = rot<T, N2 * K1, A * B>(u[K1]);
        twist<T, A, B, N2, K1 + 1>(u);
    }
}
template <typename T, int N>
__device__ __forceinline__ void dft(Cx<T> (&v)[N]);
template <typename T, int A, int B, int N2>
__device__ __forceinline__ void dft_inner(Cx<T> (&v)[A * B], Cx<T> (&w)[B][A]) {
    if constexpr (N2 < B) {
        Cx<T> u[A];
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) u[n1] = v[B * n1 + N2];
        dft<T, A>(u);
        twist<T, A, B, N2, 1>(u);
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) w[N2][k1] = u[k1];
        dft_inner<T, A, B, N2 + 1>(v, w);
    }
}
template <typename T, int N>
__device__ __forceinline__ void dft(Cx<T> (&v)[N]) {
    if constexpr (N == 2) {
        const Cx<T> a = v[0], b = v[1];
        v[0] = add(a, b);
        v[1] = sub(a, b);
    } else if constexpr (N == 3) {
        constexpr T h = (T)sin2pi(1, 3);
        const Cx<T> t = add(v[1], v[2]), d = sub(v[1], v[2]);
        const Cx<T> m{fma(T(-0.5), t.x, v[0].x), fma(T(-0.5), t.y, v[0].y)};
        v[0] = add(v[0], t);
        v[1] = {fma(h, d.y, m.x), fma(-h, d.x, m.y)};
        v[2] = {fma(-h, d.y, m.x), fma(h, d.x, m.y)};
    } else if constexpr (N == 4) {
        const Cx<T> a = add(v[0], v[2]), b = sub(v[0], v[2]);
        const Cx<T> c = add(v[1], v[3]), d = sub(v[1], v[3]);
        v[0] = add(a, c);
        v[2] = sub(a, c);
        v[1] = {b.x + d.y, b.y - d.x};
        v[3] = {b.x - d.y, b.y + d.x};
    } else if constexpr (N == 5) {
        constexpr T c1 = (T)cos2pi(1, 5), c2 = (T)cos2pi(2, 5);
        constexpr T s1 = (T)sin2pi(1, 5), s2 = (T)sin2pi(2, 5);
        const Cx<T> a1 = add(v[1], v[4]), b1 = sub(v[1], v[4]);
        const Cx<T> a2 = add(v[2], v[3]), b2 = sub(v[2], v[3]);
        const Cx<T> m1{fma(c2, a2.x, fma(c1, a1.x, v[0].x)), fma(c2, a2.y, fma(c1, a1.y, v[0].y))};
        const Cx<T> m2{fma(c1, a2.x, fma(c2, a1.x, v[0].x)), fma(c1, a2.y, fma(c2, a1.y, v[0].y))};
        const Cx<T> n1{fma(s2, b2.x, s1 * b1.x), fma(s2, b2.y, s1 * b1.y)};
        const Cx<T> n2{fma(-s1, b2.x, s2 * b1.x), fma(-s1, b2.y, s2 * b1.y)};
        v[0] = add(v[0], add(a1, a2));
        v[1] = {m1.x + n1.y, m1.y - n1.x};
        v[4] = {m1.x - n1.y, m1.y + n1.x};
        v[2] = {m2.x + n2.y, m2.y - n2.x};
        v[3] = {m2.x - n2.y, m2.y + n2.x};
    } else {
        // n = B n1 + n2, k = k1 + A k2
        constexpr int A = split_of(N), B = N / A;
        Cx<T> w[B][A];
        dft_inner<T, A, B, 0>(v, w);
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
            Cx<T> u[B];
#pragma unroll
            for (int n2 = 0; n2 < B; ++n2) u[n2] = w[n2][k1];
            dft<T, B>(u);
#pragma unroll
            for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = u[k2];
        }
    }
}

// ------------------------------------------------------------------- stages

// One Stockham stage: butterfly j < L / R of a span-Ns stage reads elements
// j + k L / R, twiddles input k by exp(-2 pi i k (j mod Ns) / (Ns R)) and
// writes elements (j / Ns) Ns R + (j mod Ns) + k Ns.  The first stage (Ns = 1)
// reads through ld, the last (Ns R = L) writes through st; at(e) is element
// e's place in LDS.  tw is the stage's own table, [k - 1][j mod Ns]:
// neighbouring threads read neighbouring entries.
template <typename T, int R, bool FIRST, bool LAST, typename At, typename Ld, typename St>
__device__ __forceinline__ void fft_stage(int L, int Ns, const Cx<T> *__restrict__ tw, Cx<T> *lds,
                                          int j, bool live, At at, Ld ld, St st) {
    const int m = L / R;
    const bool act = live && j < m;
    Cx<T> v[R];
    int o = j * R;
    if (act) {
        if constexpr (FIRST) {
#pragma unroll
            for (int k = 0; k < R; ++k) v[k] = ld(j + k * m);
        } else {
#pragma unroll
            for (int k = 0; k < R; ++k) v[k] = lds[at(j + k * m)];
            int q = j;
            if constexpr (!LAST) {
                q = j % Ns;
                o = (j - q) * R + q;
            }
#pragma unroll
            for (int k = 1; k < R; ++k) {
                const Cx<T> w = tw[(k - 1) * Ns + q];  // (cos, sin)
                v[k] = {v[k].x * w.x + v[k].y * w.y, v[k].y * w.x - v[k].x * w.y};
            }
        }
        dft<T, R>(v);
        if constexpr (LAST) {
#pragma unroll
            for (int k = 0; k < R; ++k) st(j + k * m, v[k]);
        }
    }
    if constexpr (!LAST) {
        if constexpr (!FIRST) __syncthreads();  // every input is in registers
        if (act) {
#pragma unroll
            for (int k = 0; k < R; ++k) lds[at(o + k * Ns)] = v[k];
        }
        __syncthreads();
    }
}

// A stage of radix r <= MAXR (MAXR bounds the kernel's registers).
template <typename T, int MAXR, bool FIRST, bool LAST, typename At, typename Ld, typename St>
__device__ __forceinline__ void fft_stage_r(int r, int L, int Ns, const Cx<T> *__restrict__ tw,
                                            Cx<T> *lds, int j, bool live, At at, Ld ld, St st) {
    switch (r) {
#define JFA_STAGE(R)                                                                  \
    case R:                                                                           \
        if constexpr (R <= MAXR)                                                      \
            fft_stage<T, R, FIRST, LAST>(L, Ns, tw, lds, j, live, at, ld, st);        \
        break;
        JFA_STAGE(2)
        JFA_STAGE(3)
        JFA_STAGE(4)
        JFA_STAGE(5)
        JFA_STAGE(6)
        JFA_STAGE(8)
        JFA_STAGE(9)
        JFA_STAGE(10)
        JFA_STAGE(12)
        JFA_STAGE(15)
        JFA_STAGE(16)
#undef JFA_STAGE
    }
}

template <typename T, int MAXR, typename At, typename Ld, typename St>
__device__ __forceinline__ void fft_run(const AxisFft &f, const Cx<T> *__restrict__ tw,
                                        Cx<T> *lds, int j, bool live, At at, Ld ld, St st) {
    const int last = f.count - 1;
    if (last == 0) {
        fft_stage_r<T, MAXR, true, true>(f.r[0], f.L, 1, tw, lds, j, live, at, ld, st);
        return;
    }
    fft_stage_r<T, MAXR, true, false>(f.r[0], f.L, 1, tw, lds, j, live, at, ld, st);
    int Ns = f.r[0];
#pragma unroll 1
    for (int s = 1; s < last; ++s) {
        // opaque to the compiler, which would otherwise compute every radix's
        // addresses before the loop and spill
        int jj = j;
        asm volatile("" : "+v"(jj));
        fft_stage_r<T, MAXR, false, false>(f.r[s], f.L, Ns, tw + f.t[s], lds, jj, live, at, ld, st);
        Ns *= f.r[s];
    }
    fft_stage_r<T, MAXR, false, true>(f.r[last], f.L, Ns, tw + f.t[last], lds, j, live, at, ld, st);
}

// frequency at fine index e of an axis of n modes and length L; false where no
// mode lives there
__device__ __forceinline__ bool mode_at(int e, int n, int L, int &k) {
    k = e < (n + 1) / 2 ? e : e - L;
    return e < (n + 1) / 2 || e >= L - n / 2;
}
// place of frequency k along a mode axis (modeord 0: centred, 1: FFT order)
__device__ __forceinline__ int mode_index(int k, int n, int modeord) {
    return modeord == 0 ? k + n / 2 : (k < 0 ? k + n : k);
}
// frequency of place i along a mode axis
__device__ __forceinline__ int mode_freq(int i, int n, int modeord) {
    if (modeord == 0) return i - n / 2;
    return i < (n + 1) / 2 ? i : i - n;
}

// The transforms below are exp(-i ...); the +i sign swaps real and imaginary
// parts on the way in and out (swap(DFT(swap(x))) is the conjugate kernel).
template <typename T>
__device__ __forceinline__ Cx<T> turned(Cx<T> v, int swap) { return swap ? Cx<T>{v.y, v.x} : v; }

// Place of element e in LDS: one element (or row of TC) of padding per 8 puts
// the strided writes of a radix-8 stage on distinct banks.
__host__ __device__ __forceinline__ int padded(int e) { return e + (e >> 3); }

// x pass.  grid rows [rows][L] and mode rows [rows][n]; TO_GRID: modes ->
// grid (type 2), else grid -> modes.  NR rows per workgroup, P threads each.
template <typename T, int MAXR, bool TO_GRID>
__global__ void __launch_bounds__(1024)
    fft_rows_kernel(AxisFft f, int P, int NR, int64_t rows, int n, int modeord, int swap,
                    const T *__restrict__ tw_, const T *__restrict__ in_, T *__restrict__ out_) {
    extern __shared__ __align__(16) unsigned char fft_smem[];
    const int rr = threadIdx.x / P, j = threadIdx.x - rr * P;
    const int64_t row = (int64_t)blockIdx.x * NR + rr;
    const bool live = rr < NR && row < rows;
    const int L = f.L;
    Cx<T> *lds = reinterpret_cast<Cx<T> *>(fft_smem) + rr * padded(L);
    const Cx<T> *in = reinterpret_cast<const Cx<T> *>(in_) + row * (TO_GRID ? n : L);
    Cx<T> *out = reinterpret_cast<Cx<T> *>(out_) + row * (TO_GRID ? L : n);
    fft_run<T, MAXR>(
        f, reinterpret_cast<const Cx<T> *>(tw_), lds, j, live,
        [](int e) { return padded(e); },
        [&](int e) {
            if constexpr (TO_GRID) {
                int k;
                if (!mode_at(e, n, L, k)) return Cx<T>{T(0), T(0)};
                return turned(in[mode_index(k, n, modeord)], swap);
            } else {
                return turned(in[e], swap);
            }
        },
        [&](int e, Cx<T> v) {
            if constexpr (TO_GRID) {
                out[e] = turned(v, swap);
            } else {
                int k;
                if (mode_at(e, n, L, k)) out[mode_index(k, n, modeord)] = turned(v, swap);
            }
        });
}

// y / z pass over [outer][axis][inner] arrays: the axis holds n modes on the
// mode side and the rows w0 .. w0 + wl - 1 (mod L) on the grid side (all of
// them unless a type-2 plan keeps fewer, GridGeom::wstart).  With dkl, the
// modes are scaled by dk0[k0] dkm[km] dkl[k], (k0, km) the frequencies of the
// column's place i0 + n0 im.
struct ColsShape {
    int64_t inner;      // columns
    int tiles;          // ceil(inner / TC)
    int n, w0, wl;
    int n0, nm;         // modes along x and (3D z pass) y of the columns
    int modeord, swap;
};
template <typename T, int TC, int MAXR, bool TO_GRID>
__global__ void __launch_bounds__(1024)
    fft_cols_kernel(AxisFft f, ColsShape sh, const T *__restrict__ tw_, const T *__restrict__ dk0,
                    const T *__restrict__ dkm, const T *__restrict__ dkl,
                    const T *__restrict__ in_, T *__restrict__ out_) {
    extern __shared__ __align__(16) unsigned char fft_smem[];
    Cx<T> *lds = reinterpret_cast<Cx<T> *>(fft_smem);
    const int c = threadIdx.x & (TC - 1), j = threadIdx.x / TC;
    // workgroup b runs on XCD b mod 8: hand each XCD runs of neighbouring
    // tiles, which share cache lines when TC is less than a line
    unsigned b = blockIdx.x;
    if (b < (gridDim.x & ~63u)) b = (b & ~63u) | ((b & 7) << 3) | ((b >> 3) & 7);
    const unsigned o = b / (unsigned)sh.tiles;
    const int64_t col = (int64_t)(b - o * (unsigned)sh.tiles) * TC + c;
    const bool live = col < sh.inner;
    const int L = f.L, n = sh.n;
    const int64_t mode_base = (int64_t)o * n * sh.inner + col;
    const int64_t grid_base = (int64_t)o * sh.wl * sh.inner + col;
    const Cx<T> *in = reinterpret_cast<const Cx<T> *>(in_) + (TO_GRID ? mode_base : grid_base);
    Cx<T> *out = reinterpret_cast<Cx<T> *>(out_) + (TO_GRID ? grid_base : mode_base);
    T s0 = T(1);
    if (dkl && live) {
        const unsigned cc = (unsigned)col, im = cc / (unsigned)sh.n0;
        s0 = dk0[mode_freq((int)(cc - im * sh.n0), sh.n0, sh.modeord) + sh.n0 / 2];
        if (sh.nm > 1) s0 *= dkm[mode_freq((int)im, sh.nm, sh.modeord) + sh.nm / 2];
    }
    fft_run<T, MAXR>(
        f, reinterpret_cast<const Cx<T> *>(tw_), lds, j, live,
        [&](int e) { return padded(e) * TC + c; },
        [&](int e) {
            if constexpr (TO_GRID) {
                int k;
                if (!mode_at(e, n, L, k)) return Cx<T>{T(0), T(0)};
                Cx<T> v = turned(in[mode_index(k, n, sh.modeord) * sh.inner], sh.swap);
                if (dkl) {
                    const T s = s0 * dkl[k + n / 2];
                    v = {v.x * s, v.y * s};
                }
                return v;
            } else {
                return turned(in[e * sh.inner], sh.swap);
            }
        },
        [&](int e, Cx<T> v) {
            if constexpr (TO_GRID) {
                int r = e - sh.w0;
                if (r < 0) r += L;
                if (r < sh.wl) out[r * sh.inner] = turned(v, sh.swap);
            } else {
                int k;
                if (!mode_at(e, n, L, k)) return;
                if (dkl) {
                    const T s = s0 * dkl[k + n / 2];
                    v = {v.x * s, v.y * s};
                }
                out[mode_index(k, n, sh.modeord) * sh.inner] = turned(v, sh.swap);
            }
        });
}

// tw of stage s at f.t[s]: exp(+2 pi i k q / (Ns R)) for k in [1, R), q < Ns.
template <typename T>
__global__ void __launch_bounds__(256) axis_twiddle_kernel(AxisFft f, T *__restrict__ tw) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= f.ntw) return;
    int s = 1, Ns = f.r[0];
    while (s + 1 < f.count && i >= f.t[s + 1]) Ns *= f.r[s++];
    const int e = i - f.t[s], k = e / Ns + 1, q = e - (k - 1) * Ns;
    double sn, cs;
    sincospi(2.0 * k * q / ((double)Ns * f.r[s]), &sn, &cs);
    tw[2 * i] = (T)cs;
    tw[2 * i + 1] = (T)sn;
}

constexpr int kRadices[] = {16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2};
constexpr int kMaxThreads = 1024;
constexpr size_t kMaxLds = 144 * 1024;
// Most threads of one launch; larger passes (16 transforms on 1024^3 cells) take several.
constexpr int64_t kLaunchThreads = UINT32_MAX;

// The stages of length n: as few as possible, then with the largest smallest
// radix (a stage of radix r uses n / r threads per column).
void search_stages(int n, int max_r, AxisFft &cur, AxisFft &best) {
    if (n == 1) {
        const bool fewer = best.count == 0 || cur.count < best.count;
        if (fewer || (cur.count == best.count && cur.r[cur.count - 1] > best.r[best.count - 1]))
            best = cur;
        return;
    }
    if (cur.count == 8 || (best.count && cur.count >= best.count)) return;
    for (int r : kRadices) {
        if (r > max_r || n % r) continue;
        cur.r[cur.count++] = r;
        search_stages(n / r, r, cur, best);
        --cur.count;
    }
}

template <typename K>
int allow_lds(K kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        JFA_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize,
                                          (int)bytes));
    return JFA_OK;
}

template <typename T, bool TO_GRID>
int launch_rows(const AxisFft &f, const T *tw, int64_t rows, int64_t n, int modeord, int swap,
                const T *in, T *out, hipStream_t s) {
    if (rows == 0) return JFA_OK;
    const int P = f.P;
    const size_t row_bytes = (size_t)padded(f.L) * 2 * sizeof(T);
    // about 256 threads per workgroup
    const int NR = std::max(1, std::min<int>(256 / P, (int)(48 * 1024 / row_bytes)));
    const size_t lds = NR * row_bytes;
    const unsigned threads = (unsigned)((P * NR + 63) / 64 * 64);
    const int64_t most = kLaunchThreads / threads * NR;  // rows of a launch
    auto go = [&](auto kernel) -> int {
        if (int rc = allow_lds(kernel, lds)) return rc;
        for (int64_t r0 = 0; r0 < rows; r0 += most) {
            const int64_t part = std::min(most, rows - r0);
            kernel<<<(unsigned)((part + NR - 1) / NR), threads, lds, s>>>(
                f, P, NR, part, (int)n, modeord, swap, tw, in + 2 * r0 * (TO_GRID ? n : f.L),
                out + 2 * r0 * (TO_GRID ? f.L : n));
            JFA_HIP_CHECK(hipGetLastError());
        }
        return JFA_OK;
    };
    if (f.r[0] <= 8) return go(fft_rows_kernel<T, 8, TO_GRID>);
    if (f.r[0] <= 10) return go(fft_rows_kernel<T, 10, TO_GRID>);
    return go(fft_rows_kernel<T, sizeof(T) == 8 ? 10 : 16, TO_GRID>);
}

// Columns per workgroup: 128 bytes of them when P threads per column and the
// LDS tile (80 KiB, for two workgroups per CU; up to 144 KiB for the longest
// axes) allow, 32 bytes at least; fewer too while the launch has under 512
// workgroups (a 2-byte-per-flop pass needs every CU busy, and such small
// arrays sit in L2, where short segments cost little).
template <typename T>
int cols_per_group(const AxisFft &f, int64_t columns) {
    const int least = 32 / (2 * sizeof(T));
    int tc = 128 / (2 * sizeof(T));
    const size_t col = (size_t)padded(f.L) * 2 * sizeof(T);
    while (tc > least && (tc * f.P > kMaxThreads || tc * col > 80 * 1024)) tc /= 2;
    while (tc > least && columns / tc < 512) tc /= 2;
    return tc;
}

template <typename T, bool TO_GRID>
int launch_cols(const AxisFft &f, const T *tw, int64_t outer, const ColsShape &shape,
                const T *dk0, const T *dkm, const T *dkl, const T *in, T *out, hipStream_t s) {
    ColsShape sh = shape;
    if (outer == 0 || sh.inner == 0) return JFA_OK;
    const int tc = cols_per_group<T>(f, outer * sh.inner);
    const int64_t tiles = (sh.inner + tc - 1) / tc;
    const unsigned threads = (unsigned)((f.P * tc + 63) / 64 * 64);
    if (sh.inner > INT32_MAX || tiles * threads > kLaunchThreads) {
        set_error("FFT pass of %lld columns is too large", (long long)sh.inner);
        return JFA_ERR_TOO_LARGE;
    }
    sh.tiles = (int)tiles;
    const size_t lds = f.count > 1 ? (size_t)padded(f.L) * tc * 2 * sizeof(T) : 0;
    const int64_t most = kLaunchThreads / threads / tiles;  // outer indices of a launch
    const int64_t mode_step = 2 * sh.n * sh.inner, grid_step = 2 * sh.wl * sh.inner;
    auto go = [&](auto kernel) -> int {
        if (int rc = allow_lds(kernel, lds)) return rc;
        for (int64_t o0 = 0; o0 < outer; o0 += most) {
            const unsigned blocks = (unsigned)(tiles * std::min(most, outer - o0));
            kernel<<<blocks, threads, lds, s>>>(f, sh, tw, dk0, dkm, dkl,
                                                in + o0 * (TO_GRID ? mode_step : grid_step),
                                                out + o0 * (TO_GRID ? grid_step : mode_step));
            JFA_HIP_CHECK(hipGetLastError());
        }
        return JFA_OK;
    };
    auto pick = [&](auto tcc) -> int {
        constexpr int TC = decltype(tcc)::value;
        if (f.r[0] <= 8) return go(fft_cols_kernel<T, TC, 8, TO_GRID>);
        if (f.r[0] <= 10) return go(fft_cols_kernel<T, TC, 10, TO_GRID>);
        return go(fft_cols_kernel<T, TC, sizeof(T) == 8 ? 10 : 16, TO_GRID>);
    };
    constexpr int kWide = 128 / (2 * sizeof(T));
    if (tc == kWide) return pick(std::integral_constant<int, kWide>{});
    if (tc == kWide / 2) return pick(std::integral_constant<int, kWide / 2>{});
    return pick(std::integral_constant<int, kWide / 4>{});
}

}  // namespace

bool axis_fft(int64_t L, size_t real_size, AxisFft *f) {
    if (L < 2 || L > 4096) return false;
    // 32 bytes of columns have to fit a workgroup
    const int least = 32 / (2 * (int)real_size);
    if ((size_t)padded((int)L) * 32 > kMaxLds) return false;
    auto stages = [&](int max_r) {
        AxisFft cur{}, best{};
        search_stages((int)L, max_r, cur, best);
        best.L = (int)L;
        best.P = best.count ? best.L / best.r[best.count - 1] : 0;
        if (best.P * least > kMaxThreads) best.count = 0;
        return best;
    };
    // Radices above 10 only where they leave one or two stages, or where
    // nothing else fits: their butterflies take twice the registers and idle
    // half the threads of the other stages (y pass of 512 columns of 1024 points:
    // stages 16 8 8 17.7 us, 8 8 4 4 13.9 us; of 256 x 128 columns of 256: 16 16
    // 18.7 us, 8 8 4 22.7 us).  Doubles never: a radix-16 butterfly of complex
    // doubles needs more than the 128 registers a 1024-thread workgroup has.
    *f = stages(10);
    if (real_size == 4) {
        const AxisFft wide = stages(16);
        if (wide.count && (f->count == 0 || (wide.count < f->count && wide.count <= 2))) *f = wide;
    }
    if (f->count == 0) return false;
    int Ns = f->r[0];
    f->ntw = 0;
    for (int s = 1; s < f->count; ++s) {
        f->t[s] = f->ntw;
        f->ntw += (f->r[s] - 1) * Ns;
        Ns *= f->r[s];
    }
    return true;
}

template <typename T>
int launch_axis_twiddles(const AxisFft &f, T *tw, hipStream_t s) {
    if (f.ntw == 0) return JFA_OK;
    axis_twiddle_kernel<T><<<(unsigned)((f.ntw + 255) / 256), 256, 0, s>>>(f, tw);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

static ColsShape cols_shape(int64_t inner, int64_t n, int64_t w0, int64_t wl, jfa_plan p) {
    ColsShape sh{};
    sh.inner = inner;
    sh.n = (int)n;
    sh.w0 = (int)w0;
    sh.wl = (int)wl;
    sh.n0 = (int)p->nmodes[0];
    sh.nm = 1;
    sh.modeord = p->opts.modeord;
    sh.swap = p->iflag > 0;
    return sh;
}

template <typename T>
int axis_grid_to_modes(jfa_plan p, T *fw, T *work, T *fk, int nb) {
    const int64_t *n = p->nmodes, *nf = p->geom.nf;
    const T *tw[3] = {(const T *)p->d_tw[0], (const T *)p->d_tw[1], (const T *)p->d_tw[2]};
    const T *dk[3] = {(const T *)p->d_dk[0], (const T *)p->d_dk[1], (const T *)p->d_dk[2]};
    const int swap = p->iflag > 0;
    if (int rc = launch_rows<T, false>(p->axis[0], tw[0], nb * nf[1] * nf[2], n[0],
                                       p->opts.modeord, swap, fw, work, p->stream))
        return rc;
    ColsShape y = cols_shape(n[0], n[1], 0, nf[1], p);
    if (p->dim == 2)
        return launch_cols<T, false>(p->axis[1], tw[1], nb, y, dk[0], dk[0], dk[1], work, fk,
                                     p->stream);
    if (int rc = launch_cols<T, false>(p->axis[1], tw[1], nb * nf[2], y, nullptr, nullptr,
                                       (const T *)nullptr, work, fw, p->stream))
        return rc;
    ColsShape z = cols_shape(n[0] * n[1], n[2], 0, nf[2], p);
    z.nm = (int)n[1];
    return launch_cols<T, false>(p->axis[2], tw[2], nb, z, dk[0], dk[1], dk[2], fw, fk,
                                 p->stream);
}

template <typename T>
int axis_modes_to_grid(jfa_plan p, const T *fk, T *work, T *fw, int nb) {
    const GridGeom &g = p->geom;
    const int64_t *n = p->nmodes;
    const T *tw[3] = {(const T *)p->d_tw[0], (const T *)p->d_tw[1], (const T *)p->d_tw[2]};
    const T *dk[3] = {(const T *)p->d_dk[0], (const T *)p->d_dk[1], (const T *)p->d_dk[2]};
    const int swap = p->iflag > 0;
    const int64_t ry = window_rows(g, 1), rz = window_rows(g, 2);
    ColsShape y = cols_shape(n[0], n[1], g.wlen[1] ? g.wstart[1] : 0, ry, p);
    if (p->dim == 2) {
        if (int rc = launch_cols<T, true>(p->axis[1], tw[1], nb, y, dk[0], dk[0], dk[1], fk,
                                          work, p->stream))
            return rc;
    } else {
        ColsShape z = cols_shape(n[0] * n[1], n[2], g.wlen[2] ? g.wstart[2] : 0, rz, p);
        z.nm = (int)n[1];
        if (int rc = launch_cols<T, true>(p->axis[2], tw[2], nb, z, dk[0], dk[1], dk[2], fk, fw,
                                          p->stream))
            return rc;
        if (int rc = launch_cols<T, true>(p->axis[1], tw[1], nb * rz, y, nullptr, nullptr,
                                          (const T *)nullptr, fw, work, p->stream))
            return rc;
    }
    return launch_rows<T, true>(p->axis[0], tw[0], nb * ry * rz, n[0], p->opts.modeord, swap,
                                work, fw, p->stream);
}

#define JFA_INST(T)                                                        \
    template int launch_axis_twiddles<T>(const AxisFft &, T *, hipStream_t); \
    template int axis_grid_to_modes<T>(jfa_plan, T *, T *, T *, int);      \
    template int axis_modes_to_grid<T>(jfa_plan, const T *, T *, T *, int);
JFA_INST(float)
JFA_INST(double)
#undef JFA_INST

}  // namespace jfa
