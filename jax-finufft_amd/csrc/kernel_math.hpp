// Plan-time kernel mathematics of the NUFFT method (params.cpp), shared by
// the HIP library and the CPU target: plain C++, no device headers.
#pragma once

#include <cstdint>

namespace jfa {

constexpr int kMaxNs = 16;  // widest ES kernel supported (taps per dimension)
constexpr int kMaxNc = 19;  // most Horner coefficients per kernel interval
// Largest fine grid (cells per transform) a plan accepts: the FFT sizes this
// backend validates.
constexpr int64_t kMaxFineCells = (int64_t)1 << 32;

// Horner coefficients per interval for width ns: degree ns+2 below ns = 14,
// else 18.  The Chebyshev-interpolation error is then at most 0.54 exp(-beta)
// for every width and both upsampling factors, below the kernel's own
// truncation value; higher degrees gain little (0.46 exp(-beta) at ns+4),
// since the kernel's square-root edge limits the convergence.
constexpr int horner_nc(int ns) { return ns < 14 ? ns + 3 : kMaxNc; }

// ------------------------------------------------------------ host math

struct KernelParams {
    int ns = 0;        // width in fine-grid cells
    int nc = 0;        // Horner coefficients per interval
    double beta = 0;   // ES shape parameter
    int warn = 0;      // 1 = eps below what the width cap / precision reaches
};

// Width, beta for tolerance eps at upsampling factor sigma (params.cpp).
KernelParams choose_kernel(double eps, double sigma, int rule, int is_double, int forced_ns);
int64_t next235even(int64_t n);
int64_t fine_size(int64_t n, double sigma, int ns);
// Monomial Horner coefficients, power-major: coef[p*ns + i] multiplies t^p on
// interval i (tap i of a point; t = 2*frac - 1 in [-1, 1)).
void horner_fit(int ns, int nc, double beta, double *coef);
// psi_hat(k h) for k = kmin .. kmin+n-1 on a fine grid of nf cells.
void kernel_fourier(int ns, double beta, double nf, double kmin, int64_t n, double *out);
// psi_hat at arbitrary frequencies omega (radians per fine-grid cell).
void kernel_fourier_at(int ns, double beta, const double *omega, int64_t n, double *out);
void gauss_legendre(int n, double *x, double *w);
// The quadrature behind kernel_fourier_at: psi_hat(omega) = ns * sum_p wt[p]
// cos(omega ns sn[p] / 2) over q = 2 ns + 40 <= kMaxFourierNodes nodes;
// returns q.
constexpr int kMaxFourierNodes = 2 * kMaxNs + 40;
int kernel_fourier_nodes(int ns, double beta, double *sn, double *wt);
// The same as a series for |omega| <= range <= 1.02 pi: psi_hat(omega) / ns = sum_j
// coef[j] T_j(2 (omega / range)^2 - 1) over nt = ns + 20 Chebyshev polynomials;
// returns nt.
int kernel_fourier_series(int ns, double beta, double range, double *coef);

// ------------------------------------------------------------ errors

void set_error(const char *fmt, ...);
const char *last_error();

}  // namespace jfa
