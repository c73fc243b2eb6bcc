// Internal declarations of the MI355X NUFFT backend: kernel-parameter math
// (host), plan state, and the kernel launchers the plan drives.
#pragma once

#include <hip/hip_runtime.h>
#include <rocfft/rocfft.h>

#include <cstdint>
#include <mutex>
#include <string>

#include "jax_finufft_amd.h"

#include "kernel_math.hpp"

namespace jfa {

#define JFA_HIP_CHECK(expr)                                                              \
    do {                                                                                 \
        hipError_t _e = (expr);                                                          \
        if (_e != hipSuccess) {                                                          \
            ::jfa::set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e),      \
                             __FILE__, __LINE__);                                        \
            (void)hipGetLastError(); /* reported here; do not leak into later checks */  \
            return JFA_ERR_HIP;                                                          \
        }                                                                                \
    } while (0)

// ------------------------------------------------------------ launch args

// Geometry of the fine grid and of the point bins, passed by value to kernels.
struct GridGeom {
    int64_t nf[3];       // fine grid, x fastest (1 for unused dims)
    double scale[3];     // grid units per coordinate unit: u = (x - shift) * scale
    double shift[3];     // 0 for types 1/2; the type-3 centre otherwise
    int bs[3];           // bin size in cells
    int nb[3];           // bins per dimension
    int64_t nbins;       // product of nb
    int ns;              // kernel width
    int dim;
    int ymajor;          // 2D bins ordered y fastest (bin = by + nb1*bx), for strips
    int keyshift;        // sort key = bin << keyshift | (first-tap offset bits); 0 = bin only
    int subw[3];         // bits of the first tap's offset within its bin per dimension
                         // (LDS-tile / global methods without a gather; see SortedPts)
    // Rows a type-2 plan keeps (set for the inner plan of type 3 only): along
    // axes 1 and 2 the fine grid holds just cells wstart[d] .. wstart[d] +
    // wlen[d] - 1 (mod nf[d]), which cover every tile and tap its points read;
    // wlen[d] = 0 keeps the whole axis.  Axis 0 is always whole.
    int64_t wstart[3], wlen[3];
};

// Row index of wrapped cell c of axis d within the kept rows, and the number of
// kept rows (see GridGeom::wstart).
__host__ __device__ inline int64_t window_cell(const GridGeom &g, int d, int64_t c) {
    if (g.wlen[d] == 0) return c;
    const int64_t r = c - g.wstart[d];
    return r < 0 ? r + g.nf[d] : r;
}
__host__ __device__ inline int64_t window_rows(const GridGeom &g, int d) {
    return g.wlen[d] ? g.wlen[d] : g.nf[d];
}
// Complex cells per transform of a plan's fine grid as stored.
inline int64_t stored_cells(const GridGeom &g) {
    return g.nf[0] * window_rows(g, 1) * window_rows(g, 2);
}

// Geometry of the 2D strip spreader (kernels_strip.hip): strips of SW = 64 -
// ns + 1 columns, units of H rows, K units per strip.
struct StripGeom {
    int64_t nf0, nf1;
    int SW, S;      // strip width (owned first taps) and strip count
    int H, K;       // rows per unit, units per strip
    int nz;         // slices (nf2 for a 3D grid, 1 in 2D)
    int nunits;     // nz * S * K
    int ns;
    int pmax;       // most points per piece (a unit has ceil(count / pmax) pieces)
};

constexpr int kStripPiece = 4096;  // default pmax

// Complex cells of one piece's scratch tile, and the most pieces M points can
// make (sum over units of ceil(count / pmax) <= units + M / pmax).
inline int64_t strip_tile_cells(const StripGeom &sg) { return (int64_t)(sg.H + sg.ns - 1) * 64; }
inline int64_t strip_max_pieces(const StripGeom &sg, int64_t M) {
    return std::min<int64_t>(sg.nunits, M) + M / sg.pmax + 1;
}
// Units with more than one piece hold more than pmax points each.
inline int64_t strip_max_heavy(const StripGeom &sg, int64_t M) { return M / (sg.pmax + 1) + 1; }

// Most rows of a unit: short units, whose tile the spreading kernel's accumulators hold,
// and the tall ones of sparse grids.
constexpr int strip_short_rows(int ns) { return ns <= 8 ? 9 : 33 - ns; }
constexpr int strip_tall_rows(int ns) { return ns <= 8 ? 33 - ns : 128; }
// Strips of a grid g (nf and ns set) in short units; also sets g's bins to (strip, row),
// rows fastest, which do not depend on the units.
StripGeom strip_geometry(GridGeom &g, int pmax);
// Sets the height of the units, as near `rows` as they may have.
void strip_set_rows(StripGeom &sg, int64_t rows);
// Whether tall units suit that many points (slice points in 3D) in all of so many short
// units, over every transform.
bool strip_tall(int ns, double points, double units);
// Sets the height that suits M points of nb transforms; rows > 0 asks for one
// (gpu_binsizey).
void strip_units(StripGeom &sg, int64_t M, int nb, int rows);
int ensure_rocfft();

// Batched 1D FFTs in LDS (fft_lds.hip), for rows of length n = 2^a 3^b 5^c <=
// kLdsFftMax: the stage radices, the twiddle table tw[k] = (cos, sin)(2 pi k /
// n) (n complex values, built by launch_fft_twiddles) and the in-place
// transform of `batch` contiguous rows, sign +1 or -1, unnormalised.
constexpr int kLdsFftMax = 4096;
struct LdsFftRadices {
    int count;
    int r[16];
};
bool lds_fft_radices(int64_t n, LdsFftRadices *f);
template <typename T>
int launch_fft_twiddles(int64_t n, T *tw, hipStream_t stream);
template <typename T>
int launch_fft_lds(T *data, int64_t n, int64_t batch, const T *tw, int sign, hipStream_t stream);
// Stages of one axis of the pruned FFT passes (fft_axis.hip): length L (2, 3, 5
// -smooth, at most 4096) as `count` radices, P = L / the smallest of them
// threads per transform.  False where those passes cannot run an axis.
struct AxisFft {
    int L, P, count;
    int r[8];
    int t[8];  // first entry of stage s's twiddles (s >= 1), ntw of them in all
    int ntw;
};
bool axis_fft(int64_t L, size_t real_size, AxisFft *f);
template <typename T>
int launch_axis_twiddles(const AxisFft &f, T *tw, hipStream_t s);
// Held around every rocFFT plan creation and destruction: calls from several
// host threads (concurrent transforms through the plan cache) are serialised
// there rather than relying on the library's own locking.
std::mutex &rocfft_mutex();

// Ragged batch of 2D type-1 problems (ragged.hip).  Per problem: its grid and
// bins for setpts.  Per virtual problem (problem, transform): what spreading,
// merging and deconvolution need.  Offsets count complex cells.
struct RaggedProb {
    GridGeom g;
    int64_t moff;     // first point in the concatenated point order
    int64_t bin_off;  // first global bin
};
struct RaggedVirt {
    StripGeom sg;
    int prob, t;
    int nt;            // transforms this one spreads: 2 (itself and t + 1, which
                       // shares its points), 1, or 0 (spread with t - 1)
    int64_t tile_next; // tile_off of transform t + 1 minus this tile_off
    int64_t m;         // the problem's point count
    int64_t bin_off;   // the problem's first global bin
    int64_t fw_off;    // into the concatenated fine grids
    int64_t g_off;     // into the concatenated pruned-FFT buffers ([n0][nf1] each)
    int64_t tile_off;  // into the concatenated scratch tiles
    int unit_off;      // first global unit
    int64_t n0, n1;    // modes, x fastest
    int64_t dk_off;    // 1/psi_hat: dk0 at dk + dk_off, dk1 at dk + dk_off + n0
    int64_t moff;      // the problem's first point in the concatenated order
                       // (sorted indices are concatenated-order indices)
};
// Device tables and sizes of one ragged launch sequence.
struct RaggedLaunch {
    const RaggedProb *probs;
    const RaggedVirt *virt;
    const int64_t *moff;       // nprob + 1
    const int *vunit_off;      // nv + 1
    const int64_t *mode_blk;   // nv + 1: first deconv block (32 x 32 modes)
    const void *const *ptrs;   // x[nprob], y[nprob], c[nprob], f[nprob]
    const int *unit_virt;      // nunits: virtual problem of every global unit
    int *bin_start, *piece_start, *npieces;
    int *piece_unit;           // global unit of every piece
    int *heavy;                // [count, units with more than one piece ...]
    int64_t max_heavy;         // most such units
    int64_t max_pieces;        // most pieces, over every virtual problem
    bool tall;                 // units of more than strip_short_rows rows
    int reduce_chunks;         // 256-cell chunks of the largest tile
    int *blocksum;             // 2 * ceil(nunits / 256) + 1 ints of piece-scan scratch
    int nprob, nv, ns, pmax, keyshift;
    int64_t mtot, nbins, nunits, mode_blocks;
};
// Transforms of a problem that one wave spreads together.
constexpr int ragged_transforms(size_t real) { return real == 4 ? 2 : 1; }
// Workgroups of the spreading launch, one per piece.  Every transform of a problem
// has its own pieces, so the points of a problem with T transforms count T times
// (mtot counts them once).
inline int64_t ragged_strip_blocks(const RaggedLaunch &rl) { return rl.max_pieces; }

// Points after setpts, in bin-sorted order: original index, first tap
// (wrapped into [0, nf)) and the Horner variable t = 2*frac - 1 per dim.
// Either as arrays in sorted order (l0, t), or, when key != NULL, without a
// gather: the sorted key holds the bin and the first taps' offsets within it
// (GridGeom::keyshift / subw) and rec[j*dim + d] holds t_d of input point j.
template <typename T>
struct SortedPts {
    int64_t M;
    const int *idx;
    const int *l0[3];
    const T *t[3];
    const unsigned *key;
    const T *rec;
};

// Points as the 2D strip spreader reads them: the sorted keys and original
// indices from its setpts, and one 4-value record per input point built at
// execute time (launch_strip_pack) from the strength and the Horner variables
// setpts wrote in input order: pack[4j..4j+3] = (Re c_j, Im c_j, tx_j, ty_j).
// One record read per point instead of two scattered reads; setpts needs no
// gather.  key = (bin << kStripKeyShift) | X with bin = bin_off + s*nf1 + l0y
// (s the strip) and X = l0x - s*SW in [0, SW).
constexpr int kStripKeyShift = 6;
// Lowest key bit the strip sorts order by: points of a (strip, row) bin keep
// input order (the spreader groups each batch by column itself).
constexpr int kStripSortLowBit = kStripKeyShift;
template <typename T>
struct StripPts {
    int64_t M;
    const int *idx;       // sorted position -> input point P (over all problems)
    const unsigned *key;  // sorted keys
    const T *pack;        // records of the problem's transform, by local index j;
                          // NULL: read c[j] (this transform's strengths) and rec[P]
    const T *c;
    const T *rec;         // (tx, ty) of input point P at rec[2*P], written by setpts
    int64_t bin_off;      // the problem's first global bin (0 for one plan)
    int64_t idx_off;      // the problem's first input point: j = P - idx_off
    int64_t c_tstride;    // reals from one transform's strengths to the next (c path)
};

// Per-bin bookkeeping for the LDS-subproblem method.
struct BinIndex {
    const int *bin_start;  // nbins+1 exclusive prefix of counts
    const int *sub_start;  // nbins+1 exclusive prefix of subproblems per bin
    const int *nsub;       // total subproblems (device scalar)
    int maxsub;
};

// Scratch of the point sort: the keys before and after, and radix_temp_bytes of
// scratch.
struct SortScratch {
    unsigned *key_in, *key_out;
    void *temp;
};
// Stable sort of kin[0 .. M) by bits [b0, b1) (bits above b1 are zero): sorted
// keys to kout, their input positions to vout.  Where one workgroup holds all
// keys and the bins are few it also writes bin_start (see bin_bounds_kernel)
// and sets *bounded.  temp: radix_temp_bytes(M, b1 - b0), or of more keys.
constexpr int kWidestSortBits = 22;  // the span with the largest scratch
size_t radix_temp_bytes(int64_t M, int bits = kWidestSortBits);
int radix_sort(void *temp, const unsigned *kin, unsigned *kout, unsigned *vout, int64_t M,
               int b0, int b1, int64_t nbins, int bin_shift, int *bin_start, bool *bounded,
               hipStream_t stream);
// Bits the strip sorts order by, for nbins (strip, row) bins.
int strip_sort_bits(int64_t nbins);

// Launchers (kernels_*.hip).  All queue work on `stream` and return a JFA code.
// Bin, radix-sort and gather M points: idx/l0/tv in bin order, bin_start
// (nbins + 1) and, when sub_start is non-null, the LDS-subproblem prefix
// (sub_start holds nbins + 1 + 2 * ceil(nbins / 256) + 1 ints: the prefix, then
// scan scratch).
template <typename T>
int launch_sort_points(const GridGeom &g, int64_t M, const T *x, const T *y, const T *z,
                       const SortScratch &s, int *bin_start, int *sub_start, int *nsub,
                       int maxsub, int *idx, int *l0, T *tv, hipStream_t stream);
// The same without the gather (g.keyshift = sum of g.subw > 0): keys with the
// offset bits, the Horner variables in input order in rec (dim per point), the
// sorted keys left in s.key_out.
template <typename T>
int launch_sort_points_keyed(const GridGeom &g, int64_t M, const T *x, const T *y, const T *z,
                             const SortScratch &s, int *bin_start, int *sub_start, int *nsub,
                             int maxsub, int *idx, T *rec, hipStream_t stream);
// Same per-point data in input order (no sort).
template <typename T>
int launch_fold_points(const GridGeom &g, int64_t M, const T *x, const T *y, const T *z,
                       int *idx, int *l0, T *tv, hipStream_t stream);
int launch_fill_zero(void *p, int64_t bytes, hipStream_t stream);
// Setpts of the 2D strip spreader: keys (with the first-tap column, see
// StripPts) radix-sorted with the original indices, bin_start, and the Horner
// variables written in input order to rec; no gather.
template <typename T>
int launch_sort_points_strip(const GridGeom &g, int64_t M, const T *x, const T *y,
                             const SortScratch &s, int *bin_start, int *idx, T *rec,
                             hipStream_t stream);
// 3D slices of S strips each: keys of the ns slice points of every point
// (M * ns of them), sorted; rec3 = (tx, ty, tz) per point.
template <typename T>
int launch_sort_points_slices(const GridGeom &g, int S, int64_t M, const T *x, const T *y,
                              const T *z, const SortScratch &s, int *bin_start, int *idx,
                              T *rec3, hipStream_t stream);

template <typename T>
int launch_spread(int method, const GridGeom &g, const SortedPts<T> &pts, const BinIndex &bi,
                  const T *coef, int kerevalmeth, double beta, const T *c, int64_t c_stride,
                  T *fw, int64_t fw_stride, int ntr, hipStream_t stream);
template <typename T>
int launch_spread_strip(const StripGeom &sg, const StripPts<T> &pts, const int *bin_start,
                        int *piece_start, int *npieces, int *piece_unit, int *heavy,
                        int *blocksum, const T *coef, int kerevalmeth, double beta,
                        int64_t pack_stride, T *fw,
                        int64_t fw_stride, T *scratch, int64_t scratch_stride, int ntr,
                        int phases, hipStream_t stream);
// 3D slices: pack[t][j * ns + dz] = (c[t][j] * kz_j[dz], tx_j, ty_j) for the ns
// slice points of point j; rec3[3j .. 3j+2] = (tx, ty, tz) from setpts
template <typename T>
int launch_strip3_pack(const T *c, int64_t c_stride, const T *rec3, const T *coef,
                       int kerevalmeth, double beta, int ns, int64_t M, int ntr, T *pack,
                       hipStream_t stream);
// pack[t][j] = (c[t][j], rec[j]) for t < ntr, j < M (records of 4 reals)
template <typename T>
int launch_strip_pack(const T *c, int64_t c_stride, const T *rec, int64_t M, int ntr, T *pack,
                      hipStream_t stream);
// Column gather / scatter transposes of the pruned FFT (fft_pruned.hip).  For
// each of `outer` blocks: B[j][r] = A[r][col(j)] (j < J, r < R, A rows of C
// complex values), col(j) = (j / nsel) * cblk + (i < (nsel+1)/2 ? i : cblk -
// nsel + i) with i = j % nsel; scatter writes all of A, zeros where no j maps.
template <typename T>
int gather_cols(const T *A, T *B, int64_t outer, int64_t R, int64_t C, int64_t J, int64_t nsel,
                int64_t cblk, hipStream_t s);
// scatter_cols writes A's rows r < Rout from B's rows (r0 + r) mod R (all of
// them: r0 = 0, Rout = R).
template <typename T>
int scatter_cols(const T *B, T *A, int64_t outer, int64_t R, int64_t C, int64_t J, int64_t nsel,
                 int64_t cblk, int64_t r0, int64_t Rout, hipStream_t s);
// 2D deconvolution of one transform from the compact buffer G[j0][y] (n0 x
// nf1) into the n0 x n1 modes, without a plan (dk_d[k + n_d/2] = 1/psi_hat).
template <typename T>
int launch_deconv_pruned_2d(int64_t n0, int64_t n1, int64_t nf1, const T *dk0, const T *dk1,
                            int modeord, const T *G, T *out, hipStream_t stream);

// phases of launch_spread_strip (a bit mask): piece table, spreading, merge
constexpr int kStripUnits = 1, kStripSpread = 2, kStripMerge = 4, kStripAll = 7;
// Ragged batch: sort every problem's points at once (global bins), then the
// strip phases over every virtual problem's units, then deconvolution.
template <typename T>
int launch_ragged_sort(const RaggedLaunch &rl, const SortScratch &s, int *idx, T *rec,
                       hipStream_t stream);
template <typename T>
int launch_ragged_strip(const RaggedLaunch &rl, const StripPts<T> &pts, const T *coef,
                        int kerevalmeth, double beta, T *fw_all, T *scratch_all, int phases,
                        hipStream_t stream);
template <typename T>
int launch_ragged_deconv(const RaggedLaunch &rl, const T *dk, int modeord, const T *g_all,
                         hipStream_t stream);
template <typename T>
int launch_interp(int method, const GridGeom &g, const SortedPts<T> &pts, const BinIndex &bi,
                  const T *coef, int kerevalmeth, double beta, const T *fw, int64_t fw_stride,
                  T *c, int64_t c_stride, int ntr, hipStream_t stream);
// Fused interpolation + point gradient, grad[d*grad_stride + j]: LDS tiles
// for JFA_METHOD_SM, taps read from the fine grid otherwise.
template <typename T>
int launch_interp_grad(int method, const GridGeom &g, const SortedPts<T> &pts,
                       const BinIndex &bi, const T *coef, const T *fw, int64_t fw_stride,
                       int ntr, const T *w, int64_t w_stride, T *val, int64_t val_stride,
                       T *grad, int64_t grad_stride, int accumulate, hipStream_t stream);
template <typename T>
int launch_deconv(int dim, const int64_t *n, const int64_t *nf, const T *dk0, const T *dk1,
                  const T *dk2, int modeord, const T *fw, int64_t fw_stride, T *out,
                  int64_t out_stride, int ntr, hipStream_t stream);
template <typename T>
int launch_amplify(int dim, const int64_t *n, const int64_t *nf, const T *dk0, const T *dk1,
                   const T *dk2, int modeord, const T *f, int64_t f_stride, T *fw,
                   int64_t fw_stride, int ntr, hipStream_t stream);

// Type-3 helpers (kernels_type3.hip).
// Per-array [min, max] of n values into out2 (device doubles).
template <typename T>
int launch_minmax(int64_t n, const T *a, double *out2, hipStream_t s);
// The same with the partials (2 * 1024 doubles) at `part`.
template <typename T>
int launch_minmax_to(int64_t n, const T *a, double *out2, double *part, hipStream_t s);
// Type 3 over a partition of the targets into k[0] x k[1] x k[2] boxes of
// width `width` from `lo` (box index x fastest): count (2 nbox ints of
// scratch), start (nbox + 1 offsets), the box order perm and the coordinates
// in that order (sorted[d * N + q]); then the reordering of box-ordered
// outputs (box b's nb transforms as [t][N_b] at out + 2 nb start[b]) into f.
struct BoxGrid {
    double lo[3], width[3];
    int k[3];
};
template <typename T>
int launch_t3_box_sort(int dim, int64_t N, const T *s, const T *t, const T *u,
                       const BoxGrid &bg, int nbox, int *count, int64_t *start, int *perm,
                       T *sorted, hipStream_t stream);
template <typename T>
int launch_t3_unsort(int64_t N, int nb, int nbox, const int64_t *start, const int *perm,
                     const T *out, T *f, hipStream_t stream);
// cp[t][j] = c[t][j] * exp(i iflag sum_d D_d (x_dj - C_d))
template <typename T>
int launch_t3_prephase(int dim, int64_t M, int ntr, const T *x, const T *y, const T *z,
                       const double *C, const double *D, int iflag, const T *c, T *cp,
                       hipStream_t stream);
// dec[k] = 1 / prod_d psi_hat(h_d gam_d (s_dk - D_d)) from the plan's table: in fp64
// the quadrature's (wt[q], sn[q]), psi_hat(w) = ns sum_q wt[q] cos(w ns sn[q] / 2); in
// fp32 the series of kernel_fourier_series over |w| <= range.
template <typename T>
int launch_t3_deconv_factors(int dim, int64_t N, const T *s, const T *t, const T *u,
                             const double *D, const double *hg, int ns, double range,
                             const double *table, T *dec, hipStream_t stream);
// f[t][k] *= exp(i iflag sum_d s_dk C_d) * dec[k]
template <typename T>
int launch_t3_postphase(int dim, int64_t N, int ntr, const T *s, const T *t, const T *u,
                        const double *C, int iflag, const T *dec, T *f, hipStream_t stream);

}  // namespace jfa
