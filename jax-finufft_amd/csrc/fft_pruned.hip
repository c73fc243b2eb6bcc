// Pruned multi-dimensional FFT between the fine grid and the modes, for 2D and
// 3D plans.  Replaces the full nf0 x nf1 (x nf2) FFT cuFINUFFT runs inside
// execute (called at lib/kernels.cc.cu:75; source absent from the reference)
// with 1D passes that skip the columns no mode needs.
//
// Of the nf_d fine-grid frequencies along an axis only the n_d mode
// frequencies k in [-n_d/2, (n_d-1)/2] are kept; they sit at fine index
// k mod nf_d.  Compact index j in [0, n_d) stands for k = j (j < (n_d+1)/2)
// or k = j - n_d, i.e. fine index sel(j) = j or nf_d - n_d + j.
//
// Type 1 (fine grid -> modes), 2D: x-FFT of every row (length nf0); gather the
// n0 needed columns transposed into G[t][j0][y]; y-FFT of those n0 rows
// (length nf1); deconvolve from G.  3D: x-FFT; gather into
// G1[t][z][j0][y]; y-FFT; gather the n1 needed y of each (z, j0) transposed
// into G2[t][j0][j1][z] (in the fine grid's memory, dead by then); z-FFT;
// deconvolve from G2.  Type 2 runs the same steps backwards: amplify into the
// compact buffer (zero outside the mode rows), FFT, scatter-transpose into the
// next larger buffer writing zeros in the unused columns, ..., x-FFT of the
// full grid.  Data moved per transform, 2D: 2F + F/2 + F/2 + F/2 against 8F
// for rocFFT's row-FFT / transpose / row-FFT / transpose of the full grid.
#include "jfa_device.hpp"
#include "plan_state.hpp"

namespace jfa {
namespace {

// fine index of compact index j, and the compact index of fine index c or -1
// when no mode lives there (32-bit: every axis and every product of the mode
// counts the transposes below see is below 2^31; addresses are 64-bit)
__device__ __forceinline__ int sel_of(int j, int n, int nf) { return j < (n + 1) / 2 ? j : nf - n + j; }
__device__ __forceinline__ int unsel_of(int c, int n, int nf) {
    if (c < (n + 1) / 2) return c;
    if (c >= nf - n / 2) return c - nf + n;
    return -1;
}

constexpr int kTile = 32;

// One complex value, moved as one 8- (16-) byte access.
template <typename T>
struct alignas(2 * sizeof(T)) Cx {
    T x, y;
};

// B[o][j][r] = A[o][r][col(j)] for j < J, r < R; col(j) = (j / nsel) * cblk +
// sel_of(j % nsel, nsel, cblk); A rows hold C complex values.  One 32 x 32
// tile of (j, r) per workgroup of 32 x 8 threads, through LDS, each value one
// complex-wide access.  Index arithmetic is 32-bit (one division pair per
// thread for its column); the host checks the extents.
template <typename T>
__global__ void __launch_bounds__(256)
    gather_cols_kernel(const T *__restrict__ A, T *__restrict__ B, int R, int C, int J, int nsel,
                       int cblk, int jt, int rt) {
    __shared__ Cx<T> tt[kTile][kTile + 1];
    unsigned tile = blockIdx.x;
    const int jb = (int)(tile % (unsigned)jt);
    tile /= (unsigned)jt;
    const int rb = (int)(tile % (unsigned)rt);
    const int64_t o = tile / (unsigned)rt;
    const int tx = threadIdx.x & (kTile - 1), ty = threadIdx.x / kTile;
    const Cx<T> *Ac = reinterpret_cast<const Cx<T> *>(A) + o * R * C;
    Cx<T> *Bc = reinterpret_cast<Cx<T> *>(B) + o * J * R;
    // read: lanes along j (columns of A), rows r
    const int j = jb * kTile + tx;
    int col = -1;
    if (j < J) col = (j / nsel) * cblk + sel_of(j % nsel, nsel, cblk);
    for (int k = ty; k < kTile; k += 8) {
        const int r = rb * kTile + k;
        tt[k][tx] = (col >= 0 && r < R) ? Ac[(int64_t)r * C + col] : Cx<T>{T(0), T(0)};
    }
    __syncthreads();
    // write: lanes along r (rows of B)
    const int r = rb * kTile + tx;
    for (int k = ty; k < kTile; k += 8) {
        const int jj = jb * kTile + k;
        if (jj < J && r < R) Bc[(int64_t)jj * R + r] = tt[tx][k];
    }
}

// A[o][r][c] = B[o][unsel(c)][(r0 + r) mod R] for every c < C and r < Rout (0
// where no compact column maps to c); the inverse of gather_cols_kernel,
// writing every element of A.  One tile of 64 columns x 32 rows per workgroup
// (each thread has eight reads in flight, then eight writes); the tile's 64
// source rows of B are found once, into LDS.
constexpr int kScatterCols = 64;
template <typename T>
__global__ void __launch_bounds__(256)
    scatter_cols_kernel(const T *__restrict__ B, T *__restrict__ A, int R, int C, int J, int nsel,
                        int cblk, int r0, int Rout, int ct, int rt) {
    __shared__ Cx<T> tt[kScatterCols][kTile + 1];
    __shared__ int src[kScatterCols];
    unsigned tile = blockIdx.x;
    const int cb = (int)(tile % (unsigned)ct);
    tile /= (unsigned)ct;
    const int rb = (int)(tile % (unsigned)rt);
    const int64_t o = tile / (unsigned)rt;
    if (threadIdx.x < kScatterCols) {
        // compact row of B that column cb * 64 + t of A comes from, or -1
        const int c = cb * kScatterCols + (int)threadIdx.x;
        int u = -1;
        if (c < C) {
            const int uc = unsel_of(c % cblk, nsel, cblk);
            if (uc >= 0) u = (c / cblk) * nsel + uc;
        }
        src[threadIdx.x] = u;
    }
    __syncthreads();
    Cx<T> *Ac = reinterpret_cast<Cx<T> *>(A) + o * Rout * C;
    const Cx<T> *Bc = reinterpret_cast<const Cx<T> *>(B) + o * J * R;
    {
        // read: lanes along r (rows of B), one compact column per k
        const int tx = threadIdx.x & (kTile - 1), ty = threadIdx.x / kTile;
        const int r = rb * kTile + tx;
        int rs = r0 + r;
        if (rs >= R) rs -= R;
#pragma unroll
        for (int k = ty; k < kScatterCols; k += 8) {
            const int u = src[k];
            Cx<T> v{T(0), T(0)};
            if (u >= 0 && r < Rout) v = Bc[(int64_t)u * R + rs];
            tt[k][tx] = v;
        }
    }
    __syncthreads();
    // write: lanes along c (rows of A)
    const int tx = threadIdx.x & (kScatterCols - 1), ty = threadIdx.x / kScatterCols;
    const int c = cb * kScatterCols + tx;
    if (c >= C) return;
#pragma unroll
    for (int k = ty; k < kTile; k += 4) {
        const int rr = rb * kTile + k;
        if (rr < Rout) Ac[(int64_t)rr * C + c] = tt[tx][k];
    }
}

// The compact buffer of one transform is G[j0][jm][l]: j0 < n0 the compact
// x column, jm < nm the compact y index (3D; nm = 1 in 2D), l < nfl the
// full-length last axis (y in 2D, z in 3D).  Mode (i0, im, il) of the output
// (i0 fastest; il the last axis' mode index) sits at G[j0(k0)][jm(km)][kl mod
// nfl].  Both kernels below move one 32 x 32 tile of (x, last axis) through
// LDS so that G is read / written along l and the modes along i0.
struct PrunedShape {
    int64_t n0, nm, nl;    // modes along x, the middle axis, the last axis
    int64_t nfl;           // fine size of the last axis
    int64_t t0, tl, nmid;  // tiles along x and the last axis, middle count
};

__device__ __forceinline__ int idx_of(int k, int n, int modeord) {
    return modeord == 0 ? k + n / 2 : (k < 0 ? k + n : k);
}
// frequency of output index i (modeord 0: centred, 1: FFT order)
__device__ __forceinline__ int freq_of(int i, int n, int modeord) {
    if (modeord == 0) return i - n / 2;
    return i < (n + 1) / 2 ? i : i - n;
}

// out[t][i0 + n0*(im + nm*il)] = G[...] * dk0 dkm dkl.  Axis extents and tile
// counts are below 2^31, so indices are 32-bit and only addresses 64-bit.
template <typename T>
__global__ void __launch_bounds__(256)
    deconv_pruned_kernel(PrunedShape sh, const T *__restrict__ dk0, const T *__restrict__ dkm,
                         const T *__restrict__ dkl, int modeord, const T *__restrict__ G,
                         int64_t g_stride, T *__restrict__ out, int64_t out_stride) {
    __shared__ Cx<T> tt[kTile][kTile + 1];
    const int n0 = (int)sh.n0, nm = (int)sh.nm, nl = (int)sh.nl, nfl = (int)sh.nfl;
    unsigned b = blockIdx.x;
    const int xb = (int)(b % (unsigned)sh.t0);
    b /= (unsigned)sh.t0;
    const int lb = (int)(b % (unsigned)sh.tl);
    b /= (unsigned)sh.tl;
    const int im = (int)(b % (unsigned)sh.nmid);
    const int64_t t = b / (unsigned)sh.nmid;
    G += 2 * g_stride * t;
    out += 2 * out_stride * t;
    const int tx = threadIdx.x & (kTile - 1), ty = threadIdx.x / kTile;
    const int km = nm > 1 ? freq_of(im, nm, modeord) : 0;
    const int jm = km < 0 ? km + nm : km;
    // read along the last axis
    const int il = lb * kTile + tx;
    int l = -1;
    if (il < nl) {
        const int kl = freq_of(il, nl, modeord);
        l = kl < 0 ? kl + nfl : kl;
    }
    for (int k = ty; k < kTile; k += 8) {
        const int i0 = xb * kTile + k;
        Cx<T> v{T(0), T(0)};
        if (l >= 0 && i0 < n0) {
            const int k0 = freq_of(i0, n0, modeord);
            const int j0 = k0 < 0 ? k0 + n0 : k0;
            v = reinterpret_cast<const Cx<T> *>(G)[((int64_t)j0 * nm + jm) * nfl + l];
        }
        tt[k][tx] = v;
    }
    __syncthreads();
    // write along x
    const int i0 = xb * kTile + tx;
    if (i0 >= n0) return;
    const int k0 = freq_of(i0, n0, modeord);
    const T s0 = dk0[k0 + n0 / 2] * (nm > 1 ? dkm[km + nm / 2] : T(1));
    for (int k = ty; k < kTile; k += 8) {
        const int ill = lb * kTile + k;
        if (ill >= nl) break;
        const T s = s0 * dkl[freq_of(ill, nl, modeord) + nl / 2];
        const int64_t q = i0 + (int64_t)n0 * (im + (int64_t)nm * ill);
        const Cx<T> v = tt[tx][k];
        reinterpret_cast<Cx<T> *>(out)[q] = Cx<T>{v.x * s, v.y * s};
    }
}

// G[t][j0][jm][l] for every l < nfl: the mode value times 1/psi_hat where l
// holds a mode frequency, 0 elsewhere (every element of G is written)
template <typename T>
__global__ void __launch_bounds__(256)
    amplify_pruned_kernel(PrunedShape sh, const T *__restrict__ dk0, const T *__restrict__ dkm,
                          const T *__restrict__ dkl, int modeord, const T *__restrict__ f,
                          int64_t f_stride, T *__restrict__ G, int64_t g_stride) {
    __shared__ Cx<T> tt[kTile][kTile + 1];
    const int n0 = (int)sh.n0, nm = (int)sh.nm, nl = (int)sh.nl, nfl = (int)sh.nfl;
    unsigned b = blockIdx.x;
    const int xb = (int)(b % (unsigned)sh.t0);  // tiles of compact x columns
    b /= (unsigned)sh.t0;
    const int lb = (int)(b % (unsigned)sh.tl);  // tiles of the full last axis
    b /= (unsigned)sh.tl;
    const int jm = (int)(b % (unsigned)sh.nmid);
    const int64_t t = b / (unsigned)sh.nmid;
    f += 2 * f_stride * t;
    G += 2 * g_stride * t;
    const int tx = threadIdx.x & (kTile - 1), ty = threadIdx.x / kTile;
    const int km = nm > 1 ? (jm < (nm + 1) / 2 ? jm : jm - nm) : 0;
    // read the modes along x
    const int j0 = xb * kTile + tx;
    int i0 = -1;
    T s0 = T(0);
    if (j0 < n0) {
        const int k0 = j0 < (n0 + 1) / 2 ? j0 : j0 - n0;
        i0 = idx_of(k0, n0, modeord);
        s0 = dk0[k0 + n0 / 2] * (nm > 1 ? dkm[km + nm / 2] : T(1));
    }
    const int im = nm > 1 ? idx_of(km, nm, modeord) : 0;
    for (int k = ty; k < kTile; k += 8) {
        const int l = lb * kTile + k;
        Cx<T> v{T(0), T(0)};
        if (i0 >= 0 && l < nfl) {
            const int kl = l < (nfl + 1) / 2 ? l : l - nfl;
            if (kl >= -(nl / 2) && kl <= (nl - 1) / 2) {
                const int64_t q =
                    i0 + (int64_t)n0 * (im + (int64_t)nm * idx_of(kl, nl, modeord));
                const T s = s0 * dkl[kl + nl / 2];
                const Cx<T> fv = reinterpret_cast<const Cx<T> *>(f)[q];
                v = Cx<T>{fv.x * s, fv.y * s};
            }
        }
        tt[k][tx] = v;
    }
    __syncthreads();
    // write G along the last axis
    const int l = lb * kTile + tx;
    if (l >= nfl) return;
    for (int k = ty; k < kTile; k += 8) {
        const int jj = xb * kTile + k;
        if (jj >= n0) break;
        reinterpret_cast<Cx<T> *>(G)[((int64_t)jj * nm + jm) * nfl + l] = tt[tx][k];
    }
}

bool fits_int(std::initializer_list<int64_t> v) {
    for (int64_t x : v)
        if (x < 0 || x > INT32_MAX) return false;
    return true;
}

}  // namespace

template <typename T>
int gather_cols(const T *A, T *B, int64_t outer, int64_t R, int64_t C, int64_t J, int64_t nsel,
                int64_t cblk, hipStream_t s) {
    const int64_t jt = (J + kTile - 1) / kTile, rt = (R + kTile - 1) / kTile;
    const int64_t blocks = jt * rt * outer;
    if (blocks == 0) return JFA_OK;
    if (blocks > INT32_MAX) {
        set_error("pruned FFT transpose of %lld tiles is too large", (long long)blocks);
        return JFA_ERR_TOO_LARGE;
    }
    if (!fits_int({R, C, J, nsel, cblk, (J + nsel - 1) / nsel * cblk})) {
        set_error("pruned FFT transpose extents beyond 32-bit indexing");
        return JFA_ERR_TOO_LARGE;
    }
    gather_cols_kernel<T><<<(unsigned)blocks, 256, 0, s>>>(A, B, (int)R, (int)C, (int)J, (int)nsel,
                                                           (int)cblk, (int)jt, (int)rt);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int scatter_cols(const T *B, T *A, int64_t outer, int64_t R, int64_t C, int64_t J, int64_t nsel,
                 int64_t cblk, int64_t r0, int64_t Rout, hipStream_t s) {
    if (r0 < 0 || r0 >= R || Rout < 0 || Rout > R) {
        set_error("pruned FFT scatter: rows %lld + %lld of %lld", (long long)r0,
                  (long long)Rout, (long long)R);
        return JFA_ERR_BAD_ARG;
    }
    const int64_t ct = (C + kScatterCols - 1) / kScatterCols, rt = (Rout + kTile - 1) / kTile;
    const int64_t blocks = ct * rt * outer;
    if (blocks == 0) return JFA_OK;
    if (blocks > INT32_MAX) {
        set_error("pruned FFT transpose of %lld tiles is too large", (long long)blocks);
        return JFA_ERR_TOO_LARGE;
    }
    if (!fits_int({R, C, J, nsel, cblk, C + kScatterCols})) {
        set_error("pruned FFT transpose extents beyond 32-bit indexing");
        return JFA_ERR_TOO_LARGE;
    }
    scatter_cols_kernel<T><<<(unsigned)blocks, 256, 0, s>>>(B, A, (int)R, (int)C, (int)J,
                                                            (int)nsel, (int)cblk, (int)r0,
                                                            (int)Rout, (int)ct, (int)rt);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

namespace {

// complex elements per transform of the separate compact buffer: G (2D) or
// G1 (3D)
int64_t fwt_cells(jfa_plan p) {
    const int64_t *n = p->nmodes, *nf = p->geom.nf;
    return p->dim == 2 ? n[0] * nf[1] : n[0] * nf[1] * nf[2];
}

}  // namespace

bool fft_is_pruned(jfa_plan p) { return p->dim >= 2; }

int reserve_fwt(jfa_plan p) {
    const size_t bytes = (size_t)p->batch * fwt_cells(p) * 2 * (p->is_double ? 8 : 4);
    if (bytes <= p->fwt_bytes) return JFA_OK;
    if (p->d_fwt) (void)hipFree(p->d_fwt);
    p->d_fwt = nullptr;
    p->fwt_bytes = 0;
    hipError_t e = hipMalloc(&p->d_fwt, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        release_strip_scratch(p);  // idle by now
        e = hipMalloc(&p->d_fwt, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        p->d_fwt = nullptr;
        set_error("could not allocate %zu bytes for the pruned FFT", bytes);
        return JFA_ERR_ALLOC;
    }
    p->fwt_bytes = bytes;
    return JFA_OK;
}

// The compact mode buffer the deconvolution reads / the amplification writes.
template <typename T>
static T *compact_modes(jfa_plan p, T *fw) {
    return p->dim == 2 ? (T *)p->d_fwt : fw;
}

template <typename T>
int pruned_grid_fft(jfa_plan p, T *fw, int nb) {
    if (int rc = reserve_fwt(p)) return rc;
    const int64_t *n = p->nmodes, *nf = p->geom.nf;
    T *G = (T *)p->d_fwt;
    if (int rc = fft1d(p, fw, nf[0], (int64_t)nb * nf[1] * nf[2])) return rc;
    if (p->dim == 2) {
        if (int rc = gather_cols<T>(fw, G, nb, nf[1], nf[0], n[0], n[0], nf[0], p->stream))
            return rc;
        return fft1d(p, G, nf[1], (int64_t)nb * n[0]);
    }
    // 3D: G1[t][z][j0][y], then G2[t][j0][j1][z] in fw
    if (int rc = gather_cols<T>(fw, G, (int64_t)nb * nf[2], nf[1], nf[0], n[0], n[0], nf[0],
                                p->stream))
        return rc;
    if (int rc = fft1d(p, G, nf[1], (int64_t)nb * nf[2] * n[0])) return rc;
    if (int rc = gather_cols<T>(G, fw, nb, nf[2], n[0] * nf[1], n[0] * n[1], n[1], nf[1],
                                p->stream))
        return rc;
    return fft1d(p, fw, nf[2], (int64_t)nb * n[0] * n[1]);
}

// Type 2 (modes -> fine grid).  With kept-row windows (GridGeom::wstart,
// type-3 inner plans) only the kept z planes go through the y pass and only the
// kept (y, z) rows through the x pass; the grid is stored as those rows.
template <typename T>
int pruned_modes_fft(jfa_plan p, T *fw, int nb) {
    if (int rc = reserve_fwt(p)) return rc;
    const GridGeom &g = p->geom;
    const int64_t *n = p->nmodes, *nf = g.nf;
    const int64_t ry = window_rows(g, 1), y0 = g.wlen[1] ? g.wstart[1] : 0;
    T *G = (T *)p->d_fwt;
    if (p->dim == 2) {
        if (int rc = fft1d(p, G, nf[1], (int64_t)nb * n[0])) return rc;
        if (int rc = scatter_cols<T>(G, fw, nb, nf[1], nf[0], n[0], n[0], nf[0], y0, ry,
                                     p->stream))
            return rc;
        return fft1d(p, fw, nf[0], (int64_t)nb * ry);
    }
    // 3D: G2 (in fw) -> G1 -> fw
    const int64_t rz = window_rows(g, 2), z0 = g.wlen[2] ? g.wstart[2] : 0;
    if (int rc = fft1d(p, fw, nf[2], (int64_t)nb * n[0] * n[1])) return rc;
    if (int rc = scatter_cols<T>(fw, G, nb, nf[2], n[0] * nf[1], n[0] * n[1], n[1], nf[1], z0,
                                 rz, p->stream))
        return rc;
    if (int rc = fft1d(p, G, nf[1], (int64_t)nb * rz * n[0])) return rc;
    if (int rc = scatter_cols<T>(G, fw, (int64_t)nb * rz, nf[1], nf[0], n[0], n[0], nf[0], y0,
                                 ry, p->stream))
        return rc;
    return fft1d(p, fw, nf[0], (int64_t)nb * ry * rz);
}

// Shape of the compact buffer and the tiling of the deconvolution /
// amplification kernels; g_stride = complex elements per transform.
static PrunedShape pruned_shape(jfa_plan p, bool over_fine_last, int64_t *g_stride) {
    const int64_t *n = p->nmodes, *nf = p->geom.nf;
    PrunedShape sh;
    sh.n0 = n[0];
    sh.nm = p->dim == 3 ? n[1] : 1;
    sh.nl = p->dim == 3 ? n[2] : n[1];
    sh.nfl = p->dim == 3 ? nf[2] : nf[1];
    sh.nmid = sh.nm;
    sh.t0 = (sh.n0 + kTile - 1) / kTile;
    sh.tl = ((over_fine_last ? sh.nfl : sh.nl) + kTile - 1) / kTile;
    *g_stride = sh.n0 * sh.nm * sh.nfl;
    return sh;
}

template <typename T>
int pruned_deconv(jfa_plan p, T *fw, T *fk, int nb) {
    int64_t gs;
    const PrunedShape sh = pruned_shape(p, false, &gs);
    const int64_t blocks = sh.t0 * sh.tl * sh.nmid * nb;
    if (blocks == 0) return JFA_OK;
    const T *G = compact_modes<T>(p, fw);
    const T *dk[3] = {(const T *)p->d_dk[0], (const T *)p->d_dk[1], (const T *)p->d_dk[2]};
    const T *dkm = p->dim == 3 ? dk[1] : dk[0];
    const T *dkl = p->dim == 3 ? dk[2] : dk[1];
    deconv_pruned_kernel<T><<<(unsigned)blocks, 256, 0, p->stream>>>(
        sh, dk[0], dkm, dkl, p->opts.modeord, G, gs, fk, p->Ntot);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int pruned_amplify(jfa_plan p, const T *fk, T *fw, int nb) {
    if (int rc = reserve_fwt(p)) return rc;
    int64_t gs;
    const PrunedShape sh = pruned_shape(p, true, &gs);
    const int64_t blocks = sh.t0 * sh.tl * sh.nmid * nb;
    if (blocks == 0) return JFA_OK;
    T *G = compact_modes<T>(p, fw);
    const T *dk[3] = {(const T *)p->d_dk[0], (const T *)p->d_dk[1], (const T *)p->d_dk[2]};
    const T *dkm = p->dim == 3 ? dk[1] : dk[0];
    const T *dkl = p->dim == 3 ? dk[2] : dk[1];
    amplify_pruned_kernel<T><<<(unsigned)blocks, 256, 0, p->stream>>>(
        sh, dk[0], dkm, dkl, p->opts.modeord, fk, p->Ntot, G, gs);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

// 2D deconvolution from a compact buffer G[j0][y] (n0 x nf1, one transform)
// without a plan: the allocation-free entry point's last step.
template <typename T>
int launch_deconv_pruned_2d(int64_t n0, int64_t n1, int64_t nf1, const T *dk0, const T *dk1,
                            int modeord, const T *G, T *out, hipStream_t stream) {
    PrunedShape sh;
    sh.n0 = n0;
    sh.nm = 1;
    sh.nl = n1;
    sh.nfl = nf1;
    sh.nmid = 1;
    sh.t0 = (n0 + kTile - 1) / kTile;
    sh.tl = (n1 + kTile - 1) / kTile;
    const int64_t blocks = sh.t0 * sh.tl;
    if (blocks == 0) return JFA_OK;
    deconv_pruned_kernel<T><<<(unsigned)blocks, 256, 0, stream>>>(
        sh, dk0, dk0, dk1, modeord, G, n0 * nf1, out, n0 * n1);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

#define JFA_INST(T)                                                 \
    template int launch_deconv_pruned_2d<T>(int64_t, int64_t, int64_t, const T *, const T *, \
                                            int, const T *, T *, hipStream_t);              \
    template int gather_cols<T>(const T *, T *, int64_t, int64_t, int64_t, int64_t, int64_t, \
                                int64_t, hipStream_t);                                      \
    template int scatter_cols<T>(const T *, T *, int64_t, int64_t, int64_t, int64_t, int64_t, \
                                 int64_t, int64_t, int64_t, hipStream_t);                    \
    template int pruned_grid_fft<T>(jfa_plan, T *, int);            \
    template int pruned_modes_fft<T>(jfa_plan, T *, int);           \
    template int pruned_deconv<T>(jfa_plan, T *, T *, int);         \
    template int pruned_amplify<T>(jfa_plan, const T *, T *, int);
JFA_INST(float)
JFA_INST(double)
#undef JFA_INST

}  // namespace jfa
