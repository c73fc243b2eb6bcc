// setpts: fold points onto the fine grid, bin them and sort them by bin.
// Replaces the point sort cuFINUFFT runs inside setpts (called at
// lib/kernels.cc.cu:63-68; device code absent from the reference).
//
//   1. keys:   key[j] = bin of point j (from its first tap)
//   2. sort:   stable radix sort of (key, j) pairs over the bits the bin count
//              needs (radix.hip; no data-dependent order or cost, so clustered
//              inputs cost the same)
//   3. bounds: bin_start[b] = first sorted position with key >= b (binary
//              search per bin), and for the LDS method the subproblem prefix
//   4. gather: for sorted position p, j = idx[p]: write the point's wrapped
//              first tap and Horner variable per dimension at p (coalesced
//              writes; the coordinates are read by index)
//
// The 2D strip spreader skips the gather: its key also carries the first tap's
// column within the strip (low kStripKeyShift bits), which with the bin gives
// both first taps, and the keys kernel writes the Horner variables in input
// order, where the spreader reads them by original index.
//
// The bin of a point and the tap window the spreader uses both come from
// fold_point() on the coordinate in double, so they agree exactly.
#include <algorithm>

#include "jfa_device.hpp"

namespace jfa {

namespace {

// Sort key of a point at (xj, yj, zj): its bin.
template <typename T, int DIM>
__device__ __forceinline__ unsigned key_of_values(const GridGeom &g, T xj, T yj, T zj) {
    Folded f0 = fold_point((double)xj, g.nf[0], g.scale[0], g.shift[0], g.ns);
    int64_t b = f0.l0w / g.bs[0];
    if constexpr (DIM > 1) {
        Folded f1 = fold_point((double)yj, g.nf[1], g.scale[1], g.shift[1], g.ns);
        if (DIM == 2 && g.ymajor)
            b = b * g.nb[1] + f1.l0w / g.bs[1];
        else
            b += (int64_t)(f1.l0w / g.bs[1]) * g.nb[0];
    }
    if constexpr (DIM > 2) {
        Folded f2 = fold_point((double)zj, g.nf[2], g.scale[2], g.shift[2], g.ns);
        b += (int64_t)(f2.l0w / g.bs[2]) * g.nb[0] * g.nb[1];
    }
    return (unsigned)b;
}
// Sort key of point j.
template <typename T, int DIM>
__device__ __forceinline__ unsigned key_of_point(const GridGeom &g, const T *x, const T *y,
                                                 const T *z, int64_t j) {
    return key_of_values<T, DIM>(g, x[j], DIM > 1 ? y[j] : T(0), DIM > 2 ? z[j] : T(0));
}

// Strip key of 2D point j: ((bin_off + s*nf1 + l0y) << kStripKeyShift) | X
// with s = l0x / SW and X = l0x - s*SW, and its Horner variables.
template <typename T>
__device__ __forceinline__ unsigned strip_key_of(const GridGeom &g, int64_t bin_off, T xj, T yj,
                                                 T &tx, T &ty) {
    const Folded f0 = fold_point((double)xj, g.nf[0], g.scale[0], g.shift[0], g.ns);
    const Folded f1 = fold_point((double)yj, g.nf[1], g.scale[1], g.shift[1], g.ns);
    const int s = f0.l0w / g.bs[0];
    const int X = f0.l0w - s * g.bs[0];
    tx = (T)f0.t;
    ty = (T)f1.t;
    const int64_t b = bin_off + (int64_t)s * g.nb[1] + f1.l0w;
    return (unsigned)((b << kStripKeyShift) | X);
}
template <typename T>
__device__ __forceinline__ unsigned strip_key(const GridGeom &g, int64_t bin_off, const T *x,
                                              const T *y, int64_t j, T &tx, T &ty) {
    return strip_key_of<T>(g, bin_off, x[j], y[j], tx, ty);
}

// 3D slices: the ns slice points of point j, keys ((z * S + s) * nf1 + l0y) << 6
// | X for slices z = l0z + dz (mod nf2), values j * ns + dz; rec3 = (tx, ty, tz).
template <typename T>
__global__ void __launch_bounds__(256)
    slice_keys_kernel(GridGeom g, int S, int64_t M, const T *__restrict__ x,
                      const T *__restrict__ y, const T *__restrict__ z, unsigned *key,
                      T *rec3) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= M) return;
    const Folded f0 = fold_point((double)x[j], g.nf[0], g.scale[0], g.shift[0], g.ns);
    const Folded f1 = fold_point((double)y[j], g.nf[1], g.scale[1], g.shift[1], g.ns);
    const Folded f2 = fold_point((double)z[j], g.nf[2], g.scale[2], g.shift[2], g.ns);
    const int s = f0.l0w / g.bs[0];
    const int X = f0.l0w - s * g.bs[0];
    rec3[3 * j] = (T)f0.t;
    rec3[3 * j + 1] = (T)f1.t;
    rec3[3 * j + 2] = (T)f2.t;
    const int nf2 = (int)g.nf[2];
    for (int dz = 0; dz < g.ns; ++dz) {
        int zz = f2.l0w + dz;
        if (zz >= nf2) zz -= nf2;
        const int64_t b = ((int64_t)zz * S + s) * g.nf[1] + f1.l0w;
        key[j * g.ns + dz] = (unsigned)((b << kStripKeyShift) | X);
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
    strip_keys_kernel(GridGeom g, int64_t M, const T *__restrict__ x, const T *__restrict__ y,
                      unsigned *key, T *rec) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= M) return;
    T tx, ty;
    key[j] = strip_key<T>(g, 0, x, y, j, tx, ty);
    rec[2 * j] = tx;
    rec[2 * j + 1] = ty;
}

// The same for FP32 points four at a time, when x and y are 16-byte aligned:
// 16-byte loads of x and y, one 16-byte store of the keys and two of the
// Horner pairs per thread.
__global__ void __launch_bounds__(256)
    strip_keys4_kernel(GridGeom g, int64_t M, const float *__restrict__ x,
                       const float *__restrict__ y, unsigned *key, float *rec) {
    const int64_t j0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (j0 >= M) return;
    if (j0 + 4 > M) {
        for (int64_t j = j0; j < M; ++j) {
            float tx, ty;
            key[j] = strip_key<float>(g, 0, x, y, j, tx, ty);
            rec[2 * j] = tx;
            rec[2 * j + 1] = ty;
        }
        return;
    }
    const float4 xv = *reinterpret_cast<const float4 *>(x + j0);
    const float4 yv = *reinterpret_cast<const float4 *>(y + j0);
    float4 r0, r1;
    uint4 k;
    k.x = strip_key_of<float>(g, 0, xv.x, yv.x, r0.x, r0.y);
    k.y = strip_key_of<float>(g, 0, xv.y, yv.y, r0.z, r0.w);
    k.z = strip_key_of<float>(g, 0, xv.z, yv.z, r1.x, r1.y);
    k.w = strip_key_of<float>(g, 0, xv.w, yv.w, r1.z, r1.w);
    *reinterpret_cast<uint4 *>(key + j0) = k;
    *reinterpret_cast<float4 *>(rec + 2 * j0) = r0;
    *reinterpret_cast<float4 *>(rec + 2 * j0 + 4) = r1;
}

// Key with the offset bits, and the Horner variables, of a point at
// coordinates v[0 .. DIM).
template <typename T, int DIM>
__device__ __forceinline__ unsigned keyed_key(const GridGeom &g, const T *v, T *t) {
    int64_t b = 0, stride = 1;
    unsigned off = 0;
    int sh = 0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const Folded f = fold_point((double)v[d], g.nf[d], g.scale[d], g.shift[d], g.ns);
        const int bd = f.l0w >> g.subw[d];
        b += bd * stride;
        stride *= g.nb[d];
        off |= (unsigned)(f.l0w - (bd << g.subw[d])) << sh;
        sh += g.subw[d];
        t[d] = (T)f.t;
    }
    return (unsigned)((b << g.keyshift) | off);
}

// Key with the offset bits, and the Horner variables, of point j.
template <typename T, int DIM>
__global__ void __launch_bounds__(256)
    bin_keys_rec_kernel(GridGeom g, int64_t M, const T *__restrict__ x, const T *__restrict__ y,
                        const T *__restrict__ z, unsigned *key, T *rec) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= M) return;
    const T *xs[3] = {x, y, z};
    T v[DIM], t[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) v[d] = xs[d][j];
    key[j] = keyed_key<T, DIM>(g, v, t);
#pragma unroll
    for (int d = 0; d < DIM; ++d) rec[j * DIM + d] = t[d];
}

// The same for 16-byte aligned FP32 coordinates, four points per thread: one
// 16-byte load per axis, one 16-byte store of the keys and DIM of the Horner
// variables.
template <int DIM>
__global__ void __launch_bounds__(256)
    bin_keys_rec4_kernel(GridGeom g, int64_t M, const float *__restrict__ x,
                         const float *__restrict__ y, const float *__restrict__ z, unsigned *key,
                         float *rec) {
    const int64_t j0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (j0 >= M) return;
    const float *xs[3] = {x, y, z};
    if (j0 + 4 > M) {
        for (int64_t j = j0; j < M; ++j) {
            float v[DIM], t[DIM];
            for (int d = 0; d < DIM; ++d) v[d] = xs[d][j];
            key[j] = keyed_key<float, DIM>(g, v, t);
            for (int d = 0; d < DIM; ++d) rec[j * DIM + d] = t[d];
        }
        return;
    }
    float4 c[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) c[d] = *reinterpret_cast<const float4 *>(xs[d] + j0);
    float t[4 * DIM];
    uint4 k;
    {
        float v[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) v[d] = c[d].x;
        k.x = keyed_key<float, DIM>(g, v, t);
#pragma unroll
        for (int d = 0; d < DIM; ++d) v[d] = c[d].y;
        k.y = keyed_key<float, DIM>(g, v, t + DIM);
#pragma unroll
        for (int d = 0; d < DIM; ++d) v[d] = c[d].z;
        k.z = keyed_key<float, DIM>(g, v, t + 2 * DIM);
#pragma unroll
        for (int d = 0; d < DIM; ++d) v[d] = c[d].w;
        k.w = keyed_key<float, DIM>(g, v, t + 3 * DIM);
    }
    *reinterpret_cast<uint4 *>(key + j0) = k;
    float4 *r = reinterpret_cast<float4 *>(rec + j0 * DIM);
#pragma unroll
    for (int q = 0; q < DIM; ++q) r[q] = float4{t[4 * q], t[4 * q + 1], t[4 * q + 2], t[4 * q + 3]};
}

template <typename T, int DIM>
__global__ void __launch_bounds__(256)
    bin_keys_kernel(GridGeom g, int64_t M, const T *__restrict__ x, const T *__restrict__ y,
                    const T *__restrict__ z, unsigned *key) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= M) return;
    key[j] = key_of_point<T, DIM>(g, x, y, z, j);
}

// The same for 16-byte aligned FP32 coordinates, four points per thread (one
// 16-byte load per axis and one 16-byte store of the keys: more reads in
// flight and fewer memory instructions per point).
template <int DIM>
__global__ void __launch_bounds__(256)
    bin_keys4_kernel(GridGeom g, int64_t M, const float *__restrict__ x,
                     const float *__restrict__ y, const float *__restrict__ z, unsigned *key) {
    const int64_t j0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (j0 >= M) return;
    if (j0 + 4 > M) {
        for (int64_t j = j0; j < M; ++j) key[j] = key_of_point<float, DIM>(g, x, y, z, j);
        return;
    }
    const float4 xv = *reinterpret_cast<const float4 *>(x + j0);
    float4 yv{0, 0, 0, 0}, zv{0, 0, 0, 0};
    if constexpr (DIM > 1) yv = *reinterpret_cast<const float4 *>(y + j0);
    if constexpr (DIM > 2) zv = *reinterpret_cast<const float4 *>(z + j0);
    uint4 k;
    k.x = key_of_values<float, DIM>(g, xv.x, yv.x, zv.x);
    k.y = key_of_values<float, DIM>(g, xv.y, yv.y, zv.y);
    k.z = key_of_values<float, DIM>(g, xv.z, yv.z, zv.z);
    k.w = key_of_values<float, DIM>(g, xv.w, yv.w, zv.w);
    *reinterpret_cast<uint4 *>(key + j0) = k;
}

// 16-byte aligned (x, y, z), key and rec: the four-points-per-thread kernels
// apply.
template <typename T>
bool aligned4(int dim, const T *x, const T *y, const T *z, const void *a, const void *b) {
    const uintptr_t m = (uintptr_t)x | (dim > 1 ? (uintptr_t)y : 0) | (dim > 2 ? (uintptr_t)z : 0) |
                        (uintptr_t)a | (uintptr_t)b;
    return sizeof(T) == 4 && m % 16 == 0;
}

// bin_start[b] = first p with skey[p] >= b << shift, for b in [0, nbins]
__global__ void __launch_bounds__(256)
    bin_bounds_kernel(int64_t M, int64_t nbins, int shift, const unsigned *__restrict__ skey,
                      int *bin_start) {
    const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (b > nbins) return;
    const int64_t kb = b << shift;
    int64_t lo = 0, hi = M;  // answer in [lo, hi]
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)skey[mid] < kb)
            lo = mid + 1;
        else
            hi = mid;
    }
    bin_start[b] = (int)lo;
}

// Exclusive prefix of the subproblems per bin (ceil(count / maxsub)) in three
// launches: per-bin counts with 256-bin block sums, a one-workgroup scan of
// the block sums, then the block-local scans.  Total at sub_start[nbins] and
// *nsub.  blk holds 2 * ceil(nbins / 256) + 1 ints.
__device__ __forceinline__ int block_excl_scan256(int v, int *total) {
    __shared__ int sa[256];
    const int tid = threadIdx.x;
    sa[tid] = v;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const int w = tid >= off ? sa[tid - off] : 0;
        __syncthreads();
        sa[tid] += w;
        __syncthreads();
    }
    *total = sa[255];
    const int e = sa[tid] - v;
    __syncthreads();
    return e;
}

__global__ void __launch_bounds__(256)
    sub_count_kernel(int64_t nbins, const int *__restrict__ bin_start, int maxsub, int *sub_start,
                     int *blk) {
    const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int c = 0;
    if (b < nbins) {
        const int cnt = bin_start[b + 1] - bin_start[b];
        c = (cnt + maxsub - 1) / maxsub;
        sub_start[b] = c;
    }
    int total;
    block_excl_scan256(c, &total);
    if (threadIdx.x == 0) blk[blockIdx.x] = total;
}

// one workgroup: blk[nblk ..] = exclusive scan of blk[0, nblk)
__global__ void __launch_bounds__(1024)
    sub_blocks_kernel(int64_t nbins, int nblk, int *blk, int *sub_start, int *nsub) {
    __shared__ int sa[1024];
    const int tid = threadIdx.x;
    const int per = (nblk + 1023) / 1024;
    const int lo = min(tid * per, nblk), hi = min(lo + per, nblk);
    int a = 0;
    for (int i = lo; i < hi; ++i) a += blk[i];
    sa[tid] = a;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int v = tid >= off ? sa[tid - off] : 0;
        __syncthreads();
        sa[tid] += v;
        __syncthreads();
    }
    int e = sa[tid] - a;
    int *off = blk + nblk;
    for (int i = lo; i < hi; ++i) {
        const int c = blk[i];
        off[i] = e;
        e += c;
    }
    if (tid == 1023) {
        off[nblk] = sa[1023];
        sub_start[nbins] = sa[1023];
        *nsub = sa[1023];
    }
}

__global__ void __launch_bounds__(256)
    sub_apply_kernel(int64_t nbins, int nblk, const int *__restrict__ blk, int *sub_start) {
    const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int c = b < nbins ? sub_start[b] : 0;
    int total;
    const int e = block_excl_scan256(c, &total);
    if (b < nbins) sub_start[b] = blk[nblk + blockIdx.x] + e;
}

// The subproblem prefix in one workgroup for at most kSmallBins bins (one
// launch instead of three): sub_start = exclusive prefix of ceil(count /
// maxsub) over the bins, with the total at sub_start[nbins] and *nsub.
constexpr int kSmallBins = 4095;
__global__ void __launch_bounds__(1024)
    subs_small_kernel(int nbins, const int *__restrict__ bin_start, int maxsub, int *sub_start,
                      int *nsub) {
    __shared__ int bs[kSmallBins + 1];
    __shared__ int sa[1024];
    const int tid = threadIdx.x;
    for (int b = tid; b <= nbins; b += 1024) bs[b] = bin_start[b];
    __syncthreads();
    const int per = (nbins + 1023) / 1024;
    const int b0 = min(tid * per, nbins), b1 = min(b0 + per, nbins);
    int a = 0;
    for (int b = b0; b < b1; ++b) a += (bs[b + 1] - bs[b] + maxsub - 1) / maxsub;
    sa[tid] = a;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int v = tid >= off ? sa[tid - off] : 0;
        __syncthreads();
        sa[tid] += v;
        __syncthreads();
    }
    int e = sa[tid] - a;
    for (int b = b0; b < b1; ++b) {
        sub_start[b] = e;
        e += (bs[b + 1] - bs[b] + maxsub - 1) / maxsub;
    }
    if (tid == 1023) {
        sub_start[nbins] = sa[1023];
        *nsub = sa[1023];
    }
}

// Sorted position p holds point j = idx[p] (written by the sort): store its
// wrapped first tap and Horner variable per dimension at p.
template <typename T, int DIM>
__global__ void __launch_bounds__(256)
    gather_points_kernel(GridGeom g, int64_t M, const T *__restrict__ x, const T *__restrict__ y,
                         const T *__restrict__ z, const int *__restrict__ idx, int *l0, T *tv) {
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= M) return;
    const int64_t j = idx[p];
    const T *xs[3] = {x, y, z};
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        Folded f = fold_point((double)xs[d][j], g.nf[d], g.scale[d], g.shift[d], g.ns);
        l0[d * M + p] = f.l0w;
        tv[d * M + p] = (T)f.t;
    }
}

// Unsorted variant (global-memory method with gpu_sort = 0): input order.
template <typename T, int DIM>
__global__ void __launch_bounds__(256)
    fold_points_kernel(GridGeom g, int64_t M, const T *__restrict__ x, const T *__restrict__ y,
                       const T *__restrict__ z, int *idx, int *l0, T *tv) {
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= M) return;
    idx[p] = (int)p;
    const T *xs[3] = {x, y, z};
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        Folded f = fold_point((double)xs[d][p], g.nf[d], g.scale[d], g.shift[d], g.ns);
        l0[d * M + p] = f.l0w;
        tv[d * M + p] = (T)f.t;
    }
}

// ---------------------------------------------------------------- ragged batch
// Global point P belongs to problem i with moff[i] <= P < moff[i+1]; its
// coordinates are x_i[P - moff[i]], y_i[...] from the pointer table.  Keys are
// offset by the problem's first global bin, so one sort orders every problem.

__device__ __forceinline__ int problem_of(const int64_t *__restrict__ moff, int nprob, int64_t P) {
    int lo = 0, hi = nprob;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (moff[mid] <= P)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// kRaggedKeysPer points per thread (strided by the workgroup size), so that the
// problem lookup is paid once per thread rather than once per point
constexpr int kRaggedKeysPer = 8;

template <typename T>
__global__ void __launch_bounds__(256)
    ragged_keys_kernel(const RaggedProb *__restrict__ probs, const int64_t *__restrict__ moff,
                       int nprob, const void *const *__restrict__ ptrs, int64_t mtot,
                       unsigned *key, T *rec) {
    const int64_t Pb = (int64_t)blockIdx.x * 256 * kRaggedKeysPer;
    const int64_t P0 = Pb + threadIdx.x;
    // most workgroups lie inside one problem: then the geometry is uniform
    // (scalar loads) and the points independent
    const int64_t Pe = min(Pb + 256 * kRaggedKeysPer, mtot) - 1;
    const int ib = problem_of(moff, nprob, Pb);
    if (Pe < moff[ib + 1]) {
        const RaggedProb &pr = probs[ib];
        const T *x = (const T *)ptrs[ib], *y = (const T *)ptrs[nprob + ib];
#pragma unroll
        for (int r = 0; r < kRaggedKeysPer; ++r) {
            const int64_t P = P0 + (int64_t)r * 256;
            if (P > Pe) break;
            T tx, ty;
            key[P] = strip_key<T>(pr.g, pr.bin_off, x, y, P - pr.moff, tx, ty);
            rec[2 * P] = tx;
            rec[2 * P + 1] = ty;
        }
        return;
    }
    if (P0 >= mtot) return;
    int i = problem_of(moff, nprob, P0);
    for (int r = 0; r < kRaggedKeysPer; ++r) {
        const int64_t P = P0 + (int64_t)r * 256;
        if (P >= mtot) break;
        while (P >= moff[i + 1]) ++i;  // points ascend: the next problems
        const RaggedProb &pr = probs[i];
        T tx, ty;
        key[P] = strip_key<T>(pr.g, pr.bin_off, (const T *)ptrs[i], (const T *)ptrs[nprob + i],
                              P - pr.moff, tx, ty);
        rec[2 * P] = tx;
        rec[2 * P + 1] = ty;
    }
}

__global__ void fill_zero_kernel(uint4 *p, int64_t n16, unsigned char *tail, int ntail) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n16; i += stride) p[i] = make_uint4(0, 0, 0, 0);
    if (blockIdx.x == 0 && (int)threadIdx.x < ntail) tail[threadIdx.x] = 0;
}

int key_bits(int64_t nbins) {
    int bits = 1;
    while (bits < 32 && ((int64_t)1 << bits) < nbins) ++bits;
    return bits;
}

}  // namespace

int launch_fill_zero(void *p, int64_t bytes, hipStream_t stream) {
    if (bytes <= 0) return JFA_OK;
    if (((uintptr_t)p & 15) != 0) {
        set_error("fill_zero: pointer not 16-byte aligned");
        return JFA_ERR_BAD_ARG;
    }
    int64_t n16 = bytes / 16;
    int ntail = (int)(bytes - n16 * 16);
    int64_t blocks = (n16 + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    if (blocks < 1) blocks = 1;
    fill_zero_kernel<<<dim3((unsigned)blocks), dim3(256), 0, stream>>>(
        (uint4 *)p, n16, (unsigned char *)p + n16 * 16, ntail);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

// bin_start from the sorted keys (unless the sort wrote it) and, with sub_start, the subproblem prefix
// (block sums of the large form live after the nbins + 1 prefix entries).
static int bins_and_subproblems(const GridGeom &g, int64_t M, const unsigned *skey, int *bin_start,
                         bool bounded, int *sub_start, int *nsub, int maxsub,
                         hipStream_t stream) {
    if (!bounded) {
        const unsigned blocks = (unsigned)((g.nbins + 1 + 255) / 256);
        bin_bounds_kernel<<<blocks, 256, 0, stream>>>(M, g.nbins, g.keyshift, skey, bin_start);
        JFA_HIP_CHECK(hipGetLastError());
    }
    if (sub_start && g.nbins <= kSmallBins) {
        subs_small_kernel<<<1, 1024, 0, stream>>>((int)g.nbins, bin_start, maxsub, sub_start,
                                                  nsub);
        JFA_HIP_CHECK(hipGetLastError());
    } else if (sub_start) {
        const int nblk = (int)((g.nbins + 255) / 256);
        int *blk = sub_start + g.nbins + 1;
        sub_count_kernel<<<nblk, 256, 0, stream>>>(g.nbins, bin_start, maxsub, sub_start, blk);
        sub_blocks_kernel<<<1, 1024, 0, stream>>>(g.nbins, nblk, blk, sub_start, nsub);
        sub_apply_kernel<<<nblk, 256, 0, stream>>>(g.nbins, nblk, blk, sub_start);
        JFA_HIP_CHECK(hipGetLastError());
    }
    return JFA_OK;
}

template <typename T>
int launch_sort_points(const GridGeom &g, int64_t M, const T *x, const T *y, const T *z,
                       const SortScratch &s, int *bin_start, int *sub_start, int *nsub,
                       int maxsub, int *idx, int *l0, T *tv, hipStream_t stream) {
    bool bounded = false;
    if (M > 0) {
        if (aligned4<T>(g.dim, x, y, z, s.key_in, s.key_in)) {
            const unsigned blocks = (unsigned)((M + 1023) / 1024);
            JFA_DISPATCH_DIM(g.dim, bin_keys4_kernel<DIM_><<<blocks, 256, 0, stream>>>(
                                        g, M, (const float *)x, (const float *)y,
                                        (const float *)z, s.key_in));
        } else {
            const unsigned blocks = (unsigned)((M + 255) / 256);
            JFA_DISPATCH_DIM(g.dim, bin_keys_kernel<T, DIM_><<<blocks, 256, 0, stream>>>(
                                        g, M, x, y, z, s.key_in));
        }
        JFA_HIP_CHECK(hipGetLastError());
        if (int rc = radix_sort(s.temp, s.key_in, s.key_out, (unsigned *)idx, M, 0,
                                key_bits(g.nbins) + g.keyshift, g.nbins, g.keyshift, bin_start,
                                &bounded, stream))
            return rc;
    }
    if (int rc = bins_and_subproblems(g, M, s.key_out, bin_start, bounded, sub_start, nsub,
                                      maxsub, stream))
        return rc;
    if (M > 0) {
        const unsigned blocks = (unsigned)((M + 255) / 256);
        JFA_DISPATCH_DIM(g.dim, gather_points_kernel<T, DIM_><<<blocks, 256, 0, stream>>>(
                                    g, M, x, y, z, idx, l0, tv));
        JFA_HIP_CHECK(hipGetLastError());
    }
    return JFA_OK;
}

template <typename T>
int launch_sort_points_keyed(const GridGeom &g, int64_t M, const T *x, const T *y, const T *z,
                             const SortScratch &s, int *bin_start, int *sub_start, int *nsub,
                             int maxsub, int *idx, T *rec, hipStream_t stream) {
    bool bounded = false;
    if (M > 0) {
        if (aligned4<T>(g.dim, x, y, z, s.key_in, rec)) {
            const unsigned blocks = (unsigned)((M + 1023) / 1024);
            JFA_DISPATCH_DIM(g.dim, bin_keys_rec4_kernel<DIM_><<<blocks, 256, 0, stream>>>(
                                        g, M, (const float *)x, (const float *)y,
                                        (const float *)z, s.key_in, (float *)rec));
        } else {
            const unsigned blocks = (unsigned)((M + 255) / 256);
            JFA_DISPATCH_DIM(g.dim, bin_keys_rec_kernel<T, DIM_><<<blocks, 256, 0, stream>>>(
                                        g, M, x, y, z, s.key_in, rec));
        }
        JFA_HIP_CHECK(hipGetLastError());
        // only the bin bits are sorted; the offset bits ride along
        if (int rc = radix_sort(s.temp, s.key_in, s.key_out, (unsigned *)idx, M, g.keyshift,
                                g.keyshift + key_bits(g.nbins), g.nbins, g.keyshift, bin_start,
                                &bounded, stream))
            return rc;
    }
    if (int rc = bins_and_subproblems(g, M, s.key_out, bin_start, bounded, sub_start, nsub,
                                      maxsub, stream))
        return rc;
    return JFA_OK;
}

template <typename T>
int launch_fold_points(const GridGeom &g, int64_t M, const T *x, const T *y, const T *z,
                       int *idx, int *l0, T *tv, hipStream_t stream) {
    if (M == 0) return JFA_OK;
    const unsigned blocks = (unsigned)((M + 255) / 256);
    JFA_DISPATCH_DIM(g.dim, fold_points_kernel<T, DIM_><<<blocks, 256, 0, stream>>>(
                                g, M, x, y, z, idx, l0, tv));
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

// Shared tail of the strip sorts: radix sort of (key, index) by (strip, row), and
// bin bounds.
int strip_sort_bits(int64_t nbins) { return key_bits(nbins) + kStripKeyShift - kStripSortLowBit; }

int sort_strip_keys(int64_t M, int64_t nbins, const SortScratch &s, int *bin_start, int *idx,
                    hipStream_t stream) {
    bool bounded = false;
    if (M > 0)
        if (int rc = radix_sort(s.temp, s.key_in, s.key_out, (unsigned *)idx, M,
                                kStripSortLowBit, key_bits(nbins) + kStripKeyShift, nbins,
                                kStripKeyShift, bin_start, &bounded, stream))
            return rc;
    if (bounded) return JFA_OK;
    const unsigned blocks = (unsigned)((nbins + 1 + 255) / 256);
    bin_bounds_kernel<<<blocks, 256, 0, stream>>>(M, nbins, kStripKeyShift, s.key_out,
                                                  bin_start);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int launch_sort_points_strip(const GridGeom &g, int64_t M, const T *x, const T *y,
                             const SortScratch &s, int *bin_start, int *idx, T *rec,
                             hipStream_t stream) {
    if (M > 0) {
        if (aligned4<T>(2, x, y, (const T *)nullptr, s.key_in, rec)) {
            const unsigned blocks = (unsigned)((M + 1023) / 1024);
            strip_keys4_kernel<<<blocks, 256, 0, stream>>>(g, M, (const float *)x,
                                                           (const float *)y, s.key_in,
                                                           (float *)rec);
        } else {
            const unsigned blocks = (unsigned)((M + 255) / 256);
            strip_keys_kernel<T><<<blocks, 256, 0, stream>>>(g, M, x, y, s.key_in, rec);
        }
        JFA_HIP_CHECK(hipGetLastError());
    }
    return sort_strip_keys(M, g.nbins, s, bin_start, idx, stream);
}

template <typename T>
int launch_sort_points_slices(const GridGeom &g, int S, int64_t M, const T *x, const T *y,
                              const T *z, const SortScratch &s, int *bin_start, int *idx,
                              T *rec3, hipStream_t stream) {
    if (M > 0) {
        const unsigned blocks = (unsigned)((M + 255) / 256);
        slice_keys_kernel<T><<<blocks, 256, 0, stream>>>(g, S, M, x, y, z, s.key_in,
                                                         rec3);
        JFA_HIP_CHECK(hipGetLastError());
    }
    return sort_strip_keys(M * g.ns, g.nbins, s, bin_start, idx, stream);
}

template <typename T>
int launch_ragged_sort(const RaggedLaunch &rl, const SortScratch &s, int *idx, T *rec,
                       hipStream_t stream) {
    const int64_t M = rl.mtot;
    if (M > 0) {
        const int64_t per = 256 * kRaggedKeysPer;
        const unsigned blocks = (unsigned)((M + per - 1) / per);
        ragged_keys_kernel<T><<<blocks, 256, 0, stream>>>(rl.probs, rl.moff, rl.nprob, rl.ptrs, M,
                                                          s.key_in, rec);
        JFA_HIP_CHECK(hipGetLastError());
    }
    return sort_strip_keys(M, rl.nbins, s, rl.bin_start, idx, stream);
}

#define JFA_INST(T)                                                                          \
    template int launch_ragged_sort<T>(const RaggedLaunch &, const SortScratch &, int *, T *, \
                                       hipStream_t);                                         \
    template int launch_sort_points_slices<T>(const GridGeom &, int, int64_t, const T *,      \
                                              const T *, const T *, const SortScratch &,      \
                                              int *, int *, T *, hipStream_t);                \
    template int launch_sort_points_strip<T>(const GridGeom &, int64_t, const T *, const T *, \
                                             const SortScratch &, int *, int *, T *,          \
                                             hipStream_t);                                    \
    template int launch_sort_points_keyed<T>(const GridGeom &, int64_t, const T *, const T *, \
                                             const T *, const SortScratch &, int *, int *,     \
                                             int *, int, int *, T *, hipStream_t);             \
    template int launch_sort_points<T>(const GridGeom &, int64_t, const T *, const T *,      \
                                       const T *, const SortScratch &, int *, int *, int *,  \
                                       int, int *, int *, T *, hipStream_t);                 \
    template int launch_fold_points<T>(const GridGeom &, int64_t, const T *, const T *,      \
                                       const T *, int *, int *, T *, hipStream_t);
JFA_INST(float)
JFA_INST(double)
#undef JFA_INST

}  // namespace jfa
