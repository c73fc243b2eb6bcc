// Stable radix sort of 32-bit keys with their positions: the point sort of
// setpts (the sort cuFINUFFT runs inside setpts, called at
// lib/kernels.cc.cu:63-68; source absent from the reference).
//
// radix_sort orders key[0 .. M) by its bits [b0, b1) and writes the ordered keys
// and, for each, its position in the input; equal keys keep input order.
//
// Least significant digit first, in as few passes of at most 11 bits as the
// span needs, three launches per pass:
//   count    per tile of consecutive keys, the digit histogram (LDS integer
//            atomics), one row of a tiles x digits table
//   scan     every column of the table, exclusive, and the column totals
//   scatter  per tile: stable ranks, reorder in LDS, write runs of equal digits
// A tile's waves rank their keys without atomics: the lanes holding equal
// digits find each other with one ballot per digit bit, and a counter per wave
// and digit carries the count from one 64-key step to the next, so the order
// is fixed.  A pass over 1e7 keys moves 40 MB (count) + 160 MB (scatter); the
// ranking is about 1.2 wave instructions per key.
//
// Up to kSmallSort keys: one workgroup runs every pass in LDS, one launch.
// There launches are the cost.  Against the rocPRIM sort used before (a merge
// sort of up to 20 launches below 2^20 keys, onesweep above), all launches of
// the sort: 2^20 keys, one pass 160 -> 19 us; 1e6 keys, two passes 157 -> 44 us;
// 300,007 keys 112 -> 33 us; 1e7 keys, one pass of 10 bits 128 -> 91 us; 1.5e7
// keys of 22 bits 335 -> 248 us; 4000 keys with their bin bounds 20 -> 11 us.
#include <algorithm>

#include "jfa_device.hpp"

namespace jfa {
namespace {

// Exclusive scan over the workgroup's threads (blockDim.x = 64 * waves) of v;
// s holds a value per wave.  Ends with a barrier.
template <int WAVES>
__device__ __forceinline__ unsigned block_exclusive(unsigned v, unsigned *s) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) s[wave] = x;
    __syncthreads();
    unsigned base = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
        if (w < wave) base += s[w];
    __syncthreads();
    return base + x - v;
}

// Ranks this wave's K x 64 digits (item i of a lane follows item i - 1 of every
// lane) by digit: rank[i] = earlier items of the wave with the same digit.
// cnt: the wave's 1 << BITS counters, zero on entry, its totals on return.
template <int BITS, int K>
__device__ __forceinline__ void wave_ranks(const unsigned (&digit)[K], const bool (&live)[K],
                                           unsigned *cnt, unsigned (&rank)[K]) {
#pragma unroll
    for (int i = 0; i < K; ++i) {
        uint64_t same = __ballot(live[i]);
#pragma unroll
        for (int b = 0; b < BITS; ++b) {
            const bool bit = (digit[i] >> b) & 1;
            const uint64_t ones = __ballot(bit);
            same &= bit ? ones : ~ones;
        }
        const unsigned before =
            __builtin_amdgcn_mbcnt_hi((unsigned)(same >> 32),
                                      __builtin_amdgcn_mbcnt_lo((unsigned)same, 0u));
        unsigned c = 0;
        if (live[i]) {
            c = cnt[digit[i]];
            if (before == 0) cnt[digit[i]] = c + (unsigned)__popcll(same);
        }
        rank[i] = c + before;
        // one step's counter writes before the next step's reads (a wave's LDS
        // accesses complete in order)
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
    }
}

// ------------------------------------------------------------- large inputs

// table[tile][digit]
template <int BITS, int THREADS, int K>
__global__ void __launch_bounds__(THREADS)
    radix_count_kernel(int64_t M, int shift, const unsigned *__restrict__ key, unsigned *table) {
    constexpr int D = 1 << BITS, TILE = THREADS * K;
    __shared__ unsigned cnt[D];
    for (int d = threadIdx.x; d < D; d += THREADS) cnt[d] = 0;
    __syncthreads();
    const int64_t p0 = (int64_t)blockIdx.x * TILE;
    unsigned k[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int64_t p = p0 + i * THREADS + threadIdx.x;
        k[i] = p < M ? key[p] : 0;
    }
#pragma unroll
    for (int i = 0; i < K; ++i)
    {
        // points that arrive in order (a trajectory) give runs of equal digits:
        // one add per run of lanes, or the lanes would queue on one counter
        const bool in = p0 + i * THREADS + threadIdx.x < M;
        const unsigned d = in ? (k[i] >> shift) & (D - 1) : D;
        const unsigned prev = __shfl_up(d, 1);
        const int lane = threadIdx.x & 63;
        const uint64_t heads = __ballot(lane == 0 || d != prev);
        if (in && ((heads >> lane) & 1)) {
            const uint64_t after = lane < 63 ? heads >> (lane + 1) : 0;
            atomicAdd(&cnt[d], after ? (unsigned)__builtin_ctzll(after) + 1 : 64u - lane);
        }
    }
    __syncthreads();
    for (int d = threadIdx.x; d < D; d += THREADS) table[(int64_t)blockIdx.x * D + d] = cnt[d];
}

// Column-wise exclusive scan of table[tiles][D] and the column totals.  A
// workgroup takes 16 columns (64 bytes of a row), its 64 quarter-waves equal
// runs of tiles.
constexpr int kScanCols = 16, kScanRuns = 64;
__global__ void __launch_bounds__(kScanCols *kScanRuns)
    radix_scan_kernel(int D, int tiles, unsigned *__restrict__ table, unsigned *__restrict__ total) {
    __shared__ unsigned part[kScanRuns][kScanCols];
    const int c = threadIdx.x % kScanCols, r = threadIdx.x / kScanCols;
    const int d = blockIdx.x * kScanCols + c;
    const int per = (tiles + kScanRuns - 1) / kScanRuns;
    const int t0 = min(r * per, tiles), t1 = min(t0 + per, tiles);
    unsigned sum = 0;
#pragma unroll 8
    for (int t = t0; t < t1; ++t) sum += table[(int64_t)t * D + d];
    part[r][c] = sum;
    __syncthreads();
    unsigned run = 0;
    for (int w = 0; w < r; ++w) run += part[w][c];
    if (r == kScanRuns - 1) total[d] = run + sum;
#pragma unroll 8
    for (int t = t0; t < t1; ++t) {
        const unsigned v = table[(int64_t)t * D + d];
        table[(int64_t)t * D + d] = run;
        run += v;
    }
}

template <int BITS, int THREADS, int K>
constexpr size_t scatter_lds() {
    // per-wave counters, then (aliased) the reordered pairs; offsets; wave sums
    const size_t cnt = (size_t)(THREADS / 64) * (1 << BITS) * 4, pairs = (size_t)THREADS * K * 8;
    return (cnt > pairs ? cnt : pairs) + (size_t)(1 << BITS) * 4 + 64 * 4;
}

// vin = NULL: the positions are 0, 1, ... (first pass)
template <int BITS, int THREADS, int K>
__global__ void __launch_bounds__(THREADS)
    radix_scatter_kernel(int64_t M, int shift, const unsigned *__restrict__ kin,
                         const unsigned *__restrict__ vin, const unsigned *__restrict__ table,
                         const unsigned *__restrict__ total, unsigned *__restrict__ kout,
                         unsigned *__restrict__ vout) {
    constexpr int D = 1 << BITS, TILE = THREADS * K, WAVES = THREADS / 64;
    constexpr int PER = (D + THREADS - 1) / THREADS;  // digits per thread
    extern __shared__ __align__(16) unsigned char radix_smem[];
    constexpr size_t kFront = scatter_lds<BITS, THREADS, K>() - (size_t)D * 4 - 64 * 4;
    unsigned *cnt = reinterpret_cast<unsigned *>(radix_smem);
    uint2 *pair = reinterpret_cast<uint2 *>(radix_smem);
    unsigned *ofs = reinterpret_cast<unsigned *>(radix_smem + kFront);
    unsigned *wsum = ofs + D;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t p0 = (int64_t)blockIdx.x * TILE;
    const int n = (int)min((int64_t)TILE, M - p0);
    // this wave's keys: K steps of 64 consecutive ones
    unsigned key[K], val[K], digit[K], rank[K];
    bool live[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int q = (wave * K + i) * 64 + lane;
        live[i] = q < n;
        key[i] = live[i] ? kin[p0 + q] : 0;
        val[i] = vin && live[i] ? vin[p0 + q] : (unsigned)(p0 + q);
        digit[i] = (key[i] >> shift) & (D - 1);
    }
    for (int d = threadIdx.x; d < WAVES * D; d += THREADS) cnt[d] = 0;
    __syncthreads();
    wave_ranks<BITS, K>(digit, live, cnt + wave * D, rank);
    __syncthreads();
    // counters -> exclusive over the waves; a thread's digits are consecutive
    unsigned mine[PER], sum = 0, gsum = 0, gtot[PER];
    const int d0 = threadIdx.x * PER;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        mine[e] = gtot[e] = 0;
        if (d0 + e < D) {
            unsigned run = 0;
            for (int w = 0; w < WAVES; ++w) {
                const unsigned c = cnt[w * D + d0 + e];
                cnt[w * D + d0 + e] = run;
                run += c;
            }
            mine[e] = run;
            gtot[e] = total[d0 + e];
        }
        sum += mine[e];
        gsum += gtot[e];
    }
    unsigned lstart = block_exclusive<WAVES>(sum, wsum);
    unsigned gstart = block_exclusive<WAVES>(gsum, wsum);
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        if (d0 + e < D) {
            // local position of the digit's first key, folded into the wave
            // counters below; global position minus local position
            ofs[d0 + e] = gstart + table[(int64_t)blockIdx.x * D + d0 + e] - lstart;
            for (int w = 0; w < WAVES; ++w) cnt[w * D + d0 + e] += lstart;
        }
        lstart += mine[e];
        gstart += gtot[e];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < K; ++i)
        if (live[i]) rank[i] += cnt[wave * D + digit[i]];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < K; ++i)
        if (live[i]) pair[rank[i]] = make_uint2(key[i], val[i]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int q = i * THREADS + threadIdx.x;
        if (q < n) {
            const uint2 kv = pair[q];
            const int64_t dst = ofs[(kv.x >> shift) & (D - 1)] + (unsigned)q;
            kout[dst] = kv.x;
            vout[dst] = kv.y;
        }
    }
}

// ------------------------------------------------------------- small inputs

// Up to 1024 K keys in one workgroup: digits of 8 bits, the pairs in LDS
// between passes.  With bin_start, also its nbins + 1 entries (bin_start[b] =
// first p with key[p] >= b << bin_shift).
constexpr int kSmallBits = 8;
template <int K>
__global__ void __launch_bounds__(1024)
    radix_small_kernel(int M, int b0, int b1, const unsigned *__restrict__ kin,
                       unsigned *__restrict__ kout, unsigned *__restrict__ vout, int nbins,
                       int bin_shift, int *__restrict__ bin_start) {
    constexpr int D = 1 << kSmallBits, WAVES = 16;
    extern __shared__ __align__(16) unsigned char radix_smem[];
    uint2 *pair = reinterpret_cast<uint2 *>(radix_smem);
    unsigned *cnt = reinterpret_cast<unsigned *>(radix_smem + (size_t)1024 * K * 8);
    unsigned *wsum = cnt + WAVES * D;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned key[K], val[K], digit[K], rank[K];
    bool live[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int q = (wave * K + i) * 64 + lane;
        live[i] = q < M;
        key[i] = live[i] ? kin[q] : 0;
        val[i] = (unsigned)q;
    }
    for (int shift = b0; shift < b1; shift += kSmallBits) {
        const unsigned mask = (1u << min(kSmallBits, b1 - shift)) - 1;
        if (shift != b0) {
#pragma unroll
            for (int i = 0; i < K; ++i) {
                const uint2 kv = live[i] ? pair[(wave * K + i) * 64 + lane] : make_uint2(0, 0);
                key[i] = kv.x;
                val[i] = kv.y;
            }
        }
#pragma unroll
        for (int i = 0; i < K; ++i) digit[i] = (key[i] >> shift) & mask;
        for (int d = threadIdx.x; d < WAVES * D; d += 1024) cnt[d] = 0;
        __syncthreads();
        wave_ranks<kSmallBits, K>(digit, live, cnt + wave * D, rank);
        __syncthreads();
        // thread t < D: digit t's start, then its starts per wave
        unsigned run = 0;
        if (threadIdx.x < D)
            for (int w = 0; w < WAVES; ++w) run += cnt[w * D + threadIdx.x];
        unsigned start = block_exclusive<WAVES>(run, wsum);
        if (threadIdx.x < D)
            for (int w = 0; w < WAVES; ++w) {
                const unsigned c = cnt[w * D + threadIdx.x];
                cnt[w * D + threadIdx.x] = start;
                start += c;
            }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < K; ++i)
            if (live[i]) pair[rank[i] + cnt[wave * D + digit[i]]] = make_uint2(key[i], val[i]);
        __syncthreads();
    }
    for (int q = threadIdx.x; q < M; q += 1024) {
        const uint2 kv = pair[q];
        kout[q] = kv.x;
        vout[q] = kv.y;
    }
    if (!bin_start) return;
    for (int b = threadIdx.x; b <= nbins; b += 1024) {
        const uint64_t kb = (uint64_t)b << bin_shift;
        int lo = 0, hi = M;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (pair[mid].x < kb)
                lo = mid + 1;
            else
                hi = mid;
        }
        bin_start[b] = lo;
    }
}

constexpr int64_t kSmallSort = 16384;
// bins a small sort also bounds itself: 8 searches of 14 LDS reads per thread
constexpr int64_t kSmallBounds = 8192;

// Tile sizes of the large sort: 8192 keys from 2^21 keys up (longer runs of
// equal digits per tile, so fuller cache lines, and a smaller table; 1e7 keys,
// 10 bits, scatter + scan: 70 + 10 us, 4096-key tiles 86 + 16, 2048 119 + 39,
// 16384, one workgroup per CU, 93 + 6); 2048 below, where 8192 would leave CUs
// without a tile (1e6 keys, 9 bits: 12 + 5 us, 8192-key tiles 15 + 5).  8192 keys
// as 512 threads x 16 so that the counters of 11 bits leave room for two
// workgroups per CU.
constexpr int64_t kWideTiles = (int64_t)1 << 21;

int pass_count(int bits) { return bits <= 0 ? 0 : (bits + 10) / 11; }
int pass_bits(int bits) {
    const int p = pass_count(bits);
    return std::max(8, (bits + p - 1) / p);
}

template <typename K>
int allow_lds(K kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        JFA_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize,
                                          (int)bytes));
    return JFA_OK;
}

template <int BITS, int THREADS, int K>
int radix_pass(int64_t M, int shift, const unsigned *kin, const unsigned *vin, unsigned *kout,
               unsigned *vout, unsigned *table, hipStream_t s) {
    constexpr int D = 1 << BITS;
    constexpr size_t lds = scatter_lds<BITS, THREADS, K>();
    const unsigned tiles = (unsigned)((M + THREADS * K - 1) / (THREADS * K));
    unsigned *total = table + (size_t)tiles * D;
    auto scatter = radix_scatter_kernel<BITS, THREADS, K>;
    if (int rc = allow_lds(scatter, lds)) return rc;
    radix_count_kernel<BITS, THREADS, K><<<tiles, THREADS, 0, s>>>(M, shift, kin, table);
    radix_scan_kernel<<<D / kScanCols, kScanCols * kScanRuns, 0, s>>>(D, (int)tiles, table, total);
    scatter<<<tiles, THREADS, lds, s>>>(M, shift, kin, vin, table, total, kout, vout);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <int BITS>
int radix_pass_any(int64_t M, int shift, const unsigned *kin, const unsigned *vin,
                   unsigned *kout, unsigned *vout, unsigned *table, hipStream_t s) {
    if (M >= kWideTiles)
        return radix_pass<BITS, 512, 16>(M, shift, kin, vin, kout, vout, table, s);
    return radix_pass<BITS, 256, 8>(M, shift, kin, vin, kout, vout, table, s);
}

template <int K>
int small_sort(int64_t M, int b0, int b1, const unsigned *kin, unsigned *kout, unsigned *vout,
               int64_t nbins, int bin_shift, int *bin_start, hipStream_t s) {
    const size_t lds = (size_t)1024 * K * 8 + (16 * (1 << kSmallBits) + 64) * 4;
    auto kernel = radix_small_kernel<K>;
    if (int rc = allow_lds(kernel, lds)) return rc;
    kernel<<<1, 1024, lds, s>>>((int)M, b0, b1, kin, kout, vout, (int)nbins, bin_shift, bin_start);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

}  // namespace

// Enough for any key count up to M (a plan sorts fewer points in buffers of a
// larger call): a second pair of buffers, the table of a pass over `bits` bits
// and its totals.
size_t radix_temp_bytes(int64_t M, int bits) {
    if (M <= kSmallSort) return 16;
    const int64_t narrow = std::min(M, kWideTiles) / 2048 + 1, wide = M / 8192 + 1;
    const int64_t tiles = M < kWideTiles ? narrow : std::max(narrow, wide);
    return (size_t)M * 8 + (size_t)(tiles + 1) * ((size_t)1 << pass_bits(bits)) * 4;
}

int radix_sort(void *temp, const unsigned *kin, unsigned *kout, unsigned *vout, int64_t M,
               int b0, int b1, int64_t nbins, int bin_shift, int *bin_start, bool *bounded,
               hipStream_t s) {
    *bounded = false;
    if (M == 0) return JFA_OK;
    if (M <= kSmallSort) {
        int *bs = bin_start && nbins <= kSmallBounds ? bin_start : nullptr;
        *bounded = bs != nullptr;
        if (M <= 2048) return small_sort<2>(M, b0, b1, kin, kout, vout, nbins, bin_shift, bs, s);
        if (M <= 4096) return small_sort<4>(M, b0, b1, kin, kout, vout, nbins, bin_shift, bs, s);
        if (M <= 8192) return small_sort<8>(M, b0, b1, kin, kout, vout, nbins, bin_shift, bs, s);
        return small_sort<16>(M, b0, b1, kin, kout, vout, nbins, bin_shift, bs, s);
    }
    const int bits = std::max(1, b1 - b0), passes = pass_count(bits), per = pass_bits(bits);
    unsigned *tk = (unsigned *)temp, *tv = tk + M, *table = tv + M;
    const unsigned *ki = kin, *vi = nullptr;
    for (int q = 0; q < passes; ++q) {
        // the last pass writes the output, the one before it the second buffers
        const bool to_out = (passes - 1 - q) % 2 == 0;
        unsigned *ko = to_out ? kout : tk, *vo = to_out ? vout : tv;
        const int shift = b0 + q * per;
        int rc = JFA_OK;
        switch (per) {
            case 8: rc = radix_pass_any<8>(M, shift, ki, vi, ko, vo, table, s); break;
            case 9: rc = radix_pass_any<9>(M, shift, ki, vi, ko, vo, table, s); break;
            case 10: rc = radix_pass_any<10>(M, shift, ki, vi, ko, vo, table, s); break;
            default: rc = radix_pass_any<11>(M, shift, ki, vi, ko, vo, table, s); break;
        }
        if (rc) return rc;
        ki = ko;
        vi = vo;
    }
    return JFA_OK;
}

}  // namespace jfa
