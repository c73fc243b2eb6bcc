// Atomic-free 2D spreading ("strip" method), the default type-1 spreader in 2D.
//
// Replaces the 2D type-1 spreading cuFINUFFT runs inside execute (called at
// lib/kernels.cc.cu:75; source absent from the reference).  Designed around
// two measured facts of gfx950: LDS float atomics are ~35x slower than LDS
// integer atomics or plain LDS traffic, and coalesced plain stores are far
// cheaper than global float atomics.
//
// Layout.  The fine grid is cut into vertical strips of SW = 64 - ns + 1
// columns; strip s owns points whose first x-tap l0x lies in
// [s*SW, (s+1)*SW), so all of their taps fall in the 64 columns
// [s*SW, s*SW + 64).  Points are sorted by (strip, l0y) (the "y-major" bins
// set up by the plan).  A strip is cut into units of H consecutive l0y rows:
// short ones of 9 rows (ns <= 8) or 33 - ns, on large sparse grids tall ones of
// 33 - ns (ns <= 8) or up to 128 (strip_tall).  A unit's whole tile, 16 or 32 rows x
// 64 columns, lives in the registers of the wave that spreads it, as the
// accumulators of MFMA products; those of 128 rows roll through 32.
//
// Spreading is a contraction over points: tile[y][x] += sum_p (c_p ky_p[y])
// kx_p[x].  strip_piece takes four points at a time as the K dimension of a
// 16 x 16 x 4 MFMA, whose 16 rows are the tile's and whose 16 columns are a
// frame of the tile, one product for the real and one for the imaginary part
// (details there).  Points are staged 64 at a time: each lane evaluates one
// point's ns x-weights and ns y-weights (Horner) and writes them to
// wave-private LDS in frame order.  No atomics touch LDS.
//
// Bound by instruction issue, VALU and MFMA together (a SIMD issues one or the
// other): figures at strip_piece.
//
// Output.  A unit's points are cut into pieces of at most `pmax` points (an
// empty unit has none), one workgroup of one or four waves per piece.  A piece
// writes its rows with plain coalesced stores into its own scratch tile of
// (H + ns - 1) x 64 cells; a merge kernel then writes every fine-grid cell once,
// as the sum over the units covering it (one to four, up to nine next to a narrow
// last strip or unit) of their pieces' tiles.  The fine grid is neither zeroed
// first nor read, no float atomics are used anywhere, and the summation order is
// fixed, so results are bitwise reproducible.
//
// The same per-piece and per-cell bodies serve one plan (a single problem,
// blockIdx.y = transform) and a ragged batch of problems (descriptor tables,
// one launch over every problem's units).
//
// 3D.  A 3D grid is a stack of nz = nf2 slices of nf0 x nf1 cells.  A point
// with first taps (l0x, l0y, l0z) and z-weights kz[dz] spreads, in slice
// l0z + dz, like a 2D point at (l0x, l0y) of strength c * kz[dz]; setpts
// expands every point into its ns slice points and sorts them by (slice,
// strip, row), so the strips of all slices form one list of nz * S strips
// (strip index z * S + s) and the 2D bodies run unchanged.  Only the merge
// needs the slice: its neighbours are taken within the slice.
#include <utility>

#include "jfa_device.hpp"

namespace jfa {
namespace {

constexpr int kStripLanes = 64;

// f(integral_constant 0), ..., f(integral_constant N - 1)
template <typename F, int... Is>
__device__ __forceinline__ void unroll_seq(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void unroll(F &&f) {
    unroll_seq(f, std::make_integer_sequence<int, N>{});
}

template <typename T>
struct alignas(2 * sizeof(T)) Pair {
    T x, y;
};
template <typename T>
struct alignas(4 * sizeof(T)) Quad {
    T x, y, z, w;
};

// MFMA 16 x 16 x 4: D[i][j] += sum_k A[i][k] B[k][j].  Lane l holds A[l % 16][l / 16],
// B[l / 16][l % 16] and D[row(r, l / 16)][l % 16], r < 4.
template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
    typedef float Acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ Acc mul(float a, float b, Acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int r, int g) { return 4 * g + r; }
};
template <>
struct Mfma<double> {
    typedef double Acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ Acc mul(double a, double b, Acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int r, int g) { return 4 * r + g; }
};

// Shape of a unit's tile in MFMA terms (see strip_piece).  TALL: units of more than
// strip_short_rows rows, ns <= 8 (wider kernels' shape is always the tall one).
constexpr bool strip_rolls(int ns, bool tall) { return tall && ns > 8; }
template <int NS, bool TALL>
struct StripShape {
    static constexpr bool kNarrow = NS <= 8 && !TALL;
    static constexpr int kRowTiles = kNarrow ? 1 : 2;  // of 16 rows
    // narrow: frames start every 8 columns, so one 16-column frame holds a
    // point's taps; wide: every 16 columns, a point reaches into the next frame
    static constexpr int kFrames = kNarrow ? 8 : 4;
    static constexpr int kFrameShift = kNarrow ? 3 : 4;
    // Values per staged point and axis.  Narrow: the weights, then zeros, so that
    // any 16-value window that starts up to 8 before a point's weights (units
    // are at most 9 rows) reads zeros around them (the previous point's zeros lie
    // in front).  Wide: the
    // weights alone.  Odd, so that the points of one write are on distinct banks.
    static constexpr int kStride = kNarrow ? 17 : NS | 1;
    static constexpr int kGuard = kNarrow ? 8 : 0;  // zeros before the first point
    static constexpr int kValues = kGuard + kStripLanes * kStride - (kNarrow ? 1 : 0);
    // Slots of a batch: every frame's points rounded up to groups of four, and a
    // group read ahead.
    static constexpr int kSlots = kStripLanes + 3 * kFrames + 4;
};

// A staged point as the MFMA loop finds it: the strengths of NT transforms, and
// two 16-bit values that locate its y (high) and x weights.
template <typename T, int NT>
struct alignas(16) StripSlot {
    Pair<T> c[NT];
    unsigned at;
};

// LDS staging of one wave: the weights by point of the batch, the points by slot.
// (ns <= 8 in fp32: 10,232 bytes, so that 16 waves share a CU's 160 KiB.)
template <typename T, int NS, int NT, bool TALL>
struct StripLds {
    StripSlot<T, NT> slot[StripShape<NS, TALL>::kSlots];
    T ky[StripShape<NS, TALL>::kValues];
    T kx[StripShape<NS, TALL>::kValues];
};

// The ns weights of a point along one axis to LDS, as eval_kernel computes them.  Double
// kernels of ns >= 8 two taps at a time, in a loop: the accumulators leave no registers for
// every tap at once.
template <typename T, int NS, typename Coef>
__device__ __forceinline__ void stage_weights(Coef coef, T beta, int horner, T t, T *out) {
    if constexpr (sizeof(T) == 8 && NS >= 8) {
        if (horner) {
            constexpr int NC = horner_nc(NS), NE = (NC + 1) / 2, NO = NC / 2, half = (NS + 1) / 2;
            const T s = t * t;
#pragma unroll 1
            for (int i = 0; i < half; i += 2) {
                const Coef c = coef + i;
                T e0 = c[2 * (NE - 1) * NS], e1 = c[2 * (NE - 1) * NS + 1];
                T o0 = c[(2 * NO - 1) * NS], o1 = c[(2 * NO - 1) * NS + 1];
#pragma unroll
                for (int k = NE - 2; k >= 0; --k) {
                    e0 = fma(e0, s, c[2 * k * NS]);
                    e1 = fma(e1, s, c[2 * k * NS + 1]);
                }
#pragma unroll
                for (int k = NO - 2; k >= 0; --k) {
                    o0 = fma(o0, s, c[(2 * k + 1) * NS]);
                    o1 = fma(o1, s, c[(2 * k + 1) * NS + 1]);
                }
                out[NS - 1 - i] = fma(-t, o0, e0);
                out[i] = fma(t, o0, e0);
                if (half % 2 == 0 || i + 1 < half) {
                    out[NS - 2 - i] = fma(-t, o1, e1);
                    out[i + 1] = fma(t, o1, e1);
                }
            }
        } else {
#pragma unroll 1
            for (int i = 0; i < NS; ++i) {
                const T z = (T(-0.5 * NS) + T(i) + T(0.5) * (t + T(1))) * (T(2) / T(NS));
                const T a = T(1) - z * z;
                out[i] = a < T(0) ? T(0) : exp(beta * (sqrt(a) - T(1)));
            }
        }
        return;
    }
    T k[NS];
    if (horner)
        eval_kernel<T, NS, true>(coef, beta, t, k);
    else
        eval_kernel<T, NS, false>(coef, beta, t, k);
#pragma unroll
    for (int i = 0; i < NS; ++i) out[i] = k[i];
}

// Finite, with room for its products with weights.
__device__ __forceinline__ bool plain(float v) { return fabsf(v) <= 1e38f; }
__device__ __forceinline__ bool plain(double v) { return fabs(v) <= 1e307; }

// Order of one wave's LDS accesses: its instructions reach LDS in program order,
// so only the compiler has to keep it.
__device__ __forceinline__ void wave_sync() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// Strength and Horner pair of input point P: from the packed record, or from
// the strengths (by index within the problem) and the setpts pairs (by P).
template <typename T>
__device__ __forceinline__ Quad<T> point_record(const StripPts<T> &pts, int64_t P) {
    const int64_t j = P - pts.idx_off;
    if (pts.pack) return reinterpret_cast<const Quad<T> *>(pts.pack)[j];
    const Pair<T> cv = reinterpret_cast<const Pair<T> *>(pts.c)[j];
    const Pair<T> tv = reinterpret_cast<const Pair<T> *>(pts.rec)[P];
    return Quad<T>{cv.x, cv.y, tv.x, tv.y};
}

// The point range [pb, pe) of piece `sub` of unit u, and its strip / rows.
struct PieceRange {
    int ox, r0, pb, pe;
};
__device__ __forceinline__ PieceRange piece_range(const StripGeom &sg,
                                                  const int *__restrict__ bin_start, int u,
                                                  int sub) {
    const int s = u / sg.K, k = u - s * sg.K;
    PieceRange pr;
    pr.ox = s * sg.SW;
    pr.r0 = k * sg.H;
    const int r1 = min(pr.r0 + sg.H, (int)sg.nf1);
    const int ub = bin_start[(int64_t)s * sg.nf1 + pr.r0];
    const int ue = bin_start[(int64_t)s * sg.nf1 + r1];
    pr.pb = ub + sub * sg.pmax;
    pr.pe = min(pr.pb + sg.pmax, ue);
    return pr;
}

// ------------------------------------------------------------ one piece
//
// Spreads one piece's points for NT transforms sharing them: transform k's
// strengths at pts.c + k * pts.c_tstride (NT = 1 may read packed records instead),
// its tile at tile + k * tile_tstride.
//
// The accumulators hold the unit's tile: rows r0 .. r0 + 16 kRowTiles - 1 by
// frames of 16 columns.  ns <= 8: eight frames 8 columns apart, one row tile, so a
// point adds to exactly one frame: one MFMA each for the real and imaginary parts
// of four points (half the columns are zeros).  ns > 8, and tall units of ns <= 8
// (strip_tall): four frames, two row tiles; a point adds to its frame and the next,
// and to both row tiles where its rows straddle them (batches are in row order, so a
// row tile no point of the batch touches is skipped).  Each MFMA's four points must
// share a frame: the points of a batch are ranked by frame (one ballot per bit of
// the frame) and listed in that order in the slots, every frame's list filled up to
// a multiple of four with zero strengths; the weights stay where the point's lane
// wrote them.
//
// Counted at 1e7 uniform points on 2048^2 (fp32, ns = 8), per point: 19 MFMA
// cycles, 7.1 VALU wave instructions (of 4 cycles; 104 Horner FMAs over 64 lanes,
// ranking, operand addresses), 7 LDS cycles.  263 us, where adding one point after
// another to per-lane windows of the tile (10.4 VALU instructions and 9.6 LDS cycles
// per point) took 268; a unit's points now need no order within a row, which makes
// the sort's keys 3 bits shorter.  The walk was a chain of LDS reads and adds, so
// smaller and wider problems gain more: 1e6 fp64 points on 1024^2 cells at ns = 11
// 275 -> 152 us, 300,007 centre-dense points x 4 transforms on 301 x 255 modes at
// ns = 6 65 -> 47, 4000 points on 48 x 40 29 -> 8; 2^20 sources of a 3D type 3 at
// ns = 8 507 -> 320.
//
// Tall units of ns > 8 have up to 128 rows, which the accumulators roll over: they hold
// 32 rows, row y in place y mod 32, and whenever the points move on past the first 16
// those are complete, go to the tile and start again at zero.  A batch is staged once and
// multiplied window by window.  This costs registers (89 spilled) and waves; it is for
// grids whose tiles bound the call (1e6 points on 8192^2 cells at ns = 16, units of 17
// rows 1430 us with the merge, of 128 1150).
//
// W waves share a piece: each spreads a run of its points into accumulators of its
// own, which are added through LDS in wave order at the end.
template <typename T, int NS, int NT, int W, bool TALL>
__device__ __forceinline__ void strip_piece(const StripGeom &sg, const StripPts<T> &pts,
                                            const int *__restrict__ bin_start, int u, int sub,
                                            const T *__restrict__ coef, T beta, int horner,
                                            T *__restrict__ tile, int64_t tile_tstride,
                                            StripLds<T, NS, NT, TALL> *lds_all) {
    using Sh = StripShape<NS, TALL>;
    constexpr bool ROLL = strip_rolls(NS, TALL);
    using M = Mfma<T>;
    using Acc = typename M::Acc;
    constexpr int RT = Sh::kRowTiles, NF = Sh::kFrames, S = Sh::kStride;
    const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
    const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    StripLds<T, NS, NT, TALL> &lds = lds_all[wave];
    const PieceRange pr = piece_range(sg, bin_start, u, sub);
    const int r0 = pr.r0;
    // this wave's points: whole batches, as even as they come
    const int per = ((pr.pe - pr.pb + W - 1) / W + kStripLanes - 1) & -kStripLanes;
    const int pb = min(pr.pb + wave * per, pr.pe), pe = min(pb + per, pr.pe);
    // key >> kStripKeyShift = rowbase + l0y for every point of this strip
    const int64_t rowbase = pts.bin_off + (int64_t)(u / sg.K) * sg.nf1;
    Acc re[NT][RT][NF], im[NT][RT][NF];
    unroll<NT * RT * NF>([&](auto c) {
        constexpr int e = decltype(c)::value, t = e / (RT * NF), h = e / NF % RT, f = e % NF;
        re[t][h][f] = im[t][h][f] = Acc{0, 0, 0, 0};
    });
    // the weights' places before any is staged: zeros, as around them later
    for (int e = lane; e < Sh::kValues; e += kStripLanes) lds.ky[e] = lds.kx[e] = T(0);
    StripSlot<T, NT> none;
#pragma unroll
    for (int t = 0; t < NT; ++t) none.c[t] = Pair<T>{T(0), T(0)};
    none.at = Sh::kNarrow ? (unsigned)(Sh::kGuard * sizeof(T)) * 0x10001u : 0u;
    // Software pipeline over 64-point batches: while one batch is staged and
    // multiplied, the next batch's records (and other transforms' strengths) and
    // the key and index of the batch after it are in flight.
    constexpr int NC = NT > 1 ? NT - 1 : 1;
    unsigned key1 = 0, key2 = 0;
    int idx1 = 0, idx2 = 0;
    Quad<T> rq1{};
    Pair<T> ct1[NC];
    auto load_index = [&](int b, unsigned &k, int &i) {
        if (b + lane < pe) {
            k = pts.key[b + lane];
            i = pts.idx[b + lane];
        }
    };
    auto load_record = [&](int b, int i) {
        if (b + lane < pe) {
            rq1 = point_record(pts, i);
#pragma unroll
            for (int t = 1; t < NT; ++t)
                ct1[t - 1] = reinterpret_cast<const Pair<T> *>(
                    pts.c + t * pts.c_tstride)[i - pts.idx_off];
        }
    };
    int top = 0;  // rolling: the window's first row, from r0
    // the tile's rows to scratch: value e = (t, h, r, k) is row 16 h + row(r, g),
    // column 16 k + i16 of transform t
    const int rows_tile = sg.H + NS - 1;
    const bool upper = i16 >= 8;
    auto value = [&](auto ec) {
        constexpr int e = decltype(ec)::value, t = e / (RT * 16), h = e / 16 % RT, k = e / 4 % 4,
                      r = e % 4;
        if constexpr (!Sh::kNarrow) {
            return Pair<T>{re[t][h][k][r], im[t][h][k][r]};
        } else {
            // columns 16 k ..: the even frame 2 k, and the odd frames on either
            // side, whose lanes are 8 columns off
            T sr = re[t][h][2 * k + 1][r], si = im[t][h][2 * k + 1][r];
            if constexpr (k > 0) {
                sr = upper ? re[t][h][2 * k - 1][r] : sr;
                si = upper ? im[t][h][2 * k - 1][r] : si;
            } else {
                sr = upper ? T(0) : sr;
                si = upper ? T(0) : si;
            }
            return Pair<T>{re[t][h][2 * k][r] + __shfl_xor(sr, 8),
                           im[t][h][2 * k][r] + __shfl_xor(si, 8)};
        }
    };
    auto store = [&](int e, int row, int col, Pair<T> v) {
        const int t = e / (RT * 16), k = e / 4 % 4;
        if (row < rows_tile)
            reinterpret_cast<Pair<T> *>(tile + t * tile_tstride)[row * kStripLanes + 16 * k + col] =
                v;
    };
    // Rolling: the window's first 16 rows, one row tile, are complete; they go to the
    // tile, and the row tile starts again at zero behind the other one.
    auto flush = [&] {
        int ln = lane;  // opaque: addresses are computed here, not kept in registers
        asm volatile("" : "+v"(ln));
        auto half = [&](auto hc) {
            constexpr int h = decltype(hc)::value;
            // (both halves' code is alike but for the registers: kept apart)
            asm volatile("; row tile %0" ::"n"(h));
            unroll<NT * 16>([&](auto ec) {
                constexpr int e0 = decltype(ec)::value, e = (e0 / 16 * RT + h) * 16 + e0 % 16;
                store(e, top + M::row(e % 4, ln >> 4), ln & 15, value(std::integral_constant<int, e>{}));
            });
            asm volatile("; row tile %0 done" ::"n"(h));
        };
        if (top & 16)
            half(std::integral_constant<int, RT - 1>{});
        else
            half(std::integral_constant<int, 0>{});
        // (selected, in place: cleared in the branches they would be copied)
        int odd = top & 16;
        asm volatile("" : "+v"(odd));
        unroll<NT * RT * NF * 4>([&](auto c) {
            constexpr int e = decltype(c)::value, t = e / (RT * NF * 4), h = e / (NF * 4) % RT,
                          f = e / 4 % NF, r = e % 4;
            const bool clear = h == 0 ? odd == 0 : odd != 0;
            re[t][h][f][r] = clear ? T(0) : re[t][h][f][r];
            im[t][h][f][r] = clear ? T(0) : im[t][h][f][r];
        });
        top += 16;
    };
    load_index(pb, key1, idx1);
    load_record(pb, idx1);
    load_index(pb + kStripLanes, key2, idx2);
    for (int bb = pb; bb < pe; bb += kStripLanes) {
        const int nb = min(kStripLanes, pe - bb);
        const unsigned pkey = key1;
        Quad<T> rq = rq1;
        Pair<T> ct[NC];
#pragma unroll
        for (int t = 0; t < NC; ++t) ct[t] = ct1[t];
        key1 = key2;
        idx1 = idx2;
        load_record(bb + kStripLanes, idx1);
        load_index(bb + 2 * kStripLanes, key2, idx2);
        // opaque: hoisted out of the loop, the coefficients would not fit the scalar
        // registers and spill; constant address space: scalar loads all the same
        uintptr_t cf_bits = reinterpret_cast<uintptr_t>(coef);
        asm volatile("" : "+s"(cf_bits));
        const auto *cf = reinterpret_cast<const __attribute__((address_space(4))) T *>(cf_bits);
        // Points whose values would not stay within their taps (0 x inf is NaN) go in as
        // zeros here, and one by one below.
        bool odd = !plain(rq.x) || !plain(rq.y) || !(fabs(rq.z) <= T(2)) || !(fabs(rq.w) <= T(2));
#pragma unroll
        for (int t = 1; t < NT; ++t) odd = odd || !plain(ct[t - 1].x) || !plain(ct[t - 1].y);
        uint64_t left = __ballot(lane < nb && odd);
        if (left && odd) {
            rq.x = rq.y = T(0);
            if (!(fabs(rq.z) <= T(2))) rq.z = T(0);
            if (!(fabs(rq.w) <= T(2))) rq.w = T(0);
#pragma unroll
            for (int t = 1; t < NT; ++t) ct[t - 1] = Pair<T>{T(0), T(0)};
        }
        if (lane < nb) {
            const int v0 = Sh::kGuard + lane * S;
            stage_weights<T, NS>(cf, beta, horner, rq.z, lds.kx + v0);
            stage_weights<T, NS>(cf, beta, horner, rq.w, lds.ky + v0);
        }
        // rolling: the batch window by window (its points come in row order)
        for (int done = 0;;) {
            // opaque: what follows from the key and the lane is computed in every window,
            // or it would be computed ahead and spilled
            unsigned key = pkey;
            int ln = lane;
            if constexpr (ROLL) asm volatile("" : "+v"(key), "+v"(ln));
            const int X = (int)(key & ((1u << kStripKeyShift) - 1));
            const int Y = (int)((int64_t)(key >> kStripKeyShift) - rowbase) - r0;
            uint64_t in = nb < kStripLanes ? (uint64_t(1) << nb) - 1 : ~uint64_t(0);
            if constexpr (ROLL) in &= __ballot(Y < top + 16) & (~uint64_t(0) << done);
            const int count = ROLL ? __popcll(in) : nb;
            if (!ROLL || in) {
                // this lane's slot, and the groups of four of every frame
                constexpr int kBits = Sh::kNarrow ? 3 : 2;
                const unsigned frame = (unsigned)X >> Sh::kFrameShift;
                uint64_t bit[kBits], same = in;
#pragma unroll
                for (int b = 0; b < kBits; ++b) {
                    const bool one = (frame >> b) & 1;
                    bit[b] = __ballot(one);
                    same &= one ? bit[b] : ~bit[b];
                }
                int groups[NF];
                uint64_t starts = 0;  // first group of every frame, 5 bits each
                int base = 0;
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    uint64_t m = in;
#pragma unroll
                    for (int b = 0; b < kBits; ++b) m &= (f >> b) & 1 ? bit[b] : ~bit[b];
                    starts |= (uint64_t)base << (5 * f);
                    groups[f] = (__popcll(m) + 3) >> 2;
                    base += groups[f];
                }
                const int slot = 4 * (int)((starts >> (5 * frame)) & 31) +
                                 (int)__builtin_amdgcn_mbcnt_hi(
                                     (unsigned)(same >> 32),
                                     __builtin_amdgcn_mbcnt_lo((unsigned)same, 0u));
                // the row tiles these points reach (a rolling window: 32 rows from
                // `top`, row y in place y mod 32)
                bool low = true, high = false;
                if constexpr (ROLL) {
                    const bool both = __builtin_amdgcn_readlane(Y, done + count - 1) + NS > top + 16;
                    low = both || !(top & 16);
                    high = both || (top & 16);
                } else if constexpr (RT > 1) {
                    low = __builtin_amdgcn_readfirstlane(Y) < 16;
                    high = __builtin_amdgcn_readlane(Y, nb - 1) + NS > 16;
                }
                // (a wave's LDS writes land in order: the empty slots before the filled)
                lds.slot[ln] = none;
                if (ln + kStripLanes < Sh::kSlots) lds.slot[ln + kStripLanes] = none;
                if ((in >> ln) & 1) {
                    const int v0 = Sh::kGuard + ln * S;
                    const int ox = X & ((1 << Sh::kFrameShift) - 1);
                    StripSlot<T, NT> me;
                    me.c[0] = Pair<T>{rq.x, rq.y};
#pragma unroll
                    for (int t = 1; t < NT; ++t) me.c[t] = ct[t - 1];
                    // narrow: byte offsets of where row 0 of the tile / column 0 of the frame
                    // lie in the staged values; wide: the first row, and lane and column
                    me.at = Sh::kNarrow
                                ? (unsigned)((v0 - Y) * sizeof(T)) << 16 | (unsigned)((v0 - ox) * sizeof(T))
                                : (unsigned)(ROLL ? Y & 31 : Y) << 16 | (unsigned)(ln << 4) | (unsigned)ox;
                    lds.slot[slot] = me;
                }
                wave_sync();
                // operands of the four points from slot 4 n: lane (i16, g) reads point g's
                constexpr int NB = Sh::kNarrow ? 1 : 2;
                struct Operands {
                    T y[RT], x[NB];
                    Pair<T> c[NT];
                };
                const StripSlot<T, NT> *next = lds.slot + g;
                auto fetch = [&] {
                    Operands o;
                    const StripSlot<T, NT> s = *next;
                    next += 4;
#pragma unroll
                    for (int t = 0; t < NT; ++t) o.c[t] = s.c[t];
                    if constexpr (Sh::kNarrow) {
                        // both halves at once (neither overflows)
                        const unsigned at = s.at + (unsigned)(i16 * sizeof(T)) * 0x10001u;
                        o.y[0] = *reinterpret_cast<const T *>(
                            reinterpret_cast<const char *>(lds.ky) + (at >> 16));
                        o.x[0] = *reinterpret_cast<const T *>(
                            reinterpret_cast<const char *>(lds.kx) + (at & 0xffffu));
                    } else {
                        const int ya = (int)(s.at >> 16), xa = (int)(s.at & 15u);
                        const int v0 = (int)(s.at >> 4 & 63u) * S;
#pragma unroll
                        for (int h = 0; h < RT; ++h) {
                            const int e = (i16 + 16 * h - ya) & (ROLL ? 31 : ~0);
                            const T v = lds.ky[v0 + (unsigned(e) < NS ? e : 0)];
                            o.y[h] = unsigned(e) < NS ? v : T(0);
                        }
#pragma unroll
                        for (int h = 0; h < NB; ++h) {
                            const int e = i16 + 16 * h - xa;
                            const T v = lds.kx[v0 + (unsigned(e) < NS ? e : 0)];
                            o.x[h] = unsigned(e) < NS ? v : T(0);
                        }
                    }
                    return o;
                };
                Operands cur = fetch();
                // frames as compile-time constants, so that the accumulators are separate
                // registers to the compiler (as one array it copies it between frames)
                unroll<NF>([&](auto fc) {
                    constexpr int f = decltype(fc)::value;
                    for (int n = groups[f]; n > 0; --n) {
                        const Operands o = cur;
                        cur = fetch();
                        unroll<RT>([&](auto hc) {
                            constexpr int h = decltype(hc)::value;
                            if (RT > 1 && !(h == 0 ? low : high)) return;
                            const T y = o.y[h];
                            unroll<NT>([&](auto tc) {
                                constexpr int t = decltype(tc)::value;
                                const T ar = y * o.c[t].x, ai = y * o.c[t].y;
                                re[t][h][f] = M::mul(ar, o.x[0], re[t][h][f]);
                                im[t][h][f] = M::mul(ai, o.x[0], im[t][h][f]);
                                if constexpr (NB > 1 && f + 1 < NF) {
                                    // (no point of the last frame leaves it)
                                    re[t][h][f + 1] = M::mul(ar, o.x[NB - 1], re[t][h][f + 1]);
                                    im[t][h][f + 1] = M::mul(ai, o.x[NB - 1], im[t][h][f + 1]);
                                }
                            });
                        });
                    }
                });
                for (uint64_t m = left & in; m; m &= m - 1) {
                    const int q = __builtin_ctzll(m);
                    const unsigned key = pts.key[bb + q];
                    const int i = pts.idx[bb + q];
                    const Quad<T> p = point_record(pts, i);
                    const int qx = (int)(key & ((1u << kStripKeyShift) - 1));
                    const int qy = (int)((int64_t)(key >> kStripKeyShift) - rowbase) - r0;
                    // (a weight of NaN where the coordinate is)
                    const T u = (fabs(p.z) <= T(2) ? T(0) : p.z - p.z) + (fabs(p.w) <= T(2) ? T(0) : p.w - p.w);
                    unroll<NT>([&](auto tc) {
                        constexpr int t = decltype(tc)::value;
                        Pair<T> c{p.x, p.y};
                        if constexpr (t > 0)
                            c = reinterpret_cast<const Pair<T> *>(pts.c + t * pts.c_tstride)[i - pts.idx_off];
                        unroll<RT * NF * 4>([&](auto ec) {
                            constexpr int e = decltype(ec)::value, h = e / (NF * 4), f = e / 4 % NF,
                                          r = e % 4;
                            const int dy = (16 * h + M::row(r, g) - qy) & (ROLL ? 31 : ~0);
                            const int dx = (f << Sh::kFrameShift) + i16 - qx;
                            if (unsigned(dy) < NS && unsigned(dx) < NS &&
                                (!Sh::kNarrow || f == qx >> Sh::kFrameShift)) {
                                const int v0 = Sh::kGuard + q * S;
                                const T w = lds.kx[v0 + dx] * lds.ky[v0 + dy] + u;
                                re[t][h][f][r] += c.x * w;
                                im[t][h][f][r] += c.y * w;
                            }
                        });
                    });
                }
                wave_sync();
            }
            if constexpr (!ROLL) break;
            done += count;
            if (done == nb) break;
            flush();
        }
    }
    if constexpr (ROLL) {
        while (top < rows_tile) flush();
    } else if constexpr (W == 1) {
        unroll<NT * RT * 16>([&](auto ec) {
            constexpr int e = decltype(ec)::value;
            store(e, 16 * (e / 16 % RT) + M::row(e % 4, g), i16, value(ec));
        });
    } else {
        // eight values of every lane at a time through the staging areas; wave w
        // adds up values w, w + W, ...
        static_assert(sizeof(StripLds<T, NS, NT, TALL>) >= 8 * kStripLanes * sizeof(Pair<T>), "");
        __syncthreads();
        unroll<NT * RT * 2>([&](auto cc) {
            constexpr int e0 = 8 * decltype(cc)::value;
            unroll<8>([&](auto ec) {
                constexpr int e = e0 + decltype(ec)::value;
                reinterpret_cast<Pair<T> *>(&lds)[(e - e0) * kStripLanes + lane] =
                    value(std::integral_constant<int, e>{});
            });
            __syncthreads();
#pragma unroll
            for (int e = 0; e < 8; e += W) {
                Pair<T> v{T(0), T(0)};
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const Pair<T> x = reinterpret_cast<const Pair<T> *>(
                        lds_all + w)[(e + wave) * kStripLanes + lane];
                    v.x += x.x;
                    v.y += x.y;
                }
                store(e0 + e + wave, 16 * ((e0 + e + wave) / 16 % RT) + M::row((e0 + e + wave) % 4, g), i16, v);
            }
            __syncthreads();
        });
    }
}

// The windows of one axis that reach into window w's first ns - 1 cells from
// the left: window w - 1, or, for w = 0, the last one or two windows through
// the periodic wrap (the second when the last window owns fewer than ns - 1
// cells), w itself among them where the axis is shorter than a window.  Windows
// start every `step` cells, span `span` and n of them cover nf cells.  Appends (window, offset of w's cell 0 in its tile) to win / off.
__device__ __forceinline__ int left_windows(int w, int step, int span, int n, int64_t nf,
                                            int *win, int *off) {
    int c = 0;
    if (w > 0) {
        win[c] = w - 1;
        off[c] = step;
        ++c;
    } else {
        for (int v = n - 1; v >= 0 && v >= n - 2; --v) {
            const int o = (int)(nf - (int64_t)v * step);
            if (o < span) {
                win[c] = v;
                off[c] = o;
                ++c;
            }
        }
    }
    return c;
}

// The cells unit u owns (columns [s*SW, s*SW + SW) and rows [k*H, k*H + H),
// clipped to the grid), each written once as the sum of the tiles of every
// piece of every unit covering it: u itself, and the units to its left, above
// and diagonally where their tiles reach into u's first ns - 1 columns / rows.
// One workgroup per unit, lane = column, waves over rows; the candidate units
// and their piece ranges are uniform over the workgroup.  piece_start holds the
// problem's units' first piece numbers; tile i of `scratch` belongs to piece
// piece_start[0] + i.
template <typename T, int NS>
__device__ __forceinline__ void merge_unit(const StripGeom &sg, const int *__restrict__ piece_start,
                                           const T *__restrict__ scratch, T *__restrict__ fw,
                                           int u, int reduced) {
    constexpr int SW = 65 - NS;
    const int sz = u / sg.K, k = u - sz * sg.K;  // strip over all slices, unit row
    const int z = sz / sg.S, s = sz - z * sg.S;  // slice, strip within it
    fw += 2 * (int64_t)z * sg.nf0 * sg.nf1;
    const int x0 = s * SW, y0 = k * sg.H;
    const int wcols = min(SW, (int)(sg.nf0 - x0));
    const int wrows = min(sg.H, (int)(sg.nf1 - y0));
    const int rows_tile = sg.H + NS - 1;
    const int64_t tile_cells = (int64_t)rows_tile * kStripLanes;
    const int base = piece_start[0];
    int cs[3] = {s, 0, 0}, co[3] = {0, 0, 0}, ck[3] = {k, 0, 0}, ro[3] = {0, 0, 0};
    const int ncs = 1 + left_windows(s, SW, kStripLanes, sg.S, sg.nf0, cs + 1, co + 1);
    const int nck = 1 + left_windows(k, sg.H, rows_tile, sg.K, sg.nf1, ck + 1, ro + 1);
    // the covering units' piece ranges, once per workgroup (uniform); entry
    // 3 i + j is strip candidate i with unit-row candidate j (no pieces when
    // either does not exist)
    int pfirst[9], pcount[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            pfirst[3 * i + j] = 0;
            pcount[3 * i + j] = 0;
            if (i < ncs && j < nck) {
                const int u2 = (z * sg.S + cs[i]) * sg.K + ck[j];
                pfirst[3 * i + j] = piece_start[u2] - base;
                // reduced: a crowded unit's pieces were summed into its first tile
                const int np = piece_start[u2 + 1] - piece_start[u2];
                pcount[3 * i + j] = reduced ? min(np, 1) : np;
            }
        }
    const int c = threadIdx.x & (kStripLanes - 1);
    if (c >= wcols) return;
    const Pair<T> *tiles = reinterpret_cast<const Pair<T> *>(scratch);
    for (int r = threadIdx.x / kStripLanes; r < wrows; r += blockDim.x / kStripLanes) {
        T ar = T(0), ai = T(0);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const int q = 3 * i + j;
                const int tc = c + co[i], tr = r + ro[j];
                if (pcount[q] == 0 || tc >= kStripLanes || tr >= rows_tile) continue;
                const Pair<T> *src =
                    tiles + (int64_t)pfirst[q] * tile_cells + tr * kStripLanes + tc;
                for (int pc = 0; pc < pcount[q]; ++pc) {
                    const Pair<T> v = src[pc * tile_cells];
                    ar += v.x;
                    ai += v.y;
                }
            }
        reinterpret_cast<Pair<T> *>(fw)[(int64_t)(y0 + r) * sg.nf0 + x0 + c] = Pair<T>{ar, ai};
    }
}

// pieces of unit u: ceil(count / pmax), none for an empty unit
__device__ __forceinline__ int unit_pieces(const StripGeom &sg, const int *__restrict__ bin_start,
                                           int u) {
    const int s = u / sg.K, k = u - s * sg.K;
    const int r0 = k * sg.H, r1 = min(r0 + sg.H, (int)sg.nf1);
    const int cnt = bin_start[(int64_t)s * sg.nf1 + r1] - bin_start[(int64_t)s * sg.nf1 + r0];
    return (cnt + sg.pmax - 1) / sg.pmax;
}

// One workgroup: exclusive prefix of pieces(u) over u in [0, n); total at
// piece_start[n] and in *npieces; with piece_unit, also the unit of every piece;
// with heavy, the list [count, u ...] of the units with more than one piece.
template <typename PiecesOf>
__device__ __forceinline__ void piece_scan(int n, PiecesOf pieces, int *piece_start,
                                           int *npieces, int *piece_unit, int *heavy) {
    __shared__ int sa[1024];
    const int tid = threadIdx.x;
    if (heavy && tid == 0) heavy[0] = 0;  // ordered before the atomics by the barriers below
    const int per = (n + 1023) / 1024;
    const int lo = min(tid * per, n);
    const int hi = min(lo + per, n);
    int a = 0;
    for (int u = lo; u < hi; ++u) a += pieces(u);
    sa[tid] = a;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        int v = tid >= off ? sa[tid - off] : 0;
        __syncthreads();
        sa[tid] += v;
        __syncthreads();
    }
    int e = sa[tid] - a;
    for (int u = lo; u < hi; ++u) {
        piece_start[u] = e;
        const int np = pieces(u);
        if (piece_unit)
            for (int i = 0; i < np; ++i) piece_unit[e + i] = u;
        if (heavy && np > 1) heavy[1 + atomicAdd(&heavy[0], 1)] = u;
        e += np;
    }
    if (tid == 1023) {
        piece_start[n] = sa[1023];
        *npieces = sa[1023];
    }
}

// ------------------------------------------------------------ one plan

// Waves per SIMD the spreading kernels are compiled for, by the registers of
// their accumulators: 64 leave room for four, 128 for two, 256 for one.
template <typename T, int NT>
constexpr int strip_waves() { return sizeof(T) * NT == 4 ? 4 : sizeof(T) * NT == 8 ? 2 : 1; }

template <typename T, int NS, int W, bool TALL>
__global__ void __launch_bounds__(kStripLanes *W, (strip_waves<T, 1>()))
    spread_strip_kernel(StripGeom sg, StripPts<T> pts, const int *__restrict__ bin_start,
                        const int *__restrict__ piece_start, const int *__restrict__ npieces,
                        const int *__restrict__ piece_unit, const T *__restrict__ coef, T beta,
                        int horner, int64_t pack_stride, T *__restrict__ scratch,
                        int64_t scratch_stride) {
    __shared__ StripLds<T, NS, 1, TALL> lds[W];
    pts.pack += 4 * pack_stride * blockIdx.y;
    scratch += 2 * scratch_stride * blockIdx.y;
    const int64_t tile_cells = (int64_t)(sg.H + NS - 1) * kStripLanes;
    const int piece = blockIdx.x;  // one workgroup per piece
    if (piece >= *npieces) return;
    const int u = piece_unit[piece];
    strip_piece<T, NS, 1, W, TALL>(sg, pts, bin_start, u, piece - piece_start[u], coef, beta,
                                   horner, scratch + 2 * piece * tile_cells, 0, lds);
}

// pack[t][j] = (c[t][j], rec[j])
template <typename T>
__global__ void __launch_bounds__(256)
    strip_pack_kernel(const T *__restrict__ c, int64_t c_stride, const T *__restrict__ rec,
                      int64_t M, T *__restrict__ pack) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= M) return;
    const Pair<T> cv = reinterpret_cast<const Pair<T> *>(c + 2 * c_stride * blockIdx.y)[j];
    const Pair<T> tv = reinterpret_cast<const Pair<T> *>(rec)[j];
    reinterpret_cast<Quad<T> *>(pack + 4 * M * blockIdx.y)[j] = Quad<T>{cv.x, cv.y, tv.x, tv.y};
}

// 3D: pack[t][j * ns + dz] = (c[t][j] * kz_j[dz], tx_j, ty_j), with the
// z-weights evaluated here from tz_j (rec3[3j .. 3j+2] = tx, ty, tz).
template <typename T, int NS>
__global__ void __launch_bounds__(256)
    strip3_pack_kernel(const T *__restrict__ c, int64_t c_stride, const T *__restrict__ rec3,
                       const T *__restrict__ coef, T beta, int horner, int64_t M,
                       T *__restrict__ pack) {
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= M) return;
    const Pair<T> cv = reinterpret_cast<const Pair<T> *>(c + 2 * c_stride * blockIdx.y)[j];
    const T tx = rec3[3 * j], ty = rec3[3 * j + 1], tz = rec3[3 * j + 2];
    T kz[NS];
    if (horner)
        eval_kernel<T, NS, true>(coef, beta, tz, kz);
    else
        eval_kernel<T, NS, false>(coef, beta, tz, kz);
    Quad<T> *out = reinterpret_cast<Quad<T> *>(pack + 4 * NS * M * blockIdx.y) + j * NS;
#pragma unroll
    for (int dz = 0; dz < NS; ++dz) out[dz] = Quad<T>{cv.x * kz[dz], cv.y * kz[dz], tx, ty};
}

template <typename T, int NS>
__global__ void __launch_bounds__(256)
    strip_merge_kernel(StripGeom sg, const int *__restrict__ piece_start,
                       const T *__restrict__ scratch, int64_t scratch_stride, T *__restrict__ fw,
                       int64_t fw_stride, int reduced) {
    merge_unit<T, NS>(sg, piece_start, scratch + 2 * scratch_stride * blockIdx.y,
                      fw + 2 * fw_stride * blockIdx.y, (int)blockIdx.x, reduced);
}

// Piece table of one plan's units in three launches (counts with per-block
// sums, a scan of the block sums, block-local scans), for the many units of
// 3D grids; see the ragged form below.
__global__ void __launch_bounds__(256)
    strip_units_count_kernel(StripGeom sg, const int *__restrict__ bin_start, int *piece_start,
                             int *blocksum);
__global__ void __launch_bounds__(1024)
    strip_units_blocks_kernel(int nu, int nblk, const int *__restrict__ blocksum, int *blockoff,
                              int *piece_start, int *npieces, int *heavy);
// The same in one launch of one workgroup, for few units.
constexpr int kSmallUnits = 4096;
__global__ void __launch_bounds__(1024)
    strip_units_small_kernel(StripGeom sg, const int *__restrict__ bin_start, int *piece_start,
                             int *npieces, int *piece_unit, int *heavy) {
    piece_scan(
        sg.nunits, [&](int u) { return unit_pieces(sg, bin_start, u); }, piece_start, npieces,
        piece_unit, heavy);
}
__global__ void __launch_bounds__(256)
    strip_units_scan_kernel(int nu, const int *__restrict__ blockoff, int *piece_start,
                            int *piece_unit, int *heavy);

// Sum the tiles of every piece of a crowded unit into its first piece's tile
// (in piece order), so that the merge reads one tile per unit; work items
// (unit, 256-cell chunk of the tile) over a fixed grid.  Eight tiles' loads in flight:
// a point cluster in few units leaves few workgroups to hide them (1e7 points, almost all
// within 16 cells square, 4006 pieces: 794 us one by one, 195 so).
template <typename T, int NS>
__global__ void __launch_bounds__(256)
    strip_reduce_kernel(StripGeom sg, const int *__restrict__ piece_start,
                        const int *__restrict__ heavy, T *__restrict__ scratch,
                        int64_t scratch_stride) {
    scratch += 2 * scratch_stride * blockIdx.y;
    const int64_t tile_cells = (int64_t)(sg.H + NS - 1) * kStripLanes;
    const int chunks = (int)((tile_cells + 255) / 256);
    const int items = heavy[0] * chunks;
    Pair<T> *tiles = reinterpret_cast<Pair<T> *>(scratch);
    for (int w = blockIdx.x; w < items; w += gridDim.x) {
        const int u = heavy[1 + w / chunks];
        const int64_t cell = (int64_t)(w % chunks) * 256 + threadIdx.x;
        if (cell >= tile_cells) continue;
        const int first = piece_start[u], cnt = piece_start[u + 1] - first;
        Pair<T> acc = tiles[first * tile_cells + cell];
#pragma unroll 8
        for (int pc = 1; pc < cnt; ++pc) {
            const Pair<T> v = tiles[(first + pc) * tile_cells + cell];
            acc.x += v.x;
            acc.y += v.y;
        }
        tiles[first * tile_cells + cell] = acc;
    }
}

// ------------------------------------------------------------ ragged batch
//
// Virtual problem v = (problem, transform).  Its units are the global units
// [vunit_off[v], vunit_off[v+1]); its points are its problem's, found through
// the problem's slice of the global bins; its fine grid and scratch tiles are
// slices of the concatenated buffers; its strengths come from the pointer
// table (c of problem i at ptrs[2*nprob + i], transform-major).

// Piece table of every virtual problem's units in three launches: counts and
// per-block sums, a scan of the block sums, then the block-local scans.
__device__ __forceinline__ int ragged_unit_pieces(const RaggedVirt *__restrict__ virt,
                                                  const int *__restrict__ unit_virt,
                                                  const int *__restrict__ bin_start, int gu) {
    const int v = unit_virt[gu];
    const RaggedVirt &d = virt[v];
    return unit_pieces(d.sg, bin_start + d.bin_off, gu - d.unit_off);
}

// exclusive scan of one value per thread over a 256-thread block; returns the
// block total in *total.  sa[t] holds the inclusive sums afterwards.
__device__ __forceinline__ int block_scan256(int v, int *total, int *sa) {
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
    return sa[tid] - v;
}

// The units of a 256-unit block's pieces, the block's threads over the pieces (a crowded
// unit has thousands; the call above, scan kernel 125 us with a thread per unit, 7 so):
// piece_unit[first + i] = u0 + t for the t with sa[t - 1] <= i < sa[t].
__device__ __forceinline__ void write_piece_units(const int *sa, int total, int u0, int first,
                                                  int *piece_unit) {
    for (int i = threadIdx.x; i < total; i += 256) {
        int lo = 0;
#pragma unroll
        for (int step = 128; step > 0; step >>= 1)
            if (sa[lo + step - 1] <= i) lo += step;
        piece_unit[first + i] = u0 + lo;
    }
}

__global__ void __launch_bounds__(256)
    strip_units_count_kernel(StripGeom sg, const int *__restrict__ bin_start, int *piece_start,
                             int *blocksum) {
    const int u = blockIdx.x * 256 + threadIdx.x;
    const int c = u < sg.nunits ? unit_pieces(sg, bin_start, u) : 0;
    if (u < sg.nunits) piece_start[u] = c;
    int total;
    __shared__ int sa[256];
    block_scan256(c, &total, sa);
    if (threadIdx.x == 0) blocksum[blockIdx.x] = total;
}

__global__ void __launch_bounds__(1024)
    strip_units_blocks_kernel(int nu, int nblk, const int *__restrict__ blocksum, int *blockoff,
                              int *piece_start, int *npieces, int *heavy) {
    piece_scan(
        nblk, [&](int b) { return blocksum[b]; }, blockoff, npieces, nullptr, nullptr);
    if (threadIdx.x == 1023) piece_start[nu] = blockoff[nblk];
    if (threadIdx.x == 0) heavy[0] = 0;  // the scan kernel that follows appends to it
}

__global__ void __launch_bounds__(256)
    strip_units_scan_kernel(int nu, const int *__restrict__ blockoff, int *piece_start,
                            int *piece_unit, int *heavy) {
    const int u = blockIdx.x * 256 + threadIdx.x;
    const int c = u < nu ? piece_start[u] : 0;
    int total;
    __shared__ int sa[256];
    const int e = block_scan256(c, &total, sa);
    const int first = blockoff[blockIdx.x];
    if (u < nu) {
        piece_start[u] = first + e;
        if (c > 1) heavy[1 + atomicAdd(&heavy[0], 1)] = u;
    }
    write_piece_units(sa, total, blockIdx.x * 256, first, piece_unit);
}

__global__ void __launch_bounds__(256)
    ragged_units_count_kernel(const RaggedVirt *__restrict__ virt,
                              const int *__restrict__ vunit_off,
                              const int *__restrict__ unit_virt, int nv,
                              const int *__restrict__ bin_start, int *piece_start,
                              int *blocksum) {
    const int nu = vunit_off[nv];
    const int gu = blockIdx.x * 256 + threadIdx.x;
    const int c = gu < nu ? ragged_unit_pieces(virt, unit_virt, bin_start, gu) : 0;
    if (gu < nu) piece_start[gu] = c;
    int total;
    __shared__ int sa[256];
    block_scan256(c, &total, sa);
    if (threadIdx.x == 0) blocksum[blockIdx.x] = total;
}

// one workgroup: blockoff = exclusive scan of the nblk block sums (nblk + 1
// entries); total also at piece_start[nu] and *npieces
__global__ void __launch_bounds__(1024)
    ragged_units_blocks_kernel(const int *__restrict__ vunit_off, int nv, int nblk,
                               const int *__restrict__ blocksum, int *blockoff,
                               int *piece_start, int *npieces, int *heavy) {
    piece_scan(
        nblk, [&](int b) { return blocksum[b]; }, blockoff, npieces, nullptr, nullptr);
    if (threadIdx.x == 0) heavy[0] = 0;  // the scan kernel that follows appends to it
    if (threadIdx.x == 1023) piece_start[vunit_off[nv]] = blockoff[nblk];
}

__global__ void __launch_bounds__(256)
    ragged_units_scan_kernel(const int *__restrict__ vunit_off, int nv,
                             const int *__restrict__ blockoff, int *piece_start,
                             int *piece_unit, int *heavy) {
    const int nu = vunit_off[nv];
    const int gu = blockIdx.x * 256 + threadIdx.x;
    const int c = gu < nu ? piece_start[gu] : 0;
    int total;
    __shared__ int sa[256];
    const int e = block_scan256(c, &total, sa);
    const int first = blockoff[blockIdx.x];
    if (gu < nu) {
        piece_start[gu] = first + e;
        if (c > 1) heavy[1 + atomicAdd(&heavy[0], 1)] = gu;
    }
    write_piece_units(sa, total, blockIdx.x * 256, first, piece_unit);
}

// Waves per piece.  Problems of all densities fill the GPU together: 64 problems of
// up to 2e6 points, 1 to 8 transforms: the batch takes 4.70 ms, with four 6.03.
constexpr int kRaggedWaves = 1;
// Transforms of a problem that a wave spreads together: two in fp32, whose weights are
// then staged once.  Two in fp64 would hold 256 registers of accumulators and leave one
// wave a SIMD: 8 problems of 1e6 to 4e6 points, up to 6 transforms, w = 8 4.22 -> 3.40 ms a
// batch with one, 64 of 1e4 to 2e6 7.05 -> 6.00, w = 16 13.0 -> 11.3.
template <typename T, int NS, bool TALL>
__global__ void __launch_bounds__(kStripLanes *kRaggedWaves,
                                  (strip_waves<T, ragged_transforms(sizeof(T))>()))
    ragged_strip_kernel(const RaggedVirt *__restrict__ virt, const int *__restrict__ unit_virt,
                        StripPts<T> pts, const int *__restrict__ bin_start,
                        const int *__restrict__ piece_start, const int *__restrict__ npieces,
                        const int *__restrict__ piece_unit,
                        const T *__restrict__ coef, T beta, int horner,
                        const void *const *__restrict__ ptrs, int nprob,
                        T *__restrict__ scratch_all) {
    constexpr int NT = ragged_transforms(sizeof(T));
    __shared__ StripLds<T, NS, NT, TALL> lds[kRaggedWaves];
    const int piece = blockIdx.x;  // one workgroup per piece
    if (piece >= *npieces) return;
    const int gu = piece_unit[piece];
    const int v = unit_virt[gu];
    const RaggedVirt d = virt[v];
    if (d.nt == 0) return;  // spread together with transform t - 1
    const int sub = piece - piece_start[gu];
    StripPts<T> vp = pts;
    vp.c = (const T *)ptrs[2 * nprob + d.prob] + 2 * (int64_t)d.t * d.m;
    vp.c_tstride = 2 * d.m;
    vp.bin_off = d.bin_off;
    vp.idx_off = d.moff;
    const int64_t tile_cells = (int64_t)(d.sg.H + NS - 1) * kStripLanes;
    T *tile = scratch_all + 2 * (d.tile_off + (piece - piece_start[d.unit_off]) * tile_cells);
    if (NT > 1 && d.nt > 1)
        strip_piece<T, NS, NT, kRaggedWaves, TALL>(d.sg, vp, bin_start + d.bin_off,
                                                   gu - d.unit_off, sub, coef, beta, horner, tile,
                                                   2 * d.tile_next, lds);
    else
        strip_piece<T, NS, 1, kRaggedWaves, TALL>(d.sg, vp, bin_start + d.bin_off,
                                                  gu - d.unit_off, sub, coef, beta, horner, tile, 0,
                                                  reinterpret_cast<StripLds<T, NS, 1, TALL> *>(lds));
}

// Ragged form of strip_reduce_kernel: heavy lists global units.
template <typename T, int NS>
__global__ void __launch_bounds__(256)
    ragged_reduce_kernel(const RaggedVirt *__restrict__ virt, const int *__restrict__ unit_virt,
                         const int *__restrict__ piece_start, const int *__restrict__ heavy,
                         int chunks, T *__restrict__ scratch_all) {
    const int items = heavy[0] * chunks;
    for (int w = blockIdx.x; w < items; w += gridDim.x) {
        const int gu = heavy[1 + w / chunks];
        const RaggedVirt &d = virt[unit_virt[gu]];
        const int64_t tile_cells = (int64_t)(d.sg.H + NS - 1) * kStripLanes;
        const int64_t cell = (int64_t)(w % chunks) * 256 + threadIdx.x;
        if (cell >= tile_cells) continue;
        Pair<T> *tiles = reinterpret_cast<Pair<T> *>(scratch_all + 2 * d.tile_off);
        const int first = piece_start[gu] - piece_start[d.unit_off];
        const int cnt = piece_start[gu + 1] - piece_start[gu];
        Pair<T> acc = tiles[first * tile_cells + cell];
#pragma unroll 8
        for (int pc = 1; pc < cnt; ++pc) {
            const Pair<T> v = tiles[(first + pc) * tile_cells + cell];
            acc.x += v.x;
            acc.y += v.y;
        }
        tiles[first * tile_cells + cell] = acc;
    }
}

// block b merges global unit b (unit b - unit_off of its virtual problem)
template <typename T, int NS>
__global__ void __launch_bounds__(256)
    ragged_merge_kernel(const RaggedVirt *__restrict__ virt, const int *__restrict__ unit_virt,
                        const int *__restrict__ piece_start, const T *__restrict__ scratch_all,
                        T *__restrict__ fw_all) {
    const int gu = (int)blockIdx.x;
    const int v = unit_virt[gu];
    const RaggedVirt d = virt[v];
    merge_unit<T, NS>(d.sg, piece_start + d.unit_off, scratch_all + 2 * d.tile_off,
                      fw_all + 2 * d.fw_off, gu - d.unit_off, 1);
}

}  // namespace

// A launch of strip_reduce_kernel is worth about this many pieces read in series
// by one merge workgroup.
constexpr int kMergePieces = 16;

template <typename T>
int launch_spread_strip(const StripGeom &sg, const StripPts<T> &pts, const int *bin_start,
                        int *piece_start, int *npieces, int *piece_unit, int *heavy,
                        int *blocksum, const T *coef, int kerevalmeth, double beta,
                        int64_t pack_stride, T *fw,
                        int64_t fw_stride, T *scratch, int64_t scratch_stride, int ntr,
                        int phases, hipStream_t stream) {
    if (ntr == 0 || pts.M == 0) return JFA_OK;
    if ((phases & kStripUnits) && sg.nunits <= kSmallUnits) {
        // 24 units (4000-point call): 3 launches 8.8 us, one 3.6 us; 9216 units:
        // 13.1 against 15.9 us
        strip_units_small_kernel<<<1, 1024, 0, stream>>>(sg, bin_start, piece_start, npieces,
                                                         piece_unit, heavy);
        JFA_HIP_CHECK(hipGetLastError());
    } else if (phases & kStripUnits) {
        const unsigned nblk = (unsigned)((sg.nunits + 255) / 256);
        int *blockoff = blocksum + nblk;  // nblk + 1 entries
        strip_units_count_kernel<<<nblk, 256, 0, stream>>>(sg, bin_start, piece_start, blocksum);
        strip_units_blocks_kernel<<<1, 1024, 0, stream>>>(sg.nunits, (int)nblk, blocksum,
                                                          blockoff, piece_start, npieces, heavy);
        strip_units_scan_kernel<<<nblk, 256, 0, stream>>>(sg.nunits, blockoff, piece_start,
                                                          piece_unit, heavy);
        JFA_HIP_CHECK(hipGetLastError());
    }
    // one workgroup per piece (see launch_ragged_strip); 3D slice grids have
    // tens of thousands of units
    const int64_t ub = strip_max_pieces(sg, pts.M);
    if (ub > UINT32_MAX / kStripLanes) {  // threads of a launch
        set_error("%lld strip pieces are too many for one launch", (long long)ub);
        return JFA_ERR_TOO_LARGE;
    }
    const unsigned grid = (unsigned)ub;
    // Waves per piece: four fill the GPU where units are few, and level the last round
    // where they hold many points or the points crowd; with many units of fewer points one
    // wave does less work (a tile to sum instead of four).  Even units' points, and where
    // the line lies: w = 8 in fp32, one wave / four, uniform points: 737 units of 271 points
    // 21 / 16 us, 2052 of 292 30 / 32, of 585 51 / 46, 8208 of 487 111 / 128, of 1219 276 /
    // 263, 37,120 of 216 217 / 350; normal about the centre: 2052 of 487 58 / 40, 8208 of 365
    // 91 / 97, of 731 175 / 168; w = 5, 3073 of 375, the whole call 171 / 175.  fp64 kernels hold half as many waves and are bound by their
    // products sooner (w = 8: 2052 of 585 82 / 88, of 1170 153 / 137; 5760 of 417 138 / 156,
    // of 1389 427 / 403; w = 11: 3572 of 560 238 / 283, of 1120 442 / 468).
    const int64_t even = std::min<int64_t>(pts.M / sg.nunits, sg.pmax);
    const int64_t line = std::min<int64_t>(
        std::max<int64_t>((int64_t)sg.nunits * ntr / (sizeof(T) == 4 ? 6 : 5), 128),
        sizeof(T) == 4 ? 700 : sg.ns <= 8 ? 2048 : 1024);
    constexpr int kPieceWaves = 4;
    const bool tall = sg.H > strip_short_rows(sg.ns);
    const int waves =
        !tall && even >= line && ub <= UINT32_MAX / (kStripLanes * kPieceWaves) ? kPieceWaves : 1;
    const T b = (T)beta;
    JFA_DISPATCH_NS(sg.ns, {
        if (phases & kStripSpread) {
            auto kernel = waves > 1 ? spread_strip_kernel<T, NS_, kPieceWaves, false>
                          : tall    ? spread_strip_kernel<T, NS_, 1, true>
                                    : spread_strip_kernel<T, NS_, 1, false>;
            kernel<<<dim3(grid, ntr), kStripLanes * waves, 0, stream>>>(
                sg, pts, bin_start, piece_start, npieces, piece_unit, coef, b, kerevalmeth,
                pack_stride, scratch, scratch_stride);
        }
        // few pieces in all: the merge sums a crowded unit's itself
        const int reduced = pts.M / sg.pmax > kMergePieces;
        if ((phases & kStripMerge) && reduced) {
            const int64_t rb = strip_max_heavy(sg, pts.M) *
                               ((strip_tile_cells(sg) + 255) / 256);
            strip_reduce_kernel<T, NS_>
                <<<dim3((unsigned)(rb < 2048 ? rb : 2048), ntr), 256, 0, stream>>>(
                    sg, piece_start, heavy, scratch, scratch_stride);
        }
        if (phases & kStripMerge)
            // two waves per unit: units are 8 rows or more (256 threads: 0.044 vs
            // 0.0415 ms at the 2048^2 bench size, 0.063 vs 0.056 ms clustered)
            strip_merge_kernel<T, NS_><<<dim3((unsigned)sg.nunits, ntr), 128, 0, stream>>>(
                    sg, piece_start, scratch, scratch_stride, fw, fw_stride, reduced);
    });
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int launch_ragged_strip(const RaggedLaunch &rl, const StripPts<T> &pts, const T *coef,
                        int kerevalmeth, double beta, T *fw_all, T *scratch_all, int phases,
                        hipStream_t stream) {
    // no points anywhere: the caller zeroes the fine grids instead
    if (rl.nv == 0 || pts.M == 0) return JFA_OK;
    if (phases & kStripUnits) {
        const unsigned nblk = (unsigned)((rl.nunits + 255) / 256);
        ragged_units_count_kernel<<<nblk, 256, 0, stream>>>(rl.virt, rl.vunit_off, rl.unit_virt,
                                                            rl.nv, rl.bin_start, rl.piece_start,
                                                            rl.blocksum);
        int *blockoff = rl.blocksum + nblk;  // nblk + 1 entries
        ragged_units_blocks_kernel<<<1, 1024, 0, stream>>>(rl.vunit_off, rl.nv, (int)nblk,
                                                           rl.blocksum, blockoff,
                                                           rl.piece_start, rl.npieces, rl.heavy);
        ragged_units_scan_kernel<<<nblk, 256, 0, stream>>>(rl.vunit_off, rl.nv, blockoff,
                                                           rl.piece_start, rl.piece_unit,
                                                           rl.heavy);
        JFA_HIP_CHECK(hipGetLastError());
    }
    // one workgroup per piece (the kernel does not loop): piece costs differ by
    // problem density, and the hardware dispatcher balances them as waves finish, where a capped grid
    // looping over pieces fixes each workgroup's share up front (64-problem
    // benchmark batch: 4.97 vs 5.31 ms)
    const int64_t ub = ragged_strip_blocks(rl);
    if (ub > UINT32_MAX / (kStripLanes * kRaggedWaves)) {  // threads of a launch
        set_error("%lld strip pieces are too many for one launch", (long long)ub);
        return JFA_ERR_TOO_LARGE;
    }
    const unsigned grid = (unsigned)ub;
    const T b = (T)beta;
    JFA_DISPATCH_NS(rl.ns, {
        if (phases & kStripSpread) {
            auto kernel = rl.tall ? ragged_strip_kernel<T, NS_, true>
                                  : ragged_strip_kernel<T, NS_, false>;
            kernel<<<grid, kStripLanes * kRaggedWaves, 0, stream>>>(
                rl.virt, rl.unit_virt, pts, rl.bin_start, rl.piece_start, rl.npieces,
                rl.piece_unit, coef, b, kerevalmeth, rl.ptrs, rl.nprob, scratch_all);
        }
        if (phases & kStripMerge) {
            const int64_t rb = rl.max_heavy * rl.reduce_chunks;
            ragged_reduce_kernel<T, NS_><<<(unsigned)(rb < 2048 ? rb : 2048), 256, 0, stream>>>(
                rl.virt, rl.unit_virt, rl.piece_start, rl.heavy, rl.reduce_chunks, scratch_all);
        }
        if (phases & kStripMerge)
            ragged_merge_kernel<T, NS_><<<(unsigned)rl.nunits, 64, 0, stream>>>(
                rl.virt, rl.unit_virt, rl.piece_start, scratch_all, fw_all);
    });
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int launch_strip3_pack(const T *c, int64_t c_stride, const T *rec3, const T *coef,
                       int kerevalmeth, double beta, int ns, int64_t M, int ntr, T *pack,
                       hipStream_t stream) {
    if (M == 0 || ntr == 0) return JFA_OK;
    const dim3 grid((unsigned)((M + 255) / 256), ntr);
    const T b = (T)beta;
    JFA_DISPATCH_NS(ns, strip3_pack_kernel<T, NS_><<<grid, 256, 0, stream>>>(
                            c, c_stride, rec3, coef, b, kerevalmeth, M, pack));
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

template <typename T>
int launch_strip_pack(const T *c, int64_t c_stride, const T *rec, int64_t M, int ntr, T *pack,
                      hipStream_t stream) {
    if (M == 0 || ntr == 0) return JFA_OK;
    strip_pack_kernel<T><<<dim3((unsigned)((M + 255) / 256), ntr), 256, 0, stream>>>(
        c, c_stride, rec, M, pack);
    JFA_HIP_CHECK(hipGetLastError());
    return JFA_OK;
}

#define JFA_INST(T)                                                                           \
    template int launch_spread_strip<T>(const StripGeom &, const StripPts<T> &, const int *, \
                                        int *, int *, int *, int *, int *, const T *, int,    \
                                        double, int64_t, T *, int64_t, T *, int64_t, int, int, \
                                        hipStream_t);                                         \
    template int launch_strip3_pack<T>(const T *, int64_t, const T *, const T *, int, double, \
                                       int, int64_t, int, T *, hipStream_t);                  \
    template int launch_strip_pack<T>(const T *, int64_t, const T *, int64_t, int, T *,       \
                                      hipStream_t);                                           \
    template int launch_ragged_strip<T>(const RaggedLaunch &, const StripPts<T> &, const T *, \
                                        int, double, T *, T *, int, hipStream_t);
JFA_INST(float)
JFA_INST(double)
#undef JFA_INST

}  // namespace jfa
