// Plan interface of the MI355X NUFFT backend: makeplan / setpts / execute /
// destroy.  Replaces the cuFINUFFT plan the reference builds through
// lib/cufinufft_wrapper.cc:48-99 (makeplan/setpts/execute/destroy shims) and
// drives from run_nufft (lib/kernels.cc.cu:25-92).
//
// Differences by design:
//  * all work is queued on the plan's stream; the host never waits (the
//    reference synchronises at lib/kernels.cc.cu:83);
//  * scratch is owned by the plan and grown only when a larger point count
//    arrives, so a cached plan re-used across calls allocates nothing;
//  * rocFFT plans are made once per batch size and reused.
#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "jfa_internal.hpp"
#include "plan_state.hpp"

using namespace jfa;

namespace {
std::once_flag g_rocfft_once;
int g_rocfft_status = 0;
}  // namespace

std::mutex &jfa::rocfft_mutex() {
    static std::mutex mu;
    return mu;
}

int jfa::ensure_rocfft() {
    std::call_once(g_rocfft_once, [] {
        g_rocfft_status = rocfft_setup() == rocfft_status_success ? 0 : 1;
    });
    if (g_rocfft_status) {
        set_error("rocfft_setup failed");
        return JFA_ERR_FFT;
    }
    return JFA_OK;
}

namespace {

template <typename T>
int upload(const std::vector<double> &h, void **d) {
    std::vector<T> tmp(h.begin(), h.end());
    JFA_HIP_CHECK(hipMalloc(d, sizeof(T) * std::max<size_t>(tmp.size(), 1)));
    JFA_HIP_CHECK(hipMemcpy(*d, tmp.data(), sizeof(T) * tmp.size(), hipMemcpyHostToDevice));
    return JFA_OK;
}

void free_ptr(void *&p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}

// Bin sizes: 2D 32x32 and 1D 1024 cells; 3D 8x8x8.  Each is clamped to half
// the fine grid so that a tile origin plus its extent wraps at most once.  In
// 3D the smaller tile (14^3 cells at w = 7) keeps more workgroups resident than
// 16x16x8 (22x22x14): 3D type 2, fp32, measured 4.8 vs 6.3 ms (16.7M koosh-ball
// points, 256^3 modes), 2.35 vs 2.83 ms and 5.2 vs 6.1 ms (1e7 uniform points,
// 128^3 / 256^3 modes), 2.7 vs 4.3 ms (2e6 points, 256^3).
void default_bins(jfa_plan p) {
    int b[3] = {1, 1, 1};
    if (p->dim == 1) b[0] = 1024;
    if (p->dim == 2) {
        b[0] = b[1] = 32;
        // Interpolation: 64 x 64 bins where that still leaves at least 1024 bins
        // and the LDS tile fits in 64 KiB: each workgroup then works through
        // four times the points (with the subproblem size of default_maxsub).
        // Coarser grids keep 32 x 32, whose 1024 or fewer bins already leave
        // few workgroups per CU (4e6 points on 1024^2: 64 x 64 measured 0.137
        // vs 0.113 ms).
        const GridGeom &g = p->geom;
        const int64_t tile = (int64_t)(64 + g.ns - 1) * (64 + g.ns - 1) * 2 * (p->is_double ? 8 : 4);
        if (p->type == 2 && (g.nf[0] / 64) * (g.nf[1] / 64) >= 1024 && tile <= 64 * 1024)
            b[0] = b[1] = 64;
    }
    // 3D: 8^3 bins; interpolation takes bins twice as deep in z (LDS tiles of
    // 14 x 14 x 22 cells at w = 7 cost fewer halo cells per point: koosh-ball
    // type 2, 16.7M points on 512^3, 3.48 -> 3.29 ms per setpts + execute)
    if (p->dim == 3) {
        b[0] = b[1] = b[2] = 8;
        if (p->type == 2) b[2] = 16;
    }
    const int o[3] = {p->opts.gpu_binsizex, p->opts.gpu_binsizey, p->opts.gpu_binsizez};
    GridGeom &g = p->geom;
    g.nbins = 1;
    for (int d = 0; d < 3; ++d) {
        int bs = d < p->dim ? (o[d] > 0 ? o[d] : b[d]) : 1;
        if (d < p->dim) {
            int64_t cap = std::max<int64_t>(1, g.nf[d] / 2);
            if (bs > cap) bs = (int)cap;
        }
        g.bs[d] = bs;
        g.nb[d] = (int)((g.nf[d] + bs - 1) / bs);
        g.nbins *= g.nb[d];
    }
}

size_t tile_lds_bytes(jfa_plan p) {
    size_t cells = 1;
    for (int d = 0; d < p->dim; ++d) cells *= (size_t)(p->geom.bs[d] + p->geom.ns - 1);
    return cells * 2 * (p->is_double ? 8 : 4);
}

int resolve_method(jfa_plan p) {
    const size_t kMaxTileLds = 64 * 1024;
    int m = p->opts.gpu_method;
    const bool spreads = p->type != 2;
    if (m == JFA_METHOD_STRIP || (m == JFA_METHOD_AUTO && spreads && strip_applicable(p))) {
        if (spreads) {
            if (!strip_applicable(p) || (m == JFA_METHOD_STRIP && p->geom.nf[0] < 64)) {
                set_error("the strip method needs a 2D or 3D grid of at least 64 x %d (x %d) "
                          "cells", 2 * p->geom.ns, 2 * p->geom.ns);
                return -1;
            }
            return JFA_METHOD_STRIP;
        }
        m = JFA_METHOD_SM;  // interpolation has no strip variant
    }
    if (m == JFA_METHOD_AUTO) m = tile_lds_bytes(p) <= kMaxTileLds ? JFA_METHOD_SM : JFA_METHOD_GM_SORT;
    // an explicit LDS request with a wide kernel: halve the largest bin until
    // the tile fits
    while (m == JFA_METHOD_SM && tile_lds_bytes(p) > kMaxTileLds) {
        GridGeom &g = p->geom;
        int dmax = 0;
        for (int d = 1; d < p->dim; ++d)
            if (g.bs[d] > g.bs[dmax]) dmax = d;
        if (g.bs[dmax] <= 1) break;
        g.bs[dmax] = (g.bs[dmax] + 1) / 2;
        g.nbins = 1;
        for (int d = 0; d < 3; ++d) {
            g.nb[d] = (int)((g.nf[d] + g.bs[d] - 1) / g.bs[d]);
            g.nbins *= g.nb[d];
        }
    }
    if (m == JFA_METHOD_SM && tile_lds_bytes(p) > kMaxTileLds) {
        set_error("LDS subproblem tile of %zu bytes exceeds 64 KiB; use smaller bins or "
                  "gpu_method=1", tile_lds_bytes(p));
        return -1;
    }
    if (m != JFA_METHOD_SM && m != JFA_METHOD_GM_SORT) {
        set_error("gpu_method must be 0, 1 or 2 (got %d)", m);
        return -1;
    }
    return m;
}

struct DeviceGuard {
    int prev = -1;
    bool changed = false;
    int set(int dev) {
        if (dev < 0) return JFA_OK;
        JFA_HIP_CHECK(hipGetDevice(&prev));
        if (prev != dev) {
            JFA_HIP_CHECK(hipSetDevice(dev));
            changed = true;
        }
        return JFA_OK;
    }
    ~DeviceGuard() {
        if (changed) (void)hipSetDevice(prev);
    }
};

}  // namespace

// ------------------------------------------------------------------ strips

// Grids of fewer columns than a strip's 64 use part of the tile and are still far
// faster here than with float atomics in LDS tiles: whole calls of 200,000 points on
// 24^3 modes 1302 -> 176 us (fp32, 7 digits), 9260 -> 577 (fp64, 9 digits); 300,000
// on 31^2 319 -> 136 (fp32); 10,000 on 16 x 24 145 -> 122 (fp64, 9 digits).  Their
// tiles are up to seven times the grid, so only up to kNarrowRows rows (at most 2 GB
// of tiles in fp32, 4 in fp64 for one transform).
static constexpr int64_t kNarrowRows = 1 << 20;
// And only up to this much memory for keys, records and tiles, which in
// 3D are w times the points (fp32 at w = 8: 16.7 million points).
static constexpr size_t kNarrowBytes = (size_t)8 << 30;
bool jfa::strip_applicable(jfa_plan p) {
    const GridGeom &g = p->geom;
    if (p->dim < 2 || g.nf[0] < 2 * g.ns || g.nf[1] < 2 * g.ns) return false;
    if (p->dim == 3 && g.nf[2] < 2 * g.ns) return false;
    if (g.nf[0] < 64 && g.nf[1] * g.nf[2] > kNarrowRows) return false;
    // (slice, strip, row) bins shifted by the column bits must fit 32-bit sort keys
    const int64_t strips = (g.nf[0] + 64 - g.ns) / (64 - g.ns + 1);
    const int64_t nz = p->dim == 3 ? g.nf[2] : 1;
    return ((nz * strips * g.nf[1] + 1) << kStripKeyShift) <= (int64_t)UINT32_MAX;
}

jfa::StripGeom jfa::strip_geometry(GridGeom &g, int pmax) {
    StripGeom sg{};
    const int ns = g.ns;
    sg.nf0 = g.nf[0];
    sg.nf1 = g.nf[1];
    sg.ns = ns;
    sg.nz = g.dim == 3 ? (int)g.nf[2] : 1;
    sg.SW = 64 - ns + 1;
    sg.S = (int)((g.nf[0] + sg.SW - 1) / sg.SW);
    strip_set_rows(sg, strip_short_rows(ns));
    sg.pmax = pmax > 0 ? pmax : kStripPiece;
    // bins: (slice, strip, exact row), rows fastest
    g.bs[0] = sg.SW;
    g.bs[1] = 1;
    g.bs[2] = 1;
    g.nb[0] = sg.S;
    g.nb[1] = (int)g.nf[1];
    g.nb[2] = sg.nz;
    g.nbins = (int64_t)sg.nz * sg.S * g.nf[1];
    g.ymajor = 1;
    g.keyshift = kStripKeyShift;
    return sg;
}

// H within [ns, nf1 - ns + 1], so that a cell is covered by at most two units per axis.
void jfa::strip_set_rows(StripGeom &sg, int64_t rows) {
    int64_t H = std::min<int64_t>(rows, strip_tall_rows(sg.ns));
    H = std::max<int64_t>(std::min<int64_t>(H, sg.nf1 - sg.ns + 1), sg.ns);
    sg.H = (int)H;
    sg.K = (int)((sg.nf1 + H - 1) / H);
    sg.nunits = sg.nz * sg.S * sg.K;
}

// Tall units where the short ones hold few points and are many: a unit writes its whole
// tile and the merge reads it, 2.0 cells per grid cell in short units of ns = 8, 1.4 in
// tall ones, whose products cost twice as much per point and whose waves are fewer, which
// points that crowd make worse.  Points of an even short unit (each slice's counted in 3D),
// short / tall, ns = 8 in fp32, whole calls, uniform points and normal about the centre:
// 48,700 units of 3 252 / 234 and 221 / 216 us, of 24 268 / 252 and 246 / 250; 90,000 of 24
// 602 / 572 and 552 / 558; 16,300 of 3 191 / 177 and 170 / 168, of 24 226 / 214 and 201 / 216;
// 8200 of 8 123 / 117 and 114 / 131; 3D: 15,600 of 24 202 / 185 and 184 / 194, of 64 237 / 229
// and 220 / 244; 52,600 of 24 169 / 146 and 129 / 132, of 64 187 / 171 and 160 / 173, of 192
// 255 / 273 and 251 / 308.  Spreading + merge alone: 131,000 units of 8 826 / 543 us in fp32,
// 1242 / 879 in fp64; 262,000 of 30 1700 / 1349 and 2698 / 2162.  Below two points most short
// units are empty and write nothing (ns = 3 in fp64, 37,000 of one 160 / 197).
//
// ns > 8: short units' tiles are 2.1 (ns = 9) to 2.5 cells per cell, those of 128 rows 1.2
// to 1.5, at the cost of a slower walk.  Spreading + merge, uniform points: 60,000 units of
// 17 at ns = 12 1159 / 1053 us, 33,000 of 31 651 / 689; 81,000 of 12 at ns = 16 1430 / 1150,
// 43,000 of 23 844 / 705, 24,500 of 7 417 / 353, 5082 of 4 90 / 108.  Whole fp64 calls,
// uniform and normal points: ns = 13, 61,500 of 4 1011 / 974 and 888 / 922, ns = 16, 76,800 of
// 4 1087 / 1009 and 930 / 959, of 12 1108 / 1048 and 979 / 1041; ns = 10, 50,600 of 40 1047 /
// 1080 and 990 / 1093; 3D, ns = 16, 21,100 of 64 218 / 260 and 202 / 280.
bool jfa::strip_tall(int ns, double points, double units) {
    const double even = points / units;
    if (even < 2) return false;
    if (ns > 13) return units >= 20000 && even < 32;
    if (ns > 8) return units >= 80000 && even < 24;
    return units >= 12000 && even < std::min(64.0, units / 1500);
}

void jfa::strip_units(StripGeom &sg, int64_t M, int nb, int rows) {
    strip_set_rows(sg, rows > 0 ? rows : strip_short_rows(sg.ns));
    if (rows <= 0 && strip_tall(sg.ns, (double)M * nb, (double)sg.nunits * nb))
        strip_set_rows(sg, strip_tall_rows(sg.ns));
}

int jfa::setup_strip(jfa_plan p) {
    GridGeom &g = p->geom;
    StripGeom &sg = p->sg;
    sg = strip_geometry(g, p->opts.gpu_maxsubprobsize);
    // piece table, for the most units (of ns rows); the tiles are sized by the point count
    // (reserve_strip_scratch)
    const int64_t units = (int64_t)sg.nz * sg.S * ((g.nf[1] + g.ns - 1) / g.ns);
    free_ptr(reinterpret_cast<void *&>(p->d_piece_start));
    JFA_HIP_CHECK(hipMalloc(&p->d_piece_start, sizeof(int) * (units + 1)));
    if (!p->d_npieces) JFA_HIP_CHECK(hipMalloc(&p->d_npieces, sizeof(int) * 4));
    free_ptr(reinterpret_cast<void *&>(p->d_strip_blocksum));
    JFA_HIP_CHECK(hipMalloc(&p->d_strip_blocksum,
                            sizeof(int) * (2 * ((units + 255) / 256) + 2)));
    return JFA_OK;
}

// Buffers of the strip spreader for up to M points and one transform.  Neither the piece
// size (size_chunks) nor the unit height (strip_units) grows evenly with M, and a plan
// that holds the buffers of M points takes fewer without allocating (a captured call must
// not), so this bounds every count up to M: pieces of the most units, and one more per
// piece size, of which size_chunks allows 4096 points, or 256 and at most 4096 pieces of
// the batch or half the units' number (512 pieces of the batch).
struct StripNeed {
    int64_t pieces, heavy;
    size_t tile_bytes, pack_bytes;  // per transform
};
static StripNeed strip_need(jfa_plan p, int64_t M) {
    const size_t real = p->is_double ? 8 : 4;
    const int rows = p->opts.gpu_binsizey;
    const int64_t nb = p->batch;
    StripNeed n{};
    int64_t cells = 0;
    auto add = [&](int64_t height, int64_t most) {
        StripGeom g = p->sg;
        strip_set_rows(g, height);
        int64_t more;
        if (p->opts.gpu_maxsubprobsize > 0) {
            more = most / p->opts.gpu_maxsubprobsize + 1;
        } else {
            more = std::min(std::min(most / 256, 4096 / nb),
                            std::max<int64_t>(g.nunits / 2, 512 / nb));
            more = std::max(most / kStripPiece, more + more / 64) + 2;  // (sizes are rounded)
        }
        const int64_t pieces = std::min<int64_t>(g.nunits, most) + more;
        n.pieces = std::max(n.pieces, pieces);
        n.heavy = std::max(n.heavy, more + 1);
        cells = std::max(cells, pieces * strip_tile_cells(g));
    };
    add(rows > 0 ? rows : strip_short_rows(p->geom.ns), M);
    if (rows <= 0) {
        // tall units, of the counts up to M that they suit
        StripGeom g = p->sg;
        strip_set_rows(g, strip_short_rows(g.ns));
        const int64_t units = g.nunits;
        if (M >= 2 * units && strip_tall(g.ns, 2.0 * units * nb, (double)units * nb))
            add(strip_tall_rows(g.ns), std::min(M, 64 * units));
    }
    n.tile_bytes = (size_t)cells * 2 * real;
    n.pack_bytes = (size_t)M * 4 * real;
    return n;
}

void jfa::release_strip_scratch(jfa_plan p) {
    free_ptr(p->d_strip_scratch);
    free_ptr(p->d_pack);
    p->strip_scratch_bytes = p->pack_bytes = 0;
}

// Tiles for every piece of M points and a record (c, tx, ty) per point, for as many
// transforms at a time as there is memory for, up to `most`.
static int reserve_strip_scratch(jfa_plan p, int64_t M, int most) {
    const StripNeed n = strip_need(p, M);
    p->strip_scratch_stride = strip_max_pieces(p->sg, M) * strip_tile_cells(p->sg);
    if (n.heavy + 1 > p->heavy_cap) {
        free_ptr(reinterpret_cast<void *&>(p->d_heavy));
        p->heavy_cap = 0;
        JFA_HIP_CHECK(hipMalloc(&p->d_heavy, sizeof(int) * (n.heavy + 1)));
        p->heavy_cap = n.heavy + 1;
    }
    if (n.pieces > p->piece_unit_cap) {
        free_ptr(reinterpret_cast<void *&>(p->d_piece_unit));
        p->piece_unit_cap = 0;
        JFA_HIP_CHECK(hipMalloc(&p->d_piece_unit, sizeof(int) * n.pieces));
        p->piece_unit_cap = n.pieces;
    }
    auto grow = [](void *&q, size_t &have, size_t want) {
        if (want <= have) return true;
        free_ptr(q);
        have = 0;
        if (hipMalloc(&q, want) != hipSuccess) {
            (void)hipGetLastError();
            q = nullptr;
            return false;
        }
        have = want;
        return true;
    };
    int k = std::min(most, p->strip_batch_most);
    if (p->geom.nf[0] < 64)
        while (k > 1 && k * (n.tile_bytes + n.pack_bytes) > kNarrowBytes) k = (k + 1) / 2;
    for (bool last = false;;) {
        if (grow(p->d_strip_scratch, p->strip_scratch_bytes, k * n.tile_bytes) &&
            grow(p->d_pack, p->pack_bytes, k * n.pack_bytes)) {
            p->strip_batch = k;
            return JFA_OK;
        }
        release_strip_scratch(p);
        if (k > 1) {
            p->strip_batch_most = k = (k + 1) / 2;
        } else if (!last) {
            // the FFT's buffers are idle while points are spread
            last = true;
            free_ptr(p->d_fwt);
            free_ptr(p->d_fft_work);
            p->fwt_bytes = p->fft_work_bytes = 0;
        } else {
            set_error("could not allocate %zu bytes of strip tiles and records",
                      n.tile_bytes + n.pack_bytes);
            return JFA_ERR_ALLOC;
        }
    }
}

// ------------------------------------------------------------------ fft

// Work buffer large enough for `plan`, shared by all of the plan's FFTs.
static int grow_fft_work(jfa_plan p, rocfft_plan plan) {
    size_t ws = 0;
    rocfft_plan_get_work_buffer_size(plan, &ws);
    if (ws > p->fft_work_bytes) {
        free_ptr(p->d_fft_work);
        p->fft_work_bytes = 0;
        if (hipMalloc(&p->d_fft_work, ws) != hipSuccess) {
            (void)hipGetLastError();
            release_strip_scratch(p);  // idle by now
            JFA_HIP_CHECK(hipMalloc(&p->d_fft_work, ws));
        }
        p->fft_work_bytes = ws;
    }
    return JFA_OK;
}

static int run_fft(jfa_plan p, rocfft_plan plan, void *data) {
    if (!p->fft_info) {
        if (rocfft_execution_info_create(&p->fft_info) != rocfft_status_success) {
            set_error("rocfft_execution_info_create failed");
            return JFA_ERR_FFT;
        }
    }
    rocfft_execution_info_set_stream(p->fft_info, p->stream);
    if (p->fft_work_bytes)
        rocfft_execution_info_set_work_buffer(p->fft_info, p->d_fft_work, p->fft_work_bytes);
    void *bufs[1] = {data};
    rocfft_status st = rocfft_execute(plan, bufs, nullptr, p->fft_info);
    if (st != rocfft_status_success) {
        set_error("rocfft_execute failed (status %d)", (int)st);
        return JFA_ERR_FFT;
    }
    return JFA_OK;
}

int jfa::fft_exec(jfa_plan p, void *data, int nbatch) {
    if (nbatch <= 0) return JFA_OK;
    rocfft_plan plan = nullptr;
    auto it = p->fft_plans.find(nbatch);
    if (it == p->fft_plans.end()) {
        size_t lengths[3];
        for (int d = 0; d < p->dim; ++d) lengths[d] = (size_t)p->geom.nf[d];
        std::lock_guard<std::mutex> lk(rocfft_mutex());
        rocfft_status st = rocfft_plan_create(
            &plan, rocfft_placement_inplace,
            p->iflag > 0 ? rocfft_transform_type_complex_inverse
                         : rocfft_transform_type_complex_forward,
            p->is_double ? rocfft_precision_double : rocfft_precision_single, (size_t)p->dim,
            lengths, (size_t)nbatch, nullptr);
        if (st != rocfft_status_success) {
            set_error("rocfft_plan_create failed (status %d)", (int)st);
            return JFA_ERR_FFT;
        }
        if (int rc = grow_fft_work(p, plan)) {
            rocfft_plan_destroy(plan);
            return rc;
        }
        p->fft_plans[nbatch] = plan;
    } else {
        plan = it->second;
    }
    return run_fft(p, plan, data);
}

int jfa::fft1d(jfa_plan p, void *data, int64_t len, int64_t batch) {
    if (batch <= 0) return JFA_OK;
    const auto key = std::make_pair(len, batch);
    rocfft_plan plan = nullptr;
    auto it = p->fft1_plans.find(key);
    if (it == p->fft1_plans.end()) {
        const size_t lengths[1] = {(size_t)len};
        std::lock_guard<std::mutex> lk(rocfft_mutex());
        rocfft_status st = rocfft_plan_create(
            &plan, rocfft_placement_inplace,
            p->iflag > 0 ? rocfft_transform_type_complex_inverse
                         : rocfft_transform_type_complex_forward,
            p->is_double ? rocfft_precision_double : rocfft_precision_single, 1, lengths,
            (size_t)batch, nullptr);
        if (st != rocfft_status_success) {
            set_error("rocfft_plan_create (1D, length %lld, batch %lld) failed (status %d)",
                      (long long)len, (long long)batch, (int)st);
            return JFA_ERR_FFT;
        }
        if (int rc = grow_fft_work(p, plan)) {
            rocfft_plan_destroy(plan);
            return rc;
        }
        p->fft1_plans[key] = plan;
    } else {
        plan = it->second;
    }
    return run_fft(p, plan, data);
}

// ------------------------------------------------------------------ timing

namespace jfa {
// Per-stage timing on the plan's stream.  debug = 1 prints each call's stages
// to stderr (synchronising); debug = 2 only records event pairs, which
// jfa_plan_timing() resolves later, so timed loops are not perturbed.
struct StageTimer {
    jfa_plan p;
    bool on;
    std::vector<std::pair<const char *, hipEvent_t>> marks;
    explicit StageTimer(jfa_plan pl) : p(pl), on(pl->opts.debug > 0) { mark("start"); }
    ~StageTimer() {
        for (auto &m : marks) (void)hipEventDestroy(m.second);
    }
    void mark(const char *name) {
        if (!on) return;
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
        (void)hipEventRecord(e, p->stream);
        marks.push_back({name, e});
    }
    void report(const char *what) {
        if (!on || marks.size() < 2) return;
        if (p->opts.debug >= 2) {
            for (size_t i = 1; i < marks.size(); ++i)
                p->timing_pairs.push_back({marks[i].first, marks[i - 1].second, marks[i].second});
            for (auto &m : marks) p->timing_events.push_back(m.second);
            marks.clear();
            return;
        }
        (void)hipEventSynchronize(marks.back().second);
        fprintf(stderr, "[jfa %s] type %d, %dd, ntransf=%d, M=%lld:", what, p->type, p->dim,
                p->ntransf, (long long)p->M);
        for (size_t i = 1; i < marks.size(); ++i) {
            float ms = 0;
            (void)hipEventElapsedTime(&ms, marks[i - 1].second, marks[i].second);
            fprintf(stderr, " %s %.4f ms", marks[i].first, ms);
        }
        fprintf(stderr, "\n");
        for (auto &m : marks) (void)hipEventDestroy(m.second);
        marks.clear();
    }
};
}  // namespace jfa

extern "C" int jfa_plan_timing(jfa_plan p, const char *stage, int reset, double *total_ms,
                               int64_t *count) {
    if (!p) {
        set_error("plan is NULL");
        return JFA_ERR_BAD_ARG;
    }
    if (!p->timing_pairs.empty()) {
        JFA_HIP_CHECK(hipEventSynchronize(p->timing_events.back()));
        for (auto &tp : p->timing_pairs) {
            float ms = 0;
            JFA_HIP_CHECK(hipEventElapsedTime(&ms, tp.a, tp.b));
            auto &acc = p->timing_acc[tp.name];
            acc.first += ms;
            acc.second += 1;
        }
        for (hipEvent_t e : p->timing_events) (void)hipEventDestroy(e);
        p->timing_pairs.clear();
        p->timing_events.clear();
    }
    double t = 0;
    int64_t n = 0;
    if (stage) {
        auto it = p->timing_acc.find(stage);
        if (it != p->timing_acc.end()) {
            t = it->second.first;
            n = it->second.second;
        }
    }
    if (total_ms) *total_ms = t;
    if (count) *count = n;
    if (reset) p->timing_acc.clear();
    return JFA_OK;
}

// ------------------------------------------------------------------ plan API

extern "C" void jfa_default_opts(jfa_opts *o) {
    std::memset(o, 0, sizeof(*o));
    o->modeord = 0;
    o->upsampfac = 2.0;
    o->gpu_method = JFA_METHOD_AUTO;
    o->gpu_sort = 1;
    o->gpu_kerevalmeth = 1;
    o->gpu_maxbatchsize = 0;
    o->debug = 0;
    o->gpu_maxsubprobsize = 0;
    o->gpu_spreadinterponly = 0;
    o->gpu_device_id = -1;
    o->gpu_stream = nullptr;
    o->width_rule = 0;
    o->kernel_width = 0;
}

extern "C" const char *jfa_last_error(void) { return jfa::last_error(); }

// Stages and twiddles of every axis for the one-kernel-per-axis FFT passes;
// plans with an axis those passes cannot run keep axis_ok = false (rocFFT).
static int setup_axis_fft(jfa_plan p) {
    const size_t real = p->is_double ? 8 : 4;
    for (int d = 0; d < p->dim; ++d)
        if (!axis_fft(p->geom.nf[d], real, &p->axis[d])) return JFA_OK;
    for (int d = 0; d < p->dim; ++d) {
        const AxisFft &f = p->axis[d];
        JFA_HIP_CHECK(hipMalloc(&p->d_tw[d], 2 * real * std::max(f.ntw, 1)));
        const int rc = p->is_double ? launch_axis_twiddles<double>(f, (double *)p->d_tw[d], p->stream)
                                    : launch_axis_twiddles<float>(f, (float *)p->d_tw[d], p->stream);
        if (rc) return rc;
    }
    p->used = true;  // work on p->stream
    p->axis_ok = true;
    return JFA_OK;
}

// Fill the kernel tables (Horner coefficients and per-dimension 1/psi_hat) for
// a grid geometry that is already set.
int jfa::upload_kernel_tables(jfa_plan p, const int64_t *nmodes_for_dk) {
    const KernelParams &kp = p->kp;
    std::vector<double> coef((size_t)kp.nc * kp.ns);
    horner_fit(kp.ns, kp.nc, kp.beta, coef.data());
    free_ptr(p->d_coef);
    int rc = p->is_double ? upload<double>(coef, &p->d_coef) : upload<float>(coef, &p->d_coef);
    if (rc) return rc;
    for (int d = 0; d < 3; ++d) {
        free_ptr(p->d_dk[d]);
        int64_t n = (d < p->dim && nmodes_for_dk) ? nmodes_for_dk[d] : 1;
        std::vector<double> ph((size_t)n, 1.0);
        if (d < p->dim && nmodes_for_dk) {
            kernel_fourier(kp.ns, kp.beta, (double)p->geom.nf[d], (double)(-(n / 2)), n, ph.data());
            for (auto &v : ph) v = 1.0 / v;
        }
        rc = p->is_double ? upload<double>(ph, &p->d_dk[d]) : upload<float>(ph, &p->d_dk[d]);
        if (rc) return rc;
    }
    return JFA_OK;
}

extern "C" int jfa_makeplan(int type, int dim, const int64_t *nmodes, int iflag, int ntransf,
                            double eps, int is_double, const jfa_opts *opts,
                            jfa_plan *plan_out) {
    if (!plan_out) {
        set_error("plan_out is NULL");
        return JFA_ERR_BAD_ARG;
    }
    *plan_out = nullptr;
    if (type < 1 || type > 3) {
        set_error("type must be 1, 2 or 3 (got %d)", type);
        return JFA_ERR_BAD_ARG;
    }
    if (dim < 1 || dim > 3) {
        set_error("dim must be 1, 2 or 3 (got %d)", dim);
        return JFA_ERR_BAD_ARG;
    }
    if (ntransf < 1) {
        set_error("ntransf must be >= 1 (got %d)", ntransf);
        return JFA_ERR_BAD_ARG;
    }
    if (!(eps > 0)) {
        set_error("eps must be positive");
        return JFA_ERR_BAD_ARG;
    }
    if (int rc = ensure_rocfft()) return rc;

    jfa_opts o;
    if (opts) o = *opts;
    else jfa_default_opts(&o);
    if (!(o.upsampfac >= 1.0)) {
        set_error("upsampfac must be >= 1 (got %g)", o.upsampfac);
        return JFA_ERR_BAD_ARG;
    }
    if (o.kernel_width != 0 && (o.kernel_width < 2 || o.kernel_width > kMaxNs)) {
        set_error("kernel_width must be in [2, %d]", kMaxNs);
        return JFA_ERR_BAD_ARG;
    }
    if (o.modeord != 0 && o.modeord != 1) {
        set_error("modeord must be 0 or 1");
        return JFA_ERR_BAD_ARG;
    }

    DeviceGuard dg;
    if (int rc = dg.set(o.gpu_device_id)) return rc;

    auto *p = new jfa_plan_s();
    p->type = type;
    p->dim = dim;
    p->is_double = is_double ? 1 : 0;
    p->iflag = iflag >= 0 ? 1 : -1;
    p->ntransf = ntransf;
    p->eps = eps;
    p->opts = o;
    p->stream = (hipStream_t)o.gpu_stream;
    if (hipGetDevice(&p->device) != hipSuccess) p->device = 0;
    p->batch = o.gpu_maxbatchsize > 0 ? std::min(o.gpu_maxbatchsize, ntransf) : ntransf;
    p->kp = choose_kernel(eps, o.upsampfac, o.width_rule, p->is_double, o.kernel_width);
    p->maxsub = o.gpu_maxsubprobsize > 0 ? o.gpu_maxsubprobsize : default_maxsub(p);

    GridGeom &g = p->geom;
    g.dim = dim;
    g.ns = p->kp.ns;
    for (int d = 0; d < 3; ++d) {
        p->nmodes[d] = 1;
        g.nf[d] = 1;
        g.scale[d] = 1.0;
        g.shift[d] = 0.0;
    }
    if (type != 3) {
        for (int d = 0; d < dim; ++d) {
            if (!nmodes || nmodes[d] < 1) {
                jfa_destroy(p);
                set_error("nmodes[%d] must be >= 1", d);
                return JFA_ERR_BAD_ARG;
            }
            p->nmodes[d] = nmodes[d];
            if (o.gpu_spreadinterponly) {
                if (nmodes[d] < 2 * p->kp.ns) {
                    jfa_destroy(p);
                    set_error("spread/interp-only grid %lld is smaller than 2*width %d",
                              (long long)nmodes[d], 2 * p->kp.ns);
                    return JFA_ERR_BAD_ARG;
                }
                g.nf[d] = nmodes[d];
            } else {
                g.nf[d] = fine_size(nmodes[d], o.upsampfac, p->kp.ns);
            }
            g.scale[d] = (double)g.nf[d] / (2.0 * M_PI);
        }
        p->Ntot = p->nmodes[0] * p->nmodes[1] * p->nmodes[2];
        p->F = g.nf[0] * g.nf[1] * g.nf[2];
        if (p->F > kMaxFineCells) {
            jfa_destroy(p);
            set_error("fine grid of %lld cells per transform exceeds the supported 2^32",
                      (long long)(g.nf[0] * g.nf[1] * g.nf[2]));
            return JFA_ERR_TOO_LARGE;
        }
        default_bins(p);
        p->method = resolve_method(p);
        if (p->method < 0) {
            jfa_destroy(p);
            return JFA_ERR_BAD_ARG;
        }
        p->method_by_density = o.gpu_method == JFA_METHOD_AUTO && p->method == JFA_METHOD_SM;
        if (p->method == JFA_METHOD_STRIP) {
            if (int rc = setup_strip(p)) {
                jfa_destroy(p);
                return rc;
            }
        }
        int rc = upload_kernel_tables(p, p->nmodes);
        if (rc) {
            jfa_destroy(p);
            return rc;
        }
        if (!o.gpu_spreadinterponly && dim > 1) {
            if (int rc2 = setup_axis_fft(p)) {
                jfa_destroy(p);
                return rc2;
            }
        }
        if (!o.gpu_spreadinterponly) {
            const size_t bytes = (size_t)p->batch * p->F * 2 * (p->is_double ? 8 : 4);
            if (hipMalloc(&p->d_fw, bytes) != hipSuccess) {
                (void)hipGetLastError();
                jfa_destroy(p);
                set_error("could not allocate the %zu-byte fine grid", bytes);
                return JFA_ERR_ALLOC;
            }
        }
    } else {
        p->Ntot = 0;
        p->F = 0;
        int rc = jfa::type3_init(p);
        if (rc) {
            jfa_destroy(p);
            return rc;
        }
    }
    *plan_out = p;
    return p->kp.warn ? JFA_WARN_EPS_TOO_SMALL : JFA_OK;
}

int jfa::default_maxsub(jfa_plan p) {
    // Spreading: 1024 points per LDS subproblem (cuFINUFFT's published
    // default).  Each subproblem sums its points into its tile in fp32/fp64
    // before one global add per cell, so this also bounds the length of the
    // sequential sums a crowded cell sees.  Interpolation accumulates nothing
    // across points, and larger subproblems load each tile fewer times in 2D
    // (12288: a 64 x 64 bin is one subproblem up to 3 points per cell, and a
    // crowded bin splits into equal chunks; 2D type 2 on 2048^2 against 32 x 32
    // bins of 4096: 1e7 uniform points 0.348 -> 0.278 ms interpolation, 1e7
    // clustered 0.354 -> 0.334, 3e7 uniform 1.13 -> 0.86); in 3D, 1024
    // measured faster (more subproblems in flight: koosh-ball type 2 on 16.7M
    // points, 4.56 vs 4.80 ms with 8^3 bins).
    if (p->type == 2 && p->dim == 2) return 12288;
    return p->type == 2 && p->dim < 3 ? 4096 : 1024;
}

// Subproblem and piece sizes for M points, unless the caller chose one.
//
// LDS subproblems: the full size (default_maxsub) once that many bins or chunks
// fill the GPU; with under 512 of them, M nb / 2048 points (nb transforms read the
// points; 2D type 2, 64^2 modes, 300,000 points, 8 transforms: 256 points 59 us in
// fp32 and 155 in fp64, 1171 points 47 and 127), never below the 256 lanes of a
// workgroup (30,011 fp64 points on 2048 cells, 1D interpolation:
// 8 workgroups 187 us, 118 workgroups 7 us).  Splitting where there are enough
// only reloads tiles: 1e7 points in 1024 bins of 64 x 64, halves instead of
// whole bins, 0.265 -> 0.367 ms.
//
// Strip pieces: a wave walks its piece in series, so one crowded unit in full
// pieces can outlast the rest of the launch.  Units are split above twice the
// mean unit, and above a wave slot's share of the points of all nb transforms
// (300,007 centre-dense points, 4 transforms, 640 x 512 cells: spreading 168 us in
// pieces of 4096, 65 us by this rule, 46 on matrix instructions); evenly filled units stay whole, since every
// extra piece writes a tile and is summed again (4e6 uniform points on 1024^2
// in halves: 121 -> 137 us, and 10 us of reduction).  Grids of so few units that they
// leave the GPU idle are split into 512 pieces, down to 256 points (10,000 fp64 points
// on 16 x 24 modes, 3 units: 330 -> 123 us a call).
static void size_chunks(jfa_plan p, int64_t M) {
    const int64_t Mq = p->dim == 3 ? M * p->geom.ns : M;
    if (p->method == JFA_METHOD_STRIP)
        strip_units(p->sg, Mq, p->batch, p->opts.gpu_binsizey);
    if (p->opts.gpu_maxsubprobsize > 0) return;
    auto chunk = [](int64_t v, int64_t most) {
        return (int)std::min(most, std::max<int64_t>(256, (v + 63) / 64 * 64));
    };
    const int full = default_maxsub(p);
    p->maxsub = std::max(p->geom.nbins, M / full) < 512 ? chunk(M * p->batch / 2048, full) : full;
    if (p->method == JFA_METHOD_STRIP) {
        const int64_t all = Mq * p->batch;
        p->sg.pmax = chunk(std::max(std::min(2 * Mq / p->sg.nunits, all / 512), all / 4096),
                           kStripPiece);
    }
}

// Grow the point-dependent scratch to hold M points.
int jfa::reserve_points(jfa_plan p, int64_t M) {
    const size_t real = p->is_double ? 8 : 4;
    auto get = [](auto *&q, size_t bytes) {
        if (hipMalloc(&q, bytes) == hipSuccess) return true;
        (void)hipGetLastError();
        q = nullptr;
        set_error("could not allocate %zu bytes for the sorted points", bytes);
        return false;
    };
    if (p->geom.nbins + 1 > p->cap_bins) {
        p->cap_bins = 0;
        for (int **q : {&p->d_bin_start, &p->d_sub_start})
            free_ptr(reinterpret_cast<void *&>(*q));
        const size_t nb = (size_t)p->geom.nbins + 1;
        // the subproblem prefix, then the block sums of its scan
        if (!get(p->d_bin_start, sizeof(int) * nb) ||
            !get(p->d_sub_start, sizeof(int) * (nb + 2 * ((nb + 255) / 256) + 2)))
            return JFA_ERR_ALLOC;
        if (!p->d_nsub && !get(p->d_nsub, sizeof(int) * 4)) return JFA_ERR_ALLOC;
        p->cap_bins = (int64_t)nb;
    }
    if (M > p->cap_M) {
        p->cap_M = 0;
        for (void **q : {(void **)&p->d_idx, (void **)&p->d_l0, (void **)&p->d_key_in,
                         (void **)&p->d_key_out, &p->d_t, &p->d_sort_temp})
            free_ptr(*q);
        const int64_t cap = std::max<int64_t>(M, 1);
        if (!get(p->d_idx, sizeof(int) * cap) || !get(p->d_l0, sizeof(int) * cap * p->dim) ||
            !get(p->d_key_in, sizeof(unsigned) * cap) ||
            !get(p->d_key_out, sizeof(unsigned) * cap) || !get(p->d_t, real * cap * p->dim) ||
            !get(p->d_sort_temp, radix_temp_bytes(cap)))
            return JFA_ERR_ALLOC;
        p->cap_M = cap;
    }
    return JFA_OK;
}

// Auto method between LDS subproblem tiles and global atomics in sorted order,
// from a cost model evaluated once the point count is known: the tile method
// moves every bin's (bin + halo) tile between HBM and LDS once per
// subproblem, the global method touches w^d fine-grid cells per point (in
// sorted order, mostly through L2).  Tiles win when the taps outnumber the tile
// cells, i.e. when the points are dense enough to amortize the halo.
static void choose_method_by_density(jfa_plan p, int64_t M) {
    if (!p->method_by_density) return;
    const GridGeom &g = p->geom;
    double taps = (double)M, tiles = (double)g.nbins;
    for (int d = 0; d < p->dim; ++d) {
        taps *= g.ns;
        tiles *= g.bs[d] + g.ns - 1;
    }
    p->method = taps >= tiles ? JFA_METHOD_SM : JFA_METHOD_GM_SORT;
}

// The sorted LDS-tile / global methods read the first taps from the sorted
// key when every bin extent is a power of two and bin plus offset bits fit
// the 32-bit key: setpts then writes no gathered copy of the points.  1D and
// 2D only: in 3D the kernels' scattered reads of the Horner variables cost
// more than the gather they replace (3D type 2, 16.7M points on 512^3:
// 7.7 -> 8.6 ms per transform with keys).
static bool keyed_bins(GridGeom &g) {
    if (g.ymajor || g.dim > 2) return false;
    int bits = 0;
    for (int d = 0; d < 3; ++d) {
        g.subw[d] = 0;
        if (d >= g.dim) continue;
        const int b = g.bs[d];
        if (b <= 0 || (b & (b - 1))) return false;
        while ((1 << g.subw[d]) < b) ++g.subw[d];
        bits += g.subw[d];
    }
    if (bits == 0 || ((g.nbins + 1) << bits) > (int64_t)UINT32_MAX) return false;
    g.keyshift = bits;
    return true;
}

template <typename T>
static int sort_points(jfa_plan p, int64_t M, const T *x, const T *y, const T *z) {
    choose_method_by_density(p, M);
    GridGeom &g = p->geom;
    p->keyed = false;
    if (p->method == JFA_METHOD_STRIP) {
        SortScratch s{p->d_key_in, p->d_key_out, p->d_sort_temp};
        if (p->dim == 3)
            return launch_sort_points_slices<T>(g, p->sg.S, M, x, y, z, s, p->d_bin_start,
                                                p->d_idx, (T *)p->d_t, p->stream);
        return launch_sort_points_strip<T>(g, M, x, y, s, p->d_bin_start, p->d_idx,
                                           (T *)p->d_t, p->stream);
    }
    const bool sorted = p->method == JFA_METHOD_SM || p->opts.gpu_sort;
    if (!sorted)
        return launch_fold_points<T>(g, M, x, y, z, p->d_idx, p->d_l0, (T *)p->d_t, p->stream);
    SortScratch s{p->d_key_in, p->d_key_out, p->d_sort_temp};
    if (keyed_bins(g)) {
        p->keyed = true;
        return launch_sort_points_keyed<T>(g, M, x, y, z, s, p->d_bin_start,
                                           p->method == JFA_METHOD_SM ? p->d_sub_start : nullptr,
                                           p->d_nsub, p->maxsub, p->d_idx, (T *)p->d_t, p->stream);
    }
    g.keyshift = 0;
    return launch_sort_points<T>(g, M, x, y, z, s, p->d_bin_start,
                                 p->method == JFA_METHOD_SM ? p->d_sub_start : nullptr, p->d_nsub,
                                 p->maxsub, p->d_idx, p->d_l0, (T *)p->d_t, p->stream);
}

// Auto method for spreading, once the point count is known.  In 3D the strip spreader
// sorts ns slice points per point, so it needs M * ns < 2^31; grids narrower than a strip
// have a bound on its memory (kNarrowBytes), others what the device has.  Above that the
// LDS-tile or global method spreads instead, with the plan's ordinary bins.  An explicit
// gpu_method is never changed.
static int choose_spread_method(jfa_plan p, int64_t M) {
    if (p->dim < 2 || p->type == 2 || p->opts.gpu_method != JFA_METHOD_AUTO) return JFA_OK;
    GridGeom &g = p->geom;
    bool want_strip = strip_applicable(p) && M <= p->strip_most_M;
    const int64_t Mq = p->dim == 3 ? M * (int64_t)g.ns : M;
    if (p->dim == 3) want_strip = want_strip && Mq <= (int64_t)INT_MAX;
    if (want_strip && g.nf[0] < 64) {
        // keys, indices and their sort's scratch, first taps and Horner variables, records
        // and tiles (of which a narrow grid has few)
        const size_t real = p->is_double ? 8 : 4;
        const size_t per_point = 4 * 3 + 12 + (4 + real) * p->dim + 4 * real;
        want_strip = (size_t)Mq * per_point <= kNarrowBytes;
    }
    if (want_strip == (p->method == JFA_METHOD_STRIP)) return JFA_OK;
    if (want_strip) {
        if (int rc = setup_strip(p)) return rc;
        p->method = JFA_METHOD_STRIP;
        p->method_by_density = false;
        return JFA_OK;
    }
    g.ymajor = 0;
    g.keyshift = 0;
    default_bins(p);
    p->method = tile_lds_bytes(p) <= 64 * 1024 ? JFA_METHOD_SM : JFA_METHOD_GM_SORT;
    p->method_by_density = p->method == JFA_METHOD_SM;
    return JFA_OK;
}

int jfa::setpts_12(jfa_plan p, int64_t M, const void *x, const void *y, const void *z) {
    if (M < 0 || M > INT_MAX) {
        set_error("number of points %lld outside [0, 2^31)", (long long)M);
        return JFA_ERR_TOO_LARGE;
    }
    const void *xs[3] = {x, y, z};
    for (int d = 0; d < p->dim; ++d)
        if (M > 0 && !xs[d]) {
            set_error("points for dimension %d are NULL", d);
            return JFA_ERR_BAD_ARG;
        }
    for (;;) {
        if (int rc = choose_spread_method(p, M)) return rc;
        // the 3D strip spreader sorts ns slice points per point
        const bool strips = p->method == JFA_METHOD_STRIP;
        const int64_t sorted_count = strips && p->dim == 3 ? M * p->geom.ns : M;
        if (sorted_count > INT_MAX) {
            set_error("%lld points make %lld slice points, beyond 2^31 - 1 (use gpu_method 1 or 2)",
                      (long long)M, (long long)sorted_count);
            return JFA_ERR_TOO_LARGE;
        }
        int rc = reserve_points(p, sorted_count);
        if (rc == JFA_OK) {
            p->M = M;
            if (M == 0) return JFA_OK;
            size_chunks(p, M);
            if (strips && p->type == 1) rc = reserve_strip_scratch(p, sorted_count, p->batch);
        }
        if (rc == JFA_OK) break;
        if (rc != JFA_ERR_ALLOC || !strips || M < 1 || p->opts.gpu_method != JFA_METHOD_AUTO)
            return rc;
        // no memory for strips: by LDS tiles
        release_strip_scratch(p);
        p->strip_most_M = M - 1;
    }
    if (p->is_double)
        return sort_points<double>(p, M, (const double *)x, (const double *)y,
                                   (const double *)z);
    return sort_points<float>(p, M, (const float *)x, (const float *)y, (const float *)z);
}

extern "C" int jfa_setpts(jfa_plan p, int64_t M, const void *x, const void *y, const void *z,
                          int64_t N, const void *s, const void *t, const void *u) {
    if (!p) {
        set_error("plan is NULL");
        return JFA_ERR_BAD_ARG;
    }
    DeviceGuard dg;
    if (int rc = dg.set(p->device)) return rc;
    p->used = true;
    StageTimer tm(p);
    int rc = p->type == 3 ? jfa::type3_setpts(p, M, x, y, z, N, s, t, u)
                          : jfa::setpts_12(p, M, x, y, z);
    tm.mark("setpts");
    tm.report("setpts");
    return rc;
}

template <typename T>
SortedPts<T> jfa::sorted_view(jfa_plan p) {
    SortedPts<T> s;
    s.M = p->M;
    s.idx = p->d_idx;
    for (int d = 0; d < 3; ++d) {
        s.l0[d] = d < p->dim ? p->d_l0 + d * p->M : nullptr;
        s.t[d] = d < p->dim ? (const T *)p->d_t + d * p->M : nullptr;
    }
    s.key = p->keyed ? p->d_key_out : nullptr;
    s.rec = p->keyed ? (const T *)p->d_t : nullptr;
    return s;
}
template SortedPts<float> jfa::sorted_view<float>(jfa_plan);
template SortedPts<double> jfa::sorted_view<double>(jfa_plan);

BinIndex jfa::bin_view(jfa_plan p) {
    BinIndex b;
    b.bin_start = p->d_bin_start;
    b.sub_start = p->d_sub_start;
    b.nsub = p->d_nsub;
    b.maxsub = p->maxsub;
    return b;
}

// Spread ntr transforms (strengths c with stride c_stride, grids fw with
// stride fw_stride) with the plan's method.  fw must be zeroed first except
// for the strip method, which writes every cell.
// With a stage timer, the strip method's three launches are marked as the
// stages "units", "spread" (the spreading kernel alone) and "merge".
template <typename T>
static int spread_timed(jfa_plan p, const T *c, int64_t c_stride, T *fw, int64_t fw_stride,
                        int ntr, StageTimer *tm) {
    const int kem = p->opts.gpu_kerevalmeth ? 1 : 0;
    if (p->method != JFA_METHOD_STRIP) {
        int rc = launch_spread<T>(p->method, p->geom, sorted_view<T>(p), bin_view(p),
                                  (const T *)p->d_coef, kem, p->kp.beta, c, c_stride, fw,
                                  fw_stride, ntr, p->stream);
        if (tm) tm->mark("spread");
        return rc;
    }
    // the merge writes every cell of fw, unless there are no points at all
    const int64_t M = p->M;
    if (M == 0) return launch_fill_zero(fw, (int64_t)sizeof(T) * 2 * fw_stride * ntr, p->stream);
    // points the spreader walks: M, or the ns slice points of each in 3D
    const int64_t Mq = p->dim == 3 ? M * p->geom.ns : M;
    // (with one record (c, tx, ty) per point and transform: the spreader's only
    // scattered read)
    if (int rc = reserve_strip_scratch(p, Mq, std::min(p->batch, ntr))) return rc;
    const StripPts<T> pts{Mq, p->d_idx, p->d_key_out, (const T *)p->d_pack, nullptr, nullptr, 0, 0};
    for (int t0 = 0; t0 < ntr; t0 += p->strip_batch) {
        const int nb = std::min(p->strip_batch, ntr - t0);
        const int rc =
            p->dim == 3
                ? launch_strip3_pack<T>(c + 2 * t0 * c_stride, c_stride, (const T *)p->d_t,
                                        (const T *)p->d_coef, kem, p->kp.beta, p->geom.ns, M,
                                        nb, (T *)p->d_pack, p->stream)
                : launch_strip_pack<T>(c + 2 * t0 * c_stride, c_stride, (const T *)p->d_t, M,
                                       nb, (T *)p->d_pack, p->stream);
        if (rc) return rc;
        if (tm) tm->mark("pack");
        const int phases[3] = {kStripUnits, kStripSpread, kStripMerge};
        const char *names[3] = {"units", "spread", "merge"};
        for (int ph = 0; ph < 3; ++ph) {
            if (!tm && ph > 0) break;
            int rc = launch_spread_strip<T>(
                p->sg, pts, p->d_bin_start, p->d_piece_start, p->d_npieces, p->d_piece_unit,
                p->d_heavy, p->d_strip_blocksum, (const T *)p->d_coef,
                kem, p->kp.beta, Mq, fw + 2 * t0 * fw_stride, fw_stride, (T *)p->d_strip_scratch,
                p->strip_scratch_stride, nb, tm ? phases[ph] : kStripAll, p->stream);
            if (rc) return rc;
            if (tm) tm->mark(names[ph]);
        }
    }
    return JFA_OK;
}

template <typename T>
int jfa::spread_any(jfa_plan p, const T *c, int64_t c_stride, T *fw, int64_t fw_stride, int ntr) {
    return spread_timed<T>(p, c, c_stride, fw, fw_stride, ntr, nullptr);
}
template int jfa::spread_any<float>(jfa_plan, const float *, int64_t, float *, int64_t, int);
template int jfa::spread_any<double>(jfa_plan, const double *, int64_t, double *, int64_t, int);

// Amplify nb transforms of modes (stride Ntot) onto the fine grid fw (stride
// F) and FFT them: the type-2 / interpolation input.
template <typename T>
static int modes_to_grid(jfa_plan p, const T *fk, T *fw, int nb, StageTimer &tm) {
    const GridGeom &g = p->geom;
    int rc;
    if (p->axis_ok) {
        if ((rc = reserve_fwt(p))) return rc;
        if ((rc = axis_modes_to_grid<T>(p, fk, (T *)p->d_fwt, fw, nb))) return rc;
    } else if (fft_is_pruned(p)) {
        if ((rc = pruned_amplify<T>(p, fk, fw, nb))) return rc;
        tm.mark("amplify");
        if ((rc = pruned_modes_fft<T>(p, fw, nb))) return rc;
    } else {
        const T *dk[3] = {(const T *)p->d_dk[0], (const T *)p->d_dk[1], (const T *)p->d_dk[2]};
        if ((rc = launch_amplify<T>(p->dim, p->nmodes, g.nf, dk[0], dk[1], dk[2],
                                    p->opts.modeord, fk, p->Ntot, fw, p->F, nb, p->stream)))
            return rc;
        tm.mark("amplify");
        if ((rc = fft_exec(p, fw, nb))) return rc;
    }
    tm.mark("fft");
    return JFA_OK;
}

// Type 1 / type 2 execution on the plan's current points.  c has ntransf*M
// complex values, fk ntransf*Ntot.
template <typename T>
int jfa::execute_12(jfa_plan p, T *c, T *fk) {
    const GridGeom &g = p->geom;
    const SortedPts<T> pts = sorted_view<T>(p);
    const BinIndex bi = bin_view(p);
    const T *coef = (const T *)p->d_coef;
    const T *dk[3] = {(const T *)p->d_dk[0], (const T *)p->d_dk[1], (const T *)p->d_dk[2]};
    const int kem = p->opts.gpu_kerevalmeth ? 1 : 0;
    const int64_t M = p->M;
    StageTimer tm(p);
    int rc = JFA_OK;
    if (p->opts.gpu_spreadinterponly) {
        // the mode array is the fine grid itself
        if (p->type == 1) {
            if (p->method != JFA_METHOD_STRIP) {
                if ((rc = launch_fill_zero(fk, sizeof(T) * 2 * p->F * p->ntransf, p->stream)))
                    return rc;
                tm.mark("zero");
            }
            rc = spread_timed<T>(p, c, M, fk, p->F, p->ntransf, tm.on ? &tm : nullptr);
        } else {
            rc = launch_interp<T>(p->method, g, pts, bi, coef, kem, p->kp.beta, fk, p->F, c, M,
                                  p->ntransf, p->stream);
            tm.mark("interp");
        }
        tm.report("execute");
        return rc;
    }
    T *fw = (T *)p->d_fw;
    for (int t0 = 0; t0 < p->ntransf; t0 += p->batch) {
        const int nb = std::min(p->batch, p->ntransf - t0);
        T *cb = c + 2 * (int64_t)t0 * M;
        T *fb = fk + 2 * (int64_t)t0 * p->Ntot;
        if (p->type == 1) {
            if (p->method != JFA_METHOD_STRIP) {
                if ((rc = launch_fill_zero(fw, sizeof(T) * 2 * p->F * nb, p->stream))) return rc;
                tm.mark("zero");
            }
            if ((rc = spread_timed<T>(p, cb, M, fw, p->F, nb, tm.on ? &tm : nullptr))) return rc;
            if (p->axis_ok) {
                if ((rc = reserve_fwt(p))) return rc;
                if ((rc = axis_grid_to_modes<T>(p, fw, (T *)p->d_fwt, fb, nb))) return rc;
                tm.mark("fft");
                continue;
            }
            if (fft_is_pruned(p)) {
                if ((rc = pruned_grid_fft<T>(p, fw, nb))) return rc;
                tm.mark("fft");
                if ((rc = pruned_deconv<T>(p, fw, fb, nb))) return rc;
            } else {
                if ((rc = fft_exec(p, fw, nb))) return rc;
                tm.mark("fft");
                if ((rc = launch_deconv<T>(p->dim, p->nmodes, g.nf, dk[0], dk[1], dk[2],
                                           p->opts.modeord, fw, p->F, fb, p->Ntot, nb,
                                           p->stream)))
                    return rc;
            }
            tm.mark("deconv");
        } else {
            if ((rc = modes_to_grid<T>(p, fb, fw, nb, tm))) return rc;
            if ((rc = launch_interp<T>(p->method, g, pts, bi, coef, kem, p->kp.beta, fw,
                                       stored_cells(g), cb, M, nb, p->stream)))
                return rc;
            tm.mark("interp");
        }
    }
    // the fine grid of a single-batch type-2 pass can serve a later gradient pass
    p->fw_modes = p->type == 2 && p->ntransf <= p->batch;
    tm.report("execute");
    return rc;
}
template int jfa::execute_12<float>(jfa_plan, float *, float *);
template int jfa::execute_12<double>(jfa_plan, double *, double *);

extern "C" int jfa_execute(jfa_plan p, void *c, void *fk) {
    if (!p) {
        set_error("plan is NULL");
        return JFA_ERR_BAD_ARG;
    }
    DeviceGuard dg;
    if (int rc = dg.set(p->device)) return rc;
    p->used = true;
    if (p->type == 3) return jfa::type3_execute(p, c, fk);
    if ((p->M > 0 && !c) || (p->Ntot > 0 && !fk)) {
        set_error("execute: NULL data pointer");
        return JFA_ERR_BAD_ARG;
    }
    if (p->M == 0) {
        // no points: type 1 output is zero, type 2 has nothing to write (and its
        // fine grid is not computed, so it no longer matches the last modes)
        p->fw_modes = false;
        if (p->type == 1)
            return launch_fill_zero(fk, (int64_t)(p->is_double ? 16 : 8) * p->Ntot * p->ntransf,
                                    p->stream);
        return JFA_OK;
    }
    if (p->is_double) return execute_12<double>(p, (double *)c, (double *)fk);
    return execute_12<float>(p, (float *)c, (float *)fk);
}

// Fused adjoint pass of a type-2 plan: val = the type-2 transform of fk at the
// plan's points (optional), grad[d*M + j] = sum_t Re(conj(w_t,j) dval_t,j/dx_d)
// (optional, needs w).  One amplify + FFT per batch, then one interpolation
// pass that evaluates the kernel and its derivative together.
template <typename T>
static int interp_grad_t(jfa_plan p, const T *fk, const T *w, T *val, T *grad) {
    const GridGeom &g = p->geom;
    const SortedPts<T> pts = sorted_view<T>(p);
    const BinIndex bi = bin_view(p);
    const T *dk[3] = {(const T *)p->d_dk[0], (const T *)p->d_dk[1], (const T *)p->d_dk[2]};
    const int64_t M = p->M;
    T *fw = (T *)p->d_fw;
    StageTimer tm(p);
    for (int t0 = 0; t0 < p->ntransf; t0 += p->batch) {
        const int nb = std::min(p->batch, p->ntransf - t0);
        int rc = JFA_OK;
        if (fk) {
            if ((rc = modes_to_grid<T>(p, fk + 2 * (int64_t)t0 * p->Ntot, fw, nb, tm)))
                return rc;
        }
        rc = launch_interp_grad<T>(p->method, g, pts, bi, (const T *)p->d_coef, fw, p->F, nb,
                                   w ? w + 2 * (int64_t)t0 * M : nullptr, M,
                                   val ? val + 2 * (int64_t)t0 * M : nullptr, M, grad, M, t0 > 0,
                                   p->stream);
        if (rc) return rc;
        tm.mark("interp_grad");
    }
    p->fw_modes = p->ntransf <= p->batch;
    tm.report("interp_grad");
    return JFA_OK;
}

extern "C" int jfa_interp_grad(jfa_plan p, const void *fk, const void *w, void *val,
                               void *grad) {
    if (!p) {
        set_error("plan is NULL");
        return JFA_ERR_BAD_ARG;
    }
    if (p->type != 2 || p->opts.gpu_spreadinterponly) {
        set_error("interp_grad needs a type-2 plan");
        return JFA_ERR_BAD_ARG;
    }
    if (grad && !w) {
        set_error("interp_grad: weights are required for the gradient");
        return JFA_ERR_BAD_ARG;
    }
    if (!fk && !p->fw_modes) {
        // a limitation of the plan's state, not a bad call: the last execute ran
        // in several batches (gpu_maxbatchsize < ntransf) or had no points, so
        // no fine grid of all transforms is held; the caller passes fk instead
        set_error("interp_grad without modes needs the fine grid of a preceding single-batch "
                  "type-2 execute on this plan");
        return JFA_ERR_NOT_SUPPORTED;
    }
    DeviceGuard dg;
    if (int rc = dg.set(p->device)) return rc;
    p->used = true;
    if (p->M == 0) return JFA_OK;
    if (p->is_double)
        return interp_grad_t<double>(p, (const double *)fk, (const double *)w, (double *)val,
                                     (double *)grad);
    return interp_grad_t<float>(p, (const float *)fk, (const float *)w, (float *)val,
                                (float *)grad);
}

extern "C" int jfa_set_stream(jfa_plan p, jfa_stream_t stream) {
    if (!p) {
        set_error("plan is NULL");
        return JFA_ERR_BAD_ARG;
    }
    hipStream_t s = (hipStream_t)stream;
    if (s == p->stream) return JFA_OK;
    DeviceGuard dg;
    if (int rc = dg.set(p->device)) return rc;
    if (p->used) {
        if (!p->order_event)
            JFA_HIP_CHECK(hipEventCreateWithFlags(&p->order_event, hipEventDisableTiming));
        JFA_HIP_CHECK(hipEventRecord(p->order_event, p->stream));
        JFA_HIP_CHECK(hipStreamWaitEvent(s, p->order_event, 0));
    }
    p->stream = s;
    if (p->inner) return jfa_set_stream(p->inner, stream);
    return JFA_OK;
}

extern "C" int jfa_destroy(jfa_plan p) {
    if (!p) return JFA_OK;
    DeviceGuard dg;
    (void)dg.set(p->device);
    if (p->used) (void)hipStreamSynchronize(p->stream);
    if (p->inner) jfa_destroy(p->inner);
    {
        std::lock_guard<std::mutex> lk(rocfft_mutex());
        for (auto &kv : p->fft_plans) rocfft_plan_destroy(kv.second);
        for (auto &kv : p->fft1_plans) rocfft_plan_destroy(kv.second);
    }
    free_ptr(p->d_fwt);
    for (auto &d : p->d_tw) free_ptr(d);
    if (p->fft_info) rocfft_execution_info_destroy(p->fft_info);
    free_ptr(p->d_fft_work);
    free_ptr(p->d_coef);
    for (auto &d : p->d_dk) free_ptr(d);
    free_ptr(p->d_fw);
    for (void **q : {(void **)&p->d_idx, (void **)&p->d_l0, (void **)&p->d_key_in,
                     (void **)&p->d_key_out, &p->d_sort_temp, &p->d_t,
                     (void **)&p->d_bin_start, (void **)&p->d_sub_start, (void **)&p->d_nsub,
                     (void **)&p->d_piece_start, (void **)&p->d_npieces,
                     (void **)&p->d_piece_unit, (void **)&p->d_heavy,
                     (void **)&p->d_strip_blocksum, &p->d_strip_scratch,
                     &p->d_pack})
        free_ptr(*q);
    jfa::type3_free(p);
    for (hipEvent_t e : p->timing_events) (void)hipEventDestroy(e);
    if (p->order_event) (void)hipEventDestroy(p->order_event);
    delete p;
    return JFA_OK;
}

// Layout of the sort setpts ran (see jfa_setpts_info in the header).
extern "C" int jfa_setpts_info(jfa_plan p, int64_t *info) {
    if (!p || !info) {
        set_error("setpts_info: NULL argument");
        return JFA_ERR_BAD_ARG;
    }
    const GridGeom &g = p->geom;
    const bool strip = p->method == JFA_METHOD_STRIP;
    const bool sorted = strip || p->method == JFA_METHOD_SM || p->opts.gpu_sort;
    for (int i = 0; i < 24; ++i) info[i] = 0;
    info[0] = !sorted ? 0 : (strip && p->dim == 3 ? p->M * g.ns : p->M);
    info[1] = g.nbins;
    info[2] = strip ? kStripKeyShift : g.keyshift;
    info[3] = strip ? kStripSortLowBit : (p->keyed ? g.keyshift : 0);
    info[4] = p->method;
    info[5] = strip ? 2 : (p->keyed ? 1 : 0);
    for (int d = 0; d < 3; ++d) {
        info[6 + d] = g.bs[d];
        info[9 + d] = g.nb[d];
        info[12 + d] = g.nf[d];
        info[18 + d] = g.subw[d];
    }
    info[15] = g.ns;
    info[16] = g.ymajor;
    info[17] = strip ? p->sg.S : 0;
    info[21] = strip ? p->sg.SW : 0;
    info[22] = p->type == 3 ? p->t3_nbox : 0;
    return JFA_OK;
}

// Copy the sort's integer outputs into caller device buffers, on the plan's
// stream (see the header).
extern "C" int jfa_setpts_copy(jfa_plan p, void *keys, void *perm, void *bin_start) {
    int64_t info[24];
    if (int rc = jfa_setpts_info(p, info)) return rc;
    if (info[0] == 0 && p->M > 0) {
        set_error("setpts_copy: this plan does not sort its points (gpu_sort = 0)");
        return JFA_ERR_NOT_SUPPORTED;
    }
    DeviceGuard dg;
    if (int rc = dg.set(p->device)) return rc;
    const size_t n = (size_t)info[0];
    if (keys && n)
        JFA_HIP_CHECK(hipMemcpyAsync(keys, p->d_key_out, 4 * n, hipMemcpyDeviceToDevice,
                                     p->stream));
    if (perm && n)
        JFA_HIP_CHECK(hipMemcpyAsync(perm, p->d_idx, 4 * n, hipMemcpyDeviceToDevice, p->stream));
    if (bin_start && p->d_bin_start)
        JFA_HIP_CHECK(hipMemcpyAsync(bin_start, p->d_bin_start, 4 * (size_t)(info[1] + 1),
                                     hipMemcpyDeviceToDevice, p->stream));
    return JFA_OK;
}

extern "C" int jfa_plan_info(jfa_plan p, int *ns, double *beta, int64_t *nf) {
    if (!p) {
        set_error("plan is NULL");
        return JFA_ERR_BAD_ARG;
    }
    if (ns) *ns = p->kp.ns;
    if (beta) *beta = p->kp.beta;
    if (nf)
        for (int d = 0; d < 3; ++d) nf[d] = p->geom.nf[d];
    return JFA_OK;
}
