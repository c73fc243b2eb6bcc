// Ragged batches of 2D type-1 problems: one launch sequence for many
// independent problems with their own point counts, mode grids and numbers of
// stacked strength vectors.  No reference counterpart: with the reference a
// batch like this is a Python loop of nufft1 calls, each making, using and
// destroying its own plan (run_nufft, lib/kernels.cc.cu:25-92).
//
// Layout.  The points of all problems form one concatenated index space
// (problem i owns [moff[i], moff[i+1])) and are sorted together: a point's key
// is its bin within its problem offset by the problem's first global bin.  A
// virtual problem is one (problem, transform) pair; virtual problems are
// ordered by fine-grid size (then mode count n0) so that the fine grids of one
// class are contiguous and transform together: one batched 1D rocFFT along x,
// a gather of the n0 needed columns (transposed) into the class's pruned-FFT
// buffer, one batched 1D rocFFT along y there.  The spreading and merge
// kernels walk the global list of units of every virtual problem;
// deconvolution walks the global list of 256-mode blocks.  The
// device pointer table (x, y, c, f of every problem) is rewritten before each
// run, so a captured graph stays valid for new arrays of the same shapes.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <numeric>
#include <mutex>
#include <vector>

#include "jfa_internal.hpp"

using namespace jfa;

struct jfa_ragged_s {
    int dim = 2, nprob = 0, is_double = 0, iflag = 1, device = 0;
    double eps = 1e-6;
    jfa_opts opts{};
    KernelParams kp;
    std::vector<int64_t> npts, ntr, n0, n1;
    std::vector<RaggedProb> probs;
    std::vector<RaggedVirt> virt;
    std::vector<int64_t> moff, mode_blk;
    std::vector<int> vunit_off, unit_virt;
    int64_t max_pieces = 0;  // pieces of every virtual problem at most
    int64_t max_heavy = 0;   // crowded units (more than one piece) at most
    RaggedLaunch rl{};

    // device tables
    void *d_probs = nullptr, *d_virt = nullptr, *d_moff = nullptr, *d_vunit_off = nullptr,
         *d_unit_virt = nullptr, *d_mode_blk = nullptr;
    void *d_ptrs = nullptr;
    const void **h_ptrs = nullptr;  // pinned staging of the pointer table
    hipEvent_t ptrs_copied = nullptr;
    void *d_coef = nullptr, *d_dk = nullptr;

    // sorted points
    int64_t mtot = 0;
    int *d_idx = nullptr, *d_l0 = nullptr;
    void *d_t = nullptr;
    unsigned *d_key_in = nullptr, *d_key_out = nullptr;
    void *d_sort_temp = nullptr;
    int *d_bin_start = nullptr, *d_piece_start = nullptr, *d_npieces = nullptr,
        *d_piece_unit = nullptr, *d_heavy = nullptr,
        *d_blocksum = nullptr;

    // fine grids and strip scratch (complex cells)
    int64_t fw_cells = 0, tile_cells = 0;
    void *d_fw = nullptr, *d_scratch = nullptr;

    // one batched rocFFT per fine-grid size
    struct FftClass {
        int64_t nf0, nf1, n0, fw_off, g_off;
        int count;
        rocfft_plan plan_x, plan_y;
    };
    std::vector<FftClass> fft;
    int64_t g_cells = 0;  // pruned-FFT buffers [n0][nf1] per virtual problem, in d_scratch
                          // (written once the tiles are merged)
    rocfft_execution_info fft_info = nullptr;
    void *d_fft_work = nullptr;
    size_t fft_work_bytes = 0;

    // streams and graph
    hipStream_t stream = nullptr;  // the caller's stream
    hipStream_t work = nullptr;    // own stream that graphs are captured on
    hipEvent_t ev_in = nullptr, ev_out = nullptr;
    bool use_graph = false;
    int graph_state = 0;           // 0 not captured yet, 1 captured, -1 capture failed
    hipGraphExec_t gexec = nullptr;
};

namespace {

void free_dev(void *&p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}

template <typename V>
int upload_vec(const std::vector<V> &h, void **d) {
    JFA_HIP_CHECK(hipMalloc(d, sizeof(V) * std::max<size_t>(h.size(), 1)));
    if (!h.empty())
        JFA_HIP_CHECK(hipMemcpy(*d, h.data(), sizeof(V) * h.size(), hipMemcpyHostToDevice));
    return JFA_OK;
}

template <typename T>
int upload_real(const std::vector<double> &h, void **d) {
    std::vector<T> tmp(h.begin(), h.end());
    return upload_vec(tmp, d);
}

void release(jfa_ragged r) {
    for (void **q : {&r->d_probs, &r->d_virt, &r->d_moff, &r->d_vunit_off, &r->d_unit_virt,
                     &r->d_mode_blk, &r->d_ptrs, &r->d_coef, &r->d_dk, (void **)&r->d_idx,
                     (void **)&r->d_l0, &r->d_t, (void **)&r->d_key_in,
                     (void **)&r->d_key_out, &r->d_sort_temp, (void **)&r->d_bin_start,
                     (void **)&r->d_piece_start, (void **)&r->d_npieces,
                     (void **)&r->d_piece_unit, (void **)&r->d_heavy, &r->d_fw, &r->d_scratch,
                     &r->d_fft_work, (void **)&r->d_blocksum})
        free_dev(*q);
    if (r->h_ptrs) (void)hipHostFree((void *)r->h_ptrs);
    r->h_ptrs = nullptr;
    {
        std::lock_guard<std::mutex> lk(rocfft_mutex());
        for (auto &c : r->fft)
            for (rocfft_plan pl : {c.plan_x, c.plan_y})
                if (pl) rocfft_plan_destroy(pl);
    }
    r->fft.clear();
    if (r->fft_info) rocfft_execution_info_destroy(r->fft_info);
    r->fft_info = nullptr;
    if (r->gexec) (void)hipGraphExecDestroy(r->gexec);
    r->gexec = nullptr;
    for (hipEvent_t *e : {&r->ev_in, &r->ev_out, &r->ptrs_copied})
        if (*e) (void)hipEventDestroy(*e), *e = nullptr;
    if (r->work) (void)hipStreamDestroy(r->work);
    r->work = nullptr;
}

struct DeviceScope {
    int prev = -1;
    bool changed = false;
    int set(int dev) {
        JFA_HIP_CHECK(hipGetDevice(&prev));
        if (prev != dev) {
            JFA_HIP_CHECK(hipSetDevice(dev));
            changed = true;
        }
        return JFA_OK;
    }
    ~DeviceScope() {
        if (changed) (void)hipSetDevice(prev);
    }
};

// Transforms that the wave of transform t of problem i spreads: in fp32 t and t + 1
// share the points, and the wave of t + 1 does nothing.
int wave_transforms(jfa_ragged r, int i, int t) {
    if (ragged_transforms(r->is_double ? 8 : 4) == 1) return 1;
    return (t & 1) ? 0 : (t + 1 < r->ntr[i] ? 2 : 1);
}

// Rows of the units of sparse batches (layout).
constexpr int kSparseRows = 16;

// Problem geometry, virtual problems, offsets; host only.
int layout(jfa_ragged r) {
    const int ns = r->kp.ns;
    const int np = r->nprob;
    r->probs.assign(np, RaggedProb{});
    r->moff.assign(np + 1, 0);
    std::vector<StripGeom> sg(np);
    double units = 0, unit_points = 0;  // over every transform, units short
    int64_t bins = 0;
    for (int i = 0; i < np; ++i) {
        GridGeom &g = r->probs[i].g;
        g.dim = 2;
        g.ns = ns;
        const int64_t n[2] = {r->n0[i], r->n1[i]};
        for (int d = 0; d < 3; ++d) {
            g.nf[d] = d < 2 ? fine_size(n[d], r->opts.upsampfac, ns) : 1;
            g.scale[d] = d < 2 ? (double)g.nf[d] / (2.0 * M_PI) : 1.0;
            g.shift[d] = 0.0;
        }
        if (g.nf[0] < 64 || g.nf[1] < 2 * ns) {
            set_error("ragged problem %d: fine grid %lld x %lld is below the strip spreader's "
                      "64 x %d minimum", i, (long long)g.nf[0], (long long)g.nf[1], 2 * ns);
            return JFA_ERR_NOT_SUPPORTED;
        }
        if (g.nf[0] * g.nf[1] > kMaxFineCells) {
            set_error("ragged problem %d: fine grid exceeds %lld cells", i,
                      (long long)kMaxFineCells);
            return JFA_ERR_TOO_LARGE;
        }
        sg[i] = strip_geometry(g, r->opts.gpu_maxsubprobsize);
        if (r->opts.gpu_binsizey > 0) strip_set_rows(sg[i], r->opts.gpu_binsizey);
        units += (double)sg[i].nunits * r->ntr[i];
        unit_points += (double)r->npts[i] * r->ntr[i];
        r->probs[i].moff = r->moff[i];
        r->probs[i].bin_off = bins;
        r->moff[i + 1] = r->moff[i] + r->npts[i];
        bins += g.nbins;
    }
    // One height for the batch, whose units share one launch (a launch for each height:
    // 28 problems of 1e4 to 3.1e5 points 790 -> 858 us).  ns <= 8: 16 rows halve the tiles to
    // merge, but dense problems' units, taller, end late, so there have to be few points or
    // many units to level them.  9 / 16 rows in us: 41,466 units of 3 points on the mean 511 /
    // 498, 10,676 of 34 290 / 366, 44,600 of 34 689 / 774, 56,208 of 52 856 / 992, 68,000 of
    // 49 988 / 1046, 72,206 of 54 1042 / 1010, 79,952 of 112 1265 / 1336, 89,834 of 64 1285 /
    // 1182, 98,028 of 126 1576 / 1534, 151,500 of 37 1956 / 1721, 128,558 of 6 1601 / 1441, 111,926 of 186 1938 / 1982 (25 rows: 44,600 of 34 889,
    // 151,500 of 37 1817, 128,558 of 6 1441).  ns > 8: small grids have few rolling units, so
    // there have to be many, and few points in dense problems: 200 of 1e3 to 1e4 points, one
    // transform each (128,558 short units), 2.42 / 2.77 ms at ns = 11, up to six each 7.52 /
    // 7.15.
    if (r->opts.gpu_binsizey <= 0 && ns <= 8) {
        const double line = units < 75000 ? 16 : std::min(units / 1300, 125.0);
        if (unit_points <= line * units)
            for (StripGeom &s : sg) strip_set_rows(s, kSparseRows);
    } else if (r->opts.gpu_binsizey <= 0) {
        double dense = 0;  // points of dense problems
        for (int i = 0; i < np; ++i)
            if (r->npts[i] > 256 * (int64_t)sg[i].nunits)
                dense += (double)r->npts[i] * r->ntr[i];
        if (strip_tall(ns, unit_points, units) && 3 * dense <= unit_points && units >= 200000)
            for (StripGeom &s : sg) strip_set_rows(s, strip_tall_rows(ns));
    }
    r->rl.tall = false;
    for (const StripGeom &s : sg) r->rl.tall = r->rl.tall || s.H > strip_short_rows(ns);
    r->mtot = r->moff[np];
    if (r->mtot > INT_MAX) {
        set_error("ragged batch of %lld points exceeds 2^31 - 1", (long long)r->mtot);
        return JFA_ERR_TOO_LARGE;
    }
    const int keyshift = r->probs.empty() ? 0 : r->probs[0].g.keyshift;
    if (((bins + 1) << keyshift) > (int64_t)UINT32_MAX) {
        set_error("ragged batch has too many bins for 32-bit sort keys");
        return JFA_ERR_TOO_LARGE;
    }
    // virtual problems, grouped by fine-grid size
    std::vector<int> order(np);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        const GridGeom &ga = r->probs[a].g, &gb = r->probs[b].g;
        if (ga.nf[0] != gb.nf[0]) return ga.nf[0] < gb.nf[0];
        if (ga.nf[1] != gb.nf[1]) return ga.nf[1] < gb.nf[1];
        return r->n0[a] < r->n0[b];
    });
    std::vector<int64_t> dk_off(np);
    int64_t dk = 0;
    for (int i = 0; i < np; ++i) {
        dk_off[i] = dk;
        dk += r->n0[i] + r->n1[i];
    }
    r->virt.clear();
    r->vunit_off.assign(1, 0);
    r->unit_virt.clear();
    r->max_pieces = 0;
    r->max_heavy = 0;
    r->mode_blk.assign(1, 0);
    r->fft.clear();
    int64_t fw = 0, tiles = 0, gc = 0;
    for (int i : order) {
        const GridGeom &g = r->probs[i].g;
        const int64_t F = g.nf[0] * g.nf[1];
        if (r->fft.empty() || r->fft.back().nf0 != g.nf[0] || r->fft.back().nf1 != g.nf[1] ||
            r->fft.back().n0 != r->n0[i])
            r->fft.push_back({g.nf[0], g.nf[1], r->n0[i], fw, gc, 0, nullptr, nullptr});
        for (int t = 0; t < r->ntr[i]; ++t) {
            RaggedVirt v{};
            v.sg = sg[i];
            v.prob = i;
            v.t = t;
            v.nt = wave_transforms(r, i, t);
            v.tile_next = strip_max_pieces(sg[i], r->npts[i]) * strip_tile_cells(sg[i]);
            v.m = r->npts[i];
            v.bin_off = r->probs[i].bin_off;
            v.fw_off = fw;
            v.g_off = gc;
            v.tile_off = tiles;
            v.unit_off = r->vunit_off.back();
            v.n0 = r->n0[i];
            v.n1 = r->n1[i];
            v.dk_off = dk_off[i];
            v.moff = r->moff[i];
            r->virt.push_back(v);
            fw += F;
            gc += r->n0[i] * g.nf[1];
            tiles += strip_max_pieces(sg[i], r->npts[i]) * strip_tile_cells(sg[i]);
            r->max_pieces += strip_max_pieces(sg[i], r->npts[i]);
            r->max_heavy += strip_max_heavy(sg[i], r->npts[i]);
            r->unit_virt.insert(r->unit_virt.end(), sg[i].nunits, (int)r->virt.size() - 1);
            r->vunit_off.push_back(r->vunit_off.back() + sg[i].nunits);
            r->mode_blk.push_back(r->mode_blk.back() + ((v.n0 + 31) / 32) * ((v.n1 + 31) / 32));
            r->fft.back().count++;
        }
    }
    r->fw_cells = fw;
    r->g_cells = gc;
    r->tile_cells = tiles;
    if ((int64_t)r->vunit_off.back() > INT_MAX / 2) {
        set_error("ragged batch has too many spreading units");
        return JFA_ERR_TOO_LARGE;
    }

    RaggedLaunch &rl = r->rl;
    rl.nprob = np;
    rl.nv = (int)r->virt.size();
    rl.ns = ns;
    rl.pmax = sg.empty() ? 4096 : sg[0].pmax;
    rl.keyshift = keyshift;
    rl.mtot = r->mtot;
    rl.nbins = bins;
    rl.nunits = r->vunit_off.back();
    rl.mode_blocks = r->mode_blk.back();
    rl.max_pieces = r->max_pieces;
    return JFA_OK;
}

// Consistency of the host tables layout() built, against the sizes
// allocate() gives the device buffers: every offset and range of every
// problem, virtual problem, unit, tile, pruned-FFT buffer and mode block stays
// inside its table.  Host only.
int check_layout(jfa_ragged r) {
    auto bad = [](const char *what, long long a, long long b) {
        set_error("ragged layout: %s (%lld vs %lld)", what, a, b);
        return JFA_ERR_INTERNAL;
    };
    const int np = r->nprob;
    if ((int)r->moff.size() != np + 1 || r->moff[0] != 0) return bad("moff size", r->moff.size(), np + 1);
    int64_t bins = 0, dk = 0, nv = 0;
    for (int i = 0; i < np; ++i) {
        if (r->moff[i + 1] - r->moff[i] != r->npts[i]) return bad("moff step", r->moff[i + 1] - r->moff[i], r->npts[i]);
        if (r->probs[i].moff != r->moff[i]) return bad("problem moff", r->probs[i].moff, r->moff[i]);
        if (r->probs[i].bin_off != bins) return bad("problem bin_off", r->probs[i].bin_off, bins);
        if (r->probs[i].g.keyshift != r->rl.keyshift) return bad("keyshift", r->probs[i].g.keyshift, r->rl.keyshift);
        bins += r->probs[i].g.nbins;
        dk += r->n0[i] + r->n1[i];
        nv += r->ntr[i];
    }
    if (r->mtot != r->moff[np]) return bad("total points", r->mtot, r->moff[np]);
    if (r->rl.nbins != bins) return bad("bins", r->rl.nbins, bins);
    if (((bins + 1) << r->rl.keyshift) > (int64_t)UINT32_MAX) return bad("key bits", bins, r->rl.keyshift);
    if ((int64_t)r->virt.size() != nv || r->rl.nv != nv) return bad("virtual problems", r->virt.size(), nv);
    if ((int64_t)r->vunit_off.size() != nv + 1 || (int64_t)r->mode_blk.size() != nv + 1)
        return bad("per-virtual tables", r->vunit_off.size(), nv + 1);
    if ((int64_t)r->unit_virt.size() != r->vunit_off.back() || r->rl.nunits != r->vunit_off.back())
        return bad("units", r->unit_virt.size(), r->vunit_off.back());
    int64_t pieces = 0, heavy = 0, fw_end = 0, g_end = 0, tile_end = 0;
    for (int64_t k = 0; k < nv; ++k) {
        const RaggedVirt &v = r->virt[k];
        if (v.prob < 0 || v.prob >= np || v.t < 0 || v.t >= r->ntr[v.prob]) return bad("virtual problem index", v.prob, v.t);
        const GridGeom &g = r->probs[v.prob].g;
        const int64_t F = g.nf[0] * g.nf[1];
        const int want_nt = wave_transforms(r, v.prob, v.t);
        if (v.nt != want_nt) return bad("transforms per wave", v.nt, want_nt);
        if (v.m != r->npts[v.prob] || v.moff != r->moff[v.prob] || v.bin_off != r->probs[v.prob].bin_off)
            return bad("virtual problem points", v.m, r->npts[v.prob]);
        if (v.n0 != r->n0[v.prob] || v.n1 != r->n1[v.prob]) return bad("virtual problem modes", v.n0, r->n0[v.prob]);
        if (v.fw_off < 0 || v.fw_off + F > r->fw_cells) return bad("fine grid range", v.fw_off + F, r->fw_cells);
        if (v.g_off < 0 || v.g_off + v.n0 * g.nf[1] > r->g_cells) return bad("pruned buffer range", v.g_off + v.n0 * g.nf[1], r->g_cells);
        const int64_t tiles = strip_max_pieces(v.sg, v.m) * strip_tile_cells(v.sg);
        if (v.tile_next != tiles) return bad("tile stride", v.tile_next, tiles);
        if (v.tile_off < 0 || v.tile_off + tiles > r->tile_cells) return bad("tile range", v.tile_off + tiles, r->tile_cells);
        if (v.nt == 2 && (k + 1 >= nv || r->virt[k + 1].tile_off != v.tile_off + v.tile_next ||
                          r->virt[k + 1].prob != v.prob))
            return bad("paired transform tiles", k, v.prob);
        if (v.unit_off != r->vunit_off[k] || r->vunit_off[k + 1] - r->vunit_off[k] != v.sg.nunits)
            return bad("unit range", v.unit_off, r->vunit_off[k]);
        for (int u = r->vunit_off[k]; u < r->vunit_off[k + 1]; ++u)
            if (r->unit_virt[u] != k) return bad("unit owner", r->unit_virt[u], k);
        if (v.dk_off < 0 || v.dk_off + v.n0 + v.n1 > dk) return bad("1/psi_hat range", v.dk_off + v.n0 + v.n1, dk);
        const int64_t blocks = ((v.n0 + 31) / 32) * ((v.n1 + 31) / 32);
        if (r->mode_blk[k + 1] - r->mode_blk[k] != blocks) return bad("mode blocks", r->mode_blk[k + 1] - r->mode_blk[k], blocks);
        if (v.sg.nunits < 1 || v.sg.H < v.sg.ns || v.sg.S * v.sg.SW < g.nf[0] ||
            (int64_t)v.sg.K * v.sg.H < g.nf[1])
            return bad("strip geometry", v.sg.S * v.sg.SW, g.nf[0]);
        // the units' pieces: one per unit at least, one more per pmax points
        if (strip_max_pieces(v.sg, v.m) < std::min<int64_t>(v.sg.nunits, v.m) + v.m / v.sg.pmax) return bad("piece bound", strip_max_pieces(v.sg, v.m), v.sg.nunits);
        pieces += strip_max_pieces(v.sg, v.m);
        heavy += strip_max_heavy(v.sg, v.m);
        fw_end = std::max(fw_end, v.fw_off + F);
        g_end = std::max(g_end, v.g_off + v.n0 * g.nf[1]);
        tile_end = std::max(tile_end, v.tile_off + tiles);
    }
    if (ragged_strip_blocks(r->rl) < pieces) return bad("spreading workgroups", ragged_strip_blocks(r->rl), pieces);
    if (pieces != r->max_pieces || heavy != r->max_heavy) return bad("piece totals", pieces, r->max_pieces);
    if (fw_end != r->fw_cells || g_end != r->g_cells || tile_end != r->tile_cells) return bad("buffer totals", fw_end, r->fw_cells);
    if (r->rl.mode_blocks != r->mode_blk.back()) return bad("mode block total", r->rl.mode_blocks, r->mode_blk.back());
    int64_t counted = 0;
    for (const auto &c : r->fft) {
        // a class is a run of virtual problems of one fine grid and n0, contiguous in
        // fine-grid and pruned-buffer memory
        int64_t k0 = -1;
        for (int64_t k = 0; k < nv; ++k)
            if (r->virt[k].fw_off == c.fw_off) { k0 = k; break; }
        if (k0 < 0) return bad("fft class start", c.fw_off, 0);
        for (int64_t k = k0; k < k0 + c.count; ++k) {
            const RaggedVirt &v = r->virt[k];
            const GridGeom &g = r->probs[v.prob].g;
            if (g.nf[0] != c.nf0 || g.nf[1] != c.nf1 || v.n0 != c.n0 ||
                v.fw_off != c.fw_off + (k - k0) * c.nf0 * c.nf1 ||
                v.g_off != c.g_off + (k - k0) * c.n0 * c.nf1)
                return bad("fft class member", k, k0);
        }
        counted += c.count;
    }
    if (counted != nv) return bad("fft class total", counted, nv);
    return JFA_OK;
}

int allocate(jfa_ragged r) {
    const size_t real = r->is_double ? 8 : 4;
    const int np = r->nprob;
    if (int rc = upload_vec(r->probs, &r->d_probs)) return rc;
    if (int rc = upload_vec(r->virt, &r->d_virt)) return rc;
    if (int rc = upload_vec(r->moff, &r->d_moff)) return rc;
    if (int rc = upload_vec(r->vunit_off, &r->d_vunit_off)) return rc;
    if (int rc = upload_vec(r->unit_virt, &r->d_unit_virt)) return rc;
    if (int rc = upload_vec(r->mode_blk, &r->d_mode_blk)) return rc;
    JFA_HIP_CHECK(hipMalloc(&r->d_ptrs, sizeof(void *) * 4 * np));
    JFA_HIP_CHECK(hipHostMalloc((void **)&r->h_ptrs, sizeof(void *) * 4 * np, 0));
    JFA_HIP_CHECK(hipEventCreateWithFlags(&r->ptrs_copied, hipEventDisableTiming));

    // kernel tables: Horner coefficients, and 1 / psi_hat per problem and axis
    const KernelParams &kp = r->kp;
    std::vector<double> coef((size_t)kp.nc * kp.ns);
    horner_fit(kp.ns, kp.nc, kp.beta, coef.data());
    std::vector<double> dk;
    for (int i = 0; i < np; ++i) {
        for (int d = 0; d < 2; ++d) {
            const int64_t n = d == 0 ? r->n0[i] : r->n1[i];
            std::vector<double> ph((size_t)n);
            kernel_fourier(kp.ns, kp.beta, (double)r->probs[i].g.nf[d], (double)(-(n / 2)), n,
                           ph.data());
            for (double v : ph) dk.push_back(1.0 / v);
        }
    }
    int rc = r->is_double ? upload_real<double>(coef, &r->d_coef)
                          : upload_real<float>(coef, &r->d_coef);
    if (rc) return rc;
    rc = r->is_double ? upload_real<double>(dk, &r->d_dk) : upload_real<float>(dk, &r->d_dk);
    if (rc) return rc;

    // sort scratch
    const int64_t cap = std::max<int64_t>(r->mtot, 1);
    JFA_HIP_CHECK(hipMalloc(&r->d_idx, sizeof(int) * cap));
    JFA_HIP_CHECK(hipMalloc(&r->d_t, real * cap * 2));
    JFA_HIP_CHECK(hipMalloc(&r->d_key_in, sizeof(unsigned) * cap));
    JFA_HIP_CHECK(hipMalloc(&r->d_key_out, sizeof(unsigned) * cap));
    JFA_HIP_CHECK(hipMalloc(&r->d_sort_temp, radix_temp_bytes(cap)));
    JFA_HIP_CHECK(hipMalloc(&r->d_bin_start, sizeof(int) * (r->rl.nbins + 1)));
    JFA_HIP_CHECK(hipMalloc(&r->d_piece_start, sizeof(int) * (r->rl.nunits + 1)));
    JFA_HIP_CHECK(hipMalloc(&r->d_npieces, sizeof(int) * 4));
    JFA_HIP_CHECK(hipMalloc(&r->d_piece_unit, sizeof(int) * std::max<int64_t>(r->max_pieces, 1)));
    JFA_HIP_CHECK(hipMalloc(&r->d_heavy, sizeof(int) * (r->max_heavy + 1)));
    JFA_HIP_CHECK(hipMalloc(&r->d_blocksum, sizeof(int) * (2 * ((r->rl.nunits + 255) / 256) + 1)));
    const int64_t scratch = std::max<int64_t>({r->tile_cells, r->g_cells, 1});
    if (hipMalloc(&r->d_fw, 2 * real * std::max<int64_t>(r->fw_cells, 1)) != hipSuccess ||
        hipMalloc(&r->d_scratch, 2 * real * scratch) != hipSuccess) {
        (void)hipGetLastError();
        set_error("could not allocate the ragged batch's fine grids (%lld cells) and tiles (%lld)",
                  (long long)r->fw_cells, (long long)scratch);
        return JFA_ERR_ALLOC;
    }
    // per class: in-place 1D FFTs along x of every row, then along y of the
    // n0 gathered columns
    for (auto &c : r->fft) {
        const size_t len[2] = {(size_t)c.nf0, (size_t)c.nf1};
        const size_t batch[2] = {(size_t)(c.count * c.nf1), (size_t)(c.count * c.n0)};
        rocfft_plan *pl[2] = {&c.plan_x, &c.plan_y};
        for (int a = 0; a < 2; ++a) {
            std::lock_guard<std::mutex> lk(rocfft_mutex());
            rocfft_status st = rocfft_plan_create(
                pl[a], rocfft_placement_inplace,
                r->iflag > 0 ? rocfft_transform_type_complex_inverse
                             : rocfft_transform_type_complex_forward,
                r->is_double ? rocfft_precision_double : rocfft_precision_single, 1, &len[a],
                batch[a], nullptr);
            if (st != rocfft_status_success) {
                *pl[a] = nullptr;
                set_error("rocfft_plan_create failed (status %d)", (int)st);
                return JFA_ERR_FFT;
            }
            size_t ws = 0;
            rocfft_plan_get_work_buffer_size(*pl[a], &ws);
            r->fft_work_bytes = std::max(r->fft_work_bytes, ws);
        }
    }
    if (r->fft_work_bytes) JFA_HIP_CHECK(hipMalloc(&r->d_fft_work, r->fft_work_bytes));
    if (rocfft_execution_info_create(&r->fft_info) != rocfft_status_success) {
        set_error("rocfft_execution_info_create failed");
        return JFA_ERR_FFT;
    }
    if (r->fft_work_bytes)
        rocfft_execution_info_set_work_buffer(r->fft_info, r->d_fft_work, r->fft_work_bytes);

    if (r->use_graph) {
        JFA_HIP_CHECK(hipStreamCreateWithFlags(&r->work, hipStreamNonBlocking));
        JFA_HIP_CHECK(hipEventCreateWithFlags(&r->ev_in, hipEventDisableTiming));
        JFA_HIP_CHECK(hipEventCreateWithFlags(&r->ev_out, hipEventDisableTiming));
    }

    RaggedLaunch &rl = r->rl;
    rl.probs = (const RaggedProb *)r->d_probs;
    rl.virt = (const RaggedVirt *)r->d_virt;
    rl.moff = (const int64_t *)r->d_moff;
    rl.vunit_off = (const int *)r->d_vunit_off;
    rl.unit_virt = (const int *)r->d_unit_virt;
    rl.mode_blk = (const int64_t *)r->d_mode_blk;
    rl.ptrs = (const void *const *)r->d_ptrs;
    rl.bin_start = r->d_bin_start;
    rl.piece_start = r->d_piece_start;
    rl.npieces = r->d_npieces;
    rl.piece_unit = r->d_piece_unit;
    rl.heavy = r->d_heavy;
    rl.max_heavy = r->max_heavy;
    rl.reduce_chunks = 1;
    for (const RaggedVirt &v : r->virt)
        rl.reduce_chunks =
            std::max<int>(rl.reduce_chunks, (int)((strip_tile_cells(v.sg) + 255) / 256));
    rl.blocksum = r->d_blocksum;
    return JFA_OK;
}

// sorted keys and concatenated-order indices; the spreader reads each virtual
// problem's strengths through the pointer table and the Horner pairs setpts
// wrote.  (Packing (c, tx, ty) records first, as one plan does, costs more than
// it saves here: most problems are small enough for their strengths to stay in
// cache, and a problem with T transforms would pack its pairs T times.)
template <typename T>
StripPts<T> sorted(jfa_ragged r) {
    return StripPts<T>{r->mtot, r->d_idx, r->d_key_out, nullptr, nullptr, (const T *)r->d_t,
                       0, 0};
}

// Everything after the sort: spread, merge, FFT, deconvolve.
template <typename T>
int enqueue_execute(jfa_ragged r, hipStream_t s) {
    const int kem = r->opts.gpu_kerevalmeth ? 1 : 0;
    // the merge writes every fine-grid cell; with no points at all it does not run
    if (r->mtot == 0)
        if (int rc = launch_fill_zero(r->d_fw, (int64_t)(2 * sizeof(T)) * r->fw_cells, s))
            return rc;
    if (int rc = launch_ragged_strip<T>(r->rl, sorted<T>(r), (const T *)r->d_coef, kem,
                                        r->kp.beta, (T *)r->d_fw, (T *)r->d_scratch, kStripAll,
                                        s))
        return rc;
    rocfft_execution_info_set_stream(r->fft_info, s);
    for (auto &c : r->fft) {
        T *fw = (T *)r->d_fw + 2 * c.fw_off;
        T *G = (T *)r->d_scratch + 2 * c.g_off;
        void *bx[1] = {fw}, *by[1] = {G};
        rocfft_status st = rocfft_execute(c.plan_x, bx, nullptr, r->fft_info);
        if (st == rocfft_status_success) {
            if (int rc = gather_cols<T>(fw, G, c.count, c.nf1, c.nf0, c.n0, c.n0, c.nf0, s))
                return rc;
            st = rocfft_execute(c.plan_y, by, nullptr, r->fft_info);
        }
        if (st != rocfft_status_success) {
            set_error("rocfft_execute failed (status %d)", (int)st);
            return JFA_ERR_FFT;
        }
    }
    return launch_ragged_deconv<T>(r->rl, (const T *)r->d_dk, r->opts.modeord,
                                   (const T *)r->d_scratch, s);
}

template <typename T>
int run_t(jfa_ragged r, hipStream_t s) {
    SortScratch ss{r->d_key_in, r->d_key_out, r->d_sort_temp};
    if (int rc = launch_ragged_sort<T>(r->rl, ss, r->d_idx, (T *)r->d_t, s)) return rc;
    if (!r->use_graph || r->graph_state < 0) return enqueue_execute<T>(r, s);
    if (r->graph_state == 0) {
        // capture once; a library call that cannot be captured ends graph use
        // for this plan (jfa_ragged_uses_graph then returns -1 and
        // jfa_last_error says why) and the run proceeds eagerly
        auto give_up = [&](const char *where, hipError_t e) {
            (void)hipGetLastError();
            r->graph_state = -1;
            set_error("ragged plan: graph %s failed (%s); this plan launches eagerly from now on",
                      where, hipGetErrorString(e));
            return enqueue_execute<T>(r, s);
        };
        hipGraph_t graph = nullptr;
        hipError_t e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
        if (e != hipSuccess) return give_up("capture start", e);
        const int rc = enqueue_execute<T>(r, s);
        e = hipStreamEndCapture(s, &graph);
        if (rc != JFA_OK || e != hipSuccess || !graph) {
            if (graph) (void)hipGraphDestroy(graph);
            return give_up("capture", e != hipSuccess ? e : hipErrorUnknown);
        }
        e = hipGraphInstantiate(&r->gexec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (e != hipSuccess) {
            r->gexec = nullptr;
            return give_up("instantiation", e);
        }
        r->graph_state = 1;
    }
    JFA_HIP_CHECK(hipGraphLaunch(r->gexec, s));
    return JFA_OK;
}

}  // namespace

extern "C" int jfa_ragged_makeplan(int dim, int nprob, const int64_t *nmodes,
                                   const int64_t *ntransf, const int64_t *npoints, int iflag,
                                   double eps, int is_double, const jfa_opts *opts, int use_graph,
                                   jfa_ragged *plan_out) {
    if (!plan_out) {
        set_error("plan_out is NULL");
        return JFA_ERR_BAD_ARG;
    }
    *plan_out = nullptr;
    if (dim != 2) {
        set_error("ragged batches are 2D type-1 problems (dim %d requested)", dim);
        return JFA_ERR_NOT_SUPPORTED;
    }
    if (nprob < 1 || !nmodes || !ntransf || !npoints) {
        set_error("ragged batch needs nprob >= 1 and the nmodes / ntransf / npoints arrays");
        return JFA_ERR_BAD_ARG;
    }
    for (int i = 0; i < nprob; ++i) {
        if (nmodes[2 * i] < 1 || nmodes[2 * i + 1] < 1 || ntransf[i] < 1 || npoints[i] < 0) {
            set_error("ragged problem %d: modes >= 1, ntransf >= 1, npoints >= 0 required", i);
            return JFA_ERR_BAD_ARG;
        }
    }
    if (!(eps > 0)) {
        set_error("eps must be positive");
        return JFA_ERR_BAD_ARG;
    }
    jfa_opts o;
    if (opts) o = *opts;
    else jfa_default_opts(&o);
    if (!(o.upsampfac >= 1.0) || (o.modeord != 0 && o.modeord != 1) ||
        (o.kernel_width != 0 && (o.kernel_width < 2 || o.kernel_width > kMaxNs))) {
        set_error("bad options: upsampfac >= 1, modeord 0/1, kernel_width 0 or in [2, %d]",
                  kMaxNs);
        return JFA_ERR_BAD_ARG;
    }
    if (int rc = ensure_rocfft()) return rc;
    DeviceScope ds;
    if (o.gpu_device_id >= 0)
        if (int rc = ds.set(o.gpu_device_id)) return rc;

    auto *r = new jfa_ragged_s();
    r->nprob = nprob;
    r->is_double = is_double ? 1 : 0;
    r->iflag = iflag >= 0 ? 1 : -1;
    r->eps = eps;
    r->opts = o;
    r->stream = (hipStream_t)o.gpu_stream;
    r->use_graph = use_graph != 0;
    if (hipGetDevice(&r->device) != hipSuccess) r->device = 0;
    r->kp = choose_kernel(eps, o.upsampfac, o.width_rule, r->is_double, o.kernel_width);
    for (int i = 0; i < nprob; ++i) {
        r->n0.push_back(nmodes[2 * i]);
        r->n1.push_back(nmodes[2 * i + 1]);
        r->ntr.push_back(ntransf[i]);
        r->npts.push_back(npoints[i]);
    }
    int rc = layout(r);
    if (!rc) rc = check_layout(r);
    if (!rc) rc = allocate(r);
    if (rc) {
        release(r);
        delete r;
        return rc;
    }
    *plan_out = r;
    return r->kp.warn ? JFA_WARN_EPS_TOO_SMALL : JFA_OK;
}

extern "C" int jfa_ragged_check_layout(int dim, int nprob, const int64_t *nmodes,
                                       const int64_t *ntransf, const int64_t *npoints,
                                       double eps, int is_double, const jfa_opts *opts,
                                       int64_t *info) {
    if (dim != 2 || nprob < 1 || !nmodes || !ntransf || !npoints || !(eps > 0)) {
        set_error("ragged layout check: dim 2, nprob >= 1, the arrays and eps > 0 required");
        return JFA_ERR_BAD_ARG;
    }
    for (int i = 0; i < nprob; ++i)
        if (nmodes[2 * i] < 1 || nmodes[2 * i + 1] < 1 || ntransf[i] < 1 || npoints[i] < 0) {
            set_error("ragged problem %d: modes >= 1, ntransf >= 1, npoints >= 0 required", i);
            return JFA_ERR_BAD_ARG;
        }
    jfa_ragged_s r;
    if (opts) r.opts = *opts;
    else jfa_default_opts(&r.opts);
    r.nprob = nprob;
    r.is_double = is_double ? 1 : 0;
    r.eps = eps;
    r.kp = choose_kernel(eps, r.opts.upsampfac, r.opts.width_rule, r.is_double,
                         r.opts.kernel_width);
    for (int i = 0; i < nprob; ++i) {
        r.n0.push_back(nmodes[2 * i]);
        r.n1.push_back(nmodes[2 * i + 1]);
        r.ntr.push_back(ntransf[i]);
        r.npts.push_back(npoints[i]);
    }
    int rc = layout(&r);
    if (!rc) rc = check_layout(&r);
    if (!rc && info) {
        info[0] = r.mtot;
        info[1] = r.rl.nbins;
        info[2] = r.rl.nunits;
        info[3] = r.rl.nv;
        info[4] = r.fw_cells;
        info[5] = r.g_cells;
        info[6] = r.tile_cells;
        info[7] = r.max_pieces;
    }
    return rc;
}

extern "C" int jfa_ragged_run(jfa_ragged r, const void *const *points, const void *const *c,
                              void *const *f) {
    if (!r || !points || !c || !f) {
        set_error("ragged run: NULL plan or pointer table");
        return JFA_ERR_BAD_ARG;
    }
    const int np = r->nprob;
    for (int i = 0; i < np; ++i) {
        if (r->npts[i] > 0 && (!points[i] || !points[np + i] || !c[i])) {
            set_error("ragged problem %d: NULL points or strengths", i);
            return JFA_ERR_BAD_ARG;
        }
        if (!f[i]) {
            set_error("ragged problem %d: NULL output", i);
            return JFA_ERR_BAD_ARG;
        }
    }
    DeviceScope ds;
    if (int rc = ds.set(r->device)) return rc;
    hipStream_t s = r->stream;
    if (r->use_graph) {
        JFA_HIP_CHECK(hipEventRecord(r->ev_in, r->stream));
        JFA_HIP_CHECK(hipStreamWaitEvent(r->work, r->ev_in, 0));
        s = r->work;
    }
    // the previous run's table copy must have left the pinned staging buffer
    JFA_HIP_CHECK(hipEventSynchronize(r->ptrs_copied));
    for (int i = 0; i < np; ++i) {
        r->h_ptrs[i] = points[i];
        r->h_ptrs[np + i] = points[np + i];
        r->h_ptrs[2 * np + i] = c[i];
        r->h_ptrs[3 * np + i] = f[i];
    }
    JFA_HIP_CHECK(hipMemcpyAsync(r->d_ptrs, r->h_ptrs, sizeof(void *) * 4 * np,
                                 hipMemcpyHostToDevice, s));
    JFA_HIP_CHECK(hipEventRecord(r->ptrs_copied, s));
    int rc = r->is_double ? run_t<double>(r, s) : run_t<float>(r, s);
    if (rc) return rc;
    if (r->use_graph) {
        JFA_HIP_CHECK(hipEventRecord(r->ev_out, r->work));
        JFA_HIP_CHECK(hipStreamWaitEvent(r->stream, r->ev_out, 0));
    }
    return JFA_OK;
}

extern "C" int jfa_ragged_uses_graph(jfa_ragged r) {
    if (!r || !r->use_graph) return 0;
    return r->graph_state;  // 1 replaying, 0 not captured yet, -1 capture failed
}

extern "C" int jfa_ragged_set_stream(jfa_ragged r, jfa_stream_t stream) {
    if (!r) {
        set_error("plan is NULL");
        return JFA_ERR_BAD_ARG;
    }
    if ((hipStream_t)stream == r->stream) return JFA_OK;
    if (!r->use_graph) {
        // order the new stream after this plan's previous work
        hipEvent_t e;
        JFA_HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        JFA_HIP_CHECK(hipEventRecord(e, r->stream));
        JFA_HIP_CHECK(hipStreamWaitEvent((hipStream_t)stream, e, 0));
        (void)hipEventDestroy(e);
    }
    r->stream = (hipStream_t)stream;
    return JFA_OK;
}

extern "C" int jfa_ragged_destroy(jfa_ragged r) {
    if (!r) return JFA_OK;
    DeviceScope ds;
    (void)ds.set(r->device);
    hipStream_t s = r->use_graph ? r->work : r->stream;
    (void)hipStreamSynchronize(s);
    release(r);
    delete r;
    return JFA_OK;
}
