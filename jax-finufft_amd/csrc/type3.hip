// Type-3 driver: sizes the spread grid from the extents of sources and
// targets, spreads pre-phased strengths at the rescaled sources, evaluates the
// grid at the rescaled targets with an inner type-2 plan, and post-phases.
// Replaces the type-3 path of cuFINUFFT's setpts/execute
// (lib/kernels.cc.cu:65-75).
//
// Grid rule (published FINUFFT type-3 scheme), per dimension with source
// half-width X and target half-width S:
//   X, S made safe so that X*S >= 1 (X = 0 and/or S = 0 handled);
//   nf  = next235even(max(2 sigma X S / pi + ns + 1, 2 ns));
//   h   = 2 pi / nf;   gamma = nf / (2 sigma S).
// Setpts has to read the extents back to size the grid, so type-3 setpts
// waits for the stream once (all extents in one copy); with target boxes
// (below) once more, for the box sizes.  Types 1 and 2 never wait.
//
// Target boxes.  The grid grows with the space-bandwidth product X * S; when
// the spread grid or the inner grid would exceed the cell limit (2^32, or
// opts.t3_max_cells) or half the device memory, the targets are split into
// k[0] x k[1] x k[2] boxes of half-width S / k, and every box is its own type
// 3 from all the sources to its targets, centred on the box (D_b): the grids
// shrink by k per axis at the same accuracy, for k^3 spreads of the sources.
// All boxes share one grid size, so one spread grid and one inner plan serve
// them in turn; the sources are sorted once.  The targets are put in box
// order at setpts and the outputs put back in input order at the end.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <vector>

#include "jfa_internal.hpp"
#include "plan_state.hpp"

using namespace jfa;

namespace {

void free_ptr(void *&p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}

void type3_grid(double X, double S, double sigma, int ns, int64_t *nf, double *h,
                double *gam) {
    double Xs = X, Ss = S;
    if (X == 0.0) {
        if (S == 0.0) {
            Xs = 1.0;
            Ss = 1.0;
        } else {
            Xs = std::max(Xs, 1.0 / S);
        }
    } else {
        Ss = std::max(Ss, 1.0 / X);
    }
    double nfd = 2.0 * sigma * Ss * Xs / M_PI + (ns + 1);
    if (!std::isfinite(nfd)) nfd = 0.0;
    int64_t n = (int64_t)nfd;
    if (n < 2 * ns) n = 2 * ns;
    n = next235even(n);
    *nf = n;
    *h = 2.0 * M_PI / (double)n;
    *gam = (double)n / (2.0 * sigma * Ss);
}

// Every target's frequency is at most h gam S = pi / sigma radians per cell (see
// type3_grid; boxes of targets overlap by rounding only).
double fourier_range(jfa_plan p) { return 1.02 * M_PI / p->opts.upsampfac; }

}  // namespace

int jfa::type3_init(jfa_plan p) {
    p->geom.dim = p->dim;
    p->geom.ns = p->kp.ns;
    // Horner table (the spread kernel) and the table for psi_hat
    int rc = upload_kernel_tables(p, nullptr);
    if (rc) return rc;
    const int ns = p->kp.ns;
    std::vector<double> table(2 * kMaxFourierNodes);
    int n;
    if (p->is_double) {
        n = kernel_fourier_nodes(ns, p->kp.beta, table.data() + kMaxFourierNodes, table.data());
        std::copy_n(table.begin() + kMaxFourierNodes, n, table.begin() + n);
        n *= 2;
    } else {
        n = kernel_fourier_series(ns, p->kp.beta, fourier_range(p), table.data());
    }
    JFA_HIP_CHECK(hipMalloc(&p->d_quad, sizeof(double) * n));
    JFA_HIP_CHECK(hipMemcpy(p->d_quad, table.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    // [min, max] of up to six arrays, then the partials of one pass
    JFA_HIP_CHECK(hipMalloc(&p->d_minmax, sizeof(double) * (12 + 2 * 1024)));
    return JFA_OK;
}

void jfa::type3_free(jfa_plan p) {
    free_ptr(p->d_cp);
    free_ptr(p->d_t3_deconv);
    free_ptr(reinterpret_cast<void *&>(p->d_t3_count));
    free_ptr(reinterpret_cast<void *&>(p->d_t3_start));
    free_ptr(reinterpret_cast<void *&>(p->d_t3_perm));
    free_ptr(p->d_t3_sorted);
    free_ptr(p->d_t3_out);
    free_ptr(reinterpret_cast<void *&>(p->d_minmax));
    free_ptr(p->d_quad);
}

// [min, max] of every source and target coordinate array (2 dim arrays), one
// copy and one wait for all of them.
template <typename T>
static int extents(jfa_plan p, int64_t M, const T *const xs[3], int64_t N,
                   const T *const ss[3], double mm[12]) {
    const int dim = p->dim;
    for (int i = 0; i < 12; ++i) mm[i] = 0.0;
    for (int d = 0; d < dim; ++d) {
        if (M > 0)
            if (int rc = launch_minmax_to<T>(M, xs[d], p->d_minmax + 4 * d, p->d_minmax + 12,
                                             p->stream))
                return rc;
        if (N > 0)
            if (int rc = launch_minmax_to<T>(N, ss[d], p->d_minmax + 4 * d + 2,
                                             p->d_minmax + 12, p->stream))
                return rc;
    }
    if (M == 0 && N == 0) return JFA_OK;
    double h[12];
    JFA_HIP_CHECK(hipMemcpyAsync(h, p->d_minmax, sizeof(double) * 4 * dim,
                                 hipMemcpyDeviceToHost, p->stream));
    JFA_HIP_CHECK(hipStreamSynchronize(p->stream));
    for (int d = 0; d < dim; ++d) {
        if (M > 0) {
            mm[4 * d] = h[4 * d];
            mm[4 * d + 1] = h[4 * d + 1];
        }
        if (N > 0) {
            mm[4 * d + 2] = h[4 * d + 2];
            mm[4 * d + 3] = h[4 * d + 3];
        }
    }
    return JFA_OK;
}

// Boxes per axis for the targets: the fewest (growing the axis with the
// largest grid first) whose spread and inner grids stay within the cell limit
// and, with the inner plan's pruned-FFT buffer, within half the device memory.
static int choose_boxes(jfa_plan p, const double X[3], const double S[3], int k[3]) {
    const int dim = p->dim, ns = p->kp.ns;
    const double sigma = p->opts.upsampfac;
    const int64_t cell_limit = p->opts.t3_max_cells > 0
                                   ? std::min<int64_t>(p->opts.t3_max_cells, kMaxFineCells)
                                   : kMaxFineCells;
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) {
        (void)hipGetLastError();
        total_b = (size_t)64 << 30;
    }
    const double budget = 0.5 * (double)total_b;
    const double cell_bytes = 2.0 * (p->is_double ? 8 : 4) * p->batch;
    for (int d = 0; d < 3; ++d) k[d] = 1;
    for (;;) {
        int64_t nf[3] = {1, 1, 1}, nfi[3] = {1, 1, 1};
        double F = 1, Fi = 1;
        for (int d = 0; d < dim; ++d) {
            double h, gam;
            type3_grid(X[d], S[d] / k[d], sigma, ns, &nf[d], &h, &gam);
            nfi[d] = fine_size(nf[d], sigma, ns);
            F *= (double)nf[d];
            Fi *= (double)nfi[d];
        }
        const double compact = dim >= 2 ? Fi * (double)nf[0] / (double)nfi[0] : 0.0;
        const bool fits = F <= (double)cell_limit && Fi <= (double)cell_limit &&
                          (F + Fi + compact) * cell_bytes <= budget;
        bool axis_ok = true;
        for (int d = 0; d < dim; ++d) axis_ok = axis_ok && nf[d] <= ((int64_t)1 << 30);
        if (fits && axis_ok) return JFA_OK;
        int dbig = -1;
        for (int d = 0; d < dim; ++d)
            if (S[d] > 0 && (dbig < 0 || nf[d] > nf[dbig])) dbig = d;
        if (dbig < 0 || (int64_t)k[0] * k[1] * k[2] >= 4096) {
            set_error("type-3 grids of %.3g / %.3g cells exceed the limits even with %d target "
                      "boxes (space-bandwidth product too large)",
                      F, Fi, k[0] * k[1] * k[2]);
            return JFA_ERR_TOO_LARGE;
        }
        ++k[dbig];
    }
}

// Centre of target box b (x fastest) along every axis.
static void box_centre(jfa_plan p, int b, double D[3]) {
    for (int d = 0; d < 3; ++d) {
        const int bd = b % p->t3_k[d];
        b /= p->t3_k[d];
        D[d] = d < p->dim ? p->t3_box_lo[d] + (bd + 0.5) * p->t3_box_w[d] : 0.0;
    }
}

template <typename T>
static int type3_setpts_t(jfa_plan p, int64_t M, const T *const xs[3], int64_t N,
                          const T *const ss[3]) {
    const int dim = p->dim;
    const int ns = p->kp.ns;
    const double sigma = p->opts.upsampfac;
    GridGeom &g = p->geom;
    double hg[3] = {1, 1, 1}, X[3] = {0, 0, 0}, S[3] = {0, 0, 0}, smin[3] = {0, 0, 0};
    for (int d = 0; d < 3; ++d) {
        g.nf[d] = 1;
        g.scale[d] = 1.0;
        g.shift[d] = 0.0;
        p->t3_C[d] = p->t3_D[d] = 0.0;
        p->t3_box_lo[d] = 0.0;
        p->t3_box_w[d] = 1.0;
    }
    double mm[12];
    if (int rc = extents<T>(p, M, xs, N, ss, mm)) return rc;
    for (int d = 0; d < dim; ++d) {
        p->t3_C[d] = 0.5 * (mm[4 * d + 1] + mm[4 * d]);
        X[d] = 0.5 * (mm[4 * d + 1] - mm[4 * d]);
        p->t3_D[d] = 0.5 * (mm[4 * d + 3] + mm[4 * d + 2]);
        S[d] = 0.5 * (mm[4 * d + 3] - mm[4 * d + 2]);
        smin[d] = mm[4 * d + 2];
    }
    int k[3];
    if (int rc = choose_boxes(p, X, S, k)) return rc;
    const int nbox = k[0] * k[1] * k[2];
    for (int d = 0; d < dim; ++d) {
        int64_t nf;
        double h, gam;
        type3_grid(X[d], S[d] / k[d], sigma, ns, &nf, &h, &gam);
        g.nf[d] = nf;
        g.scale[d] = (double)nf / (2.0 * M_PI) / gam;  // u = (x - C)/gam / h
        g.shift[d] = p->t3_C[d];
        p->t3_gam[d] = gam;
        p->t3_h[d] = h;
        hg[d] = h * gam;
        p->t3_box_lo[d] = smin[d];
        // a flat axis (no target extent) has one box of width 0 centred on
        // the targets' common coordinate
        p->t3_box_w[d] = S[d] > 0 ? 2.0 * S[d] / k[d] : 0.0;
        p->t3_k[d] = k[d];
    }
    for (int d = dim; d < 3; ++d) p->t3_k[d] = 1;
    p->t3_nbox = nbox;
    p->F = g.nf[0] * g.nf[1] * g.nf[2];
    p->Ntot = N;
    // bins and method for the new grid
    {
        const int b2 = 32, b1 = 1024;
        int bs[3] = {1, 1, 1};
        if (dim == 1) bs[0] = b1;
        if (dim == 2) bs[0] = bs[1] = b2;
        if (dim == 3) bs[0] = bs[1] = bs[2] = 8;
        g.nbins = 1;
        for (int d = 0; d < 3; ++d) {
            int b = d < dim ? bs[d] : 1;
            if (d < dim) b = (int)std::min<int64_t>(b, std::max<int64_t>(1, g.nf[d] / 2));
            g.bs[d] = b;
            g.nb[d] = (int)((g.nf[d] + b - 1) / b);
            g.nbins *= g.nb[d];
        }
        size_t cells = 1;
        for (int d = 0; d < dim; ++d) cells *= (size_t)(g.bs[d] + ns - 1);
        const bool fits = cells * 2 * sizeof(T) <= 64 * 1024;
        g.ymajor = 0;
        p->method = p->opts.gpu_method == JFA_METHOD_GM_SORT || !fits ? JFA_METHOD_GM_SORT
                                                                      : JFA_METHOD_SM;
        p->method_by_density = p->opts.gpu_method == JFA_METHOD_AUTO && fits;
        const int om = p->opts.gpu_method;
        if ((om == JFA_METHOD_AUTO || om == JFA_METHOD_STRIP) && strip_applicable(p)) {
            int rc = setup_strip(p);
            if (rc) return rc;
            p->method = JFA_METHOD_STRIP;
            p->method_by_density = false;  // the density choice is between the other two
        }
    }
    // fine grid and prephase buffers
    if (p->F * p->batch > p->t3_nf_cap) {
        free_ptr(p->d_fw);
        p->t3_nf_cap = 0;
        const size_t bytes = (size_t)p->F * p->batch * 2 * sizeof(T);
        if (hipMalloc(&p->d_fw, bytes) != hipSuccess) {
            (void)hipGetLastError();
            set_error("could not allocate the %zu-byte type-3 grid", bytes);
            return JFA_ERR_ALLOC;
        }
        p->t3_nf_cap = p->F * p->batch;
    }
    if (M * p->batch > p->cap_cp) {
        free_ptr(p->d_cp);
        JFA_HIP_CHECK(hipMalloc(&p->d_cp, (size_t)std::max<int64_t>(M * p->batch, 1) * 2 * sizeof(T)));
        p->cap_cp = M * p->batch;
    }
    if (N > p->cap_t3_deconv) {
        free_ptr(p->d_t3_deconv);
        JFA_HIP_CHECK(hipMalloc(&p->d_t3_deconv, (size_t)std::max<int64_t>(N, 1) * sizeof(T)));
        p->cap_t3_deconv = N;
    }
    // sort the sources on the spread grid
    int rc = setpts_12(p, M, xs[0], xs[1], xs[2]);
    if (rc) return rc;
    // inner type-2 plan from the spread grid (FFT-ordered modes) to the targets
    const int64_t nm[3] = {g.nf[0], g.nf[1], g.nf[2]};
    if (p->inner) {
        bool same = true;
        for (int d = 0; d < dim; ++d) same = same && p->inner->nmodes[d] == nm[d];
        if (!same) {
            jfa_destroy(p->inner);
            p->inner = nullptr;
        }
    }
    if (!p->inner) {
        jfa_opts io = p->opts;
        io.modeord = 1;
        io.gpu_spreadinterponly = 0;
        io.kernel_width = ns;
        io.gpu_stream = p->stream;
        io.gpu_device_id = p->device;
        // cubic bins: the inner plan's few targets per bin take the global method
        // by density, whose sort only wants locality
        io.gpu_binsizex = io.gpu_binsizey = io.gpu_binsizez = dim == 3 ? 8 : 0;
        rc = jfa_makeplan(2, dim, nm, p->iflag, p->batch, p->eps, p->is_double, &io, &p->inner);
        if (rc > 1) return rc;
    }
    p->inner->stream = p->stream;
    p->inner->used = true;
    for (int d = 0; d < dim; ++d) {
        p->inner->geom.shift[d] = p->t3_D[d];
        p->inner->geom.scale[d] = (double)p->inner->geom.nf[d] / (2.0 * M_PI) * hg[d];
    }
    // Kept rows of the inner grid.  A box's targets lie within S/k of its
    // centre, i.e. within +-nf_i / (2 sigma) cells of cell 0 of the inner grid
    // (about its middle half at sigma = 2); their first taps, the LDS tiles of
    // their bins (at most one bin before and bs + ns - 1 cells after a first
    // tap) and a cell of rounding margin are all the interpolation reads.  The
    // y (and z) axes keep only those rows, so the last FFT passes run over them
    // alone; the x axis, transformed last, stays whole.
    {
        GridGeom &gi = p->inner->geom;
        for (int d = 0; d < 3; ++d) gi.wstart[d] = gi.wlen[d] = 0;
        for (int d = 1; d < dim; ++d) {
            const double half = S[d] / k[d] * gi.scale[d];
            const int64_t nfi = gi.nf[d], bs = gi.bs[d];
            const int64_t lo = (int64_t)std::floor(-half - 0.5 * ns) - 1;
            const int64_t hi = (int64_t)std::ceil(half - 0.5 * ns) + 1;
            const int64_t a = lo - bs - 1, b = hi + bs + ns + 1;  // inclusive, unwrapped
            if (b - a + 1 < nfi) {
                gi.wstart[d] = ((a % nfi) + nfi) % nfi;
                gi.wlen[d] = b - a + 1;
            }
        }
    }
    for (int d = 0; d < 3; ++d) {
        p->t3_x[d] = xs[d];
        p->t3_s[d] = ss[d];
    }
    if (nbox == 1) {
        rc = setpts_12(p->inner, N, ss[0], ss[1], ss[2]);
        if (rc) return rc;
        return launch_t3_deconv_factors<T>(dim, N, ss[0], ss[1], ss[2], p->t3_D, hg, ns,
                                           fourier_range(p), (const double *)p->d_quad,
                                           (T *)p->d_t3_deconv, p->stream);
    }
    // target boxes: box order, box sizes on the host, per-box deconvolution
    // factors, and room for the largest box in the inner plan
    if (nbox > p->t3_cap_box) {
        free_ptr(reinterpret_cast<void *&>(p->d_t3_count));
        free_ptr(reinterpret_cast<void *&>(p->d_t3_start));
        p->t3_cap_box = 0;
        JFA_HIP_CHECK(hipMalloc(&p->d_t3_count, sizeof(int) * 2 * nbox));
        JFA_HIP_CHECK(hipMalloc(&p->d_t3_start, sizeof(int64_t) * (nbox + 1)));
        p->t3_cap_box = nbox;
    }
    if (N > p->t3_cap_n) {
        free_ptr(reinterpret_cast<void *&>(p->d_t3_perm));
        free_ptr(p->d_t3_sorted);
        free_ptr(p->d_t3_out);
        p->t3_cap_n = 0;
        JFA_HIP_CHECK(hipMalloc(&p->d_t3_perm, sizeof(int) * std::max<int64_t>(N, 1)));
        JFA_HIP_CHECK(hipMalloc(&p->d_t3_sorted, sizeof(T) * 3 * std::max<int64_t>(N, 1)));
        JFA_HIP_CHECK(hipMalloc(&p->d_t3_out,
                                sizeof(T) * 2 * p->batch * std::max<int64_t>(N, 1)));
        p->t3_cap_n = N;
    }
    BoxGrid bg;
    for (int d = 0; d < 3; ++d) {
        bg.lo[d] = p->t3_box_lo[d];
        bg.width[d] = p->t3_box_w[d];
        bg.k[d] = p->t3_k[d];
    }
    T *sorted = (T *)p->d_t3_sorted;
    rc = launch_t3_box_sort<T>(dim, N, ss[0], ss[1], ss[2], bg, nbox, p->d_t3_count,
                               p->d_t3_start, p->d_t3_perm, sorted, p->stream);
    if (rc) return rc;
    p->t3_box_start.assign((size_t)nbox + 1, 0);
    if (N > 0) {
        JFA_HIP_CHECK(hipMemcpyAsync(p->t3_box_start.data(), p->d_t3_start,
                                     sizeof(int64_t) * (nbox + 1), hipMemcpyDeviceToHost,
                                     p->stream));
        JFA_HIP_CHECK(hipStreamSynchronize(p->stream));
    }
    int64_t biggest = 0;
    for (int b = 0; b < nbox; ++b) {
        const int64_t s0 = p->t3_box_start[b], nb = p->t3_box_start[b + 1] - s0;
        biggest = std::max(biggest, nb);
        if (nb == 0) continue;
        double Db[3];
        box_centre(p, b, Db);
        const T *sb[3] = {nullptr, nullptr, nullptr};
        for (int d = 0; d < dim; ++d) sb[d] = sorted + (int64_t)d * N + s0;
        rc = launch_t3_deconv_factors<T>(dim, nb, sb[0], sb[1], sb[2], Db, hg, ns,
                                         fourier_range(p), (const double *)p->d_quad,
                                         (T *)p->d_t3_deconv + s0, p->stream);
        if (rc) return rc;
    }
    return reserve_points(p->inner, biggest);
}

int jfa::type3_setpts(jfa_plan p, int64_t M, const void *x, const void *y, const void *z,
                      int64_t N, const void *s, const void *t, const void *u) {
    if (M < 0 || M > INT32_MAX || N < 0 || N > INT32_MAX) {
        set_error("type-3 point counts must be in [0, 2^31)");
        return JFA_ERR_TOO_LARGE;
    }
    const void *xs[3] = {x, y, z}, *ss[3] = {s, t, u};
    for (int d = 0; d < p->dim; ++d) {
        if ((M > 0 && !xs[d]) || (N > 0 && !ss[d])) {
            set_error("type-3 coordinates for dimension %d are NULL", d);
            return JFA_ERR_BAD_ARG;
        }
    }
    for (int d = p->dim; d < 3; ++d) xs[d] = ss[d] = nullptr;
    if (p->is_double) {
        const double *xd[3] = {(const double *)xs[0], (const double *)xs[1], (const double *)xs[2]};
        const double *sd[3] = {(const double *)ss[0], (const double *)ss[1], (const double *)ss[2]};
        return type3_setpts_t<double>(p, M, xd, N, sd);
    }
    const float *xf[3] = {(const float *)xs[0], (const float *)xs[1], (const float *)xs[2]};
    const float *sf[3] = {(const float *)ss[0], (const float *)ss[1], (const float *)ss[2]};
    return type3_setpts_t<float>(p, M, xf, N, sf);
}

// Execute over target boxes: per box, pre-phase with its centre, spread all
// sources, evaluate its targets with the inner plan (set to the box centre)
// and post-phase; then every output back to the input order of the targets.
template <typename T>
static int type3_execute_boxes(jfa_plan p, const T *c, T *f) {
    const int dim = p->dim;
    const int64_t M = p->M, N = p->Ntot;
    const T *x[3] = {(const T *)p->t3_x[0], (const T *)p->t3_x[1], (const T *)p->t3_x[2]};
    const T *sorted = (const T *)p->d_t3_sorted;
    const T *dec = (const T *)p->d_t3_deconv;
    T *fw = (T *)p->d_fw;
    T *out = (T *)p->d_t3_out;
    int rc;
    for (int t0 = 0; t0 < p->ntransf; t0 += p->batch) {
        const int nb = std::min(p->batch, p->ntransf - t0);
        const T *cb = c + 2 * (int64_t)t0 * M;
        for (int b = 0; b < p->t3_nbox; ++b) {
            const int64_t s0 = p->t3_box_start[b], nbx = p->t3_box_start[b + 1] - s0;
            if (nbx == 0) continue;
            double Db[3];
            box_centre(p, b, Db);
            const T *sb[3] = {nullptr, nullptr, nullptr};
            for (int d = 0; d < dim; ++d) sb[d] = sorted + (int64_t)d * N + s0;
            if ((rc = launch_t3_prephase<T>(dim, M, nb, x[0], x[1], x[2], p->t3_C, Db, p->iflag,
                                            cb, (T *)p->d_cp, p->stream)))
                return rc;
            if (p->method != JFA_METHOD_STRIP)
                if ((rc = launch_fill_zero(fw, (int64_t)sizeof(T) * 2 * p->F * nb, p->stream)))
                    return rc;
            if ((rc = spread_any<T>(p, (const T *)p->d_cp, M, fw, p->F, nb))) return rc;
            for (int d = 0; d < dim; ++d) p->inner->geom.shift[d] = Db[d];
            if ((rc = setpts_12(p->inner, nbx, sb[0], sb[1], sb[2]))) return rc;
            T *ob = out + 2 * (int64_t)nb * s0;  // this box's outputs, [t][nbx]
            const int saved = p->inner->ntransf;
            p->inner->ntransf = nb;
            rc = execute_12<T>(p->inner, ob, fw);
            p->inner->ntransf = saved;
            if (rc) return rc;
            if ((rc = launch_t3_postphase<T>(dim, nbx, nb, sb[0], sb[1], sb[2], p->t3_C,
                                             p->iflag, dec + s0, ob, p->stream)))
                return rc;
        }
        if ((rc = launch_t3_unsort<T>(N, nb, p->t3_nbox, p->d_t3_start, p->d_t3_perm, out,
                                      f + 2 * (int64_t)t0 * N, p->stream)))
            return rc;
    }
    return JFA_OK;
}

template <typename T>
static int type3_execute_t(jfa_plan p, const T *c, T *f) {
    const int dim = p->dim;
    const int64_t M = p->M, N = p->Ntot;
    if (N == 0) return JFA_OK;
    if (M == 0) return launch_fill_zero(f, (int64_t)sizeof(T) * 2 * N * p->ntransf, p->stream);
    const T *x[3] = {(const T *)p->t3_x[0], (const T *)p->t3_x[1], (const T *)p->t3_x[2]};
    const T *s[3] = {(const T *)p->t3_s[0], (const T *)p->t3_s[1], (const T *)p->t3_s[2]};
    const SortedPts<T> pts = sorted_view<T>(p);
    const BinIndex bi = bin_view(p);
    const int kem = p->opts.gpu_kerevalmeth ? 1 : 0;
    bool phase = false;
    for (int d = 0; d < dim; ++d) phase = phase || p->t3_D[d] != 0.0;
    T *fw = (T *)p->d_fw;
    int rc;
    if (p->t3_nbox > 1) return type3_execute_boxes<T>(p, c, f);
    for (int t0 = 0; t0 < p->ntransf; t0 += p->batch) {
        const int nb = std::min(p->batch, p->ntransf - t0);
        const T *cb = c + 2 * (int64_t)t0 * M;
        T *fb = f + 2 * (int64_t)t0 * N;
        const T *src = cb;
        if (phase) {
            if ((rc = launch_t3_prephase<T>(dim, M, nb, x[0], x[1], x[2], p->t3_C, p->t3_D,
                                            p->iflag, cb, (T *)p->d_cp, p->stream)))
                return rc;
            src = (const T *)p->d_cp;
        }
        // the strip spreader writes every cell itself
        if (p->method != JFA_METHOD_STRIP)
            if ((rc = launch_fill_zero(fw, (int64_t)sizeof(T) * 2 * p->F * nb, p->stream)))
                return rc;
        if ((rc = spread_any<T>(p, src, M, fw, p->F, nb))) return rc;
        const int saved = p->inner->ntransf;
        p->inner->ntransf = nb;
        rc = execute_12<T>(p->inner, fb, fw);
        p->inner->ntransf = saved;
        if (rc) return rc;
        if ((rc = launch_t3_postphase<T>(dim, N, nb, s[0], s[1], s[2], p->t3_C, p->iflag,
                                         (const T *)p->d_t3_deconv, fb, p->stream)))
            return rc;
    }
    return JFA_OK;
}

int jfa::type3_execute(jfa_plan p, void *c, void *fk) {
    if ((p->M > 0 && !c) || (p->Ntot > 0 && !fk)) {
        set_error("execute: NULL data pointer");
        return JFA_ERR_BAD_ARG;
    }
    if (!p->inner && p->M > 0 && p->Ntot > 0) {
        set_error("type-3 execute before setpts");
        return JFA_ERR_BAD_ARG;
    }
    if (p->is_double) return type3_execute_t<double>(p, (const double *)c, (double *)fk);
    return type3_execute_t<float>(p, (const float *)c, (float *)fk);
}
