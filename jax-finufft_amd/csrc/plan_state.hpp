// The plan object behind the opaque jfa_plan handle.
#pragma once

#include <climits>
#include <map>
#include <utility>
#include <string>
#include <vector>

#include "jfa_internal.hpp"

struct jfa_plan_s {
    int type = 1, dim = 1, is_double = 0, iflag = 1, ntransf = 1, batch = 1;
    double eps = 1e-6;
    int64_t nmodes[3] = {1, 1, 1};  // x fastest; 1 for unused dims
    int64_t Ntot = 1;               // modes per transform (targets for type 3)
    int64_t F = 1;                  // fine-grid cells per transform
    jfa_opts opts{};
    jfa::KernelParams kp;
    jfa::GridGeom geom{};
    int method = JFA_METHOD_SM;
    bool method_by_density = false;  // auto method: LDS tiles or global atomics, chosen
                                     // at setpts from the point density
    bool keyed = false;              // sorted points without a gather: d_key_out + d_t
                                     // (point-major), see SortedPts
    int maxsub = 4096;               // most points per LDS subproblem on the current points
    hipStream_t stream = nullptr;
    int device = 0;
    bool used = false;                 // work has been queued on `stream`
    hipEvent_t order_event = nullptr;  // orders work across jfa_set_stream

    // stage timing (opts.debug == 2): recorded event pairs, resolved on query
    struct TimingPair {
        const char *name;
        hipEvent_t a, b;
    };
    std::vector<TimingPair> timing_pairs;
    std::vector<hipEvent_t> timing_events;
    std::map<std::string, std::pair<double, int64_t>> timing_acc;

    // kernel tables
    void *d_coef = nullptr;            // Horner coefficients (nc x ns)
    void *d_dk[3] = {nullptr, nullptr, nullptr};  // 1 / psi_hat per dim
    void *d_fw = nullptr;              // batch x F complex fine grid
    bool fw_modes = false;             // d_fw holds the amplified, transformed modes of
                                       // every transform of the last type-2 pass

    // rocFFT
    std::map<int, rocfft_plan> fft_plans;  // by batch count
    std::map<std::pair<int64_t, int64_t>, rocfft_plan> fft1_plans;  // 1D, by (length, batch)
    // pruned FFT passes (fft_axis.hip) where every axis supports them
    bool axis_ok = false;
    jfa::AxisFft axis[3] = {};
    void *d_tw[3] = {nullptr, nullptr, nullptr};  // twiddles, by axis
    void *d_fwt = nullptr;             // compact buffer of the pruned 2D / 3D FFT
    size_t fwt_bytes = 0;
    rocfft_execution_info fft_info = nullptr;
    void *d_fft_work = nullptr;
    size_t fft_work_bytes = 0;

    // sorted points
    int64_t M = 0, cap_M = 0, cap_bins = 0;
    int *d_idx = nullptr, *d_l0 = nullptr;
    void *d_t = nullptr;
    unsigned *d_key_in = nullptr, *d_key_out = nullptr;  // radix sort
    void *d_sort_temp = nullptr;
    int *d_bin_start = nullptr, *d_sub_start = nullptr, *d_nsub = nullptr;

    // 2D strip spreader
    jfa::StripGeom sg{};
    int *d_piece_start = nullptr, *d_npieces = nullptr;
    int *d_piece_unit = nullptr;  // unit of every piece
    int64_t piece_unit_cap = 0;
    int *d_heavy = nullptr;       // [count, crowded units], 1 + strip_max_heavy(sg, M)
    int64_t heavy_cap = 0;
    int *d_strip_blocksum = nullptr;   // piece-scan block sums, 2 ceil(units / 256) + 1
    void *d_strip_scratch = nullptr;
    size_t strip_scratch_bytes = 0;
    int64_t strip_scratch_stride = 0;  // complex cells per transform
    void *d_pack = nullptr;            // strip_batch x M records (c, tx, ty)
    size_t pack_bytes = 0;
    int strip_batch = 1;               // transforms spread at a time: the batch, or as many as
                                       // there was memory for
    int strip_batch_most = INT_MAX;    // (found by a failed allocation)
    int64_t strip_most_M = INT64_MAX;  // point counts up to which auto spreads by strips
                                       // (there was no memory for more)

    // type 3
    jfa_plan inner = nullptr;     // type-2 plan from the spread grid to the targets
    const void *t3_x[3] = {nullptr, nullptr, nullptr};   // user source coordinates
    const void *t3_s[3] = {nullptr, nullptr, nullptr};   // user target coordinates
    double t3_C[3] = {0, 0, 0}, t3_D[3] = {0, 0, 0};      // source / target centres
    double t3_gam[3] = {1, 1, 1}, t3_h[3] = {1, 1, 1};
    int64_t t3_nf_cap = 0;        // fine-grid cells allocated for d_fw
    void *d_cp = nullptr;         // prephased strengths, batch x M complex
    int64_t cap_cp = 0;
    void *d_t3_deconv = nullptr;  // per-target 1 / prod psi_hat (real)
    int64_t cap_t3_deconv = 0;
    double *d_minmax = nullptr;   // scratch for extents (6 x [min, max]) and their partials
    void *d_quad = nullptr;       // quadrature (fp64) or series (fp32) of psi_hat at arbitrary omega
    // type 3 over boxes of targets, when one pair of grids would exceed the
    // cell limit or the memory budget: k[d] boxes per axis of width
    // t3_box_w[d] from t3_box_lo[d]; targets in box order
    int t3_k[3] = {1, 1, 1};
    int t3_nbox = 1;
    double t3_box_lo[3] = {0, 0, 0}, t3_box_w[3] = {1, 1, 1};
    std::vector<int64_t> t3_box_start;  // host copy, nbox + 1
    int *d_t3_count = nullptr;          // 2 * nbox
    int64_t *d_t3_start = nullptr;      // nbox + 1
    int *d_t3_perm = nullptr;           // box order -> target
    void *d_t3_sorted = nullptr;        // dim x N coordinates in box order
    void *d_t3_out = nullptr;           // batch x N outputs in box order
    int64_t t3_cap_box = 0, t3_cap_n = 0;
};

namespace jfa {

int fft_exec(jfa_plan p, void *data, int nbatch);
// In-place 1D FFTs of `batch` contiguous rows of `len` complex values.
int fft1d(jfa_plan p, void *data, int64_t len, int64_t batch);
// Pruned FFT between the fine grid and the modes (fft_pruned.hip), 2D / 3D:
// type 1 runs pruned_grid_fft then pruned_deconv, type 2 pruned_amplify then
// pruned_modes_fft; fw holds nb transforms at stride F.
bool fft_is_pruned(jfa_plan p);
template <typename T>
int pruned_grid_fft(jfa_plan p, T *fw, int nb);
template <typename T>
int pruned_deconv(jfa_plan p, T *fw, T *fk, int nb);
template <typename T>
int pruned_amplify(jfa_plan p, const T *fk, T *fw, int nb);
template <typename T>
int pruned_modes_fft(jfa_plan p, T *fw, int nb);
// The same between the grid fw and the modes fk in one pass per axis, scaling
// included (fft_axis.hip; plans with axis_ok), through a work buffer of n0 x nf1
// (x nf2) values per transform.
int reserve_fwt(jfa_plan p);
template <typename T>
int axis_grid_to_modes(jfa_plan p, T *fw, T *work, T *fk, int nb);
template <typename T>
int axis_modes_to_grid(jfa_plan p, const T *fk, T *work, T *fw, int nb);
// Gives back the spreader's tiles and records; the next call allocates them again.
void release_strip_scratch(jfa_plan p);
bool strip_applicable(jfa_plan p);
int setup_strip(jfa_plan p);
int upload_kernel_tables(jfa_plan p, const int64_t *nmodes_for_dk);
int default_maxsub(jfa_plan p);
int reserve_points(jfa_plan p, int64_t M);
int setpts_12(jfa_plan p, int64_t M, const void *x, const void *y, const void *z);
template <typename T>
SortedPts<T> sorted_view(jfa_plan p);
BinIndex bin_view(jfa_plan p);
template <typename T>
int execute_12(jfa_plan p, T *c, T *fk);
template <typename T>
int spread_any(jfa_plan p, const T *c, int64_t c_stride, T *fw, int64_t fw_stride, int ntr);

int type3_init(jfa_plan p);
int type3_setpts(jfa_plan p, int64_t M, const void *x, const void *y, const void *z, int64_t N,
                 const void *s, const void *t, const void *u);
int type3_execute(jfa_plan p, void *c, void *fk);
void type3_free(jfa_plan p);

}  // namespace jfa
