// jfa_nufft2d1f_noalloc: the 2D type-1 single-precision transform of
// jfa_nufft2d1f, for callers that may not allocate device memory (code under
// HIP graph capture, serving loops, harnesses that forbid hipMalloc).  It has
// no counterpart in the reference.
//
// Every buffer the transform needs beyond the caller's inputs and output
// lives in one file-scope device array, `scratch`, of kNoallocBytes per GPU:
// the sort keys and the sort's scratch, the strip bins and piece tables, the
// spreading records and tiles, the fine grid, the compact pruned-FFT buffer,
// the FFT twiddles and the kernel tables.  Its address on the current device
// is looked up once per device with hipGetSymbolAddress and kept; kernels are
// handed that address, never the symbol.  The kernel tables are written by
// small kernels that take them by value, and the FFTs are the LDS kernels of
// fft_lds.hip (rocFFT allocates when a plan is made), so a call queues
// kernels only: no hipMalloc, hipFree, memset or host-to-device copy.
//
// Every call on a GPU shares that GPU's array, and each call rewrites what it
// reads, so overlapping calls on one GPU (several streams or host threads)
// race; calls must be ordered.  The same kernels as jfa_nufft2d1f spread
// (strip method), so results agree with it to rounding of the FFT.
#include <algorithm>
#include <cmath>
#include <mutex>

#include "jfa_device.hpp"

using namespace jfa;

namespace {

constexpr size_t kNoallocBytes = (size_t)192 << 20;  // 192 MiB per GPU
constexpr int kNoallocMaxDevices = 64;

__device__ __align__(256) unsigned char scratch[kNoallocBytes];

std::mutex g_scratch_mu;
void *g_scratch_ptr[kNoallocMaxDevices] = {};

// The device address of `scratch` on the current device (looked up once).
int scratch_on_device(unsigned char **out) {
    int dev = 0;
    JFA_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kNoallocMaxDevices) {
        set_error("device %d beyond the %d the allocation-free path tracks", dev,
                  kNoallocMaxDevices);
        return JFA_ERR_NOT_SUPPORTED;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        JFA_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) {
            set_error("hipGetSymbolAddress returned no address for the scratch array");
            return JFA_ERR_HIP;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = static_cast<unsigned char *>(g_scratch_ptr[dev]);
    return JFA_OK;
}

// Sub-buffers of the scratch array, 256-byte aligned; with base == nullptr
// it only counts.
struct Carve {
    unsigned char *base;
    size_t off = 0;
    template <typename P>
    P *take(size_t bytes) {
        off = (off + 255) & ~(size_t)255;
        P *p = base ? reinterpret_cast<P *>(base + off) : nullptr;
        off += bytes;
        return p;
    }
};

struct HornerArg {
    float coef[kMaxNc * kMaxNs];
    int n;
};
struct FourierArg {
    double sn[kMaxFourierNodes], wt[kMaxFourierNodes];
    int q, ns;
};

__global__ void __launch_bounds__(256) write_horner_kernel(HornerArg a, float *coef) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < a.n) coef[i] = a.coef[i];
}

// dk[i] = 1 / psi_hat(2 pi (i - n/2) / nf), i < n (as kernel_fourier)
__global__ void __launch_bounds__(256)
    inv_psi_kernel(FourierArg a, double nf, int64_t n, float *dk) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double om = 2.0 * M_PI * (double)(i - n / 2) / nf;
    const double h = 0.5 * om * a.ns;
    double acc = 0.0;
    for (int p = 0; p < a.q; ++p) acc += a.wt[p] * cos(h * a.sn[p]);
    dk[i] = (float)(1.0 / (a.ns * acc));
}

// Everything one call needs, carved from the scratch array.
struct Buffers {
    unsigned *key_in, *key_out;
    void *sort_temp;
    int *idx, *bin_start, *piece_start, *npieces, *piece_unit, *heavy, *blocksum;
    float *rec, *pack, *tiles, *fw, *G, *tw0, *tw1, *coef, *dk0, *dk1;
    int64_t tile_stride;
};

Buffers carve(Carve &c, const StripGeom &sg, const GridGeom &g, int64_t M, int64_t n0,
              int64_t n1, int nc) {
    Buffers b{};
    const int64_t m = std::max<int64_t>(M, 1);
    b.key_in = c.take<unsigned>(4 * m);
    b.key_out = c.take<unsigned>(4 * m);
    b.idx = c.take<int>(4 * m);
    b.rec = c.take<float>(8 * m);
    // the sort is done before the records are packed, and has its scratch there
    b.pack = c.take<float>(std::max<size_t>(16 * m, radix_temp_bytes(m)));
    b.sort_temp = b.pack;
    b.bin_start = c.take<int>(4 * (g.nbins + 1));
    b.piece_start = c.take<int>(4 * (sg.nunits + 1));
    b.npieces = c.take<int>(16);
    b.piece_unit = c.take<int>(4 * strip_max_pieces(sg, M));
    b.heavy = c.take<int>(4 * (strip_max_heavy(sg, M) + 1));
    b.blocksum = c.take<int>(4 * (2 * ((sg.nunits + 255) / 256) + 2));
    b.tile_stride = strip_max_pieces(sg, M) * strip_tile_cells(sg);
    b.tiles = c.take<float>(8 * std::max(b.tile_stride, n0 * g.nf[1]));
    b.fw = c.take<float>(8 * g.nf[0] * g.nf[1]);
    // the FFT's compact buffer is written once the tiles are merged
    b.G = b.tiles;
    b.tw0 = c.take<float>(8 * g.nf[0]);
    b.tw1 = c.take<float>(8 * g.nf[1]);
    b.coef = c.take<float>(4 * (size_t)nc * g.ns);
    b.dk0 = c.take<float>(4 * n0);
    b.dk1 = c.take<float>(4 * n1);
    return b;
}

int run_noalloc(jfa_stream_t stream_, float eps, int64_t iflag, int64_t n_tot, int64_t n_transf,
                int64_t n_j, int64_t n_k_1, int64_t n_k_2, int64_t modeord, double upsampfac,
                int64_t gpu_method, int64_t gpu_kerevalmeth, const float *source,
                const float *px, const float *py, float *output) {
    const hipStream_t stream = (hipStream_t)stream_;
    if (n_tot < 0 || n_transf < 1 || n_j < 0 || n_j > INT32_MAX || n_k_1 < 1 || n_k_2 < 1) {
        set_error("bad sizes: n_tot=%lld n_transf=%lld n_j=%lld n_k=(%lld, %lld)",
                  (long long)n_tot, (long long)n_transf, (long long)n_j, (long long)n_k_1,
                  (long long)n_k_2);
        return JFA_ERR_BAD_ARG;
    }
    if (gpu_method != JFA_METHOD_AUTO && gpu_method != JFA_METHOD_STRIP) {
        set_error("the allocation-free entry point spreads with the strip method only "
                  "(gpu_method 0 or 3, got %lld)", (long long)gpu_method);
        return JFA_ERR_NOT_SUPPORTED;
    }
    if (modeord != 0 && modeord != 1) {
        set_error("modeord must be 0 or 1");
        return JFA_ERR_BAD_ARG;
    }
    if (!(upsampfac >= 1.0) || !(eps > 0)) {
        set_error("eps must be > 0 and upsampfac >= 1");
        return JFA_ERR_BAD_ARG;
    }
    const KernelParams kp = choose_kernel(eps, upsampfac, 0, 0, 0);
    GridGeom g{};
    g.dim = 2;
    g.ns = kp.ns;
    const int64_t n0 = n_k_1, n1 = n_k_2;
    g.nf[0] = fine_size(n0, upsampfac, kp.ns);
    g.nf[1] = fine_size(n1, upsampfac, kp.ns);
    g.nf[2] = 1;
    for (int d = 0; d < 3; ++d) {
        g.scale[d] = d < 2 ? (double)g.nf[d] / (2.0 * M_PI) : 1.0;
        g.shift[d] = 0.0;
    }
    LdsFftRadices r0, r1;
    if (!lds_fft_radices(g.nf[0], &r0) || !lds_fft_radices(g.nf[1], &r1)) {
        set_error("fine grid %lld x %lld: the allocation-free entry point handles fine grids "
                  "up to %d per axis", (long long)g.nf[0], (long long)g.nf[1], kLdsFftMax);
        return JFA_ERR_TOO_LARGE;
    }
    if (g.nf[0] < 64 || g.nf[1] < 2 * g.ns) {
        set_error("fine grid %lld x %lld is below the strip method's 64 x %d",
                  (long long)g.nf[0], (long long)g.nf[1], 2 * g.ns);
        return JFA_ERR_NOT_SUPPORTED;
    }
    StripGeom sg = strip_geometry(g, kStripPiece);
    strip_units(sg, n_j, 1, 0);

    // sizes first, against the array's capacity
    Carve count{nullptr};
    (void)carve(count, sg, g, n_j, n0, n1, kp.nc);
    if (count.off > kNoallocBytes) {
        set_error("%lld points on a %lld x %lld fine grid need %zu bytes of scratch; the "
                  "allocation-free entry point has %zu",
                  (long long)n_j, (long long)g.nf[0], (long long)g.nf[1], count.off,
                  kNoallocBytes);
        return JFA_ERR_TOO_LARGE;
    }
    if (n_tot == 0) return kp.warn ? JFA_WARN_EPS_TOO_SMALL : JFA_OK;
    unsigned char *base = nullptr;
    if (int rc = scratch_on_device(&base)) return rc;
    Carve cv{base};
    const Buffers b = carve(cv, sg, g, n_j, n0, n1, kp.nc);

    // kernel tables and twiddles
    {
        HornerArg ha{};
        double coef[kMaxNc * kMaxNs];
        horner_fit(kp.ns, kp.nc, kp.beta, coef);
        ha.n = kp.nc * kp.ns;
        for (int i = 0; i < ha.n; ++i) ha.coef[i] = (float)coef[i];
        write_horner_kernel<<<(unsigned)((ha.n + 255) / 256), 256, 0, stream>>>(ha, b.coef);
        FourierArg fa{};
        fa.ns = kp.ns;
        fa.q = kernel_fourier_nodes(kp.ns, kp.beta, fa.sn, fa.wt);
        inv_psi_kernel<<<(unsigned)((n0 + 255) / 256), 256, 0, stream>>>(fa, (double)g.nf[0],
                                                                          n0, b.dk0);
        inv_psi_kernel<<<(unsigned)((n1 + 255) / 256), 256, 0, stream>>>(fa, (double)g.nf[1],
                                                                          n1, b.dk1);
        JFA_HIP_CHECK(hipGetLastError());
        if (int rc = launch_fft_twiddles<float>(g.nf[0], b.tw0, stream)) return rc;
        if (int rc = launch_fft_twiddles<float>(g.nf[1], b.tw1, stream)) return rc;
    }
    const int sign = iflag >= 0 ? 1 : -1;
    const int kem = gpu_kerevalmeth ? 1 : 0;
    const int64_t Ntot = n0 * n1, F = g.nf[0] * g.nf[1];
    const SortScratch ss{b.key_in, b.key_out, b.sort_temp};
    const StripPts<float> pts{n_j, b.idx, b.key_out, b.pack, nullptr, nullptr, 0, 0, 0};
    for (int64_t idx = 0; idx < n_tot; ++idx) {
        // the reference's offsets (lib/kernels.cc.cu:57-60)
        const float *x = px + idx * n_j, *y = py + idx * n_j;
        const float *c = source + 2 * idx * n_j * n_transf;
        float *out = output + 2 * idx * Ntot * n_transf;
        if (n_j > 0)
            if (int rc = launch_sort_points_strip<float>(g, n_j, x, y, ss, b.bin_start, b.idx,
                                                         b.rec, stream))
                return rc;
        for (int64_t t = 0; t < n_transf; ++t) {
            if (n_j == 0) {
                if (int rc = launch_fill_zero(b.fw, 8 * F, stream)) return rc;
            } else {
                if (int rc = launch_strip_pack<float>(c + 2 * t * n_j, n_j, b.rec, n_j, 1,
                                                      b.pack, stream))
                    return rc;
                if (int rc = launch_spread_strip<float>(
                        sg, pts, b.bin_start, b.piece_start, b.npieces, b.piece_unit, b.heavy,
                        b.blocksum, b.coef, kem, kp.beta, n_j, b.fw, F, b.tiles, b.tile_stride,
                        1, kStripAll, stream))
                    return rc;
            }
            // pruned FFT: rows along x, the n0 mode columns gathered, then along y
            if (int rc = launch_fft_lds<float>(b.fw, g.nf[0], g.nf[1], b.tw0, sign, stream))
                return rc;
            if (int rc = gather_cols<float>(b.fw, b.G, 1, g.nf[1], g.nf[0], n0, n0, g.nf[0],
                                            stream))
                return rc;
            if (int rc = launch_fft_lds<float>(b.G, g.nf[1], n0, b.tw1, sign, stream)) return rc;
            if (int rc = launch_deconv_pruned_2d<float>(n0, n1, g.nf[1], b.dk0, b.dk1,
                                                        (int)modeord, b.G,
                                                        out + 2 * t * Ntot, stream))
                return rc;
        }
    }
    JFA_HIP_CHECK(hipGetLastError());
    return kp.warn ? JFA_WARN_EPS_TOO_SMALL : JFA_OK;
}

}  // namespace

extern "C" int jfa_nufft2d1f_noalloc(JFA_ATTRS_F, const void *source, const void *points_x,
                                     const void *points_y, void *output) {
    (void)n_k_3;
    (void)gpu_sort;
    (void)gpu_maxbatchsize;
    (void)debug;
    return run_noalloc(stream, eps, iflag, n_tot, n_transf, n_j, n_k_1, n_k_2, modeord,
                       upsampfac, gpu_method, gpu_kerevalmeth, (const float *)source,
                       (const float *)points_x, (const float *)points_y, (float *)output);
}
