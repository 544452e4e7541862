// cuna_plan.hpp -- per-x plan: binned points, filter constants, workspaces.
//
// A plan is the MI355X counterpart of the reference's filter_properties +
// plan pair (inc/cuna_typedefs.h:92-148, src/gaussian_filter.cu:102-164): it
// is built once per set of sample positions and reused for every y.
#pragma once

#include <memory>
#include <vector>

#include "cuna_launch.hpp"

namespace cuna {

// Device blocks kept between plans.  A plan made for one call (a training step,
// a survey of new curves, the host interface) allocates and frees the same large
// blocks each time, and hipFree of a large block takes 70 - 260 us, hipMalloc 20 -
// 60 us.  A freed block of kMinBlock bytes or more is kept for the next
// allocation of its size class on its device instead.  As hipFree does, a release
// waits for the device first, so a kept block has no work outstanding on any
// stream and may go to any other.  At most kMaxKept bytes are kept (the oldest
// block leaves first); all go back on cuna_batch_cache_clear(), and before an
// allocation that would otherwise fail.
struct BlockPool {
    static constexpr size_t kMinBlock = size_t(64) << 10, kMaxBlock = size_t(256) << 20;
    static constexpr size_t kMaxKept = size_t(512) << 20;
    // a block of at least nbytes on the current device (its size in *got).  Like
    // hipMalloc, refused while `s` is being captured.
    static void *take(size_t nbytes, size_t *got, int *dev, hipStream_t s);
    static void give(void *p, size_t bytes, int dev);
    static void clear();
};

// true while `s` is being captured into a graph (the null stream never is)
inline bool capturing(hipStream_t s) {
    if (!s) return false;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    CUNA_HIP(hipStreamIsCapturing(s, &st));
    return st != hipStreamCaptureStatusNone;
}

// Persistent device allocation.
struct DevMem {
    void *ptr = nullptr;
    size_t bytes = 0;
    int dev = 0;
    bool owned = true;  // false: a view into another allocation
    // a captured call used this memory: its graph holds the address, so a block
    // that ensure() outgrows stays this object's own until release()
    bool in_graph = false;
    struct Outgrown {
        void *p;
        size_t bytes;
        int dev;
    };
    std::vector<Outgrown> outgrown;
    DevMem() = default;
    DevMem(const DevMem &) = delete;
    DevMem &operator=(const DevMem &) = delete;
    // s: the stream of the call that allocates (only checked for capture)
    void alloc(size_t nbytes, hipStream_t s) {
        release();
        if (nbytes) ptr = BlockPool::take(nbytes, &bytes, &dev, s);
    }
    void view(void *p, size_t nbytes) {
        release();
        ptr = p;
        bytes = nbytes;
        owned = false;
    }
    // at least nbytes, for a call on s (its contents are not kept).  A captured
    // call that is refused memory leaves what there was.
    void ensure(size_t nbytes, hipStream_t s) {
        const bool now = capturing(s);
        if (nbytes > bytes) {
            if (!now && !in_graph) {
                drop();
                ptr = BlockPool::take(nbytes, &bytes, &dev, s);
            } else {
                size_t got = 0;
                int d = 0;
                void *p = BlockPool::take(nbytes, &got, &d, s);
                if (ptr) outgrown.push_back(Outgrown{ptr, bytes, dev});
                ptr = p;
                bytes = got;
                dev = d;
                in_graph = false;
            }
        }
        in_graph = in_graph || now;
    }
    // a call on s reads or writes this memory as it is
    void use(hipStream_t s) { in_graph = in_graph || capturing(s); }
    // gives up the current memory, not what graphs hold of earlier memory
    void drop() {
        if (ptr && owned) BlockPool::give(ptr, bytes, dev);
        ptr = nullptr;
        bytes = 0;
        owned = true;
    }
    void release() {
        drop();
        for (const Outgrown &o : outgrown) BlockPool::give(o.p, o.bytes, o.dev);
        outgrown.clear();
        in_graph = false;
    }
    ~DevMem() { release(); }
    template <typename U>
    U *as() const {
        return static_cast<U *>(ptr);
    }
};

// Points of one or more curves binned by grid tile (stable counting sort).
template <typename T>
struct TiledPoints {
    // host sources of the async uploads (offsets and curve order; the sort's
    // chunk tables), declared first so that they are destroyed after the
    // device buffers (whose release synchronises)
    std::vector<int> plan_h, sort_h;
    int ncurves = 0;
    long n = 0;
    std::vector<int> coff_h;
    int longest = 0;  // points of the longest curve
    int G = 0, tlog = 0, ntiles = 0, Kc = 0, olo = 0, ntaps = 0;
    bool periodic = true;
    // two allocations; the buffers below are views into them
    DevMem arena, tile_arena;
    DevMem coff, eps_orig;
    DevMem rec_orig;  // (anchor, e) by original index
    DevMem order;     // curves by decreasing length (work-queue order)
    // the points sorted by tile, for the paths that work by tiles (see tiles())
    bool tiled = false;
    DevMem rec, perm, bucket;
    DevMem tile_desc;   // per curve: the scatter's work order (TileDesc per tile)

    // src: setup arguments with x/t/mode/compat fields filled.  lazy: the points
    // are sorted when a call first needs them (the fused kernels of small grids
    // take them in their original order)
    void build(SetupArgs<T> A, const std::vector<int> &offsets, int G_, int tlog_, int ntaps_,
               bool periodic_, bool keep_eps, bool lazy, hipStream_t s);
    // sorted points, buckets and work order, made on the first call
    void tiles(hipStream_t s);

  private:
    void sort_points(hipStream_t s);
};

struct ModeSpec {
    int mode = 0;  // CUNA_MODE_*
    int sigma = 2, m = 8, tile_log2 = 0, flags = 0;
    int fft_w = 0, fft_h = 0;  // FFT workgroup shape (0: heuristic)
};

// Bluestein (chirp-z) transform of length ng, for grids whose length is not
// a power of two >= 4 (the reference hands any ng to cuFFT,
// src/cuna_kernel.cu:82,169,208,261):
//   A[r] = sum_g z_g e^{+2 pi i g r/n} = c_r sum_g (z_g c_g) conj(c_{r-g}),
//   c_k = exp(+i pi k^2/n),
// a circular convolution of length L = 2^lgL >= 2 n - 1 done with the
// power-of-two FFT: conv = FFT_+(FFT_-(z c) * FFT_-(b)) / L, with
// b_k = b_{L-k} = conj(c_k) for 0 <= k < n and zero between.
template <typename T>
struct LoadChirp;
template <typename T>
struct ChirpSink;

template <typename T>
struct Bluestein {
    // host source of the (async) upload, declared first so that it is destroyed
    // after the device buffers (whose release synchronises)
    std::vector<cplx<T>> tab_h;
    int ng = 0, n = 0, lgL = 0;  // n: complex values transformed
    bool pairs = false;          // an even real grid: n = ng/2 pairs of cells
    long L = 0;
    DevMem tab;   // c_k, k < n, then (pairs) exp(2 pi i r/ng), r <= n/2
    DevMem bt;    // FFT_-(b) / L, in the order of the passes
    DevMem bt_rows;  // both_forms(): bt in the order of the three passes
    DevMem work;  // batch x L complex, batch as large as ensure() asked for
    // real: run_real will be called (else run_complex)
    void init(int length, bool real, hipStream_t s);
    void ensure(int batch, hipStream_t s);
    // real grids (batch rows of stride gstride, the first ng cells used) ->
    // the compat deconvolution sink, one row per grid (rows: see FftShape)
    void run_real(const T *grid, long gstride, int batch, int rows, const SinkCompat<T> &sk,
                  hipStream_t s);
    // in place on batch x ng complex values: data[r] = sum_g data[g] e^{sign 2 pi i g r/ng}
    void run_complex(cplx<T> *data, int batch, int sign, hipStream_t s);

  private:
    const cplx<T> *chirp() const { return tab.template as<cplx<T>>(); }
    bool both_forms() const;
    void run(const LoadChirp<T> &ld, const ChirpSink<T> &sink, int batch, int rows,
             hipStream_t s);
};

// true when a real grid of G cells takes the power-of-two FFT (else Bluestein)
inline bool pow2_grid(long G) { return G >= 4 && is_pow2(G); }

template <typename T>
struct Plan {
    ModeSpec spec;
    int M = 0;  // accurate: modes per curve; compat: ng
    int G = 0, lgN = 0, ntaps = 0, olo = 0;
    T beta = 0, wscale = 1;
    T e3[kMaxTaps] = {};
    // compat constants (src/gaussian_filter.cu:54-57)
    T b_c = 0, normfac_c = 0;
    int R_f = 0;
    // compat plans over several curves with their own b (device arrays, set
    // by the batched transform): per curve (1/b, 1/sqrt(pi b), exp(-1/b)),
    // b/4, and the output offset of the curve's spectrum
    const T *cpar_c = nullptr;
    const T *qb_row_c = nullptr;
    const long *row_off_c = nullptr;
    // kept to identify the x a registered plan belongs to
    const void *x_key = nullptr;
    TiledPoints<T> pts, pts2;  // pts2: points 2x (window at 2f)
    bool has_pts2 = false;
    DevMem grid, work, counts, counter;
    std::unique_ptr<Bluestein<T>> blu;  // compat grids of any other length
    // fused bootstrap: queue entries (BootCurve) and densest tap window of x and 2x
    DevMem boot_curves, cover;
    DevMem boot_list;  // draws of the resident workgroups
    DevMem ls_work;  // Lomb-Scargle: window spectra of the resident workgroups
    bool cover_ready = false;
    // optional profiling events, recorded on the execution stream before the
    // first kernel of adjoint() and after each of its kernels
    hipEvent_t prof[4] = {nullptr, nullptr, nullptr, nullptr};

    long n() const { return pts.n; }
    int ncurves() const { return pts.ncurves; }

    // y -> out (ncurves x M complex)
    void adjoint(const T *y, cplx<T> *out, hipStream_t s);
    // the same with the real grid (ncurves x G) in caller-provided memory;
    // allocates nothing
    void adjoint_into(const T *y, cplx<T> *out, T *grid_ptr, hipStream_t s) const;
    // nrhs value vectors (rows of n) -> out (ncurves x nrhs x M), one spread
    // launch and one batched FFT
    void adjoint_many(const T *y, int nrhs, cplx<T> *out, hipStream_t s);
    // compat bootstrap of src/cuna_kernel.cu:236-289 (single curve)
    void bootstrap_compat(const T *y, cplx<T> *out, int nbs, uint32_t seed, hipStream_t s);
    // accurate bootstrap (resampled points)
    void bootstrap(const T *y, int nbs, uint32_t seed, cplx<T> *out_y, cplx<T> *out_w,
                   hipStream_t s);
    // Lomb-Scargle power of each replicate (fused kernel sizes only)
    void bootstrap_ls(const T *y, int nbs, uint32_t seed, T *power, T *peak, int *kpeak,
                      hipStream_t s);
    void backward(const T *y, const cplx<T> *g, T *dy, T *dx, hipStream_t s);
    // forward (type-2) NFFT: fhat (ncurves x M) -> f (n complex)
    void forward(const cplx<T> *fhat, cplx<T> *f, hipStream_t s);
    // allocate every workspace a later call with these sizes needs (so that
    // the call can be captured into a graph without allocating)
    void prepare_bootstrap(int nbs, bool window, hipStream_t s);
    bool bootstrap_fused_ok(bool window) const;
    int boot_list_cap() const;

    bool fused_adjoint = false;  // adjoint() and adjoint_many() by launch_adjoint_fused
    void adjoint_fused(const T *y, int nrhs, cplx<T> *out, hipStream_t s);
    // per-curve cover of x (and 2x) for the fused kernels, once per plan
    const int *covers(hipStream_t s);
    SpreadArgs<T> spread_args(const TiledPoints<T> &P) const;
    GatherArgs<T> gather_args() const;
    SinkAccurate<T> accurate_sink(cplx<T> *out) const;
    void spectrum_to_grid(const cplx<T> *g, int parts, int rot, hipStream_t s);
    bool room_for_both_parts(hipStream_t s);
    BootArgs<T> fused_args(const T *y, int nbs, uint32_t seed, hipStream_t s);
    // rows: see FftShape
    void run_fft(T *grid_ptr, cplx<T> *out, int batch, int rows, hipStream_t s,
                 hipEvent_t mid = nullptr) const;
    // twiddle tables (and the Bluestein set-up for other lengths) for this
    // plan's transform; run once at plan creation
    void prepare_fft(hipStream_t s);
};

template <typename T>
std::unique_ptr<Plan<T>> make_plan_accurate(const T *x, const double *t, double df,
                                            const std::vector<int> &offsets, int M,
                                            const ModeSpec &spec, hipStream_t s);
template <typename T>
std::unique_ptr<Plan<T>> make_plan_compat(const T *x, int n, int ng, T *E1, T *E2, T *E3,
                                          const ModeSpec &spec, hipStream_t s);
// b and normfac of the compat filter in the build's precision
template <typename T>
void compat_constants(int n, int ng, T &b, T &normfac, int &R_f);

}  // namespace cuna
