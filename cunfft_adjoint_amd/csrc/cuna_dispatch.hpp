// cuna_dispatch.hpp -- host helpers of the kernel launchers: LDS limits, FFT
// workgroup shapes and compile-time dispatch on transform sizes.
#pragma once

#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <type_traits>

#include "cuna_launch.hpp"

namespace cuna {

// raise the dynamic LDS limit of a kernel once per device (not on every
// launch, so that launches can be captured into a graph).  The record is a
// fixed table: the lookup never allocates host memory (a full table only
// means the attribute is set again on each launch).
template <typename K>
static void set_lds(K kernel, size_t bytes) {
    if (bytes <= 64 * 1024) return;
    struct Entry {
        const void *key;
        int dev;
        size_t bytes;
    };
    constexpr int kEntries = 512;
    static std::mutex mu;
    static Entry done[kEntries];
    static int used = 0;
    const void *key = reinterpret_cast<const void *>(kernel);
    int dev = 0;
    CUNA_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    Entry *e = nullptr;
    for (int i = 0; i < used && !e; ++i)
        if (done[i].key == key && done[i].dev == dev) e = &done[i];
    if (e && e->bytes >= bytes) return;
    CUNA_HIP(hipFuncSetAttribute(key, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    if (!e && used < kEntries) e = &done[used++];
    if (e) *e = Entry{key, dev, bytes};
}

static constexpr int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// ----------------------------------------------------------- FFT config --
// threads per workgroup for W sequences of length 2^LG, 2^mr values per thread
constexpr int fft_threads(int lg, int w, int mr = 4) {
    return clampi(((1 << lg) * w) >> mr, 64, 1024);
}

// threads of the fused kernels: as the FFT takes them, at least 256 for the spread
constexpr int fused_threads(int lg) {
    return fft_threads(lg, 1, small_mr(lg)) < 256 ? 256 : fft_threads(lg, 1, small_mr(lg));
}
// two-pass split N = L1 * L2, L2 >= L1
constexpr int split_lg1(int lgN) { return lgN / 2; }
// largest log2 N of the single-workgroup inverse (Hermitian) transform
constexpr int kC2rSmallLg = 13;

// Sequences per workgroup of a pass: the largest count whose LDS tile fits in
// 64 KB that still gives >= min_wg workgroups; an environment override
// (CUNA_FFT_W, CUNA_FFT_H) exists for tuning runs.  Measured at N = 2^20
// (1024 x 1024): the column pass is fastest at one 256-thread workgroup per
// CU (W = 4), the row pass with mirror pairs at two or more per CU (H = 1).
template <typename T, int LG, int W>
constexpr bool lds_fits() {
    return (long)W * (1L << LG) * (long)sizeof(cplx<T>) <= 65536;
}

static int env_int(const char *name) {
    const char *v = getenv(name);
    return v ? atoi(v) : 0;
}

// compute units of the current device (cached per device, fixed table)
static int num_cus() {
    constexpr int kDevices = 64;
    static std::mutex mu;
    static int cache[kDevices] = {};
    int dev = 0;
    CUNA_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    if (dev >= 0 && dev < kDevices && cache[dev] > 0) return cache[dev];
    int n = 0;
    CUNA_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
    n = std::max(n, 1);
    if (dev >= 0 && dev < kDevices) cache[dev] = n;
    return n;
}

template <typename T>
static int pick_seq(int lg, long nseq, int batch, int per_wg_mult, const char *env,
                    int requested = 0, long min_wg = 512) {
    int forced = requested ? requested : env_int(env);
    auto valid = [&](int w) {
        long lds = (long)w * per_wg_mult * (1L << lg) * (long)sizeof(cplx<T>);
        return w >= 1 && w <= 8 && (w & (w - 1)) == 0 && lds <= 65536 &&
               nseq % (w * per_wg_mult) == 0;
    };
    if (forced && valid(forced)) return forced;
    int best = 1;
    for (int w = 8; w >= 1; w >>= 1) {
        if (!valid(w)) continue;
        if ((nseq / (w * per_wg_mult)) * (long)batch >= min_wg) return w;
        best = std::min(best, w);
    }
    return best;
}

template <typename T, int LG, class F>
static void dispatch_w(int w, F &&f) {
    if constexpr (lds_fits<T, LG, 8>())
        if (w == 8) return f(std::integral_constant<int, 8>{});
    if constexpr (lds_fits<T, LG, 4>())
        if (w == 4) return f(std::integral_constant<int, 4>{});
    if constexpr (lds_fits<T, LG, 2>())
        if (w == 2) return f(std::integral_constant<int, 2>{});
    if (w == 1) return f(std::integral_constant<int, 1>{});
    fail(CUNA_ERROR_UNSUPPORTED, "fft workgroup shape");
}

// dispatch for the row pass with mirror pairs (2H sequences per workgroup)
template <typename T, int LG, class F>
static void dispatch_h(int h, F &&f) {
    if constexpr (lds_fits<T, LG, 8>())
        if (h == 4) return f(std::integral_constant<int, 4>{});
    if constexpr (lds_fits<T, LG, 4>())
        if (h == 2) return f(std::integral_constant<int, 2>{});
    if constexpr (lds_fits<T, LG, 2>())
        if (h == 1) return f(std::integral_constant<int, 1>{});
    fail(CUNA_ERROR_UNSUPPORTED, "fft workgroup shape");
}

// compile-time dispatch on a runtime log2 size
template <int LO, int HI, class F>
static void dispatch_lg(int lg, F &&f) {
    if constexpr (LO <= HI) {
        if (lg == LO) {
            f(std::integral_constant<int, LO>{});
            return;
        }
        dispatch_lg<LO + 1, HI>(lg, std::forward<F>(f));
    } else {
        fail(CUNA_ERROR_UNSUPPORTED, "transform size out of range");
    }
}

}  // namespace cuna
