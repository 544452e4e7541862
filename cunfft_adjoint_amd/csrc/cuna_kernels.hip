// cuna_kernels.hip -- instantiation and launch of the FFT and spread kernels
// for the library's real type (float in libcunaf.so, double in libcunad.so).
#include <hip/hip_ext.h>

#include <algorithm>
#include <cstdlib>

#include "cuna_dispatch.hpp"
#include "cuna_launch.hpp"

namespace cuna {

template <typename T, int S, int LG, class Loader, class Sink, int MODE>
static void run_small(const FftShape &sh, const Loader &ld, const Sink &sk, cplx<T> *plain_out,
                      hipStream_t s) {
    constexpr int MR = small_mr(LG), NT = fft_threads(LG, 1, MR);
    auto &tc = TwiddleCache<T>::get();
    constexpr int CAP = small_cap(LG);
    const cplx<T> *tw = LG > CAP ? tc.fine(LG) : nullptr;
    const cplx<T> *tw_lds = tc.rows(LG, MR, CAP);
    Tw2<T> twG = tc.two_level(LG + 1);
    constexpr size_t lds = sizeof(cplx<T>) * (((size_t)1 << LG) + rows_count(LG, MR, CAP));
    static_assert(lds <= kMaxLds, "FFT LDS");
    auto k = k_fft_small<T, S, LG, NT, Loader, Sink, MODE, MR>;
    set_lds(k, lds);
    hipLaunchKernelGGL(k, dim3(sh.batch), dim3(NT), lds, s, ld, sk, plain_out, tw, tw_lds, twG);
    CUNA_LAUNCH_CHECK();
}

template <typename T, int S, int LG2, int W, class Loader>
static void run_col(const FftShape &sh, const Loader &ld, cplx<T> *dst, int L1, hipStream_t s) {
    constexpr int NT = fft_threads(LG2, W, kColMr);
    auto &tc = TwiddleCache<T>::get();
    const long N = 1L << sh.lgN;
    const size_t lds = sizeof(cplx<T>) * (((size_t)W << LG2) + rows_count(LG2, kColMr, LG2));
    auto k = k_fft_col<T, S, LG2, W, NT, Loader, kColMr>;
    set_lds(k, lds);
    require(L1 % W == 0, "fft column split");
    for (long b0 = 0; b0 < sh.batch; b0 += kMaxGridY) {
        const int nb = (int)std::min<long>(kMaxGridY, sh.batch - b0);
        hipLaunchKernelGGL(k, dim3(L1 / W, nb), dim3(NT), lds, s, ld, dst, N, L1,
                           tc.rows(LG2, kColMr, LG2), tc.two_level(sh.lgN), b0);
        CUNA_LAUNCH_CHECK();
    }
}

template <typename T, int LG1, int H, class Sink>
static void run_row_real(const FftShape &sh, const cplx<T> *src, int L2, const Sink &sk,
                         hipStream_t s) {
    constexpr int NT = fft_threads(LG1, 2 * H, kRowMr);
    auto &tc = TwiddleCache<T>::get();
    const long N = 1L << sh.lgN;
    const size_t lds =
        sizeof(cplx<T>) * (((size_t)(2 * H) << LG1) + rows_count(LG1, kRowMr, LG1));
    auto k = k_fft_row_real<T, LG1, H, NT, Sink, kRowMr>;
    set_lds(k, lds);
    require(L2 % (2 * H) == 0, "fft row split");
    for (long b0 = 0; b0 < sh.batch; b0 += kMaxGridY) {
        const int nb = (int)std::min<long>(kMaxGridY, sh.batch - b0);
        hipLaunchKernelGGL(k, dim3(L2 / (2 * H), nb), dim3(NT), lds, s, src, N, L2, sk,
                           tc.rows(LG1, kRowMr, LG1), tc.two_level(sh.lgN + 1), b0);
        CUNA_LAUNCH_CHECK();
    }
}

template <typename T, int S, int LG1, int H>
static void run_row_plain(const FftShape &sh, const cplx<T> *src, int L2, cplx<T> *dst,
                          hipStream_t s) {
    constexpr int NT = fft_threads(LG1, H, kRowMr);
    auto &tc = TwiddleCache<T>::get();
    const long N = 1L << sh.lgN;
    const size_t lds = sizeof(cplx<T>) * (((size_t)H << LG1) + rows_count(LG1, kRowMr, LG1));
    auto k = k_fft_row_plain<T, S, LG1, H, NT, kRowMr>;
    set_lds(k, lds);
    require(L2 % H == 0, "fft row split");
    for (long b0 = 0; b0 < sh.batch; b0 += kMaxGridY) {
        const int nb = (int)std::min<long>(kMaxGridY, sh.batch - b0);
        hipLaunchKernelGGL(k, dim3(L2 / H, nb), dim3(NT), lds, s, src, N, L2, dst, N,
                           tc.rows(LG1, kRowMr, LG1), b0);
        CUNA_LAUNCH_CHECK();
    }
}

// Whether the largest transform that one workgroup holds goes through two passes
// all the same: for few rows, which leave the chip idle at one workgroup per row and
// take the whole transform's LDS passes in a row.  sh.rows decides, not the batch,
// and the passes have one shape (kFewW, kFewH), because calls that are promised to
// agree bit for bit differ in their batches.  Measured with the spread, values of one
// plan, one workgroup per row / two passes: FP32, 2^14, 20,000 points: 1 row 22.4 /
// 12.3 us, 64 rows 31.4 / 27.5, 100 rows 38.0 / 37.4, 128 rows 42.7 / 43.9, 256 rows
// 62 / 75; FP64, 2^13, 8000 points: 1 row 19.8 / 14.8, 32 rows 23.2 / 19.6, 64 rows
// 28.4 / 27.1, 100 rows 34.4 / 36.8.  Other shapes: 12.2 us at one row and 95 at 256
// with one sequence per workgroup, 14.3 and 70 with eight and four.
constexpr int kFewW = 8, kFewH = 1;
template <typename T>
static bool few_rows(const FftShape &sh) {
    const int rows = sh.rows > 0 ? sh.rows : sh.batch;
    return sh.lgN == max_small_lg<T>() &&
           rows <= (sizeof(T) == 4 ? num_cus() * 3 / 8 : num_cus() * 3 / 16);
}

template <typename T, class Sink>
static void real_forward_impl(const FftShape &sh, T *grid, const Sink &sk, hipStream_t s,
                              hipEvent_t mid) {
    require(sh.lgN >= 1 && sh.lgN <= max_fft_lg<T>(), "grid size out of range",
            CUNA_ERROR_UNSUPPORTED);
    LoadGrid<T> ld;
    ld.z = reinterpret_cast<const cplx<T> *>(grid);
    ld.stride = 1L << sh.lgN;
    const bool few = few_rows<T>(sh);
    if (sh.lgN <= max_small_lg<T>() && !few) {
        dispatch_lg<1, max_small_lg<T>()>(sh.lgN, [&](auto c) {
            run_small<T, 1, decltype(c)::value, LoadGrid<T>, Sink, 0>(sh, ld, sk, nullptr, s);
        });
        return;
    }
    const int lg1 = split_lg1(sh.lgN), lg2 = sh.lgN - lg1;
    cplx<T> *z = reinterpret_cast<cplx<T> *>(grid);
    const int W = pick_seq<T>(lg2, 1L << lg1, sh.batch, 1, "CUNA_FFT_W",
                              few && !sh.w ? kFewW : sh.w, num_cus());
    const int H = std::min(4, pick_seq<T>(lg1, 1L << lg2, sh.batch, 2, "CUNA_FFT_H",
                                          few && !sh.h ? kFewH : sh.h));
    dispatch_lg<7, 12>(lg2, [&](auto c) {
        constexpr int LG2 = decltype(c)::value;
        dispatch_w<T, LG2>(W, [&](auto w) {
            run_col<T, 1, LG2, decltype(w)::value, LoadGrid<T>>(sh, ld, z, 1 << lg1, s);
        });
    });
    if (mid) CUNA_HIP(hipEventRecord(mid, s));
    dispatch_lg<6, 12>(lg1, [&](auto c) {
        constexpr int LG1 = decltype(c)::value;
        dispatch_h<T, LG1>(H, [&](auto h) {
            run_row_real<T, LG1, decltype(h)::value, Sink>(sh, z, 1 << lg2, sk, s);
        });
    });
}

template <typename T>
void fft_real_forward(const FftShape &sh, T *grid, const SinkAccurate<T> &sk, hipStream_t s,
                      hipEvent_t mid) {
    real_forward_impl<T, SinkAccurate<T>>(sh, grid, sk, s, mid);
}
template <typename T>
void fft_real_forward(const FftShape &sh, T *grid, const SinkCompat<T> &sk, hipStream_t s,
                      hipEvent_t mid) {
    real_forward_impl<T, SinkCompat<T>>(sh, grid, sk, s, mid);
}

template <typename T>
void fft_c2r_inverse(const FftShape &sh, const LoadHermitian<T> &ld, cplx<T> *work, T *grid,
                     hipStream_t s) {
    require(sh.lgN >= 1 && sh.lgN <= max_fft_lg<T>(), "grid size out of range",
            CUNA_ERROR_UNSUPPORTED);
    cplx<T> *z = reinterpret_cast<cplx<T> *>(grid);
    SinkAccurate<T> dummy{};
    // the Hermitian loader is register-heavy: a 1024-thread workgroup (N =
    // 2^14) would spill, so N >= 2^14 takes the two-pass path in both
    // libraries; FP64 at 2^13 does so for few rows, as the forward transform (18.4 ->
    // 15.4 us with the gather, one curve)
    const bool few = sh.lgN == max_small_lg<T>() && sh.batch <= num_cus() / 8;
    if (sh.lgN <= kC2rSmallLg && !few) {
        dispatch_lg<1, kC2rSmallLg>(sh.lgN, [&](auto c) {
            run_small<T, -1, decltype(c)::value, LoadHermitian<T>, SinkAccurate<T>, 1>(
                sh, ld, dummy, z, s);
        });
        return;
    }
    const int lg1 = split_lg1(sh.lgN), lg2 = sh.lgN - lg1;
    const int W = pick_seq<T>(lg2, 1L << lg1, sh.batch, 1, "CUNA_FFT_W", sh.w, num_cus());
    const int H = pick_seq<T>(lg1, 1L << lg2, sh.batch, 1, "CUNA_FFT_H", sh.h, num_cus());
    dispatch_lg<7, 12>(lg2, [&](auto c) {
        constexpr int LG2 = decltype(c)::value;
        dispatch_w<T, LG2>(W, [&](auto w) {
            run_col<T, -1, LG2, decltype(w)::value, LoadHermitian<T>>(sh, ld, work, 1 << lg1, s);
        });
    });
    dispatch_lg<6, 12>(lg1, [&](auto c) {
        constexpr int LG1 = decltype(c)::value;
        dispatch_w<T, LG1>(H, [&](auto h) {
            run_row_plain<T, -1, LG1, decltype(h)::value>(sh, work, 1 << lg2, z, s);
        });
    });
}

template <typename T>
void fft_complex(const FftShape &sh, cplx<T> *data, cplx<T> *work, int sign, hipStream_t s) {
    require(sh.lgN >= 1 && sh.lgN <= max_fft_lg<T>(), "transform size out of range",
            CUNA_ERROR_UNSUPPORTED);
    require(sign == 1 || sign == -1, "sign must be +1 or -1");
    LoadGrid<T> ld;
    ld.z = data;
    ld.stride = 1L << sh.lgN;
    SinkAccurate<T> dummy{};
    if (sh.lgN <= max_small_lg<T>()) {
        dispatch_lg<1, max_small_lg<T>()>(sh.lgN, [&](auto c) {
            if (sign > 0)
                run_small<T, 1, decltype(c)::value, LoadGrid<T>, SinkAccurate<T>, 1>(sh, ld, dummy,
                                                                                     data, s);
            else
                run_small<T, -1, decltype(c)::value, LoadGrid<T>, SinkAccurate<T>, 1>(
                    sh, ld, dummy, data, s);
        });
        return;
    }
    const int lg1 = split_lg1(sh.lgN), lg2 = sh.lgN - lg1;
    const int W = pick_seq<T>(lg2, 1L << lg1, sh.batch, 1, "CUNA_FFT_W", sh.w, num_cus());
    const int H = pick_seq<T>(lg1, 1L << lg2, sh.batch, 1, "CUNA_FFT_H", sh.h, num_cus());
    dispatch_lg<7, 12>(lg2, [&](auto c) {
        constexpr int LG2 = decltype(c)::value;
        dispatch_w<T, LG2>(W, [&](auto w) {
            constexpr int WW = decltype(w)::value;
            if (sign > 0)
                run_col<T, 1, LG2, WW, LoadGrid<T>>(sh, ld, work, 1 << lg1, s);
            else
                run_col<T, -1, LG2, WW, LoadGrid<T>>(sh, ld, work, 1 << lg1, s);
        });
    });
    dispatch_lg<7, 12>(lg1, [&](auto c) {
        constexpr int LG1 = decltype(c)::value;
        dispatch_w<T, LG1>(H, [&](auto h) {
            constexpr int HH = decltype(h)::value;
            if (sign > 0)
                run_row_plain<T, 1, LG1, HH>(sh, work, 1 << lg2, data, s);
            else
                run_row_plain<T, -1, LG1, HH>(sh, work, 1 << lg2, data, s);
        });
    });
}

// ----------------------------------------------------------------- sort --
template <typename T>
void launch_point_setup(const SetupArgs<T> &A, hipStream_t s) {
    const long n = std::max(A.n, (long)A.R_f);
    if (n <= 0) return;
    hipLaunchKernelGGL(k_point_setup<T>, dim3(ceil_div(n, 256)), dim3(256), 0, s, A);
    CUNA_LAUNCH_CHECK();
}

template <typename T>
void launch_sort_pass(const SortWork &W, int shift, int bits, const PointRec<T> *rec_in,
                      const int *perm_in, PointRec<T> *rec_out, int *perm_out, hipStream_t s) {
    if (W.nchunks == 0) return;
    require(bits >= 1 && bits <= kSortBits, "sort digit too wide");
    SortArgs S;
    S.chunks = W.chunks;
    S.chunk_base = W.chunk_base;
    S.nch = W.nch;
    S.nchunks = W.nchunks;
    S.K = 1 << bits;
    S.shift = shift;
    S.hist = W.hist;
    constexpr int wpb = 4;  // waves per block
    const size_t lds = sizeof(int) * (size_t)wpb * S.K;
    const int nblk = (int)ceil_div(W.nchunks, wpb);
    hipLaunchKernelGGL(k_hist<T>, dim3(nblk), dim3(64 * wpb), lds, s, S, rec_in);
    CUNA_LAUNCH_CHECK();
    // exclusive scan of the key-major count matrix
    const long n = (long)S.K * W.total_chunks;
    const long nb = ceil_div(std::max(n, 1L), kScanTile);
    size_t slds = sizeof(int) * kScanNT;
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(kScanNT), slds, s, W.hist, n, W.bsum);
    CUNA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(kScanNT), slds, s, W.hist, n, W.bsum, W.hist);
    CUNA_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_scatter<T>, dim3(nblk), dim3(64 * wpb), lds, s, S, rec_in, perm_in,
                       rec_out, perm_out);
    CUNA_LAUNCH_CHECK();
}

template <typename T>
void launch_buckets(const int *coff, int ncurves, int Kc, const PointRec<T> *rec, int tlog,
                    int olo, int ohi, int G, int *bucket, hipStream_t s) {
    const long nbk = (long)ncurves * (Kc + 1);
    if (nbk <= 0) return;
    hipLaunchKernelGGL(k_buckets<T>, dim3(ceil_div(nbk, 256)), dim3(256), 0, s, coff, ncurves, Kc,
                       rec, tlog, olo, ohi, G, bucket);
    CUNA_LAUNCH_CHECK();
}

// --------------------------------------------------------------- spread --
// with ev0/ev1 set, the kernel's own start and stop times are recorded in
// them (as its dispatch begins and ends, without separate event packets)
template <typename K, typename T>
static void launch_timed(K k, dim3 grid, dim3 block, size_t lds, hipStream_t s, hipEvent_t ev0,
                         hipEvent_t ev1, const SpreadArgs<T> &A) {
    if (ev0 || ev1)
        hipExtLaunchKernelGGL(k, grid, block, (uint32_t)lds, s, ev0, ev1, 0, A);
    else
        hipLaunchKernelGGL(k, grid, block, lds, s, A);
    CUNA_LAUNCH_CHECK();
}

// grid (ntiles, slabs) in launches of at most kMaxGridY slabs; ev0 records
// the first launch's start, ev1 the last one's stop
template <typename K, typename T>
static void launch_slabs(K k, const SpreadArgs<T> &A, int nslabs, dim3 block, size_t lds,
                         hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    for (int s0 = 0; s0 < nslabs; s0 += kMaxGridY) {
        const int ns = std::min(kMaxGridY, nslabs - s0);
        SpreadArgs<T> B = A;
        B.slab0 = s0;
        launch_timed(k, dim3(A.ntiles, ns), block, lds, s, s0 == 0 ? ev0 : nullptr,
                     s0 + ns == nslabs ? ev1 : nullptr, B);
    }
}

// The scatter form (default): one wave per tile, fixed-point cells per wave
// (32-bit in FP32, 64-bit in FP64), nothing measured at plan time needed to be
// safe.  CUNA_PLAN_GATHER selects the gather form.
template <typename T, int NTAPS, int VM>
static void spread_one(const SpreadArgs<T> &A, int nslabs, hipStream_t s, hipEvent_t ev0,
                       hipEvent_t ev1) {
    if (!A.gather) {
        constexpr int WPT = 1;
        const size_t lds = spread_wv_lds_bytes<T>(A.tlog, NTAPS, WPT);
        require(lds <= kMaxLds, "spread tile too large", CUNA_ERROR_UNSUPPORTED);
        auto k = k_spread_wv<T, NTAPS, VM, WPT>;
        set_lds(k, lds);
        launch_slabs(k, A, nslabs, dim3(64 * WPT), lds, s, ev0, ev1);
        return;
    }
    const size_t lds = spread_lds_bytes<T>(A.tlog, NTAPS, A.cap);
    require(lds <= kMaxLds, "spread tile too large", CUNA_ERROR_UNSUPPORTED);
    auto k = k_spread<T, NTAPS, VM>;
    set_lds(k, lds);
    launch_slabs(k, A, nslabs, dim3(256), lds, s, ev0, ev1);
}

// accurate filters have 2m taps, m in [2, kMaxTaps/2]; compat filters have
// 2 R_f - 1 = 11 (float build) or 23 (double build) taps
template <int LO, int HI, class F>
static void dispatch_m(int m, F &&f) {
    if constexpr (LO <= HI) {
        if (m == LO) {
            f(std::integral_constant<int, 2 * LO>{});
            return;
        }
        dispatch_m<LO + 1, HI>(m, std::forward<F>(f));
    } else {
        fail(CUNA_ERROR_UNSUPPORTED, "unsupported filter width");
    }
}

template <typename T>
void launch_spread(const SpreadArgs<T> &A, int ntaps, int vm, int nslabs, hipStream_t s,
                   hipEvent_t ev0, hipEvent_t ev1) {
    if (ntaps == 11 || ntaps == 23) {
        require(vm != VAL_COUNTS, "counts spread needs an accurate filter");
        if (ntaps == 11) {
            if (vm == VAL_PLAIN)
                spread_one<T, 11, VAL_PLAIN>(A, nslabs, s, ev0, ev1);
            else
                spread_one<T, 11, VAL_COMPAT_BOOT>(A, nslabs, s, ev0, ev1);
        } else {
            if (vm == VAL_PLAIN)
                spread_one<T, 23, VAL_PLAIN>(A, nslabs, s, ev0, ev1);
            else
                spread_one<T, 23, VAL_COMPAT_BOOT>(A, nslabs, s, ev0, ev1);
        }
        return;
    }
    require(ntaps % 2 == 0 && vm != VAL_COMPAT_BOOT, "unsupported filter width",
            CUNA_ERROR_UNSUPPORTED);
    dispatch_m<2, kMaxTaps / 2>(ntaps / 2, [&](auto c) {
        constexpr int NTP = decltype(c)::value;
        if (vm == VAL_PLAIN)
            spread_one<T, NTP, VAL_PLAIN>(A, nslabs, s, ev0, ev1);
        else
            spread_one<T, NTP, VAL_COUNTS>(A, nslabs, s, ev0, ev1);
    });
}

template <typename T>
void launch_tile_order(const SpreadArgs<T> &A, int ncurves, TileDesc *desc, hipStream_t s) {
    if (ncurves <= 0 || A.ntiles <= 0) return;
    require(A.ntiles <= kOrderMaxTiles, "too many spread tiles for the work order",
            CUNA_ERROR_UNSUPPORTED);
    hipLaunchKernelGGL(k_tile_order, dim3(ncurves), dim3(kOrderThreads), 0, s, A.bucket, A.Kc,
                       A.ntiles, desc);
    CUNA_LAUNCH_CHECK();
    const size_t lds = sizeof(int) * kDescWaves * (((size_t)1 << A.tlog) + 2 * (size_t)A.ntaps + 1);
    require(lds <= kMaxLds, "spread tile too large", CUNA_ERROR_UNSUPPORTED);
    set_lds(k_tile_desc<T>, lds);
    // a launch holds fewer than 2^32 threads
    const long npos = (long)ncurves * A.ntiles, most = 1L << 25;
    for (long p0 = 0; p0 < npos; p0 += most) {
        const long p1 = std::min(npos, p0 + most);
        hipLaunchKernelGGL(k_tile_desc<T>, dim3(ceil_div(p1 - p0, kDescWaves)),
                           dim3(64 * kDescWaves), lds, s, A, p0, p1, desc);
        CUNA_LAUNCH_CHECK();
    }
}

// sort and buckets of short curves in one launch; false when a curve is too
// long or its (anchor, index) pairs too wide for it
template <typename T>
bool launch_plan_curves(const PointRec<T> *rec_orig, const int *coff, int ncurves, int longest,
                        int tlog, int G, int Kc, int olo, int ohi, PointRec<T> *rec, int *perm,
                        int *bucket, hipStream_t s) {
    const int ibits = std::max(1, ilog2(std::max(longest, 1)));
    if (longest > kPlanCurveMax || std::max(1, ilog2(G)) + ibits > 32) return false;
    if (ncurves <= 0) return true;
    // 256 threads where they hold a curve in 8 points each, so that several
    // curves share a CU
    const int NT = longest <= 2048 ? 256 : 1024;
    // as many workgroups per curve as keep to one per CU (their LDS takes all of
    // it) and have a point per thread on average; one curve of 20,011 points takes
    // 53 us with one workgroup, 26 with 16
    int parts = 1;
    while (NT == 1024 && parts < 16 && 2L * parts * ncurves <= num_cus() &&
           longest >= 2 * parts * NT && G >= 128 * parts)
        parts *= 2;
    const int abits = std::max(1, ilog2(ceil_div(G, parts)));  // of an anchor in its part
    const int cap = (std::max(longest, 1) + 7) & ~7;
    const int npass = (int)ceil_div(abits, kPlanDigitBits), bits = (int)ceil_div(abits, npass);
    const size_t lds = (sizeof(unsigned) + sizeof(short)) * (size_t)cap +
                       sizeof(short) * ((size_t)(NT / 64) << bits);
    auto go = [&](auto k) {
        set_lds(k, lds);
        hipLaunchKernelGGL(k, dim3(ncurves, parts), dim3(NT), lds, s, rec_orig, coff, cap, abits,
                           ibits, tlog, G, Kc, olo, ohi, rec, perm, bucket);
        CUNA_LAUNCH_CHECK();
    };
    if (NT == 256)
        go(k_plan_curve<T, 256, 8>);
    else if (longest <= 8 * 1024)
        go(k_plan_curve<T, 1024, 8>);
    else
        go(k_plan_curve<T, 1024, 23>);
    return true;
}

template <typename T, int NTP, int NG>
static void gather_one(GatherArgs<T> A, int nslabs, long npts, hipStream_t s) {
    // tiles per workgroup: on average at most one point per thread, LDS for
    // 4096 cells, and still a few workgroups per CU
    const long slots = (long)nslabs * A.ntiles;
    const long per_tile = std::max(1L, npts / std::max(1L, slots));
    int gl = 0;
    while (gl < 4 && (per_tile << (gl + 1)) <= 256 && A.tlog + gl + 1 <= 12 &&
           (1 << (gl + 1)) <= A.ntiles && (slots >> (gl + 1)) >= 4L * num_cus())
        ++gl;
    A.glog = gl;
    const size_t lds = NG * sizeof(T) * (((size_t)1 << (A.tlog + gl)) + NTP);
    require(lds <= kMaxLds, "gather tile too large", CUNA_ERROR_UNSUPPORTED);
    auto k = k_gather<T, NTP, NG>;
    set_lds(k, lds);
    const int nblk = (int)ceil_div(A.ntiles, 1L << gl);
    for (int s0 = 0; s0 < nslabs; s0 += kMaxGridY) {
        GatherArgs<T> B = A;
        B.slab0 = s0;
        hipLaunchKernelGGL(k, dim3(nblk, std::min(kMaxGridY, nslabs - s0)), dim3(256), lds, s, B);
        CUNA_LAUNCH_CHECK();
    }
}

template <typename T>
void launch_gather(const GatherArgs<T> &A, int ntaps, int nslabs, int ngrids, long npts,
                   hipStream_t s) {
    require(ntaps % 2 == 0, "unsupported filter width", CUNA_ERROR_UNSUPPORTED);
    dispatch_m<2, kMaxTaps / 2>(ntaps / 2, [&](auto c) {
        constexpr int NTP = decltype(c)::value;
        if (ngrids == 2)
            gather_one<T, NTP, 2>(A, nslabs, npts, s);
        else
            gather_one<T, NTP, 1>(A, nslabs, npts, s);
    });
}

// ------------------------------------------------------ fused bootstrap --
// grids up to 2^15 cells (float) / 2^14 (double): 128 KB of LDS, so one
// persistent workgroup per CU
template <typename T>
bool boot_fused_supported(int lgN, int ntaps) {
    return lgN >= 6 && lgN <= max_small_lg<T>() && (ntaps == 12 || ntaps == 16 || ntaps == 20 ||
                                                    ntaps == 24 || ntaps == 26 || ntaps == 32);
}

// workgroups that a fused kernel is launched with at most: as many as a CU's LDS
// holds, on every CU (rows of their workspaces)
template <typename T>
int fused_slots(int lgN) {
    return num_cus() * std::max(1, (int)(kMaxLds / boot_lds_bytes<T>(lgN)));
}

template <typename T, int LG>
static void adjoint_fused_tables(AdjointArgs<T> &A) {
    auto &tc = TwiddleCache<T>::get();
    constexpr int CAP = adjoint_cap<T>(LG);
    A.twT = tc.rows(LG, small_mr(LG), CAP);
    A.fine = sizeof(T) == 4 && LG > CAP ? tc.fine(LG) : nullptr;
    A.twN = tc.two_level(LG);
    A.twH = tc.head(LG + 1, fused_threads(LG));
}

template <typename T>
void warm_adjoint_fused(int lgN) {
    dispatch_lg<6, max_small_lg<T>()>(lgN, [&](auto c) {
        AdjointArgs<T> A{};
        adjoint_fused_tables<T, decltype(c)::value>(A);
    });
}

template <typename T, int LG, int NTAPS>
static void adjoint_fused_one(AdjointArgs<T> A, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
    constexpr int NT = fused_threads(LG);
    adjoint_fused_tables<T, LG>(A);
    constexpr size_t lds = adjoint_lds_bytes<T>(LG);
    static_assert(lds <= kMaxLds - 256, "fused adjoint LDS");
    auto k = k_adjoint_fused<T, LG, NTAPS, NT>;
    set_lds(k, lds);
    const int nblk = std::max(1, std::min(A.total, fused_slots<T>(LG)));
    if (ev0 || ev1)
        hipExtLaunchKernelGGL(k, dim3(nblk), dim3(NT), (uint32_t)lds, s, ev0, ev1, 0, A);
    else
        hipLaunchKernelGGL(k, dim3(nblk), dim3(NT), lds, s, A);
    CUNA_LAUNCH_CHECK();
}

// f(integral_constant) of a filter width that the fused kernels have
template <class F>
static void dispatch_fused_taps(int ntaps, F &&f) {
    switch (ntaps) {
        case 12: f(std::integral_constant<int, 12>{}); break;
        case 16: f(std::integral_constant<int, 16>{}); break;
        case 20: f(std::integral_constant<int, 20>{}); break;
        case 24: f(std::integral_constant<int, 24>{}); break;
        case 26: f(std::integral_constant<int, 26>{}); break;
        default: f(std::integral_constant<int, 32>{}); break;
    }
}

template <typename T>
void launch_adjoint_fused(const AdjointArgs<T> &A, int lgN, int ntaps, hipStream_t s,
                          hipEvent_t ev0, hipEvent_t ev1) {
    require(boot_fused_supported<T>(lgN, ntaps), "no fused adjoint kernel for this size",
            CUNA_ERROR_UNSUPPORTED);
    dispatch_lg<6, max_small_lg<T>()>(lgN, [&](auto c) {
        dispatch_fused_taps(ntaps, [&](auto t) {
            adjoint_fused_one<T, decltype(c)::value, decltype(t)::value>(A, s, ev0, ev1);
        });
    });
}

template <typename T, int LG, int NTAPS, int MODE>
static void boot_fused_one(BootArgs<T> A, hipStream_t s) {
    constexpr int NT = fused_threads(LG);
    auto &tc = TwiddleCache<T>::get();
    A.twT = tc.rows(LG, small_mr(LG), boot_cap<T>(LG));
    A.twN = tc.two_level(LG);
    A.twH = tc.head(LG + 1, NT);
    const size_t lds = boot_lds_bytes<T>(LG);
    static_assert(boot_lds_bytes<T>(LG) <= kMaxLds, "fused bootstrap LDS");
    auto k = k_boot_fused<T, LG, NTAPS, NT, MODE>;
    set_lds(k, lds);
    int dev = 0, ncu = 0;
    CUNA_HIP(hipGetDevice(&dev));
    CUNA_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    int per_cu = 0;
    CUNA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(k),
                                                          NT, lds));
    // one workspace row per workgroup
    require(A.list != nullptr && A.slots >= 1, "bootstrap workspace missing");
    const int resident = std::min(ncu * std::max(per_cu, 1), A.slots);
    if constexpr (MODE == 0) {
        // a replicate's transforms share its draws, unless there are too few
        // replicates to fill the chip a few times over.  Measured together /
        // apart: 128 curves x 25 replicates 528 / 583 us, 128 x 100 2004 / 2174 us
        A.split = A.ntr > 1 && A.total < 4 * resident;
        if (A.split) A.total *= A.ntr;
    }
    const int nblk = std::max(1, std::min(A.total, resident));
    hipLaunchKernelGGL(k, dim3(nblk), dim3(NT), lds, s, A);
    CUNA_LAUNCH_CHECK();
}

template <typename T>
void launch_curve_cover(const PointRec<T> *rec, const int *coff, int ncurves, int G, int ntaps,
                        int *cover, hipStream_t s) {
    require(is_pow2(G) && G <= (1 << 15), "cover histogram needs a power-of-two grid <= 2^15");
    if (ncurves <= 0) return;
    const size_t lds = 16 * (((size_t)cover_slot(G) + 3) / 4);
    set_lds(k_curve_cover<T>, lds);
    hipLaunchKernelGGL(k_curve_cover<T>, dim3(ncurves), dim3(1024), lds, s, rec, coff, G, ntaps,
                       cover);
    CUNA_LAUNCH_CHECK();
}

template <typename T>
void launch_boot_prepare(const T *y, const int *coff, const int *order, const int *cover_x,
                         const int *cover_2x, int ncurves, BootCurve *curves, int *counter,
                         hipStream_t s) {
    hipLaunchKernelGGL(k_boot_prepare<T>, dim3(ncurves), dim3(kPrepThreads), 0, s, y, coff, order,
                       cover_x, cover_2x, curves, counter);
    CUNA_LAUNCH_CHECK();
}

template <typename T>
void launch_boot_fused(BootArgs<T> A, int lgN, int ntaps, int mode, hipStream_t s) {
    require(boot_fused_supported<T>(lgN, ntaps), "no fused bootstrap kernel for this size",
            CUNA_ERROR_UNSUPPORTED);
    dispatch_lg<6, max_small_lg<T>()>(lgN, [&](auto c) {
        constexpr int LG = decltype(c)::value;
        auto go = [&](auto m) {
            dispatch_fused_taps(ntaps, [&](auto t) {
                boot_fused_one<T, LG, decltype(t)::value, decltype(m)::value>(A, s);
            });
        };
        if (mode == 0)
            go(std::integral_constant<int, 0>{});
        else
            go(std::integral_constant<int, 1>{});
    });
}

// ------------------------------------------------------- instantiation --
template void fft_real_forward<dTyp>(const FftShape &, dTyp *, const SinkAccurate<dTyp> &,
                                     hipStream_t, hipEvent_t);
template void fft_real_forward<dTyp>(const FftShape &, dTyp *, const SinkCompat<dTyp> &,
                                     hipStream_t, hipEvent_t);
template void fft_c2r_inverse<dTyp>(const FftShape &, const LoadHermitian<dTyp> &, cplx<dTyp> *,
                                    dTyp *, hipStream_t);
template void fft_complex<dTyp>(const FftShape &, cplx<dTyp> *, cplx<dTyp> *, int, hipStream_t);
template void launch_point_setup<dTyp>(const SetupArgs<dTyp> &, hipStream_t);
template void launch_sort_pass<dTyp>(const SortWork &, int, int, const PointRec<dTyp> *,
                                     const int *, PointRec<dTyp> *, int *, hipStream_t);
template void launch_buckets<dTyp>(const int *, int, int, const PointRec<dTyp> *, int, int, int, int,
                                   int *, hipStream_t);
template void launch_spread<dTyp>(const SpreadArgs<dTyp> &, int, int, int, hipStream_t, hipEvent_t,
                                  hipEvent_t);
template void launch_gather<dTyp>(const GatherArgs<dTyp> &, int, int, int, long, hipStream_t);
template void launch_tile_order<dTyp>(const SpreadArgs<dTyp> &, int, TileDesc *, hipStream_t);
template bool launch_plan_curves<dTyp>(const PointRec<dTyp> *, const int *, int, int, int, int, int,
                                       int, int, PointRec<dTyp> *, int *, int *, hipStream_t);
template bool boot_fused_supported<dTyp>(int, int);
template int fused_slots<dTyp>(int);
template void warm_adjoint_fused<dTyp>(int);
template void launch_adjoint_fused<dTyp>(const AdjointArgs<dTyp> &, int, int, hipStream_t,
                                         hipEvent_t, hipEvent_t);
template void launch_boot_fused<dTyp>(BootArgs<dTyp>, int, int, int, hipStream_t);
template void launch_curve_cover<dTyp>(const PointRec<dTyp> *, const int *, int, int, int, int *,
                                       hipStream_t);
template void launch_boot_prepare<dTyp>(const dTyp *, const int *, const int *, const int *,
                                        const int *, int, BootCurve *, int *, hipStream_t);

}  // namespace cuna
