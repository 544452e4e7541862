// cuna_chirp.hip -- Bluestein (chirp-z) transform for lengths that are not
// powers of two, on top of the power-of-two Stockham FFT.
//
// The reference's cuFFT stage takes any ng (cufftPlan1d / cufftPlanMany,
// src/cuna_kernel.cu:82,169,208,261; its test program uses ng = R*N,
// test.cpp:114).  A length-n transform is
//   A[r] = c_r * sum_g (z_g c_g) conj(c_{r-g}),  c_k = exp(+i pi k^2/n),
// with the convolution done circularly at L = 2^lgL >= 2 n - 1.  A real grid of
// even ng is read as n = ng/2 complex values, and its spectrum recovered from
// Z[r], Z[n-r] as in the power-of-two path; an odd one is transformed as n = ng
// complex values.  The chirp is tabulated on the host in long double from
// k^2 mod 2 n (exact integer), so its phase carries no error that grows with k.
//
// The chirp products, the two FFTs and the product with the convolution kernel's
// transform are fused: one launch when L fits a workgroup's LDS (and, at its
// largest, the rows are many), else three (the first column pass reads and
// premultiplies the grid; a row pass transforms each row forward, multiplies and
// transforms it back in LDS; the last column pass applies the chirp and writes the
// output), plus the even grid's pairing.  Bound by the passes' loads and stores, as
// the power-of-two FFT.  Measured at ng = 300,000, FP32: 63 us in seven launches
// over L = 2^20 -> 27 us in four over 2^19 (rocprofv3 sums).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "cuna_dispatch.hpp"
#include "cuna_plan.hpp"

namespace cuna {

// z_g c_g, zero from n on: the input of the first transform (row stride `stride`
// in elements of the source)
template <typename T>
struct LoadChirp {
    const cplx<T> *zc;  // complex values (a real grid's pairs), or
    const T *zr;        // a real grid of odd length
    const cplx<T> *chirp;
    long stride;
    int n;
    int conj_in;
    __device__ __forceinline__ void advance(long b) {
        if (zr)
            zr += b * stride;
        else
            zc += b * stride;
    }
    __device__ __forceinline__ cplx<T> at(int g) const {
        if (g >= n) return cmk(T(0), T(0));
        const cplx<T> c = chirp[(unsigned)g];
        if (zr) return c * zr[(unsigned)g];
        cplx<T> w = zc[(unsigned)g];
        if (conj_in) w.y = -w.y;
        return c * w;
    }
};

// what becomes of y_r, r < n: the transform is c_r y_r
enum ChirpOut {
    CHIRP_STORE = 0,   // kept in place (row stride L) for the pairing launch
    CHIRP_COMPAT = 1,  // through the compat deconvolution (odd real grids)
    CHIRP_PLAIN = 2    // data[b][r], conjugated on request
};
template <typename T>
struct ChirpSink {
    const cplx<T> *chirp;
    int n, mode, conj_out;
    cplx<T> *data;  // CHIRP_STORE / CHIRP_PLAIN
    long stride;
    SinkCompat<T> sk;  // CHIRP_COMPAT
    // the sink of batch row b (its data pointer advanced)
    __device__ __forceinline__ ChirpSink for_row(long b) const {
        ChirpSink r = *this;
        if (mode == CHIRP_COMPAT) {
            r.sk = sk.for_row(b);
            r.data = sk.row_out(b);
        } else {
            r.data = data + b * stride;
        }
        return r;
    }
    __device__ __forceinline__ void operator()(int r, cplx<T> y) const {
        if (r >= n) return;
        cplx<T> v = chirp[(unsigned)r] * y;
        if (mode == CHIRP_COMPAT) v = v * sk.fac(r);
        if (mode == CHIRP_PLAIN && conj_out) v.y = -v.y;
        *row_at(data, r) = v;
    }
};

// Row pass of the convolution: H consecutive rows r2 of the L1-contiguous data
// per workgroup.  Length-L1 transform (sign -1), product with bt (the kernel's
// transform over L, row-major: bt[r2 L1 + r1] = bhat[r2 + L2 r1] / L), length-L1
// transform (sign +1) and the twiddle w_L^(r2 n1), in place.
template <typename T, int LG1, int H, int NT, int MR>
__global__ __launch_bounds__(NT) void k_chirp_row(cplx<T> *a, long stride, int L2,
                                                  const cplx<T> *bt, const cplx<T> *tw,
                                                  Tw2<T> twL, long b0) {
    constexpr int L1 = 1 << LG1, NTAB = rows_count(LG1, MR, LG1);
    constexpr int NV = (H * L1 + NT - 1) / NT;
    static_assert(NV <= (1 << MR), "one butterfly per thread");
    cplx<T> *lds = reinterpret_cast<cplx<T> *>(cuna_smem);
    cplx<T> *twl = lds + H * L1;
    const int tid = threadIdx.x;
    const int2 bs = xcd_block(blockIdx.x, blockIdx.y, L2 / H, gridDim.y);
    const int i = bs.x;
    cplx<T> *z = a + (b0 + bs.y) * stride;
    TableStage<T, NTAB, NT> tab;
    tab.load(tw, tid);
    // the kernel's values in the order in which the second transform's first
    // pass takes them, and the epilogue's twiddles: loaded behind the data
    cplx<T> bv[1 << MR];
    Tw2Parts<T> ot[NV];
    auto row_index = [&](int e, int h) __attribute__((always_inline)) {
        return (unsigned)((i * H + h) * L1 + e);
    };
    auto fetch = [&](int e, int h) __attribute__((always_inline)) { return z[row_index(e, h)]; };
    auto hook = [&]() __attribute__((always_inline)) {
        tab.store(twl, tid);
        constexpr int Q = L1 >> pass_log2(LG1, 0, MR);
#pragma unroll
        for (int r = 0; r < (1 << pass_log2(LG1, 0, MR)); ++r)
            if ((H * Q) % NT == 0 || tid < H * Q) bv[r] = bt[row_index(tid / H + r * Q, tid % H)];
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int idx = tid + k * NT;
            if ((H * L1) % NT == 0 || idx < H * L1)
                ot[k].load(twL, (i * H + idx % H) * (idx / H));
        }
    };
    const TwRows<T, LG1, const cplx<T> *> rows{twl, tw};
    lds_fft<T, -1, LG1, H, NT, MR>(lds, rows, fetch, hook);
    int nv = 0;
    auto product = [&](int e, int h) __attribute__((always_inline)) {
        return lds[lds_sw(e * H + h)] * bv[nv++];
    };
    fft_pass<T, 1, LG1, H, NT, 0, 0, decltype(product), true, NoHook, decltype(rows), MR>(
        lds, rows, product, NoHook());
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int idx = tid + k * NT;
        if ((H * L1) % NT == 0 || idx < H * L1) {
            const int h = idx % H, n1 = idx / H;
            z[row_index(n1, h)] = lds[lds_sw(n1 * H + h)] * ot[k].get();
        }
    }
}

// Last column pass: W columns n1 per workgroup, length-L2 transform over r2 (sign
// +1); element n2 of column n1 is y_r, r = n1 + L1 n2.
template <typename T, int LG2, int W, int NT, int MR>
__global__ __launch_bounds__(NT) void k_chirp_col(const cplx<T> *a, long stride, int L1,
                                                  ChirpSink<T> sink, const cplx<T> *tw, long b0) {
    constexpr int L2 = 1 << LG2, NTAB = rows_count(LG2, MR, LG2);
    cplx<T> *lds = reinterpret_cast<cplx<T> *>(cuna_smem);
    cplx<T> *twl = lds + W * L2;
    const int tid = threadIdx.x;
    const int2 bs = xcd_block(blockIdx.x, blockIdx.y, L1 / W, gridDim.y);
    const int n10 = bs.x * W;
    const long b = b0 + bs.y;
    const cplx<T> *z = a + b * stride;
    TableStage<T, NTAB, NT> tab;
    tab.load(tw, tid);
    auto fetch = [&](int e, int w) __attribute__((always_inline)) {
        return z[(unsigned)(n10 + w + L1 * e)];
    };
    auto hook = [&]() __attribute__((always_inline)) { tab.store(twl, tid); };
    lds_fft<T, 1, LG2, W, NT, MR>(lds, TwRows<T, LG2, const cplx<T> *>{twl, tw}, fetch, hook);
    const ChirpSink<T> sk = sink.for_row(b);
    for (int idx = tid; idx < W * L2; idx += NT) {
        const int w = idx % W, n2 = idx / W;
        sk(n10 + w + L1 * n2, lds[lds_sw(n2 * W + w)]);
    }
}

// The spectrum of an even real grid from Z[r] = conv row b, r < n = ng/2
// (A[r] and A[n-r] from the pair Z[r], Z[n-r]; wr = exp(2 pi i r/ng)).
template <typename T>
__global__ __launch_bounds__(256) void k_chirp_pairs(const cplx<T> *Z, long L, int n,
                                                     const cplx<T> *wng, int batch,
                                                     SinkCompat<T> sk) {
    for (int b = blockIdx.y; b < batch; b += gridDim.y) {
        const SinkCompat<T> skb = sk.for_row(b);
        cplx<T> *o = sk.row_out(b);
        const cplx<T> *z = Z + b * L;
        for (int r = blockIdx.x * blockDim.x + threadIdx.x; r <= n / 2; r += gridDim.x * blockDim.x)
            emit_pair(skb, o, r, n, z[r], z[r == 0 ? 0 : n - r], wng[r]);
    }
}

// The whole transform of one batch row in LDS (L = 2^LG).  bt[k] = bhat[k] / L;
// wng: the pairing twiddles of an even real grid, else null.
template <typename T, int LG, int NT, int MR>
__global__ __launch_bounds__(NT) void k_chirp_small(LoadChirp<T> ld, ChirpSink<T> sink,
                                                    const cplx<T> *bt, const cplx<T> *wng,
                                                    const cplx<T> *tw, const cplx<T> *tw_rows) {
    constexpr int L = 1 << LG, CAP = small_cap(LG), NTAB = rows_count(LG, MR, CAP);
    cplx<T> *lds = reinterpret_cast<cplx<T> *>(cuna_smem);
    cplx<T> *twl = lds + L;
    const int tid = threadIdx.x;
    const long b = blockIdx.x;
    LoadChirp<T> lb = ld;
    lb.advance(b);
    TableStage<T, NTAB, NT> tab;
    tab.load(tw_rows, tid);
    auto fetch = [&](int e, int) __attribute__((always_inline)) { return lb.at(e); };
    auto hook = [&]() __attribute__((always_inline)) { tab.store(twl, tid); };
    const TwRows<T, CAP, const cplx<T> *> rows{twl, tw};
    lds_fft<T, -1, LG, 1, NT, MR>(lds, rows, fetch, hook);
    auto product = [&](int e, int) __attribute__((always_inline)) {
        return lds[lds_sw(e)] * bt[(unsigned)e];
    };
    fft_pass<T, 1, LG, 1, NT, 0, 0, decltype(product), true, NoHook, decltype(rows), MR>(
        lds, rows, product, NoHook());
    const ChirpSink<T> sk = sink.for_row(b);
    const int n = sk.n;
    if (wng) {
        for (int r = tid; r <= n / 2; r += NT) {
            const int rn = r == 0 ? 0 : n - r;
            emit_pair(sk.sk, sk.data, r, n, sk.chirp[r] * lds[lds_sw(r)],
                      sk.chirp[rn] * lds[lds_sw(rn)], wng[r]);
        }
    } else {
        for (int r = tid; r < n; r += NT) sk(r, lds[lds_sw(r)]);
    }
}

// b_k = b_{L-k} = conj(c_k), k < n, zero between
template <typename T>
__global__ void k_chirp_kernel(const cplx<T> *chirp, int n, long L, cplx<T> *out) {
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= L) return;
    const long m = k < n ? k : L - k;
    out[k] = m < n ? conjg(chirp[m]) : cmk(T(0), T(0));
}
// bt[r2 L1 + r1] = bhat[r2 + L2 r1] * scale
template <typename T>
__global__ void k_chirp_rows(const cplx<T> *bhat, int L1, int L2, T scale, cplx<T> *bt) {
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long)L1 * L2) return;
    const long r2 = k / L1, r1 = k % L1;
    bt[k] = bhat[r2 + (long)L2 * r1] * scale;
}

template <typename T>
void Bluestein<T>::init(int length, bool real, hipStream_t s) {
    require(length >= 1, "transform length must be positive");
    ng = length;
    pairs = real && length % 2 == 0;
    n = pairs ? length / 2 : length;
    lgL = std::max(1, ilog2(2L * n - 1));
    L = 1L << lgL;
    require(lgL <= max_fft_lg<T>(), "transform length too large", CUNA_ERROR_UNSUPPORTED);
    const long double pi = 3.141592653589793238462643383279502884L;
    const int nw = pairs ? n / 2 + 1 : 0;
    tab_h.resize((size_t)n + nw);
    for (long k = 0; k < n; ++k) {
        const unsigned long long q =
            ((unsigned long long)k * (unsigned long long)k) % (2ull * (unsigned long long)n);
        const long double a = pi * (long double)q / (long double)n;
        tab_h[k] = cmk((T)cosl(a), (T)sinl(a));
    }
    for (long r = 0; r < nw; ++r) {
        const long double a = 2 * pi * (long double)r / (long double)ng;
        tab_h[n + r] = cmk((T)cosl(a), (T)sinl(a));
    }
    tab.alloc(sizeof(cplx<T>) * tab_h.size(), s);
    bt.alloc(sizeof(cplx<T>) * L, s);
    CUNA_HIP(hipMemcpyAsync(tab.ptr, tab_h.data(), sizeof(cplx<T>) * tab_h.size(),
                            hipMemcpyHostToDevice, s));
    TwiddleCache<T>::get().warm(lgL);
    ensure(1, s);
    // the kernel's transform, scaled, in the order in which the passes take it
    // (bt is the FFT's workspace before it receives the result)
    cplx<T> *const w = work.as<cplx<T>>();
    hipLaunchKernelGGL(k_chirp_kernel<T>, dim3(ceil_div(L, 256)), dim3(256), 0, s, chirp(), n, L,
                       w);
    CUNA_LAUNCH_CHECK();
    FftShape sh;
    sh.lgN = lgL;
    sh.batch = 1;
    fft_complex<T>(sh, w, bt.as<cplx<T>>(), -1, s);
    const int lg1 = lgL <= max_small_lg<T>() ? 0 : split_lg1(lgL);
    hipLaunchKernelGGL(k_chirp_rows<T>, dim3(ceil_div(L, 256)), dim3(256), 0, s, w, 1 << lg1,
                       1 << (lgL - lg1), T(1) / (T)L, bt.as<cplx<T>>());
    CUNA_LAUNCH_CHECK();
    if (both_forms()) {
        bt_rows.alloc(sizeof(cplx<T>) * L, s);
        const int l1 = split_lg1(lgL);
        hipLaunchKernelGGL(k_chirp_rows<T>, dim3(ceil_div(L, 256)), dim3(256), 0, s, w, 1 << l1,
                           1 << (lgL - l1), T(1) / (T)L, bt_rows.as<cplx<T>>());
        CUNA_LAUNCH_CHECK();
    }
}

// The largest length that one workgroup holds.  Its two FFTs take one CU 20 us, so
// few rows go through the three passes, which spread them over the chip.  `rows`
// decides, not the batch, and the passes have one shape (kBothW, both_h), because a
// curve's bits do not depend on the batch that it is in.  Measured with the spread,
// one workgroup per row / three passes: FP32, ng = 5001, 1 row 32.6 / 16.8 us, 64
// rows 33.9 / 27.9, 100 rows 35.7 / 36.9, 256 rows 46 / 69; FP64, ng = 2501, 1 row
// 25.5 / 18.9, 16 rows 25.5 / 19.3, 64 rows 26.6 / 26.6, 256 rows 31 / 55.  (FP32 at
// 2^13: 20.5 / 21.9 us at 2 rows.)  Eight sequences per workgroup 18.5 and 56 us.
template <typename T>
bool Bluestein<T>::both_forms() const {
    return lgL == max_small_lg<T>();
}
template <typename T>
static constexpr int cus_per_pass_row() {  // rows up to num_cus() over this are few
    return sizeof(T) == 4 ? 4 : 8;
}
constexpr int kBothW = 2;
template <typename T>
constexpr int both_h() {
    return sizeof(T) == 4 ? 2 : 4;
}

template <typename T>
void Bluestein<T>::ensure(int batch, hipStream_t s) {
    work.ensure(sizeof(cplx<T>) * (size_t)L * (size_t)batch, s);
}

template <typename T>
void Bluestein<T>::run(const LoadChirp<T> &ld, const ChirpSink<T> &sink, int batch, int rows,
                       hipStream_t s) {
    require(sizeof(cplx<T>) * (size_t)L * (size_t)batch <= work.bytes,
            "Bluestein workspace too small for this batch");
    work.use(s);
    auto &tc = TwiddleCache<T>::get();
    const cplx<T> *const wng = pairs ? chirp() + n : nullptr;
    const bool both = both_forms();
    if (lgL <= max_small_lg<T>() && !(both && rows <= num_cus() / cus_per_pass_row<T>())) {
        dispatch_lg<1, max_small_lg<T>()>(lgL, [&](auto c) {
            constexpr int LG = decltype(c)::value, MR = small_mr(LG), CAP = small_cap(LG);
            constexpr int NT = fft_threads(LG, 1, MR);
            constexpr size_t lds =
                sizeof(cplx<T>) * (((size_t)1 << LG) + rows_count(LG, MR, CAP));
            auto k = k_chirp_small<T, LG, NT, MR>;
            set_lds(k, lds);
            hipLaunchKernelGGL(k, dim3(batch), dim3(NT), lds, s, ld, sink, bt.as<cplx<T>>(), wng,
                               LG > CAP ? tc.fine(LG) : nullptr, tc.rows(LG, MR, CAP));
            CUNA_LAUNCH_CHECK();
        });
        return;
    }
    const int lg1 = split_lg1(lgL), lg2 = lgL - lg1, L1 = 1 << lg1, L2 = 1 << lg2;
    const int W = pick_seq<T>(lg2, L1, batch, 1, "CUNA_FFT_W", both ? kBothW : 0, num_cus());
    const int H = pick_seq<T>(lg1, L2, batch, 1, "CUNA_FFT_H", both ? both_h<T>() : 0, num_cus());
    cplx<T> *const a = work.as<cplx<T>>();
    const cplx<T> *const b = (both ? bt_rows : bt).template as<cplx<T>>();
    auto batches = [&](auto &&launch) {
        for (long b0 = 0; b0 < batch; b0 += kMaxGridY) {
            launch(b0, (int)std::min<long>(kMaxGridY, batch - b0));
            CUNA_LAUNCH_CHECK();
        }
    };
    dispatch_lg<7, 12>(lg2, [&](auto c) {
        constexpr int LG2 = decltype(c)::value;
        dispatch_w<T, LG2>(W, [&](auto w) {
            constexpr int WW = decltype(w)::value, NT = fft_threads(LG2, WW, kColMr);
            constexpr size_t lds =
                sizeof(cplx<T>) * (((size_t)WW << LG2) + rows_count(LG2, kColMr, LG2));
            auto k = k_fft_col<T, -1, LG2, WW, NT, LoadChirp<T>, kColMr>;
            set_lds(k, lds);
            batches([&](long b0, int nb) {
                hipLaunchKernelGGL(k, dim3(L1 / WW, nb), dim3(NT), lds, s, ld, a, L, L1,
                                   tc.rows(LG2, kColMr, LG2), tc.two_level(lgL), b0);
            });
        });
    });
    dispatch_lg<6, 12>(lg1, [&](auto c) {
        constexpr int LG1 = decltype(c)::value;
        dispatch_w<T, LG1>(H, [&](auto h) {
            constexpr int HH = decltype(h)::value, NT = fft_threads(LG1, HH, kRowMr);
            constexpr size_t lds =
                sizeof(cplx<T>) * (((size_t)HH << LG1) + rows_count(LG1, kRowMr, LG1));
            auto k = k_chirp_row<T, LG1, HH, NT, kRowMr>;
            set_lds(k, lds);
            batches([&](long b0, int nb) {
                hipLaunchKernelGGL(k, dim3(L2 / HH, nb), dim3(NT), lds, s, a, L, L2,
                                   b, tc.rows(LG1, kRowMr, LG1), tc.two_level(lgL), b0);
            });
        });
    });
    ChirpSink<T> out = sink;
    if (pairs) {
        out.mode = CHIRP_STORE;
        out.data = a;
        out.stride = L;
    }
    dispatch_lg<7, 12>(lg2, [&](auto c) {
        constexpr int LG2 = decltype(c)::value;
        dispatch_w<T, LG2>(W, [&](auto w) {
            constexpr int WW = decltype(w)::value, NT = fft_threads(LG2, WW, kColMr);
            constexpr size_t lds =
                sizeof(cplx<T>) * (((size_t)WW << LG2) + rows_count(LG2, kColMr, LG2));
            auto k = k_chirp_col<T, LG2, WW, NT, kColMr>;
            set_lds(k, lds);
            batches([&](long b0, int nb) {
                hipLaunchKernelGGL(k, dim3(L1 / WW, nb), dim3(NT), lds, s, a, L, L1, out,
                                   tc.rows(LG2, kColMr, LG2), b0);
            });
        });
    });
    if (pairs) {
        const long bx = std::min<long>(ceil_div(n / 2 + 1, 256), 4096);
        hipLaunchKernelGGL(k_chirp_pairs<T>, dim3(bx, std::min(batch, kMaxGridY)), dim3(256), 0, s,
                           a, L, n, wng, batch, sink.sk);
        CUNA_LAUNCH_CHECK();
    }
}

template <typename T>
void Bluestein<T>::run_real(const T *grid, long gstride, int batch, int rows,
                            const SinkCompat<T> &sk, hipStream_t s) {
    LoadChirp<T> ld{};
    ld.chirp = chirp();
    ld.n = n;
    if (pairs) {
        ld.zc = reinterpret_cast<const cplx<T> *>(grid);
        ld.stride = gstride / 2;
    } else {
        ld.zr = grid;
        ld.stride = gstride;
    }
    ChirpSink<T> sink{};
    sink.chirp = chirp();
    sink.n = n;
    sink.mode = CHIRP_COMPAT;
    sink.sk = sk;
    run(ld, sink, batch, rows, s);
}

template <typename T>
void Bluestein<T>::run_complex(cplx<T> *data, int batch, int sign, hipStream_t s) {
    // sign -1 as the conjugate of the sign +1 transform of the conjugate
    LoadChirp<T> ld{};
    ld.zc = data;
    ld.stride = ng;
    ld.chirp = chirp();
    ld.n = n;
    ld.conj_in = sign < 0 ? 1 : 0;
    ChirpSink<T> sink{};
    sink.chirp = chirp();
    sink.n = n;
    sink.mode = CHIRP_PLAIN;
    sink.conj_out = ld.conj_in;
    sink.data = data;
    sink.stride = ng;
    run(ld, sink, batch, batch, s);
}

template struct Bluestein<dTyp>;

}  // namespace cuna
