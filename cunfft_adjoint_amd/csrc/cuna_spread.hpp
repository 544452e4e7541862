// cuna_spread.hpp -- sort-by-tile Gaussian spread (and its transpose, the
// gather of the backward pass) for gfx950.
//
// Replaces fast_gridding / fast_gridding_bootstrap (src/gridding.cu:36-117),
// which scatter every tap of every point with a global atomicAdd.  Here the
// points of one x are sorted once per plan by anchor (a stable radix sort, in one
// launch for short curves), which orders them by the buckets key = 3*tile + class
// (class 0: taps reach the previous tile, 2: the next tile, 1: interior).  One
// workgroup owns one tile: it takes the points of its own bucket plus the
// boundary classes of its two neighbours and accumulates the taps that land
// in its tile in LDS, then writes the tile once with coalesced stores.  No
// global atomics, and every accumulation form is bitwise reproducible:
//   k_spread_wv (default): one wave per tile, integer atomics in fixed point
//     (32-bit cells in FP32, 64-bit in FP64; integer sums do not depend on
//     their order), tiles taken densest first;
//   k_spread (on request, CUNA_PLAN_GATHER): gather, each cell summed by
//     one thread in a fixed order.
// The fused bootstrap kernel (k_boot_fused) keeps a whole curve's grid in
// LDS; the backward's gather (k_gather) is the transpose of the spread.
#pragma once

#include <type_traits>

#include "cuna_common.hpp"
#include "cuna_fft.hpp"

namespace cuna {

constexpr int kMaxTaps = 32;

template <typename T>
struct PointRec {
    int a;  // anchor cell
    T e;    // weight parameter: taps at a+o weigh exp(-(o-e)^2/beta)
};

// ---------------------------------------------------- bootstrap RNG --
// src/gridding.cu:67-82
__device__ __host__ __forceinline__ uint32_t wang_hash(uint32_t s) {
    s = (s ^ 61u) ^ (s >> 16);
    s *= 9u;
    s = s ^ (s >> 4);
    s *= 0x27d4eb2du;
    s = s ^ (s >> 15);
    return s;
}
__device__ __host__ __forceinline__ uint32_t xorshift32(uint32_t s) {
    s ^= (s << 13);
    s ^= (s >> 17);
    s ^= (s << 5);
    return s;
}

// x mod d for 32-bit unsigned x and a divisor 1 <= d < 2^31 shared by many x,
// exact (Granlund & Montgomery 1994, unsigned division by a run-time
// invariant): l = ceil(log2 d), m = floor(2^32 (2^l - d) / d) + 1,
// q = (t + ((x - t) >> min(l,1))) >> max(l-1,0) with t = mulhi(m, x).
struct FastMod {
    uint32_t d, m;
    int s1, s2;
    __device__ __host__ void init(uint32_t d_) {
        d = d_;
        int l = 0;
        while ((1ull << l) < d) ++l;
        m = (uint32_t)(((1ull << 32) * ((1ull << l) - d)) / d + 1);
        s1 = l < 1 ? l : 1;
        s2 = l > 1 ? l - 1 : 0;
    }
    __device__ __forceinline__ uint32_t operator()(uint32_t x) const {
        const uint32_t t = __umulhi(m, x);
        const uint32_t q = (t + ((x - t) >> s1)) >> s2;
        return x - q * d;
    }
};

// ------------------------------------------------------ point setup --
enum SetupMode { SETUP_COMPAT = 0, SETUP_ACC_X = 1, SETUP_ACC_T = 2 };

template <typename T>
struct SetupArgs {
    const T *x;        // SETUP_COMPAT / SETUP_ACC_X
    const double *t;   // SETUP_ACC_T: x = frac(df * t) computed in FP64
    double df;
    int mode;
    int G;             // grid cells per curve (ng in compat)
    int R_f;           // compat filter radius
    T b, e1s;          // compat b and 1/sqrt(pi b)
    T *E1, *E2, *E3;   // compat filter_properties arrays (nullable)
    T *eps_orig;       // compat: eps by original index (nullable)
    long n;
    PointRec<T> *rec;  // out: (anchor, e) by original index
};

// compat decisions in the build's precision, one rounding per operation
// (src/gaussian_filter.cu:213-216): u = (int)(ng*x - R_f), eps = ng*x - u;
// src/gridding.cu:43-45: j = (int)((x + 0.5)*(ng - 1)) in double, clamped.
template <typename T>
__device__ __forceinline__ void compat_point(T x, int ng, int R_f, int &j, T &eps) {
#pragma clang fp contract(off)
    T prod = (T)ng * x;
    T v = prod - (T)R_f;
    int u = (int)v;
    eps = prod - (T)u;
    j = (int)(((double)x + 0.5) * (double)(ng - 1));
    if (j >= ng) j = ng - 1;
    if (j < 0) j = 0;
}

template <typename T>
__device__ __forceinline__ void setup_point(const SetupArgs<T> &A, long i, int &a, T &e) {
    if (A.mode == SETUP_COMPAT) {
        compat_point<T>(A.x[i], A.G, A.R_f, a, e);
        if (A.E1) {
            // src/gaussian_filter.cu:216-220
            T e2 = e / A.b;
            A.E1[i] = (T)exp(-e * e2) * A.e1s;
            A.E2[i] = (T)exp(2 * e2);
        }
        if (A.eps_orig) A.eps_orig[i] = e;
    } else {
        // accurate: t = G*x, anchor floor(t) mod G, e = t - floor(t).  With G
        // a power of two, G*x and t - floor(t) are exact in FP64 and the
        // anchor is reduced in integers: no bit of x is lost (reducing x to
        // [0, 1) first would round x + 1 for negative x).  Times: x = df*t
        // in FP64 (one rounding).
        const double xv = A.mode == SETUP_ACC_T ? A.df * A.t[i] : (double)A.x[i];
        const double tg = xv * (double)A.G;
        const double c = floor(tg);
        T f = (T)(tg - c);
        // (non-finite x: anchor 0 and a NaN e, which makes the output NaN)
        long long ci = fabs(c) < 0x1p62 ? (long long)c : 0;
        if (f >= T(1)) {  // rounding of tg - c to T
            f = T(0);
            ci += 1;
        }
        a = (int)(ci & (long long)(A.G - 1));  // G is a power of two
        e = f;
    }
}

template <typename T>
__global__ void k_point_setup(SetupArgs<T> A) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (A.E3 && i < A.R_f) {
        // src/gaussian_filter.cu:222-226: E3[m] = exp(-m^2/b)
        const int m = (int)i;
        A.E3[m] = (T)exp(-(T)(m * m) / A.b);
    }
    if (i >= A.n) return;
    int a;
    T e;
    setup_point(A, i, a, e);
    PointRec<T> pr;
    pr.a = a;
    pr.e = e;
    A.rec[i] = pr;
}

__device__ __forceinline__ int tile_key(int a, int tlog, int olo, int ohi, int G) {
    int tile = a >> tlog;
    int ts = tile << tlog;
    int te = min(ts + (1 << tlog), G);
    int cls = (a + olo < ts) ? 0 : ((a + ohi >= te) ? 2 : 1);
    return 3 * tile + cls;
}

// The lanes of the wave with the same digit (of at most NBITS bits) as this one,
// among those in `act`: rank below the lane and count (NBITS ballots, about four
// instructions each).
template <int NBITS>
__device__ __forceinline__ void match_digit(unsigned d, unsigned long long act, int &rank,
                                            int &count) {
    unsigned lo = (unsigned)act, hi = (unsigned)(act >> 32);
#pragma unroll
    for (int b = 0; b < NBITS; ++b) {  // (bits past the digit's are 0)
        const int t = __builtin_amdgcn_sbfe((int)d, b, 1);  // 0 or ~0
        const unsigned long long m = __ballot(t < 0);
        lo &= ~((unsigned)m ^ (unsigned)t);
        hi &= ~((unsigned)(m >> 32) ^ (unsigned)t);
    }
    rank = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
    count = __popc(lo) + __popc(hi);
}

// A stable counting sort pass over the digit (anchor >> shift) & (K - 1).  Points
// are cut into chunks of at most kSortChunk that never cross a curve; the
// per-chunk counts form a key-major matrix hist[curve base + key * nch + chunk],
// whose exclusive scan gives every chunk's first position for every key.  One
// wave handles one chunk, all of whose loads it issues first: with a step's loads
// issued when its turn came, the scatter of 1e6 points took 24 us, now 15 us.
constexpr int kSortChunk = 512, kSortBits = 8, kSortSteps = kSortChunk / 64;
struct SortArgs {
    const int4 *chunks;     // {curve, start, len, column}
    const int *chunk_base;  // chunks before each curve
    const int *nch;         // chunks per curve
    int nchunks, K, shift;
    int *hist;
};

__device__ __forceinline__ long hist_index(const SortArgs &S, int4 cd, int k) {
    return (long)S.K * S.chunk_base[cd.x] + (long)k * S.nch[cd.x] + cd.w;
}

template <typename T>
__global__ void k_hist(SortArgs S, const PointRec<T> *rec) {
    int *cnt_all = reinterpret_cast<int *>(cuna_smem);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int ch = blockIdx.x * (blockDim.x >> 6) + wave;
    int *cnt = cnt_all + wave * S.K;
    for (int k = lane; k < S.K; k += 64) cnt[k] = 0;
    if (ch >= S.nchunks) return;  // (no workgroup barriers)
    const int4 cd = S.chunks[ch];
    int a[kSortSteps];  // (clamped loads: all issue together)
#pragma unroll
    for (int r = 0; r < kSortSteps; ++r)
        a[r] = rec[(long)cd.y + min(r * 64 + lane, cd.z - 1)].a;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int r = 0; r < kSortSteps; ++r)
        if (r * 64 + lane < cd.z) atomicAdd(&cnt[(a[r] >> S.shift) & (S.K - 1)], 1);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int k = lane; k < S.K; k += 64) S.hist[hist_index(S, cd, k)] = cnt[k];
}

// scatter with ranks that keep the input order among equal keys
template <typename T>
__global__ void k_scatter(SortArgs S, const PointRec<T> *rec_in, const int *perm_in,
                          PointRec<T> *rec_out, int *perm_out) {
    int *cur_all = reinterpret_cast<int *>(cuna_smem);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int ch = blockIdx.x * (blockDim.x >> 6) + wave;
    int *cur = cur_all + wave * S.K;
    if (ch >= S.nchunks) return;  // (no workgroup barriers)
    const int4 cd = S.chunks[ch];
    PointRec<T> pr[kSortSteps];
    int pm[kSortSteps];
#pragma unroll
    for (int r = 0; r < kSortSteps; ++r) {
        const long i = (long)cd.y + min(r * 64 + lane, cd.z - 1);
        pr[r] = rec_in[i];
        pm[r] = perm_in ? perm_in[i] : (int)i;
    }
    for (int k = lane; k < S.K; k += 64) cur[k] = S.hist[hist_index(S, cd, k)];
#pragma unroll
    for (int r = 0; r < kSortSteps; ++r) {
        const int na = cd.z - r * 64;
        if (na <= 0) break;  // uniform
        const unsigned d = (unsigned)(pr[r].a >> S.shift) & (unsigned)(S.K - 1);
        int rank, count;
        match_digit<kSortBits>(d, na >= 64 ? ~0ull : (1ull << na) - 1ull, rank, count);
        const int pos = cur[d] + rank;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lane < na) {
            rec_out[pos] = pr[r];
            perm_out[pos] = pm[r];
            if (rank == count - 1) cur[d] = pos + 1;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// bucket[c*(Kc+1) + k] = first sorted index of the curve's points with
// tile_key >= k (k = Kc: the curve's end).  The points are sorted by anchor,
// and tile_key is non-decreasing in the anchor (the class is 0 for a prefix
// of the tile's cells and 2 for a suffix), so a binary search finds it.
template <typename T>
__global__ void k_buckets(const int *coff, int ncurves, int Kc, const PointRec<T> *rec, int tlog,
                          int olo, int ohi, int G, int *bucket) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)ncurves * (Kc + 1)) return;
    const int c = (int)(idx / (Kc + 1)), k = (int)(idx % (Kc + 1));
    int lo = k < Kc ? coff[c] : coff[c + 1], hi = coff[c + 1];
    while (lo < hi) {
        const int mid = lo + ((hi - lo) >> 1);
        if (tile_key(rec[mid].a, tlog, olo, ohi, G) < k)
            lo = mid + 1;
        else
            hi = mid;
    }
    bucket[idx] = lo;
}

// ---------------------------------------- sort of short curves: one launch --
// The sort by anchor and the buckets of a curve, for curves of at most
// kPlanCurveMax points whose (anchor, index) pairs fit 32 bits, by gridDim.y
// workgroups that share the curve's anchor range: each takes the points of its
// part of the range, in order of index, sorts them alone and writes them behind
// the points of the parts below, which it has counted on the way.  A point is the
// word anchor << ibits | index, held in LDS (room for all of the curve, so that
// clustered points change only the time); an LSD radix sort over the anchor's bits
// (digits of at most 9) permutes the words: stable, so the order is that of the
// multi-launch sort.  Wave w ranks the consecutive words [w seg, (w + 1) seg), 64
// per step: a word's rank is the count of equal digits in the wave's earlier steps
// (16-bit counters per wave) plus the lower lanes with the same digit (nine
// ballots); the scan of the counters turns it into a place, and every thread moves
// its IPT words through registers.  Bound by instruction issue in the ranking
// steps, hence the split where curves are fewer than CUs.  It stands in for the
// sort's launches (histogram, two scan steps and scatter per digit, and the
// buckets).  Measured: 64 curves of 20,000 points and 2^17 cells 34 us with 4 parts
// (50 with one); one curve of 20,011 points and 2^16 cells, FP64, 26 us with 16 (53
// with one).
constexpr int kPlanCurveMax = 23 * 1024, kPlanDigitBits = 9;

template <typename T, int NT, int IPT>
__global__ __launch_bounds__(NT) void k_plan_curve(const PointRec<T> *rec_orig, const int *coff,
                                                   int cap, int abits, int ibits, int tlog, int G,
                                                   int Kc, int olo, int ohi, PointRec<T> *rec,
                                                   int *perm, int *bucket) {
    constexpr int NW = NT / 64, UN = 4;
    unsigned *sv = reinterpret_cast<unsigned *>(cuna_smem);              // cap words
    unsigned short *rk = reinterpret_cast<unsigned short *>(sv + cap);   // cap ranks
    unsigned short *cnt = rk + cap;                                      // [wave][digit]
    __shared__ int wsum[NW], wbelow[NW];
    const int c = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // this workgroup's anchors [alo, ahi); the outer parts are open
    const int part = blockIdx.y, parts = gridDim.y;
    const int alo = part > 0 ? (int)((long)part * G / parts) : INT_MIN;
    const int ahi = part + 1 < parts ? (int)((long)(part + 1) * G / parts) : INT_MAX;
    const int abase = part > 0 ? alo : 0;  // the words' anchors count from here
    const int c0 = coff[c];
    int n = coff[c + 1] - c0;
    int below = 0;  // points of the parts below
    {
        const int len = (n + NT - 1) / NT * 64, q0 = min(wave * len, n), q1 = min(q0 + len, n);
        int a[IPT], mine = 0;
#pragma unroll
        for (int s = 0; s < IPT; ++s)  // (clamped loads: all issue together)
            a[s] = s * 64 < len ? rec_orig[c0 + max(min(q0 + s * 64 + lane, q1 - 1), 0)].a : 0;
#pragma unroll
        for (int s = 0; s < IPT; ++s) {
            if (s * 64 < len) {
                const bool in = q0 + s * 64 + lane < q1;
                below += __popcll(__ballot(in && a[s] < alo));
                mine += __popcll(__ballot(in && a[s] >= alo && a[s] < ahi));
            }
        }
        if (lane == 0) {
            wsum[wave] = mine;
            wbelow[wave] = below;
        }
        __syncthreads();
        int at = 0;
        mine = below = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            if (w < wave) at += wsum[w];
            mine += wsum[w];
            below += wbelow[w];
        }
#pragma unroll
        for (int s = 0; s < IPT; ++s) {
            if (s * 64 < len) {
                const int q = q0 + s * 64 + lane;
                const bool in = q < q1 && a[s] >= alo && a[s] < ahi;
                const unsigned long long m = __ballot(in);
                if (in)
                    sv[at + __builtin_amdgcn_mbcnt_hi(
                                (unsigned)(m >> 32),
                                __builtin_amdgcn_mbcnt_lo((unsigned)m, 0))] =
                        (unsigned)(a[s] - abase) << ibits | (unsigned)q;
                at += __popcll(m);
            }
        }
        n = __builtin_amdgcn_readfirstlane(mine);
        below = __builtin_amdgcn_readfirstlane(below);
        __syncthreads();
    }
    const int seg = (n + NT - 1) / NT * 64;  // words per wave
    const int w0 = min(wave * seg, n), w1 = min(w0 + seg, n);
    int shift = ibits, left = abits;
    for (int pass = (abits + kPlanDigitBits - 1) / kPlanDigitBits; pass > 0; --pass) {
        const int bits = (left + pass - 1) / pass, K = 1 << bits;
        const unsigned mask = K - 1;
        unsigned short *cw = cnt + wave * K;
        for (int i = tid; i < NW * K / 2; i += NT) reinterpret_cast<unsigned *>(cnt)[i] = 0;
        __syncthreads();
        for (int q0 = w0; q0 < w1; q0 += 64) {  // uniform
            const int na = min(64, w1 - q0);
            const unsigned long long act = na == 64 ? ~0ull : (1ull << na) - 1ull;
            const int q = min(q0 + lane, w1 - 1);
            const unsigned d = (sv[q] >> shift) & mask;
            // (a lane past the end counts all its peers as lower: it never writes)
            int r, peers;
            if (bits <= 6)  // uniform
                match_digit<6>(d, act, r, peers);
            else
                match_digit<kPlanDigitBits>(d, act, r, peers);
            const int cur = cw[d];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (r == peers - 1) cw[d] = (unsigned short)(cur + r + 1);
            if (lane < na) rk[q] = (unsigned short)(cur + r);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        // exclusive scan of the counters, by digit and then wave; a thread
        // takes every NT-th digit
        int carry = 0;
        for (int d0 = 0; d0 < K; d0 += NT) {
            const int d = d0 + tid;
            int own[NW], tot = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                own[w] = d < K ? cnt[w * K + d] : 0;
                tot += own[w];
            }
            int incl = tot;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int u = __shfl_up(incl, o);
                if (lane >= o) incl += u;
            }
            if (lane == 63) wsum[wave] = incl;
            __syncthreads();
            int at = carry + incl - tot, all = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                if (w < wave) at += wsum[w];
                all += wsum[w];
            }
            carry += all;
            if (d < K) {
#pragma unroll
                for (int w = 0; w < NW; ++w) {
                    cnt[w * K + d] = (unsigned short)at;
                    at += own[w];
                }
            }
            __syncthreads();
        }
        // every word to its place, through registers
        unsigned v[IPT];
        unsigned short to[IPT];
#pragma unroll
        for (int s = 0; s < IPT; ++s) {
            v[s] = 0;
            to[s] = 0;
            if (s * 64 < seg) {  // uniform
                const int q = max(min(w0 + s * 64 + lane, w1 - 1), 0);
                v[s] = sv[q];
                to[s] = (unsigned short)(rk[q] + cw[(v[s] >> shift) & mask]);
            }
            if (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // fewer registers
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < IPT; ++s)
            if (w0 + s * 64 + lane < w1) sv[to[s]] = v[s];
        __syncthreads();
        shift += bits;
        left -= bits;
    }
    // sorted records and original indices
    const unsigned imask = (1u << ibits) - 1u;
    for (int j0 = tid; j0 < n; j0 += UN * NT) {
        unsigned w[UN];
        T e[UN];
#pragma unroll
        for (int k = 0; k < UN; ++k) w[k] = sv[min(j0 + k * NT, n - 1)];
#pragma unroll
        for (int k = 0; k < UN; ++k) e[k] = rec_orig[c0 + (w[k] & imask)].e;
#pragma unroll
        for (int k = 0; k < UN; ++k) {
            const int j = j0 + k * NT;
            if (j < n) {
                PointRec<T> pr;
                pr.a = abase + (int)(w[k] >> ibits);
                pr.e = e[k];
                rec[c0 + below + j] = pr;
                perm[c0 + below + j] = c0 + (int)(w[k] & imask);
            }
        }
    }
    // bucket[k]: first sorted point with tile_key >= k, as in k_buckets; the keys
    // whose first anchor lies in this part
    const int k0 = part > 0 ? tile_key(alo - 1, tlog, olo, ohi, G) + 1 : 0;
    const int k1 = part + 1 < parts ? tile_key(ahi - 1, tlog, olo, ohi, G) : Kc;
    for (int k = k0 + tid; k <= k1; k += NT) {
        int lo = k < Kc ? 0 : n, hi = n;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (tile_key(abase + (int)(sv[mid] >> ibits), tlog, olo, ohi, G) < k)
                lo = mid + 1;
            else
                hi = mid;
        }
        bucket[(long)c * (Kc + 1) + k] = c0 + below + lo;
    }
}

// ------------------------------------------------ exclusive int scan --
constexpr int kScanNT = 1024, kScanIPT = 4, kScanTile = kScanNT * kScanIPT;

__device__ __forceinline__ int block_exclusive_scan(int v, int *sh, int &total) {
    const int tid = threadIdx.x;
    sh[tid] = v;
    __syncthreads();
    for (int off = 1; off < kScanNT; off <<= 1) {
        int add = tid >= off ? sh[tid - off] : 0;
        __syncthreads();
        sh[tid] += add;
        __syncthreads();
    }
    total = sh[kScanNT - 1];
    int incl = sh[tid];
    __syncthreads();
    return incl - v;
}

static __global__ __launch_bounds__(kScanNT) void k_scan_reduce(const int *in, long n, int *bsum) {
    int *sh = reinterpret_cast<int *>(cuna_smem);
    long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanIPT;
    int s = 0;
#pragma unroll
    for (int q = 0; q < kScanIPT; ++q)
        if (base + q < n) s += in[base + q];
    int total;
    block_exclusive_scan(s, sh, total);
    if (threadIdx.x == 0) bsum[blockIdx.x] = total;
}

static __global__ __launch_bounds__(kScanNT) void k_scan_apply(const int *in, long n, const int *bsum,
                                                        int *out) {
    int *sh = reinterpret_cast<int *>(cuna_smem);
    long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanIPT;
    int v[kScanIPT];
    int s = 0;
#pragma unroll
    for (int q = 0; q < kScanIPT; ++q) {
        v[q] = base + q < n ? in[base + q] : 0;
        s += v[q];
    }
    // the earlier blocks' sums
    int before = 0, total;
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += kScanNT) before += bsum[b];
    block_exclusive_scan(before, sh, before);
    int ex = block_exclusive_scan(s, sh, total) + before;
#pragma unroll
    for (int q = 0; q < kScanIPT; ++q) {
        if (base + q < n) out[base + q] = ex;
        ex += v[q];
    }
}

// ----------------------------------------------------------- spread --
enum ValueMode { VAL_PLAIN = 0, VAL_COMPAT_BOOT = 1, VAL_COUNTS = 2 };

// One entry of a curve's spread work order: the tile, its three sorted
// point ranges [b, e) (empty where a neighbour is absent: non-periodic grid
// edges) and its cover.  Built once per plan with the tiles in decreasing
// order of their own point counts (ties by tile index), so that the densest
// tiles start first and the launch ends on light ones.
struct TileDesc {
    int tile, b0, e0, b1, e1, b2, e2, cover;
};
// scalar loads of one entry (merged into one 32-byte s_load)
__device__ __forceinline__ TileDesc ldc_desc(const TileDesc *p) {
    const int *q = reinterpret_cast<const int *>(p);
    TileDesc d;
    d.tile = ldc(q);
    d.b0 = ldc(q + 1);
    d.e0 = ldc(q + 2);
    d.b1 = ldc(q + 3);
    d.e1 = ldc(q + 4);
    d.b2 = ldc(q + 5);
    d.e2 = ldc(q + 6);
    d.cover = ldc(q + 7);
    return d;
}

template <typename T>
struct SpreadArgs {
    const PointRec<T> *rec;  // points sorted by anchor within each curve
    const int *perm;
    const int *bucket;
    const int *coff;       // curve point offsets (ncurves + 1)
    const T *y;            // values by original index, or null (unit weights)
    long y_slab_stride;    // added per replicate/slab for VAL_PLAIN with several rhs
    int npts;              // points of all curves (rec and perm hold max(npts, 1))
    T *grid;
    long grid_stride;      // per slab
    int G, tlog, ntiles, Kc, olo, ntaps, nrep;
    int slab0;  // slab (plan-time kernels: curve) of blockIdx.y = 0
    int periodic;
    int wrap1;  // periodic and a single tile covers the grid
    int cap;    // points staged in LDS per round (gather form)
    int gather; // FP32: use the gather form instead of the fixed-point scatter
    T bi;       // 1/beta
    T wscale;   // weight prefactor
    T e3[kMaxTaps];  // exp(-o^2/beta), o = olo + q
    // nullable: per curve (bi, wscale, exp(-bi)) in place of the three above,
    // for batches of compat curves whose filter widths differ
    const T *cpar;
    // per curve, ntiles work-order entries (the scatter kernel takes the next
    // entry of its curve per workgroup)
    const TileDesc *tile_desc;
    // VAL_COMPAT_BOOT (src/gridding.cu:86-117): value y[d] and weight
    // parameter eps_orig[d] of the drawn point d, position of point p
    uint32_t seed;
    const T *eps_orig;
    // VAL_COUNTS: value counts[rep][p] * y[p]
    const int *counts;
    long counts_stride;
};

// Tap q (0 <= q < NTAPS) sits at offset o = q - Q0 from the anchor,
// Q0 = (NTAPS-1)/2: compat (NTAPS = 2R_f - 1) has o in [-R_f+1, R_f-1]
// (src/gridding.cu:53-58), accurate (NTAPS = 2m) has o in [-m+1, m].
// Weights by the Greengard-Lee factorisation exp(-(o-e)^2/beta) =
// E1 * E2^o * E3[o]: three exponentials per point, one multiply per tap.
template <typename T, int NTAPS>
__device__ __forceinline__ void tap_weights(T v, T e, T bi, const T *e3, T *w) {
    constexpr int Q0 = (NTAPS - 1) / 2;
    const T E1 = dexp(-e * e * bi);
    const T E2 = dexp(T(2) * e * bi);
    const T E2i = dexp(T(-2) * e * bi);
    T up = v * E1;
#pragma unroll
    for (int q = Q0; q < NTAPS; ++q) {
        w[q] = up * e3[q];
        up *= E2;
    }
    T dn = v * E1 * E2i;
#pragma unroll
    for (int q = Q0 - 1; q >= 0; --q) {
        w[q] = dn * e3[q];
        dn *= E2i;
    }
}

// value and weight parameter of sorted point s (original index p)// value and weight parameter of sorted point s (original index p)
template <typename T, int VM>
__device__ __forceinline__ void point_value(const SpreadArgs<T> &A, int p, int c, int rep, T &v,
                                            T &e) {
    if constexpr (VM == VAL_PLAIN) {
        v = A.y ? A.y[p + rep * A.y_slab_stride] : T(1);
    } else if constexpr (VM == VAL_COMPAT_BOOT) {
        if (A.y) {
            const int c0 = A.coff[c];
            const uint32_t nc = (uint32_t)(A.coff[c + 1] - c0);
            const uint32_t t = (uint32_t)rep * nc + (uint32_t)(p - c0);
            const int d = c0 + (int)(xorshift32(wang_hash(A.seed + t)) % nc);
            v = A.y[d];
            e = A.eps_orig[d];
        } else {
            v = T(1);
        }
    } else {
        v = (T)A.counts[p + rep * A.counts_stride] * (A.y ? A.y[p] : T(1));
    }
}

template <typename T>
struct StagedPoint {
    int a;  // anchor relative to the tile's first cell
    T e, v;
};

// LDS bytes of one spread workgroup
template <typename T>
__host__ __device__ inline size_t spread_lds_bytes(int tlog, int ntaps, int cap) {
    size_t b = sizeof(T) * ((size_t)1 << tlog) + sizeof(int) * (((size_t)1 << tlog) + 2 * ntaps + 1);
    b = (b + 15) & ~(size_t)15;
    return b + sizeof(StagedPoint<T>) * (size_t)cap;
}

// The sorted points a tile's cells depend on, as up to three ranges with the
// offset that maps their anchors to this tile's cells, in increasing order of
// mapped anchor: the previous tile's right-edge class, this tile, the next
// tile's left-edge class.  A tiny periodic grid (taps wrap more than once)
// instead uses 2S+1 shifted copies of all its points.
struct TileRanges {
    int b0, n0, o0, b1, n1, b2, n2, o2, tstart, total, S, G;
    bool tiny;
    template <typename T>
    __device__ __forceinline__ void init(const SpreadArgs<T> &A, int tile, int c, int ntaps) {
        load(A, tile, c, ntaps);
        finish();
    }
    // issues the bucket loads (b* = first sorted index, n* = one past the
    // last until finish()); nothing here waits for them
    template <typename T>
    __device__ __forceinline__ void load(const SpreadArgs<T> &A, int tile, int c, int ntaps) {
        const int nt = A.ntiles;
        const int *bk = A.bucket + (long)c * (A.Kc + 1);
        const int TT = 1 << A.tlog;
        G = A.G;
        tstart = tile << A.tlog;
        tiny = A.wrap1 && A.G < 2 * ntaps;
        S = tiny ? (ntaps + A.G - 1) / A.G + 1 : 0;
        b0 = n0 = o0 = b2 = n2 = o2 = 0;
        b1 = ldc(bk + 3 * tile);
        n1 = ldc(bk + 3 * tile + 3);
        if (!tiny) {
            int prev = tile - 1, next = tile + 1;
            bool hp = true, hn = true;
            if (prev < 0) {
                prev = nt - 1;
                hp = A.periodic;
            }
            if (next >= nt) {
                next = 0;
                hn = A.periodic;
            }
            if (hp) {
                b0 = ldc(bk + 3 * prev + 2);
                n0 = ldc(bk + 3 * prev + 3);
                o0 = (prev << A.tlog) + TT;
            }
            if (hn) {
                b2 = ldc(bk + 3 * next);
                n2 = ldc(bk + 3 * next + 1);
                o2 = (next << A.tlog) - TT;
            }
        }
    }
    // the same ranges from a work-order entry (one scalar load of 32 bytes
    // in place of the bucket loads)
    template <typename T>
    __device__ __forceinline__ void from_desc(const SpreadArgs<T> &A, const TileDesc &d,
                                              int ntaps) {
        const int nt = A.ntiles;
        const int TT = 1 << A.tlog;
        G = A.G;
        tstart = d.tile << A.tlog;
        tiny = A.wrap1 && A.G < 2 * ntaps;
        S = tiny ? (ntaps + A.G - 1) / A.G + 1 : 0;
        b0 = d.b0;
        n0 = d.e0;
        b1 = d.b1;
        n1 = d.e1;
        b2 = d.b2;
        n2 = d.e2;
        const int prev = d.tile > 0 ? d.tile - 1 : nt - 1;
        const int next = d.tile + 1 < nt ? d.tile + 1 : 0;
        o0 = (prev << A.tlog) + TT;
        o2 = (next << A.tlog) - TT;
        finish();
    }
    // counts and total from the loaded bounds
    __device__ __forceinline__ void finish() {
        n0 -= b0;
        n1 -= b1;
        n2 -= b2;
        total = tiny ? n1 * (2 * S + 1) : n0 + n1 + n2;
    }
    // an interior tile: its three ranges are adjacent buckets (keys 3t-1 ..
    // 3t+3) and share the offset tstart, so point j is sorted index b0 + j
    __device__ __forceinline__ bool contiguous() const {
        return !tiny && b0 + n0 == b1 && b1 + n1 == b2 && o0 == tstart && o2 == tstart;
    }
    // j-th point of the tile: sorted index s and the offset ro (mapped anchor
    // = a - ro); selects rather than branches, so that loads indexed by it
    // stay in one basic block and issue together
    __device__ __forceinline__ void get(int j, int &s, int &ro) const {
        if (tiny) {  // uniform
            s = b1 + j % n1;
            ro = -(j / n1 - S) * G;
            return;
        }
        // (selects between computed values only: a select between two
        // fields would become a select of their addresses and keep this
        // struct out of registers)
        const bool in0 = j < n0, in1 = j < n0 + n1;
        const int s0 = b0 + j, s1 = b1 + (j - n0), s2 = b2 + (j - n0 - n1);
        s = in0 ? s0 : (in1 ? s1 : s2);
        ro = o2 + (in1 ? tstart - o2 : 0) + (in0 ? o0 - tstart : 0);
    }
};

// grid: blockIdx.x = tile, blockIdx.y = slab (curve * nrep + replicate).
// Output-driven: every cell of the tile is owned by one thread, which sums
// v_i exp(-(o_i - e_i)^2/beta) over the points i whose taps reach it (o_i =
// cell - anchor_i).  Points are sorted by anchor, so those are a contiguous
// window of the staged list; start[L] (first point with anchor >= L) is built
// in one pass over the points.  Deterministic: each cell sums in a fixed order.
template <typename T, int NTAPS, int VM>
__global__ __launch_bounds__(256) void k_spread(SpreadArgs<T> A) {
    constexpr int NT = 256, Q0 = (NTAPS - 1) / 2, QH = NTAPS - 1 - Q0;
    constexpr int LMIN = -NTAPS;
    const int TT = 1 << A.tlog;
    const int LMAX = TT + NTAPS + 1;  // start[] covers cells LMIN .. LMAX-1
    T *gacc = reinterpret_cast<T *>(cuna_smem);
    int *start = reinterpret_cast<int *>(gacc + TT);
    size_t off_pts = sizeof(T) * TT + sizeof(int) * (TT + 2 * NTAPS + 1);
    off_pts = (off_pts + 15) & ~(size_t)15;
    StagedPoint<T> *pts = reinterpret_cast<StagedPoint<T> *>(cuna_smem + off_pts);

    // consecutive tiles go to different XCDs (hardware round-robin): dense
    // regions of clustered points are spread over all of them
    const int tile = blockIdx.x;
    const int slab = A.slab0 + blockIdx.y;
    const int c = slab / A.nrep, rep = slab % A.nrep;
    TileRanges R;
    R.init(A, tile, c, NTAPS);
    const int tstart = R.tstart, total = R.total;
    const T bi = A.cpar ? A.cpar[3 * c] : A.bi;
    const T wscale = A.cpar ? A.cpar[3 * c + 1] : A.wscale;

    for (int g = threadIdx.x; g < TT; g += NT) gacc[g] = T(0);
    for (int base = 0; base < total; base += A.cap) {
        const int cnt = min(A.cap, total - base);
        __syncthreads();
        // stage this round's points: anchor in tile coordinates, e, value;
        // four per thread at a time with branch-free loads (slots past the
        // end read point 0 of the round and are not stored)
        for (int i0 = 0; i0 < cnt; i0 += 4 * NT) {
            int ak[4], pk[4];
            T ek[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = i0 + k * NT + threadIdx.x;
                int s, ro;
                R.get(base + (i < cnt ? i : 0), s, ro);
                const PointRec<T> pr = A.rec[s];
                ak[k] = pr.a - ro;
                ek[k] = pr.e;
                pk[k] = A.perm[s];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = i0 + k * NT + threadIdx.x;
                T v, e = ek[k];
                point_value<T, VM>(A, pk[k], c, rep, v, e);
                if (i < cnt) {
                    StagedPoint<T> sp;
                    sp.a = ak[k];
                    sp.e = e;
                    sp.v = v;
                    pts[i] = sp;
                }
            }
        }
        for (int L = threadIdx.x; L < LMAX - LMIN; L += NT) start[L] = cnt;
        __syncthreads();
        // start[L - LMIN] = first staged point with anchor >= L
        for (int i = threadIdx.x; i < cnt; i += NT) {
            const int hi = min(pts[i].a, LMAX - 1);
            const int lo = i == 0 ? LMIN : max(pts[i - 1].a + 1, LMIN);
            for (int L = lo; L <= hi; ++L) start[L - LMIN] = i;
        }
        __syncthreads();
        for (int g = threadIdx.x; g < TT; g += NT) {
            const int lo = start[g - QH - LMIN];
            const int hi = start[g + Q0 + 1 - LMIN];
            T sum = T(0);
            for (int i = lo; i < hi; ++i) {
                const StagedPoint<T> sp = pts[i];
                const T d = (T)(g - sp.a) - sp.e;
                sum += sp.v * dexp(-d * d * bi);
            }
            gacc[g] += sum;
        }
    }
    __syncthreads();
    T *gout = A.grid + (long)slab * A.grid_stride + tstart;
    const int tlen = min(TT, A.G - tstart);
    for (int g = threadIdx.x; g < tlen; g += NT) gout[g] = gacc[g] * wscale;
}

// ---------------------------------------------- fixed-point scatter --
// Scatter form (both libraries): a thread takes a point, forms its NTAPS
// weights with three exponentials, and adds them to the tile's LDS cells
// with integer atomics in fixed point (32-bit cells in FP32, 64-bit in
// FP64).  Integer sums do not depend on the order of the additions, so the
// result is bitwise reproducible; float LDS atomics would be neither
// reproducible nor fast on this hardware, and double LDS atomics are
// compare-and-swap loops.  A round of up to CAP points uses the scale 2^s
// with min(cnt, cover) * wmax * 2^s <= 2^headroom (cover: the most points of
// the tile in one window of ntaps anchors), wmax the largest weight the round adds
// to the tile's own cells (bounded by max|v| * wscale for accurate filters),
// so none of them can overflow (halo cells, which are not written out, may).
// Split of a scaled weight x (|x| < 2^62) into a two's-complement 64-bit
// integer: h = floor(x / 2^32) and l = x - h 2^32 in [0, 2^32).  In float,
// exact for x >= 0; for -2^31 < x < 0, l is rounded to a multiple of 2^8,
// an error far below the float weight's own rounding.  In double, l is exact
// and rounded to the nearest integer (at most 2^32 - 1, so a tiny negative x
// gives -1, one unit of the scale).
__device__ __forceinline__ unsigned long long to_fixed64(float x) {
    const float h = floorf(x * 0x1p-32f);
    const float l = fminf(fmaf(h, -0x1p32f, x), 4294967040.0f);
    return ((unsigned long long)(unsigned)(int)h << 32) | (unsigned)l;
}
__device__ __forceinline__ unsigned long long to_fixed64(double x) {
    const double h = floor(x * 0x1p-32);
    const double l = fmin(rint(fma(h, -0x1p32, x)), 4294967295.0);
    return ((unsigned long long)(unsigned)(int)h << 32) | (unsigned)l;
}

// Work order of the scatter kernels, one workgroup per curve: the curve's
// tiles by decreasing own point count, as a stable counting sort over
// kOrderBins bins of the count (exact below 128 points, in steps of 8 up to
// 1143, one bin above), ties in tile order; position i's TileDesc gets its
// tile, and k_tile_desc fills in the rest.
// The order only schedules the tiles: every tile's cells come out the same
// in any order.  Each of the 16 waves ranks a contiguous segment of tiles.
constexpr int kOrderThreads = 1024, kOrderWaves = kOrderThreads / 64, kOrderBins = 256;
constexpr int kOrderMaxTiles = 8192;
static_assert(kOrderThreads == kScanNT, "the work order scans with one value per thread");

__device__ __forceinline__ int order_bin(int npts) {
    const int r = npts < 128 ? npts : 128 + min(127, (npts - 128) >> 3);
    return kOrderBins - 1 - r;  // bin 0: the densest tiles
}

static __global__ __launch_bounds__(kOrderThreads) void k_tile_order(const int *bucket, int Kc,
                                                                     int ntiles, TileDesc *desc) {
    __shared__ int cnt[kOrderBins * kOrderWaves];  // [bin][wave]: counts, then starts
    __shared__ int scan_sh[kOrderThreads];
    __shared__ unsigned char bin_sh[kOrderMaxTiles];
    __shared__ short order[kOrderMaxTiles];
    const int c = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int *bk = bucket + (long)c * (Kc + 1);
    for (int i = tid; i < kOrderBins * kOrderWaves; i += kOrderThreads) cnt[i] = 0;
    // every thread's loads first (clamped to in-bounds tiles), then their
    // uses, so that the loads are in flight together
    constexpr int TPT = kOrderMaxTiles / kOrderThreads;
    int lo[TPT], hi[TPT];
#pragma unroll
    for (int r = 0; r < TPT; ++r) {
        const int tc = min(r * kOrderThreads + tid, ntiles - 1);
        lo[r] = bk[3 * tc];
        hi[r] = bk[3 * tc + 3];
    }
#pragma unroll
    for (int r = 0; r < TPT; ++r) {
        const int t = r * kOrderThreads + tid;
        if (t < ntiles) bin_sh[t] = (unsigned char)order_bin(hi[r] - lo[r]);
    }
    __syncthreads();
    const int seg = (ntiles + kOrderWaves - 1) / kOrderWaves;
    const int s0 = min(ntiles, wave * seg), s1 = min(ntiles, s0 + seg);
    for (int t = s0 + lane; t < s1; t += 64) atomicAdd(&cnt[bin_sh[t] * kOrderWaves + wave], 1);
    __syncthreads();
    // exclusive scan in (bin, wave) order: a wave's tiles of one bin follow
    // the earlier waves' tiles of that bin
    constexpr int IPT = kOrderBins * kOrderWaves / kOrderThreads;
    int v[IPT], sum = 0;
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
        v[q] = cnt[IPT * tid + q];
        sum += v[q];
    }
    int total;
    int ex = block_exclusive_scan(sum, scan_sh, total);
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
        cnt[IPT * tid + q] = ex;
        ex += v[q];
    }
    __syncthreads();
    // rank within the wave's 64 tiles of a step: lanes with the same bin
    const unsigned long long lt = (1ull << lane) - 1ull;
    for (int t0 = s0; t0 < s1; t0 += 64) {
        const int t = t0 + lane;
        const bool act = t < s1;
        const int b = act ? bin_sh[t] : 0;
        unsigned long long peers = __ballot(act);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const unsigned long long m = __ballot((b >> bit) & 1);
            peers &= ((b >> bit) & 1) ? m : ~m;
        }
        const int rank = __popcll(peers & lt);
        int pos = 0;
        if (act) pos = cnt[b * kOrderWaves + wave] + rank;
        __builtin_amdgcn_wave_barrier();
        if (act) {
            order[pos] = (short)t;
            if (rank == __popcll(peers) - 1) cnt[b * kOrderWaves + wave] = pos + 1;
        }
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    for (int i = tid; i < ntiles; i += kOrderThreads) desc[(long)c * ntiles + i].tile = order[i];
}

// The rest of each TileDesc, one wave per work-order position: the tile's own
// range, its neighbours' edge classes (prev = t - 1 and next = t + 1, wrapping
// when periodic) and its cover, the most of these points whose anchors fall in
// one window of ntaps consecutive anchors that reaches a cell of the tile.  The
// wave counts the anchors in LDS, turns the counts into prefix sums (lane l
// scans a contiguous piece) and takes each cell's window as a difference of
// two.  One 256-thread workgroup per tile adding ntaps counts per cell took
// 33 us at 32,768 tiles of 39 points; this takes 17.5 us.
constexpr int kDescWaves = 4;

template <typename T>
__global__ __launch_bounds__(64 * kDescWaves) void k_tile_desc(SpreadArgs<T> A, long pos0,
                                                               long npos, TileDesc *desc) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int TT = 1 << A.tlog, nt = A.ntaps, Q0 = (nt - 1) / 2, NH = TT + 2 * nt;
    int *h = reinterpret_cast<int *>(cuna_smem) + wave * (NH + 1);  // cells -nt .. TT+nt-1
    const long pos = pos0 + (long)blockIdx.x * kDescWaves + wave;  // pos0 <= pos < npos
    if (pos >= npos) return;  // no workgroup barriers below
    const int c = (int)(pos / A.ntiles);
    const int tile = desc[pos].tile;
    TileRanges R;
    R.init(A, tile, c, nt);
    for (int i = lane; i <= NH; i += 64) h[i] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int j = lane; j < R.total; j += 64) {
        int s, ro;
        R.get(j, s, ro);
        const int a = A.rec[s].a - ro + nt;
        if (a >= 0 && a < NH) atomicAdd(&h[a], 1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // h[i] := points with anchors before cell i, i = 0 .. NH
    const int per = (NH + 64) / 64, i0 = min(lane * per, NH + 1), i1 = min(i0 + per, NH + 1);
    int sum = 0;
    for (int i = i0; i < i1; ++i) sum += h[i];
    int incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(incl, o);
        if (lane >= o) incl += u;
    }
    int run = incl - sum;
    for (int i = i0; i < i1; ++i) {
        const int v = h[i];
        h[i] = run;
        run += v;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // cell g takes the points with anchors g - (nt - 1 - Q0) .. g + Q0
    int best = 0;
    for (int g = lane; g < TT; g += 64) {
        const int lo = g + Q0 + 1;  // = g - (nt - 1 - Q0) + nt
        best = max(best, h[lo + nt] - h[lo]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) best = max(best, __shfl_xor(best, o));
    if (lane == 0) {
        TileDesc d;
        d.tile = tile;
        d.b0 = R.b0;
        d.e0 = R.b0 + R.n0;
        d.b1 = R.b1;
        d.e1 = R.b1 + R.n1;
        d.b2 = R.b2;
        d.e2 = R.b2 + R.n2;
        d.cover = best;
        desc[pos] = d;
    }
}

// Accumulators of the scatter: 32-bit cells (ds_add_u32) hold sums within
// 2^30, 64-bit cells (FP64 library) within 2^62.  In FP64 each weight is also
// kept within 2^`single` = 2^50 (a second bound on the scale) and rounded to
// the nearest integer by adding 1.5 * 2^52: for |x| < 2^51 the sum lies in
// [2^52, 2^53), whose spacing is 1, so its low mantissa bits are round(x) and
//   round(x) = bits(x + 1.5 * 2^52) - bits(1.5 * 2^52)
// as 64-bit integers (one add, or one fma with the weight's product, and one
// 64-bit subtract per tap).
template <typename T>
struct Fixed64 {
    using U = unsigned long long;
    static constexpr int headroom = 62;
    static constexpr int single = sizeof(T) == 8 ? 50 : 0;  // 0: no per-weight bound
    static constexpr double kMagic = 0x1.8p52;
    static constexpr U kMagicBits = 0x4338000000000000ull;
    __device__ static U fixed(T x) {
        if constexpr (sizeof(T) == 8)
            return (U)__double_as_longlong(x + kMagic) - kMagicBits;
        else
            return to_fixed64(x);
    }
    // round(a * b), FP64 only
    __device__ static U fixed_fma(double a, double b) {
        return (U)__double_as_longlong(fma(a, b, kMagic)) - kMagicBits;
    }
};
struct Fixed32 {
    using U = unsigned;
    static constexpr int headroom = 30;
    static constexpr int single = 0;
    __device__ static U fixed(float x) { return (U)__float2int_rn(x); }
};

// The NTAPS fixed-point weights of one point, rounded to nearest:
// n_q = round(v exp(-(q - Q0 - e)^2 bi)), v already carrying the scale, each
// handed to emit(q, n_q) as soon as it is formed (outward from the anchor),
// so that no array of NTAPS values stays live.  In FP32 with the table e3
// (accurate filters), each tap is one multiply (the step E2^{+-1}), one fma
// that also adds the rounding half (with the sign of v: all taps of a point
// share it) and one truncating conversion; FP64 rounds by FX::fixed_fma.
// Otherwise (compat filters) the weights come by ratio recurrences, which
// need only c1 = exp(-bi), and FX::fixed per tap.
template <typename T, int NTAPS, class FX, bool TABLE, class Emit>
__device__ __forceinline__ void tap_fixed(T v, T e, T bi, const T *e3, T c1, Emit &&emit) {
    constexpr int Q0 = (NTAPS - 1) / 2;
    if constexpr (TABLE && sizeof(T) == 4 && std::is_same<FX, Fixed32>::value) {
        const float E1 = dexp(-e * e * bi);
        const float E2 = dexp(2.0f * e * bi);
        const float E2i = dexp(-2.0f * e * bi);
        const float h = copysignf(0.5f, v);
        float up = v * E1;
#pragma unroll
        for (int q = Q0; q < NTAPS; ++q) {
            emit(q, (unsigned)(int)fmaf(up, e3[q], h));
            up *= E2;
        }
        float dn = v * E1 * E2i;
#pragma unroll
        for (int q = Q0 - 1; q >= 0; --q) {
            emit(q, (unsigned)(int)fmaf(dn, e3[q], h));
            dn *= E2i;
        }
    } else if constexpr (TABLE && sizeof(T) == 8 && std::is_same<FX, Fixed64<T>>::value) {
        const double E1 = dexp(-e * e * bi);
        const double E2 = dexp(2.0 * e * bi);
        const double E2i = dexp(-2.0 * e * bi);
        double up = v * E1;
#pragma unroll
        for (int q = Q0; q < NTAPS; ++q) {
            emit(q, FX::fixed_fma(up, e3[q]));
            up *= E2;
        }
        double dn = v * E1 * E2i;
#pragma unroll
        for (int q = Q0 - 1; q >= 0; --q) {
            emit(q, FX::fixed_fma(dn, e3[q]));
            dn *= E2i;
        }
    } else if constexpr (TABLE) {
        T w[NTAPS];
        tap_weights<T, NTAPS>(v, e, bi, e3, w);
#pragma unroll
        for (int q = 0; q < NTAPS; ++q) emit(q, FX::fixed(w[q]));
    } else {
        // two ratio recurrences, which need exp(-bi) instead of the table:
        // with w_o = v exp(-(o-e)^2 bi), w_{o+1} = w_o R_o, R_0 = E2 exp(-bi),
        // R_{o+1} = R_o exp(-2 bi); downwards w_{o-1} = w_o L_o with
        // L_0 = exp(-bi)/E2, L_{o-1} = L_o exp(-2 bi)
        const T D = c1 * c1;
        const T E1 = dexp(-e * e * bi);
        const T E2 = dexp(T(2) * e * bi);
        const T E2i = dexp(T(-2) * e * bi);
        const T w0 = v * E1;
        T up = w0, r = E2 * c1;
#pragma unroll
        for (int q = Q0; q < NTAPS; ++q) {
            emit(q, FX::fixed(up));
            up *= r;
            r *= D;
        }
        T dn = w0, l = E2i * c1;
#pragma unroll
        for (int q = Q0 - 1; q >= 0; --q) {
            dn *= l;
            l *= D;
            emit(q, FX::fixed(dn));
        }
    }
}


// ------------------------------------------- per-wave fixed-point scatter --
// Each wave of the tile's workgroup accumulates its own share of the points
// into its own LDS cells, in fixed point with integer atomics (32-bit cells
// in FP32, 64-bit in FP64), with its own power-of-two scale:
//   min(cover * vmax, vsum) * wscale * 2^s <= 2^headroom,
// vmax and vsum = the largest and the sum of the |values| of the wave's points this
// round (at most 64 * kSpreadSlots; compat filters: of the largest kept weights /
// wscale; FP64 takes their number times vmax for vsum), cover = the tile's most
// points in one window of ntaps anchors.  No cell can overflow,
// whatever the density, so no wider fallback and no plan-time read-back is
// needed; a wave's scale needs no workgroup barrier; and the waves never
// contend for one address.  After the last round the waves' cells are
// converted and summed in a fixed wave order, so the grid is bitwise
// reproducible.  Resolution: 2^-headroom * min(cover, vsum / vmax) of the round's
// largest weight (FP32: 2^-24 for cover <= 64, 2^-22 at worst, and 2^-29 next to one
// value that dominates, whose rounding the other points of its tile share: with
// cover alone, spectra in tiles of 1024 cells were up to 1.26 times as far off as in
// tiles of 256, log-normal values, now 1.02 times).  A wave with
// several rounds folds each into its own float (double) cells.
constexpr int kSpreadSlots = 4;  // point slots per lane in a round

template <typename T>
using SpreadFixed = std::conditional_t<sizeof(T) == 4, Fixed32, Fixed64<T>>;

template <typename T>
__host__ __device__ inline size_t spread_wv_lds_bytes(int tlog, int ntaps, int waves) {
    const size_t tt = (size_t)1 << tlog;
    const size_t acc = sizeof(typename SpreadFixed<T>::U) * (tt + 2 * (size_t)ntaps);
    return (size_t)waves * (acc + sizeof(T) * tt);
}

template <typename T, int NTAPS, int VM, int WPT>
__global__ __launch_bounds__(64 * WPT) void k_spread_wv(SpreadArgs<T> A) {
    using FX = SpreadFixed<T>;
    using Acc = typename FX::U;
    using SAcc = std::make_signed_t<Acc>;
    constexpr int NT = 64 * WPT, PPT = kSpreadSlots, CAP = NT * PPT;
    constexpr int Q0 = (NTAPS - 1) / 2, HALO = NTAPS;
    constexpr T kBig = sizeof(T) == 4 ? T(3.0e38f) : T(1.0e300);
    constexpr int kMaxExp = sizeof(T) == 4 ? 100 : 1000;
    __shared__ int sexp_sh[WPT];
    __shared__ int fin_sh[WPT];
    const int TT = 1 << A.tlog;
    const int NC = TT + 2 * HALO;  // cells -HALO .. TT+HALO-1
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    Acc *acc_all = reinterpret_cast<Acc *>(cuna_smem);
    T *facc_all = reinterpret_cast<T *>(acc_all + WPT * NC);
    Acc *acc = acc_all + wave * NC;
    T *facc = facc_all + wave * TT;

    // (entry of the work order, slab); a few slabs keep the order as it is
    const int2 bs = gridDim.y < kNumXcd ? make_int2(blockIdx.x, blockIdx.y)
                                        : xcd_block(blockIdx.x, blockIdx.y, gridDim.x, gridDim.y);
    const int slab = A.slab0 + bs.y;
    const int c = slab / A.nrep, rep = slab % A.nrep;
    TileRanges R;
    const TileDesc desc = ldc_desc(A.tile_desc + (long)c * A.ntiles + bs.x);
    R.from_desc(A, desc, NTAPS);
    const int cover = desc.cover;
    const int total = R.total;
    const bool multi = total > CAP;
    const T c1 = A.cpar ? A.cpar[3 * c + 2] : A.e3[Q0 + 1];  // exp(-bi)
    const T bi = A.cpar ? A.cpar[3 * c] : A.bi;
    const T wscale = A.cpar ? A.cpar[3 * c + 1] : A.wscale;
    const int tlen = min(TT, A.G - R.tstart);  // cells of the tile inside the grid
    int ew = 0;
    (void)frexp(wscale, &ew);

    for (int g = lane; g < NC; g += 64) acc[g] = Acc(0);
    if (multi)
        for (int g = lane; g < TT; g += 64) facc[g] = T(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // the wave's clears land before its atomics
    __builtin_amdgcn_wave_barrier();
    bool finite = true;
    int sexp = 0;
    const bool contig = R.contiguous();  // uniform
    for (int base = 0; base < total; base += CAP) {
        const int cnt = min(CAP, total - base);
        // thread t takes the round's points t*spl .. t*spl + spl-1, spl the
        // fewest slots that hold cnt points: a wave's lanes then sit on
        // points spread over the whole tile, so one atomic instruction seldom
        // puts two lanes on one cell (the points are sorted by anchor), and
        // slots past spl are empty for every lane.  Branch-free loads (all
        // slots issue together); a slot past the end reads point 0.
        const int spl = (cnt + NT - 1) / NT;  // uniform
        auto slot = [&](int k) { return k < spl ? tid * spl + k : CAP; };
        int am[PPT], pk[PPT], sk[PPT], rk[PPT];
        T ev[PPT], vv[PPT];
        // this wave's points in the round
        const int wcnt = max(0, min(64 * spl, cnt - wave * 64 * spl));
        // the original indices first, then the records: the values gathered
        // through perm below wait only for perm (loads return in order), and
        // their loads overlap the records'
#pragma unroll
        for (int k = 0; k < PPT; ++k) {
            const int i = slot(k);
            const int j = base + (i < cnt ? i : 0);
            if (contig) {
                sk[k] = R.b0 + j;
                rk[k] = R.tstart;
            } else {
                R.get(j, sk[k], rk[k]);
            }
            pk[k] = A.perm[sk[k]];
        }
#pragma unroll
        for (int k = 0; k < PPT; ++k) {
            const PointRec<T> pr = A.rec[sk[k]];
            am[k] = pr.a - rk[k];
            ev[k] = pr.e;
        }
        T vmax = T(0), vsum = T(0);
#pragma unroll
        for (int k = 0; k < PPT; ++k) {
            T v, e = ev[k];
            point_value<T, VM>(A, pk[k], c, rep, v, e);
            const bool ok = slot(k) < cnt;
            vv[k] = ok ? v : T(0);
            ev[k] = e;
            T av = fabs(vv[k]);
            if constexpr (NTAPS % 2 == 1) {
                // compat filter: e lies up to R_f + 1 cells from the taps and
                // taps off the grid are dropped, so the largest weight this
                // tile keeps, at its tap o nearest e, can be far below |v|
                const int lo = max(-Q0, -am[k]), hi = min(NTAPS - 1 - Q0, tlen - 1 - am[k]);
                const T o = fmin(fmax(rint(e), T(lo)), T(hi));
                av = lo <= hi ? av * dexp(-(o - e) * (o - e) * bi) : T(0);
            }
            // a non-finite value or position (NaN x gives NaN e) makes the
            // tile's output NaN
            if (!(av <= kBig) || (ok && !(fabs(e) <= kBig))) av = T(INFINITY);
            vmax = fmax(vmax, av);
            vsum += av;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            vmax = fmax(vmax, __shfl_xor(vmax, o));
            if constexpr (sizeof(T) == 4) vsum += __shfl_xor(vsum, o);
        }
        if (!(vmax <= kBig)) finite = false;
        // (FP64: the bound on single weights decides)
        const T bound =
            (sizeof(T) == 4 ? fmin((T)cover * vmax, vsum) : (T)min(wcnt, cover) * vmax) * wscale;
        int eb = -64;
        if (bound > T(0) && finite) (void)frexp(bound, &eb);
        sexp = min(FX::headroom - eb, kMaxExp - ew);
        if constexpr (FX::single > 0) {
            int e1 = -64;
            const T b1 = vmax * wscale;
            if (b1 > T(0) && finite) (void)frexp(b1, &e1);
            sexp = min(sexp, FX::single - e1);
        }
        const T mul = ldexp(wscale, sexp);
        if (finite) {
#pragma unroll
            for (int k = 0; k < PPT; ++k) {
                if (slot(k) < cnt) {
                    // accurate filters (even NTAPS) share one table e3; compat
                    // batches carry a filter per curve (cpar), so recurrences
                    const int c0 = am[k] - Q0;  // first tap's cell
                    Acc *dst = acc + HALO + c0;
                    if (R.tiny) {
                        tap_fixed<T, NTAPS, FX, NTAPS % 2 == 0>(
                            vv[k] * mul, ev[k], bi, A.e3, c1, [&](int q, Acc n) {
                                const int cell = c0 + q;
                                if (cell >= -HALO && cell < TT + HALO) atomicAdd(dst + q, n);
                            });
                    } else {
                        tap_fixed<T, NTAPS, FX, NTAPS % 2 == 0>(
                            vv[k] * mul, ev[k], bi, A.e3, c1,
                            [&](int q, Acc n) { atomicAdd(dst + q, n); });
                    }
                }
            }
        }
        if (multi) {
            // fold the round into this wave's float cells; the wave's own
            // atomics must have landed first (LDS counter drained)
            __builtin_amdgcn_s_waitcnt(0xc07f);
            __builtin_amdgcn_wave_barrier();
            const T inv = ldexp(T(1), -sexp);
            for (int g = lane; g < TT; g += 64) {
                facc[g] += (T)(SAcc)acc[HALO + g] * inv;
                acc[HALO + g] = Acc(0);
            }
            for (int h = lane; h < 2 * HALO; h += 64) acc[h < HALO ? h : TT + h] = Acc(0);
            __builtin_amdgcn_s_waitcnt(0xc07f);
            __builtin_amdgcn_wave_barrier();
        }
    }
    if (lane == 0) {
        sexp_sh[wave] = sexp;
        fin_sh[wave] = finite ? 1 : 0;
    }
    // every wave's cells and scale are read below by all threads
    __syncthreads();
    bool all_finite = true;
    T inv[WPT];
#pragma unroll
    for (int w = 0; w < WPT; ++w) {
        all_finite = all_finite && fin_sh[w] != 0;
        inv[w] = ldexp(T(1), -sexp_sh[w]);
    }
    T *gout = A.grid + (long)slab * A.grid_stride + R.tstart;
    for (int g = tid; g < tlen; g += NT) {
        T v = T(0);
#pragma unroll
        for (int w = 0; w < WPT; ++w)
            v += multi ? facc_all[w * TT + g] : (T)(SAcc)acc_all[w * NC + HALO + g] * inv[w];
        gout[g] = all_finite ? v : T(NAN);
    }
}

// ------------------------------------------- fused batched bootstrap --
// One persistent workgroup per CU drains a queue of (curve, replicate) items.
// An item draws the replicate's points
// d = c0 + xorshift(wang(seed + rep*n_c + p)) % n_c, p < n_c, spreads them
// into a grid of G = 2N cells held entirely in LDS, transforms it in place
// (real input as N complex) and writes the deconvolved spectrum:
// transform 0 is y at the points x_d, transform 1 the unit-weight window at 2 x_d.
//
// LDS float atomics are slow on this hardware, so the grid accumulates in
// fixed point with integer atomics (int32 in the FP32 library, int64 in FP64),
// which are also order-independent.  The power-of-two scale comes from the
// curve's max |y| and its densest tap window; the draws' own density is counted on
// the way, and an item denser than the scale allows is redone.  The integer grid
// occupies the same LDS words as the complex buffer of the FFT, whose first pass
// reads and converts it.
//
// What an item needs of its curve, one entry per curve in queue order.
struct BootCurve {
    int ci, c0, nc;       // curve, its first point, its points
    uint32_t fm_m;        // FastMod of max(nc, 1)
    int fm_s1, fm_s2;
    int cover_x, cover_2x;  // most points within one tap window
    double ymax;          // max |y|, NaN values ignored (1 without y)
};
constexpr int kBootCurveWords = sizeof(BootCurve) / 4;
static_assert(sizeof(BootCurve) == 40, "BootCurve is copied word by word");

template <typename T>
struct BootArgs {
    const PointRec<T> *rec_x;   // (anchor, frac) of x by original index
    const PointRec<T> *rec_2x;  // of 2x (window), nullable
    const T *y;                 // nullable: unit weights
    const BootCurve *curves;    // longest first
    int *counter;               // work-queue head, zeroed before the launch
    cplx<T> *out_y, *out_w;
    int ncurves, nbs, ntr, total;
    int split;                  // MODE 0: a replicate's transforms are items of their own
    unsigned *list;             // one row of list_cap words per workgroup
    int list_cap;
    uint32_t seed;
    T bi, wscale;
    T e3[kMaxTaps];
    SinkAccurate<T> sink;       // out pointer set per item
    const cplx<T> *twT;         // twiddle rows up to boot_cap (staged into LDS)
    Tw2<T> twN;                 // w_N^e, e < N (two-level, staged into LDS)
    const cplx<T> *twH;         // w_G^e, e < workgroup size
    // Lomb-Scargle mode (each nullable): per replicate, power at k = 0..M/2-1,
    // and its maximum over k >= 1 with the k where it occurs
    T *ls_power;
    T *ls_peak;
    int *ls_kpeak;
    // ... and a workspace of a row of M/2 values per workgroup, which keeps its
    // current window spectrum in row blockIdx.x
    cplx<T> *ls_w;
    int slots;  // rows of list and ls_w
};

// LDS of the fused kernel: the grid (G reals = N complex) between two halos of
// kBootHalo cells, the twiddle rows of the passes of at most 2^cap points, and the
// two sub-tables of w_N for the later ones.
constexpr int kBootHalo = 32;
// cap: 18 KB of rows at FP32's largest grid, where one workgroup has a CU to
// itself; a few KB where two share it
template <typename T>
__host__ __device__ constexpr int boot_cap(int lg) {
    return sizeof(T) == 4 && lg == 14 ? 11 : lg < 10 ? lg : 10;
}
template <typename T>
__host__ __device__ constexpr int boot_tw_entries(int lg) {
    return rows_count(lg, small_mr(lg), boot_cap<T>(lg)) + (1 << ((lg + 1) / 2)) +
           (1 << (lg - (lg + 1) / 2));
}
template <typename T>
__host__ __device__ constexpr size_t boot_lds_bytes(int lg) {
    return sizeof(cplx<T>) * (((size_t)1 << lg) + (size_t)boot_tw_entries<T>(lg)) +
           2 * kBootHalo * sizeof(T);
}

// the longest curve whose draws are merged: 16-bit counters in the grid's space,
// 16-bit point indices
template <typename T>
__host__ __device__ constexpr int boot_list_max(int lg) {
    const long fit = (2L << lg) * (long)sizeof(T) / 2;
    return fit < 65535 ? (int)fit : 65535;
}

// cos and sin of 2 pi i / n for the epilogue's constant rotations (compile time
// from a table of 2 pi / 32 multiples, n <= 32 a power of two)
template <typename T>
__device__ __forceinline__ constexpr cplx<T> unit_root_32(int i) {
    constexpr double c[9] = {1.0,
                             0.98078528040323044913,
                             0.92387953251128675613,
                             0.83146961230254523708,
                             0.70710678118654752440,
                             0.55557023301960222474,
                             0.38268343236508977173,
                             0.19509032201612826785,
                             0.0};
    return i <= 8 ? cplx<T>{(T)c[i], (T)c[8 - i]} : cplx<T>{(T)-c[16 - i], (T)c[i - 8]};
}

template <typename I>
struct alignas(2 * sizeof(I)) FixedPair {
    I x, y;
};

template <typename T>
struct FixedOf;
template <>
struct FixedOf<float> {
    using I = int;
    static constexpr int headroom_bits = 30;
    __device__ static I round(float v) { return __float2int_rn(v); }
};
template <>
struct FixedOf<double> {
    using I = long long;
    static constexpr int headroom_bits = 61;
    __device__ static I round(double v) { return __double2ll_rn(v); }
};

// Spectrum value 2 A[r] of the real grid from the pair (Z[r], Z[N-r]) of its
// complex transform (the first of the two values emit_pair produces).
template <typename T>
__device__ __forceinline__ cplx<T> real_spectrum_at(cplx<T> Zr, cplx<T> Znr, cplx<T> wr) {
    cplx<T> c = conjg(Znr);
    cplx<T> E = Zr + c;
    cplx<T> D = Zr - c;
    return E + wr * cmk(D.y, -D.x);
}

// Lomb-Scargle power (Press & Rybicki 1989, "standard" normalisation, data
// centred) from F = sum (y_i - ybar) e^{i w t_i} and W = sum e^{2 i w t_i}
// over n points with yy = sum (y_i - ybar)^2:
//   tan 2wtau = Im W / Re W,  YC = Re F cos wtau + Im F sin wtau,
//   YS = Im F cos wtau - Re F sin wtau,  CC = (n + |W|)/2,  SS = (n - |W|)/2,
//   P = (YC^2/CC + YS^2/SS) / yy   (a term whose denominator vanishes is 0).
// Reciprocals: the FP32 library uses the hardware's (v_rcp_f32, v_rsq_f32,
// about 1 ulp; the periodogram's error budget is far larger), FP64 divides.
__device__ __forceinline__ float ls_rcp(float v) { return __builtin_amdgcn_rcpf(v); }
__device__ __forceinline__ double ls_rcp(double v) { return 1.0 / v; }
__device__ __forceinline__ float ls_rsqrt(float v) { return __builtin_amdgcn_rsqf(v); }
__device__ __forceinline__ double ls_rsqrt(double v) { return 1.0 / sqrt(v); }

template <typename T>
__device__ __forceinline__ T ls_power(cplx<T> F, cplx<T> W, T n, T yy) {
    const T h2 = W.x * W.x + W.y * W.y;
    const T ih = h2 > T(0) ? ls_rsqrt(h2) : T(0);
    const T h = h2 * ih;
    const T c2 = h2 > T(0) ? W.x * ih : T(1), s2 = h2 > T(0) ? W.y * ih : T(0);
    const T cw = sqrt(fmax(T(0), (T(1) + c2) * T(0.5)));
    const T sw = copysign(sqrt(fmax(T(0), (T(1) - c2) * T(0.5))), s2);
    const T yc = F.x * cw + F.y * sw, ys = F.y * cw - F.x * sw;
    const T cc = (n + h) * T(0.5), ss = (n - h) * T(0.5);
    const T tiny = n * T(sizeof(T) == 4 ? 1e-6 : 1e-14);
    T p = (cc > tiny ? yc * yc * ls_rcp(cc) : T(0)) + (ss > tiny ? ys * ys * ls_rcp(ss) : T(0));
    return yy > T(0) ? p * ls_rcp(yy) : T(0);
}

// A value every thread of the workgroup holds equally, moved to scalar
// registers (it then takes no vector registers across the transforms).
__device__ __forceinline__ double uniform_f64(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readfirstlane((int)b);
    const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// MODE 0: items (curve, replicate) -> the deconvolved spectra of its transforms
// (or one of them, with A.split: few items would leave CUs idle).
// MODE 1: items (curve, replicate) -> Lomb-Scargle power of the replicate:
// the window transform (unit weights at 2x) goes to the workgroup's row of
// the workspace (each thread writes, and later reads back, its own
// frequencies), then the transform of the mean-subtracted values at x gives
// the power directly; nothing else is written.
template <typename T, int LG, int NTAPS, int NT, int MODE>
__global__ __launch_bounds__(NT) void k_boot_fused(BootArgs<T> A) {
    using I = typename FixedOf<T>::I;
    using U = std::make_unsigned_t<I>;
    static_assert(sizeof(I) == sizeof(T), "fixed-point grid aliases the real grid");
    constexpr int N = 1 << LG, G = 2 * N, Q0 = (NTAPS - 1) / 2;
    constexpr int LBN = (LG + 1) / 2;  // as TwiddleCache::two_level
    constexpr int NLN = 1 << LBN, NHN = 1 << (LG - LBN);
    constexpr int PB = 4;  // resampled points per thread whose loads are in flight together
    constexpr int kMaxExp = sizeof(T) == 4 ? 100 : 1000;
    // the grid's cell 0; kBootHalo cells before it and after cell G - 1 take the
    // taps that wrap, so that a tap's cell needs no reduction mod G
    T *grid = reinterpret_cast<T *>(cuna_smem) + kBootHalo;
    U *gu = reinterpret_cast<U *>(grid);
    cplx<T> *z = reinterpret_cast<cplx<T> *>(grid);
    cplx<T> *tl = reinterpret_cast<cplx<T> *>(grid + G + kBootHalo);  // staged once per workgroup
    constexpr int MR = small_mr(LG), CAP = boot_cap<T>(LG), NLT = rows_count(LG, MR, CAP);
    const int tid = threadIdx.x;
    for (int i = tid; i < NLT; i += NT) tl[i] = A.twT[i];
    for (int i = tid; i < NLN; i += NT) tl[NLT + i] = A.twN.lo[i];
    for (int i = tid; i < NHN; i += NT) tl[NLT + NLN + i] = A.twN.hi[i];
    TwRows<T, CAP, Tw2<T>> tw;
    tw.lds = tl;
    tw.rest.lo = tl + NLT;
    tw.rest.hi = tl + NLT + NLN;
    tw.rest.lb = LBN;
    // the epilogue's twiddle w_G^(tid + i NT) = w_G^tid w_(G/NT)^i
    constexpr int NE = (N / 2 + NT) / NT;  // values of i with tid + i NT <= N/2
    static_assert(G / NT <= 32 || NE <= 1, "epilogue rotations");
    const cplx<T> wtid = A.twH[tid];
    // (thread index and twiddle opaque in each item's epilogue, and its steps
    // kept apart: the compiler would hoist every step's addresses and rotations
    // out of the item loop and spill them)
    auto epilogue = [&](auto &&step) __attribute__((always_inline)) {
        int t = tid;
        cplx<T> w0 = wtid;
        asm volatile("" : "+v"(t), "+v"(w0.x), "+v"(w0.y));
        unroll<NE>([&](auto i) __attribute__((always_inline)) {
            constexpr int k = decltype(i)::value;
            step(t + k * NT, k == 0 ? w0 : w0 * unit_root_32<T>(k * (G / NT > 0 ? 32 * NT / G : 1)));
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    __shared__ int item_sh[kBootCurveWords + 1];
    __shared__ int nlist_sh;
    __shared__ int dmax_sh[NT / 64];
    // draws per block of 32 anchors (at most G/32 = 1024 blocks)
    constexpr int NB = G / 32;
    static_assert(NB >= 2 && NTAPS <= 32, "a tap window spans at most two anchor blocks");
    __shared__ int hist_sh[NB];
    __shared__ double red_sh[2 * (NT / 64)];
    __shared__ T peak_sh[NT / 64];
    __shared__ int kpk_sh[NT / 64];

    // The draws of replicate `rep` of the curve at c0 (nc points).  Up to
    // A.list_cap points, equal draws are merged: their multiplicities are counted
    // in 16-bit LDS counters (in the grid's space), and the distinct points, about
    // 63 % of nc, go to this workgroup's list with their counts, in any order (the
    // grid's integer sums do not depend on it).  The spread, bound by its LDS
    // atomics, then adds each point once with the weight count * y.  A longer curve
    // is drawn point by point in the spread.  With `moments`, red_sh receives the
    // sums over the draws of (y - shift) and its square.  Returns the length of the
    // list (nc without one).
    const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned *const list = A.list + (long)blockIdx.x * A.list_cap;
    auto draw = [&](int nc, int rep, const FastMod &fm, int p) __attribute__((always_inline)) {
        const uint32_t t = (uint32_t)rep * (uint32_t)nc + (uint32_t)p;
        return fm(xorshift32(wang_hash(A.seed + t)));
    };
    auto prepare_draws = [&](auto moments, int c0, int nc, int rep, const FastMod &fm,
                             T shift) __attribute__((always_inline)) -> int {
        constexpr bool MOM = decltype(moments)::value;
        double s1 = 0.0, s2 = 0.0;
        auto moment = [&](double mult, T yv) __attribute__((always_inline)) {
            const double d = (double)yv - (double)shift;
            s1 += mult * d;
            s2 += mult * d * d;
        };
        const bool merged = nc <= A.list_cap;  // uniform
        if (merged) {
            unsigned *cw = reinterpret_cast<unsigned *>(gu);
            const int nw = (nc + 1) / 2;
            for (int i = tid; i < (nw + 3) / 4; i += NT)
                reinterpret_cast<uint4 *>(cw)[i] = make_uint4(0, 0, 0, 0);
            if (tid == 0) nlist_sh = 0;
            __syncthreads();
            for (int p = tid; p < nc; p += NT) {
                const unsigned d = draw(nc, rep, fm, p);
                atomicAdd(&cw[d >> 1], 1u << (16 * (d & 1)));
            }
            __syncthreads();
            for (int i0 = wave_id * 64; i0 < nw; i0 += NT) {  // uniform
                const int i = i0 + (tid & 63);
                const unsigned w = i < nw ? cw[i] : 0u, lo = w & 0xffffu, hi = w >> 16;
                if constexpr (MOM) {
                    if (lo) moment((double)lo, A.y[c0 + 2 * i]);
                    if (hi) moment((double)hi, A.y[c0 + 2 * i + 1]);
                }
                const unsigned long long b0 = __ballot(lo != 0), b1 = __ballot(hi != 0);
                int at = 0;
                if ((tid & 63) == 0) at = atomicAdd(&nlist_sh, __popcll(b0) + __popcll(b1));
                at = __builtin_amdgcn_readfirstlane(at);
                at += __builtin_amdgcn_mbcnt_hi((unsigned)(b0 >> 32),
                                                __builtin_amdgcn_mbcnt_lo((unsigned)b0, 0));
                at += __builtin_amdgcn_mbcnt_hi((unsigned)(b1 >> 32),
                                                __builtin_amdgcn_mbcnt_lo((unsigned)b1, 0));
                if (lo) list[at] = (unsigned)(2 * i) | lo << 16;
                if (hi) list[at + (lo ? 1 : 0)] = (unsigned)(2 * i + 1) | hi << 16;
            }
        } else if constexpr (MOM) {
            for (int p = tid; p < nc; p += NT) moment(1.0, A.y[c0 + (int)draw(nc, rep, fm, p)]);
        }
        if constexpr (MOM) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                s1 += __shfl_xor(s1, o);
                s2 += __shfl_xor(s2, o);
            }
            if ((tid & 63) == 0) {
                red_sh[2 * (tid >> 6)] = s1;
                red_sh[2 * (tid >> 6) + 1] = s2;
            }
        }
        __syncthreads();
        return merged ? __builtin_amdgcn_readfirstlane(nlist_sh) : nc;
    };

    // Grid of one transform: the nl entries of prepare_draws, positions from P,
    // values y[d] - shift (or 1), |value| <= vm; spread in fixed point and
    // transformed in place into z.  Returns the power of two that the spectrum is
    // to be multiplied by: the integers go through the FFT as they are.
    auto transform = [&](int c0, int nc, int nl, int rep, const FastMod &fm, const PointRec<T> *P,
                         const T *y, T shift, double vm, int cover,
                         auto &&ahead) __attribute__((always_inline)) -> T {
        ahead();
        const bool merged = nc <= A.list_cap;  // uniform
        int sexp = 0;
        if (vm <= 1e300) {  // false for NaN and inf
            // No cell receives more than cnt weights of size <= vm * wscale, so
            // with cnt * vm * wscale * 2^sexp <= 2^headroom no cell can wrap.
            // First attempt: cnt = 4x the densest window of the original
            // points.  The draws' own densest window is counted on the way
            // (draws per block of 32 anchors; a cell's taps come from at most
            // 32 consecutive anchors, so from two adjacent blocks): if it
            // exceeds cnt the item is redone at that exact count.
            int cnt = 4 * max(cover, 1);
            for (int attempt = 0; attempt < 2; ++attempt) {
                const double bound = vm * (double)cnt * (double)A.wscale;
                int e = -kMaxExp;  // ceil(log2(bound))
                if (bound > 0 && frexp(bound, &e) == 0.5) --e;
                sexp = min(max(FixedOf<T>::headroom_bits - e, -kMaxExp), kMaxExp);
                const T mul = (T)ldexp((double)A.wscale, sexp);
                // thread t takes the spl consecutive entries from t spl on: the list
                // follows the points, often in order of position, and neighbouring
                // lanes on neighbouring points would put one atomic's lanes on the
                // same cells, which serialises them.  PB at a time, loaded ahead of
                // their use (slots past the end take entry 0 and are skipped below)
                const int spl = (nl + NT - 1) / NT;  // uniform
                unsigned wn[PB];
                auto entries = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
                    for (int k = 0; k < PB; ++k) {
                        int p = tid * spl + k0 + k;
                        p = k0 + k < spl && p < nl ? p : 0;
                        wn[k] = merged ? list[p] : draw(nc, rep, fm, p);
                    }
                };
                if (nl > 0) entries(0);
                for (int i = tid; i < (int)((G + 2 * kBootHalo) * sizeof(T) / 16); i += NT)
                    reinterpret_cast<uint4 *>(cuna_smem)[i] = make_uint4(0, 0, 0, 0);
                for (int i = tid; i < NB; i += NT) hist_sh[i] = 0;
                __syncthreads();
                for (int k0 = 0; k0 < spl; k0 += PB) {
                    PointRec<T> pr[PB];
                    T vv[PB];
                    int dk[PB], mk[PB];  // point and multiplicity
#pragma unroll
                    for (int k = 0; k < PB; ++k) {
                        dk[k] = c0 + (int)(merged ? wn[k] & 0xffffu : wn[k]);
                        mk[k] = merged ? (int)(wn[k] >> 16) : 1;
                    }
#pragma unroll
                    for (int k = 0; k < PB; ++k) pr[k] = P[dk[k]];
                    if (y) {
#pragma unroll
                        for (int k = 0; k < PB; ++k) vv[k] = (T)mk[k] * (y[dk[k]] - shift);
                    } else {
#pragma unroll
                        for (int k = 0; k < PB; ++k) vv[k] = (T)mk[k];
                    }
                    if (k0 + PB < spl) entries(k0 + PB);
#pragma unroll
                    for (int k = 0; k < PB; ++k) {
                        if (k0 + k < spl && tid * spl + k0 + k < nl) {
                            U *dst = gu + (pr[k].a - Q0);
                            if constexpr (sizeof(T) == 4) {
                                // each tap's rounded weight to its atomic as
                                // it is formed (weights <= 2^headroom_bits)
                                tap_fixed<T, NTAPS, Fixed32, true>(
                                    vv[k] * mul, pr[k].e, A.bi, A.e3, T(0),
                                    [&](int q, unsigned n) { atomicAdd(dst + q, (U)n); });
                            } else {
                                T w[NTAPS];
                                tap_weights<T, NTAPS>(vv[k] * mul, pr[k].e, A.bi, A.e3, w);
#pragma unroll
                                for (int q = 0; q < NTAPS; ++q)
                                    atomicAdd(dst + q, (U)FixedOf<T>::round(w[q]));
                            }
                            atomicAdd(&hist_sh[pr[k].a >> 5], mk[k]);
                        }
                    }
                }
                __syncthreads();
                // the taps that wrapped (distinct cells, read after the next barrier)
                if (tid < kBootHalo) {
                    gu[G - kBootHalo + tid] += gu[tid - kBootHalo];
                    gu[tid] += gu[G + tid];
                }
                int dmax = 0;
                for (int b = tid; b < NB; b += NT)
                    dmax = max(dmax, hist_sh[b] + hist_sh[(b + 1) & (NB - 1)]);
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) dmax = max(dmax, __shfl_xor(dmax, o));
                if ((tid & 63) == 0) dmax_sh[tid >> 6] = dmax;
                __syncthreads();
                dmax = dmax_sh[0];
#pragma unroll
                for (int w = 1; w < NT / 64; ++w) dmax = max(dmax, dmax_sh[w]);
                if (dmax <= cnt) break;  // uniform
                cnt = dmax;
                __syncthreads();  // every thread has read dmax_sh
            }
        }
        // the FFT's first pass reads the fixed-point grid (complex e = cells
        // 2e, 2e+1) and converts it to reals as it loads
        auto fetch = [&](int e, int) __attribute__((always_inline)) {
            const FixedPair<I> q = reinterpret_cast<const FixedPair<I> *>(gu)[e];
            return cmk((T)q.x, (T)q.y);
        };
        __syncthreads();
        fft_pass<T, 1, LG, 1, NT, 0, 0, decltype(fetch), true, NoHook, decltype(tw), MR>(
            z, tw, fetch, NoHook());
        // a non-finite value makes every spectrum value NaN
        return vm <= 1e300 ? (T)ldexp(1.0, -sexp) : (T)NAN;
    };
    // deconvolved spectrum, times `scale`, at frequency f (0 <= f < M/2) from z
    auto spectrum = [&](int f, cplx<T> w, T scale) __attribute__((always_inline)) -> cplx<T> {
        const SinkAccurate<T> &sk = A.sink;
        const cplx<T> a = real_spectrum_at(z[lds_sw(f)], z[lds_sw((N - f) & (N - 1))], w);
        const T kk = (T)f * sk.invG;
        return a * ((T(0.5) * sk.pref * scale) * dexp(sk.coef * kk * kk));
    };

    // The first item is the workgroup's index.  The first wave takes each further
    // one off the queue while the workgroup works on the current one, and has its
    // curve's entry in LDS by the end: an item then starts without a chain of global
    // loads.  With many items per workgroup it does so first thing, otherwise before
    // the current item's last transform, so that none waits behind a long one while
    // other workgroups run dry.  Measured, early / late: 128 curves x 25 replicates,
    // M = 2^14, 12 items each, 544 / 566 us; 64 x 25 periodograms, M = 2^13, 3 items
    // each, 158 / 148 us.  (All off the queue and early, the first workgroups had a
    // second item before the last ones had any: 8 curves x 24 replicates, M = 2^13,
    // FP64 periodograms 88 us, now 52.)
    const int per_curve = A.nbs * (A.split ? A.ntr : 1);
    const int lane = tid & 63;
    const bool first_wave = tid < 64;
    auto take = [&]() __attribute__((always_inline)) -> int {
        return lane == 0 ? (int)gridDim.x + atomicAdd(A.counter, 1) : 0;
    };
    auto stage_item = [&](int item) __attribute__((always_inline)) {
        item = __builtin_amdgcn_readfirstlane(item);
        int w = -1;
        if (item < A.total) {
            const int pos = item / per_curve;
            if (lane < kBootCurveWords)
                w = reinterpret_cast<const int *>(A.curves + pos)[lane];
            else if (lane == kBootCurveWords)
                w = item - pos * per_curve;
        }
        if (lane <= kBootCurveWords) item_sh[lane] = w;  // (rem < 0: no item left)
    };
    if (first_wave) stage_item(blockIdx.x);
    __syncthreads();
    for (;;) {
        // uniform over the workgroup: scalar registers
        auto word = [&](int k) { return __builtin_amdgcn_readfirstlane(item_sh[k]); };
        const int rem = word(kBootCurveWords);
        if (rem < 0) break;  // uniform over the workgroup
        const int ci = word(0), c0 = word(1), nc = word(2);
        FastMod fm;
        fm.d = (uint32_t)max(nc, 1);
        fm.m = (uint32_t)word(3);
        fm.s1 = word(4);
        fm.s2 = word(5);
        const int cover_x = word(6), cover_2x = word(7);
        const double ymax = __longlong_as_double(((long long)word(9) << 32) | (unsigned)word(8));
        int next = 0;
        const bool early = A.total >= 8 * (int)gridDim.x;
        if (first_wave && early) next = take();
        auto take_next = [&]() __attribute__((always_inline)) {
            if (first_wave && !early) next = take();
        };
        if constexpr (MODE == 0) {
            const int rep = A.split ? rem / A.ntr : rem;
            const int tr0 = A.split ? rem % A.ntr : 0, tr1 = A.split ? tr0 + 1 : A.ntr;
            const int nl = prepare_draws(std::false_type{}, c0, nc, rep, fm, T(0));
            for (int tr = tr0; tr < tr1; ++tr) {
                const bool usey = tr == 0 && A.y;
                const T scale = transform(c0, nc, nl, rep, fm, tr == 0 ? A.rec_x : A.rec_2x,
                                          usey ? A.y : nullptr, T(0), usey ? ymax : 1.0,
                                          tr == 0 ? cover_x : cover_2x, [&] {
                                              if (tr == tr1 - 1) take_next();
                                          });
                if (first_wave && tr == tr1 - 1) stage_item(next);
                SinkAccurate<T> sk = A.sink;
                sk.pref *= scale;
                cplx<T> *o = (tr == 0 ? A.out_y : A.out_w) + ((long)ci * A.nbs + rep) * sk.M;
                epilogue([&](int r, cplx<T> w) __attribute__((always_inline)) {
                    if (r <= N / 2)
                        emit_pair(sk, o, r, N, z[lds_sw(r)], z[lds_sw((N - r) & (N - 1))], w);
                });
                __syncthreads();
            }
        } else {
            const int rep = rem;
            const long row = (long)ci * A.nbs + rep;
            const int half = A.sink.M / 2;
            // moments of the drawn values about the first draw (shifted sums
            // keep the variance accurate when |mean| >> spread)
            const T shift = nc > 0 ? A.y[c0 + (int)draw(nc, rep, fm, 0)] : T(0);
            const int nl = prepare_draws(std::true_type{}, c0, nc, rep, fm, shift);
            double s1 = 0.0, s2 = 0.0;
            for (int w = 0; w < NT / 64; ++w) {
                s1 += red_sh[2 * w];
                s2 += red_sh[2 * w + 1];
            }
            s1 = uniform_f64(s1);
            s2 = uniform_f64(s2);
            const double nd = (double)max(nc, 1);
            const double mean_off = s1 / nd;
            const T ybar = (T)((double)shift + mean_off);
            const T yy = (T)fmax(0.0, s2 - s1 * mean_off);
            // window W(2w), parked in this workgroup's workspace row
            const T wscale =
                transform(c0, nc, nl, rep, fm, A.rec_2x, nullptr, T(0), 1.0, cover_2x, [] {});
            cplx<T> *wrow = A.ls_w + (long)blockIdx.x * half;
            epilogue([&](int f, cplx<T> w) __attribute__((always_inline)) {
                if (f < half) wrow[f] = spectrum(f, w, wscale);
            });
            __syncthreads();
            // F(w) of the mean-subtracted values, then the power
            const double vm = ymax + fabs((double)ybar);
            const T yscale =
                transform(c0, nc, nl, rep, fm, A.rec_x, A.y, ybar, vm, cover_x, take_next);
            if (first_wave) stage_item(next);
            T best = T(-1);
            int kbest = 0;
            epilogue([&](int f, cplx<T> w) __attribute__((always_inline)) {
                if (f < half) {
                    const T pw = ls_power(spectrum(f, w, yscale), wrow[f], (T)nc, yy);
                    if (A.ls_power) A.ls_power[row * half + f] = pw;
                    if (f >= 1 && pw > best) {
                        best = pw;
                        kbest = f;
                    }
                }
            });
            if (A.ls_peak || A.ls_kpeak) {
                // block arg-max (ties: smallest k)
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) {
                    const T ob = __shfl_xor(best, o);
                    const int ok = __shfl_xor(kbest, o);
                    if (ob > best || (ob == best && ok < kbest)) {
                        best = ob;
                        kbest = ok;
                    }
                }
                if ((tid & 63) == 0) {
                    peak_sh[tid >> 6] = best;
                    kpk_sh[tid >> 6] = kbest;
                }
                __syncthreads();
                if (tid == 0) {
                    for (int w = 1; w < NT / 64; ++w) {
                        if (peak_sh[w] > best || (peak_sh[w] == best && kpk_sh[w] < kbest)) {
                            best = peak_sh[w];
                            kbest = kpk_sh[w];
                        }
                    }
                    if (A.ls_peak) A.ls_peak[row] = best < T(0) ? T(0) : best;
                    if (A.ls_kpeak) A.ls_kpeak[row] = kbest;
                }
            }
            __syncthreads();
        }
    }
}

// Queue head := 0, and one BootCurve per workgroup (position in the queue order)
// with the curve's max |y|.  Latency-bound: a thread keeps 8 loads in flight.
// One workgroup of 256 threads per curve with one load in flight took 80 us for
// 128 curves of up to 50,000 values, and resetting the queue was a launch of its
// own (4.7 us).
constexpr int kPrepThreads = 1024, kPrepLoads = 8;
template <typename T>
__global__ __launch_bounds__(kPrepThreads) void k_boot_prepare(const T *y, const int *coff,
                                                               const int *order,
                                                               const int *cover_x,
                                                               const int *cover_2x,
                                                               BootCurve *curves, int *counter) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *counter = 0;
    const int ci = order[blockIdx.x];
    const int b = coff[ci], e = coff[ci + 1];
    T m = T(0);
    if (y) {
        for (long i = b + (long)threadIdx.x; i < e; i += kPrepLoads * kPrepThreads) {
            T v[kPrepLoads];
#pragma unroll
            for (int k = 0; k < kPrepLoads; ++k)
                v[k] = y[i + k * kPrepThreads < e ? i + k * kPrepThreads : i];
#pragma unroll
            for (int k = 0; k < kPrepLoads; ++k) m = fmax(m, fabs(v[k]));
        }
    } else {
        m = T(1);
    }
    __shared__ T red[kPrepThreads / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kPrepThreads / 64; ++w) m = fmax(m, red[w]);
        FastMod fm;
        fm.init((uint32_t)max(e - b, 1));
        BootCurve c;
        c.ci = ci;
        c.c0 = b;
        c.nc = e - b;
        c.fm_m = fm.m;
        c.fm_s1 = fm.s1;
        c.fm_s2 = fm.s2;
        c.cover_x = cover_x[ci];
        c.cover_2x = cover_2x ? cover_2x[ci] : 0;
        c.ymax = (double)m;
        curves[blockIdx.x] = c;
    }
}

// Per-curve densest window: the most points whose anchors fall in one cyclic run
// of ntaps cells of the G-cell grid.  One workgroup per curve, anchor histogram in
// LDS, where each thread slides the window over its share of the cells (a word of
// padding per 32 cells keeps the threads' walks on different banks).  What is left
// is the histogram's loads.  256 curves of 100 - 20,000 points on 2^15 cells
// take 10.9 us (22.6 with the windows as differences of a wave's prefix sums,
// whose chain of lane exchanges bounds it).
__host__ __device__ constexpr int cover_slot(int i) { return i + (i >> 5); }

template <typename T>
__global__ __launch_bounds__(1024) void k_curve_cover(const PointRec<T> *rec, const int *coff,
                                                      int G, int ntaps, int *cover) {
    int *h = reinterpret_cast<int *>(cuna_smem);
    __shared__ int red;
    const int c = blockIdx.x, b = coff[c], e = coff[c + 1];
    const int tid = threadIdx.x, NT = blockDim.x;
    for (int i = tid; i < (cover_slot(G) + 3) / 4; i += NT)
        reinterpret_cast<int4 *>(h)[i] = make_int4(0, 0, 0, 0);
    if (tid == 0) red = 0;
    __syncthreads();
    constexpr int U = 8;  // loads in flight
    for (int i = b + tid; i < e; i += U * NT) {
        int a[U];
#pragma unroll
        for (int k = 0; k < U; ++k) a[k] = rec[min(i + k * NT, e - 1)].a;
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (i + k * NT < e) atomicAdd(&h[cover_slot(a[k] & (G - 1))], 1);
    }
    __syncthreads();
    const int share = (G + NT - 1) / NT, g0 = tid * share, g1 = min(g0 + share, G);
    int best = 0, win = 0;  // win: cells g - ntaps .. g - 1
    if (g0 < G)
        for (int g = g0 - ntaps; g < g0; ++g) win += h[cover_slot(g & (G - 1))];
#pragma unroll 4
    for (int g = g0; g < g1; ++g) {
        win += h[cover_slot(g)] - h[cover_slot((g - ntaps) & (G - 1))];
        best = max(best, win);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) best = max(best, __shfl_xor(best, o));
    if ((tid & 63) == 0) atomicMax(&red, best);
    __syncthreads();
    if (tid == 0) cover[c] = red;
}

// --------------------------------------------- fused adjoint of small grids --
// The whole adjoint of one (curve, value vector) item in one workgroup, for grids
// that fit its LDS: the points in their original order, spread in fixed point into
// the halo grid of the fused bootstrap, transformed in place, and the deconvolved
// spectrum written.  The tile path's sort, spread launch and passes of the grid
// through memory fall away; the bound is the LDS atomics and vector instructions
// of the workgroup's points (1.15 ns each at 2^15 cells in FP32), so the host takes
// this path only for curves that are not long next to the whole batch.  256 curves
// of 100 - 20,000 points, M = 2^14, new plan each time: 100 us, 143 with the sort,
// tiles and FFT; one curve of 1000 points, M = 2^11, plan kept: 8.3 us, 8.9.
//
// Scale: with `cover` the curve's densest window of NTAPS anchors and vm its
// largest |value|, no cell sum exceeds cover * vm * wscale, kept within 2^30
// (FP32) / 2^61 (FP64).  All of the curve shares it, and with one unit of the scale
// at u the grid's rounding is 0.94 u / mean |value| of the spectrum's norm (m = 8).
// In FP32 a curve whose mean |value| has fewer than kMeanUnits of them, so that this
// would pass 0.75e-7 (the FFT's own is 2e-7), is looked at closer: the sums of the
// |values| per 16 anchors bound a cell's sum by that of the blocks which its window
// touches, a few times less than cover * vm.  If that is not enough, where one value
// dominates or the points are dense, a second round over the points accumulates what
// rounding each weight dropped, scaled by up to 2^kRestBits, and the first round's
// integers wait in the workspace row of the workgroup.  Errors with cover * vm alone /
// this / tiles, whose scales are each tile's: 4700 points, M = 2^14, one value 30 times
// the others 5.0e-7 / 2.2e-7 / 2.1e-7, log-normal values 6.9e-7 / 2.2e-7 / 2.3e-7;
// 20,000 points, one value 1000 times the others 41e-7 / 1.9e-7 / 1.9e-7.  It costs 256
// ordinary curves of 100 - 20,000 points 3.6 us of 54 for the sums; where the longest
// takes the second round they take 82.
constexpr float kMeanUnits = 0.75f * 16777216.0f;
constexpr int kRestBits = 14;

// What tap_fixed (FP32, table) rounded off each weight: it repeats its operations,
// so n_q is the same integer, and the rest up e3 - n_q is exact up to one rounding.
template <int NTAPS, class Emit>
__device__ __forceinline__ void tap_rest(float v, float e, float bi, const float *e3,
                                         Emit &&emit) {
    constexpr int Q0 = (NTAPS - 1) / 2;
    const float E1 = dexp(-e * e * bi);
    const float E2 = dexp(2.0f * e * bi);
    const float E2i = dexp(-2.0f * e * bi);
    const float h = copysignf(0.5f, v);
    float up = v * E1;
#pragma unroll
    for (int q = Q0; q < NTAPS; ++q) {
        emit(q, fmaf(up, e3[q], -(float)(int)fmaf(up, e3[q], h)));
        up *= E2;
    }
    float dn = v * E1 * E2i;
#pragma unroll
    for (int q = Q0 - 1; q >= 0; --q) {
        emit(q, fmaf(dn, e3[q], -(float)(int)fmaf(dn, e3[q], h)));
        dn *= E2i;
    }
}

// Twiddles: FP32 as the single-workgroup FFT takes them, rows in LDS and the last
// pass of 2^13 and 2^14 points from the full table in global memory (two-level
// products there raised the error of a survey's spectra from 2.3e-7 to 3.4e-7);
// FP64, whose rows of 2^13 do not fit beside the grid and whose filter's error is
// far above, as the fused bootstrap.
template <typename T>
__host__ __device__ constexpr int adjoint_cap(int lg) {
    return sizeof(T) == 4 ? small_cap(lg) : boot_cap<T>(lg);
}
template <typename T>
__host__ __device__ constexpr size_t adjoint_lds_bytes(int lg) {
    const size_t two_level =
        sizeof(T) == 4 ? 0 : ((size_t)1 << ((lg + 1) / 2)) + ((size_t)1 << (lg - (lg + 1) / 2));
    return sizeof(cplx<T>) * (((size_t)1 << lg) +
                              rows_count(lg, small_mr(lg), adjoint_cap<T>(lg)) + two_level) +
           2 * kBootHalo * sizeof(T);
}

template <typename T>
struct AdjointArgs {
    const PointRec<T> *rec;  // (anchor, e) by original index
    const T *y;              // nullable: unit weights
    long y_stride;           // per value vector
    const int *coff, *order, *cover;
    int nrhs, total;         // total = curves * nrhs
    int *hi;                 // FP32, two rounds: G integers per workgroup
    T bi, wscale;
    T e3[kMaxTaps];
    SinkAccurate<T> sink;
    const cplx<T> *twT;   // twiddle rows up to adjoint_cap
    const cplx<T> *fine;  // FP32: w_N^e
    Tw2<T> twN;           // FP64: the same by two levels
    const cplx<T> *twH;   // w_G^e, e < workgroup size
};

template <typename T, int LG, int NTAPS, int NT>
__global__ __launch_bounds__(NT) void k_adjoint_fused(AdjointArgs<T> A) {
    using I = typename FixedOf<T>::I;
    using U = std::make_unsigned_t<I>;
    constexpr int N = 1 << LG, G = 2 * N, Q0 = (NTAPS - 1) / 2, PB = 4;
    constexpr int LBN = (LG + 1) / 2, NLN = 1 << LBN, NHN = 1 << (LG - LBN);
    constexpr int MR = small_mr(LG), CAP = adjoint_cap<T>(LG), NLT = rows_count(LG, MR, CAP);
    using Rest = std::conditional_t<sizeof(T) == 4, const cplx<T> *, Tw2<T>>;
    constexpr int kMaxExp = sizeof(T) == 4 ? 100 : 1000;
    constexpr T kBig = sizeof(T) == 4 ? T(3.0e38f) : T(1.0e300);
    T *grid = reinterpret_cast<T *>(cuna_smem) + kBootHalo;
    U *gu = reinterpret_cast<U *>(grid);
    cplx<T> *z = reinterpret_cast<cplx<T> *>(grid);
    cplx<T> *tl = reinterpret_cast<cplx<T> *>(grid + G + kBootHalo);
    __shared__ T vmax_sh[NT / 64], vsum_sh[NT / 64];
    __shared__ unsigned block_sh[NT / 64];
    const int tid = threadIdx.x;
    for (int i = tid; i < NLT; i += NT) tl[i] = A.twT[i];
    TwRows<T, CAP, Rest> tw;
    tw.lds = tl;
    if constexpr (sizeof(T) == 4) {
        tw.rest = A.fine;
    } else {
        for (int i = tid; i < NLN; i += NT) tl[NLT + i] = A.twN.lo[i];
        for (int i = tid; i < NHN; i += NT) tl[NLT + NLN + i] = A.twN.hi[i];
        tw.rest.lo = tl + NLT;
        tw.rest.hi = tl + NLT + NLN;
        tw.rest.lb = LBN;
    }
    constexpr int NE = (N / 2 + NT) / NT;
    const cplx<T> wtid = A.twH[tid];
    int *const hi = A.hi + (long)blockIdx.x * G;

    for (int item = blockIdx.x; item < A.total; item += gridDim.x) {
        const int ci = A.order[item / A.nrhs], r = item % A.nrhs;
        const int c0 = A.coff[ci], nc = A.coff[ci + 1] - c0, cover = max(A.cover[ci], 1);
        const PointRec<T> *P = A.rec + c0;
        const T *y = A.y ? A.y + r * A.y_stride + c0 : nullptr;
        // f(|value|, record, counts) for every point, the last one also for the
        // slots past the end
        auto scan = [&](auto &&f) __attribute__((always_inline)) {
            for (int p0 = tid; p0 < nc; p0 += PB * NT) {
                T v[PB];
                PointRec<T> pr[PB];
#pragma unroll
                for (int k = 0; k < PB; ++k) {
                    const int p = min(p0 + k * NT, nc - 1);
                    v[k] = y ? fabs(y[p]) : T(1);
                    pr[k] = P[p];
                }
#pragma unroll
                for (int k = 0; k < PB; ++k) f(v[k], pr[k], p0 + k * NT < nc);
            }
        };
        // largest |value|; a non-finite value or position (NaN x gives NaN e)
        // makes it infinite and the spectrum NaN
        T vm = y ? T(0) : T(1), vs = T(0);  // largest, and (FP32) sum of the |values|
        scan([&](T v, const PointRec<T> &pr, bool in) __attribute__((always_inline)) {
            vm = fmax(vm, v <= kBig && fabs(pr.e) <= kBig ? v : T(INFINITY));
            vs += in ? v : T(0);
        });
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            vm = fmax(vm, __shfl_xor(vm, o));
            if constexpr (sizeof(T) == 4) vs += __shfl_xor(vs, o);
        }
        if ((tid & 63) == 0) {
            vmax_sh[tid >> 6] = vm;
            vsum_sh[tid >> 6] = vs;
        }
        for (int i = tid; i < (int)((G + 2 * kBootHalo) * sizeof(T) / 16); i += NT)
            reinterpret_cast<uint4 *>(cuna_smem)[i] = make_uint4(0, 0, 0, 0);
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) vm = fmax(vm, vmax_sh[w]);
        const bool finite = vm <= kBig;  // uniform
        // the scale's exponent for cell sums within `bound`
        auto exponent = [&](double bound) __attribute__((always_inline)) -> int {
            int eb = -kMaxExp;  // ceil(log2(bound))
            if (bound > 0 && finite && frexp(bound, &eb) == 0.5) --eb;
            return min(max(FixedOf<T>::headroom_bits - eb, -kMaxExp), kMaxExp);
        };
        int sexp = exponent((double)vm * (double)cover * (double)A.wscale);
        bool second = false;  // a second round (uniform)
        if constexpr (sizeof(T) == 4) {
            float mean = 0.0f;
#pragma unroll
            for (int w = 0; w < NT / 64; ++w) mean += vsum_sh[w];
            mean *= A.wscale / (float)max(nc, 1);
            if (finite && mean > 0.0f && ldexpf(mean, sexp) < kMeanUnits) {
                // block sums in the grid's first cells (cleared above, cleared again
                // below), in units of 2^(ev - q), rounded up: within 2^31 in all.
                // Lanes count in four copies: points in order of position meet on one
                // block.
                constexpr int NBK = G >> 4, NW = (NTAPS + 14) / 16 + 1;
                static_assert(NW <= NBK, "blocks that a window touches");
                uint4 *const blocks = reinterpret_cast<uint4 *>(gu);
                int ev = 0;
                (void)frexpf(vm, &ev);
                const int q = 30 - (32 - __clz(nc)), copy = tid & 3;
                scan([&](float v, const PointRec<T> &pr, bool in) __attribute__((always_inline)) {
                    if (in) atomicAdd(&gu[(pr.a >> 4) * 4 + copy], (U)ceilf(ldexpf(v, q - ev)));
                });
                __syncthreads();
                unsigned most = 0;
                for (int b = tid; b < NBK; b += NT) {
                    unsigned sum = 0;
#pragma unroll
                    for (int i = 0; i < NW; ++i) {
                        const uint4 u = blocks[(b + i) & (NBK - 1)];
                        sum += u.x + u.y + u.z + u.w;
                    }
                    most = max(most, sum);
                }
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) most = max(most, (unsigned)__shfl_xor((int)most, o));
                if ((tid & 63) == 0) block_sh[tid >> 6] = most;
                __syncthreads();
                for (int b = tid; b < NBK; b += NT) blocks[b] = make_uint4(0, 0, 0, 0);
#pragma unroll
                for (int w = 0; w < NT / 64; ++w) most = max(most, block_sh[w]);
                sexp = max(sexp, exponent(ldexp((double)most * (double)A.wscale, ev - q)));
                second = ldexpf(mean, sexp) < kMeanUnits;
                __syncthreads();
            }
        }
        const T mul = (T)ldexp((double)A.wscale, sexp);
        // the second round: rests of at most 1/2, `cover` of them in a cell, within 2^30
        const int lowbits = min(kRestBits, 31 - (32 - __clz(cover - 1)));
        const float lowmul = ldexpf(1.0f, lowbits);
        // one round over the points: each tap's integer, or (LOW) the scaled rest
        // of its rounding, to its cell.  Thread t takes spl consecutive points:
        // neighbours in neighbouring lanes would meet on one cell (see k_boot_fused)
        const int spl = (nc + NT - 1) / NT;
        auto round = [&](auto low) __attribute__((always_inline)) {
            constexpr bool LOW = decltype(low)::value;
            for (int k0 = 0; k0 < spl; k0 += PB) {
                PointRec<T> pr[PB];
                T vv[PB];
#pragma unroll
                for (int k = 0; k < PB; ++k) {
                    const int p = tid * spl + k0 + k, q = k0 + k < spl && p < nc ? p : 0;
                    pr[k] = P[q];
                    vv[k] = y ? y[q] : T(1);
                }
#pragma unroll
                for (int k = 0; k < PB; ++k) {
                    if (k0 + k < spl && tid * spl + k0 + k < nc) {
                        U *dst = gu + (pr[k].a - Q0);
                        if constexpr (LOW) {
                            tap_rest<NTAPS>(vv[k] * mul, pr[k].e, A.bi, A.e3,
                                            [&](int q, float rest) {
                                                atomicAdd(dst + q, (U)__float2int_rn(rest * lowmul));
                                            });
                        } else if constexpr (sizeof(T) == 4) {
                            tap_fixed<T, NTAPS, Fixed32, true>(
                                vv[k] * mul, pr[k].e, A.bi, A.e3, T(0),
                                [&](int q, unsigned n) { atomicAdd(dst + q, (U)n); });
                        } else {
                            T w[NTAPS];
                            tap_weights<T, NTAPS>(vv[k] * mul, pr[k].e, A.bi, A.e3, w);
#pragma unroll
                            for (int q = 0; q < NTAPS; ++q)
                                atomicAdd(dst + q, (U)FixedOf<T>::round(w[q]));
                        }
                    }
                }
            }
        };
        auto fold = [&]() __attribute__((always_inline)) {
            __syncthreads();
            if (tid < kBootHalo) {
                gu[G - kBootHalo + tid] += gu[tid - kBootHalo];
                gu[tid] += gu[G + tid];
            }
            __syncthreads();
        };
        if (finite) round(std::false_type{});
        fold();
        if constexpr (sizeof(T) == 4) {
            if (second) {
                for (int i = tid; i < G; i += NT) hi[i] = (int)gu[i];
                __syncthreads();
                for (int i = tid; i < (int)((G + 2 * kBootHalo) * sizeof(T) / 16); i += NT)
                    reinterpret_cast<uint4 *>(cuna_smem)[i] = make_uint4(0, 0, 0, 0);
                __syncthreads();
                round(std::true_type{});
                fold();
                // both parts as reals, in the integers' unit
                for (int i = tid; i < G; i += NT)
                    grid[i] = (T)hi[i] + (T)(int)gu[i] * (T)(1.0f / lowmul);
                __syncthreads();
            }
        }
        auto fetch = [&](int e, int) __attribute__((always_inline)) {
            const FixedPair<I> q = reinterpret_cast<const FixedPair<I> *>(gu)[e];
            return second ? z[e] : cmk((T)q.x, (T)q.y);
        };
        fft_pass<T, 1, LG, 1, NT, 0, 0, decltype(fetch), true, NoHook, decltype(tw), MR>(
            z, tw, fetch, NoHook());
        SinkAccurate<T> sk = A.sink;
        sk.pref *= finite ? (T)ldexp(1.0, -sexp) : (T)NAN;
        cplx<T> *o = sk.row_out((long)ci * A.nrhs + r);
        int t = tid;
        cplx<T> w0 = wtid;
        asm volatile("" : "+v"(t), "+v"(w0.x), "+v"(w0.y));
        unroll<NE>([&](auto i) __attribute__((always_inline)) {
            constexpr int k = decltype(i)::value;
            const int f = t + k * NT;
            const cplx<T> w =
                k == 0 ? w0 : w0 * unit_root_32<T>(k * (G / NT > 0 ? 32 * NT / G : 1));
            if (f <= N / 2)
                emit_pair(sk, o, f, N, z[lds_sw(f)], z[lds_sw((N - f) & (N - 1))], w);
            __builtin_amdgcn_sched_barrier(0);
        });
        __syncthreads();
    }
}

// ----------------------------------------------------------- gather --
// Transpose of the accurate spread, for the backward and the forward transform:
// for each point, sum_o w(o) h[a+o] and sum_o (o - e) w(o) h[a+o] over the real
// grid h; with NG = 2 grids per curve (forward) the first sum over both, as the
// real and imaginary part of one complex value.
template <typename T>
struct GatherArgs {
    const PointRec<T> *rec;
    const int *perm;
    const int *bucket;
    const T *h;         // NG real grids of G cells per slab (slab = curve * nrep + rep)
    long h_stride;
    const T *y;         // values (for d/dx), nullable -> 1
    long y_stride;      // per rep
    T *dy;              // nullable (NG = 2: interleaved complex values)
    T *dx;              // nullable
    long out_stride;    // per rep
    int dy_elem;        // element stride of dy (2: one part of an interleaved complex array)
    int G, tlog, ntiles, Kc, olo, nrep;
    int glog;  // a workgroup takes 2^glog consecutive tiles
    int slab0;  // slab of blockIdx.y = 0
    T bi, wscale, dxscale;  // dxscale = 2 G / beta
    T e3[kMaxTaps];
};

// A workgroup stages the cells of its tiles (and the taps' halo) in LDS, then
// takes their points, which are adjacent in the sorted order.  2^glog tiles
// share a workgroup so that its threads have a point each: one 256-cell tile
// per workgroup left 85 % of the threads idle at 20,000 points on 2^17 cells.
template <typename T, int NTAPS, int NG>
__global__ __launch_bounds__(256) void k_gather(GatherArgs<T> A) {
    constexpr int NT = 256;
    constexpr int Q0 = (NTAPS - 1) / 2;
    struct alignas(NG * sizeof(T)) Cell {
        T v[NG];
    };
    Cell *hs = reinterpret_cast<Cell *>(cuna_smem);  // cells tstart-Q0 .. tstart+span-Q0-1
    const int2 bs = xcd_block(blockIdx.x, blockIdx.y, gridDim.x, gridDim.y);
    const int blk = bs.x, slab = A.slab0 + bs.y;
    const int c = slab / A.nrep, rep = slab % A.nrep;
    const int *bk = A.bucket + (long)c * (A.Kc + 1);
    const int tile0 = blk << A.glog, tile1 = min(tile0 + (1 << A.glog), A.ntiles);
    const int tstart = tile0 << A.tlog;
    const T *h = A.h + (long)slab * NG * A.h_stride;
    const int span = ((tile1 - tile0) << A.tlog) + NTAPS;
    for (int i = threadIdx.x; i < span; i += NT) {
        int cell = tstart - Q0 + i;
        if (cell < 0 || cell >= A.G) {
            cell %= A.G;
            if (cell < 0) cell += A.G;
        }
        Cell v;
#pragma unroll
        for (int k = 0; k < NG; ++k) v.v[k] = h[k * A.h_stride + cell];
        hs[i] = v;
    }
    const long s0 = bk[3 * tile0], send = bk[3 * tile1];
    __syncthreads();
    for (long s = s0 + threadIdx.x; s < send; s += NT) {
        const int p = A.perm[s];
        const PointRec<T> pr = A.rec[s];
        const T e = pr.e;
        const int rel = pr.a - tstart;  // hs index of tap q is rel + q
        T w[NTAPS];
        tap_weights<T, NTAPS>(A.wscale, e, A.bi, A.e3, w);
        T sw[NG] = {}, sd = T(0);
#pragma unroll
        for (int q = 0; q < NTAPS; ++q) {
            const Cell hv = hs[rel + q];
#pragma unroll
            for (int k = 0; k < NG; ++k) {
                const T t = hv.v[k] * w[q];
                sw[k] += t;
                if constexpr (NG == 1) sd += ((T)(q - Q0) - e) * t;
            }
        }
        const long oo = (long)rep * A.out_stride;
        if constexpr (NG == 2) {
            reinterpret_cast<cplx<T> *>(A.dy)[oo + p] = cmk(sw[0], sw[1]);
        } else {
            if (A.dy) A.dy[oo + (long)p * A.dy_elem] = sw[0];
            if (A.dx) {
                const T v = A.y ? A.y[(long)rep * A.y_stride + p] : T(1);
                A.dx[oo + p] = A.dxscale * v * sd;
            }
        }
    }
}

}  // namespace cuna
