// cuna_launch.hpp -- host launchers for the FFT and spread kernels.
// Defined in cuna_kernels.hip, instantiated for the library's real type.
#pragma once

#include "cuna_common.hpp"
#include "cuna_fft.hpp"
#include "cuna_spread.hpp"

namespace cuna {

// complex length N = 2^lgN of the real grid G = 2N, `batch` transforms
struct FftShape {
    int lgN = 0;
    int batch = 1;
    int w = 0;  // columns per workgroup in pass 1 (0: heuristic)
    int h = 0;  // rows (real: row pairs) per workgroup in pass 2 (0: heuristic)
    // rows by which a form with other roundings is chosen (0: batch): the same for
    // calls that have to agree bit for bit
    int rows = 0;
};

template <typename T>
constexpr int max_small_lg() {
    return sizeof(T) == 4 ? 14 : 13;
}
template <typename T>
constexpr int max_fft_lg() {
    return sizeof(T) == 4 ? 24 : 23;
}

// Real grid (batch x G reals, read as batch x N complex, modified in place
// when two passes are used) -> spectrum through the sink.
// `mid` (optional) is recorded on s between the two passes of a two-pass FFT.
template <typename T>
void fft_real_forward(const FftShape &sh, T *grid, const SinkAccurate<T> &sk, hipStream_t s,
                      hipEvent_t mid = nullptr);
template <typename T>
void fft_real_forward(const FftShape &sh, T *grid, const SinkCompat<T> &sk, hipStream_t s,
                      hipEvent_t mid = nullptr);

// Hermitian spectrum (loader) -> real grid (batch x G reals) by an inverse
// (sign -1) transform; `work` holds batch x N complex.
template <typename T>
void fft_c2r_inverse(const FftShape &sh, const LoadHermitian<T> &ld, cplx<T> *work, T *grid,
                     hipStream_t s);

// Plain complex transform of batch sequences of N = 2^lgN values, in place
// (used by tests of the FFT stage through the library).
template <typename T>
void fft_complex(const FftShape &sh, cplx<T> *data, cplx<T> *work, int sign, hipStream_t s);

// sort-by-tile plan building
struct SortWork {
    const int4 *chunks;
    const int *chunk_base;
    const int *nch;
    const int *coff;
    int nchunks, ncurves, total_chunks;
    int *hist;  // 2^kSortBits * total_chunks entries
    int *bsum;
};
template <typename T>
void launch_point_setup(const SetupArgs<T> &A, hipStream_t s);
// one stable counting-sort pass over the anchors' bits [shift, shift + bits)
template <typename T>
void launch_sort_pass(const SortWork &W, int shift, int bits, const PointRec<T> *rec_in,
                      const int *perm_in, PointRec<T> *rec_out, int *perm_out, hipStream_t s);
// first sorted index of every (curve, 3 * tile + edge class) key, from points
// sorted by anchor
template <typename T>
void launch_buckets(const int *coff, int ncurves, int Kc, const PointRec<T> *rec, int tlog,
                    int olo, int ohi, int G, int *bucket, hipStream_t s);

// ev0/ev1 (optional) receive the spread kernel's own start and stop times
template <typename T>
void launch_spread(const SpreadArgs<T> &A, int ntaps, int vm, int nslabs, hipStream_t s,
                   hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);
template <typename T>
// ngrids real grids per slab (2: their sums are the parts of one complex
// output); npts: points of all slabs (for the launch shape)
void launch_gather(const GatherArgs<T> &A, int ntaps, int nslabs, int ngrids, long npts,
                   hipStream_t s);
// per curve, the scatter's work order (tiles by decreasing point count) with
// each tile's ranges and cover (A: rec, bucket, tiles)
template <typename T>
void launch_tile_order(const SpreadArgs<T> &A, int ncurves, TileDesc *desc, hipStream_t s);
// sort by anchor and buckets of short curves in one launch; false, and nothing
// launched, when the longest curve or the grid is too large for it
template <typename T>
bool launch_plan_curves(const PointRec<T> *rec_orig, const int *coff, int ncurves, int longest,
                        int tlog, int G, int Kc, int olo, int ohi, PointRec<T> *rec, int *perm,
                        int *bucket, hipStream_t s);

// fused batched bootstrap (grid in LDS): false when this size/filter has no
// fused kernel
template <typename T>
bool boot_fused_supported(int lgN, int ntaps);
// workgroups a fused kernel is launched with at most
template <typename T>
int fused_slots(int lgN);
// adjoint of small grids, one workgroup per (curve, value vector) item; A.hi holds
// min(A.total, fused_slots) x G integers (FP32)
template <typename T>
void launch_adjoint_fused(const AdjointArgs<T> &A, int lgN, int ntaps, hipStream_t s,
                          hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);
// the twiddle tables of its launches (made at plan creation, so that a captured
// call makes none)
template <typename T>
void warm_adjoint_fused(int lgN);
// per-curve densest tap window (G <= 2^15)
template <typename T>
void launch_curve_cover(const PointRec<T> *rec, const int *coff, int ncurves, int G, int ntaps,
                        int *cover, hipStream_t s);
// zeroes the work-queue head and fills the queue's curve entries (with max |y|);
// launched before every fused bootstrap
template <typename T>
void launch_boot_prepare(const T *y, const int *coff, const int *order, const int *cover_x,
                         const int *cover_2x, int ncurves, BootCurve *curves, int *counter,
                         hipStream_t s);
// mode 0: spectra of y at x and of the window at 2x; 1: Lomb-Scargle power
template <typename T>
void launch_boot_fused(BootArgs<T> A, int lgN, int ntaps, int mode, hipStream_t s);

// bytes of dynamic LDS a launch may use on gfx950
constexpr size_t kMaxLds = 160 * 1024;
// the largest grid y dimension; launches over more slabs or batches split
constexpr int kMaxGridY = 65535;

}  // namespace cuna
