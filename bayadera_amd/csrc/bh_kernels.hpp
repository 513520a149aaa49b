// Launchers of the ahead-of-time kernels (bh_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace bh {

// dataset kernels: threads per block, and blocks: two per CU over 256 CUs
constexpr unsigned kDatasetThreads = 512;
constexpr unsigned kMaxDatasetBlocks = 512;
// largest work-group the context accepts (WGS); the reduction trees of acor and
// the per-step means are sized for it
constexpr unsigned kMaxGroupThreads = 1024;

// bh_dataset_variance_noalloc: the rows one call may have, and the device
// array (one per GPU, held until the process ends) that takes the place of
// the buffers bh_dataset_variance allocates (4 MiB, of which the blocks' parts
// of the rows take three doubles each).
constexpr unsigned kNoAllocMaxRows = 256;
constexpr size_t kNoAllocScratchBytes = (size_t)4 << 20;
static_assert((size_t)kMaxDatasetBlocks * kNoAllocMaxRows * 3 * sizeof(double) <=
                  kNoAllocScratchBytes,
              "the parts of every row");
// Looks up the array's address on `device`, which must be the current
// device; once per device, later calls return at once.
hipError_t noalloc_scratch_init(int device);
// The address noalloc_scratch_init found for `device`.
hipError_t noalloc_scratch(int device, void** ptr);

// dst[i] = src[i] for n16 16-byte pieces (nt: non-temporal loads and stores)
hipError_t launch_copy16(hipStream_t s, const void* src, void* dst, unsigned long long n16,
                         bool nt);
hipError_t launch_init_walkers(hipStream_t s, unsigned seed, const float* limits, unsigned dim,
                               unsigned walkers, float* xs);
hipError_t launch_uniform_sample(hipStream_t s, unsigned seed, float lo, float hi, unsigned quads,
                                 float* x);
hipError_t launch_direct_sample(hipStream_t s, int kind, unsigned seed, float p0, float p1,
                                unsigned quads, float* x);
size_t dataset_scratch_bytes(unsigned m, unsigned long long n);
// limits of every row; clears its `bins` counters
hipError_t launch_min_max(hipStream_t s, const float* a, unsigned m, unsigned long long n,
                          unsigned ld, float* limits, unsigned* counts, unsigned bins,
                          void* scratch);
hipError_t launch_histogram(hipStream_t s, const float* a, unsigned m, unsigned long long n,
                            unsigned ld, const float* limits, unsigned bins, unsigned* counts);
hipError_t launch_histogram_finalize(hipStream_t s, const unsigned* counts, const float* limits,
                                     float alpha, unsigned m, unsigned bins, float* limits_out,
                                     float* pdf, float* ranks);
// step: the doubles from one sum to the next; rate, mean, sd may be null
hipError_t launch_batch_results(hipStream_t s, const unsigned long long* acc, const double* s1,
                                const double* s2, unsigned step, const unsigned* dims,
                                unsigned problems, unsigned max_dim, double count, double* rate,
                                double* mean, double* sd);
// the rows' means, or with var (mean is not written then) their variances
hipError_t launch_moments(hipStream_t s, const float* a, unsigned m, unsigned long long n,
                          unsigned ld, float* mean, float* var, void* scratch);
hipError_t launch_row_tree_sum(hipStream_t s, const float* a, unsigned rows, unsigned count,
                               unsigned local_n, unsigned long long row_stride, float* work,
                               float scale, float* out, unsigned long long out_stride);
hipError_t launch_sum_u32(hipStream_t s, const unsigned* v, unsigned n, unsigned long long* out);
hipError_t launch_sum_f64(hipStream_t s, const double* v, unsigned n, double* out);
// acor split over the chip (long series of few columns): the lengths, lags,
// offsets and slices of every level the estimator can reach, which follow
// from n, and the scratch they need.
constexpr unsigned kAcorMaxLevels = 32;  // halvings of a series of < 2^31 steps
constexpr unsigned kAcorPyramid = 11;    // levels per pyramid launch (2048 values per block)
constexpr unsigned kAcorWinMult = 5, kAcorMinLag = 10;
// the lag of the level after one of prev_n points with lag `lag` (acor.cl:143-168)
__host__ __device__ inline unsigned acor_next_lag(unsigned lag, unsigned prev_n) {
    if (lag * kAcorWinMult < prev_n) return lag;
    return prev_n / kAcorWinMult > kAcorMinLag ? prev_n / kAcorWinMult : kAcorMinLag;
}
struct AcorLevels {
    unsigned levels;
    unsigned n[kAcorMaxLevels], lag[kAcorMaxLevels], group[kAcorMaxLevels];
    size_t data[kAcorMaxLevels];
};
struct AcorSplit {
    AcorLevels t;
    unsigned total_groups, part_stride;
    size_t lev_stride, floats;  // floats: of the scratch
};
AcorSplit acor_split_plan(unsigned cols, unsigned max_stride, unsigned n, unsigned lag,
                          unsigned wgs);
// series (device) is only read; col_off and col_stride as acor_batch's, or
// null for one series of `dim` = `cols` columns.
hipError_t launch_acor_split(hipStream_t s, const float* series, const unsigned long long* col_off,
                             const unsigned* col_stride, unsigned dim, unsigned cols,
                             const AcorSplit& p, unsigned wgs, float* scratch, float* tau,
                             float* mean, float* sigma);
hipError_t launch_acor_batch(hipStream_t s, float* series, const unsigned long long* col_off,
                             const unsigned* col_stride, unsigned cols, unsigned n, unsigned lag,
                             unsigned wgs, float* scratch, unsigned scratch_per_dim, float* tau,
                             float* mean, float* sigma);
hipError_t launch_acor(hipStream_t s, float* series, unsigned dim, unsigned n, unsigned lag,
                       unsigned wgs, float* scratch, unsigned scratch_per_dim, float* tau,
                       float* mean, float* sigma);

}  // namespace bh
