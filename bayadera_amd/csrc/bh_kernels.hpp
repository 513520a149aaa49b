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
// The partners of a step found beforehand, for halves S (K walkers of dim floats)
// past what the L2s hold: tiles of kPartnerTile walkers are sorted by the region
// of S their partner starts in (for both half-steps at once), a work-group with
// a region in LDS writes all tiles' partners from it in that order, and the move
// of a tile finds walker k's at its pos[k].
constexpr unsigned kPartnerTile = 8192;
constexpr unsigned kPartnerRegions = 1024;  // at most
constexpr unsigned kPartnerMaxDim = 2;
struct PartnerPlan {
    unsigned K, dim;
    unsigned* entries;    // [2][K] the tiles' partners' first elements, by region
    unsigned short* pos;  // [2][K] a walker's place in its tile's entries
    unsigned* starts;     // [2][regions + 1][tiles] a region's first entry in a tile
    float* g;             // [K][dim] the partners' records, in the order of entries

    unsigned long long floats() const { return (unsigned long long)K * dim; }
    unsigned tiles() const { return (K + kPartnerTile - 1) / kPartnerTile; }
    // floats of a region: 64 KiB, two work-groups to a compute unit, while that
    // makes 256 of them and a tile's entries of one a line; then 128 KiB (2^23
    // floats: 32 us to read against 43)
    unsigned bits() const { return floats() <= (1ull << 22) ? 14 : 15; }
    unsigned regions() const { return (unsigned)((floats() + (1ull << bits()) - 1) >> bits()); }
};
hipError_t launch_partner_sort(hipStream_t s, const PartnerPlan& p, int partner_walker,
                               const unsigned seeds[2], const unsigned odd_even[2], unsigned step);
// of half-step `half`, from the half S
hipError_t launch_partner_read(hipStream_t s, const PartnerPlan& p, int half, const float* S);
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
