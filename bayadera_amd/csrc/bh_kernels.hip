// Model-independent kernels of the HIP engine, compiled ahead of time for
// gfx950: walker initialisation, the dataset engine (min/max, histogram with
// LDS-privatised bins, pdf + bin ranks, FP64 mean/variance), the run-sampler
// accounting reductions and the autocorrelation estimator.
//
// Matrices are the reference's DIM x n column-major blocks (element (d, j)
// at a[j*ld + d]).  The dataset kernels map a block onto a tile of TM rows x
// TN columns (TM*TN its threads, TM the next power of two >= m, capped at 64
// rows per pass), so every thread owns one row and consecutive threads read
// consecutive addresses of a column.
#include <hip/hip_runtime.h>

#include <mutex>

#include "bh_kernels.hpp"
#include "bh_philox.hpp"

// The working memory of bh_dataset_variance_noalloc (the blocks' parts), for
// callers that cannot allocate.  Each GPU holds its own copy at
// its own address; host code reaches it only through the address that
// noalloc_scratch_init looks up (the array's name is a host-side stand-in).
static __device__ __align__(256) unsigned char scratch[bh::kNoAllocScratchBytes];

namespace bh {

namespace {
constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mu;
void* g_noalloc_ptr[kNoAllocMaxDevices];
}  // namespace

hipError_t noalloc_scratch_init(int device) {
    if (device < 0 || device >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (g_noalloc_ptr[device]) return hipSuccess;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(::scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_noalloc_ptr[device] = p;
    return hipSuccess;
}

hipError_t noalloc_scratch(int device, void** ptr) {
    if (device < 0 || device >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    *ptr = g_noalloc_ptr[device];
    return *ptr ? hipSuccess : hipErrorNotInitialized;
}

// --------------------------------------------------------------------------
// init_walkers (amd-gcn-mcmc-stretch.cl:138-159)
// --------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
init_walkers_kernel(unsigned seed, const float* __restrict__ limits, unsigned dim,
                    unsigned items, float* __restrict__ xs) {
    const unsigned g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= items) return;
    const bh_f32x4 u = bh_u01x4(
        bh_philox4x32_10(bh_u32x4{g, BH_CTR1_INIT, BH_CTR2_INIT, BH_CTR3}, seed, BH_KEY1_INIT));
    const float uu[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (unsigned m = 0; m < 4; ++m) {
        const unsigned i = 4 * g + m;
        const unsigned r = i % dim;
        const float lo = limits[2 * r], hi = limits[2 * r + 1];
        xs[i] = __builtin_fmaf(uu[m], hi, (1.0f - uu[m]) * lo);
    }
}

// Uniform direct sampler (uniform-sampler.cl:19-34): x = fma(u, hi-lo, lo).
__global__ void __launch_bounds__(256)
uniform_sample_kernel(unsigned seed, float lower, float upper, unsigned quads,
                      float* __restrict__ x) {
    const unsigned g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= quads) return;
    const bh_f32x4 u = bh_u01x4(
        bh_philox4x32_10(bh_u32x4{g, BH_CTR1_INIT, BH_CTR2_INIT, BH_CTR3}, seed, BH_KEY1_INIT));
    const float range = upper - lower;
    float4 v;
    v.x = __builtin_fmaf(u.x, range, lower);
    v.y = __builtin_fmaf(u.y, range, lower);
    v.z = __builtin_fmaf(u.z, range, lower);
    v.w = __builtin_fmaf(u.w, range, lower);
    reinterpret_cast<float4*>(x)[g] = v;
}

// Gaussian (Box-Muller), exponential and Erlang direct samplers
// (gaussian-sampler.cl:17-44, exponential-sampler.cl:16-29,
// erlang-sampler.cl:20-40); kinds as BH_DIRECT_* in bayadera_hip.h.
__global__ void __launch_bounds__(256)
direct_sample_kernel(int kind, unsigned seed, float p0, float p1, unsigned quads,
                     float* __restrict__ x) {
    const unsigned g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= quads) return;
    float r[4];
    if (kind == 3) {
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (unsigned i = 0; (float)i < p1; ++i) {
            const bh_f32x4 u = bh_u01x4(
                bh_philox4x32_10(bh_u32x4{g, BH_CTR1_INIT, BH_CTR2_INIT, i}, seed, BH_KEY1_INIT));
            acc[0] += logf(u.x);
            acc[1] += logf(u.y);
            acc[2] += logf(u.z);
            acc[3] += logf(u.w);
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) r[m] = -(acc[m] / p0);
    } else {
        const bh_f32x4 u = bh_u01x4(
            bh_philox4x32_10(bh_u32x4{g, BH_CTR1_INIT, BH_CTR2_INIT, BH_CTR3}, seed, BH_KEY1_INIT));
        if (kind == 1) {
            const float two_pi = 6.2831855f;
            const float ra = sqrtf(-2.0f * logf(u.y)), rb = sqrtf(-2.0f * logf(u.w));
            r[0] = __builtin_fmaf(sinf(two_pi * u.x) * ra, p1, p0);
            r[1] = __builtin_fmaf(cosf(two_pi * u.x) * ra, p1, p0);
            r[2] = __builtin_fmaf(sinf(two_pi * u.z) * rb, p1, p0);
            r[3] = __builtin_fmaf(cosf(two_pi * u.z) * rb, p1, p0);
        } else if (kind == 2) {
            const float c = -1.0f / p0;
            r[0] = c * logf(1.0f - u.x);
            r[1] = c * logf(1.0f - u.y);
            r[2] = c * logf(1.0f - u.z);
            r[3] = c * logf(1.0f - u.w);
        } else {
            const float range = p1 - p0;
            r[0] = __builtin_fmaf(u.x, range, p0);
            r[1] = __builtin_fmaf(u.y, range, p0);
            r[2] = __builtin_fmaf(u.z, range, p0);
            r[3] = __builtin_fmaf(u.w, range, p0);
        }
    }
    reinterpret_cast<float4*>(x)[g] = make_float4(r[0], r[1], r[2], r[3]);
}

// --------------------------------------------------------------------------
// Dataset engine (amd-gcn-estimate.cl; host amd_gcn.clj:137-214)
// --------------------------------------------------------------------------
__device__ __forceinline__ float ordered_min(float a, float b) { return b < a ? b : a; }
__device__ __forceinline__ float ordered_max(float a, float b) { return b > a ? b : a; }

// What the dataset kernels do with a thread's values: every column j of the
// thread's row r with j = blockIdx * tn + cl + k * gridDim * tn, eight loads in
// flight.  They are bound by HBM: 268 MB (2^24 x 4) in 39 to 44 us, 6.1 to 6.9
// TB/s; with one load in flight 53 to 56 us, the histogram 88.
template <class F>
__device__ __forceinline__ void row_values(const float* __restrict__ a, unsigned long long n,
                                           unsigned ld, unsigned r, unsigned tn, unsigned cl,
                                           F&& use) {
    constexpr unsigned U = 8;
    const unsigned long long stride = (unsigned long long)gridDim.x * tn;
    unsigned long long j = (unsigned long long)blockIdx.x * tn + cl;
    const float* p = a + j * ld + r;
    const size_t step = (size_t)stride * ld;
    for (; j + (U - 1) * stride < n; j += U * stride) {
        float x[U];
#pragma unroll
        for (unsigned u = 0; u < U; ++u) x[u] = p[u * step];
        p += U * step;
#pragma unroll
        for (unsigned u = 0; u < U; ++u) use(x[u]);
    }
    if (j < n) {
        // the last few together (past the end the first of them again, unused)
        float x[U];
#pragma unroll
        for (unsigned u = 0; u < U; ++u) x[u] = p[j + u * stride < n ? u * step : 0];
#pragma unroll
        for (unsigned u = 0; u < U; ++u)
            if (j + u * stride < n) use(x[u]);
    }
}

// The blocks' parts of a row by one wave, kMaxDatasetBlocks / 64 to a lane, in
// flight together: `get` loads part b, `use` takes it (a lane without a part
// loads its first again, unused).  With 256 threads and a tree over LDS a
// final kernel of 65,536 values took 2.7 to 3.3 us, now 2.3 to 2.9.
template <class T, class G, class F>
__device__ __forceinline__ void row_parts(unsigned blocks, G&& get, F&& use) {
    constexpr unsigned U = kMaxDatasetBlocks / 64;
    const unsigned b0 = threadIdx.x;
    if (b0 >= blocks) return;
    T v[U];
#pragma unroll
    for (unsigned u = 0; u < U; ++u) v[u] = get(b0 + u * 64 < blocks ? b0 + u * 64 : b0);
#pragma unroll
    for (unsigned u = 0; u < U; ++u)
        if (b0 + u * 64 < blocks) use(v[u]);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Per-block [min, max] of rows [r0, r0+tm) -> partial[(blk*m + r)*2 + {0,1}].
__global__ void __launch_bounds__(kDatasetThreads)
minmax_partial_kernel(const float* __restrict__ a, unsigned m, unsigned long long n,
                      unsigned ld, unsigned r0, unsigned tm, float* __restrict__ partial) {
    const unsigned t = threadIdx.x;
    const unsigned tn = kDatasetThreads / tm;
    const unsigned rl = t % tm, cl = t / tm;
    const unsigned r = r0 + rl;
    float lo = __builtin_inff(), hi = -__builtin_inff();
    if (r < m)
        row_values(a, n, ld, r, tn, cl, [&](float x) {
            lo = ordered_min(lo, x);
            hi = ordered_max(hi, x);
        });
    __shared__ float slo[kDatasetThreads], shi[kDatasetThreads];
    slo[t] = lo;
    shi[t] = hi;
    __syncthreads();
    for (unsigned s = tn / 2; s >= 1; s >>= 1) {
        if (cl < s) {
            slo[t] = ordered_min(slo[t], slo[t + s * tm]);
            shi[t] = ordered_max(shi[t], shi[t + s * tm]);
        }
        __syncthreads();
    }
    if (cl == 0 && r < m) {
        partial[((size_t)blockIdx.x * m + r) * 2] = slo[t];
        partial[((size_t)blockIdx.x * m + r) * 2 + 1] = shi[t];
    }
}

// One wave per row; clears the row's histogram counters.
__global__ void __launch_bounds__(64)
minmax_final_kernel(const float* __restrict__ partial, unsigned blocks, unsigned m, unsigned r0,
                    float* __restrict__ limits, unsigned* __restrict__ counts, unsigned bins) {
    const unsigned r = r0 + blockIdx.x;
    float lo = __builtin_inff(), hi = -__builtin_inff();
    row_parts<float2>(
        blocks,
        [&](unsigned b) {
            const float* p = partial + ((size_t)b * m + r) * 2;
            return float2{p[0], p[1]};
        },
        [&](float2 v) {
            lo = ordered_min(lo, v.x);
            hi = ordered_max(hi, v.y);
        });
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        lo = ordered_min(lo, __shfl_xor(lo, off, 64));
        hi = ordered_max(hi, __shfl_xor(hi, off, 64));
    }
    if (threadIdx.x == 0) {
        limits[2 * r] = lo;
        limits[2 * r + 1] = hi;
    }
    for (unsigned i = threadIdx.x; i < bins; i += 64) counts[(size_t)r * bins + i] = 0;
}

// bin = (uint)((x-lo)/(hi-lo)*bins) clamped to bins-1 (amd-gcn-estimate.cl:17-18);
// v_cvt_u32_f32 saturates negative values and NaN to 0.
__device__ __forceinline__ unsigned hist_clamp(float f, unsigned bins) {
    const unsigned b = f > 0.0f ? (f >= 4294967296.0f ? 0xffffffffu : (unsigned)f) : 0u;
    return b < bins ? b : bins - 1;
}
__device__ __forceinline__ unsigned hist_bin(float x, float lo, float hi, unsigned bins) {
    return hist_clamp((x - lo) / (hi - lo) * (float)bins, bins);
}
// The same bin with the row's width w = hi - lo divided by once: with y =
// RN(1 / w), q = RN(a y) and the exact remainder r = a - q w, RN(q + r y) is
// the correctly rounded quotient a / w (Markstein), as long as r is exact
// (2^-60 <= w <= 2^60, and a quotient below 2^-24 is in bin 0 either way).
// A quotient of 2 or more, also an infinite one whose remainder is not a
// number, is in the last bin without the correction.
__device__ __forceinline__ unsigned hist_bin_by(float x, float lo, float w, float y,
                                                unsigned bins) {
    const float a = x - lo;
    float q = a * y;
    const float c = __builtin_fmaf(__builtin_fmaf(-q, w, a), y, q);
    q = q >= 2.0f ? q : c;
    return hist_clamp(q * (float)bins, bins);
}

// LDS-privatised histogram of rows [r0, r0+tm): counts[r*bins + b] += n_rb.
// Each block keeps tm x bins counters in LDS (ds_add_u32), then adds its
// non-zero counters to global memory once.  A division per value, 2048 blocks
// adding their counters and one load in flight took 88 us for 2^24 x 4 values,
// now 44.
__global__ void __launch_bounds__(kDatasetThreads)
histogram_kernel(const float* __restrict__ a, unsigned m, unsigned long long n, unsigned ld,
                 unsigned r0, unsigned tm, const float* __restrict__ limits, unsigned bins,
                 unsigned* __restrict__ counts) {
    extern __shared__ unsigned hist[];  // tm * bins
    const unsigned t = threadIdx.x;
    const unsigned tn = kDatasetThreads / tm;
    const unsigned rl = t % tm, cl = t / tm;
    const unsigned r = r0 + rl;
    for (unsigned i = t; i < tm * bins; i += kDatasetThreads) hist[i] = 0;
    __syncthreads();
    if (r < m) {
        const float lo = limits[2 * r], hi = limits[2 * r + 1], w = hi - lo;
        unsigned* h = hist + rl * bins;
        if (w >= 0x1p-60f && w <= 0x1p60f) {
            const float y = 1.0f / w;
            row_values(a, n, ld, r, tn, cl,
                       [&](float x) { atomicAdd(&h[hist_bin_by(x, lo, w, y, bins)], 1u); });
        } else {
            row_values(a, n, ld, r, tn, cl,
                       [&](float x) { atomicAdd(&h[hist_bin(x, lo, hi, bins)], 1u); });
        }
    }
    __syncthreads();
    for (unsigned i = t; i < tm * bins; i += kDatasetThreads) {
        const unsigned c = hist[i];
        const unsigned rr = r0 + i / bins;
        if (c && rr < m) atomicAdd(&counts[(size_t)rr * bins + (i % bins)], c);
    }
}

// uint_to_real + bitonic_local (amd-gcn-estimate.cl:27-34, 95-123) for one
// row per block of `bins` threads: pdf = alpha/(hi-lo) * count, then the
// reference's bitonic network on (index, pdf) pairs, which orders the bins
// by descending pdf; ties keep the network's positional order.
__global__ void __launch_bounds__(1024)
histogram_finalize_kernel(const unsigned* __restrict__ counts, const float* __restrict__ limits,
                          float alpha, unsigned bins, float* __restrict__ limits_out,
                          float* __restrict__ pdf, float* __restrict__ ranks) {
    const unsigned r = blockIdx.x;
    const unsigned lid = threadIdx.x;
    if (lid < 2) limits_out[2 * r + lid] = limits[2 * r + lid];
    __shared__ float ax[2][1024], ay[2][1024];
    const float p = alpha / (limits[2 * r + 1] - limits[2 * r]) * (float)counts[(size_t)r * bins + lid];
    pdf[(size_t)r * bins + lid] = p;
    float vx = (float)lid, vy = p;
    // partners within the wave exchange by shuffles, the others through one of
    // two LDS areas in turn, a barrier each (33 of the 36 exchanges of 256
    // bins are within the wave)
    unsigned area = 0;
    for (unsigned length = 1; length < bins; length <<= 1) {
        const bool direction = (lid & (length << 1)) != 0;
        for (unsigned inc = length; inc > 0; inc >>= 1) {
            const unsigned j = lid ^ inc;
            float ox, oy;
            if (inc < 64) {
                ox = __shfl_xor(vx, (int)inc, 64);
                oy = __shfl_xor(vy, (int)inc, 64);
            } else {
                ax[area][lid] = vx;
                ay[area][lid] = vy;
                __syncthreads();
                ox = ax[area][j];
                oy = ay[area][j];
                area ^= 1;
            }
            const bool smaller = (vy < oy) || (oy == vy && j < lid);
            const bool swap = smaller ^ (j < lid) ^ direction;
            vx = swap ? ox : vx;
            vy = swap ? oy : vy;
        }
    }
    ranks[(size_t)r * bins + lid] = vx;
}

// Mean and population variance of every row in one pass over the data, in
// double (the reference's two passes round the mean and each difference to
// float, amd-gcn-estimate.cl:146-157).  A block sums its values' differences d
// from its own first value of the row and their squares; it leaves its mean and
// the sum of squares about it.  The blocks' parts are then combined about the
// mean of all (Chan, Golub, LeVeque).  A difference is exact in double where the
// two floats' exponents are at most 29 apart, and rounded once (2^-53 of it)
// otherwise.  With a block's value as its origin, cancellation multiplies the
// rounding errors, of the sums and of such differences, by at most the block's
// count of values: an origin far from the others is itself among the values
// whose variance is taken.  partial[(blk*m + r)*3]: the block's mean of
// row r, its sum of squares, its count.  With var 0 plain sums of the values:
// partial[blk*m + r].
template <int VAR>
__global__ void __launch_bounds__(kDatasetThreads)
moments_partial_kernel(const float* __restrict__ a, unsigned m, unsigned long long n,
                       unsigned ld, unsigned r0, unsigned tm, double* __restrict__ partial) {
    const unsigned t = threadIdx.x;
    const unsigned tn = kDatasetThreads / tm;
    const unsigned rl = t % tm, cl = t / tm;
    const unsigned r = r0 + rl;
    double s1 = 0.0, s2 = 0.0, origin = 0.0;
    unsigned long long count = 0;
    if (r < m) {
        if (VAR) {
            // (blockIdx * tn < n: the launch has no block without columns)
            origin = (double)a[(size_t)blockIdx.x * tn * ld + r];
            row_values(a, n, ld, r, tn, cl, [&](float x) {
                const double d = (double)x - origin;
                s1 += d;
                s2 = __builtin_fma(d, d, s2);
                ++count;
            });
        } else {
            row_values(a, n, ld, r, tn, cl, [&](float x) { s1 += (double)x; });
        }
    }
    __shared__ double ss[VAR ? 2 : 1][kDatasetThreads];
    __shared__ unsigned long long sc[VAR ? kDatasetThreads : 1];
    ss[0][t] = s1;
    if (VAR) {
        ss[VAR ? 1 : 0][t] = s2;
        sc[VAR ? t : 0] = count;
    }
    __syncthreads();
    for (unsigned k = tn / 2; k >= 1; k >>= 1) {
        if (cl < k) {
            ss[0][t] += ss[0][t + k * tm];
            if (VAR) {
                ss[VAR ? 1 : 0][t] += ss[VAR ? 1 : 0][t + k * tm];
                sc[VAR ? t : 0] += sc[VAR ? t + k * tm : 0];
            }
        }
        __syncthreads();
    }
    if (cl == 0 && r < m) {
        if (VAR) {
            double* o = partial + ((size_t)blockIdx.x * m + r) * 3;
            const double c = (double)sc[VAR ? t : 0], mean = ss[0][t] / c;
            o[0] = origin + mean;
            o[1] = __builtin_fma(-mean, ss[0][t], ss[VAR ? 1 : 0][t]);
            o[2] = c;
        } else {
            partial[(size_t)blockIdx.x * m + r] = ss[0][t];
        }
    }
}

// out[r] = (float)(sum of partials / n), or the variance of the combined parts
// (one wave per row).
template <int VAR>
__global__ void __launch_bounds__(64)
moments_final_kernel(const double* __restrict__ partial, unsigned blocks, unsigned m,
                     unsigned r0, double inv_n, float* __restrict__ out) {
    const unsigned r = r0 + blockIdx.x;
    double s = 0.0;
    if (!VAR) {
        row_parts<double>(
            blocks, [&](unsigned b) { return partial[(size_t)b * m + r]; },
            [&](double v) { s += v; });
        s = wave_sum(s);
        if (threadIdx.x == 0) out[r] = (float)(s * inv_n);
        return;
    }
    struct Part {
        double mean, sq, count;
    };
    const auto part = [&](unsigned b) {
        const double* p = partial + ((size_t)b * m + r) * 3;
        return Part{p[0], p[1], p[2]};
    };
    row_parts<Part>(blocks, part, [&](const Part& p) { s = __builtin_fma(p.mean, p.count, s); });
    const double mean = wave_sum(s) * inv_n;
    double q = 0.0;
    row_parts<Part>(blocks, part, [&](const Part& p) {
        const double d = p.mean - mean;
        q += __builtin_fma(d * d, p.count, p.sq);
    });
    q = wave_sum(q) * inv_n;
    if (threadIdx.x == 0) out[r] = (float)(q < 0.0 ? 0.0 : q);
}

// --------------------------------------------------------------------------
// Work-group tree of the reference (amd-gcn-mcmc-stretch.cl:5-29) for a
// group of lsize <= blockDim items, including the odd-size step: while i > 0,
// item i/2-1 first adds item i/2+i/2... (2*(i/2)) when i is odd, then every
// item l < i/2 adds item l+i/2.  lacc has blockDim floats.  Returns the total
// in every thread.
// --------------------------------------------------------------------------
__device__ float group_tree(float v, unsigned lsize, float* lacc) {
    const unsigned l = threadIdx.x;
    __syncthreads();
    if (l < lsize) lacc[l] = v;
    __syncthreads();
    float pacc = v;
    unsigned i = lsize;
    while (i > 0) {
        const bool odd = (i & 1u) && (l == (i >> 1) - 1);
        i >>= 1;
        if (odd) pacc += lacc[l + i + 1];
        if (l < i) {
            pacc += lacc[l + i];
            lacc[l] = pacc;
        }
        __syncthreads();
    }
    const float r = lacc[0];
    __syncthreads();
    return r;
}

// clojurecl's enq-reduce! along the columns of one row (sum_means_vertical +
// sum_reduction_horizontal, amd_gcn.clj:437-438): groups of local_n
// consecutive values reduce with the tree, the partials reduce again until
// one is left.  One block per row; work holds a row-sized scratch area.
__global__ void __launch_bounds__(kMaxGroupThreads)
row_tree_sum_kernel(const float* __restrict__ a, unsigned count, unsigned local_n,
                    unsigned long long row_stride, float* __restrict__ work, float scale,
                    float* __restrict__ out, unsigned long long out_stride) {
    __shared__ float lacc[kMaxGroupThreads];
    const unsigned row = blockIdx.x;
    const float* src = a + row * row_stride;
    float* w = work + (size_t)row * ((count + local_n - 1) / local_n + 1);
    unsigned c = count;
    bool first = true;
    while (true) {
        const unsigned groups = (c + local_n - 1) / local_n;
        for (unsigned g = 0; g < groups; ++g) {
            const unsigned start = g * local_n;
            const unsigned len = (c - start < local_n) ? c - start : local_n;
            const float v = threadIdx.x < len ? (first ? src[start + threadIdx.x] : w[start + threadIdx.x]) : 0.0f;
            const float s = group_tree(v, len, lacc);
            // all reads of this pass read indices >= start > g unless g = 0;
            // group 0 reads before writing slot 0
            if (threadIdx.x == 0) w[g] = s;
            __syncthreads();
        }
        first = false;
        if (groups == 1) break;
        c = groups;
    }
    if (threadIdx.x == 0) out[row * out_stride] = w[0] * scale;
}

__global__ void __launch_bounds__(256)
sum_u32_kernel(const unsigned* __restrict__ v, unsigned n, unsigned long long* __restrict__ out) {
    unsigned long long s = 0;
    for (unsigned i = threadIdx.x; i < n; i += blockDim.x) s += v[i];
    __shared__ unsigned long long ss[256];
    ss[threadIdx.x] = s;
    __syncthreads();
    for (unsigned k = 128; k >= 1; k >>= 1) {
        if (threadIdx.x < k) ss[threadIdx.x] += ss[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = ss[0];
}

__global__ void __launch_bounds__(256)
sum_f64_kernel(const double* __restrict__ v, unsigned n, double* __restrict__ out) {
    double s = 0.0;
    for (unsigned i = threadIdx.x; i < n; i += blockDim.x) s += v[i];
    __shared__ double ss[256];
    ss[threadIdx.x] = s;
    __syncthreads();
    for (unsigned k = 128; k >= 1; k >>= 1) {
        if (threadIdx.x < k) ss[threadIdx.x] += ss[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = ss[0];
}

// A batch's acceptance rates, means and population deviations from its sums;
// dimensions past a problem's own are 0.
__global__ void __launch_bounds__(256)
batch_results_kernel(const unsigned long long* __restrict__ acc, const double* __restrict__ s1,
                     const double* __restrict__ s2, unsigned step,
                     const unsigned* __restrict__ dims, unsigned problems, unsigned max_dim,
                     double count, double* __restrict__ rate, double* __restrict__ mean,
                     double* __restrict__ sd) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (rate && i < problems) rate[i] = (double)acc[i] / count;
    if (i >= (size_t)problems * max_dim) return;
    const unsigned p = (unsigned)(i / max_dim);
    double m = 0.0, v = 0.0;
    if (i - (size_t)p * max_dim < dims[p]) {
        m = s1[i * step] / count;
        v = s2[i * step] / count - __dmul_rn(m, m);
        v = v > 0.0 ? v : 0.0;
    }
    if (mean) mean[i] = m;
    if (sd) sd[i] = sqrt(v);
}

// --------------------------------------------------------------------------
// Autocorrelation (GCNAcorEngine.acor, amd_gcn.clj:216-267; amd-gcn-acor.cl)
// One block of wgs threads per dimension.  The reference's device-side
// enqueue recursion (acor.cl:143-168) becomes a loop; each of its
// work-groups becomes a pass of this block over a slice of the series with
// the same loads, lag sums and trees, so the float results are the same.
// series: n x dim (series[t*dim + d]), a device copy the kernel centres and
// pair-sums in place.  scratch: >= 2*(ceil(n/wgs)+1) floats per dimension.
// --------------------------------------------------------------------------
// One column: element t at col[t*cs]; its results go to tau[0], mean[0],
// sigma[0]; c0acc: scratch_per_dim floats of scratch.
__device__ __forceinline__ void acor_column(float* __restrict__ col, unsigned cs, unsigned n,
                                            unsigned lag, float inv_n, unsigned local_n_mean,
                                            float* __restrict__ c0acc, unsigned scratch_per_dim,
                                            float* __restrict__ tau, float* __restrict__ mean,
                                            float* __restrict__ sigma) {
    const unsigned wgs = blockDim.x;
    const unsigned l = threadIdx.x;
    __shared__ float lacc[kMaxGroupThreads];
    __shared__ float lm[2 * kMaxGroupThreads];
    float* dacc = c0acc + scratch_per_dim / 2;

    // mean: enq-reduce! with local (min(16,dim), wgs/that) along n, scal! 1/n
    {
        unsigned c = n;
        bool first = true;
        while (true) {
            const unsigned groups = (c + local_n_mean - 1) / local_n_mean;
            for (unsigned g = 0; g < groups; ++g) {
                const unsigned start = g * local_n_mean;
                const unsigned len = (c - start < local_n_mean) ? c - start : local_n_mean;
                float v = 0.0f;
                if (l < len) v = first ? col[(size_t)(start + l) * cs] : c0acc[start + l];
                const float s = group_tree(v, len, lacc);
                if (l == 0) c0acc[g] = s;
                __syncthreads();
            }
            first = false;
            if (groups == 1) break;
            c = groups;
        }
    }
    const float mu = c0acc[0] * inv_n;
    __syncthreads();
    for (unsigned t = l; t < n; t += wgs) col[(size_t)t * cs] -= mu;
    __syncthreads();

    // one acor_1d level (acor.cl:26-86) over gsize points at stride
    auto level = [&](unsigned stride, unsigned lg, unsigned gsize, unsigned lw) -> unsigned {
        const unsigned groups = (gsize + lw - 1) / lw;
        for (unsigned g = 0; g < groups; ++g) {
            const unsigned start = g * lw;
            const unsigned lsize = (gsize - start < lw) ? gsize - start : lw;
            const bool has_next = g + 1 < groups;
            __syncthreads();
            lm[l] = 0.0f;
            lm[l + wgs] = 0.0f;
            __syncthreads();
            if (l < lsize) {
                const unsigned gid = start + l;
                const bool compute = gid + lg < gsize;
                const bool load_lag = (l < lg) && has_next && (gid + lsize < gsize);
                lm[l] = compute ? col[(size_t)gid * stride] : 0.0f;
                lm[l + lsize] = load_lag ? col[(size_t)(gid + lsize) * stride] : 0.0f;
            }
            __syncthreads();
            float xv = 0.0f, xacc = 0.0f;
            if (l < lsize) {
                xv = lm[l];
                for (unsigned s = 0; s < lg; ++s) {
                    const unsigned idx = l + s + 1;
                    xacc += idx < 2 * lsize ? lm[idx] : 0.0f;
                }
                xacc = xv * __builtin_fmaf(2.0f, xacc, xv);
            }
            const float c0 = group_tree(xv * xv, lsize, lacc);
            const float dd = group_tree(xacc, lsize, lacc);
            if (l == 0) {
                c0acc[g] = c0;
                dacc[g] = dd;
            }
        }
        __syncthreads();
        return groups;
    };

    // sum_reduction_acor's reduction (acor.cl:88-130)
    auto reduce = [&](unsigned groups, float& c0, float& dd) {
        const unsigned lsize = groups < wgs ? groups : wgs;
        float a = 0.0f, b = 0.0f;
        if (l < lsize) {
            for (unsigned t = l; t < groups; t += lsize) {
                a += c0acc[t];
                b += dacc[t];
            }
        }
        c0 = group_tree(a, lsize, lacc);
        dd = group_tree(b, lsize, lacc);
    };

    unsigned groups = level(cs, lag, n, wgs);
    float c0, dd;
    reduce(groups, c0, dd);
    unsigned stride = 1, cur_lag = lag, prev_n = n;
    float orig_c0 = 0.0f, prev_c0 = 0.0f;
    while (true) {
        const float start_c0 = (stride == 1) ? c0 : orig_c0;
        const float tv = dd / ((stride == 1) ? c0 : prev_c0);
        const unsigned lag2 = acor_next_lag(cur_lag, prev_n);
        if (kAcorMinLag < lag2 && (float)lag2 < tv * (float)kAcorWinMult) {
            const unsigned n2 = prev_n / 2;
            const unsigned w2 = wgs < n2 ? wgs : n2;
            const size_t step = (size_t)stride * cs;
            __syncthreads();
            for (unsigned g = l; g < n2; g += wgs) col[2 * g * step] += col[(2 * (size_t)g + 1) * step];
            __syncthreads();
            groups = level((unsigned)(2 * step), lag2, n2, w2);
            float c0n, dn;
            reduce(groups, c0n, dn);
            orig_c0 = start_c0;
            prev_c0 = c0;
            c0 = c0n;
            dd = dn;
            stride *= 2;
            cur_lag = lag2;
            prev_n = n2;
        } else {
            if (l == 0) {
                const float scale = (float)stride * (float)(prev_n - lag2);
                tau[0] = dd * (float)(n - cur_lag) / (scale * start_c0);
                sigma[0] = sqrtf(dd / (scale * (float)n));
                mean[0] = mu;
            }
            break;
        }
    }
}

__global__ void __launch_bounds__(kMaxGroupThreads)
acor_kernel(float* __restrict__ series, unsigned dim, unsigned n, unsigned lag, float inv_n,
            unsigned local_n_mean, float* __restrict__ scratch, unsigned scratch_per_dim,
            float* __restrict__ tau, float* __restrict__ mean, float* __restrict__ sigma) {
    const unsigned d = blockIdx.x;
    acor_column(series + d, dim, n, lag, inv_n, local_n_mean,
                scratch + (size_t)d * scratch_per_dim, scratch_per_dim, tau + d, mean + d,
                sigma + d);
}

// Many series of n steps in one launch, one block per column: block b takes
// the column starting at series + col_off[b] with stride col_stride[b] (its
// series' dimension, which also sets the mean's reduction shape as in
// acor_kernel), results at index b.
__global__ void __launch_bounds__(kMaxGroupThreads)
acor_batch_kernel(float* __restrict__ series, const unsigned long long* __restrict__ col_off,
                  const unsigned* __restrict__ col_stride, unsigned n, unsigned lag, float inv_n,
                  float* __restrict__ scratch, unsigned scratch_per_dim, float* __restrict__ tau,
                  float* __restrict__ mean, float* __restrict__ sigma) {
    const unsigned b = blockIdx.x;
    const unsigned cs = col_stride[b];
    const unsigned wgs = blockDim.x;
    unsigned wgsm = cs < 16 ? cs : 16;
    if (wgs < wgsm) wgsm = wgs;
    acor_column(series + col_off[b], cs, n, lag, inv_n, wgs / wgsm,
                scratch + (size_t)b * scratch_per_dim, scratch_per_dim, tau + b, mean + b,
                sigma + b);
}

// --------------------------------------------------------------------------
// The same estimator split over the chip, for long series of few columns.
// acor_column walks a column's slices in turn with ~30 barriers each, on one
// compute unit per column: 5.0 ms for 112,640 steps x 2 (440 slices per
// level-0 pass), all of it latency.  Nothing in the walk depends on an
// earlier slice, and the only data-dependent choice, at which halving of the
// series to stop, can be made last: the lags and lengths of every level
// follow from n alone.  So the mean's trees, the series of every level (the
// pairwise sums are a pyramid over the centred series), the lag sums of
// every slice of every level, and the reduction over slices each become one
// launch over all slices, and one thread per column then picks the level.
// Levels past the one that is picked cost at most as much as level 0 does.
// Every sum keeps acor_column's shape, so the results are the same bit for
// bit.  5-6 launches, 0.046 ms for 112,640 x 2.
// --------------------------------------------------------------------------

// The column a block works on: of one n x dim series, or of many (col_off and
// col_stride as in acor_batch_kernel).
struct AcorCols {
    const unsigned long long* off;  // null: one series of `dim` columns
    const unsigned* stride;
    unsigned dim;
    __device__ __forceinline__ const float* base(const float* series, unsigned c) const {
        return series + (off ? off[c] : c);
    }
    __device__ __forceinline__ unsigned step(unsigned c) const { return off ? stride[c] : dim; }
};

__device__ __forceinline__ unsigned acor_mean_group(unsigned cs, unsigned wgs) {
    unsigned w = cs < 16 ? cs : 16;
    if (wgs < w) w = wgs;
    return wgs / w;
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// group_tree's sum of v[0 .. len) by `p` lanes of one wave (lane sl of them):
// at each level an item l < i/2 adds item l + i/2 (and item i/2 - 1 first the
// last one when i is odd), which only reads at or past i/2 and only writes
// before it.  Left in v[0].  All lanes of the wave call it together.
__device__ __forceinline__ void sub_tree(float* v, unsigned len, unsigned p, unsigned sl,
                                         unsigned longest) {
    unsigned i = len;
    for (unsigned m = longest; m > 1; m >>= 1) {  // as many levels as the longest of the wave
        wave_lds_sync();
        const bool odd = i & 1u;
        const unsigned h = i >> 1;
        for (unsigned l = sl; l < h; l += p) {
            float a = v[l];
            if (odd && l == h - 1) a += v[2 * h];
            v[l] = a + v[l + h];
        }
        if (i > 1) i = h;
    }
    wave_lds_sync();
}

// Lanes that share one group of at most `longest` values: a power of two.
__device__ __forceinline__ unsigned sub_lanes(unsigned longest) {
    unsigned p = 1;
    while (p < longest && p < 64) p <<= 1;
    return p;
}

// One pass of the mean's enq-reduce!: group g of local_n values (element t at
// src[t * cs]) to dst[g], 64 / p groups per wave and round.
__device__ __forceinline__ void acor_mean_pass(const float* __restrict__ src, size_t cs, unsigned count,
                                               unsigned local_n, float* __restrict__ dst,
                                               float* lds, unsigned wave, unsigned waves) {
    const unsigned lane = threadIdx.x & 63u;
    const unsigned p = sub_lanes(local_n), per = 64 / p, sl = lane % p;
    const unsigned groups = (count + local_n - 1) / local_n;
    float* v = lds + (lane / p) * local_n;
    for (unsigned g0 = wave * per; g0 < groups; g0 += waves * per) {
        const unsigned g = g0 + lane / p;
        unsigned len = 0;
        if (g < groups) {
            const unsigned start = g * local_n;
            len = count - start < local_n ? count - start : local_n;
            for (unsigned l = sl; l < len; l += p) v[l] = src[(size_t)(start + l) * cs];
        }
        sub_tree(v, len, p, sl, local_n);
        if (g < groups && sl == 0) dst[g] = v[0];
        wave_lds_sync();
    }
}

// LDS floats of one wave in acor_mean_pass: 64 / p groups of local_n.
constexpr unsigned kAcorMeanLds = kMaxGroupThreads;

// First pass of the mean over all columns: grid (blocks, columns).
__global__ void __launch_bounds__(256)
acor_mean_kernel(const float* __restrict__ series, AcorCols cols, unsigned n, unsigned wgs,
                 float* __restrict__ part, unsigned part_stride) {
    __shared__ float lds[4][kAcorMeanLds];
    const unsigned c = blockIdx.y, cs = cols.step(c), wave = threadIdx.x >> 6;
    acor_mean_pass(cols.base(series, c), cs, n, acor_mean_group(cs, wgs),
                   part + (size_t)c * part_stride, lds[wave], blockIdx.x * 4 + wave,
                   gridDim.x * 4);
}

// The passes that are left, one block per column, back and forth between the
// two halves of its scratch; mu[c] = the mean.
__global__ void __launch_bounds__(512)
acor_mean_finish_kernel(AcorCols cols, unsigned n, unsigned wgs, float inv_n,
                        float* __restrict__ part, unsigned part_stride, float* __restrict__ part2,
                        float* __restrict__ mu) {
    __shared__ float lds[8][kAcorMeanLds];
    const unsigned c = blockIdx.x, wave = threadIdx.x >> 6;
    const unsigned local_n = acor_mean_group(cols.step(c), wgs);
    unsigned count = (n + local_n - 1) / local_n;
    float* a = part + (size_t)c * part_stride;
    float* b = part2 + (size_t)c * part_stride;
    while (count > 1) {
        acor_mean_pass(a, 1, count, local_n, b, lds[wave], wave, 8);
        __syncthreads();
        float* t = a;
        a = b;
        b = t;
        count = (count + local_n - 1) / local_n;
    }
    if (threadIdx.x == 0) mu[c] = a[0] * inv_n;
}

// The series of levels l0 .. l0 + kAcorPyramid: a block takes 2^kAcorPyramid
// values of level l0 (of the series itself minus its mean when l0 is 0) and
// sums neighbours pairwise, level by level; level l holds n >> l values at
// lev + c * lev_stride + t.data[l].  An odd last value is dropped, as the
// halved series does.
__global__ void __launch_bounds__(256)
acor_pyramid_kernel(const float* __restrict__ series, AcorCols cols, AcorLevels t, unsigned l0,
                    const float* __restrict__ mu, float* __restrict__ lev, size_t lev_stride) {
    constexpr unsigned N = 1u << kAcorPyramid;
    __shared__ float buf[2][N];
    const unsigned c = blockIdx.y;
    float* out = lev + (size_t)c * lev_stride;
    const unsigned long long first = (unsigned long long)blockIdx.x * N;
    if (l0 == 0) {
        const float* src = cols.base(series, c);
        const unsigned cs = cols.step(c);
        const float m = mu[c];
#pragma unroll
        for (unsigned q = 0; q < N / 256; ++q) {
            const unsigned i = q * 256 + threadIdx.x;
            const unsigned long long g = first + i;
            float v = 0.0f;
            if (g < t.n[0]) {
                v = src[g * cs] - m;
                out[g] = v;
            }
            buf[0][i] = v;
        }
    } else {
#pragma unroll
        for (unsigned q = 0; q < N / 256; ++q) {
            const unsigned i = q * 256 + threadIdx.x;
            const unsigned long long g = first + i;
            buf[0][i] = g < t.n[l0] ? out[t.data[l0] + g] : 0.0f;
        }
    }
    unsigned which = 0;
    for (unsigned s = 1; s <= kAcorPyramid && l0 + s < t.levels; ++s) {
        __syncthreads();
        const unsigned l = l0 + s;
        const unsigned long long at = first >> s;
        for (unsigned i = threadIdx.x; i < (N >> s); i += 256) {
            const float v = buf[which][2 * i] + buf[which][2 * i + 1];
            buf[which ^ 1][i] = v;
            if (at + i < t.n[l]) out[t.data[l] + at + i] = v;
        }
        which ^= 1;
    }
}

// Two of group_tree's sums at once (they share the barriers); lacc has twice
// blockDim floats.
__device__ __forceinline__ void group_tree2(float& a, float& b, unsigned lsize, float* lacc) {
    const unsigned l = threadIdx.x;
    float* lb = lacc + blockDim.x;
    __syncthreads();
    if (l < lsize) {
        lacc[l] = a;
        lb[l] = b;
    }
    __syncthreads();
    unsigned i = lsize;
    while (i > 0) {
        const bool odd = (i & 1u) && (l == (i >> 1) - 1);
        i >>= 1;
        if (odd) {
            a += lacc[l + i + 1];
            b += lb[l + i + 1];
        }
        if (l < i) {
            a += lacc[l + i];
            b += lb[l + i];
            lacc[l] = a;
            lb[l] = b;
        }
        __syncthreads();
    }
    a = lacc[0];
    b = lb[0];
}

// acor_1d's sums (acor.cl:26-86) of one slice of one level of one column:
// grid (slices of all levels, columns), wgs threads.
__global__ void __launch_bounds__(kMaxGroupThreads)
acor_slice_kernel(AcorLevels t, const float* __restrict__ lev, size_t lev_stride,
                  float* __restrict__ sums, unsigned total_groups) {
    __shared__ float lacc[2 * kMaxGroupThreads];
    __shared__ float lm[2 * kMaxGroupThreads];
    const unsigned wgs = blockDim.x, l = threadIdx.x, c = blockIdx.y;
    unsigned k = 0;
    while (k + 1 < t.levels && blockIdx.x >= t.group[k + 1]) ++k;
    const unsigned gsize = t.n[k], lg = t.lag[k], lw = wgs < gsize ? wgs : gsize;
    const unsigned g = blockIdx.x - t.group[k];
    const float* col = lev + (size_t)c * lev_stride + t.data[k];
    const unsigned start = g * lw;
    const unsigned lsize = gsize - start < lw ? gsize - start : lw;
    const bool has_next = start + lw < gsize;
    lm[l] = 0.0f;
    lm[l + wgs] = 0.0f;
    __syncthreads();
    if (l < lsize) {
        const unsigned gid = start + l;
        const bool load_lag = (l < lg) && has_next && (gid + lsize < gsize);
        lm[l] = gid + lg < gsize ? col[gid] : 0.0f;
        lm[l + lsize] = load_lag ? col[gid + lsize] : 0.0f;
    }
    __syncthreads();
    float xv = 0.0f, xacc = 0.0f;
    if (l < lsize) {
        xv = lm[l];
        for (unsigned s = 0; s < lg; ++s) {
            const unsigned idx = l + s + 1;
            xacc += idx < 2 * lsize ? lm[idx] : 0.0f;
        }
        xacc = xv * __builtin_fmaf(2.0f, xacc, xv);
    }
    float c0 = xv * xv;
    group_tree2(c0, xacc, lsize, lacc);
    if (l == 0) {
        float* o = sums + (size_t)c * 2 * total_groups + blockIdx.x;
        o[0] = c0;
        o[total_groups] = xacc;
    }
}

// sum_reduction_acor's reduction (acor.cl:88-130) of every level, a wave per
// level, then the choice of the level and the results by one thread: one
// block of 4 waves per column.  LDS: 8 wgs floats.
__global__ void __launch_bounds__(256)
acor_choose_kernel(AcorLevels t, unsigned wgs, const float* __restrict__ sums,
                   unsigned total_groups, const float* __restrict__ mu, float* __restrict__ tau,
                   float* __restrict__ mean, float* __restrict__ sigma) {
    extern __shared__ float red[];
    __shared__ float lc0[kAcorMaxLevels], ldd[kAcorMaxLevels];
    const unsigned c = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    float* va = red + (size_t)wave * 2 * wgs;
    float* vb = va + wgs;
    for (unsigned k = wave; k < t.levels; k += 4) {
        const unsigned lw = wgs < t.n[k] ? wgs : t.n[k];
        const unsigned groups = (t.n[k] + lw - 1) / lw;
        const unsigned lsize = groups < wgs ? groups : wgs;
        const float* sa = sums + (size_t)c * 2 * total_groups + t.group[k];
        const float* sb = sa + total_groups;
        for (unsigned i = lane; i < lsize; i += 64) {
            float a = 0.0f, b = 0.0f;
            for (unsigned q = i; q < groups; q += lsize) {
                a += sa[q];
                b += sb[q];
            }
            va[i] = a;
            vb[i] = b;
        }
        sub_tree(va, lsize, 64, lane, lsize);
        sub_tree(vb, lsize, 64, lane, lsize);
        if (lane == 0) {
            lc0[k] = va[0];
            ldd[k] = vb[0];
        }
        wave_lds_sync();
    }
    __syncthreads();
    if (threadIdx.x) return;
    // acor_column's loop over levels, on the sums that are there already
    const unsigned n = t.n[0];
    unsigned stride = 1, cur_lag = t.lag[0], prev_n = n, k = 0;
    float c0 = lc0[0], dd = ldd[0], orig_c0 = 0.0f, prev_c0 = 0.0f;
    while (true) {
        const float start_c0 = (stride == 1) ? c0 : orig_c0;
        const float tv = dd / ((stride == 1) ? c0 : prev_c0);
        const unsigned lag2 = acor_next_lag(cur_lag, prev_n);
        if (k + 1 < t.levels && (float)lag2 < tv * (float)kAcorWinMult) {
            orig_c0 = start_c0;
            prev_c0 = c0;
            ++k;
            c0 = lc0[k];
            dd = ldd[k];
            stride *= 2;
            cur_lag = lag2;
            prev_n = t.n[k];
        } else {
            const float scale = (float)stride * (float)(prev_n - lag2);
            tau[c] = dd * (float)(n - cur_lag) / (scale * start_c0);
            sigma[c] = sqrtf(dd / (scale * (float)n));
            mean[c] = mu[c];
            break;
        }
    }
}

// --------------------------------------------------------------------------
// Streaming copy (the measured HBM denominator): each thread copies four
// 16-byte pieces, 4 KB apart within its block's 16 KB chunk, the four loads
// in flight before the stores; NT: non-temporal loads and stores.
// --------------------------------------------------------------------------
typedef float bh_copy_f4 __attribute__((ext_vector_type(4)));

template <bool NT>
__global__ void __launch_bounds__(256)
copy16_kernel(const bh_copy_f4* __restrict__ src, bh_copy_f4* __restrict__ dst,
              unsigned long long n16) {
    const unsigned long long base = (unsigned long long)blockIdx.x * 1024u + threadIdx.x;
    bh_copy_f4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const unsigned long long i = base + 256u * u;
        if (i < n16) v[u] = NT ? __builtin_nontemporal_load(src + i) : src[i];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const unsigned long long i = base + 256u * u;
        if (i < n16) {
            if (NT) __builtin_nontemporal_store(v[u], dst + i);
            else dst[i] = v[u];
        }
    }
}

// --------------------------------------------------------------------------
// Partners of a half-step found beforehand
// --------------------------------------------------------------------------
// A half-step of a large ensemble of small records is bound by its partners:
// each is a line from memory (5.2e10 a second) for 4 or 8 bytes of it.  They
// are sorted by region first, and read from LDS.
//
// Sorting: a work-group takes a tile's draws (the Philox words of the move, of
// which only the partner's counts here), counts them by region in LDS and puts
// each partner's first element at its place.  The order inside a region is
// whatever the counters gave; nothing depends on it.  Draws don't depend on
// positions, so one launch sorts for both half-steps of a step: 2 x 2^23 draws
// in 43 us against 27 for 2^23.
constexpr unsigned kPartnerThreads = 1024;
__global__ void __launch_bounds__(kPartnerThreads)
    partner_sort_kernel(unsigned K, unsigned dim, int partner_walker, uint2 seeds, uint2 odd_even,
                        unsigned step, unsigned bits, unsigned regions,
                        unsigned* __restrict__ entries, unsigned short* __restrict__ pos,
                        unsigned* __restrict__ starts) {
    const unsigned seed = blockIdx.y ? seeds.y : seeds.x;
    const unsigned odd_or_even = blockIdx.y ? odd_even.y : odd_even.x;
    entries += (size_t)blockIdx.y * K;
    pos += (size_t)blockIdx.y * K;
    starts += (size_t)blockIdx.y * gridDim.x * (regions + 1);
    constexpr unsigned N = kPartnerTile / kPartnerThreads;
    static_assert(kPartnerRegions == kPartnerThreads, "a thread per region");
    __shared__ unsigned count[kPartnerRegions], first[kPartnerRegions], waves[kPartnerThreads / 64];
    __shared__ unsigned sorted[kPartnerTile];
    const unsigned t = threadIdx.x, tile = blockIdx.x * kPartnerTile;
    const unsigned n = K - tile < kPartnerTile ? K - tile : kPartnerTile;
    count[t] = 0;
    __syncthreads();
    unsigned e[N], rank[N];
#pragma unroll
    for (unsigned i = 0; i < N; ++i) {
        const unsigned w = i * kPartnerThreads + t;
        const bh_u32x4 r = bh_philox4x32_10(bh_u32x4{tile + w, step, odd_or_even, BH_CTR3}, seed,
                                            BH_KEY1_STRETCH);
        const float u = bh_u01(r.x);
        if (partner_walker) {
            unsigned j = (unsigned)(u * (float)K);
            j = j < K ? j : K - 1;
            e[i] = j * dim;
        } else {
            e[i] = (unsigned)((u * (float)K) * (float)dim);
            if (e[i] >= K * dim) e[i] -= K * dim;
        }
        if (w < n) rank[i] = atomicAdd(&count[e[i] >> bits], 1u);
    }
    __syncthreads();
    const unsigned own = count[t];
    unsigned s = own;
#pragma unroll
    for (unsigned i = 1; i < 64; i *= 2) {
        const unsigned v = __shfl_up(s, i);
        if ((t & 63u) >= i) s += v;
    }
    if ((t & 63u) == 63u) waves[t >> 6] = s;
    __syncthreads();
    for (unsigned w = 0; w < (t >> 6); ++w) s += waves[w];
    first[t] = s - own;
    const unsigned tiles = gridDim.x;
    if (t < regions) starts[(size_t)t * tiles + blockIdx.x] = s - own;
    if (t == 0) starts[(size_t)regions * tiles + blockIdx.x] = n;
    __syncthreads();
#pragma unroll
    for (unsigned i = 0; i < N; ++i) {
        const unsigned w = i * kPartnerThreads + t;
        if (w < n) {
            const unsigned at = first[e[i] >> bits] + rank[i];
            sorted[at] = e[i];
            pos[tile + w] = (unsigned short)at;
        }
    }
    __syncthreads();
#pragma unroll
    for (unsigned i = 0; i < N; ++i) {
        const unsigned w = i * kPartnerThreads + t;
        if (w < n) entries[tile + w] = sorted[w];
    }
}

// Reading: a work-group's region of S lies in LDS (and the floats that a record
// starting at its end runs on to); `lanes` lanes take a tile's entries of it,
// and four tiles at a time so that the loads of eight groups of entries are in
// flight.
template <unsigned DIM>
__global__ void __launch_bounds__(kPartnerThreads)
    partner_read_kernel(const unsigned* __restrict__ entries, const unsigned* __restrict__ starts,
                        unsigned bits, unsigned lanes, unsigned tiles,
                        const float* __restrict__ S, unsigned total, float* __restrict__ g) {
    constexpr unsigned NS = 4, NU = 2;
    extern __shared__ __attribute__((aligned(16))) float region[];
    const unsigned t = threadIdx.x, r0 = blockIdx.x << bits;
    const unsigned n = total - r0 < (1u << bits) ? total - r0 : 1u << bits;
    // total is a multiple of 4 (K is one of 64), and so is n
    for (unsigned i = t * 4; i < n; i += kPartnerThreads * 4)
        *reinterpret_cast<float4*>(region + i) = *reinterpret_cast<const float4*>(S + r0 + i);
    if (t < DIM - 1) region[n + t] = S[r0 + n == total ? t : r0 + n + t];
    const unsigned* row = starts + (size_t)blockIdx.x * tiles;
    const unsigned lane = t & (lanes - 1), groups = kPartnerThreads / lanes;
    __syncthreads();
    for (unsigned t0 = t / lanes; t0 < tiles; t0 += NS * groups) {
        unsigned at[NS], end[NS], longest = 0;
#pragma unroll
        for (unsigned c = 0; c < NS; ++c) {
            const unsigned tile = t0 + c * groups;
            const bool has = tile < tiles;
            const unsigned lo = has ? row[tile] : 0, hi = has ? row[tiles + tile] : 0;
            at[c] = tile * kPartnerTile + lo;
            end[c] = tile * kPartnerTile + hi;
            longest = longest > hi - lo ? longest : hi - lo;
        }
        for (unsigned i0 = lane; i0 < longest; i0 += lanes * NU) {
            unsigned e[NS][NU];
#pragma unroll
            for (unsigned c = 0; c < NS; ++c)
#pragma unroll
                for (unsigned j = 0; j < NU; ++j) {
                    const unsigned i = at[c] + i0 + lanes * j;
                    e[c][j] = i < end[c] ? entries[i] : r0;
                }
#pragma unroll
            for (unsigned c = 0; c < NS; ++c)
#pragma unroll
                for (unsigned j = 0; j < NU; ++j) {
                    const unsigned i = at[c] + i0 + lanes * j;
                    if (i < end[c])
#pragma unroll
                        for (unsigned d = 0; d < DIM; ++d)
                            __builtin_nontemporal_store(region[e[c][j] - r0 + d],
                                                        g + (size_t)i * DIM + d);
                }
        }
    }
}

// --------------------------------------------------------------------------
// Host-side launchers (all on the caller's stream)
// --------------------------------------------------------------------------
static unsigned tile_rows(unsigned m) {
    unsigned tm = 1;
    while (tm < m && tm < 64) tm <<= 1;
    return tm;
}

// blocks of a dataset kernel over n columns in tiles of tm rows: each with
// columns of its own, a few rounds of its eight loads when there are enough
static unsigned dataset_blocks(unsigned long long n, unsigned tm) {
    const unsigned tn = kDatasetThreads / tm;
    const unsigned long long b = (n + tn - 1) / tn;
    return b < kMaxDatasetBlocks ? (unsigned)b : kMaxDatasetBlocks;
}

hipError_t launch_copy16(hipStream_t s, const void* src, void* dst, unsigned long long n16,
                         bool nt) {
    const unsigned long long blocks = (n16 + 1023) / 1024;
    if (blocks == 0) return hipSuccess;
    if (nt)
        copy16_kernel<true><<<(unsigned)blocks, 256, 0, s>>>(
            static_cast<const bh_copy_f4*>(src), static_cast<bh_copy_f4*>(dst), n16);
    else
        copy16_kernel<false><<<(unsigned)blocks, 256, 0, s>>>(
            static_cast<const bh_copy_f4*>(src), static_cast<bh_copy_f4*>(dst), n16);
    return hipGetLastError();
}

hipError_t launch_partner_sort(hipStream_t s, const PartnerPlan& p, int partner_walker,
                               const unsigned seeds[2], const unsigned odd_even[2],
                               unsigned step) {
    partner_sort_kernel<<<dim3(p.tiles(), 2), kPartnerThreads, 0, s>>>(
        p.K, p.dim, partner_walker, make_uint2(seeds[0], seeds[1]),
        make_uint2(odd_even[0], odd_even[1]), step, p.bits(), p.regions(), p.entries, p.pos,
        p.starts);
    return hipGetLastError();
}

hipError_t launch_partner_read(hipStream_t s, const PartnerPlan& p, int half, const float* S) {
    const unsigned regions = p.regions(), tiles = p.tiles();
    // twice the lanes cover a tile's entries of a region but for rare ones
    unsigned lanes = 64;
    while (lanes > 8 && lanes * regions > kPartnerTile) lanes /= 2;
    const unsigned* entries = p.entries + (size_t)half * p.K;
    const unsigned* starts = p.starts + (size_t)half * tiles * (regions + 1);
    const size_t lds = ((size_t)4 << p.bits()) + 16;
    if (p.dim == 1)
        partner_read_kernel<1><<<regions, kPartnerThreads, lds, s>>>(entries, starts, p.bits(), lanes,
                                                                     tiles, S, p.K, p.g);
    else
        partner_read_kernel<2><<<regions, kPartnerThreads, lds, s>>>(entries, starts, p.bits(), lanes,
                                                                     tiles, S, 2 * p.K, p.g);
    return hipGetLastError();
}

hipError_t launch_init_walkers(hipStream_t s, unsigned seed, const float* limits, unsigned dim,
                               unsigned walkers, float* xs) {
    const unsigned items = dim * walkers / 4;
    init_walkers_kernel<<<(items + 255) / 256, 256, 0, s>>>(seed, limits, dim, items, xs);
    return hipGetLastError();
}

hipError_t launch_uniform_sample(hipStream_t s, unsigned seed, float lo, float hi, unsigned quads,
                                 float* x) {
    uniform_sample_kernel<<<(quads + 255) / 256, 256, 0, s>>>(seed, lo, hi, quads, x);
    return hipGetLastError();
}

hipError_t launch_direct_sample(hipStream_t s, int kind, unsigned seed, float p0, float p1,
                                unsigned quads, float* x) {
    direct_sample_kernel<<<(quads + 255) / 256, 256, 0, s>>>(kind, seed, p0, p1, quads, x);
    return hipGetLastError();
}

size_t dataset_scratch_bytes(unsigned m, unsigned long long n) {
    (void)n;
    return (size_t)kMaxDatasetBlocks * m * 3 * sizeof(double) + 64;
}

hipError_t launch_min_max(hipStream_t s, const float* a, unsigned m, unsigned long long n,
                          unsigned ld, float* limits, unsigned* counts, unsigned bins,
                          void* scratch) {
    float* partial = (float*)scratch;
    for (unsigned r0 = 0; r0 < m; r0 += 64) {
        const unsigned rows = m - r0 < 64 ? m - r0 : 64;
        const unsigned tm = tile_rows(rows);
        const unsigned blocks = dataset_blocks(n, tm);
        minmax_partial_kernel<<<blocks, kDatasetThreads, 0, s>>>(a, m, n, ld, r0, tm, partial);
        minmax_final_kernel<<<rows, 64, 0, s>>>(partial, blocks, m, r0, limits, counts, bins);
    }
    return hipGetLastError();
}

hipError_t launch_histogram(hipStream_t s, const float* a, unsigned m, unsigned long long n,
                            unsigned ld, const float* limits, unsigned bins, unsigned* counts) {
    // rows per pass so that rows x bins counters take at most 32 KB of LDS
    unsigned per_pass = 8192 / bins;
    per_pass = per_pass < 1 ? 1 : (per_pass > 64 ? 64 : per_pass);
    for (unsigned r0 = 0; r0 < m; r0 += per_pass) {
        const unsigned rows = m - r0 < per_pass ? m - r0 : per_pass;
        const unsigned tm = tile_rows(rows);
        const unsigned blocks = dataset_blocks(n, tm);
        const size_t lds = (size_t)tm * bins * sizeof(unsigned);
        histogram_kernel<<<blocks, kDatasetThreads, lds, s>>>(a, m, n, ld, r0, tm, limits, bins,
                                                              counts);
    }
    return hipGetLastError();
}

hipError_t launch_histogram_finalize(hipStream_t s, const unsigned* counts, const float* limits,
                                     float alpha, unsigned m, unsigned bins, float* limits_out,
                                     float* pdf, float* ranks) {
    histogram_finalize_kernel<<<m, bins, 0, s>>>(counts, limits, alpha, bins, limits_out, pdf,
                                                 ranks);
    return hipGetLastError();
}

hipError_t launch_moments(hipStream_t s, const float* a, unsigned m, unsigned long long n,
                          unsigned ld, float* mean, float* var, void* scratch) {
    double* partial = (double*)scratch;
    const double inv_n = 1.0 / (double)n;
    for (unsigned r0 = 0; r0 < m; r0 += 64) {
        const unsigned rows = m - r0 < 64 ? m - r0 : 64;
        const unsigned tm = tile_rows(rows);
        const unsigned blocks = dataset_blocks(n, tm);
        if (var) {
            moments_partial_kernel<1>
                <<<blocks, kDatasetThreads, 0, s>>>(a, m, n, ld, r0, tm, partial);
            moments_final_kernel<1><<<rows, 64, 0, s>>>(partial, blocks, m, r0, inv_n, var);
        } else {
            moments_partial_kernel<0>
                <<<blocks, kDatasetThreads, 0, s>>>(a, m, n, ld, r0, tm, partial);
            moments_final_kernel<0><<<rows, 64, 0, s>>>(partial, blocks, m, r0, inv_n, mean);
        }
    }
    return hipGetLastError();
}

hipError_t launch_row_tree_sum(hipStream_t s, const float* a, unsigned rows, unsigned count,
                               unsigned local_n, unsigned long long row_stride, float* work,
                               float scale, float* out, unsigned long long out_stride) {
    // the tree of a group of local_n values needs local_n threads (local_n <= WGS)
    const unsigned threads = local_n > 256 ? local_n : 256;
    row_tree_sum_kernel<<<rows, threads, 0, s>>>(a, count, local_n, row_stride, work, scale, out,
                                                 out_stride);
    return hipGetLastError();
}

hipError_t launch_sum_u32(hipStream_t s, const unsigned* v, unsigned n, unsigned long long* out) {
    sum_u32_kernel<<<1, 256, 0, s>>>(v, n, out);
    return hipGetLastError();
}

hipError_t launch_sum_f64(hipStream_t s, const double* v, unsigned n, double* out) {
    sum_f64_kernel<<<1, 256, 0, s>>>(v, n, out);
    return hipGetLastError();
}

hipError_t launch_batch_results(hipStream_t s, const unsigned long long* acc, const double* s1,
                                const double* s2, unsigned step, const unsigned* dims,
                                unsigned problems, unsigned max_dim, double count, double* rate,
                                double* mean, double* sd) {
    const size_t n = (size_t)problems * max_dim;
    batch_results_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(
        acc, s1, s2, step, dims, problems, max_dim, count, rate, mean, sd);
    return hipGetLastError();
}

hipError_t launch_acor_batch(hipStream_t s, float* series, const unsigned long long* col_off,
                             const unsigned* col_stride, unsigned cols, unsigned n, unsigned lag,
                             unsigned wgs, float* scratch, unsigned scratch_per_dim, float* tau,
                             float* mean, float* sigma) {
    const float inv_n = (float)(1.0 / (double)n);
    acor_batch_kernel<<<cols, wgs, 0, s>>>(series, col_off, col_stride, n, lag, inv_n, scratch,
                                           scratch_per_dim, tau, mean, sigma);
    return hipGetLastError();
}

AcorSplit acor_split_plan(unsigned cols, unsigned max_stride, unsigned n, unsigned lag,
                          unsigned wgs) {
    AcorSplit p{};
    AcorLevels& t = p.t;
    size_t data = 0;
    unsigned nn = n, lg = lag, groups = 0;
    while (true) {
        const unsigned k = t.levels++, lw = wgs < nn ? wgs : nn;
        t.n[k] = nn;
        t.lag[k] = lg;
        t.data[k] = data;
        t.group[k] = groups;
        data += nn;
        groups += (nn + lw - 1) / lw;
        const unsigned lag2 = acor_next_lag(lg, nn);
        if (lag2 <= kAcorMinLag || t.levels == kAcorMaxLevels) break;
        lg = lag2;
        nn /= 2;
    }
    p.total_groups = groups;
    p.lev_stride = (data + 63) / 64 * 64;
    // the smallest group of the mean's reduction leaves the most partial sums
    unsigned w = max_stride < 16 ? max_stride : 16;
    if (wgs < w) w = wgs;
    p.part_stride = (n + wgs / w - 1) / (wgs / w);
    p.floats = (size_t)cols * (p.lev_stride + 2 * (size_t)p.part_stride + 2 * (size_t)groups + 1);
    return p;
}

hipError_t launch_acor_split(hipStream_t s, const float* series, const unsigned long long* col_off,
                             const unsigned* col_stride, unsigned dim, unsigned cols,
                             const AcorSplit& p, unsigned wgs, float* scratch, float* tau,
                             float* mean, float* sigma) {
    const AcorLevels& t = p.t;
    const unsigned n = t.n[0];
    const AcorCols c{col_off, col_stride, dim};
    const float inv_n = (float)(1.0 / (double)n);
    float* lev = scratch;
    float* part = lev + (size_t)cols * p.lev_stride;
    float* part2 = part + (size_t)cols * p.part_stride;
    float* sums = part2 + (size_t)cols * p.part_stride;
    float* mu = sums + (size_t)cols * 2 * p.total_groups;
    const unsigned waves = (p.part_stride + 3) / 4;
    const unsigned mb = waves < 1024 ? waves : 1024;
    acor_mean_kernel<<<dim3(mb, cols), 256, 0, s>>>(series, c, n, wgs, part, p.part_stride);
    acor_mean_finish_kernel<<<cols, 512, 0, s>>>(c, n, wgs, inv_n, part, p.part_stride, part2, mu);
    for (unsigned l0 = 0; l0 == 0 || l0 + 1 < t.levels; l0 += kAcorPyramid) {
        const unsigned blocks = (t.n[l0] + (1u << kAcorPyramid) - 1) >> kAcorPyramid;
        acor_pyramid_kernel<<<dim3(blocks, cols), 256, 0, s>>>(series, c, t, l0, mu, lev,
                                                               p.lev_stride);
    }
    acor_slice_kernel<<<dim3(p.total_groups, cols), wgs, 0, s>>>(t, lev, p.lev_stride, sums,
                                                                 p.total_groups);
    acor_choose_kernel<<<cols, 256, 8 * wgs * sizeof(float), s>>>(t, wgs, sums, p.total_groups, mu,
                                                                   tau, mean, sigma);
    return hipGetLastError();
}

hipError_t launch_acor(hipStream_t s, float* series, unsigned dim, unsigned n, unsigned lag,
                       unsigned wgs, float* scratch, unsigned scratch_per_dim, float* tau,
                       float* mean, float* sigma) {
    unsigned wgsm = dim < 16 ? dim : 16;
    if (wgs < wgsm) wgsm = wgs;
    const unsigned local_n_mean = wgs / wgsm;
    const float inv_n = (float)(1.0 / (double)n);
    acor_kernel<<<dim, wgs, 0, s>>>(series, dim, n, lag, inv_n, local_n_mean, scratch,
                                    scratch_per_dim, tau, mean, sigma);
    return hipGetLastError();
}

}  // namespace bh
