// Model-dependent kernels of the HIP engine, compiled at run time by hipRTC
// together with the user's model source (the reference compiles its OpenCL
// engine the same way: amd_gcn.clj:573-631, with -DLOGFN/-DLOGPDF/-DLOGLIK,
// -DDIM and -DWGS).  The host defines:
//   WGS     reference work-group size: accounting groups and block size
//   DIM     model dimension (stretch kernels only)
//   LOGFN   mcmc log-density  REAL f(uint data_len, uint params_len, const REAL* params, uint dim, const REAL* x)
//   LOGPDF  log-density       (same signature)
//   LOGLIK  log-likelihood    REAL f(uint data_len, const REAL* data, uint dim, const REAL* x)
//
// Walker state is AoS, x[walker*DIM + d], the two half-ensembles contiguous,
// exactly the layout the reference hands across its boundary (DIM x W
// column-major).  The stretch move reads the partner walker's DIM floats as
// one contiguous run, so a random partner costs one cache line rather than
// DIM of them.

#include "bh_philox.hpp"

#define BH_PARTNER_FLAT 0
#define BH_PARTNER_WALKER 1

// The last six levels of the work-group tree inside one wave, for lane 0:
// level i adds lane t + i to lane t (i = 32, 16, 8, 4, 2, 1), the pairing
// of the reference's tree; v_permlane32_swap / v_permlane16_swap bring
// lanes t + 32 / t + 16 to lanes t < 32 / t < 16 (the builtins' second
// result), DPP row_shl:i lanes t + i within each 16-lane row.
__device__ __forceinline__ float bh_wave_tree_sum(float x) {
    const unsigned u = __float_as_uint(x);
    x = x + __uint_as_float(__builtin_amdgcn_permlane32_swap(u, u, false, false)[1]);
    const unsigned u16 = __float_as_uint(x);
    x = x + __uint_as_float(__builtin_amdgcn_permlane16_swap(u16, u16, false, false)[1]);
    x = x + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x108, 0xf, 0xf, false));
    x = x + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x104, 0xf, 0xf, false));
    x = x + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x102, 0xf, 0xf, false));
    x = x + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x101, 0xf, 0xf, false));
    return x;
}

#if defined(LOGFN) || defined(BH_GLM)

// A walker's DIM coordinates.  Walkers start at multiples of DIM floats from
// 256-byte aligned bases (and half-ensembles at K*DIM floats, K a multiple of
// 256), so for DIM % 4 == 0 they are 16-byte aligned: one 128-bit access per
// four coordinates.
__device__ __forceinline__ void bh_load_walker(const float* p, float (&v)[DIM]) {
    if constexpr (DIM % 4 == 0) {
        const float4* q = reinterpret_cast<const float4*>(__builtin_assume_aligned(p, 16));
#pragma unroll
        for (int i = 0; i < DIM / 4; ++i) {
            const float4 t = q[i];
            v[4 * i] = t.x;
            v[4 * i + 1] = t.y;
            v[4 * i + 2] = t.z;
            v[4 * i + 3] = t.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < DIM; ++i) v[i] = p[i];
    }
}

__device__ __forceinline__ void bh_store_walker(float* p, const float (&v)[DIM]) {
    if constexpr (DIM % 4 == 0) {
        float4* q = reinterpret_cast<float4*>(__builtin_assume_aligned(p, 16));
#pragma unroll
        for (int i = 0; i < DIM / 4; ++i)
            q[i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < DIM; ++i) p[i] = v[i];
    }
}

// The draws of the stretch move (amd-gcn-mcmc-stretch.cl:46-57):
//   counter {k, step, odd_or_even, 0xbeeff00d}, key {seed, 0xdecafbad}
//   z  = fma((a-2+1/a)*u1, u1, (2(1-1/a))*u1) + 1/a                     (:53-54)
// Partner: FLAT reads the complementary half at element offset
// j0 = (uint)((u0*K)*DIM) (:57), wrapping modulo K*DIM where the reference
// reads out of bounds; WALKER reads walker min((uint)(u0*K), K-1), i.e.
// element offset j*DIM.  Sets z and the partner's first element offset
// (< K*DIM); returns u2, the uniform of the accept test.
template <int PARTNER>
__device__ __forceinline__ float bh_stretch_draw(unsigned k, unsigned K, unsigned seed,
                                                 unsigned odd_or_even, unsigned step, float a,
                                                 float& z, unsigned& start) {
    const bh_f32x4 u = bh_u01x4(
        bh_philox4x32_10(bh_u32x4{k, step, odd_or_even, BH_CTR3}, seed, BH_KEY1_STRETCH));
    const float inv_a = 1.0f / a;
    const float ca = a - 2.0f + inv_a;
    const float cb = 2.0f * (1.0f - inv_a);
    z = __builtin_fmaf(ca * u.y, u.y, cb * u.y) + inv_a;
    if constexpr (PARTNER == BH_PARTNER_FLAT) {
        const unsigned total = K * DIM;
        unsigned e = (unsigned)((u.x * (float)K) * (float)DIM);
        if (e >= total) e -= total;
        start = e;
    } else {
        unsigned j = (unsigned)(u.x * (float)K);
        j = j < K ? j : K - 1;
        start = j * DIM;
    }
    return u.z;
}

// The proposal half of the stretch move (amd-gcn-mcmc-stretch.cl:46-65):
// the draws above, then Y = fma(z, Xk - Xj, Xj) (:64) with the partner's
// coordinates read from S (FLAT: element i at (start + i) mod K*DIM).
// Returns u2, the uniform of the accept test.
template <int PARTNER>
__device__ __forceinline__ float bh_propose(unsigned k, unsigned K, unsigned seed,
                                           unsigned odd_or_even, unsigned step, float a,
                                           const float* S, const float (&xk)[DIM],
                                           float (&y)[DIM], float& z) {
    unsigned e;
    const float u2 = bh_stretch_draw<PARTNER>(k, K, seed, odd_or_even, step, a, z, e);
    if constexpr (PARTNER == BH_PARTNER_FLAT) {
        const unsigned total = K * DIM;
#pragma unroll
        for (int i = 0; i < DIM; ++i) {
            const float xj = S[e];
            y[i] = __builtin_fmaf(z, xk[i] - xj, xj);
            e = (e + 1 == total) ? 0u : e + 1;
        }
    } else {
        float sj[DIM];
        bh_load_walker(S + e, sj);
#pragma unroll
        for (int i = 0; i < DIM; ++i) y[i] = __builtin_fmaf(z, xk[i] - sj[i], sj[i]);
    }
    return u2;
}

// z^(DIM-1) by repeated multiplication
__device__ __forceinline__ float bh_zpow(float z) {
    float zp = 1.0f;
#pragma unroll
    for (int i = 0; i < DIM - 1; ++i) zp *= z;
    return zp;
}

// Accounting of stretch_move_accu (amd-gcn-mcmc-stretch.cl:98-114) for the
// work-group of WGS threads holding group g: accept[g] += accepted count;
// means[groups*DIM*step + i*groups + g] += tree sum of coordinate i.
// Coordinates are staged BH_ACCU_CHUNK at a time, so that the staging area
// stays at BH_ACCU_CHUNK floats per thread whatever DIM is, and the
// work-group's waves take the trees of a chunk between them (wave w the
// coordinates w, w + WGS/64, ...).  What the sums are added to is read before
// the move (BhAccuOld): lane i of a wave holds the old value, later the new
// one, of the wave's i-th coordinate.  The kernel's end is then a staging, a
// barrier, two trees and a store; with one wave taking every tree and its
// first lane reading, adding and writing the sums one after the other, a
// half-step of 32,768 walkers x 7 took 6.96 us, now 4.54 (bound by the latency
// of the walker's and then the partner's loads).
#define BH_ACCU_CHUNK (DIM < 8 ? DIM : 8)
constexpr unsigned kBhWaves = WGS / 64;
constexpr unsigned kBhAccuChunks = (DIM + BH_ACCU_CHUNK - 1) / BH_ACCU_CHUNK;
constexpr unsigned kBhAccuPer = (BH_ACCU_CHUNK + kBhWaves - 1) / kBhWaves;  // of a chunk, per wave
constexpr unsigned kBhAccuRegs = (kBhAccuChunks * kBhAccuPer + 63) / 64;

// The accounting's LDS staging, one area for every instantiation of a
// half-step in a kernel.
struct BhAccuLds {
    float red[BH_ACCU_CHUNK * WGS];
    unsigned wave_counts[WGS / 64];
};

__device__ __forceinline__ BhAccuLds& bh_accu_lds() {
    __shared__ BhAccuLds st;
    return st;
}

// Sum of row c of the staged values (WGS of them) with the reference's
// work-group tree (amd-gcn-mcmc-stretch.cl:5-29 for power-of-two WGS: level i
// adds item l+i into item l, i = WGS/2 ... 1), by one wave: lane l takes the
// items l + 64j and their levels i >= 64 in the tree's pairing, then the
// levels 32 ... 1 with cross-lane moves.  Float addition is not associative,
// so the tree's shape is kept exactly.
__device__ __forceinline__ float bh_row_tree_sum(const float* red, unsigned c) {
    const float* p = red + c * WGS + (threadIdx.x & 63u);
    float x[kBhWaves];
#pragma unroll
    for (unsigned j = 0; j < kBhWaves; ++j) x[j] = p[64 * j];
#pragma unroll
    for (unsigned h = kBhWaves / 2; h >= 1; h >>= 1)
#pragma unroll
        for (unsigned j = 0; j < h; ++j) x[j] = x[j] + x[j + h];
    return __uint_as_float(
        __builtin_amdgcn_readfirstlane(__float_as_uint(bh_wave_tree_sum(x[0]))));
}

struct BhAccuOld {
    float m[kBhAccuRegs];
    unsigned accept;

    // the coordinate of this lane's item in register r, or DIM
    __device__ __forceinline__ static unsigned dim_of(unsigned r) {
        const unsigned it = r * 64 + (threadIdx.x & 63u);
        const unsigned c = (threadIdx.x >> 6) + it % kBhAccuPer * kBhWaves;
        const unsigned d = it / kBhAccuPer * BH_ACCU_CHUNK + c;
        return it < kBhAccuChunks * kBhAccuPer && c < BH_ACCU_CHUNK && d < DIM ? d : DIM;
    }
    __device__ __forceinline__ void load(unsigned g, unsigned groups, unsigned mstep,
                                         const unsigned* acc, const float* means) {
        accept = acc[g];
        const float* p = means + (size_t)groups * DIM * mstep + g;
#pragma unroll
        for (unsigned r = 0; r < kBhAccuRegs; ++r) {
            const unsigned d = dim_of(r);
            m[r] = d < DIM ? p[(size_t)d * groups] : 0.0f;
        }
    }
};

__device__ __forceinline__ void bh_accu(const float (&xk)[DIM], bool accepted, unsigned g,
                                        unsigned groups, unsigned mstep, unsigned* accept,
                                        float* means, BhAccuOld& old, BhAccuLds& lds) {
    const unsigned t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const unsigned long long b = __ballot(accepted);
    if (lane == 0) lds.wave_counts[wave] = (unsigned)__popcll(b);
#pragma unroll
    for (unsigned n = 0; n < kBhAccuChunks; ++n) {
        const unsigned d0 = n * BH_ACCU_CHUNK;
        if (n > 0) __syncthreads();  // the previous chunk's trees have read it
#pragma unroll
        for (unsigned c = 0; c < BH_ACCU_CHUNK; ++c)
            if (d0 + c < DIM) lds.red[c * WGS + t] = xk[d0 + c];
        __syncthreads();
#pragma unroll
        for (unsigned q = 0; q < kBhAccuPer; ++q) {
            const unsigned c = wave + q * kBhWaves;
            if (c < BH_ACCU_CHUNK && d0 + c < DIM) {
                const float sum = bh_row_tree_sum(lds.red, c);
                const unsigned it = n * kBhAccuPer + q;
                if (lane == it % 64) old.m[it / 64] += sum;
            }
        }
    }
    float* p = means + (size_t)groups * DIM * mstep + g;
#pragma unroll
    for (unsigned r = 0; r < kBhAccuRegs; ++r) {
        const unsigned d = BhAccuOld::dim_of(r);
        if (d < DIM) p[(size_t)d * groups] = old.m[r];
    }
    if (t == 0) {
        unsigned cnt = 0;
        for (unsigned w = 0; w < kBhWaves; ++w) cnt += lds.wave_counts[w];
        accept[g] = old.accept + cnt;
    }
}

#endif  // LOGFN || BH_GLM

#ifdef LOGFN

// The accept test of a proposal (:66-76).
__device__ __forceinline__ bool bh_accept(const float (&y)[DIM], float z, float u2, float beta,
                                          float (&xk)[DIM], float& lx, unsigned data_len,
                                          unsigned params_len, const float* params) {
    const float ly = LOGFN(data_len, params_len, params, DIM, y);
    const float q = __builtin_isfinite(ly) ? bh_zpow(z) * expf(beta * (ly - lx)) : 0.0f;
    const bool accepted = u2 <= q;
    if (accepted) {
#pragma unroll
        for (int i = 0; i < DIM; ++i) xk[i] = y[i];
        lx = ly;
    }
    return accepted;
}

// One walker's stretch move (amd-gcn-mcmc-stretch.cl:31-81).
//   counter {k, step, odd_or_even, 0xbeeff00d}, key {seed, 0xdecafbad}
//   z  = fma((a-2+1/a)*u1, u1, (2(1-1/a))*u1) + 1/a                     (:53-54)
//   Y  = fma(z, Xk - Xj, Xj)                                           (:64)
//   q  = isfinite(ly) ? z^(DIM-1) exp(beta (ly - lX)) : 0; accept iff u2 <= q (:68-71)
// Partner: FLAT reads the complementary half at element offset
// j0 = (uint)((u0*K)*DIM) (:57), wrapping modulo K*DIM where the reference
// reads out of bounds; WALKER reads walker min((uint)(u0*K), K-1).
// xk holds the walker's coordinates on entry and its new ones on exit.
template <int PARTNER>
__device__ __forceinline__ bool bh_stretch_walker(unsigned k, unsigned K, unsigned seed,
                                                  unsigned odd_or_even, unsigned step, float a,
                                                  float beta, const float* S,
                                                  float (&xk)[DIM], float& lx,
                                                  unsigned data_len, unsigned params_len,
                                                  const float* params) {
    float y[DIM];
    float z;
    const float u2 = bh_propose<PARTNER>(k, K, seed, odd_or_even, step, a, S, xk, y, z);
    return bh_accept(y, z, u2, beta, xk, lx, data_len, params_len, params);
}

// The modules of a model: its per-half-step kernels, and on their own (a user's
// density is compiled into each kernel) the resident and the batched ones.
#if !defined(BH_RESIDENT) && !defined(BH_BATCH)
// logfn kernel (amd-gcn-mcmc-stretch.cl:161-167): res[w] = LOGFN(x + DIM*w).
extern "C" __global__ void __launch_bounds__(WGS)
bh_logfn(unsigned data_len, unsigned params_len, const float* __restrict__ params,
         const float* __restrict__ x, float* __restrict__ res, unsigned n) {
    const unsigned w = blockIdx.x * WGS + threadIdx.x;
    if (w < n) res[w] = LOGFN(data_len, params_len, params, DIM, x + (size_t)w * DIM);
}

// One half-step over K walkers, one thread per walker, WGS walkers per block
// (stretch_move_bare / stretch_move_accu, amd-gcn-mcmc-stretch.cl:83-134).
// The walker's own record and log density are read and written once per
// half-step: streamed with non-temporal loads and stores, so that the
// caches keep the complementary half, which is read at random.
__device__ __forceinline__ void bh_load_walker_nt(const float* p, float (&v)[DIM]) {
    if constexpr (DIM % 4 == 0) {
        typedef float bh_f4 __attribute__((ext_vector_type(4)));
        const bh_f4* q = reinterpret_cast<const bh_f4*>(__builtin_assume_aligned(p, 16));
#pragma unroll
        for (int i = 0; i < DIM / 4; ++i) {
            const bh_f4 t = __builtin_nontemporal_load(q + i);
            v[4 * i] = t.x;
            v[4 * i + 1] = t.y;
            v[4 * i + 2] = t.z;
            v[4 * i + 3] = t.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < DIM; ++i) v[i] = __builtin_nontemporal_load(p + i);
    }
}

__device__ __forceinline__ void bh_store_walker_nt(float* p, const float (&v)[DIM]) {
    if constexpr (DIM % 4 == 0) {
        typedef float bh_f4 __attribute__((ext_vector_type(4)));
        bh_f4* q = reinterpret_cast<bh_f4*>(__builtin_assume_aligned(p, 16));
#pragma unroll
        for (int i = 0; i < DIM / 4; ++i)
            __builtin_nontemporal_store(bh_f4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]},
                                        q + i);
    } else {
#pragma unroll
        for (int i = 0; i < DIM; ++i) __builtin_nontemporal_store(v[i], p + i);
    }
}

// Staged half-step for DIM >= 8: a thread's own record and its partner's
// span DIM/4 16-byte pieces (DIM floats when DIM % 4 != 0), and reading them
// thread by thread makes every load instruction of a wave touch up to 64
// separate lines (4 to 16 times the requests of a contiguous read).  Here
// the block's WGS records, contiguous in X, are read and written as
// consecutive pieces by consecutive threads, and each partner's pieces by
// consecutive threads too; an LDS tile transposes between that order and
// one record per thread.  Rows of the tile are an odd number of 16-byte
// units (odd number of floats for DIM % 4 != 0) apart, so threads reading
// consecutive rows hit distinct banks.  Arithmetic and results are those of
// the thread-per-record path.
#define BH_STAGE_STRIDE \
    (DIM % 4 == 0 ? ((DIM / 4) % 2 ? DIM : DIM + 4) : (DIM % 2 ? DIM : DIM + 1))
#define BH_STAGE (DIM >= 8 && WGS * BH_STAGE_STRIDE * 4 <= 49152)
constexpr int kBhStageStride = BH_STAGE_STRIDE;
constexpr bool kBhStage = BH_STAGE;

// One LDS staging area for every instantiation of the staged half-step in a
// kernel (a __shared__ array declared in each instantiation would be
// allocated once per instantiation, halving the blocks that fit on a CU).
struct BhStageLds {
    float tile[kBhStage ? WGS * kBhStageStride : 1];
    unsigned pstart[WGS];
    unsigned long long acc_mask[WGS / 64];
};

__device__ __forceinline__ BhStageLds& bh_stage_lds() {
    __shared__ __attribute__((aligned(16))) BhStageLds st;
    return st;
}

template <bool ACCU, int PARTNER>
__device__ __forceinline__ void bh_stretch_half_staged(unsigned seed, unsigned odd_or_even,
                                                       unsigned data_len, unsigned params_len,
                                                       const float* __restrict__ params,
                                                       const float* __restrict__ S,
                                                       float* __restrict__ X,
                                                       float* __restrict__ logfn_X, float a,
                                                       float beta, unsigned step, unsigned K,
                                                       unsigned* __restrict__ accept,
                                                       float* __restrict__ means,
                                                       float* __restrict__ out) {
    typedef float bh_f4 __attribute__((ext_vector_type(4)));
    constexpr int ST = kBhStageStride;
    constexpr bool V4 = DIM % 4 == 0;                     // records as 16-byte pieces
    constexpr bool SV4 = V4 && PARTNER == BH_PARTNER_WALKER;  // partners too
    constexpr int NP = V4 ? DIM / 4 : DIM;                 // pieces per record
    BhStageLds& lds = bh_stage_lds();
    float* tile = lds.tile;
    unsigned* pstart = lds.pstart;
    unsigned long long* acc_mask = lds.acc_mask;
    const unsigned t = threadIdx.x;
    const unsigned k = blockIdx.x * WGS + t;
    float* xb = X + (size_t)blockIdx.x * WGS * DIM;
    BhAccuOld old;
    if (ACCU) old.load(blockIdx.x, gridDim.x, step, accept, means);
    // own records: piece g = i*WGS + t is piece g % NP of record g / NP
    float xs[NP * (V4 ? 4 : 1)];
    if constexpr (V4) {
        const bh_f4* q = reinterpret_cast<const bh_f4*>(__builtin_assume_aligned(xb, 16));
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const bh_f4 v = __builtin_nontemporal_load(q + i * WGS + t);
            xs[4 * i] = v.x;
            xs[4 * i + 1] = v.y;
            xs[4 * i + 2] = v.z;
            xs[4 * i + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < NP; ++i) xs[i] = __builtin_nontemporal_load(xb + i * WGS + t);
    }
    float lx = __builtin_nontemporal_load(logfn_X + k);
    float z;
    unsigned e;
    const float u2 = bh_stretch_draw<PARTNER>(k, K, seed, odd_or_even, step, a, z, e);
    pstart[t] = e;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const unsigned g = i * WGS + t, w = g / NP, c = g % NP;
        if constexpr (V4) {
            *reinterpret_cast<bh_f4*>(&tile[w * ST + 4 * c]) =
                bh_f4{xs[4 * i], xs[4 * i + 1], xs[4 * i + 2], xs[4 * i + 3]};
        } else {
            tile[w * ST + c] = xs[i];
        }
    }
    __syncthreads();
    // partner pieces, consecutive threads on consecutive pieces of a partner
    constexpr int NPS = SV4 ? DIM / 4 : DIM;
    float ss[DIM];
    if constexpr (SV4) {
        const bh_f4* q = reinterpret_cast<const bh_f4*>(__builtin_assume_aligned(S, 16));
#pragma unroll
        for (int i = 0; i < NPS; ++i) {
            const unsigned g = i * WGS + t, w = g / NPS, c = g % NPS;
            const bh_f4 v = q[pstart[w] / 4 + c];
            ss[4 * i] = v.x;
            ss[4 * i + 1] = v.y;
            ss[4 * i + 2] = v.z;
            ss[4 * i + 3] = v.w;
        }
    } else {
        const unsigned total = K * DIM;
#pragma unroll
        for (int i = 0; i < NPS; ++i) {
            const unsigned g = i * WGS + t, w = g / NPS, c = g % NPS;
            unsigned idx = pstart[w] + c;
            if (PARTNER == BH_PARTNER_FLAT && idx >= total) idx -= total;
            ss[i] = S[idx];
        }
    }
    float xk[DIM];
#pragma unroll
    for (int i = 0; i < DIM; ++i) xk[i] = tile[t * ST + i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NPS; ++i) {
        const unsigned g = i * WGS + t, w = g / NPS, c = g % NPS;
        if constexpr (SV4) {
            *reinterpret_cast<bh_f4*>(&tile[w * ST + 4 * c]) =
                bh_f4{ss[4 * i], ss[4 * i + 1], ss[4 * i + 2], ss[4 * i + 3]};
        } else {
            tile[w * ST + c] = ss[i];
        }
    }
    __syncthreads();
    float y[DIM];
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
        const float xj = tile[t * ST + i];
        y[i] = __builtin_fmaf(z, xk[i] - xj, xj);
    }
    const float ly = LOGFN(data_len, params_len, params, DIM, y);
    const float qv = __builtin_isfinite(ly) ? bh_zpow(z) * expf(beta * (ly - lx)) : 0.0f;
    const bool accepted = u2 <= qv;
    if (accepted) {
#pragma unroll
        for (int i = 0; i < DIM; ++i) {
            xk[i] = y[i];
            tile[t * ST + i] = y[i];
        }
        lx = ly;
    } else if (out) {
#pragma unroll
        for (int i = 0; i < DIM; ++i) tile[t * ST + i] = xk[i];
    }
    // where any of a wave's walkers moved, all their log densities: whole lines of
    // 32 take less than masked ones (2^21 x 16, us per half-step: 70.7 -> 69.7)
    const unsigned long long m = __ballot(accepted);
    if (m) __builtin_nontemporal_store(lx, logfn_X + k);
    if ((t & 63u) == 0) acc_mask[t >> 6] = m;
    __syncthreads();
    // accepted records back to X as consecutive pieces
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const unsigned g = i * WGS + t, w = g / NP, c = g % NP;
        if ((acc_mask[w >> 6] >> (w & 63u)) & 1ull) {
            if constexpr (V4) {
                bh_f4* q = reinterpret_cast<bh_f4*>(__builtin_assume_aligned(xb, 16));
                __builtin_nontemporal_store(*reinterpret_cast<const bh_f4*>(&tile[w * ST + 4 * c]),
                                            q + g);
            } else {
                __builtin_nontemporal_store(tile[w * ST + c], xb + g);
            }
        }
    }
    if (out) {
        float* ob = out + (size_t)blockIdx.x * WGS * DIM;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const unsigned g = i * WGS + t, w = g / NP, c = g % NP;
            if constexpr (V4) {
                bh_f4* q = reinterpret_cast<bh_f4*>(__builtin_assume_aligned(ob, 16));
                __builtin_nontemporal_store(*reinterpret_cast<const bh_f4*>(&tile[w * ST + 4 * c]),
                                            q + g);
            } else {
                __builtin_nontemporal_store(tile[w * ST + c], ob + g);
            }
        }
    }
    if (ACCU)
        bh_accu(xk, accepted, blockIdx.x, gridDim.x, step, accept, means, old, bh_accu_lds());
}

template <bool ACCU, int PARTNER>
__device__ __forceinline__ void bh_stretch_half(unsigned seed, unsigned odd_or_even,
                                                unsigned data_len, unsigned params_len,
                                                const float* __restrict__ params,
                                                const float* __restrict__ S, float* __restrict__ X,
                                                float* __restrict__ logfn_X, float a, float beta,
                                                unsigned step, unsigned K,
                                                unsigned* __restrict__ accept,
                                                float* __restrict__ means,
                                                float* __restrict__ out) {
    if constexpr (kBhStage) {
        bh_stretch_half_staged<ACCU, PARTNER>(seed, odd_or_even, data_len, params_len, params, S,
                                              X, logfn_X, a, beta, step, K, accept, means, out);
        return;
    } else {
        const unsigned k = blockIdx.x * WGS + threadIdx.x;
        float xk[DIM];
        float* xp = X + (size_t)k * DIM;
        bh_load_walker_nt(xp, xk);
        float lx = __builtin_nontemporal_load(logfn_X + k);
        BhAccuOld old;
        if (ACCU) old.load(blockIdx.x, gridDim.x, step, accept, means);
        const bool accepted = bh_stretch_walker<PARTNER>(k, K, seed, odd_or_even, step, a, beta, S,
                                                         xk, lx, data_len, params_len, params);
        // A line holds several of these small records, and whole lines take less
        // than masked ones: from so many of a wave's walkers moved on, all are
        // written (us per half-step with 60%, 20% and none moved, the moved ones
        // written against all: 2^22 x 1 69 68 60 / 63 63 65, 2^22 x 4 101 95 83 /
        // 96 96 97, 2^22 x 7 146 131 106 / 137 137 138).  A record of 8
        // coordinates or more that is too wide to stage fills lines of its own:
        // the moved ones only (2^18 walkers x 48 coordinates, 15% moved, 101 -> 62).
        const unsigned moved = (unsigned)__popcll(__ballot(accepted));
        if ((DIM < 8 && moved >= 3 + DIM * 5 / 2) || accepted) bh_store_walker_nt(xp, xk);
        if (moved >= 5 || accepted) __builtin_nontemporal_store(lx, logfn_X + k);
        if (DIM < 8 && out) bh_store_walker_nt(out + (size_t)k * DIM, xk);
        if (ACCU)
            bh_accu(xk, accepted, blockIdx.x, gridDim.x, step, accept, means, old, bh_accu_lds());
    }
}

// With `out` the half's records after the move go there too: a sample of an
// ensemble is written by its last step instead of being copied from it (2^21
// x 16 walkers a half: the copy read and wrote 2 x 134 MB, 100 us for both
// halves; writing alone 43).  A record that does not move then stays in registers
// while the density runs, which costs wide ones a wave on each SIMD: past 12
// coordinates the moves that write a sample are a kernel of their own (2^19
// walkers a half, correlated Gaussian, us without a sample: 28 coordinates 64 ->
// 57, 38 167 -> 98; 9 and 12 take 1% less as one kernel).  Records of 8 and more
// that are not staged have none: a thread's own stores of 48 coordinates take
// 152 us with 2^18 walkers, the move and a copy 80.
#define BH_BARE_KERNEL(NAME, OUT)                                                                 \
    extern "C" __global__ void __launch_bounds__(WGS) NAME(                                       \
        unsigned seed, unsigned odd_or_even, unsigned data_len, unsigned params_len,              \
        const float* __restrict__ params, const float* __restrict__ S, float* __restrict__ X,     \
        float* __restrict__ logfn_X, float a, float beta, unsigned step, unsigned K, int partner, \
        float* __restrict__ out) {                                                                \
        if (partner == BH_PARTNER_FLAT)                                                           \
            bh_stretch_half<false, BH_PARTNER_FLAT>(seed, odd_or_even, data_len, params_len,      \
                                                    params, S, X, logfn_X, a, beta, step, K,      \
                                                    nullptr, nullptr, (OUT) ? out : nullptr);     \
        else                                                                                      \
            bh_stretch_half<false, BH_PARTNER_WALKER>(seed, odd_or_even, data_len, params_len,    \
                                                      params, S, X, logfn_X, a, beta, step, K,    \
                                                      nullptr, nullptr, (OUT) ? out : nullptr);   \
    }
BH_BARE_KERNEL(bh_stretch_move_bare, DIM <= 12)
#if DIM > 12 && BH_STAGE
BH_BARE_KERNEL(bh_stretch_move_bare_out, true)
#endif
#undef BH_BARE_KERNEL

extern "C" __global__ void __launch_bounds__(WGS)
bh_stretch_move_accu(unsigned seed, unsigned odd_or_even, unsigned data_len,
                     unsigned params_len, const float* __restrict__ params,
                     const float* __restrict__ S, float* __restrict__ X,
                     float* __restrict__ logfn_X, unsigned* __restrict__ accept,
                     float* __restrict__ means, float a, unsigned step, unsigned K,
                     int partner) {
    if (partner == BH_PARTNER_FLAT)
        bh_stretch_half<true, BH_PARTNER_FLAT>(seed, odd_or_even, data_len, params_len, params, S,
                                               X, logfn_X, a, 1.0f, step, K, accept, means, nullptr);
    else
        bh_stretch_half<true, BH_PARTNER_WALKER>(seed, odd_or_even, data_len, params_len, params,
                                                 S, X, logfn_X, a, 1.0f, step, K, accept, means, nullptr);
}

#if DIM <= 2
// A half-step whose partners were found beforehand (see partner_sort_kernel in
// bh_kernels.hip): a work-group takes a tile of kBhFoundTile walkers, puts the
// tile's partners in LDS as they come (found) and reads walker k's at pos[k].
// Its arithmetic is bh_stretch_move_bare's.  Bound by its traffic: 34 us for 2^23
// walkers of one coordinate, 185 MB, 5.4 TB/s; reading the partners from memory
// by pos takes 42 to 60, a line's lookup in the L2 each.  Tiles of 16384 take 36,
// and leave records of two coordinates one work-group to a compute unit.
constexpr unsigned kBhFoundTile = 8192, kBhFoundThreads = 1024;
extern "C" __global__ void __launch_bounds__(kBhFoundThreads)
bh_stretch_move_found(unsigned seed, unsigned odd_or_even, unsigned data_len, unsigned params_len,
                      const float* __restrict__ params, const float* __restrict__ found,
                      const unsigned short* __restrict__ pos, float* __restrict__ X,
                      float* __restrict__ logfn_X, float a, float beta, unsigned step, unsigned K,
                      float* __restrict__ out) {
    __shared__ __attribute__((aligned(16))) float partners[kBhFoundTile * DIM];
    const unsigned t = threadIdx.x, tile = blockIdx.x * kBhFoundTile;
    const unsigned n = K - tile < kBhFoundTile ? K - tile : kBhFoundTile;
    // the next walker's record, log density and place are read ahead
    float nx[DIM], nl = 0.0f;
    unsigned np = 0;
    const auto load = [&](unsigned w) {
        if (w < n) {
            const unsigned k = tile + w;
            bh_load_walker_nt(X + (size_t)k * DIM, nx);
            nl = __builtin_nontemporal_load(logfn_X + k);
            np = __builtin_nontemporal_load(pos + k);
        }
    };
    load(t);
    {
        typedef float bh_f4 __attribute__((ext_vector_type(4)));
        const bh_f4* q = reinterpret_cast<const bh_f4*>(found + (size_t)tile * DIM);
        for (unsigned i = t; i < n * DIM / 4; i += kBhFoundThreads)
            reinterpret_cast<bh_f4*>(partners)[i] = __builtin_nontemporal_load(q + i);
    }
    __syncthreads();
    for (unsigned w = t; w < n; w += kBhFoundThreads) {
        const unsigned k = tile + w;
        float xk[DIM], lx = nl, y[DIM], z;
        const unsigned p = np;
#pragma unroll
        for (int i = 0; i < DIM; ++i) xk[i] = nx[i];
        load(w + kBhFoundThreads);
        unsigned e;
        const float u2 =
            bh_stretch_draw<BH_PARTNER_WALKER>(k, K, seed, odd_or_even, step, a, z, e);
#pragma unroll
        for (int i = 0; i < DIM; ++i) {
            const float xj = partners[p * DIM + i];
            y[i] = __builtin_fmaf(z, xk[i] - xj, xj);
        }
        bh_accept(y, z, u2, beta, xk, lx, data_len, params_len, params);
        bh_store_walker_nt(X + (size_t)k * DIM, xk);
        __builtin_nontemporal_store(lx, logfn_X + k);
        if (out) bh_store_walker_nt(out + (size_t)k * DIM, xk);
    }
}
#endif

#endif  // !BH_RESIDENT && !BH_BATCH

#ifdef BH_RESIDENT
// Small ensembles: one work-group holds the whole ensemble (positions and
// log densities) in LDS and runs many full steps without returning to the
// host, so that no launch sits between half-steps.  What bounds it is then
// what one compute unit must do per half-step, in sequence, and two thirds of
// that does not depend on the ensemble: the draws (Philox alone is ~20
// quarter-rate multiplies per walker) and the accounting's trees (two barriers
// and a reduction per half-step).  With both inside, 1024 walkers x 4 took 1.5
// us per bare step and 2.9 per accounted one; without, 0.69 and 0.73.  So each
// chunk of steps is three launches:
//   bh_stretch_draws     z, the partner's offset, u2 and z^(DIM-1) of every
//                        walker of every half-step of the chunk (whole chip)
//   bh_stretch_resident  the steps: partner from LDS, density, accept test;
//                        the positions after each half-step go to a trace
//                        (accounting) or straight to the caller's samples
//   bh_trace_accu        the accounting's sums of every step from the trace
//                        (whole chip)
// Every walker's arithmetic and every tree is that of the per-half-step
// kernels, so the results are bit-identical.

// Draw i of the launch is half-step i / Kp, walker i % Kp of the Kp >= K
// slots per half-step (those past K are not filled).
extern "C" __global__ void __launch_bounds__(256)
bh_stretch_draws(unsigned seed_odd, unsigned seed_even, unsigned c_odd, unsigned c_even,
                 unsigned K, unsigned Kp, float a, unsigned step0, unsigned nsteps, int partner,
                 float4* __restrict__ draws) {
    const unsigned k = blockIdx.x * 256 + threadIdx.x;
    if (k >= K) return;
    for (unsigned hs = blockIdx.y; hs < 2 * nsteps; hs += gridDim.y) {
        const bool even = hs & 1u;
        const unsigned seed = even ? seed_even : seed_odd, oe = even ? c_even : c_odd;
        const unsigned step = step0 + hs / 2;
        float z;
        unsigned e;
        const float u2 =
            partner == BH_PARTNER_FLAT
                ? bh_stretch_draw<BH_PARTNER_FLAT>(k, K, seed, oe, step, a, z, e)
                : bh_stretch_draw<BH_PARTNER_WALKER>(k, K, seed, oe, step, a, z, e);
        draws[(size_t)hs * Kp + k] = make_float4(z, __uint_as_float(e), u2, bh_zpow(z));
    }
}

// Floats from one half-ensemble to the next in LDS: the K * DIM coordinates,
// then the first DIM - 1 of them again, so that every partner's coordinates
// are read in a row from its offset, without wrapping and whatever the
// partner mode; a multiple of 4, so that records stay aligned.
__device__ __forceinline__ unsigned bh_resident_half(unsigned K) {
    return (K * DIM + DIM - 1 + 3) / 4 * 4;
}

// The ensemble in LDS: both halves, then the log densities, then the accept
// counts per group of WGS walkers.
__device__ __forceinline__ void bh_resident_load(float* sx, unsigned H, unsigned K,
                                                 const float* __restrict__ xs) {
    for (unsigned h = 0; h < 2; ++h) {
        for (unsigned i = threadIdx.x; i < K * DIM; i += blockDim.x)
            sx[h * H + i] = xs[h * K * DIM + i];
        for (unsigned i = threadIdx.x; i < DIM - 1; i += blockDim.x)
            sx[h * H + K * DIM + i] = xs[h * K * DIM + i];
    }
}

__device__ __forceinline__ void bh_resident_accept(float* X, unsigned K, unsigned k,
                                                   const float (&y)[DIM]) {
    bh_store_walker(X + k * DIM, y);
    if (DIM > 1 && k == 0) {
#pragma unroll
        for (int i = 0; i < DIM - 1; ++i) X[K * DIM + i] = y[i];
    }
}

// Each thread keeps the draws of its next BH_RESIDENT_AHEAD walkers in
// flight: they come from another XCD's writes, some 0.7 us away, a half-step
// takes 0.35.  These loads, and the stores of the positions, sit in no
// branch: the hardware retires both in order through one counter, and only
// where every path issues the same number of them can the compiler wait for
// the one load it needs instead of for all (which would be 0.7 us every
// half-step).  For the same reason the loops have one way out, after whole
// rounds of BH_RESIDENT_AHEAD; in what is past the last half-step nothing is
// decided and the positions go to `sink` (K * DIM floats).  The draws there
// were never made: the density, whose loops may depend on its argument, is
// evaluated at a position of the other half instead (z = 0).
#define BH_RESIDENT_AHEAD 4

// nsteps steps with one walker of each half per thread (blockDim.x == K): the
// thread's own records and log densities stay in registers, LDS holds what
// the other half reads.  Eight waves share four SIMDs, so at 1024 walkers the
// half-step takes the instructions it issues, ~65 VALU at dim 4 (500 of its
// 830 cycles, the rest LDS and barrier latency); the general form below reads
// and addresses everything anew: 0.45 us per half-step where this takes 0.35.
//   draws: K per half-step, and 2 * BH_RESIDENT_AHEAD * K more that are read
//        but not used
//   betas: one inverse temperature per step, or null (beta for all)
//   out (OUT): the positions after each half-step, half after half
//   accept: null, or the accept counts per group of WGS walkers, added to
template <bool OUT>
__device__ __forceinline__ void bh_resident_one(
    const float4* __restrict__ draws, unsigned data_len, unsigned params_len,
    const float* __restrict__ params, float* __restrict__ xs, float* __restrict__ logfn,
    unsigned K, float beta, const float* __restrict__ betas, unsigned nsteps,
    unsigned* __restrict__ accept, float* __restrict__ out, float* __restrict__ sink) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    static_assert(BH_RESIDENT_AHEAD == 4, "two steps per round");
    typedef float bh_f4 __attribute__((ext_vector_type(4)));
    const unsigned k = threadIdx.x, H = bh_resident_half(K);
    float* sx = lds;
    bh_resident_load(sx, H, K, xs);
    float x[2][DIM], lx[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        bh_load_walker(xs + ((size_t)h * K + k) * DIM, x[h]);
        lx[h] = logfn[h * K + k];
    }
    const bh_f4* dp = reinterpret_cast<const bh_f4*>(draws);
    bh_f4 d[BH_RESIDENT_AHEAD];
#pragma unroll
    for (int r = 0; r < BH_RESIDENT_AHEAD; ++r) {
        d[r] = dp[k];
        dp += K;
        __builtin_amdgcn_sched_barrier(0);  // in this order, which the waits count on
    }
    unsigned count = 0;  // of the wave's walkers, which are of one group
    float b[2] = {beta, beta};
    __syncthreads();
    for (unsigned s = 0; s < nsteps; s += 2) {
        if (betas) {
            b[0] = betas[s];
            b[1] = betas[s + 1 < nsteps ? s + 1 : s];
        }
#pragma unroll
        for (int r = 0; r < BH_RESIDENT_AHEAD; ++r) {
            constexpr int NH = 2;
            const int h = r % NH;
            const bool live = r < NH || s + 1 < nsteps;  // (uniform)
            // (used as a whole, so that the draw goes round the loop in one
            // register tuple: copied in parts it would be waited for there)
            asm volatile("" : "+v"(d[r]));
            float* X = sx + (h ? H : 0u);
            float sj[DIM], y[DIM];
            const float z = live ? d[r].x : 0.0f;
            const float* S = sx + (h ? 0u : H) + (live ? __float_as_uint(d[r].y) : 0u);
#pragma unroll
            for (int i = 0; i < DIM; ++i) sj[i] = S[i];
#pragma unroll
            for (int i = 0; i < DIM; ++i) y[i] = __builtin_fmaf(z, x[h][i] - sj[i], sj[i]);
            const float ly = LOGFN(data_len, params_len, params, DIM, y);
            // (u2 > 0: a log density that is not finite is never accepted)
            const float q = d[r].w * expf(b[r / NH] * (ly - lx[h]));
            const bool acc = live && __builtin_isfinite(ly) && d[r].z <= q;
#pragma unroll
            for (int i = 0; i < DIM; ++i) x[h][i] = acc ? y[i] : x[h][i];
            lx[h] = acc ? ly : lx[h];
            if (acc) bh_resident_accept(X, K, k, x[h]);
            count += (unsigned)__popcll(__ballot(acc));
            if constexpr (OUT) {
                float* dst = live ? out : sink;
#pragma unroll
                for (int i = 0; i < DIM; ++i) dst[k * DIM + i] = x[h][i];
                out += K * DIM;
            }
            d[r] = dp[k];  // BH_RESIDENT_AHEAD half-steps on, into the registers now free
            dp += K;
            __syncthreads();
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        bh_store_walker(xs + ((size_t)h * K + k) * DIM, x[h]);
        logfn[h * K + k] = lx[h];
    }
    if (accept && (k & 63u) == 0) atomicAdd(&accept[k / WGS], count);
}

// The same for larger halves, slots = ceil(K / blockDim.x) walkers per thread
// and half (draws: slots * blockDim.x per half-step, and 2 *
// BH_RESIDENT_AHEAD * blockDim.x more); threads past K take walker K - 1,
// decide nothing and write to the sink.
template <bool OUT>
__device__ __forceinline__ void bh_resident_slots(
    const float4* __restrict__ draws, unsigned data_len, unsigned params_len,
    const float* __restrict__ params, float* __restrict__ xs, float* __restrict__ logfn,
    unsigned K, float beta, const float* __restrict__ betas, unsigned nsteps,
    unsigned* __restrict__ accept, float* __restrict__ out, float* __restrict__ sink) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    constexpr int AHEAD = 2;
    typedef float bh_f4 __attribute__((ext_vector_type(4)));
    const unsigned nb = blockDim.x, t = threadIdx.x;
    const unsigned H = bh_resident_half(K), W = 2 * K, groups = K / WGS;
    float* sx = lds;                          // 2 H
    float* sl = sx + 2 * H;                   // W
    unsigned* acc_lds = (unsigned*)(sl + W);  // groups
    bh_resident_load(sx, H, K, xs);
    for (unsigned i = t; i < W; i += nb) sl[i] = logfn[i];
    for (unsigned i = t; i < groups; i += nb) acc_lds[i] = 0u;
    const unsigned total = 2 * nsteps * ((K + nb - 1) / nb);
    const bh_f4* dp = reinterpret_cast<const bh_f4*>(draws) + t;
    bh_f4 d[AHEAD];
#pragma unroll
    for (int r = 0; r < AHEAD; ++r) {
        d[r] = *dp;
        dp += nb;
        __builtin_amdgcn_sched_barrier(0);
    }
    float b = betas ? betas[0] : beta;
    float b_next = betas && nsteps > 1 ? betas[1] : beta;
    unsigned h = 0, k0 = 0, s = 0;
    __syncthreads();
    for (unsigned i0 = 0; i0 < total; i0 += AHEAD) {
#pragma unroll
        for (int r = 0; r < AHEAD; ++r) {
            const unsigned kt = k0 + t;
            const bool live = kt < K && i0 + r < total;
            const unsigned k = kt < K ? kt : K - 1;
            asm volatile("" : "+v"(d[r]));
            float* X = sx + h * H;
            float xk[DIM], sj[DIM], y[DIM];
            const float z = live ? d[r].x : 0.0f;
            const float* S = sx + (h ^ 1u) * H + (live ? __float_as_uint(d[r].y) : 0u);
#pragma unroll
            for (int i = 0; i < DIM; ++i) sj[i] = S[i];
            bh_load_walker(X + k * DIM, xk);
            const float lx = sl[h * K + k];
#pragma unroll
            for (int i = 0; i < DIM; ++i) y[i] = __builtin_fmaf(z, xk[i] - sj[i], sj[i]);
            const float ly = LOGFN(data_len, params_len, params, DIM, y);
            const float q = d[r].w * expf(b * (ly - lx));
            const bool acc = live && __builtin_isfinite(ly) && d[r].z <= q;
#pragma unroll
            for (int i = 0; i < DIM; ++i) xk[i] = acc ? y[i] : xk[i];
            if (acc) {
                bh_resident_accept(X, K, k, xk);
                sl[h * K + k] = ly;
            }
            if constexpr (OUT) {
                float* dst = live ? out : sink;
#pragma unroll
                for (int i = 0; i < DIM; ++i) dst[(size_t)k * DIM + i] = xk[i];
            }
            if (accept) {
                const unsigned long long m = __ballot(acc);
                if ((t & 63u) == 0) atomicAdd(&acc_lds[k / WGS], (unsigned)__popcll(m));
            }
            d[r] = *dp;
            dp += nb;
            k0 += nb;
            if (k0 >= K) {
                k0 = 0;
                if constexpr (OUT) out += K * DIM;
                if (h) {
                    ++s;
                    b = b_next;
                    if (betas && s + 1 < nsteps) b_next = betas[s + 1];
                }
                h ^= 1u;
                __syncthreads();
            }
        }
    }
    for (unsigned hh = 0; hh < 2; ++hh)
        for (unsigned i = t; i < K * DIM; i += nb) xs[hh * K * DIM + i] = sx[hh * H + i];
    for (unsigned i = t; i < W; i += nb) logfn[i] = sl[i];
    if (accept)
        for (unsigned i = t; i < groups; i += nb) accept[i] += acc_lds[i];
}

// With and without positions to write: two kernels, so that each has its own
// registers and its own loops.  The host bounds their threads by the ensembles
// that fit in LDS: records of 38 coordinates and more leave at most 512 walkers
// to a half, whose threads may have 256 registers each.  Bounded by 1024 threads
// all had 128, and records from 21 coordinates on spilled (us per bare step,
// independent / correlated Gaussian: 512 walkers x 48 13.3 / 39.9 -> 3.1 / 29.9,
// 1024 x 32 6.6 / 22.0 -> 3.1 / 17.9; 256 x 128 independent 37.5 -> 10.9).
#define BH_RESIDENT_KERNEL(NAME, OUT)                                                             \
    extern "C" __global__ void __launch_bounds__(BH_RESIDENT_THREADS) NAME(                       \
        const float4* __restrict__ draws, unsigned data_len, unsigned params_len,                 \
        const float* __restrict__ params, float* __restrict__ xs, float* __restrict__ logfn,      \
        unsigned K, float beta, const float* __restrict__ betas, unsigned nsteps,                 \
        unsigned* __restrict__ accept, float* __restrict__ out, float* __restrict__ sink) {       \
        if (blockDim.x == K)                                                                      \
            bh_resident_one<OUT>(draws, data_len, params_len, params, xs, logfn, K, beta, betas,  \
                                 nsteps, accept, out, sink);                                      \
        else                                                                                      \
            bh_resident_slots<OUT>(draws, data_len, params_len, params, xs, logfn, K, beta,       \
                                   betas, nsteps, accept, out, sink);                             \
    }
BH_RESIDENT_KERNEL(bh_stretch_resident, false)
BH_RESIDENT_KERNEL(bh_stretch_resident_out, true)
#undef BH_RESIDENT_KERNEL

// The accounting of stretch_move_accu for steps step0 .. step0 + gridDim.y
// from their traced positions (each step's two halves of K records): the
// group sums of the odd half, then (0 + odd) + even, the value the two
// read-modify-writes of the per-half-step kernels leave in a zeroed slot.
// One work-group per group and step.
extern "C" __global__ void __launch_bounds__(WGS)
bh_trace_accu(const float* __restrict__ trace, unsigned K, unsigned step0,
              float* __restrict__ means) {
    __shared__ float red[2][BH_ACCU_CHUNK * WGS];
    const unsigned g = blockIdx.x, groups = gridDim.x, t = threadIdx.x;
    const unsigned lane = t & 63u, wave = t >> 6;
    const float* rec = trace + ((size_t)blockIdx.y * 2 * K + g * WGS + t) * DIM;
    float xo[DIM], xe[DIM];
    bh_load_walker(rec, xo);
    bh_load_walker(rec + (size_t)K * DIM, xe);
    float* m = means + (size_t)groups * DIM * (step0 + blockIdx.y) + g;
#pragma unroll
    for (unsigned n = 0; n < kBhAccuChunks; ++n) {
        const unsigned d0 = n * BH_ACCU_CHUNK;
        if (n > 0) __syncthreads();
#pragma unroll
        for (unsigned c = 0; c < BH_ACCU_CHUNK; ++c)
            if (d0 + c < DIM) {
                red[0][c * WGS + t] = xo[d0 + c];
                red[1][c * WGS + t] = xe[d0 + c];
            }
        __syncthreads();
#pragma unroll
        for (unsigned q = 0; q < kBhAccuPer; ++q) {
            const unsigned c = wave + q * kBhWaves;
            if (c < BH_ACCU_CHUNK && d0 + c < DIM) {
                const float odd = bh_row_tree_sum(red[0], c), even = bh_row_tree_sum(red[1], c);
                if (lane == 0) m[(size_t)(d0 + c) * groups] = (0.0f + odd) + even;
            }
        }
    }
}

#endif  // BH_RESIDENT
#endif  // LOGFN

#ifdef BH_BATCH
// Many independent posteriors of one model source in one launch: a
// work-group per problem (or two), its W walkers advanced for all steps of the call
// inside the work-group.  A problem b with dimension dims[b] <= DIM and
// params params + poff[b] runs exactly the single-sampler algorithm
// (move-bare!, constants 3333/4444) with bare seed seed0 + 2b: the same
// streams, moves and accept tests as a sampler created for that problem
// alone.  Positions are packed with the problem's own dimension; a proposal
// is built in the thread's LDS slot, where the model reads it.  The records of
// a wave's 64 walkers are read, and the accepted ones written, as one run of
// floats, 64 a pass, and the partners' beside them: with each lane at its own
// walker's record a load took 64 lines, and the L1's lookups bounded the
// kernel.  16 accounted steps of 4096 posteriors of 7 to 52 dimensions, 256
// walkers each: 2.0 -> 1.1 ms.  (Groups of 16 to 64 lanes at a record each
// need fewer instructions a pass but leave lanes idle: 5% faster there, 6%
// slower than a lane per record at 192 posteriors of up to 34 dimensions,
// where this is 12% faster.)  What bounds it now is the vector instructions,
// the model's half of them.  A lane still takes its own record where that needs
// fewer instructions and no more lookups: of models of less than 8 coordinates, for
// which a run of eight passes is mostly idle, and in LDS records of no multiple of
// 8, which keep the lanes' banks apart (us per bare step of 1000 posteriors of 256
// walkers, independent Gaussian, runs / lanes: in LDS 1 coordinate 3.8 / 1.9,
// 4 4.6 / 3.0, 10 6.9 / 4.5, 16 7.6 / 14, 20 10.4 / 8.0, 100 129 / 103; in place
// 1 4.2 / 1.9, 4 4.9 / 3.6, 10 7.3 / 8.8).  The form of small models is fixed when
// they are compiled, which leaves them a third to half the registers.  The slots' stride is odd where the LDS has the
// room (ypad 1), so that the lanes' loads of one coordinate take different
// banks.  A work-group of 2 nb threads runs two problems, the i-th largest and
// the i-th smallest of its launch, in step (see batch_paired); the largest
// problems start first.
// State placement (gstate): 0 copies the problem's positions and log
// densities into LDS for the call (partner reads from LDS; the LDS a
// problem needs bounds how many share a CU), 1 works on them in place in
// the problem's global slot (L2-resident; many more problems per CU).
// Mode 1 also accumulates per problem, in double, the sums over steps of the
// ensemble sums of x and x^2; each step's ensemble sum of a coordinate is a
// float sum in a fixed order (threads own (coordinate, walker residue)
// pairs, P = nb / dim residues: a serial sum over walkers p, p + P, ..., then
// the P partial sums in order).  With series non-null it also writes each
// step's ensemble mean (that sum over W), problem b's n x dims[b] block
// starting at series + soff[b].  A launch runs the problems
// order[base .. base + count), ascending in dimension.
// LDS of each problem: 2*DIM doubles + 2*nb floats + nb*ld floats (+ W*dim + W
// floats for gstate 0).

// The value of lane r4 / 4.
__device__ __forceinline__ unsigned bh_lane(unsigned v, unsigned r4) {
    return (unsigned)__builtin_amdgcn_ds_bpermute((int)r4, (int)v);
}
__device__ __forceinline__ float bh_lane(float v, unsigned r4) {
    return __builtin_bit_cast(float, bh_lane(__builtin_bit_cast(unsigned, v), r4));
}

// A wave's 64 records of dim coordinates as one run of floats, 64 a pass: the
// record (r4 / 4) and the coordinate (iy, in bytes, with the offset of the
// wave's proposals in the LDS added) of a lane's element of a pass.
struct BhRun {
    unsigned r4, iy;
    struct Steps {
        unsigned dr4, di4, dim4, end;  // end: where iy is past a record
    };
    __device__ __forceinline__ void next(const Steps& s) {
        iy += s.di4;
        const bool past = iy >= s.end;
        r4 += past ? s.dr4 + 4u : s.dr4;
        iy -= past ? s.dim4 : 0u;
    }
};

struct BhTrue {
    static constexpr bool v = true;
};
struct BhFalse {
    static constexpr bool v = false;
};

// A place in the LDS as a byte offset, and the float at one.
__device__ __forceinline__ unsigned bh_lds_offset(const float* p) {
    return (unsigned)(size_t)(__attribute__((address_space(3))) const float*)p;
}
__device__ __forceinline__ float& bh_lds(unsigned bytes) {
    return *(float*)(__attribute__((address_space(3))) float*)(size_t)bytes;
}

// The float at a byte offset of 32 bits (one address register on a scalar base).
__device__ __forceinline__ float& bh_at(float* p, unsigned bytes) {
    return *reinterpret_cast<float*>(reinterpret_cast<char*>(p) + bytes);
}
__device__ __forceinline__ float bh_at(const float* p, unsigned bytes) {
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + bytes);
}

// A wave's LDS stores before, its other lanes' loads after (LDS operations of
// a wave complete in order).
__device__ __forceinline__ void bh_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

template <bool GSTATE>
__device__ __forceinline__ void bh_batch_impl(
    unsigned seed0, const unsigned* __restrict__ dims, const unsigned long long* __restrict__ poff,
    const unsigned* __restrict__ dlen, const unsigned* __restrict__ plen,
    const float* __restrict__ params, float* __restrict__ xs, float* __restrict__ logfn,
    unsigned W, float a, unsigned step0, unsigned nsteps, int partner, int mode,
    unsigned long long* __restrict__ accept, double* __restrict__ sums,
    const unsigned long long* __restrict__ soff, float* __restrict__ series,
    const unsigned* __restrict__ order, unsigned base, unsigned count, unsigned nb,
    unsigned ypad) {
    extern __shared__ double lds_d[];
    // the work-group's blockIdx-th largest problem, and in its second half (if
    // it has one) the blockIdx-th smallest
    const unsigned half = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >= nb));
    const unsigned big = order[base + count - 1u - blockIdx.x];
    const unsigned b = half ? order[base + blockIdx.x] : big;
    const unsigned dim = dims[b];
    const bool idle = half && b == big;  // the middle one of an odd count
    const unsigned K = idle ? 0u : W / 2;
    const unsigned t = threadIdx.x - half * nb;
    const float* prm = params + poff[b];
    const unsigned data_len = dlen[b], params_len = plen[b];
    float* gx = xs + (size_t)b * W * DIM;  // problem slot: W x DIM floats, packed by dim
    float* gl = logfn + (size_t)b * W;
    const unsigned dim0 = half ? dims[big] : 0;  // the first half's share of the LDS
    double* acc1 = lds_d;                  // DIM
    if (half)
        acc1 += 2 * DIM + (2 * nb + nb * (dim0 | ypad) + (GSTATE ? 0 : W * dim0 + W)) / 2;
    double* acc2 = acc1 + DIM;             // DIM
    float* red = reinterpret_cast<float*>(acc2 + DIM);  // 2 * nb
    float* sx;                             // W * dim
    float* sl;                             // W
    float* yb;                             // nb * ld
    if constexpr (GSTATE) {
        sx = gx;
        sl = gl;
        yb = red + 2 * nb;
    } else {
        sx = red + 2 * nb;
        sl = sx + (size_t)W * dim;
        yb = sl + W;
        for (unsigned i = t; i < W * dim; i += nb) sx[i] = gx[i];
        for (unsigned i = t; i < W; i += nb) sl[i] = gl[i];
    }
    for (unsigned i = t; i < 2 * DIM; i += nb) acc1[i] = 0.0;
    __syncthreads();
    const unsigned seed = seed0 + 2u * b;
    unsigned long long nacc = 0;
    const float inv_a = 1.0f / a;
    const float ca = a - 2.0f + inv_a;
    const float cb = 2.0f * (1.0f - inv_a);
    const unsigned ld = dim | ypad;  // odd if the LDS has the room
    const unsigned lane = t & 63u;
    float* yw = yb + (size_t)(t - lane) * ld;  // the wave's proposals
    float* y = yw + lane * ld;
    // a lane to a record
    const bool lanes = DIM < 8 || (!GSTATE && ((DIM < 12 && DIM != 8) || dim % 8 != 0));
    constexpr int N = 8;  // passes in flight
    const unsigned yw4 = (unsigned)__builtin_amdgcn_readfirstlane((int)bh_lds_offset(yw));
    const unsigned sx4 = GSTATE ? 0u : bh_lds_offset(sx), dim4 = 4 * dim;
    const BhRun run0{4 * (lane / dim), yw4 + 4 * (lane % dim)};
    const BhRun::Steps steps{4 * (64u / dim), 4 * (64u % dim), dim4, yw4 + dim4};
    // the problem's slot as a buffer of its own size
    const __amdgpu_buffer_rsrc_t xbuf =
        __builtin_amdgcn_make_buffer_rsrc(gx, 0, (int)(W * dim4), 0x00020000);
    const unsigned P = dim <= nb ? nb / dim : 1u;
    for (unsigned st = 0; st < nsteps; ++st) {
        const unsigned step = step0 + st;
        for (int h = 0; h < 2; ++h) {
            float* X = sx + (h ? (size_t)K * dim : 0);
            const float* S = sx + (h ? 0 : (size_t)K * dim);
            float* L = sl + (h ? K : 0);
            for (unsigned k = t; k < K; k += nb) {
                const bh_f32x4 u = bh_u01x4(bh_philox4x32_10(
                    bh_u32x4{k, step, h ? 4444u : 3333u, BH_CTR3}, seed + (unsigned)h,
                    BH_KEY1_STRETCH));
                const float z = __builtin_fmaf(ca * u.y, u.y, cb * u.y) + inv_a;
                // partner element i at S[(e + i) mod K*dim] (FLAT) or
                // S[j*dim + i] (WALKER)
                unsigned e;
                if (partner == BH_PARTNER_FLAT) {
                    e = (unsigned)((u.x * (float)K) * (float)dim);
                    if (e >= K * dim) e -= K * dim;
                } else {
                    unsigned j = (unsigned)(u.x * (float)K);
                    j = j < K ? j : K - 1;
                    e = j * dim;  // e + i < K * dim for i < dim
                }
                const float lk = L[k];
                if (lanes) {
                    const float* xk = X + (size_t)k * dim;
                    unsigned i = 0;
                    for (; !GSTATE && i + N <= dim; i += N) {
                        float xa[N], sa[N];
#pragma unroll
                        for (int c = 0; c < N; ++c) {
                            unsigned ec = e + c;
                            if (ec >= K * dim) ec -= K * dim;
                            xa[c] = xk[i + c];
                            sa[c] = S[ec];
                        }
#pragma unroll
                        for (int c = 0; c < N; ++c)
                            y[i + c] = __builtin_fmaf(z, xa[c] - sa[c], sa[c]);
                        e += N;
                        if (e >= K * dim) e -= K * dim;
                    }
                    for (; i < dim; ++i) {
                        const float xj = S[e];
                        y[i] = __builtin_fmaf(z, xk[i] - xj, xj);
                        e = (e + 1 == K * dim) ? 0u : e + 1;
                    }
                } else {
                    // the wave's records (a scalar base, byte offsets below)
                    const float* xw =
                        X + (size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(k - lane)) * dim;
                    const unsigned total = 4 * K * dim;
                    e = 4 * e - yw4;  // + iy: the coordinate's place
                    BhRun at = run0;
                    // N passes from the j-th, all of them in the records (FULL)
                    const auto propose = [&](unsigned j, auto FULL) {
                        float xa[N], sa[N], zr[N];
                        unsigned ec[N], yo[N];
#pragma unroll
                        for (int c = 0; c < N; ++c) {
                            ec[c] = bh_lane(e, at.r4) + at.iy;
                            zr[c] = bh_lane(z, at.r4);
                            yo[c] = __umul24(at.r4, ld) + at.iy;
                            at.next(steps);
                        }
#pragma unroll
                        for (int c = 0; c < N; ++c) {
                            // (a pass past the records loads from within them)
                            xa[c] = bh_at(xw + 64 * (FULL.v || j + c < dim ? j + c : j), 4 * lane);
                            // past the end: from the start (the smaller, unsigned)
                            sa[c] = bh_at(S, ec[c] - total < ec[c] ? ec[c] - total : ec[c]);
                        }
#pragma unroll
                        for (int c = 0; c < N; ++c)
                            if (FULL.v || j + c < dim)
                                bh_lds(yo[c]) = __builtin_fmaf(zr[c], xa[c] - sa[c], sa[c]);
                    };
                    unsigned j = 0;
                    for (; j + N <= dim; j += N) propose(j, BhTrue{});
                    if (j < dim) propose(j, BhFalse{});
                    bh_wave_sync();
                }
                const float ly = LOGFN(data_len, params_len, prm, dim, y);
                float zp = 1.0f;
#pragma unroll 4
                for (unsigned i = 1; i < dim; ++i) zp *= z;
                const float q = __builtin_isfinite(ly) ? zp * expf(ly - lk) : 0.0f;
                const bool accepted = u.z <= q;
                if (accepted) {
                    L[k] = ly;
                    nacc += 1;
                }
                if (lanes) {
                    if (accepted)
                        for (unsigned i = 0; i < dim; ++i) X[(size_t)k * dim + i] = y[i];
                    continue;
                }
                bh_wave_sync();
                if (__builtin_amdgcn_ballot_w64(accepted) != 0) {
                    // no branch: what did not move is stored past the buffer's
                    // end, which the hardware drops, or (LDS) onto the
                    // proposal itself
                    const unsigned keep = accepted ? 0u : 0x80000000u;
                    const unsigned xo =
                        ((h ? K : 0u) + (unsigned)__builtin_amdgcn_readfirstlane((int)(k - lane))) *
                        dim4;
                    BhRun at = run0;
                    const auto move = [&](unsigned j, auto FULL) {
                        float ya[N];
                        unsigned kept[N], yo[N];
#pragma unroll
                        for (int c = 0; c < N; ++c) {
                            kept[c] = bh_lane(keep, at.r4);
                            yo[c] = __umul24(at.r4, ld) + at.iy;
                            at.next(steps);
                        }
#pragma unroll
                        for (int c = 0; c < N; ++c)
                            ya[c] = bh_lds(FULL.v || j + c < dim ? yo[c] : yo[0]);
#pragma unroll
                        for (int c = 0; c < N; ++c)
                            if (FULL.v || j + c < dim) {
                                if constexpr (GSTATE)
                                    __builtin_amdgcn_raw_buffer_store_b32(
                                        __builtin_bit_cast(unsigned, ya[c]), xbuf,
                                        4 * lane | kept[c], (int)(xo + 256 * (j + c)), 0);
                                else
                                    bh_lds(kept[c] ? yo[c]
                                                   : sx4 + xo + 256 * (j + c) + 4 * lane) = ya[c];
                            }
                    };
                    unsigned j = 0;
                    for (; j + N <= dim; j += N) move(j, BhTrue{});
                    if (j < dim) move(j, BhFalse{});
                }
                bh_wave_sync();
            }
            __syncthreads();
        }
        if (mode == 1) {
            if (dim <= nb) {
                if (t < P * dim && !idle) {
                    const unsigned d = t % dim, p = t / dim;
                    float s1 = 0.0f, s2 = 0.0f;
                    // walkers p, p + P, ... in order, N loads in flight
                    const unsigned wstep = 4 * P * dim, wend = 4 * W * dim;
                    unsigned wo = 4 * (p * dim + d);
                    for (; wo + (N - 1) * wstep < wend; wo += N * wstep) {
                        float xv[N];
#pragma unroll
                        for (int c = 0; c < N; ++c) xv[c] = bh_at(sx, wo + c * wstep);
#pragma unroll
                        for (int c = 0; c < N; ++c) {
                            s1 += xv[c];
                            s2 = __builtin_fmaf(xv[c], xv[c], s2);
                        }
                    }
                    if (wo < wend) {
                        float xv[N];
#pragma unroll
                        for (int c = 0; c < N; ++c)
                            xv[c] = bh_at(sx, wo + c * wstep < wend ? wo + c * wstep : wo);
#pragma unroll
                        for (int c = 0; c < N; ++c)
                            if (wo + c * wstep < wend) {
                                s1 += xv[c];
                                s2 = __builtin_fmaf(xv[c], xv[c], s2);
                            }
                    }
                    red[t] = s1;
                    red[nb + t] = s2;
                }
            } else {
                for (unsigned d = t; d < dim && !idle; d += nb) {
                    float s1 = 0.0f, s2 = 0.0f;
                    for (unsigned w = 0; w < W; ++w) {
                        const float x = sx[(size_t)w * dim + d];
                        s1 += x;
                        s2 = __builtin_fmaf(x, x, s2);
                    }
                    acc1[d] += (double)s1;
                    acc2[d] += (double)s2;
                    if (series) series[soff[b] + (size_t)st * dim + d] = s1 / (float)W;
                }
            }
            // the next step's first half writes accepted proposals into sx,
            // which these sums read
            __syncthreads();
            if (dim <= nb) {
                if (t < dim && !idle) {
                    float s1 = 0.0f, s2 = 0.0f;
                    for (unsigned p = 0; p < P; ++p) {
                        s1 += red[p * dim + t];
                        s2 += red[nb + p * dim + t];
                    }
                    acc1[t] += (double)s1;
                    acc2[t] += (double)s2;
                    if (series) series[soff[b] + (size_t)st * dim + t] = s1 / (float)W;
                }
                // red is written again only after the next step's two
                // half-step barriers
            }
        }
    }
    if (!GSTATE && !idle) {
        for (unsigned i = t; i < W * dim; i += nb) gx[i] = sx[i];
        for (unsigned i = t; i < W; i += nb) gl[i] = sl[i];
    }
    // accept count: block reduce in the (now free) staging area
    __syncthreads();
    unsigned long long* ra = reinterpret_cast<unsigned long long*>(red);
    ra[t] = nacc;
    __syncthreads();
    for (unsigned r = nb / 2; r >= 1; r >>= 1) {
        if (t < r) ra[t] += ra[t + r];
        __syncthreads();
    }
    if (t == 0 && !idle) accept[b] += ra[0];
    if (mode == 1 && !idle) {
        for (unsigned i = t; i < dim; i += nb) {
            sums[((size_t)b * DIM + i) * 2] += acc1[i];
            sums[((size_t)b * DIM + i) * 2 + 1] += acc2[i];
        }
    }
}

// State in LDS (bh_batch_run) or in place in global memory (bh_batch_run_g):
// two kernels, so that each has the registers of one placement.
#define BH_BATCH_RUN_KERNEL(NAME, GSTATE)                                                        \
    extern "C" __global__ void __launch_bounds__(1024) NAME(                                     \
        unsigned seed0, const unsigned* __restrict__ dims,                                        \
        const unsigned long long* __restrict__ poff, const unsigned* __restrict__ dlen,           \
        const unsigned* __restrict__ plen, const float* __restrict__ params,                      \
        float* __restrict__ xs, float* __restrict__ logfn, unsigned W, float a, unsigned step0,   \
        unsigned nsteps, int partner, int mode, unsigned long long* __restrict__ accept,          \
        double* __restrict__ sums, const unsigned long long* __restrict__ soff,                   \
        float* __restrict__ series, const unsigned* __restrict__ order, unsigned base,            \
        unsigned count, unsigned nb, unsigned ypad) {                                             \
        bh_batch_impl<GSTATE>(seed0, dims, poff, dlen, plen, params, xs, logfn, W, a, step0,      \
                              nsteps, partner, mode, accept, sums, soff, series, order, base,     \
                              count, nb, ypad);                                                   \
    }
BH_BATCH_RUN_KERNEL(bh_batch_run, false)
BH_BATCH_RUN_KERNEL(bh_batch_run_g, true)
#undef BH_BATCH_RUN_KERNEL

// Initial positions and log-densities of every problem: init_walkers'
// stream (key {seed0 + b, 0xdecafaaa}) over the problem's W*dim values,
// limits (DIM x 2 per problem) taken row i % dim.
extern "C" __global__ void __launch_bounds__(256)
bh_batch_init(unsigned seed0, const unsigned* __restrict__ dims,
              const unsigned long long* __restrict__ poff, const unsigned* __restrict__ dlen,
              const unsigned* __restrict__ plen, const float* __restrict__ params,
              const float* __restrict__ limits, float* __restrict__ xs, float* __restrict__ logfn,
              unsigned W) {
    const unsigned b = blockIdx.y;
    const unsigned dim = dims[b];
    float* gx = xs + (size_t)b * W * DIM;
    const float* lim = limits + (size_t)b * DIM * 2;
    const unsigned items = dim * W / 4;
    for (unsigned g = blockIdx.x * 256 + threadIdx.x; g < items; g += gridDim.x * 256) {
        const bh_f32x4 u = bh_u01x4(bh_philox4x32_10(
            bh_u32x4{g, BH_CTR1_INIT, BH_CTR2_INIT, BH_CTR3}, seed0 + b, BH_KEY1_INIT));
        const float uu[4] = {u.x, u.y, u.z, u.w};
        for (unsigned m = 0; m < 4; ++m) {
            const unsigned i = 4 * g + m;
            const unsigned r = i % dim;
            gx[i] = __builtin_fmaf(uu[m], lim[2 * r + 1], (1.0f - uu[m]) * lim[2 * r]);
        }
    }
}

extern "C" __global__ void __launch_bounds__(256)
bh_batch_logfn(const unsigned* __restrict__ dims, const unsigned long long* __restrict__ poff,
               const unsigned* __restrict__ dlen, const unsigned* __restrict__ plen,
               const float* __restrict__ params, const float* __restrict__ xs,
               float* __restrict__ logfn, unsigned W) {
    const unsigned b = blockIdx.y;
    const unsigned w = blockIdx.x * 256 + threadIdx.x;
    if (w >= W) return;
    const unsigned dim = dims[b];
    const float* x = xs + (size_t)b * W * DIM + (size_t)w * dim;
    logfn[(size_t)b * W + w] = LOGFN(dlen[b], plen[b], params + poff[b], dim, x);
}
#endif  // BH_BATCH

#ifdef BH_GLM
#ifndef BH_GLM_KIND
#define BH_GLM_KIND 1
#endif
// Generalised linear model posteriors evaluated for a whole batch of walkers
// at once (the likelihood is a dense contraction X.Y over data rows, run by
// the ahead-of-time kernels of bh_glm.hip).  These kernels are the
// walker-side halves: the proposal, and the accept test with its accounting,
// with the same arithmetic as bh_stretch_walker.

// Writes yscale*Y as nsplit 16-bit terms (bf16, or fp16 when f16 is set),
// hi + mid + lo, each the nearest value of what the previous terms leave
// (exact residuals in fp32).  With g0 (the logistic softplus sum's gradient
// at a reference point b of the ensemble, natural units) it returns the
// correction of the log posterior for the split's rounding: with y' =
// lnscale * terms (lnscale = 1 / yscale in the epilogue's units) and
// dl = y - y', the first-order -g0 . dl, and given H0 (the sum's Hessian at
// b) also -dl . H0 (y' - b + dl / 2), so that the split's log posterior plus
// it is the log posterior at y up to terms of third order in (y' - b, dl)
// (0 when not finite).
__device__ __forceinline__ double bh_glm_split(const float (&y)[DIM], float yscale, int nsplit,
                                               int f16, void* out, unsigned k, unsigned n,
                                               const double* __restrict__ g0, double lnscale,
                                               const float* __restrict__ H0,
                                               const float* __restrict__ bref) {
    double c = 0.0;
    double dl[DIM];  // y - y', y' what the terms represent (natural units)
    float w[DIM];    // y' - b + dl / 2
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
        float r = y[i] * yscale;
        double hs = 0.0;  // what the terms represent, in units of 1 / yscale
        const size_t o = (size_t)k * DIM + i;
        for (int sp = 0; sp < nsplit; ++sp) {
            if (f16) {
                const _Float16 h = (_Float16)r;
                static_cast<_Float16*>(out)[(size_t)sp * n * DIM + o] = h;
                r = r - (float)h;
                hs += (double)(float)h;
            } else {
                const __bf16 h = (__bf16)r;
                static_cast<__bf16*>(out)[(size_t)sp * n * DIM + o] = h;
                r = r - (float)h;
                hs += (double)(float)h;
            }
        }
        const double yp = hs * lnscale;
        dl[i] = (double)y[i] - yp;
        if (g0) c = __builtin_fma(g0[i], -dl[i], c);
        if (H0) w[i] = (float)(yp - (double)bref[i] + 0.5 * dl[i]);
    }
    if (g0 && H0) {
        for (int i = 0; i < DIM; ++i) {
            float v = 0.0f;
            for (int j = 0; j < DIM; ++j) v = __builtin_fmaf(H0[i * DIM + j], w[j], v);
            c = __builtin_fma(-dl[i], (double)v, c);
        }
    }
    return __builtin_isfinite(c) ? c : 0.0;
}

// Proposals of one half-step: Y (fp32), z and u2 per walker, and the 16-bit
// split of log2(e)*Y for the MFMA kernels with, given g0 (and H0, bref), each
// proposal's correction for it in corr (as bh_glm_split); clears the guard
// list's count.  Given H0 and gscale, gscale[k] = max(1, q / (2 DIM)), q the
// larger H0-norm squared of the proposal's and the position's distances
// from b, by which the screen widens the guard for walker k.  BH_GLM_TPW
// threads per walker, thread `sub` taking coordinates sub, sub + BH_GLM_TPW,
// ... (so a walker's threads read and write consecutive coordinates); each
// draws the walker's uniforms (the same Philox call), and the corrections'
// parts are summed over the walker's threads.
#define BH_GLM_TPW 16
extern "C" __global__ void __launch_bounds__(WGS)
bh_glm_propose(unsigned seed, unsigned odd_or_even, const float* __restrict__ S,
               const float* __restrict__ X, float a, unsigned step, unsigned K, int partner,
               float* __restrict__ Y, float* __restrict__ zbuf, float* __restrict__ u2buf,
               void* __restrict__ ysplit, float yscale, int nsplit, int f16,
               unsigned* __restrict__ guard_count, const double* __restrict__ g0, double lnscale,
               double* __restrict__ corr, const float* __restrict__ H0,
               const float* __restrict__ bref, float* __restrict__ gscale) {
    constexpr int CPT = (DIM + BH_GLM_TPW - 1) / BH_GLM_TPW;  // coordinates per thread
    // H0 rows padded to a multiple of 4 floats plus 4 (16-byte reads; the
    // 16 rows a wave reads at once start in different banks)
    constexpr int HP = (DIM + 3) / 4 * 4 + 4;
    __shared__ __attribute__((aligned(16))) float wsh[WGS / BH_GLM_TPW][HP];
    __shared__ __attribute__((aligned(16))) float wxs[WGS / BH_GLM_TPW][HP];
    __shared__ __attribute__((aligned(16))) float hsh[DIM * HP];
    const unsigned gt = blockIdx.x * WGS + threadIdx.x;
    const unsigned k = gt / BH_GLM_TPW, sub = gt % BH_GLM_TPW;
    if (guard_count && gt == 0) *guard_count = 0u;
    float z;
    unsigned e;
    const float u2 = partner == BH_PARTNER_FLAT
                         ? bh_stretch_draw<BH_PARTNER_FLAT>(k, K, seed, odd_or_even, step, a, z, e)
                         : bh_stretch_draw<BH_PARTNER_WALKER>(k, K, seed, odd_or_even, step, a, z,
                                                              e);
    const unsigned total = K * DIM;
    // the loads of all the thread's coordinates (partner's and own position,
    // g0 and the reference point) issued before any of them is used; where
    // g0 or the reference point is absent the load reads the ensemble S
    // instead (at least 4 K DIM >= 8 DIM bytes; the value is never used), so
    // that no load sits in a branch of its own
    const double* g0p = g0 ? g0 : reinterpret_cast<const double*>(S);
    const float* brp = H0 ? bref : S;
    float xjv[CPT], xiv[CPT], brv[CPT];
    double g0v[CPT];
#pragma unroll
    for (int q = 0; q < CPT; ++q) {
        const unsigned i = sub + q * BH_GLM_TPW;
        xjv[q] = 0.0f;
        xiv[q] = 0.0f;
        brv[q] = 0.0f;
        g0v[q] = 0.0;
        if (i < DIM) {
            unsigned ei = e + i;
            if (partner == BH_PARTNER_FLAT && ei >= total) ei -= total;
            xjv[q] = S[ei];
            xiv[q] = X[(size_t)k * DIM + i];
            g0v[q] = g0p[i];
            brv[q] = brp[i];
        }
    }
    asm volatile("" ::: "memory");
    double c = 0.0;
    double dl[CPT];
    float wv[CPT], wx[CPT];
    int m = 0;
    for (unsigned i = sub; i < DIM; i += BH_GLM_TPW, ++m) {
        const float xj = xjv[m];
        const float xi = xiv[m];
        const float yi = __builtin_fmaf(z, xi - xj, xj);
        Y[(size_t)k * DIM + i] = yi;
        if (nsplit > 0) {
            float r = yi * yscale;
            double hs = 0.0;
            const size_t o = (size_t)k * DIM + i;
            for (int sp = 0; sp < nsplit; ++sp) {
                if (f16) {
                    const _Float16 h = (_Float16)r;
                    static_cast<_Float16*>(ysplit)[(size_t)sp * K * DIM + o] = h;
                    r = r - (float)h;
                    hs += (double)(float)h;
                } else {
                    const __bf16 h = (__bf16)r;
                    static_cast<__bf16*>(ysplit)[(size_t)sp * K * DIM + o] = h;
                    r = r - (float)h;
                    hs += (double)(float)h;
                }
            }
            const double yp = hs * lnscale;
            dl[m] = (double)yi - yp;
            if (g0) c = __builtin_fma(g0v[m], -dl[m], c);
            if (H0) {
                wv[m] = (float)(yp - (double)brv[m] + 0.5 * dl[m]);
                wx[m] = xi - brv[m];
            }
        }
    }
    float qy = 0.0f, qx = 0.0f;
    if (nsplit > 0 && g0 && H0) {
        // the second-order term: the walker's y' - b + dl / 2 through LDS,
        // each thread the rows of H0 of its coordinates (H0 staged in LDS
        // once per work-group); with it the H0-norms of the proposal's and
        // the position's distances from b
        const unsigned wl = threadIdx.x / BH_GLM_TPW;
        // rows padded with zeros past DIM; eight loads in flight per thread
        constexpr unsigned NH = (DIM * HP + WGS - 1) / WGS;
        for (unsigned t0 = 0; t0 < NH; t0 += 8) {
            float hv[8];
#pragma unroll
            for (unsigned t = 0; t < 8; ++t) {
                const unsigned q = threadIdx.x + (t0 + t) * WGS, r = q / HP, j = q % HP;
                hv[t] = q < DIM * HP && j < DIM ? H0[r * DIM + j] : 0.0f;
            }
            asm volatile("" ::: "memory");
#pragma unroll
            for (unsigned t = 0; t < 8; ++t) {
                const unsigned q = threadIdx.x + (t0 + t) * WGS;
                if (q < DIM * HP) hsh[q] = hv[t];
            }
        }
        for (unsigned j = DIM + sub; j < HP; j += BH_GLM_TPW) {
            wsh[wl][j] = 0.0f;
            wxs[wl][j] = 0.0f;
        }
        m = 0;
        for (unsigned i = sub; i < DIM; i += BH_GLM_TPW, ++m) {
            wsh[wl][i] = wv[m];
            wxs[wl][i] = wx[m];
        }
        __syncthreads();
        m = 0;
        for (unsigned i = sub; i < DIM; i += BH_GLM_TPW, ++m) {
            float v = 0.0f, vx = 0.0f;
            const float4* hr = reinterpret_cast<const float4*>(hsh + i * HP);
            const float4* ws = reinterpret_cast<const float4*>(wsh[wl]);
            const float4* wxr = reinterpret_cast<const float4*>(wxs[wl]);
#pragma unroll 4
            for (int j4 = 0; j4 < (DIM + 3) / 4; ++j4) {
                const float4 h = hr[j4], wy = ws[j4], wxx = wxr[j4];
                v = __builtin_fmaf(h.x, wy.x, v);
                v = __builtin_fmaf(h.y, wy.y, v);
                v = __builtin_fmaf(h.z, wy.z, v);
                v = __builtin_fmaf(h.w, wy.w, v);
                vx = __builtin_fmaf(h.x, wxx.x, vx);
                vx = __builtin_fmaf(h.y, wxx.y, vx);
                vx = __builtin_fmaf(h.z, wxx.z, vx);
                vx = __builtin_fmaf(h.w, wxx.w, vx);
            }
            c = __builtin_fma(-dl[m], (double)v, c);
            qy = __builtin_fmaf(wv[m], v, qy);
            qx = __builtin_fmaf(wx[m], vx, qx);
        }
    }
#pragma unroll
    for (int off = BH_GLM_TPW / 2; off >= 1; off >>= 1) {
        c += __shfl_xor(c, off, 64);
        qy += __shfl_xor(qy, off, 64);
        qx += __shfl_xor(qx, off, 64);
    }
    if (sub == 0) {
        zbuf[k] = z;
        u2buf[k] = u2;
        if (nsplit > 0 && corr) corr[k] = __builtin_isfinite(c) ? c : 0.0;
        // the guard's scale for this walker: the correction's remainder grows
        // with the square of the distance from b, which near equilibrium is
        // about DIM in the H0-norm
        if (gscale) {
            const float q = __builtin_fmaxf(qy, qx) / (2.0f * (float)DIM);
            gscale[k] = q > 1.0f ? q : 1.0f;
        }
    }
}

// 16-bit split of n given points (for the initial log-densities), with their
// corrections given g0.
extern "C" __global__ void __launch_bounds__(WGS)
bh_glm_split_points(const float* __restrict__ P, unsigned n, void* __restrict__ ysplit,
                    float yscale, int nsplit, int f16, const double* __restrict__ g0,
                    double lnscale, double* __restrict__ corr, const float* __restrict__ H0,
                    const float* __restrict__ bref) {
    const unsigned k = blockIdx.x * WGS + threadIdx.x;
    if (k >= n) return;
    float y[DIM];
#pragma unroll
    for (int i = 0; i < DIM; ++i) y[i] = P[(size_t)k * DIM + i];
    const double c = bh_glm_split(y, yscale, nsplit, f16, ysplit, k, n, g0, lnscale, H0, bref);
    if (corr) corr[k] = c;
}

// Log posterior of point y from the sum s over data rows of the likelihood
// kernel's per-row terms, in double.
// BH_GLM_KIND 1, logistic: lin.y - scale * s - |y|^2 / (2 s0^2), with s the
//   softplus sum and lin the linear coefficients of the precision.
// BH_GLM_KIND 2, linear regression, y = [beta (DIM-1), log sigma], s the sum
//   of squared residuals, lin = {N, N log(2 pi) / 2, 1 / s_beta^2,
//   1 / s_logsigma^2}: -N log sigma - N log(2 pi)/2 - s / (2 sigma^2)
//   - |beta|^2 / (2 s_beta^2) - (log sigma)^2 / (2 s_logsigma^2).
__device__ __forceinline__ double bh_glm_logpost_sum(const float (&y)[DIM], double s,
                                                     const double* __restrict__ lin, double scale,
                                                     double prior_prec) {
#if BH_GLM_KIND == 2
    (void)scale;
    (void)prior_prec;
    const double ls = (double)y[DIM - 1];
    double q = 0.0;
#pragma unroll
    for (int i = 0; i < DIM - 1; ++i) q = __builtin_fma((double)y[i], (double)y[i], q);
    return -lin[0] * ls - lin[1] - 0.5 * exp(-2.0 * ls) * s - 0.5 * (lin[2] * q + lin[3] * ls * ls);
#else
    double l = 0.0, q = 0.0;
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
        l = __builtin_fma(lin[i], (double)y[i], l);
        q = __builtin_fma((double)y[i], (double)y[i], q);
    }
    return l - scale * s - 0.5 * prior_prec * q;
#endif
}

// p[0] + p[stride] + ..., n values in this order.  The chain is one thread's
// and each load some 0.7 us away, so the time is the number of rounds of
// loads: 32 in flight, then 8, also for the last few.
__device__ __forceinline__ double bh_strided_sum(const double* __restrict__ p, size_t stride,
                                                 unsigned n) {
    double s = 0.0;
    unsigned r = 0;
    for (; r + 32 <= n; r += 32) {
        double v[32];
#pragma unroll
        for (int e = 0; e < 32; ++e) v[e] = p[(size_t)(r + e) * stride];
#pragma unroll
        for (int e = 0; e < 32; ++e) s += v[e];
    }
    for (; r < n; r += 8) {
        // past the end the first of the eight again, not added
        double v[8];
#pragma unroll
        for (unsigned e = 0; e < 8; ++e) v[e] = p[(size_t)(r + e < n ? r + e : r) * stride];
#pragma unroll
        for (unsigned e = 0; e < 8; ++e) s = r + e < n ? s + v[e] : s;
    }
    return s;
}

// The same from the per-range row sums of the likelihood kernel (the sum
// over ranges runs in range order).
__device__ __forceinline__ double bh_glm_logpost(const float (&y)[DIM], unsigned k, unsigned n,
                                                 const double* __restrict__ partial,
                                                 unsigned nranges, const double* __restrict__ lin,
                                                 double scale, double prior_prec,
                                                 const double* __restrict__ corr) {
    const double s = bh_strided_sum(partial + k, n, nranges);
    const double l = bh_glm_logpost_sum(y, s, lin, scale, prior_prec);
    return corr ? l + corr[k] : l;
}

// Sum over r < nranges of partial[r * stride + col] by one wave: lane-strided
// partial sums (eight loads in flight), then a butterfly (a fixed order).
__device__ __forceinline__ double bh_wave_range_sum(const double* __restrict__ partial,
                                                    unsigned nranges, unsigned stride,
                                                    unsigned col) {
    const unsigned lane = threadIdx.x & 63u;
    double s = 0.0;
    unsigned r = lane;
    for (; r + 7 * 64 < nranges; r += 8 * 64) {
        double v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = partial[(size_t)(r + e * 64) * stride + col];
#pragma unroll
        for (int e = 0; e < 8; ++e) s += v[e];
    }
    for (; r < nranges; r += 64) s += partial[(size_t)r * stride + col];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    return s;
}

// The log posteriors of 16 consecutive points by one work-group, WGS/16
// threads to a point: lane l of a wave takes point l % 16, so that a load of
// the partial sums reads whole lines, and the ranges and coordinates go round
// the point's threads (`sub` of BH_GLM_STPW).  With a point's threads side by
// side in a wave instead, each load touched eight half-used lines on few
// compute units: 14.4 us for 1024 points x 768 ranges, now 5.7.
#define BH_GLM_STPW (WGS / 16)
struct BhGlmLds {
    double s[WGS / 64][3][16];
    unsigned slot[16];
};

// The thread's point is k = base + lane % 16.  The result is in the first 16
// threads of the work-group.
__device__ __forceinline__ double bh_glm_logpost16(const float* __restrict__ P, unsigned k,
                                                   unsigned n,
                                                   const double* __restrict__ partial,
                                                   unsigned nranges,
                                                   const double* __restrict__ lin, double scale,
                                                   double prior_prec,
                                                   const double* __restrict__ corr,
                                                   BhGlmLds& lds) {
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const unsigned sub = threadIdx.x / 16;
    // coordinates of the linear and quadratic terms, and their coefficients
    // (linear regression: the coefficients' squares; log sigma by itself)
#if BH_GLM_KIND == 2
    constexpr unsigned QD = DIM - 1;
    const float ls = P[(size_t)k * DIM + QD];
#else
    constexpr unsigned QD = DIM;
#endif
    constexpr unsigned SC = (QD + BH_GLM_STPW - 1) / BH_GLM_STPW;
    float yc[SC];
    double lc[SC];
#pragma unroll
    for (unsigned c = 0; c < SC; ++c) {
        const unsigned i = sub + c * BH_GLM_STPW;
        yc[c] = i < QD ? P[(size_t)k * DIM + i] : 0.0f;
        lc[c] = 0.0;
#if BH_GLM_KIND != 2
        if (i < QD) lc[c] = lin[i];
#endif
    }
    double v[3] = {0.0, 0.0, 0.0};  // row sum, linear and quadratic term
    if (sub < nranges)
        v[0] = bh_strided_sum(partial + (size_t)sub * n + k, (size_t)BH_GLM_STPW * n,
                              (nranges - sub + BH_GLM_STPW - 1) / BH_GLM_STPW);
#pragma unroll
    for (unsigned c = 0; c < SC; ++c) {
        const double y = (double)yc[c];
        v[1] = __builtin_fma(lc[c], y, v[1]);
        v[2] = __builtin_fma(y, y, v[2]);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        v[j] += __shfl_xor(v[j], 16, 64);
        v[j] += __shfl_xor(v[j], 32, 64);
        if (lane < 16) lds.s[wave][j][lane] = v[j];
    }
    __syncthreads();
    double lp = 0.0;
    if (threadIdx.x < 16) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            v[j] = lds.s[0][j][lane];
            for (unsigned w = 1; w < WGS / 64; ++w) v[j] += lds.s[w][j][lane];
        }
#if BH_GLM_KIND == 2
        const double lsd = (double)ls;
        lp = -lin[0] * lsd - lin[1] - 0.5 * exp(-2.0 * lsd) * v[0] -
             0.5 * (lin[2] * v[2] + lin[3] * lsd * lsd);
#else
        lp = v[1] - scale * v[0] - 0.5 * prior_prec * v[2];
#endif
        if (corr) lp += corr[k];
    }
    return lp;
}

// Initial log posteriors of n points, 16 per work-group.
extern "C" __global__ void __launch_bounds__(WGS)
bh_glm_logpost(const float* __restrict__ P, unsigned n, const double* __restrict__ partial,
               unsigned nranges, const double* __restrict__ lin, double scale, double prior_prec,
               double* __restrict__ lp, const double* __restrict__ corr) {
    __shared__ BhGlmLds lds;
    const unsigned k = blockIdx.x * 16 + (threadIdx.x & 15u);
    const double v = bh_glm_logpost16(P, k, n, partial, nranges, lin, scale, prior_prec, corr, lds);
    if (threadIdx.x < 16) lp[k] = v;
}

// The accept decision of stretch_move (amd-gcn-mcmc-stretch.cl:66-71): q =
// z^(DIM-1) exp(beta (lp(Y) - lp(X))), u2 <= q, the difference taken in
// double and rounded to float as the kernels of every precision do.
__device__ __forceinline__ bool bh_glm_decide(double lpy, double lpx, float z, float u2,
                                              float beta) {
    const float d = (float)(lpy - lpx);
    const float q = __builtin_isfinite(lpy) ? bh_zpow(z) * expf(beta * d) : 0.0f;
    return u2 <= q;
}

// Guarded accept test of the reduced-precision likelihoods.  The decision is
// a monotone step in d = lp(Y) - lp(X); a walker whose log margin
//   m = log u2 - (DIM-1) log z - beta d
// is within `guard` of zero (times gscale[k] when given) could be decided
// differently by an error of that size in d, so it is listed (up to lmax
// walkers, the rest counting as overflow; the engine passes lmax = K, so
// none overflow) for an fp64 evaluation of lp(Y) and lp(X) and decided on
// those.
// 16 walkers per work-group (bh_glm_logpost16).
// flag[k]: 0 decided here, 3 listed (bh_glm_resolve turns it into 1 = reject
// or 2 = accept).
extern "C" __global__ void __launch_bounds__(WGS)
bh_glm_screen(const float* __restrict__ Y, const float* __restrict__ zbuf,
              const float* __restrict__ u2buf, const double* __restrict__ partial,
              unsigned nranges, const double* __restrict__ lin, double scale, double prior_prec,
              const double* __restrict__ lp, float beta, unsigned K, double guard,
              unsigned* __restrict__ flag, unsigned* __restrict__ list,
              unsigned* __restrict__ count, unsigned lmax, const float* __restrict__ Xpos,
              double* __restrict__ pts64, double* __restrict__ lpy_out,
              const double* __restrict__ corr, const float* __restrict__ gscale) {
    __shared__ BhGlmLds lds;
    const unsigned kk = threadIdx.x & 15u, sub = threadIdx.x / 16;
    const unsigned k = blockIdx.x * 16 + kk;
    // the walker's scalars, ahead of the sums
    const float u2k = u2buf[k], zk = zbuf[k];
    const double lpk = lp[k];
    const float gsk = gscale ? gscale[k] : 1.0f;
    const double lpy =
        bh_glm_logpost16(Y, k, K, partial, nranges, lin, scale, prior_prec, corr, lds);
    if (threadIdx.x < 16) {
        unsigned slot = 0xffffffffu;
        lpy_out[k] = lpy;
        unsigned f = 0;
        if (__builtin_isfinite(lpy)) {
            const double m = log((double)u2k) - (double)(DIM - 1) * log((double)zk) -
                             (double)beta * (lpy - lpk);
            const double gk = gscale ? guard * (double)gsk : guard;
            if (__builtin_fabs(m) <= gk) {
                const unsigned i = atomicAdd(count, 1u);
                if (i < lmax) {
                    list[i] = k;
                    f = 3;
                    slot = i;
                }
            }
        }
        // walkers not listed are decided here, on this precision's values
        // (1 reject, 2 accept; bh_glm_resolve decides the listed ones)
        if (f == 0) f = bh_glm_decide(lpy, lpk, zk, u2k, beta) ? 2u : 1u;
        flag[k] = f;
        lds.slot[kk] = slot;
    }
    __syncthreads();
    const unsigned slot = lds.slot[kk];
    if (slot != 0xffffffffu) {
        // the two points in double for the fp64 likelihood kernel: row 2i
        // the proposal, row 2i + 1 the current position
        for (unsigned j = sub; j < DIM; j += BH_GLM_STPW) {
            pts64[(size_t)2 * slot * DIM + j] = (double)Y[(size_t)k * DIM + j];
            pts64[((size_t)2 * slot + 1) * DIM + j] = (double)Xpos[(size_t)k * DIM + j];
        }
    }
}

// Decides the listed walkers on their fp64 log posteriors, one wave per
// walker: partial64 holds, per row range r (row stride `stride`), column
// 2i the softplus sum of Y[list[i]] and column 2i + 1 that of X[list[i]]
// (natural units).
// totals[0] += listed walkers, totals[1] += walkers past lmax.
extern "C" __global__ void __launch_bounds__(WGS)
bh_glm_resolve(const float* __restrict__ Y, const float* __restrict__ X,
               const float* __restrict__ zbuf, const float* __restrict__ u2buf,
               const double* __restrict__ partial64, unsigned nranges64, unsigned stride,
               const double* __restrict__ lin64, double prior_prec, float beta,
               const unsigned* __restrict__ list, const unsigned* __restrict__ count,
               unsigned lmax, unsigned* __restrict__ flag,
               unsigned long long* __restrict__ totals) {
    const unsigned n = *count;
    const unsigned c = n < lmax ? n : lmax;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        atomicAdd(&totals[0], (unsigned long long)c);
        atomicAdd(&totals[1], (unsigned long long)(n - c));
    }
    const unsigned waves = WGS / 64;
    for (unsigned i = blockIdx.x * waves + threadIdx.x / 64; i < c; i += gridDim.x * waves) {
#if BH_GLM_KIND != 2
        // both columns of a range in one 16-byte load (the row stride is
        // even), eight loads in flight per lane; the coordinates' terms
        // across the lanes; then one butterfly for all six sums
        const unsigned lane = threadIdx.x & 63u;
        double sy = 0.0, sx = 0.0;
        unsigned r = lane;
        for (; r + 7 * 64 < nranges64; r += 8 * 64) {
            double2 v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[e] = *reinterpret_cast<const double2*>(partial64 + (size_t)(r + e * 64) * stride +
                                                         2 * i);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sy += v[e].x;
                sx += v[e].y;
            }
        }
        for (; r < nranges64; r += 64) {
            const double2 v =
                *reinterpret_cast<const double2*>(partial64 + (size_t)r * stride + 2 * i);
            sy += v.x;
            sx += v.y;
        }
        const unsigned k = list[i];
        double ly = 0.0, lx = 0.0, qy = 0.0, qx = 0.0;
        for (unsigned j = lane; j < DIM; j += 64) {
            const double yj = (double)Y[(size_t)k * DIM + j];
            const double xj = (double)X[(size_t)k * DIM + j];
            ly = __builtin_fma(lin64[j], yj, ly);
            lx = __builtin_fma(lin64[j], xj, lx);
            qy = __builtin_fma(yj, yj, qy);
            qx = __builtin_fma(xj, xj, qx);
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            sy += __shfl_xor(sy, off, 64);
            sx += __shfl_xor(sx, off, 64);
            ly += __shfl_xor(ly, off, 64);
            lx += __shfl_xor(lx, off, 64);
            qy += __shfl_xor(qy, off, 64);
            qx += __shfl_xor(qx, off, 64);
        }
        if (lane == 0) {
            // the logistic log posterior (bh_glm_logpost_sum, scale 1)
            const double lpy = ly - sy - 0.5 * prior_prec * qy;
            const double lpx = lx - sx - 0.5 * prior_prec * qx;
            flag[k] = bh_glm_decide(lpy, lpx, zbuf[k], u2buf[k], beta) ? 2u : 1u;
        }
#else
        const double sy = bh_wave_range_sum(partial64, nranges64, stride, 2 * i);
        const double sx = bh_wave_range_sum(partial64, nranges64, stride, 2 * i + 1);
        if ((threadIdx.x & 63u) == 0) {
            const unsigned k = list[i];
            float y[DIM], xk[DIM];
#pragma unroll
            for (int j = 0; j < DIM; ++j) {
                y[j] = Y[(size_t)k * DIM + j];
                xk[j] = X[(size_t)k * DIM + j];
            }
            const double ly = bh_glm_logpost_sum(y, sy, lin64, 1.0, prior_prec);
            const double lx = bh_glm_logpost_sum(xk, sx, lin64, 1.0, prior_prec);
            flag[k] = bh_glm_decide(ly, lx, zbuf[k], u2buf[k], beta) ? 2u : 1u;
        }
#endif
    }
}

// Accept test of one half-step (amd-gcn-mcmc-stretch.cl:66-78) with accu !=
// 0 also the accounting of stretch_move_accu.  With flag non-null, walkers
// resolved in fp64 take that decision.
extern "C" __global__ void __launch_bounds__(WGS)
bh_glm_accept(const float* __restrict__ Y, const float* __restrict__ zbuf,
              const float* __restrict__ u2buf, const double* __restrict__ partial,
              unsigned nranges, const double* __restrict__ lin, double scale, double prior_prec,
              float* __restrict__ X, double* __restrict__ lp, float beta, unsigned K, int accu,
              unsigned* __restrict__ accept, float* __restrict__ means, unsigned mstep,
              const unsigned* __restrict__ flag, const double* __restrict__ corr) {
    const unsigned k = blockIdx.x * WGS + threadIdx.x;
    BhAccuOld old;
    if (accu) old.load(blockIdx.x, gridDim.x, mstep, accept, means);
    float y[DIM], xk[DIM];
#pragma unroll
    for (int i = 0; i < DIM; ++i) y[i] = Y[(size_t)k * DIM + i];
    // the stored lp stays in this sampler's precision in every case, so that
    // its common offset from the fp64 values cancels in later differences
    const double lpy = bh_glm_logpost(y, k, K, partial, nranges, lin, scale, prior_prec, corr);
    const unsigned f = flag ? flag[k] : 0u;
    const bool accepted = (f == 1u || f == 2u)
                              ? f == 2u
                              : bh_glm_decide(lpy, lp[k], zbuf[k], u2buf[k], beta);
    if (accepted) {
#pragma unroll
        for (int i = 0; i < DIM; ++i) {
            X[(size_t)k * DIM + i] = y[i];
            xk[i] = y[i];
        }
        lp[k] = lpy;
    } else if (accu) {
#pragma unroll
        for (int i = 0; i < DIM; ++i) xk[i] = X[(size_t)k * DIM + i];
    }
    if (accu)
        bh_accu(xk, accepted, blockIdx.x, gridDim.x, mstep, accept, means, old, bh_accu_lds());
}
// The guarded path's accept step, with every decision already in flag (1
// reject, 2 accept) and the proposals' log posteriors in lpy: work-group
// (g, c) handles group g's WGS walkers and coordinates
// [c*BH_ACCU_CHUNK, (c+1)*BH_ACCU_CHUNK): it copies accepted proposals of
// those coordinates into X and adds their group sums to the means (the
// same tree per coordinate as bh_accu); chunk 0 also stores the accepted
// log posteriors and the group's accept count.
extern "C" __global__ void __launch_bounds__(WGS)
bh_glm_accept_split(const float* __restrict__ Y, const double* __restrict__ lpy,
                    float* __restrict__ X, double* __restrict__ lp, int accu,
                    unsigned* __restrict__ accept, float* __restrict__ means, unsigned mstep,
                    const unsigned* __restrict__ flag) {
    const unsigned g = blockIdx.x, c = blockIdx.y;
    const unsigned k = g * WGS + threadIdx.x;
    const bool accepted = flag[k] == 2u;
    const unsigned d0 = c * BH_ACCU_CHUNK;
    // lane q of a wave: the wave's q-th coordinate of the chunk (bh_accu)
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const unsigned cm = wave + lane * kBhWaves;
    const bool mine = accu && lane < kBhAccuPer && cm < BH_ACCU_CHUNK && d0 + cm < DIM;
    float* m = means + (size_t)gridDim.x * DIM * mstep + (size_t)(d0 + cm) * gridDim.x + g;
    float old = mine ? *m : 0.0f;
    const unsigned old_acc = accu && c == 0 ? accept[g] : 0u;
    float v[BH_ACCU_CHUNK];
#pragma unroll
    for (int i = 0; i < BH_ACCU_CHUNK; ++i) {
        const unsigned d = d0 + i;
        v[i] = 0.0f;
        if (d < DIM) {
            if (accepted) {
                v[i] = Y[(size_t)k * DIM + d];
                X[(size_t)k * DIM + d] = v[i];
            } else if (accu) {
                v[i] = X[(size_t)k * DIM + d];
            }
        }
    }
    if (c == 0 && accepted) lp[k] = lpy[k];
    if (accu) {
        BhAccuLds& lds = bh_accu_lds();
        const unsigned long long b = __ballot(accepted);
        if (lane == 0) lds.wave_counts[wave] = (unsigned)__popcll(b);
#pragma unroll
        for (int i = 0; i < BH_ACCU_CHUNK; ++i) lds.red[i * WGS + threadIdx.x] = v[i];
        __syncthreads();
#pragma unroll
        for (unsigned q = 0; q < kBhAccuPer; ++q) {
            const unsigned i = wave + q * kBhWaves;
            if (i < BH_ACCU_CHUNK && d0 + i < DIM) {
                const float sum = bh_row_tree_sum(lds.red, i);
                if (lane == q) old += sum;
            }
        }
        if (mine) *m = old;
        if (c == 0 && threadIdx.x == 0) {
            unsigned cnt = 0;
            for (unsigned w = 0; w < kBhWaves; ++w) cnt += lds.wave_counts[w];
            accept[g] = old_acc + cnt;
        }
    }
}
#endif  // BH_GLM

#ifdef LOGPDF
// logpdf / pdf kernels (amd-gcn-distribution.cl:1-14).
extern "C" __global__ void __launch_bounds__(WGS)
bh_logpdf(unsigned data_len, unsigned params_len, const float* __restrict__ params, unsigned dim,
          const float* __restrict__ x, float* __restrict__ res, unsigned long long n) {
    const unsigned long long j = (unsigned long long)blockIdx.x * WGS + threadIdx.x;
    if (j < n) res[j] = LOGPDF(data_len, params_len, params, dim, x + j * dim);
}

extern "C" __global__ void __launch_bounds__(WGS)
bh_pdf(unsigned data_len, unsigned params_len, const float* __restrict__ params, unsigned dim,
       const float* __restrict__ x, float* __restrict__ res, unsigned long long n) {
    const unsigned long long j = (unsigned long long)blockIdx.x * WGS + threadIdx.x;
    if (j < n) res[j] = native_exp(LOGPDF(data_len, params_len, params, dim, x + j * dim));
}
#endif  // LOGPDF

#ifdef LOGLIK
// loglik / lik / evidence kernels (amd-gcn-likelihood.cl:1-29); the
// evidence accumulates in double (ACCUMULATOR=double, amd_gcn.clj:580).
extern "C" __global__ void __launch_bounds__(WGS)
bh_loglik(unsigned data_len, const float* __restrict__ data, unsigned dim,
          const float* __restrict__ x, float* __restrict__ res, unsigned long long n) {
    const unsigned long long j = (unsigned long long)blockIdx.x * WGS + threadIdx.x;
    if (j < n) res[j] = LOGLIK(data_len, data, dim, x + j * dim);
}

extern "C" __global__ void __launch_bounds__(WGS)
bh_lik(unsigned data_len, const float* __restrict__ data, unsigned dim,
       const float* __restrict__ x, float* __restrict__ res, unsigned long long n) {
    const unsigned long long j = (unsigned long long)blockIdx.x * WGS + threadIdx.x;
    if (j < n) res[j] = native_exp(LOGLIK(data_len, data, dim, x + j * dim));
}

extern "C" __global__ void __launch_bounds__(WGS)
bh_evidence_partial(unsigned data_len, const float* __restrict__ data, unsigned dim,
                    const float* __restrict__ x, unsigned long long n,
                    double* __restrict__ partial) {
    const unsigned long long j = (unsigned long long)blockIdx.x * WGS + threadIdx.x;
    double v = 0.0;
    if (j < n) v = (double)native_exp(LOGLIK(data_len, data, dim, x + j * dim));
#pragma unroll
    for (int i = 32; i >= 1; i >>= 1) v += __shfl_down(v, i, 64);
    __shared__ double wsum[WGS / 64];
    if ((threadIdx.x & 63u) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < WGS / 64; ++w) s += wsum[w];
        partial[blockIdx.x] = s;
    }
}
#endif  // LOGLIK
