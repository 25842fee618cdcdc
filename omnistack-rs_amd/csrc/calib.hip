// Lloyd-Max INT4 codebook calibration on the GPU (gfx950).
//
// Reference: LloydMaxCalibrator.fit (omnistack_rs/quantization/codebook.py:
// 64-108), driven per kv head by calibrate_per_group (:148-172) in the bake
// (scripts/run_criteo_benchmark.py:357-362).  Same recipe:
//   init   16 equal-count bins of the sorted samples (bin size
//          bs = n / 16; the n % 16 largest samples are in no bin), centroid
//          = mean of its bin;
//   iterate  code = first-index argmin_k fp32 |x - c_k|; c_k = mean of the
//          samples coded k (an empty cell keeps its centroid); stop after
//          max_iters or when the largest fp32 move |c_new - c_old| < tol
//          (the moved centroids are kept);
//   result sorted ascending.
//
// A Lloyd step needs no pass over the samples.  They are counted and stored
// once by bins of their order-preserving key: a bin is one exponent (of one
// sign) or a power-of-two part of it, as fine as its share of the samples
// asks for (up to 512 a bin on average).  (calib_inplace.hip calibrates where
// there is no room for that copy.)  One exponent per bin makes the fp64 sum of up
// to 2^29 of its samples exact in any order.  Under sorted centroids the
// codes ascend with x, so cell k is a run of whole bins between two boundary
// bins plus a part of each: per boundary the largest fp32 value that still
// takes the lower code is found with the fp32 distances themselves, and only
// that bin's samples are compared with it.  One block per group runs the
// initial bins and every step in one launch, a wave per boundary; the bins'
// places stay in LDS, the boundary bin's samples in registers, so a step
// waits for memory once, and only where a boundary has moved to another bin.
// 8 groups x 1.64 M fp32 samples, 300 steps (a pass over all samples and an
// update launch per step before): 17.7 ms -> 1.2 ms (0.93 ms of it the steps).
//
// Results are deterministic: sums inside a bin are exact, sums over bins are
// formed in fp64 in a fixed order, means are rounded to fp32 once.  (The
// reference's fp32 `mean()` rounds along the way: its last bits can differ,
// and so can a convergence decision taken at the tolerance.)  Where two
// distances of one sample can round to a tie with a lower index (centroids
// closer than 2^-22 of the distances compared) the step codes each bin by its
// ends, and the samples one by one only of bins where those do not decide.
// Samples must be finite.
//
// Layout: group g's samples are rows of `inner` contiguous elements:
// element e of group g is x[(e / inner) * outer_stride + g * group_stride +
// e % inner], e < outer * inner.  A flat vector is outer = 1; head h of a
// (B, H, T, D) cache is outer = B, inner = T*D, outer_stride = H*T*D,
// group_stride = T*D.
#include <float.h>
#include <math.h>

#include "calib.h"

namespace omni {

constexpr int kLmThreads = 1024;
constexpr int kLmPer = 32;                  // samples per thread of the counting and storing passes
constexpr int kLmBlock = kLmThreads * kLmPer;
constexpr int kLmOct = 512;                 // sign and exponent
constexpr int kLmMaxBins = 32768;           // bins per group at most (their places fit LDS)
// Samples per bin aimed at, where that keeps the bins within kLmMaxBins.
// Finer bins cost the passes that fill them more than they save the steps:
// count, store, bin sums and steps took 72 + 174 + 49 + 955 us at 64 samples,
// 31 + 154 + 28 + 920 at 256 and 26 + 148 + 24 + 927 at 512 (8 x 1.64 M).
constexpr int kLmFill = 512;
constexpr int kLmCache = 32;                // samples per lane a boundary bin may hold in registers

struct LmArgs {
    const void *x;
    int64_t outer, inner, outer_stride, group_stride, n, bs;
    int max_iters;
    float tol;
    int nb, nch;            // bins (the last ones may be unused) and 64-bin chunks
    int64_t fill;           // samples per bin aimed at
    int mant;               // mantissa bits of the sample type
    int vec, wide;          // 4-element loads; n >= 2^32: cursors relative to their bin
    // workspace (per group g)
    uint32_t *oct;          // [g][512] samples per sign and exponent
    uint32_t *map;          // [g][512] first bin << 5 | key bits below the bin number
    uint32_t *cnt;          // [g][nb]
    uint32_t *cursor;       // [g][nb] next free place of each bin
    uint64_t *start;        // [g][nb + 1] first place of each bin
    double *bsum;           // [g][nb]
    double *csum;           // [g][nch] sums of 64 bins
    float *buf;             // [g][n] samples by bin
    float *out;             // [g][16]
    int32_t *iters;         // [g], nullable
};

template <int DT>
__device__ __forceinline__ float lm_widen(uint16_t h) {
    return DT == OMNI_BF16 ? bf16_to_f32(h) : f16_to_f32(h);
}

// This thread's samples of the block's run of kLmBlock: bit s of the result
// says that xv[s] is one.  The (row, column) pair advances without division.
template <int DT>
__device__ __forceinline__ uint32_t lm_load_run(const LmArgs &a, int g, float (&xv)[kLmPer]) {
    const int w = a.vec ? 4 : 1;
    const int64_t first = (int64_t)blockIdx.x * kLmBlock + (int64_t)threadIdx.x * w;
    const int64_t stride = (int64_t)kLmThreads * w;
    int64_t o = 0, i = first, so = 0, si = stride;
    if (a.outer > 1) {
        o = first / a.inner;
        i = first - o * a.inner;
        so = stride / a.inner;
        si = stride - so * a.inner;
    }
    uint32_t valid = 0u;
    const int64_t gbase = (int64_t)g * a.group_stride;
    auto next = [&]() {
        o += so;
        i += si;
        if (i >= a.inner) {
            i -= a.inner;
            ++o;
        }
    };
    if (a.vec) {
#pragma unroll
        for (int j = 0; j < kLmPer / 4; ++j) {
            const bool ok = first + j * stride < a.n;
            const int64_t idx = ok ? o * a.outer_stride + gbase + i : gbase;
            if constexpr (DT == OMNI_F32) {
                const float4 t = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(a.x) + idx);
                xv[4 * j] = t.x; xv[4 * j + 1] = t.y; xv[4 * j + 2] = t.z; xv[4 * j + 3] = t.w;
            } else {
                const uint2 t = *reinterpret_cast<const uint2 *>(reinterpret_cast<const uint16_t *>(a.x) + idx);
                xv[4 * j] = lm_widen<DT>((uint16_t)t.x); xv[4 * j + 1] = lm_widen<DT>((uint16_t)(t.x >> 16));
                xv[4 * j + 2] = lm_widen<DT>((uint16_t)t.y); xv[4 * j + 3] = lm_widen<DT>((uint16_t)(t.y >> 16));
            }
            valid |= ok ? 15u << (4 * j) : 0u;
            next();
        }
    } else {
#pragma unroll
        for (int j = 0; j < kLmPer; ++j) {
            const bool ok = first + j * stride < a.n;
            const int64_t idx = ok ? o * a.outer_stride + gbase + i : gbase;
            if constexpr (DT == OMNI_F32) xv[j] = reinterpret_cast<const float *>(a.x)[idx];
            else xv[j] = lm_widen<DT>(reinterpret_cast<const uint16_t *>(a.x)[idx]);
            valid |= ok ? 1u << j : 0u;
            next();
        }
    }
    return valid;
}

__device__ __forceinline__ uint32_t lm_bin(uint32_t map, uint32_t key) {
    return (map >> 5) + ((key & 0x7fffffu) >> (map & 31u));
}

__global__ __launch_bounds__(256) void lm_clear_kernel(LmArgs a) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b < kLmOct) a.oct[(size_t)blockIdx.y * kLmOct + b] = 0u;
    if (b >= a.nb) return;
    const size_t at = (size_t)blockIdx.y * a.nb + b;
    a.cnt[at] = 0u;
    a.bsum[at] = 0.0;
}

// Samples per sign and exponent.  Most of them share a few: four copies of
// the counters per block.
template <int DT>
__global__ __launch_bounds__(kLmThreads) void lm_oct_kernel(LmArgs a) {
    __shared__ uint32_t lh[4][kLmOct];
    const int g = blockIdx.y;
    float xv[kLmPer];
    const uint32_t valid = lm_load_run<DT>(a, g, xv);
    for (int w = threadIdx.x; w < 4 * kLmOct; w += kLmThreads) lh[0][w] = 0u;
    __syncthreads();
    uint32_t *mine = lh[threadIdx.x & 3];
#pragma unroll
    for (int s = 0; s < kLmPer; ++s)
        if ((valid >> s) & 1u) atomicAdd(&mine[lm_key(xv[s]) >> 23], 1u);
    __syncthreads();
    for (int w = threadIdx.x; w < kLmOct; w += kLmThreads) {
        const uint32_t v = lh[0][w] + lh[1][w] + lh[2][w] + lh[3][w];
        if (v) atomicAdd(&a.oct[(size_t)g * kLmOct + w], v);
    }
}

// Bins of each sign and exponent: 2^m with m the smallest that leaves `fill`
// samples a bin or fewer on average (at most one per value of the sample
// type), so 2 n / fill + 512 of them at most.
__global__ __launch_bounds__(kLmOct) void lm_map_kernel(LmArgs a) {
    __shared__ uint32_t wsum[kLmOct / 64];
    const int g = blockIdx.x, t = threadIdx.x, lane = t & 63, w = t >> 6;
    const uint64_t c = a.oct[(size_t)g * kLmOct + t];
    int m = 0;
    while (m < a.mant && ((uint64_t)a.fill << m) < c) ++m;
    const uint32_t mine = 1u << m;
    uint32_t incl = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(incl, off);
        if (lane >= off) incl += y;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    uint32_t base = incl - mine;
    for (int q = 0; q < w; ++q) base += wsum[q];
    a.map[(size_t)g * kLmOct + t] = (base << 5) | (uint32_t)(23 - m);
}

// Samples per bin: 16-bit counters of a block's 32768 samples in LDS, then
// one global addition per bin that the block met.
template <int DT>
__global__ __launch_bounds__(kLmThreads) void lm_count_kernel(LmArgs a) {
    __shared__ uint32_t lh[kLmMaxBins / 2];
    __shared__ uint32_t map[kLmOct];
    const int g = blockIdx.y;
    float xv[kLmPer];
    const uint32_t valid = lm_load_run<DT>(a, g, xv);
    const int words = a.nb / 2;
    for (int w = threadIdx.x; w < words; w += kLmThreads) lh[w] = 0u;
    if (threadIdx.x < kLmOct) map[threadIdx.x] = a.map[(size_t)g * kLmOct + threadIdx.x];
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kLmPer; ++s)
        if ((valid >> s) & 1u) {
            const uint32_t k = lm_key(xv[s]), b = lm_bin(map[k >> 23], k);
            atomicAdd(&lh[b >> 1], (b & 1u) ? 65536u : 1u);
        }
    __syncthreads();
    uint32_t *cnt = a.cnt + (size_t)g * a.nb;
    for (int w = threadIdx.x; w < words; w += kLmThreads) {
        const uint32_t v = lh[w];
        if (v & 0xffffu) atomicAdd(&cnt[2 * w], v & 0xffffu);
        if (v >> 16) atomicAdd(&cnt[2 * w + 1], v >> 16);
    }
}

// First place of each bin: a block takes 4096 bins, four per thread, after
// the sum of all bins before them.
constexpr int kLmScan = 4 * kLmThreads;

__global__ __launch_bounds__(kLmThreads) void lm_scan_kernel(LmArgs a) {
    __shared__ uint64_t wsum[kLmThreads / 64], wpre[kLmThreads / 64];
    const int g = blockIdx.y, t = threadIdx.x, lane = t & 63, w = t >> 6;
    const uint4 *cnt = reinterpret_cast<const uint4 *>(a.cnt + (size_t)g * a.nb);
    uint64_t pre = 0;
    for (int k = t; k < (int)blockIdx.x * kLmThreads; k += kLmThreads) {
        const uint4 v = cnt[k];
        pre += (uint64_t)v.x + v.y + v.z + v.w;
    }
    const int b0 = (int)blockIdx.x * kLmScan + 4 * t;
    const uint4 v = b0 < a.nb ? cnt[b0 >> 2] : make_uint4(0u, 0u, 0u, 0u);
    const uint32_t cv[4] = {v.x, v.y, v.z, v.w};
    const uint64_t mine = (uint64_t)v.x + v.y + v.z + v.w;
    uint64_t incl = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint64_t y = __shfl_up((unsigned long long)incl, off);
        if (lane >= off) incl += y;
        pre += __shfl_xor((unsigned long long)pre, off);
    }
    if (lane == 63) {
        wsum[w] = incl;
        wpre[w] = pre;
    }
    __syncthreads();
    uint64_t at = incl - mine;
    for (int q = 0; q < kLmThreads / 64; ++q) at += wpre[q] + (q < w ? wsum[q] : 0);
    if (b0 >= a.nb) return;
    uint64_t *start = a.start + (size_t)g * (a.nb + 1);
    uint32_t *cursor = a.cursor + (size_t)g * a.nb;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int b = b0 + k;
        start[b] = at;
        cursor[b] = a.wide ? 0u : (uint32_t)at;
        at += cv[k];
    }
    if (b0 + 4 == a.nb) start[a.nb] = at;
}

// Samples to their bins: a block ranks its samples per bin in LDS, reserves a
// run of every bin that it met with one global addition, and writes.  The
// order inside a bin is not fixed and nothing below depends on it.
template <int DT>
__global__ __launch_bounds__(kLmThreads) void lm_store_kernel(LmArgs a) {
    __shared__ uint32_t lh[kLmMaxBins];
    __shared__ uint32_t map[kLmOct];
    const int g = blockIdx.y;
    float xv[kLmPer];
    const uint32_t valid = lm_load_run<DT>(a, g, xv);
    uint32_t *cursor = a.cursor + (size_t)g * a.nb;
    float *buf = a.buf + (size_t)g * a.n;
    for (int s = threadIdx.x; s < a.nb; s += kLmThreads) lh[s] = 0u;
    if (threadIdx.x < kLmOct) map[threadIdx.x] = a.map[(size_t)g * kLmOct + threadIdx.x];
    __syncthreads();
    uint32_t at[kLmPer];                               // bin, rank among the block's samples in it << 15
#pragma unroll
    for (int s = 0; s < kLmPer; ++s) {
        at[s] = 0u;
        if ((valid >> s) & 1u) {
            const uint32_t k = lm_key(xv[s]), b = lm_bin(map[k >> 23], k);
            at[s] = b | (atomicAdd(&lh[b], 1u) << 15);
        }
    }
    static_assert(kLmMaxBins <= 1 << 15 && kLmBlock <= 1 << 15, "bin and rank share 32 bits");
    __syncthreads();
    for (int s = threadIdx.x; s < a.nb; s += kLmThreads) {
        const uint32_t c = lh[s];
        if (c) lh[s] = atomicAdd(&cursor[s], c);
    }
    __syncthreads();
    if (a.wide) {
        const uint64_t *start = a.start + (size_t)g * (a.nb + 1);
#pragma unroll
        for (int s = 0; s < kLmPer; ++s)
            if ((valid >> s) & 1u) buf[start[at[s] & 32767u] + lh[at[s] & 32767u] + (at[s] >> 15)] = xv[s];
    } else {
#pragma unroll
        for (int s = 0; s < kLmPer; ++s)
            if ((valid >> s) & 1u) buf[lh[at[s] & 32767u] + (at[s] >> 15)] = xv[s];
    }
}

// Lane l's value as a scalar (l wave-uniform): the wave's own state stays in
// scalar registers and its branches uniform.
__device__ __forceinline__ float lm_lane(float v, int l) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), l));
}
__device__ __forceinline__ double lm_lane(double v, int l) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    return __builtin_bit_cast(double, (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, l) |
                                          ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l) << 32));
}

// Wave sums by DPP row shifts (1, 2, 4, 8: each row's last lane holds its
// sum) and row broadcasts (15 into rows 1 and 3, 31 into rows 2 and 3), no LDS
// permutes; the result is a scalar.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t lm_dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double lm_dpp_add(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint64_t t = (uint64_t)lm_dpp<CTRL, ROWS>((uint32_t)u) | ((uint64_t)lm_dpp<CTRL, ROWS>((uint32_t)(u >> 32)) << 32);
    return v + __builtin_bit_cast(double, t);
}
__device__ __forceinline__ double lm_wave_sum(double v) {
    v = lm_dpp_add<0x111, 0xf>(v);
    v = lm_dpp_add<0x112, 0xf>(v);
    v = lm_dpp_add<0x114, 0xf>(v);
    v = lm_dpp_add<0x118, 0xf>(v);
    v = lm_dpp_add<0x142, 0xa>(v);
    v = lm_dpp_add<0x143, 0xc>(v);
    return lm_lane(v, 63);
}
__device__ __forceinline__ uint32_t lm_wave_sum_u32(uint32_t v) {
    v += lm_dpp<0x111, 0xf>(v);
    v += lm_dpp<0x112, 0xf>(v);
    v += lm_dpp<0x114, 0xf>(v);
    v += lm_dpp<0x118, 0xf>(v);
    v += lm_dpp<0x142, 0xa>(v);
    v += lm_dpp<0x143, 0xc>(v);
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// fp64 sum of each bin: a wave takes 1024 consecutive stored samples, mostly
// one bin per 64, and adds once per bin.  Exact in any order (one exponent
// per bin, up to 2^29 samples).
__global__ __launch_bounds__(256) void lm_binsum_kernel(LmArgs a) {
    constexpr int kVec = 16;
    const int g = blockIdx.y, lane = threadIdx.x & 63;
    const int64_t base = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 * kVec);
    if (base >= a.n) return;
    const float *buf = a.buf + (size_t)g * a.n;
    double *bsum = a.bsum + (size_t)g * a.nb;
    const uint32_t *map = a.map + (size_t)g * kLmOct;
    float v[kVec];
    uint32_t bn[kVec];
#pragma unroll
    for (int k = 0; k < kVec; ++k) {
        const int64_t e = base + 64 * k + lane;
        v[k] = buf[e < a.n ? e : a.n - 1];
    }
#pragma unroll
    for (int k = 0; k < kVec; ++k) {
        const uint32_t key = lm_key(v[k]);
        bn[k] = lm_bin(map[key >> 23], key);
    }
    double acc = 0.0;
    uint32_t cur = 0u;
    bool open = false;
    auto flush = [&]() {
        if (open) {
            const double t = lm_wave_sum(acc);
            if (lane == 0) unsafeAtomicAdd(&bsum[cur], t);
        }
        open = false;
        acc = 0.0;
    };
#pragma unroll
    for (int k = 0; k < kVec; ++k) {
        const bool ok = base + 64 * k + lane < a.n;
        const uint32_t b = bn[k];
        const uint32_t b0 = __builtin_amdgcn_readfirstlane(b);
        if (__builtin_amdgcn_ballot_w64(!ok || b != b0) == 0ull) {
            if (open && b0 != cur) flush();
            cur = b0;
            open = true;
            acc += (double)v[k];
        } else {
            // several bins: sums over each run of equal bins, added by its last lane
            double t = ok ? (double)v[k] : 0.0;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const double u = __shfl_up(t, d);
                const uint32_t ub = __shfl_up(b, d);
                if (lane >= d && ub == b) t += u;
            }
            const uint32_t nb1 = __shfl_down(b, 1);
            const bool okn = __shfl_down(ok ? 1 : 0, 1) != 0;
            if (ok && (lane == 63 || nb1 != b || !okn)) unsafeAtomicAdd(&bsum[b], t);
        }
    }
    flush();
}

// Sums of 64 bins (a wave each).
__global__ __launch_bounds__(kLmThreads) void lm_chunk_kernel(LmArgs a) {
    const int g = blockIdx.y, lane = threadIdx.x & 63, c = blockIdx.x * (kLmThreads / 64) + (threadIdx.x >> 6);
    if (c >= a.nch) return;
    const double s = lm_wave_sum(a.bsum[(size_t)g * a.nb + 64 * c + lane]);
    if (lane == 0) a.csum[(size_t)g * a.nch + c] = s;
}

// d_a <= d_b for a < b as the fp32 distances decide it, false from b on
// (there the pairs further right decide); ascending x: true, then false.
__device__ __forceinline__ bool lm_left(float x, float a, float b) {
    return x < b && fabsf(x - a) <= fabsf(x - b);
}

// Key of the largest value that takes a's code rather than b's (wave).
__device__ __forceinline__ uint32_t lm_threshold(float a, float b, int lane) {
    uint32_t lo = lm_key(a), hi = lm_key(b);          // lm_left(lo), !lm_left(hi)
    {
        // 64 values around the midpoint: nearly always enough
        const uint32_t mid = lm_key(0.5f * a + 0.5f * b);
        const uint32_t k = mid - 32u + (uint32_t)lane;
        const bool in = mid > lo + 32u && mid + 32u < hi;
        const uint64_t t = __builtin_amdgcn_ballot_w64(in && lm_left(lm_value(k), a, b));
        const int c = __popcll(t);
        if (c > 0 && c < 64) return mid - 32u + (uint32_t)c - 1u;
    }
    while (hi - lo > 1u) {
        const uint32_t step = (hi - lo + 63u) >> 6;
        // offsets, not keys: lo + 64 step can pass 2^32
        const uint64_t off = (uint64_t)step * (uint32_t)(lane + 1);
        const uint64_t t = __builtin_amdgcn_ballot_w64(off < (uint64_t)(hi - lo) &&
                                                       lm_left(lm_value(lo + (uint32_t)off), a, b));
        const uint32_t c = (uint32_t)__popcll(t);
        const uint64_t up = (uint64_t)step * (c + 1u);
        if (up < (uint64_t)(hi - lo)) hi = lo + (uint32_t)up;
        lo += step * c;
    }
    return lo;
}

// One boundary's bin, held by a wave: its samples as the low bits of their
// ordered keys, kLmCache per lane (a larger bin is read from memory).
struct LmBin {
    int bin;                 // -1: none yet
    int sh;                  // key bits below the bin number
    uint32_t klo;            // the bin's first key
    uint32_t cnt;
    uint64_t at;             // its first place
    double sum;
    const float *src;
    uint32_t low[kLmCache];
};

// fp64 sum of c samples of the bin whose ordered low bits sum to `low`
// (exact: sign * (count * base + ulp * sum of magnitude bits)).
__device__ __forceinline__ double lm_bin_value(const LmBin &B, uint64_t c, uint64_t low) {
    const uint32_t mask = (1u << B.sh) - 1u;
    const bool neg = (B.klo & 0x80000000u) == 0u;
    const uint32_t u = neg ? ~B.klo & 0x7fffffffu : B.klo & 0x7fffffffu;   // magnitude bits of the first key
    const uint32_t ex = (u >> 23) > 1u ? u >> 23 : 1u;
    const double base = (double)__uint_as_float(u & ~mask);
    const double ulp = __builtin_bit_cast(double, (uint64_t)(ex - 150u + 1023u) << 52);   // 2^(ex - 150)
    const uint64_t mag = neg ? c * mask - low : low;
    const double s = (double)c * base + ulp * (double)mag;
    return neg ? -s : s;
}

// Samples of the bin with ordered low bits <= t: their number and the sum of
// their low bits.
__device__ __forceinline__ void lm_scan_bin(const LmArgs &a, const LmBin &B, uint32_t t, int lane, uint64_t &c_out,
                                            uint64_t &s_out) {
    const uint32_t mask = (1u << B.sh) - 1u;
    if (B.sh <= 23 - a.mant) {
        // one value of the sample type: its low bits are zeros (of a negative key: ones)
        const uint32_t l = (B.klo & 0x80000000u) ? 0u : mask;
        c_out = l <= t ? B.cnt : 0u;
        s_out = (uint64_t)l * c_out;
        return;
    }
    if (B.cnt <= 64u * kLmCache) {
        uint32_t s = 0u, n = 0u;
#pragma unroll
        for (int q = 0; q < kLmCache / 4; ++q) {
            if (256u * q < B.cnt) {                    // wave-uniform
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t l = B.low[4 * q + k];
                    const bool in = l <= t;
                    n += in ? 1u : 0u;
                    s += in ? l : 0u;
                }
            }
        }
        // two 32-bit wave sums: s < 2^28 in an 18-bit part and the rest,
        // n <= 32 above the latter
        static_assert(kLmCache <= 32, "s and n of a lane fit their parts");
        const uint32_t p0 = lm_wave_sum_u32(s & 0x3ffffu), p1 = lm_wave_sum_u32((s >> 18) | (n << 18));
        c_out = p1 >> 18;
        s_out = ((uint64_t)(p1 & 0x3ffffu) << 18) + p0;
        return;
    }
    uint64_t s = 0, c = 0;
    for (uint32_t e = 0; e < B.cnt; e += 64u * 8u) {
        uint32_t l[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint32_t i = e + 64u * k + (uint32_t)lane;
            l[k] = i < B.cnt ? lm_key(B.src[i]) & mask : 0xffffffffu;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const bool in = l[k] <= t;
            c += (uint64_t)__popcll(__builtin_amdgcn_ballot_w64(in));
            s += in ? l[k] : 0u;
        }
    }
    c_out = c;
    s_out = (uint64_t)lm_wave_sum((double)s);          // < 2^53: exact
}

// Requests the samples of bin `bin` (first key klo, sh key bits below its
// number, cnt samples from place `at` on): raw until lm_settle_bin.
__device__ __forceinline__ void lm_open_bin(const LmArgs &a, int g, LmBin &B, int bin, uint32_t klo, int sh,
                                            uint64_t at, uint32_t cnt, int lane) {
    B.bin = bin;
    B.klo = klo;
    B.sh = sh;
    B.cnt = cnt;
    B.at = at;
    B.src = a.buf + (size_t)g * a.n + at;
    if (cnt > 0u && cnt <= 64u * kLmCache && sh > 23 - a.mant) {
        const uint32_t last = cnt - 1u;
#pragma unroll
        for (int q = 0; q < kLmCache / 4; ++q) {
            if (256u * q < cnt) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t i = 64u * (4 * q + k) + (uint32_t)lane;
                    B.low[4 * q + k] = __float_as_uint(B.src[i < last ? i : last]);
                }
            }
        }
    }
}

// Raw samples to ordered low bits, lanes past the last to all ones.
__device__ __forceinline__ void lm_settle_bin(LmBin &B, int lane) {
    const uint32_t flip = (B.klo & 0x80000000u) ? 0x80000000u : 0xffffffffu;   // key = u ^ flip (one sign)
#pragma unroll
    for (int q = 0; q < kLmCache / 4; ++q) {
        if (256u * q < B.cnt && B.cnt <= 64u * kLmCache) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t i = 64u * (4 * q + k) + (uint32_t)lane;
                const uint32_t l = (B.low[4 * q + k] ^ flip) - B.klo;
                B.low[4 * q + k] = i < B.cnt ? l : 0xffffffffu;
            }
        }
    }
}

// First-index argmin of |x - c_k| (c_k NaN: no candidate), and whether the next
// distance lies far enough above the least one (by 2^-20 of it; rounding moves
// either by 2^-24) that the real distances decide, not their rounding.
__device__ __forceinline__ bool lm_code(const float *c, float x, int &code) {
    float best = fabsf(x - c[0]), second = INFINITY;
    code = 0;
#pragma unroll
    for (int k = 1; k < kLmK; ++k) {
        const float d = fabsf(x - c[k]);
        second = d < best ? best : fminf(second, d);
        code = d < best ? k : code;
        best = fminf(best, d);
    }
    return best < 1e38f && second > best * 1.00000095367431640625f;
}

// The whole calibration of a group: wave w finds order statistic w and then,
// each step, boundary w and the mean of cell w.
template <int DT>
__global__ __launch_bounds__(kLmThreads) void lm_lloyd_kernel(LmArgs a) {
    __shared__ uint32_t place[kLmMaxBins + 4];         // first places of the bins
    __shared__ double csum[kLmMaxBins / 64];
    __shared__ uint32_t map[kLmOct];
    __shared__ float cent2[2][kLmK], moved[kLmK];
    __shared__ int bbin[kLmK];                         // boundary w: its bin (nb: none),
    __shared__ uint64_t bcnt[kLmK];                    // the group's samples on its left,
    __shared__ double bval[kLmK], bright[kLmK];        // the sums of its bin's samples on its left and right,
    __shared__ double bhead[kLmK], btail[kLmK];        // and of the chunk's bins before and after that bin
    __shared__ int slow;
    __shared__ float live[kLmK];                       // step by bins: the centroids, equal ones once (else NaN),
    __shared__ double tsum[kLmThreads / 64][kLmK];                // each wave's sums and counts of the cells
    __shared__ uint64_t tcnt[kLmThreads / 64][kLmK];
    const int g = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const double *bsum = a.bsum + (size_t)g * a.nb;
    const uint64_t *start = a.start + (size_t)g * (a.nb + 1);
    if (!a.wide)                                       // (64-bit places stay in memory)
        for (int b = tid; b <= a.nb; b += kLmThreads) place[b] = (uint32_t)start[b];
    auto first_of = [&](int b) -> uint64_t { return a.wide ? start[b] : (uint64_t)place[b]; };
    for (int c = tid; c < a.nch; c += kLmThreads) csum[c] = a.csum[(size_t)g * a.nch + c];
    if (tid < kLmOct) map[tid] = a.map[(size_t)g * kLmOct + tid];
    __syncthreads();

    LmBin B;
    B.bin = -1;
    B.cnt = 0u;
    // Boundary w moves to the bin with first key klo: the one memory round
    // trip of a step.  Its samples and its chunk's sums are requested together.
    auto go_to = [&](int bin, uint32_t klo, int sh) {
        if (bin == B.bin) return;
        const uint64_t at = first_of(bin), end = first_of(bin + 1);
        const uint32_t at_lo = __builtin_amdgcn_readfirstlane((uint32_t)at);
        const uint32_t at_hi = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32));
        const uint32_t n = __builtin_amdgcn_readfirstlane((uint32_t)(end - at));
        const double mine = bsum[(bin & ~63) + lane];
        lm_open_bin(a, g, B, bin, klo, sh, ((uint64_t)at_hi << 32) | at_lo, n, lane);
        lm_settle_bin(B, lane);
        B.sum = lm_lane(mine, bin & 63);
        const double head = lm_wave_sum(lane < (bin & 63) ? mine : 0.0);
        const double tail = lm_wave_sum(lane > (bin & 63) ? mine : 0.0);
        if (lane == 0) {
            bhead[w] = head;
            btail[w] = tail;
        }
    };
    // `c` of the bin's samples, `s` the sum of their low bits, lie on the left
    auto set_left = [&](uint64_t c, uint64_t s) {
        const double left = lm_bin_value(B, c, s);
        if (lane == 0) {
            bbin[w] = B.bin;
            bcnt[w] = B.at + c;
            bval[w] = left;
            bright[w] = B.sum - left;                  // exact
        }
    };
    // first key and shift of a bin
    auto bin_key = [&](int bin, uint32_t &klo, int &sh) {
        int o = 0;
#pragma unroll
        for (int q = 0; q < kLmOct / 64; ++q)
            o += __popcll(__builtin_amdgcn_ballot_w64((int)(map[64 * q + lane] >> 5) <= bin));
        o -= 1;
        const uint32_t m = __builtin_amdgcn_readfirstlane(map[o]);
        sh = (int)(m & 31u);
        klo = ((uint32_t)o << 23) | ((uint32_t)(bin - (int)(m >> 5)) << sh);
    };
    // bin of the sample of rank k
    auto bin_of_rank = [&](uint64_t k) {
        int lo = 0, hi = a.nb;
        while (hi - lo > 1) {
            const int step = (hi - lo + 63) >> 6;
            const int at = lo + step * (lane + 1);
            const int c = __popcll(__builtin_amdgcn_ballot_w64(at < hi && first_of(at < hi ? at : hi) <= k));
            const int up = lo + step * (c + 1);
            hi = up < hi ? up : hi;
            lo += step * c;
        }
        return lo;
    };
    uint32_t klo;
    int sh;
    bin_key(bin_of_rank((uint64_t)a.n - 1u), klo, sh);
    const float xmax = lm_value(klo | ((1u << sh) - 1u));      // the data's largest value, or a little more
    {
        const uint64_t k = (uint64_t)(w + 1) * (uint64_t)a.bs - 1u;
        const int bin = bin_of_rank(k);
        bin_key(bin, klo, sh);
        go_to(bin, klo, sh);
        const uint64_t kk = k - B.at;
        // smallest low bits with more than kk samples at or below
        uint32_t lo = 0u, hi = (1u << sh) - 1u;
        uint64_t c, s;
        while (lo < hi) {
            const uint32_t mid = lo + ((hi - lo) >> 1);
            lm_scan_bin(a, B, mid, lane, c, s);
            if (c > kk) hi = mid;
            else lo = mid + 1u;
        }
        lm_scan_bin(a, B, lo, lane, c, s);
        // of the samples equal to it, those up to rank k
        set_left(kk + 1u, s - (c - (kk + 1u)) * lo);
    }
    __syncthreads();

    // samples and sum of cell w: right part of the bin of boundary w - 1, the
    // whole bins between, left part of the bin of boundary w
    int kl = -2, kr = -2;
    double kmid = 0.0;                                 // whole chunks between, kept with (kl, kr)
    auto cell = [&](uint64_t &n, double &s) {
        const int L = w > 0 ? __builtin_amdgcn_readfirstlane(bbin[w - 1]) : -1;
        const int R = __builtin_amdgcn_readfirstlane(bbin[w]);
        n = (R < a.nb ? bcnt[w] : (uint64_t)a.n) - (w > 0 ? bcnt[w - 1] : 0u);
        if (L == R) {
            s = bval[w] - bval[w - 1];
            return;
        }
        const int cl = L >= 0 ? L >> 6 : -1, cr = R >> 6;
        if (L != kl || R != kr) {
            kl = L;
            kr = R;
            double t = 0.0;
            if (cl == cr) {                            // within one chunk
                const int b = L + 1 + lane;
                if (b < R) t = bsum[b];
            } else {
                for (int c = cl + 1 + lane; c < cr; c += 64) t += csum[c];
            }
            kmid = lm_wave_sum(t);
        }
        s = kmid;
        if (cl != cr) {
            if (L >= 0) s += btail[w - 1];
            if (R < a.nb) s += bhead[w];
        }
        if (L >= 0) s += bright[w - 1];
        if (R < a.nb) s += bval[w];
    };
    {
        uint64_t n;
        double s;
        cell(n, s);
        if (lane == 0) cent2[0][w] = (float)(s / (double)a.bs);
    }
    __syncthreads();

    float pa = NAN, pb = NAN;                          // the pair this wave's boundary was found for
    int it = 0;
    for (; it < a.max_iters; ++it) {
        const float *cent = cent2[it & 1];
        const float ck = cent[lane & (kLmK - 1)];
        const float ca = lm_lane(ck, w);
        const uint32_t rest = (uint32_t)__builtin_amdgcn_ballot_w64(lane < kLmK && lane > w && ck != ca);
        const float cb = rest ? lm_lane(ck, __builtin_ctz(rest)) : ca;     // next distinct centroid
        if (w < kLmK - 1 && !(ca == pa && cb == pb)) {
            pa = ca;
            pb = cb;
            if (ca < cb) {
                const uint32_t key = lm_threshold(ca, cb, lane);
                const uint32_t m = __builtin_amdgcn_readfirstlane(map[key >> 23]);
                const uint32_t mask = (1u << (m & 31u)) - 1u;
                go_to((int)lm_bin(m, key), key & ~mask, (int)(m & 31u));
                uint64_t c, s;
                lm_scan_bin(a, B, key & mask, lane, c, s);
                set_left(c, s);
            } else if (lane == 0) {
                bbin[w] = a.nb;
            }
        }
        if (w == kLmK - 1) {
            // Boundaries decide the codes if the centroids ascend and no
            // distance to a lower centroid can round to a tie with the
            // nearest one: gap >= 2 ulp of the largest distance compared.
            bool bad = false;
            const float up = __shfl_down(ck, 1);
            if (lane < kLmK - 1) bad = !(ck <= up);
            float lower = 0.0f;
            bool have = false;
            for (int j = 0; j < kLmK; ++j) {
                const float c = lm_lane(ck, j);
                if (lane < kLmK && j < lane && c != ck) { lower = c; have = true; }
            }
            float next = fmaxf(xmax, ck);
            for (int j = kLmK - 1; j >= 0; --j) {
                const float c = lm_lane(ck, j);
                if (lane < kLmK && j > lane && c != ck) next = c;
            }
            if (lane < kLmK && have) bad = bad || !((ck - lower) >= (next - lower) * 2.384185791015625e-7f);
            if (lane < kLmK) bad = bad || !(fabsf(ck) <= FLT_MAX) || !(fabsf(xmax - ck) <= FLT_MAX);
            const bool any = __builtin_amdgcn_ballot_w64(bad) != 0ull;
            if (lane == 0) {
                slow = any ? 1 : 0;
                bbin[w] = a.nb;
            }
        }
        __syncthreads();
        uint64_t n = 0;
        double s = 0.0;
        if (!__builtin_amdgcn_readfirstlane(slow)) {
            // a centroid equal to the one before it gets no sample (first index)
            if (w == 0 || lm_lane(ck, w > 0 ? w - 1 : 0) != ca) cell(n, s);
        } else {
            // Bin by bin: both ends coded alike, and neither near a tie, code
            // the whole bin (between them |x - c_j| - (1 + 2^-22) |x - c_k| is
            // least at an end); the others' samples are coded one by one.  Sums
            // inside a bin are exact, bins and waves are added in a fixed order.
            // 8 groups x 1.64 M samples, one of them 1e8: 28 us a step (3 us
            // where boundaries decide; one by one in this block 3570 us, in
            // a pass of 240 blocks over the samples 62 us).
            if (tid < kLmK) {
                bool again = false;
                for (int j = 0; j < tid; ++j) again = again || cent[j] == cent[tid];
                live[tid] = again ? __builtin_nanf("") : cent[tid];
            }
            __syncthreads();
            const float *buf = a.buf + (size_t)g * a.n;
            double ts = 0.0;                           // lane k: cell k
            uint64_t tn = 0;
            for (int b0 = 64 * w; b0 < a.nb; b0 += kLmThreads) {
                const uint64_t at = first_of(b0 + lane), c = first_of(b0 + lane + 1) - at;
                const double sum = bsum[b0 + lane];
                int code = 0, code1 = 0;
                bool whole = false;
                if (c > 0) {
                    const uint32_t key = lm_key(buf[at]), mask = (1u << (map[key >> 23] & 31u)) - 1u;
                    const bool sure0 = lm_code(live, lm_value(key & ~mask), code);
                    const bool sure1 = lm_code(live, lm_value(key | mask), code1);
                    whole = sure0 && sure1 && code == code1;
                }
                for (uint64_t left = __builtin_amdgcn_ballot_w64(whole); left;) {
                    const int k = __builtin_amdgcn_readlane(code, __builtin_ctzll(left));
                    const bool mine = whole && code == k;
                    const double s1 = lm_wave_sum(mine ? sum : 0.0), n1 = lm_wave_sum(mine ? (double)c : 0.0);
                    ts += lane == k ? s1 : 0.0;
                    tn += lane == k ? (uint64_t)n1 : 0u;
                    left &= ~__builtin_amdgcn_ballot_w64(mine);
                }
                for (uint64_t left = __builtin_amdgcn_ballot_w64(c > 0 && !whole); left; left &= left - 1u) {
                    const int l = __builtin_ctzll(left);
                    const uint64_t first = __shfl((unsigned long long)at, l), nl = __shfl((unsigned long long)c, l);
                    double bs = 0.0;
                    for (uint64_t e = 0; e < nl; e += 256u) {
                        float x[4];
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const uint64_t i = e + 64u * q + (uint32_t)lane;
                            x[q] = buf[first + (i < nl ? i : nl - 1u)];
                        }
#pragma unroll 1
                        for (int q = 0; q < 4; ++q) {
                            const bool in = e + 64u * q + (uint32_t)lane < nl;
                            int cx;
                            lm_code(live, x[0], cx);
                            for (uint64_t some = __builtin_amdgcn_ballot_w64(in); some;) {
                                const int k = __builtin_amdgcn_readlane(cx, __builtin_ctzll(some));
                                const bool mine = in && cx == k;
                                const uint64_t m = __builtin_amdgcn_ballot_w64(mine);
                                const double s1 = lm_wave_sum(mine ? (double)x[0] : 0.0);
                                bs += lane == k ? s1 : 0.0;
                                tn += lane == k ? (uint64_t)__popcll(m) : 0u;
                                some &= ~m;
                            }
                            x[0] = x[1]; x[1] = x[2]; x[2] = x[3];
                        }
                    }
                    ts += bs;
                }
            }
            if (lane < kLmK) {
                tsum[w][lane] = ts;
                tcnt[w][lane] = tn;
            }
            __syncthreads();
            for (int v = 0; v < kLmThreads / 64; ++v) {
                s += tsum[v][w];
                n += tcnt[v][w];
            }
        }
        const float nc = n > 0 ? (float)(s / (double)n) : ca;
        if (lane == 0) {
            moved[w] = fabsf(nc - ca);
            cent2[(it + 1) & 1][w] = nc;
        }
        __syncthreads();
        const float mv = moved[lane & (kLmK - 1)];
        if (__builtin_amdgcn_ballot_w64(!(mv < a.tol) && mv == mv) == 0ull) {
            ++it;
            break;
        }
    }
    // sorted ascending
    if (tid == 0) {
        float c[kLmK];
        for (int k = 0; k < kLmK; ++k) c[k] = cent2[it & 1][k];
        for (int i = 1; i < kLmK; ++i) {
            const float v = c[i];
            int j = i - 1;
            while (j >= 0 && c[j] > v) {
                c[j + 1] = c[j];
                --j;
            }
            c[j + 1] = v;
        }
        for (int k = 0; k < kLmK; ++k) a.out[g * kLmK + k] = c[k];
        if (a.iters) a.iters[g] = it;
    }
}

// Bins by the samples per group: kLmFill samples a bin, or as many as keep
// 2 n / fill + 512 within kLmMaxBins.
static void lm_shape(int x_dtype, int64_t n, LmArgs &a) {
    const int64_t least = (n + (kLmMaxBins - kLmOct) / 2 - 1) / ((kLmMaxBins - kLmOct) / 2);
    a.fill = least > kLmFill ? least : kLmFill;
    const int64_t bins = 2 * (n / a.fill) + kLmOct;
    a.nb = (int)(bins < kLmMaxBins ? (bins + 63) / 64 * 64 : kLmMaxBins);
    a.nch = a.nb / 64;
    a.mant = x_dtype == OMNI_F32 ? 23 : (x_dtype == OMNI_BF16 ? 7 : 10);
    a.wide = n >= (int64_t(1) << 32) ? 1 : 0;
}

// Workspace carve-up; returns the total bytes (base may be null to size).
static size_t lm_layout(int groups, int64_t n, char *base, LmArgs &a) {
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char *p = base ? base + off : nullptr;
        off = lm_align256(off + bytes);
        return p;
    };
    const size_t gr = (size_t)groups;
    a.oct = reinterpret_cast<uint32_t *>(take(gr * kLmOct * 4));
    a.map = reinterpret_cast<uint32_t *>(take(gr * kLmOct * 4));
    a.cnt = reinterpret_cast<uint32_t *>(take(gr * a.nb * 4));
    a.cursor = reinterpret_cast<uint32_t *>(take(gr * a.nb * 4));
    a.start = reinterpret_cast<uint64_t *>(take(gr * (a.nb + 1) * 8));
    a.bsum = reinterpret_cast<double *>(take(gr * a.nb * 8));
    a.csum = reinterpret_cast<double *>(take(gr * a.nch * 8));
    a.buf = reinterpret_cast<float *>(take(gr * (size_t)n * 4));
    return off;
}

template <int DT>
static void lm_launch(const LmArgs &a, int groups, hipStream_t st) {
    const unsigned gr = (unsigned)groups;
    const dim3 grid((unsigned)((a.n + kLmBlock - 1) / kLmBlock), gr), block(kLmThreads);
    const int clear = a.nb > kLmOct ? a.nb : kLmOct;
    hipLaunchKernelGGL(lm_clear_kernel, dim3((unsigned)((clear + 255) / 256), gr), dim3(256), 0, st, a);
    hipLaunchKernelGGL((lm_oct_kernel<DT>), grid, block, 0, st, a);
    hipLaunchKernelGGL(lm_map_kernel, dim3(gr), dim3(kLmOct), 0, st, a);
    hipLaunchKernelGGL((lm_count_kernel<DT>), grid, block, 0, st, a);
    hipLaunchKernelGGL(lm_scan_kernel, dim3((unsigned)((a.nb + kLmScan - 1) / kLmScan), gr), block, 0, st, a);
    hipLaunchKernelGGL((lm_store_kernel<DT>), grid, block, 0, st, a);
    hipLaunchKernelGGL(lm_binsum_kernel, dim3((unsigned)((a.n + 4095) / 4096), gr), dim3(256), 0, st, a);
    hipLaunchKernelGGL(lm_chunk_kernel, dim3((unsigned)((a.nch + 15) / 16), gr), block, 0, st, a);
    hipLaunchKernelGGL((lm_lloyd_kernel<DT>), dim3(gr), block, 0, st, a);
}

}  // namespace omni

using namespace omni;

extern "C" size_t omni_lloyd_max_workspace_size(int n_groups, int64_t outer, int64_t inner) {
    if (n_groups <= 0 || outer <= 0 || inner <= 0 || outer > INT64_MAX / inner) return 0;
    LmArgs a;
    lm_shape(OMNI_F32, outer * inner, a);
    return lm_layout(n_groups, outer * inner, nullptr, a);
}

extern "C" size_t omni_lloyd_max_workspace_least(int n_groups, int64_t outer, int64_t inner) {
    if (n_groups <= 0 || outer <= 0 || inner <= 0 || outer > INT64_MAX / inner) return 0;
    const size_t all = omni_lloyd_max_workspace_size(n_groups, outer, inner);
    const size_t least = lm_inplace_bytes(n_groups, outer * inner);
    return least < all ? least : all;
}

extern "C" int omni_lloyd_max(const void *x, int x_dtype, int n_groups, int64_t outer, int64_t inner,
                              int64_t outer_stride, int64_t group_stride, int max_iters, float tol,
                              float *codebooks, int32_t *iters_out, void *workspace, size_t workspace_bytes,
                              void *stream) {
    OMNI_CHECK_ARG(dtype_ok(x_dtype), "omni_lloyd_max: bad dtype %d", x_dtype);
    OMNI_CHECK_ARG(n_groups >= 1 && n_groups <= 65535, "omni_lloyd_max: need 1 <= n_groups <= 65535");
    OMNI_CHECK_ARG(outer >= 1 && inner >= 1 && outer_stride >= 0 && group_stride >= 0,
                   "omni_lloyd_max: bad sample layout");
    OMNI_CHECK_ARG(outer <= INT64_MAX / inner, "omni_lloyd_max: too many samples");
    const int64_t n = outer * inner;
    OMNI_CHECK_ARG(n >= kLmK, "omni_lloyd_max: need at least 16 samples per group, got %lld", (long long)n);
    OMNI_CHECK_ARG(max_iters >= 0 && max_iters <= 100000, "omni_lloyd_max: max_iters must be in [0, 100000]");
    OMNI_CHECK_ARG(x && codebooks, "omni_lloyd_max: NULL pointer");
    const size_t least = omni_lloyd_max_workspace_least(n_groups, outer, inner);
    if (workspace == nullptr || workspace_bytes < least) {
        set_error("omni_lloyd_max: workspace of %zu bytes required, %zu given", least, workspace_bytes);
        return OMNI_EWORKSPACE;
    }
    hipStream_t st = as_stream(stream);
    if (workspace_bytes < omni_lloyd_max_workspace_size(n_groups, outer, inner)) {
        lm_inplace_run({x, x_dtype, n_groups, outer, inner, outer_stride, group_stride, max_iters, tol, codebooks, iters_out},
                       workspace, st);
        OMNI_CHECK_LAUNCH("omni_lloyd_max");
        return OMNI_OK;
    }
    LmArgs a;
    a.x = x;
    a.outer = outer; a.inner = inner; a.outer_stride = outer_stride; a.group_stride = group_stride;
    a.n = n;
    a.bs = n / kLmK;
    a.max_iters = max_iters;
    a.tol = tol;
    a.out = codebooks;
    a.iters = iters_out;
    lm_shape(x_dtype, n, a);
    // 4-element loads: every run of four lies in one row and is aligned
    a.vec = (inner % 4 == 0 && outer_stride % 4 == 0 && group_stride % 4 == 0 &&
             (uintptr_t)x % (4 * dtype_size(x_dtype)) == 0) ? 1 : 0;
    lm_layout(n_groups, n, reinterpret_cast<char *>(workspace), a);
    if (x_dtype == OMNI_F32) lm_launch<OMNI_F32>(a, n_groups, st);
    else if (x_dtype == OMNI_BF16) lm_launch<OMNI_BF16>(a, n_groups, st);
    else lm_launch<OMNI_F16>(a, n_groups, st);
    OMNI_CHECK_LAUNCH("omni_lloyd_max");
    return OMNI_OK;
}
