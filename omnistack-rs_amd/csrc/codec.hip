// gfx950 codec kernels: WHT rotation, fused INT4 + QJL encoder, dequantizer.
//
// Bit-level contract (reference deepsheth3/Omnistack-RS, Python/torch):
//   rotation   omnistack_rs/kernels/hadamard.py:51-85   (_wht_torch)
//   encoder    omnistack_rs/kernels/quantize.py:542-590 (quantize_heads)
//              + :361-377 (argmin, nibble pack) + :398-423 (QJL signs)
//   decoder    omnistack_rs/kernels/quantize.py:593-640 (dequantize_heads)
//              + :380-395 (unpack) + :426-451 (QJL reconstruct)
// The library is built with -ffp-contract=off: every fp32 operation below
// rounds exactly where the reference's torch ops round.
#include <math.h>

#include "omni_common.h"

namespace omni {

typedef float float4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t cvt_pk_f16(float x, float y) {
    typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
    typedef float f2_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){x, y}, h2_t));
}

// ── omni_encode ─────────────────────────────────────────────────────────
//
// Two wave kernels: encode128_kernel (16-bit input, D = 128: codes from a
// table of all values) and encode_grid_kernel (the rest).  For each row
//   code_d = argmin_k fp32 |x_d - c_k|, first index on ties; a NaN distance
//            is the minimum (torch.argmin), which only matters when the
//            codebook itself holds a NaN
//   e = x - c[code] (fp32), norm = ||e||_2, bit_i = [G_i . e >= 0]
//
// ── 16-bit input, D = 128 ───────────────────────────────────────────────
//
//   * 16 rows per wave-iteration; lane (n, g) holds elements 32 s + 8 g + i
//     (s < 4, i < 8) of row n.  The WHT runs in registers (h = 1, 2, 4, 32,
//     64) and by paired v_permlane16/32_swap butterflies (h = 8, 16), in the
//     reference stage order with the reference's fp32 operations.
//   * Codes come from a 64 KB LDS table indexed by the rotated value's
//     16-bit pattern, built exactly (brute-force first-index argmin with the
//     NaN rule) by code_table_kernel into the caller's workspace.
//   * QJL projections P = E G^T on v_mfma_f32_16x16x32_bf16: each residual
//     is split into two round-to-nearest bf16 parts (the dropped remainder is
//     below 2^-16 |e|), G is exactly +-1, so the products are exact and the
//     error (fp32 accumulation plus the remainder) is bounded by
//     1312 * 2^-24 * sum|e| (+ 2^-100 for flushed denormals).  Signs outside
//     the bound are certain; the rare rest are recomputed in fp64 with
//     compensated sums.  Rows with a non-finite residual take the
//     order-free sign of the reference's fp32 sum (NaN if it meets NaN or
//     both infinities, else the sign of the infinity).
//   * With A = G rows and B = the residual rows, lane (n, g) receives
//     P[n][16 cb + 4 g + i]: every value a lane needs for its row is local
//     or one 4-lane reduction away.

constexpr int kEncWaves = 12;
constexpr int kEncTab = 65536;                            // u8 code table (both nibbles = code)
constexpr int kEncCentOff = kEncTab;                      // f32 centroid by table byte (256 slots)
constexpr int kEncGimgOff = kEncCentOff + 256 * 4;        // [cb][s][lane] uint4: 8 bf16 +-1 of G
constexpr int kEncGbitsOff = kEncGimgOff + 4 * 4 * 64 * 16;   // G rows as bits, 64 x 4 words
constexpr int kEncFlipOff = kEncGbitsOff + 64 * 4 * 4;       // [lane][16] u32: sign-bit xor of the raw 16-bit words
constexpr int kEncStageOff = kEncFlipOff + 64 * 16 * 4;      // [wave][128] f32: one residual row (rare paths)
constexpr int kEncLdsBytes = kEncStageOff + kEncWaves * 128 * 4;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

struct EncArgs {
    const void *x[2];            // one or two tensors of the same shape (blockIdx.z)
    const uint8_t *table;        // n_tables x 65536
    const float *codebooks;
    const uint32_t *g_bits;
    const int8_t *sign_flip;
    uint8_t *nibbles[2], *qjl[2];
    float *norms[2];
    int64_t T, nrows_head, rows_per_block[2];    // per tensor
    int nx0;                                      // paged: blocks of the first tensor
    int H, per_head, rotate;
    float scale;
    // paged output (encode128_kernel<..., true>): row (b, h, t) goes to pool
    // row (page_table[b][p >> page_shift] * H + h) * page_size + p %
    // page_size, p = positions[b] + t; rows whose page is outside the pool
    // (or past the table) are not written; the second tensor (V) writes
    // its codes only
    const int32_t *page_table, *positions;
    int64_t max_pages, n_pages;
    int page_shift;
    // encode_grid_kernel: rows between a wave's groups as (batch entries, tokens)
    int64_t step_b, step_t;
};

template <int XDT>
__global__ __launch_bounds__(256) void code_table_kernel(const float *codebooks, int per_head, uint8_t *table) {
    const int h = blockIdx.y;
    const uint32_t u = blockIdx.x * 256u + threadIdx.x;
    const float v = XDT == OMNI_BF16 ? bf16_to_f32((uint16_t)u) : f16_to_f32((uint16_t)u);
    const float *cbp = codebooks + (per_head ? h * 16 : 0);
    float cb[16];
    bool cb_nan = false;
#pragma unroll
    for (int k = 0; k < 16; ++k) { cb[k] = cbp[k]; cb_nan |= (cb[k] != cb[k]); }
    float best = fabsf(v - cb[0]);
    int code = 0;
#pragma unroll
    for (int k = 1; k < 16; ++k) {
        const float dk = fabsf(v - cb[k]);
        bool take = dk < best;
        if (cb_nan) take = take || ((dk != dk) && (best == best));
        best = take ? dk : best;
        code = take ? k : code;
    }
    table[(int64_t)h * kEncTab + u] = (uint8_t)(code | (code << 4));
}

// ── omni_wht_rotate ─────────────────────────────────────────────────────
//
// Normalized WHT in the reference's butterfly order h = 1, 2, ..., D/2
// ((upper, lower) -> (upper + lower, upper - lower)), memory-bound.  A wave
// takes 16 rows of 128 (64 of 32); lane (n, g) holds 32 values of row n as
// x[s][i] (D = 32: s is a 16-row set), with the element bits spread so that
// every 16-byte access of four lanes covers 64 consecutive bytes:
//   16-bit  element 32 s + 8 g + i
//   f32     element 32 s + 16 (i / 4) + 4 g + i % 4
// 102,400 f32 rows of 128: 85 us with a lane per row before, 19 us (5.5 TB/s)
// now; 2^20 bf16 rows 1360 -> 104 us.
constexpr int64_t kWhtGridX = 65536;

template <int XDT, int D>
__global__ __launch_bounds__(256) void wht_kernel(const void *x, int64_t rows, const int8_t *sign_flip, void *out,
                                                  float scale) {
    constexpr int kSets = D == 128 ? 1 : 4;
    constexpr bool F32 = XDT == OMNI_F32;
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int64_t v0 = (((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 4 + (threadIdx.x >> 6)) * (16 * kSets);
    if (v0 >= rows) return;
    auto at = [&](int s, int i) {                      // element offset of x[s][i] (i a multiple of 4 or 8)
        const int64_t r = v0 + n + (D == 128 ? 0 : 16 * s);
        return (r < rows ? r : rows - 1) * D + (D == 128 ? 32 * s : 0) + (F32 ? 4 * i + 4 * g : 8 * g + i);
    };
    float v[4][8];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if constexpr (F32) {
#pragma unroll
            for (int i = 0; i < 8; i += 4) {
                const float4 t = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(x) + at(s, i));
                v[s][i] = t.x; v[s][i + 1] = t.y; v[s][i + 2] = t.z; v[s][i + 3] = t.w;
            }
        } else {
            const uint4 t = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(x) + at(s, 0));
            const uint32_t w[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint16_t u = (uint16_t)((i & 1) ? w[i >> 1] >> 16 : w[i >> 1] & 0xffffu);
                v[s][i] = XDT == OMNI_BF16 ? bf16_to_f32(u) : f16_to_f32(u);
            }
        }
    }
    if (sign_flip) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int d = (D == 128 ? 32 * s : 0) + (F32 ? 16 * (i >> 2) + 4 * g + (i & 3) : 8 * g + i);
                v[s][i] = sign_flip[d] < 0 ? -v[s][i] : v[s][i];
            }
    }
    auto in_lane = [&](int hh) {                       // register index bit hh
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (!(i & hh)) {
                    const float u = v[s][i], l = v[s][i + hh];
                    v[s][i] = u + l;
                    v[s][i + hh] = u - l;
                }
    };
    in_lane(1);
    in_lane(2);
    if (!F32) in_lane(4);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 8; i += 2) xlane_pair_butterfly<16>(v[s][i], v[s][i + 1]);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 8; i += 2) xlane_pair_butterfly<32>(v[s][i], v[s][i + 1]);
    if (F32) in_lane(4);
    if constexpr (D == 128) {
#pragma unroll
        for (int hs = 1; hs < 4; hs <<= 1)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (!(s & hs))
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const float u = v[s][i], l = v[s + hs][i];
                        v[s][i] = u + l;
                        v[s + hs][i] = u - l;
                    }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const bool ok = v0 + n + (D == 128 ? 0 : 16 * s) < rows;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[s][i] *= scale;
            // rounded to fp32 before f16 (v_fma_mixlo_f16 would round once)
            if (XDT == OMNI_F16) asm volatile("" : "+v"(v[s][i]));
        }
        if (!ok) continue;
        if constexpr (F32) {
#pragma unroll
            for (int i = 0; i < 8; i += 4)
                *reinterpret_cast<float4 *>(reinterpret_cast<float *>(out) + at(s, i)) =
                    make_float4(v[s][i], v[s][i + 1], v[s][i + 2], v[s][i + 3]);
        } else {
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float p = v[s][2 * j], q = v[s][2 * j + 1];
                w[j] = XDT == OMNI_BF16 ? (uint32_t)f32_to_bf16_rne(p) | ((uint32_t)f32_to_bf16_rne(q) << 16)
                                        : (uint32_t)f32_to_f16_rne(p) | ((uint32_t)f32_to_f16_rne(q) << 16);
            }
            *reinterpret_cast<uint4 *>(reinterpret_cast<uint16_t *>(out) + at(s, 0)) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

template <int HALF>
__device__ __forceinline__ double xlane_sum_f64(double v) {
    const uint64_t bits = __builtin_bit_cast(uint64_t, v);
    uint32_t lo = (uint32_t)bits, hi = (uint32_t)(bits >> 32), plo, phi;
    if constexpr (HALF == 16) {
        const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        const bool odd = (__lane_id() & 16) != 0;
        plo = odd ? a[0] : a[1];
        phi = odd ? b[0] : b[1];
    } else {
        const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        const bool up = (__lane_id() & 32) != 0;
        plo = up ? a[0] : a[1];
        phi = up ? b[0] : b[1];
    }
    return v + __builtin_bit_cast(double, ((uint64_t)phi << 32) | plo);
}

template <int HALF>
__device__ __forceinline__ uint32_t xlane_u32(uint32_t v) {
    if constexpr (HALF == 16) {
        const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (__lane_id() & 16) ? a[0] : a[1];
    } else {
        const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return (__lane_id() & 32) ? a[0] : a[1];
    }
}

__device__ __forceinline__ float xlane_sum_f32(float v) {
    v += __uint_as_float(xlane_u32<16>(__float_as_uint(v)));
    return v + __uint_as_float(xlane_u32<32>(__float_as_uint(v)));
}

// sum_j s_j e_j over one staged residual row (128 floats in LDS) for G row
// `grow` (4 words): each lane takes elements lane and lane + 64 in fp64 and
// the wave reduces (sum, error) pairs with TwoSum, so the result is the exact
// sum up to ~1e-30 relative.  Commutative steps: every lane gets the same
// value.  `fl` collects the order-free classes of the terms (1 NaN, 2 +inf,
// 4 -inf), OR-reduced over the wave.
__device__ __forceinline__ double wave_row_dot(const float *st, const uint32_t *grow, int lane, uint32_t &fl) {
    const float e1 = st[lane], e2 = st[lane + 64];
    const uint32_t b1 = (grow[lane >> 5] >> (lane & 31)) & 1u, b2 = (grow[2 + (lane >> 5)] >> (lane & 31)) & 1u;
    const float f1 = b1 ? e1 : -e1, f2 = b2 ? e2 : -e2;
    uint32_t cls = 0u;
    cls |= (f1 != f1) ? 1u : (f1 == INFINITY ? 2u : (f1 == -INFINITY ? 4u : 0u));
    cls |= (f2 != f2) ? 1u : (f2 == INFINITY ? 2u : (f2 == -INFINITY ? 4u : 0u));
    fl = (__builtin_amdgcn_ballot_w64((cls & 1u) != 0u) ? 1u : 0u) | (__builtin_amdgcn_ballot_w64((cls & 2u) != 0u) ? 2u : 0u) |
         (__builtin_amdgcn_ballot_w64((cls & 4u) != 0u) ? 4u : 0u);
    const double y1 = (double)f1, y2 = (double)f2;
    double s = y1 + y2;
    double bp = s - y1;
    double c = (y1 - (s - bp)) + (y2 - bp);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        const double so = __shfl_xor(s, m), co = __shfl_xor(c, m);
        const double t = s + so;
        bp = t - s;
        const double err = (s - (t - bp)) + (so - bp);
        s = t;
        c = (c + co) + err;
    }
    return s + c;
}

template <int XDT, bool ROT, bool PAGED>
__global__ __launch_bounds__(64 * kEncWaves) void encode128_kernel(EncArgs a) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[kEncLdsBytes];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int h = blockIdx.y;
    // tensor zb (K or V of one encode_pair call): blockIdx.z, or (paged, where
    // K and V take different block counts) blocks x >= nx0 of one row
    const int zb = PAGED ? (blockIdx.x >= (unsigned)a.nx0 ? 1 : 0) : (int)blockIdx.z;
    const int64_t xb = PAGED && zb ? (int64_t)blockIdx.x - a.nx0 : (int64_t)blockIdx.x;
    const void *const xz = a.x[zb];
    uint8_t *const nibz = a.nibbles[zb];
    uint8_t *const qjlz = a.qjl[zb];
    float *const nrmz = a.norms[zb];
    const int64_t rpb = a.rows_per_block[zb];
    const int64_t v_begin = xb * rpb;
    if (v_begin >= a.nrows_head) return;                     // block-uniform, before any barrier
    const int64_t v_end = v_begin + rpb < a.nrows_head ? v_begin + rpb : a.nrows_head;

    // ── prologue: code table, centroids, G bits and bf16 images ───────
    {
        const uint4 *src = reinterpret_cast<const uint4 *>(a.table + (int64_t)(a.per_head ? h : 0) * kEncTab);
        uint4 *dst = reinterpret_cast<uint4 *>(smem);
        for (int k = tid; k < kEncTab / 16; k += 64 * kEncWaves) dst[k] = src[k];
    }
    const float *cbp = a.codebooks + (a.per_head ? h * 16 : 0);
    if (tid < 16) reinterpret_cast<float *>(smem + kEncCentOff)[tid | (tid << 4)] = cbp[tid];
    const uint32_t *gh = a.g_bits + (int64_t)h * 64 * 4;
    if (tid < 256) reinterpret_cast<uint32_t *>(smem + kEncGbitsOff)[tid] = gh[tid];
    for (int m = tid; m < 4 * 4 * 64; m += 64 * kEncWaves) {
        const int cb = m >> 8, s = (m >> 6) & 3, l = m & 63;
        const uint32_t byte = (gh[(16 * cb + (l & 15)) * 4 + s] >> (8 * (l >> 4))) & 0xffu;
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            w[k] = (((byte >> (2 * k)) & 1u) ? 0x3F80u : 0xBF80u) | ((((byte >> (2 * k + 1)) & 1u) ? 0x3F80u : 0xBF80u) << 16);
        reinterpret_cast<uint4 *>(smem + kEncGimgOff)[m] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    // sign flip as an xor on the raw 16-bit words: word j of chunk (s, g)
    // holds elements 32 s + 8 g + 2 j (low half) and + 1 (high half)
    for (int k = tid; k < 64 * 16; k += 64 * kEncWaves) {
        const int l = k >> 4, q = k & 15, sq = q >> 2, j = q & 3;
        uint32_t m = 0u;
        if (ROT && a.sign_flip) {
            const int e0 = 32 * sq + 8 * (l >> 4) + 2 * j;
            m = (a.sign_flip[e0] < 0 ? 0x8000u : 0u) | (a.sign_flip[e0 + 1] < 0 ? 0x80000000u : 0u);
        }
        reinterpret_cast<uint32_t *>(smem + kEncFlipOff)[k] = m;
    }
    __syncthreads();

    const unsigned char *tab = smem;
    const float *cent = reinterpret_cast<const float *>(smem + kEncCentOff);
    const uint32_t *gbits = reinterpret_cast<const uint32_t *>(smem + kEncGbitsOff);

    // row of lane n in the 16-row group at virtual row v (< v_end): v + n
    // (clamped) -> (b, t) -> memory row
    auto group_bt = [&](int64_t v, int64_t &bq, int64_t &t) {
        const int64_t b0 = v / a.T;                          // uniform
        t = (v - b0 * a.T) + (v + n < v_end ? n : (v_end - 1 - v));
        bq = b0;
        while (t >= a.T) { t -= a.T; ++bq; }                 // at most 16 / T + 1 steps
    };
    auto group_row = [&](int64_t v) {
        int64_t bq, t;
        group_bt(v, bq, t);
        return (bq * a.H + h) * a.T + t;
    };
    // output row of lane n's row: the memory row, or (paged) its pool row,
    // -1 where the page is outside the pool or the position past the table
    auto group_orow = [&](int64_t v, int64_t irow) -> int64_t {
        if constexpr (!PAGED) {
            return irow;
        } else {
            int64_t bq, t;
            group_bt(v, bq, t);
            const int64_t pos = (int64_t)a.positions[bq] + t;
            const int64_t pi = pos >> a.page_shift;
            const int32_t pg = (pos >= 0 && pi < a.max_pages) ? a.page_table[bq * a.max_pages + pi] : -1;
            if (pg < 0 || pg >= a.n_pages) return -1;
            return (((int64_t)pg * a.H + h) << a.page_shift) + (pos & ((1 << a.page_shift) - 1));
        }
    };
    auto load_group = [&](uint4 (&w)[4], int64_t row) {
        const uint4 *src = reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(xz) + row * 128);
#pragma unroll
        for (int s = 0; s < 4; ++s) w[s] = src[4 * s + g];
    };
    // One 16-row group: w4 holds lane (n, g)'s four 16-byte chunks of row
    // mrow (virtual row v0 + n).
    auto encode_group = [&](const uint4 (&w4)[4], const int64_t mrow, const int64_t v0) {
        const bool store = v0 + n < v_end && g == 0 && (!PAGED || mrow >= 0);
        // wave priority by phase: the projection MFMAs 2, the rotation 1,
        // the rest 0, so that of a SIMD's three waves the ones in those
        // phases issue first (issue order only: results do not depend on it)
        __builtin_amdgcn_s_setprio(1);

        // flip signs on the raw words (8 x 16-bit per chunk), widen
        float x[4][8];
        uint32_t nib[4];
        double ss = 0.0;
        float as = 0.0f;
        {
            const uint4 *fmk = reinterpret_cast<const uint4 *>(smem + kEncFlipOff) + lane * 4;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const uint4 f = ROT ? fmk[s] : make_uint4(0u, 0u, 0u, 0u);
                const uint32_t w[4] = {w4[s].x ^ f.x, w4[s].y ^ f.y, w4[s].z ^ f.z, w4[s].w ^ f.w};
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint32_t u = (i & 1) ? (w[i >> 1] >> 16) : (w[i >> 1] & 0xffffu);
                    x[s][i] = XDT == OMNI_BF16 ? __uint_as_float(u << 16) : f16_to_f32((uint16_t)u);
                }
            }
        }
        if (ROT) {
            // h = 1, 2, 4 inside each 8-element chunk
#pragma unroll
            for (int hh = 1; hh < 8; hh <<= 1)
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (!(i & hh)) {
                            const float u = x[s][i], l = x[s][i + hh];
                            x[s][i] = u + l;
                            x[s][i + hh] = u - l;
                        }
            // h = 8 (lanes l ^ 16), h = 16 (lanes l ^ 32)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 8; i += 2) xlane_pair_butterfly<16>(x[s][i], x[s][i + 1]);
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 8; i += 2) xlane_pair_butterfly<32>(x[s][i], x[s][i + 1]);
            // h = 32 (s ^ 1), h = 64 (s ^ 2)
#pragma unroll
            for (int hs = 1; hs < 4; hs <<= 1)
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    if (!(s & hs)) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            const float u = x[s][i], l = x[s + hs][i];
                            x[s][i] = u + l;
                            x[s + hs][i] = u - l;
                        }
                    }
        }
        __builtin_amdgcn_s_setprio(0);
        // value bits of each element ((scaled and) rounded to the input dtype)
        uint32_t vb[4][8];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
                if (ROT) {
                    const float p = x[s][i] * a.scale, q = x[s][i + 1] * a.scale;
                    uint32_t pk;
                    if (XDT == OMNI_BF16) {
                        typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
                        typedef float f2_t __attribute__((ext_vector_type(2)));
                        pk = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){p, q}, bf2_t));
                        x[s][i] = __uint_as_float(pk << 16);
                        x[s][i + 1] = __uint_as_float(pk & 0xffff0000u);
                    } else {
                        pk = cvt_pk_f16(p, q);
                        x[s][i] = f16_to_f32((uint16_t)(pk & 0xffffu));
                        x[s][i + 1] = f16_to_f32((uint16_t)(pk >> 16));
                    }
                    vb[s][i] = pk & 0xffffu;
                    vb[s][i + 1] = pk >> 16;
                } else if (XDT == OMNI_BF16) {
                    vb[s][i] = __float_as_uint(x[s][i]) >> 16;
                    vb[s][i + 1] = __float_as_uint(x[s][i + 1]) >> 16;
                } else {
                    vb[s][i] = f32_to_f16_rne(x[s][i]);          // exact: the value came from f16
                    vb[s][i + 1] = f32_to_f16_rne(x[s][i + 1]);
                }
            }
        // codes (all table reads issued together), then centroids
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < 8; ++i) vb[s][i] = tab[vb[s][i]];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            uint32_t wn = 0u;
#pragma unroll
            for (int i = 0; i < 8; i += 2)
                wn |= ((vb[s][i] & 0x0Fu) | (vb[s][i + 1] & 0xF0u)) << (4 * i);
            nib[s] = wn;
        }
        if (PAGED && zb == 1) {
            // V in the paged pool: codes only (the attention reads no V
            // residual), so no residual, norm or projection
            if (v0 + n < v_end && mrow >= 0) {
                uint32_t *np = reinterpret_cast<uint32_t *>(nibz + mrow * 64);
#pragma unroll
                for (int s = 0; s < 4; ++s) np[4 * s + g] = nib[s];
            }
            return;
        }
        float cv[4][8];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < 8; ++i) cv[s][i] = cent[vb[s][i]];
        // residuals, norm (fp64 sum of the exact squares) and |e| partial
        // sums, one chain per chunk s (four independent dependency chains)
        double ssp[4] = {0.0, 0.0, 0.0, 0.0};
        float asp[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const float e = x[s][i] - cv[s][i];
                x[s][i] = e;
                const double ed = (double)e;
                ssp[s] = __builtin_fma(ed, ed, ssp[s]);
                asp[s] += fabsf(e);
            }
        ss = (ssp[0] + ssp[1]) + (ssp[2] + ssp[3]);
        as = (asp[0] + asp[1]) + (asp[2] + asp[3]);
        ss = xlane_sum_f64<16>(ss);
        ss = xlane_sum_f64<32>(ss);
        as = xlane_sum_f32(as);

        // projections: P^T = G . E^T on MFMA with each residual as two
        // round-to-nearest bf16 parts, e = h + m + l: h = bf16(e), m =
        // bf16(e - h) (e - h is exact), |l| <= 2^-16 |e|.  G is exactly +-1,
        // so the products are exact and the MFMA sum of G (h + m) is within
        // 1024 * 2^-24 * sum(|h| + |m|) <= 1032.1 * 2^-24 * sum|e| of its exact
        // value (fp32 accumulation of 256 terms in any order, rounding to
        // nearest or toward zero); sum|l| adds 256 * 2^-24 * sum|e|, and the
        // fp32 sum `as` is within a relative 127 * 2^-24 of sum|e|:
        // 1312 * 2^-24 * as bounds the total.  Rows with sum|e| >= 2^127
        // (where a part could round to infinity) take the exact path below.
        __builtin_amdgcn_s_setprio(2);
        float4_t acc[4];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) acc[cb] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            uint32_t ph[4], pm[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
                typedef float f2_t __attribute__((ext_vector_type(2)));
                const float e0 = x[s][2 * j], e1 = x[s][2 * j + 1];
                const uint32_t hp = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){e0, e1}, bf2_t));
                const float r0 = e0 - __uint_as_float(hp << 16);
                const float r1 = e1 - __uint_as_float(hp & 0xffff0000u);
                ph[j] = hp;
                pm[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){r0, r1}, bf2_t));
            }
            const bf16x8_t bh = __builtin_bit_cast(bf16x8_t, make_uint4(ph[0], ph[1], ph[2], ph[3]));
            const bf16x8_t bm = __builtin_bit_cast(bf16x8_t, make_uint4(pm[0], pm[1], pm[2], pm[3]));
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) {
                const uint4 gv = reinterpret_cast<const uint4 *>(smem + kEncGimgOff)[(cb * 4 + s) * 64 + lane];
                const bf16x8_t ga = __builtin_bit_cast(bf16x8_t, gv);
                acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga, bh, acc[cb], 0, 0, 0);
                acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga, bm, acc[cb], 0, 0, 0);
            }
        }

        __builtin_amdgcn_s_setprio(0);
        // signs: lane (n, g) holds P[n][16 cb + 4 g + i]; cb's four bits go
        // to bits 16 (cb & 1) + 4 g .. + 3 of word cb / 2
        const bool finite_row = as < 0x1p127f;                 // false for inf / NaN
        const float bound = as * 7.82012939453125e-05f + 7.888609052210118e-31f;   // 1312 * 2^-24, 2^-100
        uint32_t slo = 0u, shi = 0u;
        float amin = INFINITY;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const uint32_t nb = (acc[cb][0] >= 0.0f ? 1u : 0u) | (acc[cb][1] >= 0.0f ? 2u : 0u) |
                                (acc[cb][2] >= 0.0f ? 4u : 0u) | (acc[cb][3] >= 0.0f ? 8u : 0u);
            const uint32_t w = nb << (16 * (cb & 1) + 4 * g);
            if (cb < 2) slo |= w; else shi |= w;
            amin = fminf(amin, fminf(fminf(fabsf(acc[cb][0]), fabsf(acc[cb][1])), fminf(fabsf(acc[cb][2]), fabsf(acc[cb][3]))));
        }
        // rare: uncertain signs of finite rows (recomputed exactly: the 4
        // lanes of the row each sum their 32 elements, then combine) and
        // rows whose residual is not finite (or whose |e| sum reaches 2^127)
        const bool nf = !finite_row && v0 + n < v_end;
        if (__builtin_amdgcn_ballot_w64((finite_row && !(amin > bound)) || nf)) {
            uint32_t unc = 0u;
#pragma unroll
            for (int cb = 0; cb < 4; ++cb)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (finite_row && !(fabsf(acc[cb][i]) > bound)) unc |= 1u << (4 * cb + i);
            // one residual row at a time goes through this wave's LDS row
            float *st = reinterpret_cast<float *>(smem + kEncStageOff) + wave * 128;
            int staged = -1;
            auto stage = [&](int r) {
                if (r == staged) return;
                if (n == r) {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
#pragma unroll
                        for (int i = 0; i < 8; ++i) st[32 * q + 8 * g + i] = x[q][i];
                }
                staged = r;
            };
            uint64_t pend = __builtin_amdgcn_ballot_w64(unc != 0u);
            while (pend) {
                const int L = __builtin_ctzll(pend);
                const uint32_t uL = __builtin_amdgcn_readlane(unc, L);
                const int item = __builtin_ctz(uL);
                const int o = 16 * (item >> 2) + 4 * (L >> 4) + (item & 3);
                stage(L & 15);
                uint32_t fl;
                const double tot = wave_row_dot(st, gbits + o * 4, lane, fl);
                if (lane == L) {
                    unc &= ~(1u << item);
                    const uint32_t bit = tot >= 0.0 ? 1u : 0u;
                    const int pos = 16 * ((item >> 2) & 1) + 4 * g + (item & 3);
                    if ((item >> 2) < 2) slo = (slo & ~(1u << pos)) | (bit << pos);
                    else shi = (shi & ~(1u << pos)) | (bit << pos);
                }
                pend = __builtin_amdgcn_ballot_w64(unc != 0u);
            }
            uint64_t nfm = __builtin_amdgcn_ballot_w64(nf && g == 0);
            while (nfm) {
                const int r = __builtin_ctzll(nfm);
                nfm &= nfm - 1;
                stage(r);
#pragma unroll 1
                for (int o = 0; o < 64; ++o) {
                    // order-free sign of the fp32 sum: a NaN term or both
                    // infinities -> NaN -> 0; one infinity -> its sign; all
                    // finite (only the |e| sum overflowed) -> exact fp64 sign
                    uint32_t fl;
                    const double tot = wave_row_dot(st, gbits + o * 4, lane, fl);
                    uint32_t bit;
                    if ((fl & 1u) || (fl & 6u) == 6u) bit = 0u;
                    else if (fl & 2u) bit = 1u;
                    else if (fl & 4u) bit = 0u;
                    else bit = tot >= 0.0 ? 1u : 0u;
                    if (n == r && g == ((o & 15) >> 2)) {
                        const int pos = 16 * ((o >> 4) & 1) + 4 * g + (o & 3);
                        if ((o >> 4) < 2) slo = (slo & ~(1u << pos)) | (bit << pos);
                        else shi = (shi & ~(1u << pos)) | (bit << pos);
                    }
                }
            }
        }
        slo |= xlane_u32<16>(slo);
        slo |= xlane_u32<32>(slo);
        shi |= xlane_u32<16>(shi);
        shi |= xlane_u32<32>(shi);

        // stores: nibble dword s of lane (n, g) is bytes 16 s + 4 g .. + 3
        if (v0 + n < v_end && (!PAGED || mrow >= 0)) {
            uint32_t *np = reinterpret_cast<uint32_t *>(nibz + mrow * 64);
#pragma unroll
            for (int s = 0; s < 4; ++s) np[4 * s + g] = nib[s];
        }
        if (store) {
            reinterpret_cast<uint2 *>(qjlz + mrow * 8)[0] = make_uint2(slo, shi);
            nrmz[mrow] = ss > 3.4028234663852886e38 ? INFINITY : (float)sqrt(ss);
        }
    };

    // Groups v0, v0 + 16 nw, ... through a two-slot ring: the next group's
    // rows are requested before the current one is encoded (past the last
    // group, the current group's rows again, so every load is unconditional
    // and the compiler waits only for the slot it consumes).
    constexpr int64_t kStep = 16 * kEncWaves;
    int64_t v0 = v_begin + 16 * wave;
    if (v0 >= v_end) return;                                 // no barrier follows
    uint4 ring0[4], ring1[4];
    int64_t row0 = group_row(v0), row1;
    load_group(ring0, row0);
    for (;;) {
        row1 = v0 + kStep < v_end ? group_row(v0 + kStep) : row0;
        load_group(ring1, row1);
        encode_group(ring0, group_orow(v0, row0), v0);
        v0 += kStep;
        if (v0 >= v_end) break;
        row0 = v0 + kStep < v_end ? group_row(v0 + kStep) : row1;
        load_group(ring0, row0);
        encode_group(ring1, group_orow(v0, row1), v0);
        v0 += kStep;
        if (v0 >= v_end) break;
    }
}

// ── wave encoder without a value table: f32 input, D = 32 ───────────────
//
// The contract and the matrix-core projections of encode128_kernel for the
// inputs whose codes no table of all values can give (f32) or that are too
// short for one (D = 32).  Lane (n, g) holds 32 values as x[s][i]: elements
// 32 s + 8 g + i of row n (D = 128, 16 rows per wave iteration), or elements
// 8 g + i of row 16 s + n (D = 32, 64 rows).
//   * Codes: the values from c_0 - r to c_15 + 7 r (r = c_15 - c_0) fall into
//     1023 equal cells, and a byte table in LDS, built by each block, names
//     the lower of the two adjacent codes that a cell's values can take (the
//     codes at its edges, one percent of a cell further out, differ by at most
//     one, and codes ascend with the value).  Both fp32 distances then decide,
//     first index on ties.  Cells with more boundaries, values beyond the last
//     cell, and codebooks that do not ascend by more than a rounding error of
//     the distances compared point at a NaN centroid: such a group of rows is
//     coded again over all 16 centroids.
//   * Bound by VALU issue, as encode128_kernel.  K and V of 16 x 4096 tokens,
//     8 heads, with a lane per row and 16 distances per value before: f32 at
//     D = 128 3851 -> 176 us (3.5 TB/s), bf16 at D = 32 595 -> 86 us; one
//     token of one sequence 385 -> 10 us.  On 16-bit rows at D = 128 the value
//     table is the better of the two where it is built already (146 against
//     197 us; equal below 1000 rows per head).

constexpr int kEgWaves = 4;
constexpr int kEgCells = 1024;                        // the last one: values past the grid
constexpr float kEgBelow = 1.0f, kEgAbove = 7.0f;     // the grid's reach past the centroids, in r

template <int D>
struct EgLds {
    static constexpr int S = D == 128 ? 4 : 1;        // chunks of a row
    static constexpr int CB = D == 128 ? 4 : 1;       // blocks of 16 projections
    uint8_t cell[kEgCells];                           // 4 * lower code (64: none)
    float cent[20];                                   // 16..19: NaN
    uint4 gimg[CB * S * 64];                          // [cb][s][lane]: 8 bf16 +-1 of G
    uint32_t gbits[(D / 2) * (D / 32)];
    uint32_t flip[D];                                 // sign-bit xor of each element
    float stage[kEgWaves][D];                         // one residual row (rare paths)
};

// sum_j s_j e_j over one staged residual row of D floats (wave_row_dot for
// any D).
template <int D>
__device__ __forceinline__ double eg_row_dot(const float *st, const uint32_t *grow, int lane, uint32_t &fl) {
    if constexpr (D == 128) {
        return wave_row_dot(st, grow, lane, fl);
    } else {
        float f = 0.0f;
        if (lane < 32) f = ((grow[0] >> lane) & 1u) ? st[lane] : -st[lane];
        const uint32_t cls = (f != f) ? 1u : (f == INFINITY ? 2u : (f == -INFINITY ? 4u : 0u));
        fl = (__builtin_amdgcn_ballot_w64((cls & 1u) != 0u) ? 1u : 0u) | (__builtin_amdgcn_ballot_w64((cls & 2u) != 0u) ? 2u : 0u) |
             (__builtin_amdgcn_ballot_w64((cls & 4u) != 0u) ? 4u : 0u);
        double s = (double)f, c = 0.0;
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) {
            const double so = __shfl_xor(s, m), co = __shfl_xor(c, m);
            const double t = s + so;
            const double bp = t - s;
            const double err = (s - (t - bp)) + (so - bp);
            s = t;
            c = (c + co) + err;
        }
        return s + c;
    }
}

// First-index argmin of the fp32 distances (no NaN).
__device__ __forceinline__ int eg_code(float x, const float (&cb)[16]) {
    float best = fabsf(x - cb[0]);
    int code = 0;
#pragma unroll
    for (int k = 1; k < 16; ++k) {
        const float d = fabsf(x - cb[k]);
        code = d < best ? k : code;
        best = fminf(best, d);
    }
    return code;
}

template <int XDT, int D, bool ROT>
__global__ __launch_bounds__(64 * kEgWaves, D == 128 ? 3 : 2) void encode_grid_kernel(EncArgs a) {
    using L = EgLds<D>;
    constexpr int S = L::S, CB = L::CB;
    constexpr int kGroup = D == 128 ? 16 : 64;        // rows per wave iteration
    constexpr int QD = D / 2, W = D / 32;
    __shared__ __attribute__((aligned(16))) L sm;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int h = blockIdx.y, zb = blockIdx.z;
    const int64_t rpb = a.rows_per_block[zb];
    const int64_t v_begin = (int64_t)blockIdx.x * rpb;
    if (v_begin >= a.nrows_head) return;               // block-uniform, before any barrier
    const int64_t v_end = v_begin + rpb < a.nrows_head ? v_begin + rpb : a.nrows_head;
    const void *const xz = a.x[zb];
    uint8_t *const nibz = a.nibbles[zb];
    uint8_t *const qjlz = a.qjl[zb];
    float *const nrmz = a.norms[zb];

    // ── prologue: centroids, cells, G images, sign flips ─────────────
    const float *cbp = a.codebooks + (a.per_head ? h * 16 : 0);
    const uint32_t *gh = a.g_bits + (int64_t)h * QD * W;
    if (tid < 20) sm.cent[tid] = tid < 16 ? cbp[tid] : __builtin_nanf("");
    for (int k = tid; k < QD * W; k += 64 * kEgWaves) sm.gbits[k] = gh[k];
    for (int d = tid; d < D; d += 64 * kEgWaves) sm.flip[d] = (ROT && a.sign_flip && a.sign_flip[d] < 0) ? 0x80000000u : 0u;
    for (int m = tid; m < CB * S * 64; m += 64 * kEgWaves) {
        const int cb = m / (S * 64), s = (m / 64) % S, l = m & 63;
        const uint32_t byte = (gh[(16 * cb + (l & 15)) * W + s] >> (8 * (l >> 4))) & 0xffu;
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            w[k] = (((byte >> (2 * k)) & 1u) ? 0x3F80u : 0xBF80u) | ((((byte >> (2 * k + 1)) & 1u) ? 0x3F80u : 0xBF80u) << 16);
        sm.gimg[m] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    __syncthreads();
    const float c0 = sm.cent[0], r = sm.cent[15] - c0;
    const float g_lo = c0 - kEgBelow * r, g_hi = sm.cent[15] + kEgAbove * r;
    const float inv = (float)(kEgCells - 1) / (g_hi - g_lo), off = -g_lo * inv;
    float cb[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) cb[k] = sm.cent[k];
    // ascending, and no distance to a lower centroid can round to a tie with
    // the nearest one anywhere on the grid: gap >= 2 ulp of it (lane k: the
    // gap of centroids k and k + 1)
    const float lo = sm.cent[n < 15 ? n : 14], hi = sm.cent[n < 15 ? n + 1 : 15];
    float next = g_hi;
#pragma unroll
    for (int j = 15; j > 0; --j) next = cb[j] > hi ? cb[j] : next;
    const bool good = lo == hi || (lo < hi && hi - lo >= (next - lo) * 2.384185791015625e-7f);
    const bool grid_ok = __builtin_amdgcn_ballot_w64(!good) == 0ull && r > 0.0f && inv > 1e-30f && inv < 1e30f &&
                         fabsf(g_lo) < 1e30f && fabsf(g_hi) < 1e30f;
    const double width = 1.0 / (double)inv;
    for (int c = tid; c < kEgCells; c += 64 * kEgWaves) {
        int code = 16;
        if (grid_ok && c < kEgCells - 1) {
            const float x0 = (float)(((double)c - 0.01 - (double)off) * width);
            const float x1 = (float)(((double)c + 1.01 - (double)off) * width);
            const int k0 = c == 0 ? 0 : eg_code(x0, cb), k1 = eg_code(x1, cb);
            if (k1 >= k0 && k1 - k0 <= 1) code = k0 < 14 ? k0 : 14;
        }
        sm.cell[c] = (uint8_t)(4 * code);
    }
    __syncthreads();
    const char *cent_b = reinterpret_cast<const char *>(sm.cent);

    // (vb, vt): batch entry and token of the first row of the wave's group;
    // groups of a wave lie kEgWaves * kGroup rows apart = (step_b, step_t)
    int64_t vcur = v_begin + kGroup * wave;
    if (vcur >= v_end) return;                         // no barrier follows
    int64_t vb = vcur / a.T, vt = vcur - vb * a.T;
    constexpr int kSets = D == 128 ? 1 : 4;            // 16-row sets of a group
    auto rows_of = [&](int64_t (&row)[kSets], int64_t v, int64_t b0, int64_t t0) {
#pragma unroll
        for (int q = 0; q < kSets; ++q) {
            const int64_t left = v_end - 1 - v;
            int64_t b = b0, t = t0 + (16 * q + n < left ? (int64_t)(16 * q + n) : left);
            while (t >= a.T) {
                t -= a.T;
                ++b;
            }
            row[q] = (b * a.H + h) * a.T + t;
        }
    };
    constexpr int kRaw = XDT == OMNI_F32 ? 2 : 1;      // 16-byte loads of a chunk
    auto load = [&](uint4 (&raw)[4][kRaw], const int64_t (&row)[kSets]) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int64_t e = row[D == 128 ? 0 : s] * D + (D == 128 ? 32 * s : 0) + 8 * g;
            if constexpr (XDT == OMNI_F32) {
                const uint4 *p = reinterpret_cast<const uint4 *>(reinterpret_cast<const float *>(xz) + e);
                raw[s][0] = p[0];
                raw[s][1] = p[1];
            } else {
                raw[s][0] = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(xz) + e);
            }
        }
    };
    auto encode = [&](float (&x)[4][8], const int64_t (&row)[kSets], const int64_t v0) {
        if (ROT) {
#pragma unroll
            for (int hh = 1; hh < 8; hh <<= 1)
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (!(i & hh)) {
                            const float u = x[s][i], l = x[s][i + hh];
                            x[s][i] = u + l;
                            x[s][i + hh] = u - l;
                        }
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 8; i += 2) xlane_pair_butterfly<16>(x[s][i], x[s][i + 1]);
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 8; i += 2) xlane_pair_butterfly<32>(x[s][i], x[s][i + 1]);
            if constexpr (D == 128) {
#pragma unroll
                for (int hs = 1; hs < 4; hs <<= 1)
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        if (!(s & hs))
#pragma unroll
                            for (int i = 0; i < 8; ++i) {
                                const float u = x[s][i], l = x[s + hs][i];
                                x[s][i] = u + l;
                                x[s + hs][i] = u - l;
                            }
            }
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    float p = x[s][i] * a.scale;
                    // the product is rounded to fp32 before it is rounded to
                    // f16 (v_fma_mixlo_f16 would round once)
                    if (XDT == OMNI_F16) asm volatile("" : "+v"(p));
                    x[s][i] = round_to_dtype(p, XDT);
                }
        }
        // codes and residuals: the cell's two candidates
        float e[4][8];
        uint32_t nib[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            uint32_t cell[8], wn = 0u;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float t = __builtin_amdgcn_fmed3f(__builtin_fmaf(x[s][i], inv, off), 0.0f, (float)(kEgCells - 1));
                cell[i] = sm.cell[(uint32_t)t];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float *c = reinterpret_cast<const float *>(cent_b + cell[i]);
                const float e0 = x[s][i] - c[0], e1 = x[s][i] - c[1];
                const bool up = fabsf(e1) < fabsf(e0);
                e[s][i] = up ? e1 : e0;
                wn += ((cell[i] >> 2) + (up ? 1u : 0u)) << (4 * i);
            }
            nib[s] = wn;
        }
        // per chunk: sum |e| over the row's four lanes (and chunks, D = 128);
        // not finite where a value's cell names no code, or by itself
        float as[kSets];
        auto abs_sums = [&]() {
            float p[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                p[s] = 0.0f;
#pragma unroll
                for (int i = 0; i < 8; ++i) p[s] += fabsf(e[s][i]);
            }
            if constexpr (D == 128) {
                as[0] = xlane_sum_f32((p[0] + p[1]) + (p[2] + p[3]));
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s) as[s] = xlane_sum_f32(p[s]);
            }
        };
        abs_sums();
        bool odd = false;
#pragma unroll
        for (int q = 0; q < kSets; ++q) odd = odd || !(as[q] < 0x1p127f);
        if (__builtin_amdgcn_ballot_w64(odd)) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                nib[s] = 0u;
#pragma unroll
                for (int i = 0; i < 8; ++i) e[s][i] = x[s][i] - sm.cent[0];
            }
#pragma unroll 1
            for (int k = 1; k < 16; ++k) {
                const float c = sm.cent[k];
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const float d = x[s][i] - c;
                        const bool take = fabsf(d) < fabsf(e[s][i]) || (d != d && e[s][i] == e[s][i]);
                        e[s][i] = take ? d : e[s][i];
                        nib[s] = take ? ((nib[s] & ~(15u << (4 * i))) | ((uint32_t)k << (4 * i))) : nib[s];
                    }
            }
            abs_sums();
        }
        // norms: fp64 sums of the exact squares
        double ss[kSets];
        {
            double p[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) p[s] = 0.0;
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const double ed = (double)e[s][i];
                    p[s] = __builtin_fma(ed, ed, p[s]);
                }
            if constexpr (D == 128) {
                ss[0] = xlane_sum_f64<32>(xlane_sum_f64<16>((p[0] + p[1]) + (p[2] + p[3])));
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s) ss[s] = xlane_sum_f64<32>(xlane_sum_f64<16>(p[s]));
            }
        }
        // projections as in encode128_kernel: two bf16 parts of each residual,
        // G exact; D = 128: acc[cb] over the chunks, D = 32: acc[s] per set
        float4_t acc[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            uint32_t ph[4], pm[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
                typedef float f2_t __attribute__((ext_vector_type(2)));
                const float e0 = e[s][2 * j], e1 = e[s][2 * j + 1];
                const uint32_t hp = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){e0, e1}, bf2_t));
                const float r0 = e0 - __uint_as_float(hp << 16);
                const float r1 = e1 - __uint_as_float(hp & 0xffff0000u);
                ph[j] = hp;
                pm[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){r0, r1}, bf2_t));
            }
            const bf16x8_t bh = __builtin_bit_cast(bf16x8_t, make_uint4(ph[0], ph[1], ph[2], ph[3]));
            const bf16x8_t bm = __builtin_bit_cast(bf16x8_t, make_uint4(pm[0], pm[1], pm[2], pm[3]));
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const bf16x8_t ga = __builtin_bit_cast(bf16x8_t, sm.gimg[(cb * S + (D == 128 ? s : 0)) * 64 + lane]);
                float4_t &t = acc[D == 128 ? cb : s];
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga, bh, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga, bm, t, 0, 0, 0);
            }
        }
        // signs: bits q of `sg` is acc[q / 4][q % 4] >= 0 (lane (n, g): D = 128
        // projection 16 (q / 4) + 4 g + q % 4 of row n, D = 32 projection
        // 4 g + q % 4 of row 16 (q / 4) + n)
        uint32_t sg = 0u, unc = 0u, nf = 0u;
        float amin[kSets];
#pragma unroll
        for (int q = 0; q < kSets; ++q) amin[q] = INFINITY;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sg |= acc[q][i] >= 0.0f ? 1u << (4 * q + i) : 0u;
                float &m = amin[D == 128 ? 0 : q];
                m = fminf(m, fabsf(acc[q][i]));
            }
        // Uncertain signs of finite rows and rows whose residual is not finite
        // (or whose |e| sum reaches 2^127): encode128_kernel's bound, which was
        // derived for 128 elements and holds for 32
        bool rare = false;
        float bound[kSets];
#pragma unroll
        for (int q = 0; q < kSets; ++q) {
            bound[q] = as[q] * 7.82012939453125e-05f + 7.888609052210118e-31f;
            const bool fin = as[q] < 0x1p127f, in = v0 + 16 * q + n < v_end;
            nf |= (!fin && in) ? 1u << q : 0u;
            rare = rare || (fin && !(amin[q] > bound[q])) || (!fin && in);
        }
        if (__builtin_amdgcn_ballot_w64(rare)) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int z = D == 128 ? 0 : q;
                    if (as[z] < 0x1p127f && !(fabsf(acc[q][i]) > bound[z])) unc |= 1u << (4 * q + i);
                }
            float *st = sm.stage[wave];
            int staged = -1;
            auto stage = [&](int rr) {                 // row rr of the group
                if (rr == staged) return;
                if (n == (rr & 15)) {
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        if (D == 128 || s == (rr >> 4))
#pragma unroll
                            for (int i = 0; i < 8; ++i) st[(D == 128 ? 32 * s : 0) + 8 * g + i] = e[s][i];
                }
                staged = rr;
            };
            uint64_t pend = __builtin_amdgcn_ballot_w64(unc != 0u);
            while (pend) {
                const int Lq = __builtin_ctzll(pend);
                const uint32_t uL = __builtin_amdgcn_readlane(unc, Lq);
                const int item = __builtin_ctz(uL);
                const int o = (D == 128 ? 16 * (item >> 2) : 0) + 4 * (Lq >> 4) + (item & 3);
                stage((Lq & 15) + (D == 128 ? 0 : 16 * (item >> 2)));
                uint32_t fl;
                const double tot = eg_row_dot<D>(st, sm.gbits + o * W, lane, fl);
                if (lane == Lq) {
                    unc &= ~(1u << item);
                    sg = (sg & ~(1u << item)) | ((tot >= 0.0 ? 1u : 0u) << item);
                }
                pend = __builtin_amdgcn_ballot_w64(unc != 0u);
            }
#pragma unroll 1
            for (int q = 0; q < kSets; ++q) {
                uint64_t nfm = __builtin_amdgcn_ballot_w64(((nf >> q) & 1u) && g == 0);
                while (nfm) {
                    const int rr = __builtin_ctzll(nfm);
                    nfm &= nfm - 1;
                    stage(16 * q + rr);
#pragma unroll 1
                    for (int o = 0; o < QD; ++o) {
                        // order-free sign of the fp32 sum (see encode128_kernel)
                        uint32_t fl;
                        const double tot = eg_row_dot<D>(st, sm.gbits + o * W, lane, fl);
                        uint32_t bit;
                        if ((fl & 1u) || (fl & 6u) == 6u) bit = 0u;
                        else if (fl & 2u) bit = 1u;
                        else if (fl & 4u) bit = 0u;
                        else bit = tot >= 0.0 ? 1u : 0u;
                        const int item = (D == 128 ? 4 * (o >> 4) : 4 * q) + (o & 3);
                        if (n == rr && g == ((o & 15) >> 2)) sg = (sg & ~(1u << item)) | (bit << item);
                    }
                }
            }
        }
        // stores
        auto norm = [](double t) { return t > 3.4028234663852886e38 ? INFINITY : (float)sqrt(t); };
        if constexpr (D == 128) {
            uint32_t slo = ((sg & 15u) << (4 * g)) | (((sg >> 4) & 15u) << (16 + 4 * g));
            uint32_t shi = (((sg >> 8) & 15u) << (4 * g)) | ((sg >> 12) << (16 + 4 * g));
            slo |= xlane_u32<16>(slo);
            slo |= xlane_u32<32>(slo);
            shi |= xlane_u32<16>(shi);
            shi |= xlane_u32<32>(shi);
            if (v0 + n < v_end) {
                uint32_t *np = reinterpret_cast<uint32_t *>(nibz + row[0] * 64);
#pragma unroll
                for (int s = 0; s < 4; ++s) np[4 * s + g] = nib[s];
                if (g == 0) {
                    reinterpret_cast<uint2 *>(qjlz + row[0] * 8)[0] = make_uint2(slo, shi);
                    nrmz[row[0]] = norm(ss[0]);
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                uint32_t sw = ((sg >> (4 * q)) & 15u) << (4 * g);
                sw |= xlane_u32<16>(sw);
                sw |= xlane_u32<32>(sw);
                if (v0 + 16 * q + n < v_end) {
                    reinterpret_cast<uint32_t *>(nibz + row[q] * 16)[g] = nib[q];
                    if (g == 0) {
                        reinterpret_cast<uint16_t *>(qjlz + row[q] * 2)[0] = (uint16_t)sw;
                        nrmz[row[q]] = norm(ss[q]);
                    }
                }
            }
        }
    };

    // The next group's rows are requested as soon as the current ones are
    // widened (past the last group: the current rows again).
    uint4 raw[4][kRaw];
    int64_t row[kSets];
    rows_of(row, vcur, vb, vt);
    load(raw, row);
    for (;;) {
        float x[4][8];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const uint4 *fl = reinterpret_cast<const uint4 *>(sm.flip + (D == 128 ? 32 * s : 0) + 8 * g);
            const uint4 f0 = ROT ? fl[0] : make_uint4(0u, 0u, 0u, 0u), f1 = ROT ? fl[1] : f0;
            const uint32_t f[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
            if constexpr (XDT == OMNI_F32) {
                const uint32_t w[8] = {raw[s][0].x, raw[s][0].y, raw[s][0].z, raw[s][0].w,
                                       raw[s][1].x, raw[s][1].y, raw[s][1].z, raw[s][1].w};
#pragma unroll
                for (int i = 0; i < 8; ++i) x[s][i] = __uint_as_float(w[i] ^ f[i]);
            } else {
                const uint32_t w[4] = {raw[s][0].x, raw[s][0].y, raw[s][0].z, raw[s][0].w};
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint32_t u = (i & 1) ? (w[i >> 1] >> 16) : (w[i >> 1] & 0xffffu);
                    const float v = XDT == OMNI_BF16 ? __uint_as_float(u << 16) : f16_to_f32((uint16_t)u);
                    x[s][i] = __uint_as_float(__float_as_uint(v) ^ f[i]);
                }
            }
        }
        const int64_t v0 = vcur;
        int64_t cur[kSets];
#pragma unroll
        for (int q = 0; q < kSets; ++q) cur[q] = row[q];
        vcur += kEgWaves * kGroup;
        const bool more = vcur < v_end;
        if (more) {
            vb += a.step_b;
            vt += a.step_t;
            if (vt >= a.T) {
                vt -= a.T;
                ++vb;
            }
            rows_of(row, vcur, vb, vt);
        }
        load(raw, row);
        encode(x, cur, v0);
        if (!more) break;
    }
}

// ── omni_dequantize ─────────────────────────────────────────────────────
//
// k_hat_d = fl(cb[code_d] + fl(s_d * fl(norm * c))), c = fp32(sqrt(2/pi)/D),
// s_d = sum_i b+-_i G_h[i][d] = QD - 2 popcount(b ^ Gcol_d)  (an exact integer).

//
// Write-bound: a lane takes four consecutive elements of a row (D / 4 lanes
// per row, one 16-byte store), and keeps the G columns of those elements in
// registers over the block's run of rows of one head.  A lane per row before,
// with byte loads and 4-byte stores 512 bytes apart: 131,136 rows of 128 with
// QJL 105 -> 16 us (4.8 TB/s).
constexpr int kDqThreads = 256;

template <int D, bool QJL>
__global__ __launch_bounds__(kDqThreads) void dequant_kernel(
    const uint8_t *nibbles, const uint8_t *qjl, const float *norms, const float *codebooks,
    int per_head, const uint32_t *g_bits, int64_t T, int H, int64_t rows_head, int rows_block, uint64_t t_magic,
    float *out, float c_alpha) {
    constexpr int QD = D / 2, W = D / 32;
    constexpr int kLanes = D / 4;                      // lanes per row
    constexpr int kRows = kDqThreads / kLanes;         // rows per pass of the block
    constexpr int kU = 4;                              // passes with their loads in flight together
    __shared__ uint64_t gcol[D];
    __shared__ float cb[16];
    const int tid = threadIdx.x, lane = tid & 63;
    const int h = blockIdx.y;
    if (tid < 16) cb[tid] = codebooks[(per_head ? h * 16 : 0) + tid];
    if constexpr (QJL) {
        // columns of G_h as QD-bit masks: a wave ballots one bit of its QD rows
        const uint32_t *gh = g_bits + (int64_t)h * QD * W;
        for (int w = tid >> 6; w < W; w += kDqThreads / 64) {
            const uint32_t word = lane < QD ? gh[lane * W + w] : 0u;
            for (int j = 0; j < 32; ++j) {
                const uint64_t m = __builtin_amdgcn_ballot_w64((word >> j) & 1u);
                if (lane == 0) gcol[32 * w + j] = m;
            }
        }
    }
    __syncthreads();
    const int d4 = tid % kLanes, rl = tid / kLanes;
    uint64_t gc[4] = {0, 0, 0, 0};
    if constexpr (QJL) {
#pragma unroll
        for (int k = 0; k < 4; ++k) gc[k] = gcol[4 * d4 + k];
    }
    const int64_t v0 = (int64_t)blockIdx.x * rows_block;
    const int64_t b0 = v0 / T;
    const int64_t t0 = v0 - b0 * T;
    const int left = (int)(rows_head - v0 < rows_block ? rows_head - v0 : rows_block);
    for (int r0 = 0; r0 < left; r0 += kU * kRows) {
        int64_t row[kU];
        uint32_t nb[kU];
        uint2 sb[kU];
        float nr[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int r = r0 + u * kRows + rl, rr = r < left ? r : left - 1;
            // (t0 + rr) / T: exact below 2^16; longer sequences wrap once at most
            const int64_t t = t0 + rr;
            const int64_t wrap = t_magic ? (int64_t)(((uint64_t)(uint32_t)t * t_magic) >> 32) : (t >= T ? 1 : 0);
            row[u] = ((b0 + wrap) * H + h) * T + (t - wrap * T);
            nb[u] = reinterpret_cast<const uint16_t *>(nibbles + row[u] * (D / 2))[d4];
            if constexpr (QJL) {
                if constexpr (D == 128) sb[u] = reinterpret_cast<const uint2 *>(qjl + row[u] * (D / 16))[0];
                else sb[u] = make_uint2(reinterpret_cast<const uint16_t *>(qjl + row[u] * (D / 16))[0], 0u);
                nr[u] = norms[row[u]];
            }
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = cb[(nb[u] >> (4 * k)) & 15u];
            if constexpr (QJL) {
                const float sc = __fmul_rn(nr[u], c_alpha);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int p = __popc(sb[u].x ^ (uint32_t)gc[k]) + (D == 128 ? __popc(sb[u].y ^ (uint32_t)(gc[k] >> 32)) : 0);
                    v[k] = __fadd_rn(v[k], __fmul_rn((float)(QD - 2 * p), sc));
                }
            }
            if (r0 + u * kRows + rl < left)
                reinterpret_cast<float4 *>(out + row[u] * D)[d4] = make_float4(v[0], v[1], v[2], v[3]);
        }
    }
}

}  // namespace omni

using namespace omni;

extern "C" int omni_wht_rotate(const void *x, int dtype, int64_t rows, int head_dim,
                               const int8_t *sign_flip, void *out, void *stream) {
    OMNI_CHECK_ARG(dtype_ok(dtype), "omni_wht_rotate: bad dtype %d", dtype);
    OMNI_CHECK_ARG(head_dim_ok(head_dim), "WHT rotation requires last dim = 128 (or 32), got %d", head_dim);
    OMNI_CHECK_ARG(rows >= 0, "omni_wht_rotate: rows < 0");
    OMNI_CHECK_ARG(rows == 0 || (x && out), "omni_wht_rotate: NULL pointer");
    if (rows == 0) return OMNI_OK;
    const int per_block = 4 * (head_dim == 128 ? 16 : 64);
    // (two dimensions: a launch of 2^32 threads or more in one is cut off)
    const int64_t blocks = (rows + per_block - 1) / per_block, gx = blocks < kWhtGridX ? blocks : kWhtGridX;
    const dim3 grid((unsigned)gx, (unsigned)((blocks + gx - 1) / gx)), block(256);
    const float s = inv_sqrt_dim_f32(head_dim);
    hipStream_t st = as_stream(stream);
    if (head_dim == 128) {
        if (dtype == OMNI_F32) hipLaunchKernelGGL((wht_kernel<OMNI_F32, 128>), grid, block, 0, st, x, rows, sign_flip, out, s);
        else if (dtype == OMNI_BF16) hipLaunchKernelGGL((wht_kernel<OMNI_BF16, 128>), grid, block, 0, st, x, rows, sign_flip, out, s);
        else hipLaunchKernelGGL((wht_kernel<OMNI_F16, 128>), grid, block, 0, st, x, rows, sign_flip, out, s);
    } else {
        if (dtype == OMNI_F32) hipLaunchKernelGGL((wht_kernel<OMNI_F32, 32>), grid, block, 0, st, x, rows, sign_flip, out, s);
        else if (dtype == OMNI_BF16) hipLaunchKernelGGL((wht_kernel<OMNI_BF16, 32>), grid, block, 0, st, x, rows, sign_flip, out, s);
        else hipLaunchKernelGGL((wht_kernel<OMNI_F16, 32>), grid, block, 0, st, x, rows, sign_flip, out, s);
    }
    OMNI_CHECK_LAUNCH("omni_wht_rotate");
    return OMNI_OK;
}

// The table-driven wave kernel serves 16-bit inputs at D = 128 when each head
// has enough rows to amortise its 64 KB table; the rest (f32 inputs, D = 32,
// few rows per head) goes to launch_encode_rows.
static bool enc_fast(int64_t B, int64_t T, int head_dim, int x_dtype) {
    return head_dim == 128 && (x_dtype == OMNI_BF16 || x_dtype == OMNI_F16) && B * T >= 64;
}

extern "C" size_t omni_encode_workspace_size(int64_t B, int H, int64_t T, int head_dim, int x_dtype,
                                             int per_head_codebook) {
    if (B <= 0 || H <= 0 || T <= 0 || !enc_fast(B, T, head_dim, x_dtype)) return 0;
    return (size_t)(per_head_codebook ? H : 1) * kEncTab;
}

// Value-to-code tables for 16-bit inputs: one 64 KB table per codebook.
static void launch_code_tables(const float *codebooks, int per_head_codebook, int H, int x_dtype, uint8_t *tables,
                               hipStream_t st) {
    const int n_tab = per_head_codebook ? H : 1;
    if (x_dtype == OMNI_BF16)
        hipLaunchKernelGGL(code_table_kernel<OMNI_BF16>, dim3(kEncTab / 256, n_tab), dim3(256), 0, st, codebooks,
                           per_head_codebook, tables);
    else
        hipLaunchKernelGGL(code_table_kernel<OMNI_F16>, dim3(kEncTab / 256, n_tab), dim3(256), 0, st, codebooks,
                           per_head_codebook, tables);
}

// The wave kernel over nz (1 or 2) tensors of one shape, tables built.
// Paged output of the encoder (omni_encode_paged).  V rows there cost less
// (codes only): K takes this share (%) of the blocks.
constexpr int kEncPagedKShare = 55;
struct EncPaged {
    const int32_t *page_table, *positions;
    int64_t max_pages, n_pages;
    int page_shift;
};

static int launch_encode128(const void *const xs[2], int nz, int x_dtype, int64_t B, int H, int64_t T, int rotate,
                            const int8_t *sign_flip, const float *codebooks, int per_head_codebook,
                            const uint32_t *g_bits, const uint8_t *tables, uint8_t *const nib[2],
                            uint8_t *const qjl[2], float *const nrm[2], hipStream_t st,
                            const EncPaged *paged = nullptr) {
    EncArgs a{};
    for (int z = 0; z < 2; ++z) {
        const int zz = z < nz ? z : 0;
        a.x[z] = xs[zz]; a.nibbles[z] = nib[zz]; a.qjl[z] = qjl[zz]; a.norms[z] = nrm[zz];
    }
    a.table = tables; a.codebooks = codebooks; a.g_bits = g_bits; a.sign_flip = sign_flip;
    a.T = T; a.nrows_head = B * T; a.H = H; a.per_head = per_head_codebook; a.rotate = rotate;
    a.scale = inv_sqrt_dim_f32(128);
    // about one block per CU across the tensors and heads; each block a run
    // of rows of one head of one tensor
    const int cus = device_cus();
    // paged K and V: V writes codes only (about 0.4 of K's work per row),
    // so K's rows are spread over more blocks
    const int64_t grp = 16 * kEncWaves;
    const int64_t per_tensor = (cus + (int64_t)H - 1) / H;         // blocks per head over the tensors
    int64_t nxz[2] = {1, 1};
    for (int z = 0; z < 2; ++z) {
        int64_t blocks = (per_tensor + nz - 1) / nz;
        if (paged && nz == 2) blocks = z == 0 ? per_tensor * kEncPagedKShare / 100
                                              : per_tensor - per_tensor * kEncPagedKShare / 100;
        if (blocks < 1) blocks = 1;
        int64_t rpb = (a.nrows_head + blocks - 1) / blocks;
        rpb = (rpb + grp - 1) / grp * grp;
        a.rows_per_block[z] = rpb;
        nxz[z] = (a.nrows_head + rpb - 1) / rpb;
    }
    a.nx0 = (int)nxz[0];
    // paged: one grid row of K's blocks then V's (no empty blocks); else
    // blockIdx.z picks the tensor
    const int64_t nx = paged ? nxz[0] + (nz > 1 ? nxz[1] : 0) : nxz[0];
    OMNI_CHECK_ARG(nx <= 2147483647LL, "omni_encode: grid too large");
    const dim3 eg((unsigned)nx, (unsigned)H, paged ? 1u : (unsigned)nz), eb(64 * kEncWaves);
    if (paged) {
        a.page_table = paged->page_table; a.positions = paged->positions;
        a.max_pages = paged->max_pages; a.n_pages = paged->n_pages; a.page_shift = paged->page_shift;
        if (x_dtype == OMNI_BF16) {
            if (rotate) hipLaunchKernelGGL((encode128_kernel<OMNI_BF16, true, true>), eg, eb, 0, st, a);
            else hipLaunchKernelGGL((encode128_kernel<OMNI_BF16, false, true>), eg, eb, 0, st, a);
        } else {
            if (rotate) hipLaunchKernelGGL((encode128_kernel<OMNI_F16, true, true>), eg, eb, 0, st, a);
            else hipLaunchKernelGGL((encode128_kernel<OMNI_F16, false, true>), eg, eb, 0, st, a);
        }
    } else if (x_dtype == OMNI_BF16) {
        if (rotate) hipLaunchKernelGGL((encode128_kernel<OMNI_BF16, true, false>), eg, eb, 0, st, a);
        else hipLaunchKernelGGL((encode128_kernel<OMNI_BF16, false, false>), eg, eb, 0, st, a);
    } else {
        if (rotate) hipLaunchKernelGGL((encode128_kernel<OMNI_F16, true, false>), eg, eb, 0, st, a);
        else hipLaunchKernelGGL((encode128_kernel<OMNI_F16, false, false>), eg, eb, 0, st, a);
    }
    OMNI_CHECK_LAUNCH("omni_encode");
    return OMNI_OK;
}

// encode_grid_kernel over nz (1 or 2) tensors of one shape.
template <int XDT, int D>
static void launch_encode_grid(const EncArgs &a, dim3 grid, hipStream_t st) {
    if (a.rotate) hipLaunchKernelGGL((encode_grid_kernel<XDT, D, true>), grid, dim3(64 * kEgWaves), 0, st, a);
    else hipLaunchKernelGGL((encode_grid_kernel<XDT, D, false>), grid, dim3(64 * kEgWaves), 0, st, a);
}

// Inputs without a value table (f32, D = 32, few rows per head).
static int launch_encode_rows(const void *const xs[2], int nz, int x_dtype, int64_t B, int H, int64_t T, int head_dim,
                              int rotate, const int8_t *sign_flip, const float *codebooks, int per_head_codebook,
                              const uint32_t *g_bits, uint8_t *const nib[2], uint8_t *const qjl[2],
                              float *const nrm[2], hipStream_t st) {
    const float s = inv_sqrt_dim_f32(head_dim);
    EncArgs a{};
    for (int z = 0; z < 2; ++z) {
        const int zz = z < nz ? z : 0;
        a.x[z] = xs[zz]; a.nibbles[z] = nib[zz]; a.qjl[z] = qjl[zz]; a.norms[z] = nrm[zz];
    }
    a.codebooks = codebooks; a.g_bits = g_bits; a.sign_flip = sign_flip;
    a.T = T; a.nrows_head = B * T; a.H = H; a.per_head = per_head_codebook; a.rotate = rotate;
    a.scale = s;
    // three blocks of four waves per CU across the tensors and heads, each
    // a run of rows of one head of one tensor
    const int64_t grp = (head_dim == 128 ? 16 : 64) * kEgWaves;
    const int64_t want = ((int64_t)3 * device_cus() + (int64_t)H * nz - 1) / ((int64_t)H * nz);
    int64_t rpb = (a.nrows_head + want - 1) / want;
    rpb = (rpb + grp - 1) / grp * grp;
    a.rows_per_block[0] = a.rows_per_block[1] = rpb;
    a.step_b = grp / T;
    a.step_t = grp % T;
    const int64_t nx = (a.nrows_head + rpb - 1) / rpb;
    OMNI_CHECK_ARG(nx <= 2147483647LL, "omni_encode: grid too large");
    const dim3 eg((unsigned)nx, (unsigned)H, (unsigned)nz);
    if (head_dim == 128) {
        if (x_dtype == OMNI_F32) launch_encode_grid<OMNI_F32, 128>(a, eg, st);
        else if (x_dtype == OMNI_BF16) launch_encode_grid<OMNI_BF16, 128>(a, eg, st);
        else launch_encode_grid<OMNI_F16, 128>(a, eg, st);
    } else {
        if (x_dtype == OMNI_F32) launch_encode_grid<OMNI_F32, 32>(a, eg, st);
        else if (x_dtype == OMNI_BF16) launch_encode_grid<OMNI_BF16, 32>(a, eg, st);
        else launch_encode_grid<OMNI_F16, 32>(a, eg, st);
    }
    OMNI_CHECK_LAUNCH("omni_encode");
    return OMNI_OK;
}

extern "C" int omni_encode(const void *x, int x_dtype, int64_t B, int H, int64_t T, int head_dim,
                           int rotate, const int8_t *sign_flip, const float *codebooks,
                           int per_head_codebook, const uint32_t *g_bits,
                           uint8_t *nibbles, uint8_t *qjl, float *norms,
                           void *workspace, size_t workspace_bytes, void *stream) {
    OMNI_CHECK_ARG(dtype_ok(x_dtype), "omni_encode: bad dtype %d", x_dtype);
    OMNI_CHECK_ARG(head_dim_ok(head_dim), "omni_encode: head_dim must be 128 or 32, got %d", head_dim);
    OMNI_CHECK_ARG(B >= 0 && H >= 0 && T >= 0, "omni_encode: negative shape");
    if (B == 0 || H == 0 || T == 0) return OMNI_OK;
    OMNI_CHECK_ARG(x && codebooks && g_bits && nibbles && qjl && norms, "omni_encode: NULL pointer");
    OMNI_CHECK_ARG(B <= 65535 && H <= 65535, "omni_encode: B and H must be <= 65535");
    hipStream_t st = as_stream(stream);
    const void *xs[2] = {x, x};
    uint8_t *nib[2] = {nibbles, nibbles}, *qj[2] = {qjl, qjl};
    float *nr[2] = {norms, norms};
    if (enc_fast(B, T, head_dim, x_dtype)) {
        const size_t need = omni_encode_workspace_size(B, H, T, head_dim, x_dtype, per_head_codebook);
        if (workspace == nullptr || workspace_bytes < need) {
            set_error("omni_encode: workspace of %zu bytes required, %zu given", need, workspace_bytes);
            return OMNI_EWORKSPACE;
        }
        uint8_t *table = reinterpret_cast<uint8_t *>(workspace);
        launch_code_tables(codebooks, per_head_codebook, H, x_dtype, table, st);
        OMNI_CHECK_LAUNCH("omni_encode (code table)");
        return launch_encode128(xs, 1, x_dtype, B, H, T, rotate, sign_flip, codebooks, per_head_codebook, g_bits,
                                table, nib, qj, nr, st);
    }
    return launch_encode_rows(xs, 1, x_dtype, B, H, T, head_dim, rotate, sign_flip, codebooks, per_head_codebook,
                              g_bits, nib, qj, nr, st);
}

extern "C" size_t omni_encode_tables_size(int H, int per_head_codebook) {
    if (H <= 0) return 0;
    return (size_t)(per_head_codebook ? H : 1) * kEncTab;
}

extern "C" int omni_encode_build_tables(const float *codebooks, int per_head_codebook, int H, int x_dtype,
                                        uint8_t *tables, size_t tables_bytes, void *stream) {
    OMNI_CHECK_ARG(x_dtype == OMNI_BF16 || x_dtype == OMNI_F16,
                   "omni_encode_build_tables: tables serve 16-bit inputs (dtype %d)", x_dtype);
    OMNI_CHECK_ARG(H > 0 && H <= 65535, "omni_encode_build_tables: need 1 <= H <= 65535");
    OMNI_CHECK_ARG(codebooks && tables, "omni_encode_build_tables: NULL pointer");
    const size_t need = omni_encode_tables_size(H, per_head_codebook);
    if (tables_bytes < need) {
        set_error("omni_encode_build_tables: %zu bytes of tables required, %zu given", need, tables_bytes);
        return OMNI_EWORKSPACE;
    }
    launch_code_tables(codebooks, per_head_codebook, H, x_dtype, tables, as_stream(stream));
    OMNI_CHECK_LAUNCH("omni_encode_build_tables");
    return OMNI_OK;
}

extern "C" int omni_encode_pair(const void *x0, const void *x1, int x_dtype, int64_t B, int H, int64_t T,
                                int head_dim, int rotate, const int8_t *sign_flip, const float *codebooks,
                                int per_head_codebook, const uint32_t *g_bits, const uint8_t *tables,
                                size_t tables_bytes, uint8_t *nibbles0, uint8_t *qjl0, float *norms0,
                                uint8_t *nibbles1, uint8_t *qjl1, float *norms1, void *stream) {
    OMNI_CHECK_ARG(dtype_ok(x_dtype), "omni_encode_pair: bad dtype %d", x_dtype);
    OMNI_CHECK_ARG(head_dim_ok(head_dim), "omni_encode_pair: head_dim must be 128 or 32, got %d", head_dim);
    OMNI_CHECK_ARG(B >= 0 && H >= 0 && T >= 0, "omni_encode_pair: negative shape");
    if (B == 0 || H == 0 || T == 0) return OMNI_OK;
    const int nz = x1 ? 2 : 1;
    OMNI_CHECK_ARG(x0 && codebooks && g_bits && nibbles0 && qjl0 && norms0, "omni_encode_pair: NULL pointer");
    OMNI_CHECK_ARG(nz == 1 || (nibbles1 && qjl1 && norms1), "omni_encode_pair: NULL output for the second tensor");
    OMNI_CHECK_ARG(B <= 65535 && H <= 65535, "omni_encode_pair: B and H must be <= 65535");
    hipStream_t st = as_stream(stream);
    const void *xs[2] = {x0, x1 ? x1 : x0};
    uint8_t *nib[2] = {nibbles0, nz > 1 ? nibbles1 : nibbles0}, *qj[2] = {qjl0, nz > 1 ? qjl1 : qjl0};
    float *nr[2] = {norms0, nz > 1 ? norms1 : norms0};
    if (enc_fast(B, T, head_dim, x_dtype)) {
        const size_t need = omni_encode_tables_size(H, per_head_codebook);
        if (tables == nullptr || tables_bytes < need) {
            set_error("omni_encode_pair: %zu bytes of code tables required, %zu given", need, tables_bytes);
            return OMNI_EWORKSPACE;
        }
        return launch_encode128(xs, nz, x_dtype, B, H, T, rotate, sign_flip, codebooks, per_head_codebook, g_bits,
                                tables, nib, qj, nr, st);
    }
    return launch_encode_rows(xs, nz, x_dtype, B, H, T, head_dim, rotate, sign_flip, codebooks, per_head_codebook,
                              g_bits, nib, qj, nr, st);
}

extern "C" int omni_encode_paged(const void *k, const void *v, int x_dtype, int64_t B, int H, int64_t T,
                                 int rotate, const int8_t *sign_flip, const float *codebooks,
                                 int per_head_codebook, const uint32_t *g_bits, const uint8_t *tables,
                                 size_t tables_bytes, const int32_t *page_table, int64_t max_pages,
                                 const int32_t *positions, int64_t n_pages, int page_size, uint8_t *k_nibbles,
                                 uint8_t *k_qjl, float *k_norms, uint8_t *v_nibbles, void *stream) {
    OMNI_CHECK_ARG(x_dtype == OMNI_BF16 || x_dtype == OMNI_F16, "omni_encode_paged: K and V must be bf16 or f16");
    OMNI_CHECK_ARG(B >= 0 && H >= 0 && T >= 0, "omni_encode_paged: negative shape");
    if (B == 0 || H == 0 || T == 0) return OMNI_OK;
    OMNI_CHECK_ARG(k && codebooks && g_bits && page_table && positions && k_nibbles && k_qjl && k_norms,
                   "omni_encode_paged: NULL pointer");
    OMNI_CHECK_ARG(v == nullptr || v_nibbles, "omni_encode_paged: NULL V pool for a V input");
    OMNI_CHECK_ARG(B <= 65535 && H <= 65535, "omni_encode_paged: B and H must be <= 65535");
    int shift = 4;
    while (shift < 11 && (1 << shift) < page_size) ++shift;
    OMNI_CHECK_ARG(page_size >= 16 && page_size <= 1024 && (1 << shift) == page_size,
                   "omni_encode_paged: page_size must be a power of two in [16, 1024], got %d", page_size);
    OMNI_CHECK_ARG(n_pages >= 1 && max_pages >= 1, "omni_encode_paged: need n_pages >= 1, max_pages >= 1");
    OMNI_CHECK_ARG(n_pages * H * (int64_t)page_size < (int64_t(1) << 40), "omni_encode_paged: pool too large");
    const size_t need = omni_encode_tables_size(H, per_head_codebook);
    if (tables == nullptr || tables_bytes < need) {
        set_error("omni_encode_paged: %zu bytes of code tables required, %zu given", need, tables_bytes);
        return OMNI_EWORKSPACE;
    }
    const int nz = v ? 2 : 1;
    const void *xs[2] = {k, v ? v : k};
    uint8_t *nib[2] = {k_nibbles, v ? v_nibbles : k_nibbles}, *qj[2] = {k_qjl, k_qjl};
    float *nr[2] = {k_norms, k_norms};
    const EncPaged pg{page_table, positions, max_pages, n_pages, shift};
    return launch_encode128(xs, nz, x_dtype, B, H, T, rotate, sign_flip, codebooks, per_head_codebook, g_bits,
                            tables, nib, qj, nr, as_stream(stream), &pg);
}

extern "C" int omni_dequantize(const uint8_t *nibbles, const uint8_t *qjl, const float *norms,
                               const float *codebooks, int per_head_codebook, const uint32_t *g_bits,
                               int64_t B, int H, int64_t T, int head_dim, int with_qjl, float *out,
                               void *stream) {
    OMNI_CHECK_ARG(head_dim_ok(head_dim), "omni_dequantize: head_dim must be 128 or 32, got %d", head_dim);
    OMNI_CHECK_ARG(B >= 0 && H >= 0 && T >= 0, "omni_dequantize: negative shape");
    if (B == 0 || H == 0 || T == 0) return OMNI_OK;
    OMNI_CHECK_ARG(nibbles && codebooks && out, "omni_dequantize: NULL pointer");
    OMNI_CHECK_ARG(!with_qjl || (qjl && norms && g_bits), "omni_dequantize: NULL QJL pointer");
    OMNI_CHECK_ARG(B <= 65535 && H <= 65535, "omni_dequantize: B and H must be <= 65535");
    // runs of rows of one head, about eight blocks per CU and no shorter than
    // four passes of a block
    const int64_t rows_head = B * T;
    const int unit = 4 * (kDqThreads / (head_dim / 4));
    int64_t rpb = rows_head * H / (8 * device_cus());
    rpb = (rpb / unit) * unit;
    rpb = rpb < unit ? unit : (rpb > 2048 ? 2048 : rpb);
    const int64_t nx = (rows_head + rpb - 1) / rpb;
    OMNI_CHECK_ARG(nx <= 2147483647LL, "omni_dequantize: grid too large");
    const dim3 grid((unsigned)nx, (unsigned)H), block(kDqThreads);
    // floor(2^32 / T) + 1: exact quotients below 2^16 (t0 + 2048 stays there)
    const uint64_t magic = T < 60000 ? ((uint64_t)1 << 32) / (uint64_t)T + 1 : 0;
    const float c = (float)(sqrt(2.0 / M_PI) / (double)head_dim);
    hipStream_t st = as_stream(stream);
    if (head_dim == 128) {
        if (with_qjl) hipLaunchKernelGGL((dequant_kernel<128, true>), grid, block, 0, st, nibbles, qjl, norms, codebooks,
                                         per_head_codebook, g_bits, T, H, rows_head, (int)rpb, magic, out, c);
        else hipLaunchKernelGGL((dequant_kernel<128, false>), grid, block, 0, st, nibbles, qjl, norms, codebooks,
                                per_head_codebook, g_bits, T, H, rows_head, (int)rpb, magic, out, c);
    } else {
        if (with_qjl) hipLaunchKernelGGL((dequant_kernel<32, true>), grid, block, 0, st, nibbles, qjl, norms, codebooks,
                                         per_head_codebook, g_bits, T, H, rows_head, (int)rpb, magic, out, c);
        else hipLaunchKernelGGL((dequant_kernel<32, false>), grid, block, 0, st, nibbles, qjl, norms, codebooks,
                                per_head_codebook, g_bits, T, H, rows_head, (int)rpb, magic, out, c);
    }
    OMNI_CHECK_LAUNCH("omni_dequantize");
    return OMNI_OK;
}
