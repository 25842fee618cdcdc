// Dense fp32 GQA attention on already dequantized K / V (gfx950).
//
// Reference: reference_attn (omnistack_rs/attention/reference.py:72-177),
// the CPU path's attention: fp32 scores q . k * scale (+ an additive mask
// broadcastable to (B, Hq, T, S)), online softmax over key tiles, fp32
// P . V, output O / l; kv head of q head h = h / (Hq / Hkv) (repeat_kv,
// :49-67) without materialising the repeated K / V.
//
// One block per 64 query rows of one (batch, kv head): four waves of 16 rows
// (row r = t * G + g of that kv head).  Keys go through LDS in tiles of 32;
// scores and P . V run on v_mfma_f32_16x16x4_f32 (fp32 products, fp32
// accumulation), the softmax in fp32 with expf.  The running-max update is the
// reference's, made safe for tiles whose scores are all -inf (alpha and p are
// 0 there instead of exp(-inf - -inf)); the reference's own result for a row
// whose whole first tile of `first_tile` keys is masked (NaN) is reproduced
// explicitly, and a NaN score makes its row NaN as torch.maximum / amax
// propagate it.
#include <math.h>

#include "omni_common.h"

namespace omni {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct DenseArgs {
    const float *q, *k, *v, *mask;
    float *out;
    int64_t ms_b, ms_h, ms_t, ms_s;   // mask strides in elements (0: broadcast)
    int64_t B, T, S, rows, first_tile;
    int Hq, Hkv, G;
    float scale;
};

constexpr int kDnKeys = 32;          // keys per LDS tile
constexpr int kDnWaves = 4;
constexpr int kDnRows = 16 * kDnWaves;
constexpr int kDnKsWaves = 8;

// Raw buffer descriptor, dword 3.
constexpr int kDnBufWord3 = 0x00020000;
// Four floats at any 4-byte aligned address.
typedef float dn_f4_t __attribute__((ext_vector_type(4), aligned(4)));

// Scores are computed transposed, S^T = K Q^T (keys on M, query rows on N),
// so that lane (n, g) of the MFMA result holds keys 16 kb + 4 g + i of query
// row n: a row's maximum is a register reduction and two cross-row swaps, and
// the probabilities are the B operand of O^T += V^T P^T as they stand (k slot
// g of step i is key 4 g + i).  Both contractions take their k slots in the
// order that 16-byte reads give: dims 16 t + 4 g + u for the scores, and
// output row m of MFMA (h, j) is dim 16 VJ h + VJ m + j.
template <int D>
struct DnRow {
    static constexpr int VJ = D >= 64 ? 4 : 2, NH = D / (16 * VJ);
    f32x4_t o[NH][VJ];               // lane (n, g): dims 16 VJ h + VJ (4 g + i) + j of row n
    float m, l;                      // running maximum (of the row), denominator (of the lane's keys)
    int seen0, nan;                  // lane's keys: a score above -inf in the first tile, a NaN score
    const float *mrow;               // the row's mask
    bool ok;
};

__device__ __forceinline__ float dn_max_groups(float m) {
    auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    m = fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
    auto u = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    return fmaxf(__uint_as_float(u[0]), __uint_as_float(u[1]));
}
__device__ __forceinline__ float dn_sum_groups(float v) {
    auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(t[0]) + __uint_as_float(t[1]);
    auto u = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(u[0]) + __uint_as_float(u[1]);
}

// Query row `r` of this kv head (past the last: row 0, never stored) as B operand: qb[4 t + u] = dim 16 t + 4 g + u.
template <int D>
__device__ __forceinline__ void dn_init(const DenseArgs &a, int64_t b, int hk, int64_t r, int g, DnRow<D> &R, float (&qb)[D / 4]) {
    R.ok = r < a.rows;
    const int64_t t = R.ok ? r / a.G : 0;
    const int hq = hk * a.G + (R.ok ? (int)(r - t * a.G) : 0);
    const float *qrow = a.q + ((b * a.Hq + hq) * a.T + t) * D + 4 * g;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
        const dn_f4_t w = *reinterpret_cast<const dn_f4_t *>(qrow + 16 * s);
#pragma unroll
        for (int u = 0; u < 4; ++u) qb[4 * s + u] = w[u];
    }
#pragma unroll
    for (int h = 0; h < DnRow<D>::NH; ++h)
#pragma unroll
        for (int j = 0; j < DnRow<D>::VJ; ++j) R.o[h][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    R.m = -INFINITY;
    R.l = 0.0f;
    R.seen0 = R.nan = 0;
    R.mrow = a.mask + (b * a.ms_b + hq * a.ms_h + t * a.ms_t);
}

// Mask values of the lane's keys key .. key + 3 (`whole`: all keys of the
// wave's tile are below S; otherwise keys past S get -inf).  Lanes past the
// last row read row 0 of the kv head.
__device__ __forceinline__ void dn_mask(const DenseArgs &a, const float *mrow, int64_t key, bool whole, float (&mk)[4]) {
    if (whole && a.ms_s == 1) {
        const dn_f4_t w = *reinterpret_cast<const dn_f4_t *>(mrow + key);
#pragma unroll
        for (int i = 0; i < 4; ++i) mk[i] = w[i];
    } else {
        const float *p = mrow;
        asm volatile("" : "+v"(p));          // (nothing of this path is formed ahead, outside the loop over tiles)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t k = key + i < a.S ? key + i : a.S - 1;
            const float w = p[k * a.ms_s];
            mk[i] = key + i < a.S ? w : -INFINITY;
        }
    }
}

// Online softmax over the raw scores of KB blocks of 16 keys from key0 on:
// acc becomes the probabilities, the output and denominator are rescaled.
template <int D, int KB, bool MASK>
__device__ __forceinline__ void dn_softmax(const DenseArgs &a, DnRow<D> &R, f32x4_t (&acc)[KB], const float (&mk)[KB][4],
                                           int64_t key0, int g) {
    float mt = -INFINITY;
    const bool tail = key0 + 16 * KB > a.S, first = key0 < a.first_tile;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float v = acc[kb][i] * a.scale;
            if (MASK) v += mk[kb][i];
            acc[kb][i] = v;
        }
    if (tail) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (key0 + 16 * kb + 4 * g + i >= a.S) acc[kb][i] = -INFINITY;
    }
    if (first) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                R.seen0 |= (int)(key0 + 16 * kb + 4 * g + i < a.first_tile) & (int)(acc[kb][i] > -INFINITY);
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            R.nan |= (int)(acc[kb][i] != acc[kb][i]);       // poisons the row (torch.maximum / amax propagate NaN)
            mt = fmaxf(mt, acc[kb][i]);
        }
    const float m_new = fmaxf(R.m, dn_max_groups(mt));
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    if (__builtin_amdgcn_ballot_w64(m_new != R.m)) {         // an unchanged maximum's factor is 1
        const float alpha = expf(R.m - m_use);
        R.l *= alpha;
#pragma unroll
        for (int h = 0; h < DnRow<D>::NH; ++h)
#pragma unroll
            for (int j = 0; j < DnRow<D>::VJ; ++j) R.o[h][j] *= alpha;
        R.m = m_new;
    }
    float ps = 0.0f;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[kb][i] = expf(acc[kb][i] - m_use);
            ps += acc[kb][i];
        }
    R.l += ps;
}

template <int D>
__device__ __forceinline__ void dn_store_row(const DenseArgs &a, const DnRow<D> &R, int64_t b, int hk, int64_t r, int g) {
    const float l = dn_sum_groups(R.l);
    const bool seen = dn_max_groups(R.seen0 ? 1.0f : 0.0f) > 0.0f, nan = dn_max_groups(R.nan ? 1.0f : 0.0f) > 0.0f;
    if (!R.ok) return;
    const int64_t t = r / a.G;
    const int hq = hk * a.G + (int)(r - t * a.G);
    float *orow = a.out + ((b * a.Hq + hq) * a.T + t) * D;
    constexpr int VJ = DnRow<D>::VJ;
#pragma unroll
    for (int h = 0; h < DnRow<D>::NH; ++h)
#pragma unroll
        for (int e = 0; e < 4 * VJ; e += 4) {
            dn_f4_t w;
#pragma unroll
            for (int u = 0; u < 4; ++u)
                w[u] = (nan || !seen) ? __builtin_nanf("") : R.o[h][(e + u) % VJ][(e + u) / VJ] / l;
            *reinterpret_cast<dn_f4_t *>(orow + 16 * VJ * h + 4 * VJ * g + e) = w;
        }
}

// Bits of |x| as an integer: NaN above inf above every finite value.
__device__ __forceinline__ uint32_t dn_abs_bits(float x) { return __float_as_uint(x) & 0x7FFFFFFFu; }
__device__ __forceinline__ uint32_t dn_abs_max(uint32_t m, float4 v) {
    const uint32_t x = dn_abs_bits(v.x), y = dn_abs_bits(v.y), z = dn_abs_bits(v.z), w = dn_abs_bits(v.w);
    const uint32_t xy = x > y ? x : y, zw = z > w ? z : w, e = xy > zw ? xy : zw;
    return m > e ? m : e;
}

// Bound by the fp32 matrix rate: 2 x 1000 queries, 32 heads over 8, 1000 keys,
// head_dim 128, 294 us without a mask (111 of the 154 TFLOP/s that a large
// product reaches) and 220 us causal, where half of the tiles are hidden and
// skipped; with row-major scores, whose maxima and sums were 16-lane
// shuffles, and P through LDS 485 and 537 us.  Registers for three waves per
// SIMD: two of them 369 us.
template <int D, bool MASK>
__global__ __launch_bounds__(64 * kDnWaves, D == 256 ? 1 : (D == 128 ? 3 : 4)) void dense_attn_kernel(DenseArgs a) {
    constexpr int DP = D + 4;                     // padded LDS row (floats): 16-byte reads of 16 rows cover all banks
    constexpr int VJ = DnRow<D>::VJ, NH = DnRow<D>::NH;
    __shared__ __attribute__((aligned(16))) float ks[kDnKeys * DP];
    __shared__ __attribute__((aligned(16))) float vs[kDnKeys * DP];
    __shared__ uint32_t wild[kDnWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, g = lane >> 4;
    // the last rows first: under a causal mask they are the longest
    const int64_t bh = (int64_t)a.Hkv * a.B, id = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
    const int64_t chunk = (a.rows + kDnRows - 1) / kDnRows - 1 - id / bh, b = id % bh / a.Hkv;
    if (chunk < 0) return;                        // past the last block
    const int hk = (int)(id % bh % a.Hkv);
    const int64_t row0 = chunk * kDnRows + 16 * wave;

    DnRow<D> R;
    float qb[D / 4];
    dn_init<D>(a, b, hk, row0 + n, g, R, qb);
    const float *kb0 = a.k + ((int64_t)b * a.Hkv + hk) * a.S * D;
    const float *vb0 = a.v + ((int64_t)b * a.Hkv + hk) * a.S * D;
    // waves whose 16 rows are all past the end only help stage K / V
    const bool active = row0 < a.rows;
    // |q|, |k| < 2^48 and |scale| < 2^20: no score can leave the finite range
    constexpr uint32_t kTame = 0x57800000u;
    uint32_t qm = 0;
#pragma unroll
    for (int s = 0; s < D / 4; ++s) qm = qm > dn_abs_bits(qb[s]) ? qm : dn_abs_bits(qb[s]);
    const bool may_skip = MASK && fabsf(a.scale) < 1048576.0f && !__builtin_amdgcn_ballot_w64(qm >= kTame);

    // the next tile's K / V sit in registers while the current one is used
    constexpr int kPer = kDnKeys * D / (4 * 64 * kDnWaves);   // float4 per thread per tile
    float4 nk[kPer], nv[kPer];
    float mk[2][4] = {};
    auto fetch = [&](int64_t s0) {
        // the tile's keys below S as buffers: lanes past them read 0 (the
        // whole offset is the lane's and the instruction's: the scalar one is
        // not range-checked); a wave's loads are consecutive KB
        const int bytes = (int)(s0 + kDnKeys <= a.S ? kDnKeys : a.S - s0) * D * 4;
        const __amdgpu_buffer_rsrc_t K = __builtin_amdgcn_make_buffer_rsrc((void *)(kb0 + s0 * D), (short)0, bytes, kDnBufWord3);
        const __amdgpu_buffer_rsrc_t V = __builtin_amdgcn_make_buffer_rsrc((void *)(vb0 + s0 * D), (short)0, bytes, kDnBufWord3);
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
            nk[c] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(K, 16 * lane + 1024 * (kPer * wave + c), 0, 0));
            nv[c] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(V, 16 * lane + 1024 * (kPer * wave + c), 0, 0));
        }
    };
    if (a.S > 0) fetch(0);

    for (int64_t s0 = 0; s0 < a.S; s0 += kDnKeys) {
        if (MASK) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) dn_mask(a, R.mrow, s0 + 16 * kb + 4 * g, s0 + kDnKeys <= a.S, mk[kb]);
        }
        __syncthreads();                          // the previous tile is consumed
        uint32_t km = 0, vm = 0;
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
            const int e = 4 * (lane + 64 * (kPer * wave + c));
            const int key = e / D, d = e - key * D;
            *reinterpret_cast<float4 *>(ks + key * DP + d) = nk[c];
            *reinterpret_cast<float4 *>(vs + key * DP + d) = nv[c];
            if (MASK) {
                km = dn_abs_max(km, nk[c]);
                vm = dn_abs_max(vm, nv[c]);
            }
        }
        if (MASK) {
            const uint64_t w = __builtin_amdgcn_ballot_w64(km >= kTame || vm >= 0x7F800000u);
            if (lane == 0) wild[wave] = w != 0;
        }
        __syncthreads();
        if (s0 + kDnKeys < a.S) fetch(s0 + kDnKeys);
        if (!active) continue;
        // every key hidden from every row of the wave, K and q tame, V
        // finite: all scores are -inf, all probabilities 0 and 0 V = 0, so
        // the tile changes nothing
        if (MASK) {
            int visible = 0;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 4; ++i) visible |= (int)!(mk[kb][i] == -INFINITY);
            uint32_t w = __builtin_amdgcn_ballot_w64(visible != 0) != 0 || !may_skip;
            if (w == 0) {
#pragma unroll
                for (int k = 0; k < kDnWaves; ++k) w |= wild[k];
            }
            if (__builtin_amdgcn_readfirstlane((int)w) == 0) continue;
        }

        // one step's LDS reads ahead of the MFMAs, no more (the scheduler
        // would hoist all of them and spill)
        f32x4_t acc[2];
        acc[0] = acc[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        auto read_k = [&](int t, int kb) { return *reinterpret_cast<const f32x4_t *>(ks + (16 * kb + n) * DP + 16 * t + 4 * g); };
        f32x4_t kw[2] = {read_k(0, 0), read_k(0, 1)};
#pragma unroll
        for (int t = 0; t < D / 16; ++t) {
            f32x4_t nx[2];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) nx[kb] = read_k(t + 1 < D / 16 ? t + 1 : t, kb);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
                    acc[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kw[kb][u], qb[4 * t + u], acc[kb], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            kw[0] = nx[0];
            kw[1] = nx[1];
        }
        typedef float vj_t __attribute__((ext_vector_type(VJ)));
        auto read_v = [&](int s, int h) {                  // step s: key 16 (s / 4) + 4 g + s % 4
            return *reinterpret_cast<const vj_t *>(vs + (16 * (s / 4) + 4 * g + s % 4) * DP + 16 * VJ * h + VJ * n);
        };
        vj_t vw[NH];
#pragma unroll
        for (int h = 0; h < NH; ++h) vw[h] = read_v(0, h);
        dn_softmax<D, 2, MASK>(a, R, acc, mk, s0, g);
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            vj_t nx[NH];
#pragma unroll
            for (int h = 0; h < NH; ++h) nx[h] = read_v(s < 7 ? s + 1 : s, h);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < NH; ++h)
#pragma unroll
                for (int j = 0; j < VJ; ++j)
                    R.o[h][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vw[h][j], acc[s / 4][s % 4], R.o[h][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < NH; ++h) vw[h] = nx[h];
        }
    }
    if (active) dn_store_row<D>(a, R, b, hk, row0 + n, g);
}

// Few query rows (decode): the NW waves share one group of 16 rows and split
// the keys in 16-key chunks (wave w takes chunks w, w + NW, ...), each keeping
// its own online-softmax state; the states are merged in LDS at the end (max,
// then the exp-weighted sums in wave order).  K and V go from memory straight
// into MFMA operand registers (no LDS staging, no block barrier per tile),
// two chunks in flight per wave.  16 sequences of 4000 keys, 32 heads over 8,
// one query each: 109.8 us, 4.8 TB/s (152 us with row-major scores); one
// sequence 91 us (146), bound by the matrix work on rows that do not exist.
template <int D>
struct DnChunk {
    float k[D / 4];       // key 16 c + n: k[4 t + u] = dim 16 t + 4 g + u
    float v[D / 4];       // key 16 c + 4 g + i: v[(i NH + h) VJ + j] = dim 16 VJ h + VJ n + j
    float mk[1][4];
};

template <int D, int NW, bool MASK>
__global__ __launch_bounds__(64 * NW) void dense_attn_ks_kernel(DenseArgs a) {
    constexpr int DP = D + 4, VJ = DnRow<D>::VJ, NH = DnRow<D>::NH;
    __shared__ float wst[NW][16][4];             // per wave and row: m, l, seen0, nan
    __shared__ __attribute__((aligned(16))) float op[NW * 16 * DP];   // per wave and row: O
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, g = lane >> 4;
    const int hk = blockIdx.y;
    const int64_t b = blockIdx.z;
    const int64_t row0 = 16 * (int64_t)blockIdx.x;

    DnRow<D> R;
    float qb[D / 4];
    dn_init<D>(a, b, hk, row0 + n, g, R, qb);
    const float *kb0 = a.k + ((int64_t)b * a.Hkv + hk) * a.S * D;
    const float *vb0 = a.v + ((int64_t)b * a.Hkv + hk) * a.S * D;
    const int S = (int)a.S;                                 // < 2^27 (host check)
    const int nch = (S + 15) / 16;
    // chunk c's operands; keys past S read the last key (a valid address)
    // and their V is zeroed (their P is 0, and 0 * inf would be NaN)
    auto load = [&](DnChunk<D> &C, int c) {
        const int key = 16 * c + n, kk = key < S ? key : S - 1;
        const float4 *kp = reinterpret_cast<const float4 *>(kb0 + (int64_t)kk * D + 4 * g);
#pragma unroll
        for (int t = 0; t < D / 16; ++t) {
            const float4 w = kp[4 * t];
            C.k[4 * t] = w.x; C.k[4 * t + 1] = w.y; C.k[4 * t + 2] = w.z; C.k[4 * t + 3] = w.w;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int vk = 16 * c + 4 * g + i, vv = vk < S ? vk : S - 1;
            const bool z = vk >= S;
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                const float *vp = vb0 + (int64_t)vv * D + 16 * VJ * h + VJ * n;
                float *dst = C.v + (i * NH + h) * VJ;
                if constexpr (VJ == 4) {
                    const float4 w = *reinterpret_cast<const float4 *>(vp);
                    dst[0] = z ? 0.0f : w.x; dst[1] = z ? 0.0f : w.y; dst[2] = z ? 0.0f : w.z; dst[3] = z ? 0.0f : w.w;
                } else {
                    const float2 w = *reinterpret_cast<const float2 *>(vp);
                    dst[0] = z ? 0.0f : w.x; dst[1] = z ? 0.0f : w.y;
                }
            }
        }
        if (MASK) dn_mask(a, R.mrow, 16 * (int64_t)c + 4 * g, 16 * (c + 1) <= S, C.mk[0]);
    };
    auto step = [&](const DnChunk<D> &C, int c) {
        f32x4_t acc[1] = {f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int s = 0; s < D / 4; ++s) acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(C.k[s], qb[s], acc[0], 0, 0, 0);
        dn_softmax<D, 1, MASK>(a, R, acc, C.mk, 16 * (int64_t)c, g);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int h = 0; h < NH; ++h)
#pragma unroll
                for (int j = 0; j < VJ; ++j)
                    R.o[h][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(C.v[(i * NH + h) * VJ + j], acc[0][i], R.o[h][j], 0, 0, 0);
    };
    if (wave < nch) {
        // two chunks in flight: loads past the last chunk read valid
        // addresses and are never consumed
        DnChunk<D> r0, r1;
        load(r0, wave);
        for (int c = wave;; c += 2 * NW) {
            load(r1, c + NW);
            step(r0, c);
            if (c + NW >= nch) break;
            load(r0, c + 2 * NW);
            step(r1, c + NW);
            if (c + 2 * NW >= nch) break;
        }
    }

    // merge the waves' states
    const float l = dn_sum_groups(R.l), seen = dn_max_groups(R.seen0 ? 1.0f : 0.0f), nan = dn_max_groups(R.nan ? 1.0f : 0.0f);
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int e = 0; e < 4 * VJ; e += 4)
            *reinterpret_cast<float4 *>(op + (wave * 16 + n) * DP + 16 * VJ * h + 4 * VJ * g + e) =
                make_float4(R.o[h][e % VJ][e / VJ], R.o[h][(e + 1) % VJ][(e + 1) / VJ], R.o[h][(e + 2) % VJ][(e + 2) / VJ],
                            R.o[h][(e + 3) % VJ][(e + 3) / VJ]);
    if (g == 0) {
        wst[wave][n][0] = R.m;
        wst[wave][n][1] = l;
        wst[wave][n][2] = seen;
        wst[wave][n][3] = nan;
    }
    __syncthreads();
    for (int e = tid; e < 16 * D; e += 64 * NW) {
        const int r = e / D, d = e - r * D;
        const int64_t row = row0 + r;
        if (row >= a.rows) continue;
        float mx = -INFINITY;
        bool s0seen = false, isnan_row = false;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            mx = fmaxf(mx, wst[w][r][0]);
            s0seen = s0seen || wst[w][r][2] != 0.0f;
            isnan_row = isnan_row || wst[w][r][3] != 0.0f;
        }
        float lsum = 0.0f, osum = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float f = (wst[w][r][0] == -INFINITY) ? 0.0f : expf(wst[w][r][0] - mx);
            lsum += f * wst[w][r][1];
            osum += f * op[(w * 16 + r) * DP + d];
        }
        const int64_t t = row / a.G;
        const int hq = hk * a.G + (int)(row % a.G);
        a.out[((b * a.Hq + hq) * a.T + t) * D + d] = (isnan_row || !s0seen) ? __builtin_nanf("") : osum / lsum;
    }
}

}  // namespace omni

using namespace omni;

template <int D>
static void launch_rows(dim3 grid, dim3 block, hipStream_t st, const DenseArgs &a) {
    if (a.mask) hipLaunchKernelGGL((dense_attn_kernel<D, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((dense_attn_kernel<D, false>), grid, block, 0, st, a);
}
template <int D>
static void launch_keys(dim3 grid, dim3 block, hipStream_t st, const DenseArgs &a) {
    if (a.mask) hipLaunchKernelGGL((dense_attn_ks_kernel<D, kDnKsWaves, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((dense_attn_ks_kernel<D, kDnKsWaves, false>), grid, block, 0, st, a);
}

extern "C" int omni_dense_attn(const float *q, const float *k, const float *v, const float *mask,
                               const int64_t *mask_strides, int64_t B, int Hq, int Hkv, int64_t T, int64_t S,
                               int head_dim, float scale, int64_t first_tile, float *out, void *stream) {
    OMNI_CHECK_ARG(head_dim == 32 || head_dim == 64 || head_dim == 128 || head_dim == 256,
                   "omni_dense_attn: head_dim must be 32, 64, 128 or 256, got %d", head_dim);
    OMNI_CHECK_ARG(B >= 0 && Hq > 0 && Hkv > 0 && T >= 0 && S >= 0 && Hq % Hkv == 0,
                   "omni_dense_attn: bad shape");
    OMNI_CHECK_ARG(first_tile >= 1, "omni_dense_attn: first_tile must be >= 1");
    if (B == 0 || T == 0) return OMNI_OK;
    OMNI_CHECK_ARG(q && k && v && out, "omni_dense_attn: NULL pointer");
    OMNI_CHECK_ARG(mask == nullptr || mask_strides != nullptr, "omni_dense_attn: mask without strides");
    OMNI_CHECK_ARG(B <= 65535 && Hkv <= 65535, "omni_dense_attn: grid too large");
    const int G = Hq / Hkv;
    const int64_t rows = T * G;
    const int64_t chunks = (rows + kDnRows - 1) / kDnRows;
    OMNI_CHECK_ARG(chunks <= 2147483647, "omni_dense_attn: too many query rows");
    DenseArgs a;
    a.q = q; a.k = k; a.v = v; a.mask = mask; a.out = out;
    a.ms_b = mask ? mask_strides[0] : 0;
    a.ms_h = mask ? mask_strides[1] : 0;
    a.ms_t = mask ? mask_strides[2] : 0;
    a.ms_s = mask ? mask_strides[3] : 0;
    a.B = B; a.T = T; a.S = S; a.rows = rows; a.first_tile = first_tile < S ? first_tile : S;
    a.Hq = Hq; a.Hkv = Hkv; a.G = G;
    a.scale = scale;
    if (S == 0) a.first_tile = 0;   // no keys: every row is NaN (0 / 0), as the reference
    hipStream_t st = as_stream(stream);
    const int64_t blocks = chunks * Hkv * B, rgroups = (rows + 15) / 16, groups = rgroups * Hkv * B;
    // A block of the row kernel takes as long for one CU's worth of blocks as
    // for a chip full; while its 64-row blocks leave CUs idle, blocks of 16
    // rows whose waves split the keys are faster.  Up to two of those per CU
    // (head_dim 128: one runs at a time), three at smaller head_dims, and one
    // less where few keys leave most of their waves idle.  32 heads over 8, 700
    // keys, causal, row kernel against key kernel: head_dim 128, 120 queries
    // 71.5 / 30.7 us, 200 71.9 / 57.3, 350 75.9 / 82.9; head_dim 64, 200 47.2 /
    // 31.1, 700 x 2 69.6 / 161.  Few keys: head_dim 128, 512 groups of 16 rows,
    // 16 keys 12.5 / 16.4, 64 18.0 / 22.2; head_dim 64, 680 groups, causal, 128
    // keys 12.3 / 24.1, 600 42.5 / 44.5, 700 49.5 / 45.9; head_dim 32, 200 keys
    // 14.7 / 16.2, 300 18.5 / 16.0.
    const int64_t per_cu = head_dim == 128 ? (S > 64 ? 2 : 1) : (S > (head_dim == 64 ? 600 : 200) ? 3 : 2);
    if ((rows <= 16 || groups <= per_cu * device_cus()) && head_dim <= 128 &&
        S < (int64_t(1) << 27)) {
        // few rows: the waves split the keys instead of the rows
        const dim3 grid((unsigned)rgroups, (unsigned)Hkv, (unsigned)B), block(64 * kDnKsWaves);
        if (head_dim == 32) launch_keys<32>(grid, block, st, a);
        else if (head_dim == 64) launch_keys<64>(grid, block, st, a);
        else launch_keys<128>(grid, block, st, a);
        OMNI_CHECK_LAUNCH("omni_dense_attn");
        return OMNI_OK;
    }
    // a launch takes fewer than 2^32 threads in a dimension (more are cut off
    // without an error): 2^22 blocks in x, the rest in y
    const int64_t gx = blocks < (int64_t(1) << 22) ? blocks : int64_t(1) << 22, gy = (blocks + gx - 1) / gx;
    OMNI_CHECK_ARG(gy <= 65535, "omni_dense_attn: grid too large");
    const dim3 grid((unsigned)gx, (unsigned)gy), block(64 * kDnWaves);
    switch (head_dim) {
        case 32: launch_rows<32>(grid, block, st, a); break;
        case 64: launch_rows<64>(grid, block, st, a); break;
        case 128: launch_rows<128>(grid, block, st, a); break;
        default: launch_rows<256>(grid, block, st, a); break;
    }
    OMNI_CHECK_LAUNCH("omni_dense_attn");
    return OMNI_OK;
}
