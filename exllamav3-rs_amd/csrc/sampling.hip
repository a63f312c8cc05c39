// Row sampling for gfx950.
//
// exl3r_argmax_sample replaces exl3_shim_argmax_sample (reference csrc/exl3_shim.cpp:229-231 ->
// argmax_sample, kernels/generator/sampling_basic.cu:65-92, 151-172) and the generator's batched tch
// argmax over [bsz, vocab] logits (src/generator.rs:1596, draft.rs:121).  Rule (torch.argmax's): the
// first index of the row maximum among indices < max_logit, NaN counting as the maximum (the first
// NaN wins) and -0 equal to +0.
//
// exl3r_gumbel_sample / exl3r_gumbel_noise take the role of exl3_shim_gumbel_sample and
// exl3_shim_gumbel_noise_f32 (exl3_shim.cpp:232-237; sampling_basic.cu:94-128, gumbel.cu:45-62): a
// Gumbel-max draw, the argmax of logits + Gumbel(0, 1) noise, which picks index i with probability
// softmax(logits)_i.  The noise stream is this library's own, a function of (seed, row, column) only:
//   bits = Philox4x32-10(counter {column >> 2, row low, row high, 0}, key {seed, 0}), word column & 3
//   u    = ((bits >> 9) + 0.5) * 2^-23          exact, in [2^-24, 1 - 2^-24]
//   g    = -log(-log(u))                         log_f32 below, correctly ordered fp32 operations
// Philox4x32-10 is the published generator of Salmon, Moraes, Dror and Shaw ("Parallel random
// numbers: as easy as 1, 2, 3", SC 2011).
//
// Layout, few rows (decode): a row is cut into slices of 2048 or 8192 elements (argmax) or 2048 to 10240
// (draw), a 256-lane workgroup per slice (grid (slices, rows)), so a single decode row of 152k logits still
// spreads over ~75 CUs.  From 128 rows (argmax) or 384 rows (Gumbel draw): a workgroup of 512 or 1024 lanes per
// row, the index written directly.  Each lane keeps its
// best candidate as one 64-bit key -- an order-preserving image of the value in the high word, the
// complement of the index in the low word -- so "larger key" is exactly "larger value, then lower
// index".  With slices, the workgroup's maximum key (DPP butterfly, one LDS hop) goes to the row's
// int64 output with one atomicMax; a clear kernel before and a convert kernel after turn that slot
// into the index.  Capture-safe: no memset.
#include <mutex>

#include "abi.hpp"
#include "common.cuh"
#ifdef EXL3R_TUNING
#include "tuning.h"
#endif

namespace exl3r {

struct ArgArgs
{
    const char* x;
    int64_t ld;          // row stride, bytes
    int64_t n;           // candidates per row (masked length)
    int64_t rows;
    uint64_t* ids;
    uint32_t seed;       // Gumbel noise key
    int64_t slice;       // elements per slice of the sliced kernels (a multiple of 2048)
};

// Philox4x32-10: ten rounds of two 32 x 32 -> 64-bit products with the published multipliers,
// the key advanced by the published Weyl increments between rounds.
__device__ __forceinline__ void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0,
                                              uint32_t k1, uint32_t (&out)[4])
{
    #pragma unroll
    for (int round = 0; round < 10; ++round)
    {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        // three-way xor in one gfx950 bitop3 (truth table 0x96 = a ^ b ^ c)
        const uint32_t n0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c1, k0, 0x96);
        const uint32_t n2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c3, k1, 0x96);
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

// Natural log of a positive normal float in plain fp32 operations and explicit fmas, so that any
// IEEE implementation of the same steps gives the same bits.  x = 2^e m, m in [sqrt(1/2), sqrt(2))
// (0x3f3504f3 is sqrt(1/2)); f = m - 1 exactly; log(1 + f) = 2 atanh(s), s = f / (2 + f), arranged as
// f - (f^2/2 - s (f^2/2 + R)) with R = sum_k 2 s^2k / (2k + 1) through k = 5.  s enters only the
// correction term, so 1/(2 + f) comes from the linear minimax seed on [2 - 0.2929, 2 + 0.4143]
// (relative error 1.49e-2) and two Newton steps (5.0e-8) instead of an IEEE divide.  e ln2 is split
// so that e * ln2_hi is exact (15-bit ln2_hi, |e| < 2^9); ln2_lo is the float nearest ln2 - ln2_hi.
// Error: under 0.72 ulp on a sweep of normal floats.
__device__ __forceinline__ float log_f32(float x)
{
    #pragma clang fp contract(off)
    const uint32_t ix = __builtin_bit_cast(uint32_t, x);
    const int32_t e = ((int32_t)(ix - 0x3f3504f3u)) >> 23;
    const float m = __builtin_bit_cast(float, ix - ((uint32_t)e << 23));
    const float f = m - 1.0f;
    const float d = 2.0f + f;
    float y = __builtin_fmaf(d, -0x1.e9813ap-3f, 0x1.f859fcp-1f);
    y = __builtin_fmaf(y, __builtin_fmaf(-d, y, 1.0f), y);
    y = __builtin_fmaf(y, __builtin_fmaf(-d, y, 1.0f), y);
    const float s = f * y;
    const float z = s * s;
    const float R = z * __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, 0x1.745d18p-3f,
                    0x1.c71c72p-3f), 0x1.24924ap-2f), 0x1.99999ap-2f), 0x1.555556p-1f);
    const float hfsq = 0.5f * f * f;
    const float ef = (float)e;
    return __builtin_fmaf(ef, 0x1.62e4p-1f, -((hfsq - __builtin_fmaf(s, hfsq + R, ef * 0x1.7f7d1cp-20f)) - f));
}

__device__ __forceinline__ float gumbel_of_bits(uint32_t b)
{
    #pragma clang fp contract(off)
    const float u = ((float)(b >> 9) + 0.5f) * 1.1920928955078125e-07f;    // 2^-23
    return -log_f32(-log_f32(u));
}

// Noise for columns c .. c+7 of `row`, c a multiple of 4.
__device__ __forceinline__ void gumbel8(uint32_t seed, int64_t row, int64_t c, float (&g)[8])
{
    uint32_t w[4];
    #pragma unroll
    for (int h = 0; h < 2; ++h)
    {
        philox4x32_10((uint32_t)(c >> 2) + h, (uint32_t)row, (uint32_t)((uint64_t)row >> 32), 0u, seed, 0u, w);
        #pragma unroll
        for (int j = 0; j < 4; ++j) g[4 * h + j] = gumbel_of_bits(w[j]);
    }
}

__device__ __forceinline__ float gumbel1(uint32_t seed, int64_t row, int64_t c)
{
    uint32_t w[4];
    philox4x32_10((uint32_t)(c >> 2), (uint32_t)row, (uint32_t)((uint64_t)row >> 32), 0u, seed, 0u, w);
    const int j = (int)(c & 3);
    return gumbel_of_bits(j == 0 ? w[0] : j == 1 ? w[1] : j == 2 ? w[2] : w[3]);
}

// Order-preserving 32-bit image of a float (larger float -> larger key); -0 maps with +0 and every
// NaN to the top key.
__device__ __forceinline__ uint32_t order_key(float v)
{
    if (v != v) return 0xffffffffu;
    const uint32_t u = __builtin_bit_cast(uint32_t, v + 0.0f);   // -0 + +0 = +0
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ uint64_t cand_key(float v, int64_t idx)
{
    return ((uint64_t)order_key(v) << 32) | (uint64_t)(0xffffffffu - (uint32_t)idx);
}

__device__ __forceinline__ uint64_t max_u64(uint64_t a, uint64_t b) { return a > b ? a : b; }

// A lane's running best over candidates seen in increasing index order: a candidate replaces the
// best when none is held yet, when it is larger, or when it is the first NaN (a NaN best is final);
// ties keep the earlier index.  Float compares per element; the 64-bit key is formed once.
struct LaneBest
{
    float v = 0.0f;
    uint32_t i = 0;
    bool has = false;

    __device__ __forceinline__ void consider(float x, int64_t idx)
    {
        const bool take = (!has) | (x > v) | ((x != x) & (v == v));    // no short circuit: selects, no branches
        v = take ? x : v;
        i = take ? (uint32_t)idx : i;
        has = true;
    }
    __device__ __forceinline__ uint64_t key() const { return has ? cand_key(v, i) : 0; }
};

// f16 logits without noise: a lane keeps its best chunk of 8 instead of its best element.  The chunk's
// maximum cm comes from NaN-propagating packed maxima (v_pk_maximum3_f16: a NaN anywhere in the chunk
// makes cm NaN); the chunk replaces the held one when it is the lane's first chunk, when cm is larger
// (-0 and +0 compare equal, so the earlier chunk stays), or when cm is the first NaN (a NaN best is
// final).  The held chunk's data is kept and its element found once at the end: the first one equal
// to the maximum, or the first NaN when the maximum is NaN, which is the element LaneBest keeps over
// the same elements in the same order.  Per 8 elements: 3 maxima, 3 compares and 6 selects instead of
// 8 x LaneBest::consider.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

struct LaneBestF16
{
    _Float16 m = 0;
    uint32_t c = 0;     // first element of the held chunk
    u32x4 d = {};       // its data
    bool has = false;

    // FIRST: the lane's first chunk (taken unconditionally).
    template <bool FIRST>
    __device__ __forceinline__ void consider8(const u32x4& w, uint32_t c0)
    {
        // (uint32_t) casts: the operand of a bit_cast must be a value, not a vector element -- this
        // compiler lowers __builtin_bit_cast of an ext_vector element lvalue as a read of element 0.
        const f16x2 p = __builtin_elementwise_maximum(
            __builtin_elementwise_maximum(__builtin_bit_cast(f16x2, (uint32_t)w[0]), __builtin_bit_cast(f16x2, (uint32_t)w[1])),
            __builtin_elementwise_maximum(__builtin_bit_cast(f16x2, (uint32_t)w[2]), __builtin_bit_cast(f16x2, (uint32_t)w[3])));
        const _Float16 cm = __builtin_elementwise_maximum(p[0], p[1]);
        const bool take = FIRST || (cm > m) || ((cm != cm) & (m == m));
        m = take ? cm : m;
        c = take ? c0 : c;
        #pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = take ? w[q] : d[q];
        has = FIRST || has;
    }

    __device__ __forceinline__ LaneBest lane_best() const
    {
        LaneBest lb;
        int j = 7;
        #pragma unroll
        for (int q = 7; q >= 0; --q)
        {
            const _Float16 x = __builtin_bit_cast(f16x2, (uint32_t)d[q >> 1])[q & 1];
            j = ((x == m) | ((x != x) & (m != m))) ? q : j;
        }
        lb.v = (float)m;
        lb.i = c + (uint32_t)j;
        lb.has = has;
        return lb;
    }
};

template <int CTRL>
__device__ __forceinline__ uint64_t dpp_u64(uint64_t v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, 0xf, 0xf, false);
    return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
}

// Maximum over the wave, valid in lane 0 (and every lane).
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v)
{
    v = max_u64(v, dpp_u64<DPP_QUAD_XOR1>(v));
    v = max_u64(v, dpp_u64<DPP_QUAD_XOR2>(v));
    v = max_u64(v, dpp_u64<DPP_ROW_HALF_MIRROR>(v));
    v = max_u64(v, dpp_u64<DPP_ROW_MIRROR>(v));
    v = max_u64(v, __shfl_xor(v, 16));
    v = max_u64(v, __shfl_xor(v, 32));
    return v;
}

__global__ __launch_bounds__(256) void k_argmax_clear(uint64_t* ids, int64_t rows)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < rows) ids[i] = 0;
}

__global__ __launch_bounds__(256) void k_argmax_convert(uint64_t* ids, int64_t rows)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < rows)
    {
        const uint64_t k = ids[i];
        ids[i] = k ? (uint64_t)(0xffffffffu - (uint32_t)k) : 0;
    }
}

// A whole chunk of 8 logits.  ALIGNED: 16-byte aligned rows; otherwise (an odd vocabulary, a sliced tensor)
// the same 16-byte accesses at the alignment of one element, which the hardware splits where they cross a
// line, in place of 8 single reads and, for a draw, 8 Philox blocks instead of 2 (64 x 151935 f32 logits, us,
// before and after: argmax 24.6 -> 13.6, draw 34.8 -> 15.4).
typedef u32x4 __attribute__((aligned(2))) u32x4_u2;
typedef u32x4 __attribute__((aligned(4))) u32x4_u4;
template <class IT, bool ALIGNED>
__device__ __forceinline__ typename IT::Vec load_chunk(const void* base, int64_t c)
{
    if constexpr (ALIGNED) return load8s<IT>(base, c);
    else if constexpr (IT::code == DT_F32)
    {
        const gcptr<u32x4_u4> p = (gcptr<u32x4_u4>)((const float*)base + c);
        typename IT::Vec v;
        v.a = __builtin_nontemporal_load(p);
        v.b = __builtin_nontemporal_load(p + 1);
        return v;
    }
    else return { __builtin_nontemporal_load((gcptr<u32x4_u2>)((const uint16_t*)base + c)) };
}

// ---------------------------------------------------------------------------------------------
// The Gumbel draw's candidates.  The noise is the cost of a draw: its two logs as log_f32 evaluates them are
// 60 of 80 VALU instructions per element.  Only the winner's noise has to be that exact, so the draw first
// ranks every candidate with the hardware's log2 (v_log_f32), which needs 5 instructions, and then evaluates
// log_f32's noise for the candidates that come within a bound of the best rank, one as a rule.
//
// b = x - ln2 log2(-log2 u) is the candidate x + g less the constant -ln ln 2.  Over all 2^23 values of u
// the noise part differs from g by less than kRankErr (by 1.58e-6 at most: k_rank_error walks them), and forming b and
// x + g rounds each by at most 2^-24 of its size, so with m the largest b, a candidate with
// b < m - (2 kRankErr + 2^-20 |m|) is below the one that has b = m: |b| <= 2 |m| leaves 3 * 2^-23 |m| for the
// roundings, and a larger |b| (b far below m) is more than |b| / 2 away.  The best candidate, and any that
// ties with it, is therefore always evaluated, and the draw is the same index as before.
// Masked logits (top-k, grammar: -inf, the type's lowest value, -1e9) leave most slices without a live candidate,
// and there the noise decides nothing: from |m| = kAbsorbs on, half the spacing of the floats about m (32) is more
// than any noise (-2.9 .. 16.7), so x + g is x for every candidate that can win, and with NaN or +inf about, x + g
// is NaN or +inf where x is.  The slice's draw is then its logits' argmax, the first index where all are -inf.  (us in
// a HIP graph, 16 / 64 rows of 151936 f32 logits, live 9.3 / 14.3, all but 50 columns of a row -inf 9.0 / 14.0, -1e9
// 11.0 / 15.3, a NaN in every row 9.5 / 16.4; one by one with their noise 20.2 / 26.9, 20.2 / 25.1 and 21 / 25.3.)
// 64 rows of 151936 f32 logits took 20.9 us in a HIP graph with every candidate exact, bound by VALU issue, and take
// 14.2; 1024 rows 242 -> 122 us (5.1 TB/s).
constexpr float kRankErr = 1e-5f;
constexpr float kAbsorbs = 0x1.1p29f;

__device__ __forceinline__ float gumbel_rank(float x, uint32_t bits)
{
    // u = ((bits >> 9) + 0.5) 2^-23 exactly: 1.mantissa less 1 - 2^-24
    const float u = __builtin_bit_cast(float, __builtin_amdgcn_alignbit(0x7fu, bits, 9)) - 0x1.fffffep-1f;
    return __builtin_fmaf(__builtin_amdgcn_logf(-__builtin_amdgcn_logf(u)), -0x1.62e43p-1f, x);
}
__device__ __forceinline__ float rank_floor(float m) { return m - __builtin_fmaf(fabsf(m), 0x1p-20f, 2.0f * kRankErr); }
__device__ __forceinline__ float max_nan(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float wave_max_nan(float v)
{
    v = max_nan(v, dpp<DPP_QUAD_XOR1>(v));
    v = max_nan(v, dpp<DPP_QUAD_XOR2>(v));
    v = max_nan(v, dpp<DPP_ROW_HALF_MIRROR>(v));
    v = max_nan(v, dpp<DPP_ROW_MIRROR>(v));
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    v = max_nan(__builtin_bit_cast(float, (uint32_t)p[0]), __builtin_bit_cast(float, (uint32_t)p[1]));
    const uint32_t w = __builtin_bit_cast(uint32_t, v);
    const auto q = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return max_nan(__builtin_bit_cast(float, (uint32_t)q[0]), __builtin_bit_cast(float, (uint32_t)q[1]));
}

#ifdef EXL3R_TUNING
// out[0]: the largest distance of the ranked noise (with the constant -ln ln 2 that it leaves out) from the exact one
// over all 2^23 values of u, a lane each; out[1]: the bound that the draw allows it.
__global__ __launch_bounds__(256) void k_rank_error(float* out)
{
    const uint32_t bits = (blockIdx.x * 256 + threadIdx.x) << 9;
    const double d = (double)gumbel_rank(0.0f, bits) + 0.36651292058166432701 - (double)gumbel_of_bits(bits);
    atomicMax((unsigned*)out, __builtin_bit_cast(uint32_t, (float)fabs(d)));
    if (bits == 0) out[1] = kRankErr;
}
#endif

// The chunk's 8 logits (-inf past the row), from the loaded vector or, for a chunk that crosses n, one by one.
template <class IT>
__device__ __forceinline__ void chunk_logits(const ArgArgs& a, const char* base, const typename IT::Vec& v, int64_t c, float (&x)[8])
{
    if (c + 8 <= a.n) unpack8<IT>(v, x);
    else
    {
        #pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = c + j < a.n ? load1(base, IT::code, c + j) : -INFINITY;
    }
}

__device__ __forceinline__ void chunk_ranks(const float (&x)[8], uint32_t seed, int64_t row, int64_t c, uint32_t (&w)[8],
                                            float (&k)[8])
{
    #pragma unroll
    for (int h = 0; h < 2; ++h)
    {
        uint32_t q[4];
        philox4x32_10((uint32_t)(c >> 2) + h, (uint32_t)row, (uint32_t)((uint64_t)row >> 32), 0u, seed, 0u, q);
        #pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            w[4 * h + j] = q[j];
            k[4 * h + j] = gumbel_rank(x[4 * h + j], q[j]);
        }
    }
}

// The exact candidates of the chunk at c whose rank reaches `floor`, in index order.
template <class IT, bool VEC>
__device__ __forceinline__ void take_chunk(const ArgArgs& a, const char* base, int64_t row, int64_t c, float floor, LaneBest& lb)
{
    #pragma clang fp contract(off)
    typename IT::Vec v{};
    if (c + 8 <= a.n) v = load_chunk<IT, VEC>(base, c);
    float x[8], k[8];
    uint32_t w[8], left = 0;
    chunk_logits<IT>(a, base, v, c, x);
    chunk_ranks(x, a.seed, row, c, w, k);
    #pragma unroll
    for (int j = 0; j < 8; ++j) left |= c + j < a.n && k[j] >= floor ? 1u << j : 0u;
    while (left)
    {
        const int j = __builtin_ctz(left);
        left &= left - 1;
        float xj = x[0];
        uint32_t wj = w[0];
        #pragma unroll
        for (int i = 1; i < 8; ++i)
        {
            xj = j == i ? x[i] : xj;
            wj = j == i ? w[i] : wj;
        }
        lb.consider(xj + gumbel_of_bits(wj), c + j);
    }
}

// One lane's best candidate of the draw over elements [start, end) of `row`, end at most n, by a workgroup of
// THREADS lanes (every lane must get here; wmax: one LDS slot per wave).  A lane walks its chunks start + 8 tid,
// + 8 THREADS, ... keeping the largest chunk rank, that chunk, and the largest rank of its other chunks; the
// workgroup's largest rank then decides which chunk is looked at again.  (As a rolled loop with the next
// chunk's load issued ahead: unrolled four times it holds 140 VGPRs, 3 waves per SIMD.)
template <class IT, bool VEC, int THREADS>
__device__ __forceinline__ uint64_t gumbel_lane_key(const ArgArgs& a, int64_t row, int64_t start, int64_t end, int tid,
                                                    float* wmax)
{
    const char* base = a.x + row * a.ld;
    constexpr int STEP = THREADS * 8;
    float top = -INFINITY, other = -INFINITY;
    int64_t at = start + tid * 8;
    typename IT::Vec v{}, vn{};
    if (at + 8 <= a.n && at < end) v = load_chunk<IT, VEC>(base, at);
    #pragma unroll 1
    for (int64_t c = at; c < end; c += STEP)
    {
        const int64_t cn = c + STEP;
        if (cn + 8 <= a.n && cn < end) vn = load_chunk<IT, VEC>(base, cn);
        float x[8], k[8];
        uint32_t w[8];
        chunk_logits<IT>(a, base, v, c, x);
        chunk_ranks(x, a.seed, row, c, w, k);
        const float m = max_nan(max_nan(max_nan(k[0], k[1]), max_nan(k[2], k[3])), max_nan(max_nan(k[4], k[5]), max_nan(k[6], k[7])));
        other = fmaxf(other, fminf(top, m));
        at = m > top ? c : at;
        top = max_nan(top, m);
        v = vn;
    }
    const float mw = wave_max_nan(top);
    if ((tid & 63) == 0) wmax[tid >> 6] = mw;
    __syncthreads();
    float m = wmax[0];
    #pragma unroll
    for (int i = 1; i < THREADS / 64; ++i) m = max_nan(m, wmax[i]);
    const float floor = rank_floor(m);
    LaneBest lb;
    // (The usual way is laid out first and straight: after the other three, and as a loop, the same code took 0.2 us
    // more per launch, 7.04 against 6.82 for one row of 151936 f32 logits and 9.58 against 9.21 for 16.)
    if (__builtin_expect(fabsf(m) < kAbsorbs && !(other >= floor), 1))
    {
        if (top >= floor) take_chunk<IT, VEC>(a, base, row, at, floor, lb);
    }
    else if (m == -INFINITY)                // nothing but -inf: any noise leaves it, and the first index wins
    {
        if (start + tid * 8 < end) lb.consider(m, start + tid * 8);
    }
    else if (!(fabsf(m) < kAbsorbs))        // the logits decide: NaN, +inf, or too large for the noise to move them
    {
        #pragma unroll 1
        for (int64_t c = start + tid * 8; c < end; c += STEP)
        {
            if (c + 8 <= a.n)
            {
                float x[8];
                unpack8<IT>(load_chunk<IT, VEC>(base, c), x);
                #pragma unroll
                for (int j = 0; j < 8; ++j) lb.consider(x[j], c + j);
            }
            else
            {
                #pragma unroll 1
                for (int j = 0; j < 8 && c + j < end; ++j) lb.consider(load1(base, IT::code, c + j), c + j);
            }
        }
    }
    else                                    // two chunks of the lane come within the bound: each is looked at again
    {
        #pragma unroll 1
        for (int64_t c = start + tid * 8; c < end; c += STEP) take_chunk<IT, VEC>(a, base, row, c, floor, lb);
    }
    return lb.key();
}

// One lane's best candidate over its UNROLL chunks of the slice starting at `start` of `row`.  A chunk crossing
// n is read element by element.  GUMBEL: a slice of one chunk per lane (UNROLL 1) evaluates them all; in a longer
// one (any UNROLL above) the workgroup's largest rank (wmax: one LDS slot per wave) decides which, and every lane of
// the workgroup must get here.
template <class IT, bool VEC, int UNROLL, bool GUMBEL>
__device__ __forceinline__ uint64_t slice_lane_key(const ArgArgs& a, int64_t row, int64_t start, int tid, float* wmax)
{
    const char* base = a.x + row * a.ld;
    LaneBest lb;
    if constexpr (GUMBEL && UNROLL > 1)
    {
        const int64_t end = start + a.slice;
        return gumbel_lane_key<IT, VEC, 256>(a, row, start, end < a.n ? end : a.n, tid, wmax);
    }
    if constexpr (GUMBEL)
    {
        #pragma clang fp contract(off)
        const int64_t c = start + tid * 8;
        if (c >= a.n) return 0;
        typename IT::Vec v{};
        if (c + 8 <= a.n) v = load_chunk<IT, VEC>(base, c);
        float g[8];
        gumbel8(a.seed, row, c, g);
        if (__builtin_expect(c + 8 <= a.n, 1))
        {
            float x[8];
            unpack8<IT>(v, x);
            #pragma unroll
            for (int j = 0; j < 8; ++j) lb.consider(x[j] + g[j], c + j);
        }
        else
        {
            #pragma unroll
            for (int j = 0; j < 7; ++j)
                if (c + j < a.n) lb.consider(load1(base, IT::code, c + j) + g[j], c + j);
        }
        return lb.key();
    }
    typename IT::Vec v[UNROLL];
    #pragma unroll
    for (int u = 0; u < UNROLL; ++u)
    {
        const int64_t c = start + u * 2048 + tid * 8;
        if (c + 8 <= a.n) v[u] = load_chunk<IT, VEC>(base, c);
    }
    if constexpr (IT::code == DT_F16)
    {
        // whole chunks by LaneBestF16 (a chunk is whole only when every earlier one of the lane is)
        LaneBestF16 hb;
        #pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            const int64_t c = start + u * 2048 + tid * 8;
            if (c + 8 <= a.n)
            {
                if (u == 0) hb.consider8<true>(v[u].a, (uint32_t)c);
                else hb.consider8<false>(v[u].a, (uint32_t)c);
            }
        }
        lb = hb.lane_best();
    }
    #pragma unroll
    for (int u = 0; u < UNROLL; ++u)
    {
        const int64_t c = start + u * 2048 + tid * 8;
        if (c + 8 <= a.n)
        {
            if constexpr (IT::code == DT_F16) continue;   // taken above
            float f[8];
            unpack8<IT>(v[u], f);
            #pragma unroll
            for (int j = 0; j < 8; ++j) lb.consider(f[j], c + j);
        }
        else
        {
            for (int j = 0; j < 8 && c + j < a.n; ++j) lb.consider(load1(base, IT::code, c + j), c + j);
        }
    }
    return lb.key();
}

// First element of the workgroup's slice.  Only a draw's longer slices have a length that the kernel does not know:
// with a length from memory the argmax of four chunks per lane needs more than 96 VGPRs, a wave per SIMD less.
template <int UNROLL, bool GUMBEL>
__device__ __forceinline__ int64_t slice_start(const ArgArgs& a)
{
    if constexpr (GUMBEL && UNROLL > 1) return (int64_t)blockIdx.x * a.slice;
    else return (int64_t)blockIdx.x * UNROLL * 2048;
}

// A workgroup of 256 lanes reduces a slice (argmax: UNROLL * 2048 elements, UNROLL chunks of 8 per lane in
// flight) to one key, so a row takes only vocab / slice atomics: same-address atomics from many
// workgroups (and XCDs) serialize.
template <class IT, bool VEC, int UNROLL, bool GUMBEL>
__global__ __launch_bounds__(256) void k_argmax(ArgArgs a)
{
    __shared__ uint64_t part[4];
    __shared__ float wmax[4];
    const int tid = threadIdx.x;
    const int64_t start = slice_start<UNROLL, GUMBEL>(a);
    for (int64_t row = blockIdx.y; row < a.rows; row += gridDim.y)
    {
        uint64_t best = wave_max_u64(slice_lane_key<IT, VEC, UNROLL, GUMBEL>(a, row, start, tid, wmax));
        if ((tid & 63) == 0) part[tid >> 6] = best;
        __syncthreads();
        if (tid == 0)
        {
            best = max_u64(max_u64(part[0], part[1]), max_u64(part[2], part[3]));
            if (best) atomicMax((unsigned long long*)(a.ids + row), (unsigned long long)best);
        }
        __syncthreads();
    }
}

// The same slices in one launch with a workspace (exl3r_argmax_sample_ws, exl3r_gumbel_sample_ws):
// each workgroup folds its slice's key into the row's slot with atomicMax and then counts itself in
// count[row]; the workgroup whose count completes the row takes the slot with an atomic exchange
// (which also resets it to 0), writes the index and resets the count, so the workspace is zero again
// when the launch ends and nothing is cleared per call.  Ordering comes from completion, not fences:
// a workgroup issues its count only after its atomicMax has returned, so every slot update is
// performed before the last count, and the exchange after that (atomics on one address are
// serialized where they are performed, across XCDs too).  (Release / acquire
// fences at device scope write back and invalidate the L2 for every workgroup: 28.8 against 10.2 us
// for the three launches at 64 x 151936.)  No workgroup waits for another.
template <class IT, bool VEC, int UNROLL, bool GUMBEL>
__global__ __launch_bounds__(256) void k_argmax_ws(ArgArgs a, uint32_t* count, uint64_t* slot)
{
    __shared__ uint64_t wpart[4];
    __shared__ float wmax[4];
    const int tid = threadIdx.x;
    const uint32_t slices = gridDim.x;
    const int64_t start = slice_start<UNROLL, GUMBEL>(a);
    for (int64_t row = blockIdx.y; row < a.rows; row += gridDim.y)
    {
        uint64_t best = wave_max_u64(slice_lane_key<IT, VEC, UNROLL, GUMBEL>(a, row, start, tid, wmax));
        if ((tid & 63) == 0) wpart[tid >> 6] = best;
        __syncthreads();
        if (tid == 0)
        {
            best = max_u64(max_u64(wpart[0], wpart[1]), max_u64(wpart[2], wpart[3]));
            // The returning form, its value consumed: the count below is issued only once the slot's
            // update has been performed and answered.
            const unsigned long long prev = atomicMax((unsigned long long*)(slot + row), (unsigned long long)best);
            asm volatile("" : : "v"(prev) : "memory");
            if (atomicAdd(count + row, 1u) + 1 == slices)
            {
                const uint64_t k = atomicExch((unsigned long long*)(slot + row), 0ull);
                a.ids[row] = k ? (uint64_t)(0xffffffffu - (uint32_t)k) : 0;
                atomicExch(count + row, 0u);
            }
        }
        __syncthreads();
    }
}

// Many rows: a workgroup of THREADS lanes owns a row, walks it THREADS * 8 elements per chunk round
// with 4 chunks per lane in flight, and writes the index itself (no atomics, no clear / convert
// launches).
template <class IT, bool VEC, bool GUMBEL, int THREADS>
__global__ __launch_bounds__(THREADS) void k_argmax_rows(ArgArgs a)
{
    constexpr int WAVES = THREADS / 64;
    constexpr int STEP = THREADS * 8;          // elements per chunk round
    __shared__ uint64_t part[WAVES];
    __shared__ float wmax[WAVES];
    const int tid = threadIdx.x;
    for (int64_t row = blockIdx.x; row < a.rows; row += gridDim.x)
    {
        const char* base = a.x + row * a.ld;
        LaneBest lb;
        [[maybe_unused]] uint64_t lane_key = 0;
        if constexpr (GUMBEL)
        {
            lane_key = gumbel_lane_key<IT, VEC, THREADS>(a, row, 0, a.n, tid, wmax);
        }
        else if constexpr (IT::code == DT_F16)
        {
            // whole chunks by LaneBestF16, then the elements of a partial last chunk (after every whole
            // one) by the lane that holds it
            const int64_t nw = a.n & ~(int64_t)7;
            LaneBestF16 hb;
            auto round = [&](int64_t s0, auto FIRST) __attribute__((always_inline)) {
                u32x4 v[4];
                #pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    const int64_t c = s0 + u * STEP + tid * 8;
                    if (c < nw) v[u] = load_chunk<TF16, VEC>(base, c).a;
                }
                #pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    const int64_t c = s0 + u * STEP + tid * 8;
                    if (c < nw)
                    {
                        if (decltype(FIRST)::value && u == 0) hb.consider8<true>(v[u], (uint32_t)c);
                        else hb.consider8<false>(v[u], (uint32_t)c);
                    }
                }
            };
            if (nw > 0) round((int64_t)0, std::true_type{});
            for (int64_t s0 = 4 * STEP; s0 < nw; s0 += 4 * STEP) round(s0, std::false_type{});
            lb = hb.lane_best();
            if (nw < a.n && tid * 8 == nw % STEP)
                for (int64_t c = nw; c < a.n; ++c) lb.consider(load1(base, DT_F16, c), c);
        }
        else for (int64_t s0 = 0; s0 < a.n; s0 += 4 * STEP)
        {
            typename IT::Vec v[4];
            #pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                const int64_t c = s0 + u * STEP + tid * 8;
                if (c + 8 <= a.n) v[u] = load_chunk<IT, VEC>(base, c);
            }
            #pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                const int64_t c = s0 + u * STEP + tid * 8;
                if (c + 8 <= a.n)
                {
                    float f[8];
                    unpack8<IT>(v[u], f);
                    #pragma unroll
                    for (int j = 0; j < 8; ++j) lb.consider(f[j], c + j);
                }
                else
                {
                    for (int j = 0; j < 8 && c + j < a.n; ++j) lb.consider(load1(base, IT::code, c + j), c + j);
                }
            }
        }
        uint64_t best = wave_max_u64(GUMBEL ? lane_key : lb.key());
        if ((tid & 63) == 0) part[tid >> 6] = best;
        __syncthreads();
        if (tid == 0)
        {
            best = part[0];
            #pragma unroll
            for (int w = 1; w < WAVES; ++w) best = max_u64(best, part[w]);
            a.ids[row] = best ? (uint64_t)(0xffffffffu - (uint32_t)best) : 0;
        }
        __syncthreads();
    }
}

// out[r, c] = x[r, c] + g(seed, r, c): a lane per 8 columns (grid (column chunks, rows)).  VEC: 16-byte
// aligned rows of x and out; otherwise element by element.
struct NoiseArgs
{
    const char* x;
    char* out;
    int64_t ldx, ldo;    // bytes
    int64_t rows, cols;
    uint32_t seed;
};

template <class IT, class OT, bool VEC>
__global__ __launch_bounds__(256) void k_gumbel_noise(NoiseArgs a)
{
    #pragma clang fp contract(off)
    const int64_t c = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (c >= a.cols) return;
    for (int64_t row = blockIdx.y; row < a.rows; row += gridDim.y)
    {
        const char* xr = a.x + row * a.ldx;
        char* orow = a.out + row * a.ldo;
        if (VEC && c + 8 <= a.cols)
        {
            float f[8], g[8];
            unpack8<IT>(load8s<IT>(xr, c), f);
            gumbel8(a.seed, row, c, g);
            #pragma unroll
            for (int j = 0; j < 8; ++j) f[j] = f[j] + g[j];
            store8<OT>(orow, c, pack8<OT>(f));
        }
        else
        {
            for (int64_t j = c; j < c + 8 && j < a.cols; ++j)
                store1(orow, OT::code, j, load1(xr, IT::code, j) + gumbel1(a.seed, row, j));
        }
    }
}

}  // namespace exl3r

using namespace exl3r;

// exl3r_argmax_sample_noalloc's scratch: the one-launch kernel's row counters and slots for 384 rows
// (4608 bytes: the workspace of exl3r_argmax_sample_ws), one copy per GPU the library runs on, held
// until the process ends.  It is zero when the code object is loaded, and every completed call leaves
// it zero (the last workgroup of a row resets the row's counter and slot), so no call clears it.  Host
// code never uses the name as an address: scratch_of_current_device() asks the runtime for the
// current device's copy, once per device.
static __device__ __align__(256) unsigned char scratch[384 * 12];

namespace {

// Workspace of the single-launch sliced path: kWsMaxRows row counters (u32), then as many row slots
// (u64), all zero between calls.
constexpr int64_t kWsMaxRows = 384;
constexpr size_t kCountBytes = kWsMaxRows * 4;
constexpr size_t kWsBytes = kCountBytes + kWsMaxRows * 8;

// Elements per slice of the sliced kernels: 8192 (19 slices per 152k-token row); decode batches of a
// few rows take 2048-element slices so the row still spreads over enough CUs.
inline int slice_unroll(int64_t rows) { return rows >= 16 ? 4 : 1; }

// Chunks of 8 logits per lane of a draw's slices.  A slice costs its workgroup a reduction, the winner's evaluation
// and an atomic on the row's word, so slices are long, up to 10240 elements, while they leave half the CUs a
// workgroup.  One chunk per lane evaluates its candidates as they come: ranking them first costs a small draw a second
// read of the winner's chunk (1 row of 32000 f32 logits 6.47 us ranked, 6.26 as they come).  MI355X, HIP graph, f32,
// us for 1 / 2 / 3 / 4 / 5 / 6 / 8 chunks (1: as they come), three launches:
//     1 x 151936   6.84 / 6.97 / 7.32 / 7.80 / 8.20 / 8.61 / 9.40
//     8 x 151936  13.25 / 9.85 / 9.14 / 9.09 / 9.55 / 10.3 / 11.3
//    16 x 32000    7.75 / 7.31 / 7.52 / 7.94 / 8.70 / 9.08 / 10.9
//    16 x 151936  16.4 / 11.5 / 10.2 / 10.6 / 10.1 / 10.6 / 11.7
//    64 x 32000   10.6 / 8.63 / 9.09 / 9.04 / 9.66 / 10.4 / 11.8
//    64 x 151936  28.8 / 19.1 / 16.2 / 15.5 / 15.0 / 16.0 / 15.6
//   256 x 151936  66.6 / 42.4 / 37.0 / 35.6 / 35.6 / 36.4 / 37.1
// Over 1 to 383 rows of 32000 to 262144 logits, f16 and f32, with and without the workspace, it is 4% from the best
// of them on average, 24% at most (one slice of a few elements left over; few rows in the workspace); 2048-element
// slices below 16 rows and 10240 from there on were 13%, 150% at most.
inline int draw_chunks(int64_t n, int64_t rows)
{
    for (int k = 5; k > 1; --k)
        if (rows * ((n + k * 2048 - 1) / (k * 2048)) >= device_cus() / 2) return k;
    return 1;
}

struct Workspace
{
    void* base;      // nullptr: the three-launch path (ids as the reduction slot)
    size_t bytes;
    bool scratch;    // the library's scratch (looked up when the sliced kernel needs it); a call it cannot
                     // serve is an error, not the three-launch path
};

static_assert(sizeof(scratch) == kWsBytes, "the scratch is one workspace");

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The current device's scratch address: hipGetSymbolAddress on the first call with that device
// current, kept per device.
int scratch_of_current_device(const char* op, void** out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return set_error((int)e, "%s: hipGetDevice: %s", op, hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices)
        return set_error(EXL3R_EINVAL, "%s: device %d is beyond the %d devices this entry point serves", op, dev,
                         kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev])
    {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return set_error(e != hipSuccess ? (int)e : (int)hipErrorInvalidSymbol, "%s: hipGetSymbolAddress(scratch): %s",
                             op, hipGetErrorString(e != hipSuccess ? e : hipErrorInvalidSymbol));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return EXL3R_OK;
}

// Shared by the argmax and the Gumbel draw: validation, then the slice or row-per-workgroup kernels.
template <bool GUMBEL>
int sample_entry(const char* op, const void* logits, int dtype, int64_t rows, int64_t vocab, int64_t ld,
                 int max_logit, uint32_t seed, int64_t* ids, void* stream, Workspace ws = { nullptr, 0, false })
{

    if (!is_float_dtype(dtype)) return set_error(EXL3R_EDTYPE, "%s: unsupported logits dtype %s", op, dtype_name(dtype));
    if (rows < 0 || vocab <= 0 || vocab > 0xffffffffLL || (rows > 1 && ld < vocab))
        return set_error(EXL3R_EINVAL, "%s: invalid shape rows=%lld vocab=%lld ld=%lld", op, (long long)rows,
                         (long long)vocab, (long long)ld);
    if (rows == 0) return EXL3R_OK;
    if (!logits || !ids) return set_error(EXL3R_EINVAL, "%s: logits and ids must be non-null", op);
    const int64_t n = (max_logit <= 0 || max_logit > vocab) ? vocab : max_logit;
    const int es = dtype_bytes(dtype);
    ArgArgs a{ (const char*)logits, (rows > 1 ? ld : vocab) * es, n, rows, (uint64_t*)ids, seed, 0 };
    hipStream_t s = (hipStream_t)stream;
    const bool vec = aligned16(logits) && a.ld % 16 == 0;
    // Measured on MI355X over f16 [rows, 151936] logits (us; sliced / a workgroup per row with 512 /
    // 1024 lanes): argmax 64 rows 11.2 / 25.0 / 16.4, 128 rows 16.8 / 25.7 / 17.0, 192 rows 21.8 /
    // 26.3 / 17.4, 512 rows - / 32.0 / 33.5 (256 lanes 57.0), 1024 rows - / 62.3 / 64.5.  The Gumbel draw keeps
    // the sliced kernel longer (f16: 383 rows sliced 44.6, 400 rows by rows 55.3, 1024 rows 96.2; f32 48.8 /
    // 54.4 / 122.5, when every candidate was evaluated exactly 121.5 / 227.7 and 119.8 / 247.1 at 400 / 1024),
    // up to the rows that the workspace holds.
    const Tuning& tu = tuning();
    const int64_t rows_min = tu.sample_rows_min > 0 ? tu.sample_rows_min : GUMBEL ? 384 : 128;
    if (rows >= rows_min)
    {
        const unsigned grid = (unsigned)(rows < kMaxGridX ? rows : kMaxGridX);
        int threads = GUMBEL || rows >= 512 ? 512 : 1024;
        if (tu.sample_threads == 256 || tu.sample_threads == 512 || tu.sample_threads == 1024) threads = tu.sample_threads;
        with_float_type(dtype, [&](auto T) {
            using Ty = decltype(T);
            if (threads == 1024)
            {
                if (vec) launch(k_argmax_rows<Ty, true, GUMBEL, 1024>, grid, 1024, 0, s, a);
                else launch(k_argmax_rows<Ty, false, GUMBEL, 1024>, grid, 1024, 0, s, a);
            }
            else if (threads == 512)
            {
                if (vec) launch(k_argmax_rows<Ty, true, GUMBEL, 512>, grid, 512, 0, s, a);
                else launch(k_argmax_rows<Ty, false, GUMBEL, 512>, grid, 512, 0, s, a);
            }
            else
            {
                if (vec) launch(k_argmax_rows<Ty, true, GUMBEL, 256>, grid, 256, 0, s, a);
                else launch(k_argmax_rows<Ty, false, GUMBEL, 256>, grid, 256, 0, s, a);
            }
        });
        return launch_status(op);
    }
    int unroll = slice_unroll(rows);
    if (GUMBEL) unroll = tu.sample_slice > 0 ? tu.sample_slice : draw_chunks(n, rows);
    const int64_t slice = (int64_t)unroll * 2048;
    a.slice = slice;
    const dim3 grid((unsigned)((n + slice - 1) / slice), (unsigned)rows);
    if (ws.scratch)
    {
        if (rows > kWsMaxRows)
            return set_error(EXL3R_EINVAL, "%s: %lld rows take the sliced kernel, whose scratch holds %lld rows", op,
                             (long long)rows, (long long)kWsMaxRows);
        const int rc = scratch_of_current_device(op, &ws.base);
        if (rc) return rc;
    }
    if (ws.base && rows <= kWsMaxRows)
    {
        // One launch: the slice keys and row counters in the workspace.
        if (((uintptr_t)ws.base & 255) || ws.bytes < kWsBytes)
            return set_error(EXL3R_EINVAL, "%s: the workspace must be 256-byte aligned and hold %zu bytes (%zu given)",
                             op, kWsBytes, ws.bytes);
        uint32_t* count = (uint32_t*)ws.base;
        uint64_t* part = (uint64_t*)((char*)ws.base + kCountBytes);
        with_float_type(dtype, [&](auto T) {
            using Ty = decltype(T);
            if (unroll > 1)
            {
                if (vec) launch(k_argmax_ws<Ty, true, 4, GUMBEL>, grid, 256, 0, s, a, count, part);
                else launch(k_argmax_ws<Ty, false, 4, GUMBEL>, grid, 256, 0, s, a, count, part);
            }
            else
            {
                if (vec) launch(k_argmax_ws<Ty, true, 1, GUMBEL>, grid, 256, 0, s, a, count, part);
                else launch(k_argmax_ws<Ty, false, 1, GUMBEL>, grid, 256, 0, s, a, count, part);
            }
        });
        return launch_status(op);
    }
    const unsigned small = (unsigned)((rows + 255) / 256);
    launch(k_argmax_clear, small, 256, 0, s, a.ids, rows);
    with_float_type(dtype, [&](auto T) {
        using Ty = decltype(T);
        if (unroll > 1)
        {
            if (vec) launch(k_argmax<Ty, true, 4, GUMBEL>, grid, 256, 0, s, a);
            else launch(k_argmax<Ty, false, 4, GUMBEL>, grid, 256, 0, s, a);
        }
        else
        {
            if (vec) launch(k_argmax<Ty, true, 1, GUMBEL>, grid, 256, 0, s, a);
            else launch(k_argmax<Ty, false, 1, GUMBEL>, grid, 256, 0, s, a);
        }
    });
    launch(k_argmax_convert, small, 256, 0, s, a.ids, rows);
    return launch_status(op);
}

}  // namespace

#ifdef EXL3R_TUNING
extern "C" int exl3r_tune_gumbel_rank_error(float* out, void* stream)
{
    begin_call();
    launch(k_argmax_clear, 1, 256, 0, (hipStream_t)stream, (uint64_t*)out, 1);
    launch(k_rank_error, (1u << 23) / 256, 256, 0, (hipStream_t)stream, out);
    return launch_status("exl3r_tune_gumbel_rank_error");
}
#endif

extern "C" int exl3r_argmax_sample_noalloc(const void* logits, int dtype, int64_t rows, int64_t vocab, int64_t ld,
                                           int max_logit, int64_t* ids, void* stream)
{
    begin_call();
    const char* op = "exl3r_argmax_sample_noalloc";
    return sample_entry<false>(op, logits, dtype, rows, vocab, ld, max_logit, 0u, ids, stream, { nullptr, kWsBytes, true });
}

extern "C" int exl3r_argmax_sample(const void* logits, int dtype, int64_t rows, int64_t vocab, int64_t ld,
                                   int max_logit, int64_t* ids, void* stream)
{
    begin_call();
    return sample_entry<false>("exl3r_argmax_sample", logits, dtype, rows, vocab, ld, max_logit, 0u, ids, stream);
}

extern "C" size_t exl3r_sample_workspace_bytes(void) { return kWsBytes; }

extern "C" int exl3r_argmax_sample_ws(const void* logits, int dtype, int64_t rows, int64_t vocab, int64_t ld,
                                      int max_logit, int64_t* ids, void* workspace, size_t workspace_bytes,
                                      void* stream)
{
    begin_call();
    if (!workspace) return set_error(EXL3R_EINVAL, "exl3r_argmax_sample_ws: workspace must be non-null");
    return sample_entry<false>("exl3r_argmax_sample_ws", logits, dtype, rows, vocab, ld, max_logit, 0u, ids, stream,
                               { workspace, workspace_bytes, false });
}

extern "C" int exl3r_gumbel_sample_ws(const void* logits, int dtype, int64_t rows, int64_t vocab, int64_t ld,
                                      int max_logit, uint32_t random, int64_t* ids, void* workspace,
                                      size_t workspace_bytes, void* stream)
{
    begin_call();
    if (!workspace) return set_error(EXL3R_EINVAL, "exl3r_gumbel_sample_ws: workspace must be non-null");
    return sample_entry<true>("exl3r_gumbel_sample_ws", logits, dtype, rows, vocab, ld, max_logit, random, ids,
                              stream, { workspace, workspace_bytes, false });
}

extern "C" int exl3r_gumbel_sample(const void* logits, int dtype, int64_t rows, int64_t vocab, int64_t ld,
                                   int max_logit, uint32_t random, int64_t* ids, void* stream)
{
    begin_call();
    return sample_entry<true>("exl3r_gumbel_sample", logits, dtype, rows, vocab, ld, max_logit, random, ids, stream);
}

extern "C" int exl3r_gumbel_noise(const void* x, int x_dtype, int64_t ldx, void* out, int out_dtype, int64_t ldo,
                                  int64_t rows, int64_t cols, uint32_t random, void* stream)
{
    begin_call();
    const char* op = "exl3r_gumbel_noise";
    if (!is_float_dtype(x_dtype) || !is_float_dtype(out_dtype))
        return set_error(EXL3R_EDTYPE, "%s: unsupported dtypes x=%s out=%s", op, dtype_name(x_dtype),
                         dtype_name(out_dtype));
    if (rows < 0 || cols < 0 || cols > 0xffffffffLL * 4 || (rows > 1 && (ldx < cols || ldo < cols)))
        return set_error(EXL3R_EINVAL, "%s: invalid shape rows=%lld cols=%lld ldx=%lld ldo=%lld", op, (long long)rows,
                         (long long)cols, (long long)ldx, (long long)ldo);
    if (rows == 0 || cols == 0) return EXL3R_OK;
    if (!x || !out) return set_error(EXL3R_EINVAL, "%s: x and out must be non-null", op);
    const int xs = dtype_bytes(x_dtype), os = dtype_bytes(out_dtype);
    NoiseArgs a{ (const char*)x, (char*)out, (rows > 1 ? ldx : cols) * xs, (rows > 1 ? ldo : cols) * os, rows, cols,
                 random };
    const bool vec = aligned16(x) && aligned16(out) && a.ldx % 16 == 0 && a.ldo % 16 == 0;
    const dim3 grid((unsigned)((cols + 2047) / 2048), (unsigned)(rows < 65535 ? rows : 65535));
    hipStream_t s = (hipStream_t)stream;
    with_float_type(x_dtype, [&](auto TI) {
        with_float_type(out_dtype, [&](auto TO) {
            if (vec) launch(k_gumbel_noise<decltype(TI), decltype(TO), true>, grid, 256, 0, s, a);
            else launch(k_gumbel_noise<decltype(TI), decltype(TO), false>, grid, 256, 0, s, a);
        });
    });
    return launch_status(op);
}
