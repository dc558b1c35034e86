// Index-build producer: the unit vectors, balanced cosine bisection and page
// assembly that turn a 1024-token bucket (16 native pages) into the permuted
// pages, member map and FP8 centers the query path reads.
//
// Semantics: sglang/srt/layers/attention/v1_deepseek/kernels.py:9-54
// (initialize, assemble), sglang/srt/layers/attention/v1_native/
// fused_grouping.py:38-61 (_dots, _anchor; _sort lives in sort64.hip / the
// group sort), chain order runtime.py:171-216.
//
// Arithmetic (this build's contract; the reference's Triton reductions have no
// specified order): every 128-wide fp32 sum keeps four partial sums over dims
// d = r (mod 4), each in ascending d with one rounding per product and per
// addition (no fused multiply-add), then (p0 + p1) + (p2 + p3).  Unit vectors
// follow kernels.py:17-28: x_d = fl(c_d * s), m = max(sqrt(sum x_d^2), 1e-12),
// u_d = fl(x_d / m), c_d the FP8 key and s its scale.  Center means add the 8
// members in order, times 1/8.
//
// Two forms: per-kernel drop-ins with the reference's launch shapes, and three
// launches that build a batch of buckets (thread = position in the order):
// build_top_kernel takes a bucket through the groups of 1024 and, launched
// again, of 512 with the tokens' FP8 keys in registers, build_quarter_kernel a
// quarter of it through the groups of 256 to 16 with their unit vectors there
// (and build_write_kernel writes outputs that lie over the pool).  An argmin winner
// stages its vector in LDS, each group is sorted by a bitonic network over its
// unique (score, -position) words, and members move through LDS or lane
// permutes.
//
// Bound by vector issue: 21 dots of 1024 x 128 terms per bucket, each product
// and each sum rounded on its own (no FMA, no matrix core can follow that
// order).  A unit component takes 4.5 operations from its FP8 byte, so the
// lower levels keep the components (128 registers a token, which is why a
// work-group is a quarter: three share a CU) and a term of a dot costs its
// product and its sum; the anchor's components come by DPP row broadcast as
// an operand of the product, from 8 registers a lane.  2048 buckets take 695-712
// us (under the profiler, which slows them, 164 + 131 + 464; one launch with
// every component made anew for every dot 1266), four 63.6 us (24 + 14 + 26;
// 155); the vector units issue 94-96% of the time.
#include <type_traits>

#include "common.h"

// No contraction in this file: every product and every sum written here rounds
// on its own (plain operators: the header's __f*_rn helpers are compiled with
// contraction on and fuse once inlined), and sqrtf / division are correctly
// rounded with the HIP defaults.
#pragma clang fp contract(off)

namespace v1 {
namespace {

constexpr int kTokens = 1024;
constexpr int kWords = 32;                      // 128 FP8 bytes per token
constexpr int kPageWords = V1_PAGE_BYTES / 4;   // 2112
constexpr int kScaleWord = 2048;                // first scale word of a page

// FP8 byte r (0..3) of a packed word, as fp32 (exact).
template <int R>
__device__ __forceinline__ float fp8_at(uint32_t w) {
    return __builtin_amdgcn_cvt_f32_fp8((int)w, R);
}

// The four-partial 128-wide sum.
struct Acc4 {
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    __device__ __forceinline__ void add(float p0, float p1, float p2, float p3) {
        a0 = (a0 + p0);
        a1 = (a1 + p1);
        a2 = (a2 + p2);
        a3 = (a3 + p3);
    }
    __device__ __forceinline__ float total() const { return ((a0 + a1) + (a2 + a3)); }
};

// Divisor m of a token's unit vector: max(||x||, 1e-12), x_d = c_d * s.
__device__ __forceinline__ float unit_norm(const uint32_t (&c)[kWords], float s) {
    Acc4 acc;
#pragma unroll
    for (int w = 0; w < kWords; ++w) {
        const float x0 = (fp8_at<0>(c[w]) * s), x1 = (fp8_at<1>(c[w]) * s);
        const float x2 = (fp8_at<2>(c[w]) * s), x3 = (fp8_at<3>(c[w]) * s);
        acc.add((x0 * x0), (x1 * x1), (x2 * x2), (x3 * x3));
    }
    return fmaxf(sqrtf(acc.total()), 1e-12f);
}

// fl(x / m) from r = fl(1 / m): q0 = fl(x * r), then one correction with the
// exact residual x - q0 * m (an FMA).  With a correctly rounded reciprocal the
// corrected quotient is the correctly rounded one (Markstein's division
// theorem; checked against the division on 3.9e8 x = fp8 * s, m >= |x| pairs,
// significands of m all ones and near powers of two included).  x = -0 gives
// +0 where the division gives -0: the dots cannot tell, every partial sum
// starts at +0.
__device__ __forceinline__ float unit_div(float x, float m, float r) {
    const float q0 = x * r;
    return __builtin_fmaf(__builtin_fmaf(-q0, m, x), r, q0);
}

// Where a token's scale s is a power of two (the format's own scales are),
// x = c s is exact and x / m = c / (m / s), so its components are quotients of
// 4-bit significands: fl(c / d) = fl(c h + fl(c l)) with h = fl(1 / d) and
// l = fl((1 - h d) / d), two operations instead of four.  Checked against the
// division for all 8 significands and all 2^23 significands of d; within the
// exponents allowed here no step leaves the normal range.  (With l = e h in
// place of e / d, 9 of the 67 million pairs differ.)
__device__ __forceinline__ bool short_units(float s) {
    const uint32_t bits = __float_as_uint(s);
    return (bits & 0x807fffffu) == 0 && bits >= (127u - 40u) << 23 && bits <= (127u + 40u) << 23;
}

struct Recip {
    float h, l;  // of d = m / s
};

__device__ __forceinline__ Recip unit_recip(float s, float m, float rm) {
    return {rm * s, (__builtin_fmaf(-rm, m, 1.0f) / m) * s};
}

__device__ __forceinline__ float unit_short(float c, Recip r) { return __builtin_fmaf(c, r.h, c * r.l); }

__device__ __forceinline__ void load_key(const uint8_t* row, uint32_t (&c)[kWords]) {
    const uint4* src = reinterpret_cast<const uint4*>(row);
#pragma unroll
    for (int i = 0; i < kWords / 4; ++i) {
        const uint4 v = src[i];
        c[4 * i] = v.x;
        c[4 * i + 1] = v.y;
        c[4 * i + 2] = v.z;
        c[4 * i + 3] = v.w;
    }
}

// Power of two >= fl(max(amax, 1e-4) / 448): the smallest such.
__device__ __forceinline__ float center_scale(float amax) {
    const float v = fmaxf(amax, 1e-4f) / 448.0f;
    int e;
    const float m = frexpf(v, &e);
    return __builtin_ldexpf(1.0f, m == 0.5f ? e - 1 : e);
}

// ------------------------------------------------------------ drop-ins
// kernels.py:9-30: 16 tokens per program.
__global__ __launch_bounds__(64) void initialize_kernel(const uint8_t* __restrict__ K, const float* __restrict__ KS,
                                                        const int32_t* __restrict__ table, const int32_t* meta,
                                                        float* __restrict__ unit, int32_t* __restrict__ perm,
                                                        int32_t* flag) {
    const int32_t active = meta[2];
    if (blockIdx.x == 0 && threadIdx.x == 0) *flag = active != 0 ? -1 : 0;
    if (!active || threadIdx.x >= 16) return;
    const int32_t i = blockIdx.x * 16 + threadIdx.x;
    const int64_t page = table[i / 64];
    const int32_t slot = i % 64;
    uint32_t c[kWords];
    load_key(K + page * V1_PAGE_BYTES + slot * 128, c);
    const float s = KS[page * kPageWords + kScaleWord + slot];
    const float m = unit_norm(c, s);
    float4* dst = reinterpret_cast<float4*>(unit + (int64_t)i * 128);
#pragma unroll
    for (int w = 0; w < kWords; ++w)
        dst[w] = make_float4((fp8_at<0>(c[w]) * s) / m, (fp8_at<1>(c[w]) * s) / m,
                             (fp8_at<2>(c[w]) * s) / m, (fp8_at<3>(c[w]) * s) / m);
    perm[i] = i;
}

// fused_grouping.py:38-52: 16 positions per program, head = blockIdx.y.
__global__ __launch_bounds__(64) void dots_kernel(const float* __restrict__ U, const int32_t* __restrict__ P,
                                                  const int32_t* __restrict__ A, float* S, const int32_t* flag,
                                                  int32_t N, int32_t start, int32_t mode) {
    if (*flag >= 0 || threadIdx.x >= 16) return;
    const int32_t i = blockIdx.x * 16 + threadIdx.x, h = blockIdx.y;
    const int32_t group = i / N;
    const int64_t id = P[h * 4096 + i] - start;
    const int64_t anchor = (mode == 0 ? P[h * 4096 + group * N] : A[(h * 256 + group) * 2 + (mode - 1)]) - start;
    const float4* x = reinterpret_cast<const float4*>(U + ((int64_t)h * 4096 + id) * 128);
    const float4* y = reinterpret_cast<const float4*>(U + ((int64_t)h * 4096 + anchor) * 128);
    Acc4 acc;
#pragma unroll 8
    for (int w = 0; w < kWords; ++w) {
        const float4 a = x[w], b = y[w];
        acc.add((a.x * b.x), (a.y * b.y), (a.z * b.z), (a.w * b.w));
    }
    float value = acc.total();
    if (mode == 2) value = (value - S[h * 4096 + i]);
    S[h * 4096 + i] = value;
}

// Minimum of (ascending score key, position) words over a block.
__device__ __forceinline__ uint64_t umin64(uint64_t a, uint64_t b) { return a < b ? a : b; }

__device__ __forceinline__ uint64_t shfl_xor64(uint64_t v, int off) {
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, off, kWave);
    const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), off, kWave);
    return ((uint64_t)hi << 32) | lo;
}

// fused_grouping.py:54-61: one 256-thread program per (group, head).
__global__ __launch_bounds__(256) void anchor_kernel(const int32_t* __restrict__ P, int32_t* A,
                                                     const float* __restrict__ S, const int32_t* flag, int32_t N,
                                                     int32_t slot) {
    __shared__ unsigned long long best;
    if (*flag >= 0) return;
    const int32_t group = blockIdx.x, h = blockIdx.y;
    if (threadIdx.x == 0) best = ~0ull;
    __syncthreads();
    uint64_t k = ~0ull;
    for (int32_t i = threadIdx.x; i < N; i += blockDim.x)
        k = umin64(k, ((uint64_t)score_key(S[h * 4096 + group * N + i]) << 32) | (uint32_t)i);
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) k = umin64(k, shfl_xor64(k, off));
    if (__lane_id() == 0) atomicMin(&best, (unsigned long long)k);
    __syncthreads();
    if (threadIdx.x == 0) A[(h * 256 + group) * 2 + slot] = P[h * 4096 + group * N + (int32_t)(uint32_t)best];
}

// kernels.py:33-54: program (page, g) handles members g*8 .. g*8+7 of page,
// one thread per dim.
__global__ __launch_bounds__(128) void assemble_kernel(const uint8_t* __restrict__ K, const float* __restrict__ KS,
                                                       const int32_t* __restrict__ table, const int32_t* meta,
                                                       const int32_t* __restrict__ ids, uint8_t* tmp, float* tmps,
                                                       uint8_t* centers, float* cs, int32_t* map) {
    __shared__ float red[2];
    if (!meta[2]) return;
    const int32_t page = blockIdx.x, g = blockIdx.y, d = threadIdx.x;
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int32_t i = g * 8 + j;
        const int32_t src = ids[page * 64 + i];
        const int64_t native = table[src / 64];
        const uint8_t code = K[native * V1_PAGE_BYTES + (src % 64) * 128 + d];
        const float scale = KS[native * kPageWords + kScaleWord + src % 64];
        tmp[(int64_t)page * V1_PAGE_BYTES + i * 128 + d] = code;
        if (d == 0) {
            tmps[(int64_t)page * kPageWords + kScaleWord + i] = scale;
            map[page * 64 + i] = meta[0] + src;
        }
        const float x = (__builtin_amdgcn_cvt_f32_fp8((int)code, 0) * scale);
        acc = j == 0 ? x : (acc + x);
    }
    const float mean = (acc * 0.125f);
    float amax = fabsf(mean);
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off, kWave));
    if (__lane_id() == 0) red[d / kWave] = amax;
    __syncthreads();
    const float scale = center_scale(fmaxf(red[0], red[1]));
    const int32_t c = page * 8 + g;
    centers[(int64_t)(c / 64) * V1_PAGE_BYTES + (c % 64) * 128 + d] = (uint8_t)e4m3_code(mean / scale);
    if (d == 0) cs[(int64_t)(c / 64) * kPageWords + kScaleWord + c % 64] = scale;
}

// ------------------------------------------------------------- fused
constexpr int kQuarter = 256;  // tokens of a quarter bucket

// A position's token (of the bucket) and its unit divisor between the launches,
// in memory that the last one writes: a quarter's part is written by the
// quarter's own work-group, after it has read it.
struct Carry {
    int32_t* tok;
    float* m;
    int64_t bucket;   // words from a bucket to the next
    int32_t quarter;  // and from a quarter to the next
    __device__ int64_t at(int64_t b, int32_t pos) const {
        return b * bucket + pos / kQuarter * quarter + pos % kQuarter;
    }
};

// FP8 bytes 2H and 2H+1 of a packed word, as fp32 (exact).
template <bool H>
__device__ __forceinline__ float2 fp8_pair(uint32_t w) {
    const auto v = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, H);
    return make_float2(v[0], v[1]);
}

// Lane p ^ J's value (J < 64, every lane active): DPP quad permutes and a
// row rotate for 1, 2 and 8, swizzle bit masks for 4 and 16, a permute for 32.
template <int J>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
    if constexpr (J == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false);
    else if constexpr (J == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false);
    else if constexpr (J == 8) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, false);
    else if constexpr (J == 4 || J == 16) return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (J << 10) | 0x1F);
    else return (uint32_t)__shfl_xor((int)v, J, kWave);
}

template <int J>
__device__ __forceinline__ uint64_t lane_xor64(uint64_t v) {
    return ((uint64_t)lane_xor<J>((uint32_t)(v >> 32)) << 32) | lane_xor<J>((uint32_t)v);
}

// Lanes (of 64) whose bit J is clear, and those that keep the larger key of
// the pair (lane, lane ^ J) while runs of S lanes sort in turn down and up.
constexpr uint64_t lanes_without(int J) {
    uint64_t m = 0;
    for (int l = 0; l < kWave; ++l)
        if ((l & J) == 0) m |= 1ull << l;
    return m;
}

// One compare-exchange step of a descending bitonic network over groups of
// N (i = position in the group, partner i ^ J, merge size S).  Keys of a
// group are distinct, so one compare decides: keep the partner's key when it
// is the larger and this position keeps the maximum, or the smaller and it
// keeps the minimum.  Which positions keep the maximum is a constant lane
// mask, but for strides and runs of whole waves, where it is one bit of the
// wave's number: five vector operations a step.
template <int N, int S, int J, int T>
__device__ __forceinline__ uint64_t bitonic_step(uint64_t key, int32_t p, int32_t wave, uint64_t (*buf)[T], int32_t& nb) {
    uint64_t other, keep_max;
    if constexpr (J >= kWave) {
        buf[nb][p] = key;
        __syncthreads();
        other = buf[nb][p ^ J];
        nb ^= 1;
        const bool low = ((wave * kWave) & J) == 0, down = S == N || ((wave * kWave) & S) == 0;
        keep_max = low == down ? ~0ull : 0ull;
    } else {
        other = lane_xor64<J>(key);
        if constexpr (S == N) keep_max = lanes_without(J);
        else if constexpr (S < kWave) keep_max = ~(lanes_without(J) ^ lanes_without(S));
        else keep_max = ((wave * kWave) & S) == 0 ? lanes_without(J) : ~lanes_without(J);
    }
    const uint64_t larger = __builtin_amdgcn_ballot_w64(other > key);
    return __builtin_amdgcn_inverse_ballot_w64(~(larger ^ keep_max)) ? other : key;
}

template <int N, int S, int J, int T>
__device__ __forceinline__ uint64_t bitonic_merge(uint64_t key, int32_t p, int32_t wave, uint64_t (*buf)[T], int32_t& nb) {
    key = bitonic_step<N, S, J>(key, p, wave, buf, nb);
    if constexpr (J > 1) key = bitonic_merge<N, S, J / 2>(key, p, wave, buf, nb);
    return key;
}

// Descending sort of every aligned group of N keys (unique); strides of a
// wave or more exchange through buf (double-buffered, barriers between).
template <int N, int S = 2, int T>
__device__ __forceinline__ uint64_t bitonic_sort(uint64_t key, int32_t p, int32_t wave, uint64_t (*buf)[T], int32_t& nb) {
    key = bitonic_merge<N, S, S / 2>(key, p, wave, buf, nb);
    if constexpr (S < N) key = bitonic_sort<N, S * 2>(key, p, wave, buf, nb);
    return key;
}

// Minimum of (ascending score, position) words over the `width` lanes that
// share a group (16, 32 or 64), in every lane.
__device__ __forceinline__ uint64_t lanes_min(uint64_t k, int32_t width) {
    k = umin64(k, lane_xor64<1>(k));
    k = umin64(k, lane_xor64<2>(k));
    k = umin64(k, lane_xor64<4>(k));
    k = umin64(k, lane_xor64<8>(k));
    if (width > 16) k = umin64(k, lane_xor64<16>(k));
    if (width > 32) k = umin64(k, lane_xor64<32>(k));
    return k;
}

// Component 16 J + I of the anchor that the lanes of a row share: lane I of
// the row holds it in a[J].
template <int I>
__device__ __forceinline__ float row_bcast(float a) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(a), 0x150 + I, 0xF, 0xF, true));
}

// acc += unit components u0 .. u3 (dims 4 W .. 4 W + 3) times the anchor's.
template <int W>
__device__ __forceinline__ void add_terms(Acc4& acc, const float (&a)[8], float u0, float u1, float u2, float u3) {
    constexpr int I = 4 * (W & 3), J = W >> 2;
    acc.add(row_bcast<I>(a[J]) * u0, row_bcast<I + 1>(a[J]) * u1, row_bcast<I + 2>(a[J]) * u2,
            row_bcast<I + 3>(a[J]) * u3);
    __builtin_amdgcn_sched_barrier(0);  // (products made ahead of their sums would need registers of their own)
}

// Page of token t of a bucket (ids outside the pool read page 0).
__device__ __forceinline__ int64_t page_of(const int32_t* table, int32_t t, int64_t pool_pages) {
    const int64_t page = table[t / 64];
    return (uint64_t)page < (uint64_t)pool_pages ? page : 0;
}

// ---- groups of 1024 and 512: one group per work-group, keys in registers
// A token's FP8 key, scale and unit divisor, staged for the lanes that expand it.
struct Stage {
    uint32_t c[kWords];
    float s, m, rm;
};

template <int N>
struct TopSmem {
    Stage first;                   // the group's first member
    Stage win[2][N / kWave];       // each wave's argmin of the first and second dot
    unsigned long long amin[2];    // the group's argmin words
    uint64_t k[2][N];              // sort keys crossing waves, double-buffered
    float m[N];                    // unit divisors
    int32_t tok[N];
};

template <bool SHORT, int W = 0>
__device__ __forceinline__ void dot_keys(Acc4& acc, const float (&a)[8], const uint32_t (&c)[kWords], float s, float m,
                                         float rm, Recip r) {
    uint32_t cw = c[W];
    asm volatile("" : "+v"(cw));  // recomputed per dot: kept, the components would need 128 more registers
    const float2 lo = fp8_pair<false>(cw), hi = fp8_pair<true>(cw);
    if constexpr (SHORT)
        add_terms<W>(acc, a, unit_short(lo.x, r), unit_short(lo.y, r), unit_short(hi.x, r), unit_short(hi.y, r));
    else
        add_terms<W>(acc, a, unit_div(lo.x * s, m, rm), unit_div(lo.y * s, m, rm), unit_div(hi.x * s, m, rm),
                     unit_div(hi.y * s, m, rm));
    if constexpr (W + 1 < kWords) dot_keys<SHORT, W + 1>(acc, a, c, s, m, rm, r);
}

// Thread = position in the group (the bucket, or a half of it in the order
// that the launch before left).  Three dots against the group's anchors
// (first member, b = argmin s0, a = argmin sb), score = dot_a - sb, and a
// stable descending sort by (score, -position).  64 registers: two groups of
// 1024 share a CU, one's sort beside the other's dots.
template <int N>
__global__ __launch_bounds__(N, 8) void build_top_kernel(const uint8_t* __restrict__ pool, int64_t pool_pages,
                                                         const int32_t* __restrict__ tables, Carry carry) {
    __shared__ TopSmem<N> sm;
    const int32_t p = threadIdx.x, lane = p & (kWave - 1);
    const int32_t wave = __builtin_amdgcn_readfirstlane(p / kWave);
    const int64_t b = blockIdx.x / (kTokens / N);
    const int64_t at = carry.at(b, (int32_t)(blockIdx.x % (kTokens / N)) * N + p);

    const int32_t tok = N == kTokens ? p : carry.tok[at];
    const int64_t page = page_of(tables + b * 16, tok, pool_pages);
    uint32_t c[kWords];
    load_key(pool + page * V1_PAGE_BYTES + (tok % 64) * 128, c);
    // the token's scale, unit divisor and its reciprocal
    const float s = reinterpret_cast<const float*>(pool)[page * kPageWords + kScaleWord + tok % 64];
    const float m = N == kTokens ? unit_norm(c, s) : carry.m[at];
    const float rm = 1.0f / m;
    const Recip r = unit_recip(s, m, rm);
    const bool all_short = __builtin_amdgcn_ballot_w64(!short_units(s)) == 0;

    auto stage_put = [&](Stage& st) __attribute__((always_inline)) {
        uint4* dst = reinterpret_cast<uint4*>(st.c);
#pragma unroll
        for (int i = 0; i < kWords / 4; ++i) dst[i] = make_uint4(c[4 * i], c[4 * i + 1], c[4 * i + 2], c[4 * i + 3]);
        st.s = s;
        st.m = m;
        st.rm = rm;
    };
    // dot with the staged token: lane i of a row expands its dims i, 16 + i, ...
    auto dot = [&](const Stage& st) __attribute__((always_inline)) {
        float a[8];
        const float sa = st.s, ma = st.m, ra = st.rm;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t w = st.c[4 * j + ((lane & 15) >> 2)] >> (8 * (lane & 3));
            a[j] = unit_div(fp8_at<0>(w) * sa, ma, ra);
        }
        Acc4 acc;
        if (all_short) dot_keys<true>(acc, a, c, s, m, rm, r);
        else dot_keys<false>(acc, a, c, s, m, rm, r);
        return acc.total();
    };
    // group argmin (leftmost minimum, -0.0 == +0.0): every wave's winner stages
    // its key; returns the group's winner's wave
    auto argmin = [&](float v, int32_t i) __attribute__((always_inline)) {
        const uint64_t k = lanes_min(((uint64_t)score_key(v) << 32) | (uint32_t)p, kWave);
        if ((uint32_t)k == (uint32_t)p) {
            stage_put(sm.win[i][wave]);
            atomicMin(&sm.amin[i], (unsigned long long)k);
        }
        __syncthreads();
        return (int32_t)(uint32_t)sm.amin[i] / kWave;
    };
    if (p < 2) sm.amin[p] = ~0ull;
    if (p == 0) stage_put(sm.first);
    sm.m[p] = m;
    sm.tok[p] = tok;
    __syncthreads();

    const float s0 = dot(sm.first);
    const float sb = dot(sm.win[0][argmin(s0, 0)]);
    const float score = dot(sm.win[1][argmin(sb, 1)]) - sb;
    int32_t nb = 0;
    const uint64_t key = bitonic_sort<N>(((uint64_t)score_key(score) << 32) | (0xffffffffu - (uint32_t)p), p, wave,
                                         sm.k, nb);
    const int32_t from = (int32_t)(0xffffffffu - (uint32_t)key);  // old position of the new member
    carry.tok[at] = sm.tok[from];
    carry.m[at] = sm.m[from];
}

// ---- groups of 256 to 16: a quarter of a bucket per work-group
constexpr int kQuarterWaves = kQuarter / kWave;

// Tokens are numbered by their first position in the quarter; a thread's
// token moves as its number.
struct QuarterSmem {
    uint4 c[kQuarter][8];             // keys: 16-byte chunk j of token t at j ^ (t % 8)
    float4 v[kQuarter];               // scale, unit divisor, its reciprocal, token in the bucket (int bits)
    Recip r[kQuarter];
    unsigned long long amin[2][2];    // argmin words of the groups above one wave
    uint64_t k[2][kQuarter];          // sort keys crossing waves, double-buffered
    int32_t first[kQuarterWaves];     // first token of every wave
};

template <int W = 0>
__device__ __forceinline__ void dot_units(Acc4& acc, const float (&a)[8], const float (&u)[128]) {
    add_terms<W>(acc, a, u[4 * W], u[4 * W + 1], u[4 * W + 2], u[4 * W + 3]);
    if constexpr (W + 1 < kWords) dot_units<W + 1>(acc, a, u);
}

// Outputs of position `at` of bucket b, whose member is `id` of the work-group's
// keys and token `tok` of the bucket: perm, its row of the assembled pages, the
// member map, and its part of a center.  key(t, j) is 16-byte chunk j of key t.
template <class Key, class Scale>
__device__ __forceinline__ void write_member(int64_t b, int32_t at, int32_t id, int32_t tok, int32_t start,
                                             int32_t* perm_out, uint8_t* tmp_out, int32_t* map_out,
                                             uint8_t* centers_out, Key key, Scale scale_of) {
    perm_out[b * kTokens + at] = tok;
    map_out[b * kTokens + at] = start + tok;
    uint8_t* tp = tmp_out + (b * 16 + at / 64) * V1_PAGE_BYTES;
    uint4* row = reinterpret_cast<uint4*>(tp + (at % 64) * 128);
#pragma unroll
    for (int j = 0; j < 8; ++j) row[j] = key(id, j);
    reinterpret_cast<float*>(tp)[kScaleWord + at % 64] = scale_of(id);
    // center at / 8: lane r of the 8 members computes dims 16r .. 16r+15
    const int32_t lane = __lane_id(), r = lane & 7;
    float mean[16];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int32_t t = __builtin_amdgcn_ds_bpermute(((lane & ~7) + j) << 2, id);
        const uint4 w4 = key(t, r);
        const float sj = scale_of(t);
        const uint32_t words[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float x0 = (fp8_at<0>(words[q]) * sj), x1 = (fp8_at<1>(words[q]) * sj);
            const float x2 = (fp8_at<2>(words[q]) * sj), x3 = (fp8_at<3>(words[q]) * sj);
            if (j == 0) {
                mean[4 * q] = x0;
                mean[4 * q + 1] = x1;
                mean[4 * q + 2] = x2;
                mean[4 * q + 3] = x3;
            } else {
                mean[4 * q] = (mean[4 * q] + x0);
                mean[4 * q + 1] = (mean[4 * q + 1] + x1);
                mean[4 * q + 2] = (mean[4 * q + 2] + x2);
                mean[4 * q + 3] = (mean[4 * q + 3] + x3);
            }
        }
    }
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        mean[i] = (mean[i] * 0.125f);
        amax = fmaxf(amax, fabsf(mean[i]));
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off, kWave));
    const float scale = center_scale(amax);
    const float inv = 1.0f / scale;  // (a power of two from 2^-22 to 2^120: the products are the quotients)
    uint32_t packed[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
        packed[q] = e4m3_code(mean[4 * q] * inv) | (e4m3_code(mean[4 * q + 1] * inv) << 8) |
                    (e4m3_code(mean[4 * q + 2] * inv) << 16) |
                    (e4m3_code(mean[4 * q + 3] * inv) << 24);
    const int32_t center = at / 8;
    uint8_t* cp = centers_out + (b * 2 + center / 64) * V1_PAGE_BYTES;
    *reinterpret_cast<uint4*>(cp + (center % 64) * 128 + 16 * r) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
    if (r == 0) reinterpret_cast<float*>(cp)[kScaleWord + center % 64] = scale;
}

// Thread = position in the quarter; the levels as above.  A level makes its
// token's unit vector from the key in LDS (moving 128 registers instead costs
// more LDS time than that takes vector time: 740 against 527 us for 2048
// buckets when both were tried) and holds it through three dots.  Groups of at most one wave run
// without barriers.  Then the outputs of the quarter, or (tmp_out null) its
// order alone.
__global__ __launch_bounds__(kQuarter, 3) void build_quarter_kernel(const uint8_t* __restrict__ pool, int64_t pool_pages,
                                                                    const int32_t* __restrict__ tables,
                                                                    const int32_t* __restrict__ starts, Carry carry,
                                                                    int32_t* perm_out, uint8_t* tmp_out,
                                                                    int32_t* map_out, uint8_t* centers_out) {
    __shared__ QuarterSmem sm;
    const int32_t p = threadIdx.x, lane = p & (kWave - 1);
    const int32_t wave = __builtin_amdgcn_readfirstlane(p / kWave);
    const int64_t b = blockIdx.x / (kTokens / kQuarter);
    const int32_t at = (int32_t)(blockIdx.x % (kTokens / kQuarter)) * kQuarter + p;  // position in the bucket

    int32_t id = p;
    bool all_short;
    {
        const int32_t tok = carry.tok[carry.at(b, at)];
        const float m = carry.m[carry.at(b, at)];
        const int64_t page = page_of(tables + b * 16, tok, pool_pages);
        const uint4* src = reinterpret_cast<const uint4*>(pool + page * V1_PAGE_BYTES + (tok % 64) * 128);
#pragma unroll
        for (int j = 0; j < 8; ++j) sm.c[p][j ^ (p & 7)] = src[j];
        const float s = reinterpret_cast<const float*>(pool)[page * kPageWords + kScaleWord + tok % 64], rm = 1.0f / m;
        sm.v[p] = make_float4(s, m, rm, __int_as_float(tok));
        sm.r[p] = unit_recip(s, m, rm);
        all_short = __syncthreads_and(short_units(s));
    }
    float u[128];  // the token's unit vector
    auto make_units = [&]() __attribute__((always_inline)) {
        auto each_word = [&](auto unit) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint4 w4 = sm.c[id][j ^ (id & 7)];
                const uint32_t words[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float2 lo = fp8_pair<false>(words[q]), hi = fp8_pair<true>(words[q]);
                    float* d = u + 16 * j + 4 * q;
                    d[0] = unit(lo.x);
                    d[1] = unit(lo.y);
                    d[2] = unit(hi.x);
                    d[3] = unit(hi.y);
                }
            }
        };
        if (all_short) {
            const Recip r = sm.r[id];
            each_word([&](float c) __attribute__((always_inline)) { return unit_short(c, r); });
        } else {
            const float4 v = sm.v[id];
            each_word([&](float c) __attribute__((always_inline)) { return unit_div(c * v.x, v.y, v.z); });
        }
    };
    // dot with token t's unit vector: lane i of a row expands its dims i, 16 + i, ...
    auto dot = [&](int32_t t) __attribute__((always_inline)) {
        const uint8_t* row = reinterpret_cast<const uint8_t*>(sm.c[t]) + (lane & 15);
        float a[8];
        if (all_short) {
            const Recip r = sm.r[t];
#pragma unroll
            for (int j = 0; j < 8; ++j) a[j] = unit_short(fp8_at<0>(row[16 * (j ^ (t & 7))]), r);
        } else {
            const float4 v = sm.v[t];
#pragma unroll
            for (int j = 0; j < 8; ++j) a[j] = unit_div(fp8_at<0>(row[16 * (j ^ (t & 7))]) * v.x, v.y, v.z);
        }
        Acc4 acc;
        dot_units(acc, a, u);
        return acc.total();
    };
    // token of the group's minimum (leftmost, -0.0 == +0.0)
    auto argmin = [&](float v, auto group, int32_t i) __attribute__((always_inline)) {
        constexpr int32_t n = decltype(group)::value;
        uint64_t k = lanes_min(((uint64_t)score_key(v) << 32) | (uint32_t)(p << 8 | id), n < kWave ? n : kWave);
        if constexpr (n > kWave) {
            if (lane == 0) atomicMin(&sm.amin[i][wave / (n / kWave)], (unsigned long long)k);
            __syncthreads();
            k = sm.amin[i][wave / (n / kWave)];
        }
        return (int32_t)(k & 255);
    };
    if (p < 4) (&sm.amin[0][0])[p] = ~0ull;
    __syncthreads();

    int32_t first = 0;  // first token of the group
    auto level = [&](auto group) __attribute__((always_inline)) {
        constexpr int32_t n = decltype(group)::value, half = n >> 1;
        make_units();
        const float s0 = dot(first);
        const float sb = dot(argmin(s0, group, 0));
        const float score = dot(argmin(sb, group, 1)) - sb;
        int32_t nb = 0;
        const uint64_t key = bitonic_sort<n>(((uint64_t)score_key(score) << 32) | ~(uint32_t)(p << 8 | id), p, wave,
                                             sm.k, nb);
        id = (int32_t)(~(uint32_t)key & 255u);
        if constexpr (half > kWave) {
            // (the sort's barriers lie between the argmin words' last use and this)
            if (lane == 0) sm.first[wave] = id;
            if (p < 4) (&sm.amin[0][0])[p] = ~0ull;
            __syncthreads();
            first = sm.first[wave & ~(half / kWave - 1)];
        } else if constexpr (half >= 16) {
            first = __builtin_amdgcn_ds_bpermute((lane & ~(half - 1)) << 2, id);
        }
    };
    level(std::integral_constant<int32_t, 256>());
    level(std::integral_constant<int32_t, 128>());
    level(std::integral_constant<int32_t, 64>());
    level(std::integral_constant<int32_t, 32>());
    level(std::integral_constant<int32_t, 16>());

    const int32_t tok = __float_as_int(sm.v[id].w);
    if (tmp_out == nullptr) {  // (build_write_kernel writes the outputs)
        carry.tok[carry.at(b, at)] = tok;
        return;
    }
    write_member(b, at, id, tok, starts[b], perm_out, tmp_out, map_out, centers_out,
                 [&](int32_t t, int32_t j) __attribute__((always_inline)) { return sm.c[t][j ^ (t & 7)]; },
                 [&](int32_t t) __attribute__((always_inline)) { return sm.v[t].x; });
}

// The outputs of a bucket in the order that the launches before left, by one
// work-group that has read all of the bucket before it writes: for outputs that
// lie over the bucket's own pages.
__global__ __launch_bounds__(kTokens) void build_write_kernel(const uint8_t* pool, int64_t pool_pages,
                                                              const int32_t* tables, const int32_t* starts, Carry carry,
                                                              int32_t* perm_out, uint8_t* tmp_out, int32_t* map_out,
                                                              uint8_t* centers_out) {
    __shared__ uint4 c[kTokens][8];
    __shared__ float s[kTokens];
    const int32_t p = threadIdx.x;
    const int64_t b = blockIdx.x;
    const int32_t tok = carry.tok[carry.at(b, p)], start = starts[b];
    const int64_t page = page_of(tables + b * 16, tok, pool_pages);
    const uint4* src = reinterpret_cast<const uint4*>(pool + page * V1_PAGE_BYTES + (tok % 64) * 128);
#pragma unroll
    for (int j = 0; j < 8; ++j) c[p][j ^ (p & 7)] = src[j];
    s[p] = reinterpret_cast<const float*>(pool)[page * kPageWords + kScaleWord + tok % 64];
    __syncthreads();
    write_member(b, p, p, tok, start, perm_out, tmp_out, map_out, centers_out,
                 [&](int32_t t, int32_t j) __attribute__((always_inline)) { return c[t][j ^ (t & 7)]; },
                 [&](int32_t t) __attribute__((always_inline)) { return s[t]; });
}

}  // namespace
}  // namespace v1

using namespace v1;

extern "C" int v1_build_initialize(const void* K, const float* KS, const int32_t* table, const int32_t* meta,
                                   float* unit, int32_t* perm, int32_t* flag, int32_t programs, void* stream) {
    V1_REQUIRE(programs >= 0, "initialize: negative grid");
    V1_REQUIRE((reinterpret_cast<uintptr_t>(K) & 15) == 0 && (reinterpret_cast<uintptr_t>(unit) & 15) == 0,
               "initialize: K and UNIT must be 16-byte aligned");
    if (programs == 0) return V1_OK;
    hipLaunchKernelGGL(initialize_kernel, dim3((uint32_t)programs), dim3(64), 0, as_stream(stream),
                       static_cast<const uint8_t*>(K), KS, table, meta, unit, perm, flag);
    return V1_LAUNCHED("initialize");
}

extern "C" int v1_group_dots(const float* U, const int32_t* P, const int32_t* A, float* S, const int32_t* flag,
                             int32_t N, int32_t start, int32_t mode, int32_t programs, int32_t heads, void* stream) {
    V1_REQUIRE(N > 0 && mode >= 0 && mode <= 2 && programs >= 0 && heads >= 0, "_dots: bad arguments");
    V1_REQUIRE((reinterpret_cast<uintptr_t>(U) & 15) == 0, "_dots: U must be 16-byte aligned");
    if (programs == 0 || heads == 0) return V1_OK;
    hipLaunchKernelGGL(dots_kernel, dim3((uint32_t)programs, (uint32_t)heads), dim3(64), 0, as_stream(stream), U, P, A,
                       S, flag, N, start, mode);
    return V1_LAUNCHED("_dots");
}

extern "C" int v1_group_anchor(const int32_t* P, int32_t* A, const float* S, const int32_t* flag, int32_t N,
                               int32_t slot, int32_t groups, int32_t heads, void* stream) {
    V1_REQUIRE(N > 0 && (slot == 0 || slot == 1) && groups >= 0 && heads >= 0, "_anchor: bad arguments");
    if (groups == 0 || heads == 0) return V1_OK;
    hipLaunchKernelGGL(anchor_kernel, dim3((uint32_t)groups, (uint32_t)heads), dim3(256), 0, as_stream(stream), P, A,
                       S, flag, N, slot);
    return V1_LAUNCHED("_anchor");
}

extern "C" int v1_build_assemble(const void* K, const float* KS, const int32_t* table, const int32_t* meta,
                                 const int32_t* ids, void* tmp, float* tmps, void* centers, float* cs, int32_t* map,
                                 int32_t pages, int32_t groups, void* stream) {
    V1_REQUIRE(pages >= 0 && groups >= 0 && groups <= 8, "assemble: bad grid");
    if (pages == 0 || groups == 0) return V1_OK;
    hipLaunchKernelGGL(assemble_kernel, dim3((uint32_t)pages, (uint32_t)groups), dim3(128), 0, as_stream(stream),
                       static_cast<const uint8_t*>(K), KS, table, meta, ids, static_cast<uint8_t*>(tmp), tmps,
                       static_cast<uint8_t*>(centers), cs, map);
    return V1_LAUNCHED("assemble");
}

extern "C" int v1_build_buckets(const void* pool, int64_t pool_pages, const int32_t* tables, const int32_t* starts,
                                int32_t buckets, int32_t* perm, void* tmp, int32_t* mapping, void* centers,
                                void* stream) {
    V1_REQUIRE(buckets >= 0 && pool_pages > 0, "build_buckets: bad shape");
    V1_REQUIRE((reinterpret_cast<uintptr_t>(pool) & 15) == 0 && (reinterpret_cast<uintptr_t>(tmp) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(centers) & 15) == 0,
               "build_buckets: pool, tmp and centers must be 16-byte aligned");
    if (buckets == 0) return V1_OK;
    // Outputs over a bucket's own pages are allowed (all of the bucket is read
    // before any of them is written); quarters that read and write side by side
    // are for outputs elsewhere.  The order between the launches lies in tmp, or
    // where tmp is over the pool in centers, or else in perm and mapping.
    const int64_t pool_bytes = pool_pages * V1_PAGE_BYTES, order_bytes = (int64_t)buckets * kTokens * 4;
    auto meet = [](const void* a, int64_t na, const void* b, int64_t nb) {
        const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
        return x < y + (uintptr_t)nb && y < x + (uintptr_t)na;
    };
    const bool tmp_meets = meet(pool, pool_bytes, tmp, (int64_t)buckets * 16 * V1_PAGE_BYTES);
    const bool order_meets = meet(pool, pool_bytes, perm, order_bytes) || meet(pool, pool_bytes, mapping, order_bytes);
    const bool centers_meet = meet(pool, pool_bytes, centers, (int64_t)buckets * 2 * V1_PAGE_BYTES);
    const bool in_place = tmp_meets || order_meets || centers_meet;
    V1_REQUIRE(!tmp_meets || !centers_meet || !(order_meets || meet(perm, order_bytes, mapping, order_bytes)),
               "build_buckets: with tmp and centers over the pool, perm and mapping must be apart from it and from "
               "each other");
    Carry carry{perm, reinterpret_cast<float*>(mapping), kTokens, kQuarter};
    if (!tmp_meets) {
        carry = Carry{static_cast<int32_t*>(tmp), static_cast<float*>(tmp) + kQuarter, 16 * kPageWords, 4 * kPageWords};
    } else if (!centers_meet) {
        static_assert(2 * kTokens <= 2 * kPageWords, "order and divisors of a bucket in its two center pages");
        carry = Carry{static_cast<int32_t*>(centers), static_cast<float*>(centers) + kTokens, 2 * kPageWords, kQuarter};
    }
    const uint8_t* const from = static_cast<const uint8_t*>(pool);
    uint8_t* const pages = static_cast<uint8_t*>(tmp);
    uint8_t* const means = static_cast<uint8_t*>(centers);
    hipStream_t st = as_stream(stream);
    hipLaunchKernelGGL(build_top_kernel<1024>, dim3((uint32_t)buckets), dim3(1024), 0, st, from, pool_pages, tables, carry);
    int rc = V1_LAUNCHED("build_buckets: 1024");
    if (rc != V1_OK) return rc;
    hipLaunchKernelGGL(build_top_kernel<512>, dim3((uint32_t)buckets * 2), dim3(512), 0, st, from, pool_pages, tables, carry);
    rc = V1_LAUNCHED("build_buckets: 512");
    if (rc != V1_OK) return rc;
    hipLaunchKernelGGL(build_quarter_kernel, dim3((uint32_t)buckets * (kTokens / kQuarter)), dim3(kQuarter), 0, st, from,
                       pool_pages, tables, starts, carry, perm, in_place ? nullptr : pages, mapping, means);
    rc = V1_LAUNCHED("build_buckets: quarters");
    if (rc != V1_OK || !in_place) return rc;
    hipLaunchKernelGGL(build_write_kernel, dim3((uint32_t)buckets), dim3(kTokens), 0, st, from, pool_pages, tables, starts,
                       carry, perm, pages, mapping, means);
    return V1_LAUNCHED("build_buckets: outputs");
}
