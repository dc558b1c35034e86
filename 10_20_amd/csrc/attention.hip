// Decode attention over the gathered workspace: the consumer that follows the
// slot gather (sglang/srt/layers/attention/v1_native/backend.py:306-315 calls
// flash_attn_with_kvcache(q[:, None], kg, vg, causal=False,
// softmax_scale=scaling) on the GatherWorkspace rows).  One query position
// per batch row, Hq query heads sharing each of Hkv KV heads (GQA group
// G = Hq / Hkv <= 4, the reference's group of 4), head dim 128, bf16 in, fp32 math, bf16 out:
//   O[b, h] = sum_j p_j v[b, j, h / G],  p = softmax_j(scale * q[b, h] . k[b, j, h / G])
// over the row's first n_b keys (n_b = seqlens[b] clamped to [0, S], or S);
// a row with no keys gives zeros.
//
// One wave attends one part of a row's keys (attn_parts: at most 8, 1 from 2049
// rows on), tile by tile of 32 keys on the matrix cores with a running maximum;
// the parts' sums are joined at the end.  Both products are
// v_mfma_f32_16x16x32_bf16:
//   scores  S^T = K Q^T: 16 keys x 16 columns, column n = head n % 4 (the same
//           scores for n / 4 = 0 .. 3).  K goes memory -> LDS without passing
//           registers (16-byte chunks of a 256-byte row XOR-swizzled by its
//           row in the fragment), and comes back as A fragments.
//   output  O = P V: the 16 rows of P are head m % 4, part m / 4 of the fp32
//           probability split exactly into three bf16 parts (8 + 8 + 8
//           significant bits), so the product keeps fp32 probabilities; the
//           parts' rows are added at the end.  Lane (g, c) loads dims
//           8c .. 8c+7 of keys 8g .. 8g+7, whole 256-byte rows per 16 lanes,
//           and turns its own 8 x 8 block into eight B fragments (MFMA t takes
//           dim 8c + t) with byte permutes: no lane needs another's data.
// The key order inside a tile is chosen so that a lane's 8 scores are the 8
// keys of its P fragment.  Scores stay fp32; exponentials are base 2.
//
// Bound by the memory path: K and V rows are read once per (row, key) in
// 256-byte pieces, 4.3 GB for 4096 rows of 2048 keys.  The form before this
// one (16 lanes per key, fp32 products, two passes) spent ~130 vector
// operations per 8 dims of a key and was bound by them: 717 us for those rows
// over a context of 131072 slots, 4 heads; now 193-217 us (4.3 GB in that time
// is 20-22 TB/s, which the L2s must give; 1 head 486 -> 190 us), one row 97 ->
// 15 us, 1024 rows of 128 keys 18 -> 15 us.  One head of at most 96 keys alone
// is slower than it was, by 0.1-0.5 us up to 1024 rows (4096 rows of 64 keys 23
// -> 26 us): the prologue's and the join's latency.  So are gathered keys of one
// head per KV head, by 2-10% (512 rows x 1024 keys 39.5 -> 43.3 us).  Over rows of contiguous
// keys (nothing shared) 822 -> 704 us, HBM's rate.
//
// Slot form: keys come straight from the K / V pools of one KV head through
// the row's slot ids (req[ids[b, j]], the GatherWorkspace mapping of
// sglang/srt/layers/attention/v1_native/kernels.py:62-77); an id below zero
// or past req, or a slot outside the pool, is a zero key and value, exactly
// what the gather writes: its loads go to a row of zeros.  Same arithmetic,
// without the workspace round trip; ids are fetched two steps (of 64 keys)
// and slots one step before their keys.
#include <algorithm>

#include "common.h"

namespace v1 {
namespace {

constexpr int kAttnDim = 128;
constexpr int kMaxGroup = 4;       // heads of a P fragment: 16 rows / (3 parts, one unused)
constexpr int kMaxScores = 12288;  // keys x heads that a call may have (the entries' limit, not these kernels')
constexpr int kTile = 32;          // keys per step of a wave
constexpr int kMaxWaves = 16;      // waves of a work-group
constexpr int kXcds = 8;
constexpr int kMaxParts = kXcds;   // parts of a row's keys
constexpr int kWaitAll = 0x0f70, kWaitButEight = 0x0f78;  // s_waitcnt vmcnt(0), vmcnt(8)

// Lane p ^ J within 16-lane rows, every lane active.
template <int J>
__device__ __forceinline__ float row_xor(float v) {
    const int x = __float_as_int(v);
    if constexpr (J == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false));
    else if constexpr (J == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false));
    else if constexpr (J == 8) return __int_as_float(__builtin_amdgcn_mov_dpp(x, 0x128, 0xF, 0xF, false));
    else return __int_as_float(__builtin_amdgcn_ds_swizzle(x, (J << 10) | 0x1F));
}

__device__ __forceinline__ float row_sum16(float v) {
    v += row_xor<8>(v);
    v += row_xor<4>(v);
    v += row_xor<2>(v);
    v += row_xor<1>(v);
    return v;
}

// 8 bf16 (16 bytes) -> fp32, exact.
__device__ __forceinline__ void bf16x8(const uint4 w, float (&f)[8]) {
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = __uint_as_float(u[i] << 16);
        f[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
    }
}

// fp32 -> bf16, round to nearest even (NaN stays NaN).
__device__ __forceinline__ uint16_t to_bf16(float x) {
    const uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

struct AttnParams {
    const uint16_t* q;
    int64_t q_batch, q_head;
    const uint16_t* k;
    int64_t k_batch, k_token, k_head;
    const uint16_t* v;
    int64_t v_batch, v_token, v_head;
    const int32_t* seqlens;
    uint16_t* out;
    int64_t o_batch, o_head;
    int32_t keys, group, rows, parts;
    float scale;
    // slot form
    const int32_t* ids;
    int64_t ids_stride;
    const int32_t* req;
    int64_t req_len;
    int64_t pool_rows;
    float* partial;  // lined form: [rows][parts][max G, sum G, out G x 128]
};

using bf16x8_t = __attribute__((ext_vector_type(8))) __bf16;
using f32x4_t = __attribute__((ext_vector_type(4))) float;
using u32x4_t = __attribute__((ext_vector_type(4))) uint32_t;

union Frag {
    uint4 u;
    uint32_t w[4];
    bf16x8_t v;
};

__device__ __forceinline__ f32x4_t mfma_bf16(const Frag& a, const Frag& b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0);
}

// K and V rows of the keys that a call has not: one row of zeros.
__device__ const uint4 zero_row[16] = {};

// LDS of one wave: a tile of K rows (row 4i + g of the buffer is key 8g + i),
// reused for the wave's partial sums, and the K / V row addresses of 64 keys.
struct WaveLds {
    union {
        uint4 k[kTile][16];
        float part[4][kMaxGroup][kAttnDim];
    } u;
    uint64_t addr[2 * kTile];
};

__device__ __forceinline__ void wave_lds_fence() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// The wave's sums again with fp32 products, for tiles whose accumulators are
// not finite: a part of a probability that is exactly zero meets an infinite
// value in the split product and gives NaN where the whole probability gives
// an infinity.  16 lanes per key, lane c dims 8c .. 8c+7, as the loads above.
template <bool SLOTS>
__device__ __forceinline__ void plain_sums(const AttnParams& p, int64_t b, const char* kb, const char* vb, int32_t kvh,
                                           int32_t first, int32_t end, float sub, WaveLds& my) {
    const int32_t lane = (int32_t)threadIdx.x % kWave, g = lane >> 4, c = lane & 15;
    const float scale2 = p.scale * 1.44269504088896341f;
    float acc[kMaxGroup][8] = {};
    for (int32_t j = first + g; j < end; j += 4) {
        int32_t slot = j;
        if constexpr (SLOTS) {
            const int32_t id = p.ids[b * p.ids_stride + j];
            slot = id >= 0 && id < p.req_len ? p.req[id] : -1;
            if (slot >= p.pool_rows) slot = -1;
        }
        uint4 kw = make_uint4(0, 0, 0, 0), vw = kw;
        if (slot >= 0) {
            kw = *reinterpret_cast<const uint4*>(kb + (int64_t)slot * p.k_token * 2 + 16 * c);
            vw = *reinterpret_cast<const uint4*>(vb + (int64_t)slot * p.v_token * 2 + 16 * c);
        }
        float kf[8], vf[8];
        bf16x8(kw, kf);
        bf16x8(vw, vf);
#pragma unroll
        for (int32_t h = 0; h < kMaxGroup; ++h) {
            if (h >= p.group) break;
            float qf[8], part = 0.f;
            bf16x8(*reinterpret_cast<const uint4*>(p.q + b * p.q_batch + (int64_t)(kvh * p.group + h) * p.q_head + 8 * c),
                   qf);
#pragma unroll
            for (int i = 0; i < 8; ++i) part = fmaf(qf[i], kf[i], part);
            const float e = __builtin_amdgcn_exp2f(row_sum16(part) * scale2 - __shfl(sub, 16 * g + h, kWave));
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[h][i] = fmaf(e, vf[i], acc[h][i]);
        }
    }
#pragma unroll
    for (int32_t h = 0; h < kMaxGroup; ++h) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float x = acc[h][i];
            x += __shfl_xor(x, 16, kWave);
            x += __shfl_xor(x, 32, kWave);
            my.u.part[g][h][8 * c + i] = g == 0 ? x : 0.f;
        }
    }
}

// Sums of a row's parts: parts' sums scaled to the largest of their maxima.
template <class Max, class Sum, class Out>
__device__ __forceinline__ float join_parts(int32_t parts, Max max_of, Sum sum_of, Out out_of) {
    float m = max_of(0);
    for (int32_t i = 1; i < parts; ++i) m = fmaxf(m, max_of(i));
    if (m == -__builtin_inff()) m = 0.f;
    float o = 0.f, s = 0.f;
    for (int32_t i = 0; i < parts; ++i) {
        const float f = __builtin_amdgcn_exp2f(max_of(i) - m);
        o = fmaf(f, out_of(i), o);
        s = fmaf(f, sum_of(i), s);
    }
    return o / s;
}

// One wave per part of a row.  LINED (slot form): a work-group is the same
// part of `blockDim / 64` rows, whose waves keep step tile by tile: with ids
// that ascend along each row, the rows of an XCD then pass the same stretch of
// the context together and find each other's keys in its 4 MB L2 (4096 rows
// over 131072 slots 205 us; without the barrier the rows drift apart and it
// takes 385-411 us; with ids in no order 543 us either way).  Else it is the
// parts of one (KV head, row), added through LDS.
template <bool SLOTS, bool LINED>
__global__ __launch_bounds__(64 * kMaxWaves) void decode_attn_kernel(AttnParams p) {
    extern __shared__ WaveLds wave_lds[];
    __shared__ float wave_max[kMaxParts][kMaxGroup], wave_sum_[kMaxParts][kMaxGroup];
    const int32_t wave = __builtin_amdgcn_readfirstlane((int32_t)threadIdx.x / kWave);
    const int32_t lane = (int32_t)threadIdx.x % kWave, g = lane >> 4, c = lane & 15;
    int32_t part = wave, kvh = blockIdx.x;
    int64_t b = blockIdx.y;
    bool extra = false;  // a wave past the last row: keeps the others' step, stores nothing
    if constexpr (LINED) {
        // work-groups reach the XCDs in turn: each part's rows on 8 / parts of them
        const int32_t rpb = (int32_t)blockDim.x / kWave, groups = (p.rows + rpb - 1) / rpb;
        const int32_t xcd = (int32_t)(blockIdx.x % kXcds), i = (int32_t)(blockIdx.x / kXcds), per = kXcds / p.parts;
        part = xcd / per;
        const int32_t rg = i * per + xcd % per;
        if (rg >= groups) return;
        kvh = 0;
        b = (int64_t)rg * rpb + wave;
        extra = b >= p.rows;
        if (extra) b = p.rows - 1;
    }
    const int32_t S = p.keys, G = p.group;
    const int32_t n = p.seqlens ? min(max(p.seqlens[b], 0), S) : S;
    // this wave's part of the row's tiles: `mine` of them from tile `first`
    const int32_t tiles = (n + kTile - 1) / kTile, each = (tiles + p.parts - 1) / p.parts;
    const int32_t first = min(part * each, tiles), mine = min(each, tiles - first);
    const int32_t end = min((first + mine) * kTile, n);  // of its keys: what is fetched past them is the row of zeros
    WaveLds& my = wave_lds[wave];

    const char* kb = reinterpret_cast<const char*>(p.k + (SLOTS ? 0 : b * p.k_batch) + (int64_t)kvh * p.k_head);
    const char* vb = reinterpret_cast<const char*>(p.v + (SLOTS ? 0 : b * p.v_batch) + (int64_t)kvh * p.v_head);

    // the tile's keys: lanes 0-31 resolve their K rows, lanes 32-63 their V
    // rows; the loads are unconditional (clamped), the conditions come after
    const uint32_t ids_end = (uint32_t)min(p.req_len, (int64_t)1 << 31);
    const uint32_t slots_end = (uint32_t)min(p.pool_rows, (int64_t)1 << 31);
    auto key_of = [&](int32_t it) __attribute__((always_inline)) { return (first + it) * kTile + (lane & 31); };
    auto fetch_id = [&](int32_t it) __attribute__((always_inline)) -> int32_t {
        if constexpr (!SLOTS) return 0;
        else return p.ids[b * p.ids_stride + min(key_of(it), end - 1)];
    };
    auto id_ok = [&](int32_t it, int32_t id) __attribute__((always_inline)) -> int32_t {
        return key_of(it) < end && (!SLOTS || (uint32_t)id < ids_end) ? -1 : 0;
    };
    auto fetch_slot = [&](int32_t id) __attribute__((always_inline)) -> int32_t {
        if constexpr (!SLOTS) return 0;
        else return p.req[min((uint32_t)id, ids_end - 1)];
    };
    const uint64_t my_base = reinterpret_cast<uint64_t>(lane < 32 ? kb : vb);
    const uint64_t my_pitch = (uint64_t)(lane < 32 ? p.k_token : p.v_token) * 2;
    auto put_addr = [&](int32_t it, int32_t ok_id, int32_t slot) __attribute__((always_inline)) {
        const int32_t row = SLOTS ? slot : key_of(it);
        const bool ok = ok_id != 0 && (!SLOTS || (uint32_t)slot < slots_end);
        const uint64_t base = ok ? my_base : reinterpret_cast<uint64_t>(&zero_row[0]);
        my.addr[lane] = base + (uint64_t)(ok ? (uint32_t)row : 0u) * my_pitch;
    };
    uint32_t k_chunk = 16 * (c ^ (4 * g)), v_chunk = 16 * c;
    uint32_t k_read = 256 * (4 * (c & 3) + (c >> 2)) + 16 * (g ^ c);  // A fragment 0: row of key 8 (c / 4) + c % 4
    // K rows of the tile in the address table, memory -> LDS: load i brings keys 8g + i, chunk c of a row at its place c ^ (4g + i % 4)
    auto load_k = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint64_t a = my.addr[8 * g + i] + (uint64_t)(k_chunk ^ (16u * (i & 3)));
            __builtin_amdgcn_global_load_lds(
                reinterpret_cast<const __attribute__((address_space(1))) void*>(a),
                reinterpret_cast<__attribute__((address_space(3))) void*>(
                    (__attribute__((address_space(3))) uint4*)&my.u.k[4 * i][0]),
                16, 0, 0);
        }
    };
    u32x4_t v[8];
    auto load_v = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint64_t a = my.addr[32 + 8 * g + i] + (uint64_t)v_chunk;
            v[i] = *reinterpret_cast<const __attribute__((address_space(1))) u32x4_t*>(a);
        }
    };

    f32x4_t acc[8];  // MFMA t: rows 4 part + head, dim 8c + t
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+v"(acc[t]));  // (zeros set in place: as constants they are copied as one block, past the registers)
    }
    // of head c % 4, base-2 exponents: the maximum so far, what is subtracted
    // (0 while the maximum is -inf), and this lane's share of the sum
    float mx = -__builtin_inff(), sub = 0.f, sum = 0.f;
    const float scale2 =
        __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(p.scale * 1.44269504088896341f)));
    const uint32_t cut1 = c >= 4 ? 0xffff0000u : 0u, cut2 = c >= 8 ? 0xffff0000u : 0u;

    // B fragments of Q^T: column c = head c % 4 (those past the group repeat its last head, for nothing)
    Frag q[4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
        q[s].u = *reinterpret_cast<const uint4*>(p.q + b * p.q_batch + (int64_t)(kvh * G + min(c & 3, G - 1)) * p.q_head +
                                                 32 * s + 8 * g);
    // The first ids and slots are fetched side by side: a wave with one tile
    // waits three times for memory (ids, slots, keys) before its first product.
    int32_t slot = 0, ok = 0, id = 0;  // slot and "id is in range" of tile it + 1, id of tile it + 2
    if (mine > 0) {
        const int32_t id0 = fetch_id(0), id1 = fetch_id(1);
        id = fetch_id(2);
        const int32_t slot0 = fetch_slot(id0);
        slot = fetch_slot(id1);
        ok = id_ok(1, id1);
        put_addr(0, id_ok(0, id0), slot0);
        // (landed before the keys are fetched: the loop's own waits count only its own loads)
#pragma unroll
        for (int s = 0; s < 4; ++s)
            asm volatile("" : "+v"(q[s].w[0]), "+v"(q[s].w[1]), "+v"(q[s].w[2]), "+v"(q[s].w[3]));
        asm volatile("" : "+v"(slot), "+v"(id)::"memory");
        wave_lds_fence();
        load_k();
        asm volatile("" ::: "memory");
        load_v();
    }
#pragma unroll 1
    for (int32_t it = 0; it < mine; ++it) {
        asm volatile("" : "+v"(k_chunk), "+v"(v_chunk), "+v"(k_read));  // (offsets made in place: kept, they spill)
        // This tile's K, before ids and slots are fetched behind it (the wait
        // that the compiler puts before the LDS reads would be for those too).
        // Rows in step wait for V as well: it keeps them closer together (4096
        // rows 197 us, 201 without; the other form 58-64 us for 64 rows, 66-80).
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(LINED ? kWaitAll : kWaitButEight);
        asm volatile("" ::: "memory");
        put_addr(it + 1, ok, slot);  // this tile's addresses have been read
        slot = fetch_slot(id);
        ok = id_ok(it + 2, id);
        asm volatile("" : "+v"(ok)::"memory");  // the old id is read before the next one is fetched into its register
        id = fetch_id(it + 3);
        // scores: rows r of MFMA group u are keys 8 (r / 4) + 4u + r % 4
        float s[8];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            f32x4_t d = {0.f, 0.f, 0.f, 0.f};
            Frag k[4];
#pragma unroll
            for (int st = 0; st < 4; ++st)  // (chunk 4 st + g of the row, at its place ^ c)
                k[st].u = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(my.u.k) + 4096 * u + (k_read ^ (64u * st)));
#pragma unroll
            for (int st = 0; st < 4; ++st) d = mfma_bf16(k[st], q[st], d);
#pragma unroll
            for (int i = 0; i < 4; ++i) s[4 * u + i] = d[i] * scale2;
            __builtin_amdgcn_sched_barrier(0);
        }
        wave_lds_fence();
        if (it + 1 < mine) load_k();
        asm volatile("" ::: "memory");  // the next V loads stay behind: the next tile's wait counts on it
        const int32_t left = end - (first + it) * kTile - 8 * g;  // keys of this lane's eight
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] = i < left ? s[i] : -__builtin_inff();
        float top = s[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) top = fmaxf(top, s[i]);
        if (__ballot(top > mx)) {
            top = fmaxf(top, mx);
            top = fmaxf(top, __shfl_xor(top, 16, kWave));
            top = fmaxf(top, __shfl_xor(top, 32, kWave));
            const float keep = mx == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(sub - top);
            mx = top;
            sub = top == -__builtin_inff() ? 0.f : top;
            sum *= keep;
            // row i of an accumulator is head i: lane i of every quad holds its factor
            const int x = __float_as_int(keep);
            const f32x4_t f = {__int_as_float(__builtin_amdgcn_mov_dpp(x, 0x00, 0xF, 0xF, false)),
                               __int_as_float(__builtin_amdgcn_mov_dpp(x, 0x55, 0xF, 0xF, false)),
                               __int_as_float(__builtin_amdgcn_mov_dpp(x, 0xAA, 0xF, 0xF, false)),
                               __int_as_float(__builtin_amdgcn_mov_dpp(x, 0xFF, 0xF, 0xF, false))};
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                acc[t][0] *= f[0];
                acc[t][1] *= f[1];
                acc[t][2] *= f[2];
                acc[t][3] *= f[3];
            }
        }
        Frag pf;  // part c / 4 of the probabilities of the lane's eight keys
        uint32_t e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float x = __builtin_amdgcn_exp2f(s[i] - sub);
            sum += x;
            const float r1 = x - __uint_as_float(__float_as_uint(x) & cut1);
            const float r2 = r1 - __uint_as_float(__float_as_uint(r1) & cut2);
            e[i] = __float_as_uint(r2);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) pf.w[i] = __builtin_amdgcn_perm(e[2 * i + 1], e[2 * i], 0x07060302u);
        // V: word w of the eight keys holds dims 8c + 2w (low halves) and 8c + 2w + 1 (high halves)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            Frag lo, hi;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                lo.w[i] = __builtin_amdgcn_perm(v[2 * i + 1][w], v[2 * i][w], 0x05040100u);
                hi.w[i] = __builtin_amdgcn_perm(v[2 * i + 1][w], v[2 * i][w], 0x07060302u);
            }
            acc[2 * w] = mfma_bf16(pf, lo, acc[2 * w]);
            acc[2 * w + 1] = mfma_bf16(pf, hi, acc[2 * w + 1]);
            __builtin_amdgcn_sched_barrier(0);
        }
        load_v();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (LINED) __builtin_amdgcn_s_barrier();  // (`mine` is the same for all of the work-group)
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load still writes the K buffer
    sum += __shfl_xor(sum, 16, kWave);
    sum += __shfl_xor(sum, 32, kWave);
    float odd = 0.f;  // NaN if an accumulator is not finite
#pragma unroll
    for (int t = 0; t < 8; ++t) odd += ((acc[t][0] + acc[t][1]) + (acc[t][2] + acc[t][3])) * 0.f;
    wave_lds_fence();
    if (__ballot(odd != odd) == 0) {
#pragma unroll
        for (int i = 0; i < kMaxGroup; ++i) {
            *reinterpret_cast<float4*>(&my.u.part[g][i][8 * c]) = make_float4(acc[0][i], acc[1][i], acc[2][i], acc[3][i]);
            *reinterpret_cast<float4*>(&my.u.part[g][i][8 * c + 4]) =
                make_float4(acc[4][i], acc[5][i], acc[6][i], acc[7][i]);
        }
    } else {
        plain_sums<SLOTS>(p, b, kb, vb, kvh, first * kTile, end, sub, my);
    }
    if constexpr (LINED) {
        wave_lds_fence();
        if (extra) return;
        auto out_at = [&](int32_t i) __attribute__((always_inline)) {
            const float* x = &my.u.part[0][0][0] + i;
            return (x[0] + x[kMaxGroup * kAttnDim]) + x[2 * kMaxGroup * kAttnDim];
        };
        if (p.parts == 1) {
            for (int32_t i = lane; i < G * kAttnDim; i += kWave) {
                const int32_t h = i / kAttnDim;  // (the same for the wave)
                const float m = __shfl(mx, h, kWave), l = __shfl(sum, h, kWave);
                const float o = join_parts(
                    1, [&](int32_t) { return m; }, [&](int32_t) { return l; }, [&](int32_t) { return out_at(i); });
                p.out[b * p.o_batch + (int64_t)h * p.o_head + i % kAttnDim] = to_bf16(n > 0 ? o : 0.f);
            }
            return;
        }
        float* o = p.partial + (b * p.parts + part) * (int64_t)(G * (kAttnDim + 2));
        if (lane < G) {
            o[lane] = mx;
            o[G + lane] = sum;
        }
        for (int32_t i = 2 * lane; i < G * kAttnDim; i += 2 * kWave)
            *reinterpret_cast<float2*>(o + 2 * G + i) = make_float2(out_at(i), out_at(i + 1));
        return;
    }
    if (lane < kMaxGroup) {
        wave_max[wave][lane] = mx;
        wave_sum_[wave][lane] = sum;
    }
    __syncthreads();
    for (int32_t idx = (int32_t)threadIdx.x; idx < G * kAttnDim; idx += (int32_t)blockDim.x) {
        const int32_t h = idx / kAttnDim, d = idx % kAttnDim;
        const auto& w = wave_lds;
        const float o = join_parts(
            p.parts, [&](int32_t i) { return wave_max[i][h]; }, [&](int32_t i) { return wave_sum_[i][h]; },
            [&](int32_t i) { return (w[i].u.part[0][h][d] + w[i].u.part[1][h][d]) + w[i].u.part[2][h][d]; });
        p.out[b * p.o_batch + (int64_t)(kvh * G + h) * p.o_head + d] = to_bf16(n > 0 ? o : 0.f);
    }
}

// Output of the lined form with several parts: one thread per (row, head, dim).
__global__ __launch_bounds__(256) void join_kernel(AttnParams p) {
    const int32_t G = p.group, idx = (int32_t)(blockIdx.x * 256 + threadIdx.x);
    const int32_t b = idx / (G * kAttnDim), hd = idx % (G * kAttnDim), h = hd / kAttnDim;
    if (b >= p.rows) return;
    const int32_t pitch = G * (kAttnDim + 2);
    const float* x = p.partial + (int64_t)b * p.parts * pitch;
    const float o = join_parts(
        p.parts, [&](int32_t i) { return x[i * pitch + h]; }, [&](int32_t i) { return x[i * pitch + G + h]; },
        [&](int32_t i) { return x[i * pitch + 2 * G + hd]; });
    p.out[b * p.o_batch + (int64_t)h * p.o_head + hd % kAttnDim] = to_bf16(p.keys > 0 ? o : 0.f);
}

// Parts of a row's keys, a function of the call's (rows x KV heads) and keys
// alone, so that every form adds the same sums in the same order: at most 8,
// at most one per tile, and no more than give each SIMD two waves, or four
// (what 128 registers allow) where each part keeps 8 tiles: a part costs a
// prologue of three dependent loads and its share of the join. Measured, us:
//   rows x keys      1      2      4      8     16 parts
//     64 x 2048     64     36     22     19     20
//    256 x  512     21     16     14     14     16
//    512 x 2048     74     49     38     41     53
//   1024 x  128     15     15     16
//   2048 x 2048    114    110    120    137    178
// (Up to 16 parts of one tile each, as many as four waves per SIMD, cost 1024
// rows x 128 keys 27 us and 2048 rows x 64 28, more than the form before the
// matrix cores.)
inline int32_t attn_parts(int64_t groups, int32_t keys) {
    const int64_t waves = 8ll * device_cus(), tiles = cdiv(keys, kTile);
    int32_t parts = 1;
    while (parts < kMaxParts && 2 * parts <= tiles &&
           2 * parts * groups <= (tiles >= 16 * parts ? 2 * waves : waves))
        parts *= 2;
    return parts;
}

// Parts in work-groups of their own, joined by a second launch, or the parts of
// a row in one work-group: rows in step meet in the L2s, which pays for the
// launch once the keys no longer fit them: 256 rows x 2048 keys 28 us, 38 in
// one launch; 128 x 2048 24 / 25, 512 x 512 24 / 24, 256 x 128 10 / 6.
inline bool attn_two_launches(int32_t rows, int32_t keys, int32_t parts) {
    return parts > 1 && (int64_t)rows * keys > 1ll << 18;
}

inline int64_t attn_partial_bytes(int32_t rows, int32_t group, int32_t parts) {
    return (int64_t)rows * parts * group * (kAttnDim + 2) * (int64_t)sizeof(float);
}

template <bool SLOTS, bool LINED>
int launch_waves(const AttnParams& p, dim3 grid, int32_t waves, hipStream_t st) {
    const size_t lds = sizeof(WaveLds) * (size_t)waves;
    static OncePerDevice lds_once;  // (to the most that any call takes: a smaller value would cut another thread's)
    const int rc = allow_lds(lds_once, reinterpret_cast<const void*>(decode_attn_kernel<SLOTS, LINED>),
                             sizeof(WaveLds) * (LINED ? kMaxWaves : kMaxParts), "decode_attention: LDS");
    if (rc != V1_OK) return rc;
    hipLaunchKernelGGL((decode_attn_kernel<SLOTS, LINED>), grid, dim3(64 * waves), lds, st, p);
    return V1_LAUNCHED("decode_attention");
}

// Slot form with room for its parts (or with one part): lined.
inline int launch_lined(const AttnParams& p, hipStream_t st) {
    const int64_t all = (int64_t)p.rows * p.parts, cus = device_cus();
    const int64_t rounds = cdiv(all, kMaxWaves * cus);
    const int32_t rpb = (int32_t)cdiv(all, rounds * cus);  // rows per work-group: one work-group per CU and round
    const int64_t groups = cdiv(p.rows, rpb);
    const int64_t blocks = kXcds * cdiv(groups, kXcds / p.parts);
    const int rc = launch_waves<true, true>(p, dim3((uint32_t)blocks), rpb, st);
    if (rc != V1_OK || p.parts == 1) return rc;
    hipLaunchKernelGGL(join_kernel, dim3((uint32_t)cdiv((int64_t)p.rows * p.group * kAttnDim, 256)), dim3(256), 0, st, p);
    return V1_LAUNCHED("decode_attention: join");
}

}  // namespace
}  // namespace v1

using namespace v1;

extern "C" int v1_decode_attention(const void* q, int64_t q_batch, int64_t q_head, const void* k, int64_t k_batch,
                                   int64_t k_token, int64_t k_head, const void* v, int64_t v_batch, int64_t v_token,
                                   int64_t v_head, const int32_t* seqlens, void* out, int64_t o_batch, int64_t o_head,
                                   int32_t batch, int32_t heads_q, int32_t heads_kv, int32_t keys, float scale,
                                   void* stream) {
    V1_REQUIRE(batch >= 0 && heads_kv > 0 && heads_q > 0 && heads_q % heads_kv == 0 && keys >= 0,
               "decode_attention: bad shape");
    const int32_t G = heads_q / heads_kv;
    V1_REQUIRE(G <= kMaxGroup, "decode_attention: at most %d query heads per KV head", kMaxGroup);
    V1_REQUIRE((int64_t)G * keys <= kMaxScores, "decode_attention: keys x group above %d", kMaxScores);
    const int64_t strides[] = {q_batch, q_head, k_batch, k_token, k_head, v_batch, v_token, v_head, o_batch, o_head};
    bool aligned = (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) % 16 == 0;
    for (int64_t s : strides) aligned = aligned && s % 8 == 0;
    V1_REQUIRE(aligned, "decode_attention: q, k, v must be 16-byte aligned with strides in multiples of 8 elements");
    if (batch == 0) return V1_OK;
    AttnParams p{static_cast<const uint16_t*>(q), q_batch, q_head, static_cast<const uint16_t*>(k), k_batch, k_token,
                 k_head, static_cast<const uint16_t*>(v), v_batch, v_token, v_head, seqlens,
                 static_cast<uint16_t*>(out), o_batch, o_head, keys, G, batch,
                 attn_parts((int64_t)batch * heads_kv, keys), scale, nullptr, 0, nullptr, 0, 0, nullptr};
    return launch_waves<false, false>(p, dim3((uint32_t)heads_kv, (uint32_t)batch), p.parts, as_stream(stream));
}

extern "C" int v1_decode_attention_slots_ws(const void* q, int64_t q_batch, int64_t q_head, const void* k_pool,
                                         int64_t k_slot, int64_t k_head, const void* v_pool, int64_t v_slot,
                                         int64_t v_head, int64_t pool_slots, int32_t head, const int32_t* req,
                                         int64_t req_len, const int32_t* ids, int64_t ids_stride, void* out,
                                         int64_t o_batch, int64_t o_head, int32_t rows, int32_t heads_q, int32_t keys,
                                         float scale, void* workspace, int64_t workspace_bytes, void* stream) {
    V1_REQUIRE(rows >= 0 && heads_q > 0 && heads_q <= kMaxGroup && keys >= 0 && head >= 0 && pool_slots >= 0,
               "decode_attention_slots: bad shape (at most %d query heads)", kMaxGroup);
    V1_REQUIRE((int64_t)heads_q * keys + keys <= kMaxScores, "decode_attention_slots: keys x (heads + 1) above %d",
               kMaxScores);
    V1_REQUIRE(req != nullptr && req_len > 0 && ids != nullptr, "decode_attention_slots: empty slot map");
    const int64_t strides[] = {q_batch, q_head, k_slot, k_head, v_slot, v_head, o_batch, o_head};
    bool aligned = (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_pool) |
                    reinterpret_cast<uintptr_t>(v_pool)) % 16 == 0;
    for (int64_t s : strides) aligned = aligned && s % 8 == 0;
    V1_REQUIRE(aligned, "decode_attention_slots: q and the pools must be 16-byte aligned, strides multiples of 8");
    if (rows == 0) return V1_OK;
    // the chosen KV head becomes head 0 of a one-head problem
    AttnParams p{static_cast<const uint16_t*>(q), q_batch, q_head,
                 static_cast<const uint16_t*>(k_pool) + (int64_t)head * k_head, 0, k_slot, 0,
                 static_cast<const uint16_t*>(v_pool) + (int64_t)head * v_head, 0, v_slot, 0, nullptr,
                 static_cast<uint16_t*>(out), o_batch, o_head, keys, heads_q, rows,
                 attn_parts(rows, keys), scale, ids, ids_stride, req, req_len, pool_slots, static_cast<float*>(workspace)};
    const int64_t need = attn_partial_bytes(rows, heads_q, p.parts);
    if (p.parts == 1 || (attn_two_launches(rows, keys, p.parts) && workspace != nullptr && workspace_bytes >= need))
        return launch_lined(p, as_stream(stream));
    return launch_waves<true, false>(p, dim3(1, (uint32_t)rows), p.parts, as_stream(stream));
}

extern "C" int v1_decode_attention_slots(const void* q, int64_t q_batch, int64_t q_head, const void* k_pool,
                                         int64_t k_slot, int64_t k_head, const void* v_pool, int64_t v_slot,
                                         int64_t v_head, int64_t pool_slots, int32_t head, const int32_t* req,
                                         int64_t req_len, const int32_t* ids, int64_t ids_stride, void* out,
                                         int64_t o_batch, int64_t o_head, int32_t rows, int32_t heads_q, int32_t keys,
                                         float scale, void* stream) {
    return v1_decode_attention_slots_ws(q, q_batch, q_head, k_pool, k_slot, k_head, v_pool, v_slot, v_head, pool_slots,
                                        head, req, req_len, ids, ids_stride, out, o_batch, o_head, rows, heads_q, keys,
                                        scale, nullptr, 0, stream);
}

extern "C" int64_t v1_decode_attention_slots_workspace(int32_t rows, int32_t heads_q, int32_t keys) {
    if (rows <= 0 || heads_q <= 0 || heads_q > kMaxGroup || keys <= 0) return 0;
    const int32_t parts = attn_parts(rows, keys);
    return attn_two_launches(rows, keys, parts) ? attn_partial_bytes(rows, heads_q, parts) : 0;
}
