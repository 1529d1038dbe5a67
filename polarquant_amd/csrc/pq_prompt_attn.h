// Causal attention of a prompt (flash attention on the matrix cores), shared by the polar-key and the latent-attention libraries.
#pragma once
#include "pq_mfma.h"

namespace pq {

struct PromptAttnArgs {
    const void *q, *k, *v;                    // q element (b, t, h, d) at b q_b + t q_t + h q_h + d; k likewise with key head h / (H / G)
    int64_t q_b, q_t, q_h, k_b, k_t, k_h;
    int64_t v_b, v_t, v_h;                    // a row per token: (b, t, g, c) at b v_b + t v_t + g v_h + c; a row per channel: v_t apart
    const float* sink;                        // [H] or null
    const void* gate;                         // [B * L, H * Dv] rows gate_row apart, or null
    int64_t gate_row;
    const int32_t* start;                     // [B]: keys before it do not exist; or null
    void* out;                                // [B * L, H * Dv] rows out_row apart
    int64_t out_row;
    int B, L, Lk, H, G, D, Dv;                // the L queries are the last of the Lk tokens
    float scale;
    // of a sliding window (WINDOW): k and v hold the call's own tokens, those before it are row (position % cap) of [B, G, cap, ..] rings
    const void *k_ring, *v_ring;
    const float* slopes;                      // [H] taken off a score per position of distance, or null
    int cap, window;
    float out_scale;                          // (times the result)
};

constexpr int kPromptTileRows = 128, kPromptTileKeys = 64;
constexpr int kAhead = 4;                     // steps of the score product whose keys are on their way from LDS

// 16 bytes per lane from global memory into 1 KiB of LDS at `lds` (uniform), lane after lane.  Not known to the compiler's count
// of loads in flight: wait_lds_loads() before the barrier behind which the data is read.  (The builtin is known to it, and makes every
// read of LDS wait for the next tile's loads.)  The load reads M0 one wait state after a scalar write at the earliest; the compiler
// leaves that to us inside an asm statement.  (M0 is named as written, so that nothing else relies on it; it is never allocated, which is
// what the warning would say.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_to_lds(const void* p, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(p), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ void wait_lds_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// the larger of lanes l and l ^ 32, by an exchange of half wavefronts that stays in the vector unit
__device__ __forceinline__ float both_halves_max(float v) {
    typedef unsigned int uint2_x __attribute__((ext_vector_type(2)));
    const uint2_x r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
}

// The order of a basic block's instructions by kind (a rule for the compiler's scheduler, which takes the calls in their order): so many
// of one kind next.
constexpr int kMatrix = 0x8, kDsRead = 0x100;
template <int KIND, int N>
__device__ __forceinline__ void order() { __builtin_amdgcn_sched_group_barrier(KIND, N, 0); }

typedef float floatx2_a __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_a __attribute__((ext_vector_type(2)));
typedef _Float16 halfx2_a __attribute__((ext_vector_type(2)));
template <typename T> __device__ __forceinline__ uint32_t pack_pair(float a, float b);
template <> __device__ __forceinline__ uint32_t pack_pair<BF16>(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2_a{a, b}, bf16x2_a));
}
template <> __device__ __forceinline__ uint32_t pack_pair<F16>(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2_a{a, b}, halfx2_a));
}

// grid (heads, query tiles, sequences), longest query tiles first.  Four wavefronts with 32 query rows each over 64-key tiles of K
// and V that are double-buffered in LDS.  The transposed score tile S^T = K Q^T makes a query a lane, its softmax state a
// register, and P^T the right operand of O^T = V^T P^T as it stands.  TOKEN_ROWS: V has a row per token and is transposed on the
// way out of LDS; otherwise a row per channel, as a product with the weights on the left leaves it.
//
// What bounds it: matrix cores and vector unit are both busy for half of the time (32 products of 32 cycles a tile; 32 exponentials and
// some 150 other vector instructions a lane), and the two wavefronts of a SIMD overlap little of it beyond what each has side by
// side itself.  So the order of a tile's instructions is laid down: keys for four steps of the score product are on their way from
// LDS, and each product with V stands beside two of the next step's weights and the reads of its operand (left alone, the compiler waits
// for LDS every second product and makes all weights before the first).  Tiles go to LDS directly (no registers, no store instructions);
// the addresses that the lanes load from swizzle them so that 16 lanes' reads of 16 bytes, or 32 lanes' of 8, meet every bank once (by
// 8 rows instead of 16 half of the LDS cycles were conflicts).  The scale is part of the exponential's multiply-add.
// In turn with the kernel before (compiler's order, 8-row swizzle), bf16, us: 8192 tokens, 32 heads of 128, a row per token 586 -> 567,
// per channel 585 -> 584 (its reads of V meet a bank twice whatever the swizzle); 2048 tokens 58.5 -> 54.7, 59.2 -> 56.0; 4096 tokens,
// 16 heads of 192 / 256 143.6 -> 133.1, 238.7 -> 202.1.  No gain: three or four buffers; eight wavefronts that take turns at scores and
// products; eight wavefronts over one tile of keys without turns 545 for 560.
// A step that makes the next tile's scores beside this tile's weights needs more registers than two wavefronts have; raised wavefront
// priority around the products changes nothing.
// The maximum is raised whenever it is exceeded: the largest weight of a row is then 1, which its 16 bits hold exactly.  Raised at an
// excess of 2^8 only, which saves most of the rescaling (615 and 592 us), that weight is rounded like the others and the error against
// 64 bits grows: by 3 % with normal scores, by 15 % where a few keys have most of the weight.
// WINDOW: a query sees the last `window` positions, with a bias per position of distance; tiles that a workgroup's windows do not touch
// are not visited, those before the call come from a ring, or from both where the call begins inside a tile.  8192 tokens, window
// 2048, 32 query and 8 KV heads of 128: 394 -> 341 us against tiles passed through registers (16 heads of 256: 649 -> 506).  The bias is
// added to a finished score in one multiply-add.  (As the start of the score's accumulator it takes 327 us, but every partial sum
// then rounds at the bias's size: where a bias of 2^17 cancels against the product, 1.7 times the error.)  Rows come from ring or call
// by selection (with branches: 3 % more at 5000 tokens before the call).
template <typename T, int DKP, int DVP, bool TOKEN_ROWS, bool WINDOW = false>
__global__ __launch_bounds__(256, DKP <= 128 ? 2 : 1) void prompt_attn_kernel(PromptAttnArgs a) {
    constexpr int KS = DKP / 16, VT = DVP / 32, KC = DKP / 8, VC = TOKEN_ROWS ? DVP / 8 : 8;        // 16-byte chunks of a row of K, of V
    constexpr int KBYTES = kPromptTileKeys * DKP * 2, VBYTES = kPromptTileKeys * DVP * 2;
    constexpr int KL = KBYTES / 4096, VL = VBYTES / 4096;                                          // loads per lane and tile
    static_assert(TOKEN_ROWS || !WINDOW, "a ring has a row per token");
    extern __shared__ __attribute__((aligned(1024))) uint8_t sm[];                                // two K tiles, then two V tiles
    const uint32_t lds0 = lds_addr(sm);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 31, hi = lane >> 5;
    const int H = a.H, D = a.D, Dv = a.Dv, b = blockIdx.z;
    const int h = blockIdx.x, g = h / (H / a.G);
    const int tile = static_cast<int>(gridDim.y) - 1 - static_cast<int>(blockIdx.y);
    const int past = a.Lk - a.L;
    const int qw = tile * kPromptTileRows + wv * 32, qi = qw + col;                 // the wavefront's first query token; this lane's
    const bool valid = qi < a.L;
    const int qc = valid ? qi : a.L - 1, limit = past + qc;                         // last key this row sees
    const int lo = a.start ? a.start[b] : 0;
    const int q_last = tile * kPromptTileRows + kPromptTileRows - 1 < a.L - 1 ? tile * kPromptTileRows + kPromptTileRows - 1 : a.L - 1;
    const int wave_last = past + (qw + 31 < a.L - 1 ? qw + 31 : a.L - 1);
    const int wave_first = past + (qw < a.L - 1 ? qw : a.L - 1);
    // the first key that any row of the workgroup sees
    int key_lo = WINDOW ? past + tile * kPromptTileRows - a.window + 1 : lo;
    key_lo = key_lo > lo ? key_lo : lo;
    key_lo = !WINDOW || key_lo > 0 ? key_lo : 0;
    const int it0 = key_lo / kPromptTileKeys, it1 = (past + q_last) / kPromptTileKeys + 1;
    // a scale of zero: the scores of zero queries, times one (a masked score, -inf, stays one)
    const float scale2 = a.scale != 0.0f ? fabsf(a.scale) * kLog2e : 1.0f;
    const float slope2 = WINDOW && a.slopes ? a.slopes[h] * kLog2e : 0.0f;

    // the queries: requested here, and masked once the first tile is on its way.  (A selection of what is loaded becomes a branch around each
    // load, and each is waited for by itself: 20 tokens, 32 heads of 128 9.0 us, 8.4 so; 16 heads of 192 10.4 and 9.5, 8 of 256 14.1 and
    // 12.4; with tiles passed through registers 8.0, 9.0, 12.7.)
    u32x4_a q[KS];
    {
        const uint16_t* qp = static_cast<const uint16_t*>(a.q) + b * a.q_b + qc * a.q_t + h * a.q_h;
        static_for<KS>([&](auto I) {
            const int c = decltype(I)::value * 16 + 8 * hi;
            q[I] = *reinterpret_cast<const u32x4_a*>(qp + (c < D ? c : 0));
        });
    }
    auto mask_queries = [&]() {
        const uint32_t flip = a.scale < 0.0f ? 0x80008000u : 0u, zero = a.scale != 0.0f ? 0xffffffffu : 0u;
        static_for<KS>([&](auto I) {
            const uint32_t keep = decltype(I)::value * 16 + 8 * hi < D ? zero : 0u;
            q[I] = u32x4_a{(q[I].x ^ flip) & keep, (q[I].y ^ flip) & keep, (q[I].z ^ flip) & keep, (q[I].w ^ flip) & keep};
        });
    };
    // where this lane's 16 bytes of each load come from: load i of a wavefront fills chunks (wv KL + i) 64 .. + 63 of a tile
    const uint16_t* kb = static_cast<const uint16_t*>(a.k) + b * a.k_b + g * a.k_h;
    const uint16_t* vb = static_cast<const uint16_t*>(a.v) + b * a.v_b + g * a.v_h;
    auto k_swz = [](int row) { return DKP % 128 ? (row >> 1) & 7 : row & 15; };
    auto v_swz = [](int row) { return TOKEN_ROWS ? (DVP == 64 ? ((row >> 1) & 1) << 2 : (row & 3) << 2) : (row >> 1) & 7; };
    // with WINDOW, row (first + row) of the sequence: the ring's before this call's own
    auto either = [&](const uint16_t* own, int64_t own_t, const void* ring, int width, int first, int slot, int row, int last) {
        const int key = first + (row < last ? row : last);
        const bool past_key = key < past;                           // (selected, not branched on)
        return (past_key ? static_cast<const uint16_t*>(ring) + (static_cast<int64_t>(b) * a.G + g) * a.cap * width : own) +
               static_cast<int64_t>(past_key ? slot + row : key - past) * (past_key ? width : own_t);
    };
    auto k_src = [&](int i, int first, int slot, int last) {
        const int u = (wv * KL + i) * 64 + lane, row = u / KC, c = ((u % KC) ^ k_swz(row)) * 8;
        const uint16_t* at = WINDOW ? either(kb, a.k_t, a.k_ring, D, first, slot, row, last) : kb + static_cast<int64_t>(first + (row < last ? row : last)) * a.k_t;
        return at + (c < D ? c : 0);
    };
    auto v_src = [&](int i, int first, int slot, int last) {
        const int u = (wv * VL + i) * 64 + lane, row = u / VC, c = ((u % VC) ^ v_swz(row)) * 8;
        if (!TOKEN_ROWS) return vb + static_cast<int64_t>(row < Dv ? row : Dv - 1) * a.v_t + first + c;
        const uint16_t* at = WINDOW ? either(vb, a.v_t, a.v_ring, Dv, first, slot, row, last) : vb + static_cast<int64_t>(first + (row < last ? row : last)) * a.v_t;
        return at + (c < Dv ? c : 0);
    };
    const uint16_t *ks[KL], *vs[VL];
    if (!WINDOW) {
        const int last = a.Lk - 1 - it0 * kPromptTileKeys > 0 ? a.Lk - 1 - it0 * kPromptTileKeys : 0;
        static_for<KL>([&](auto I) { ks[I] = k_src(I, it0 * kPromptTileKeys, 0, last); });
        static_for<VL>([&](auto I) { vs[I] = v_src(I, it0 * kPromptTileKeys, 0, last); });
    }
    auto fetch = [&](int it, auto BUF) {
        constexpr int buf = decltype(BUF)::value;
        const int last = a.Lk - 1 - it * kPromptTileKeys;          // rows past the end: copies of the last one, with weight zero
        // (the addresses of whole tiles of this call's tokens only advance)
        if ((it > it0 && last < kPromptTileKeys - 1) || (WINDOW && (it == it0 || (it - 1) * kPromptTileKeys < past))) {
            const int first = it * kPromptTileKeys, slot = WINDOW ? first % a.cap : 0;
            static_for<KL>([&](auto I) { ks[I] = k_src(I, first, slot, last); });
            if (TOKEN_ROWS) static_for<VL>([&](auto I) { vs[I] = v_src(I, first, slot, last); });
        }
        static_for<KL>([&](auto I) {
            load_to_lds(ks[I], lds0 + buf * KBYTES + (wv * KL + I) * 1024);
            ks[I] += kPromptTileKeys * a.k_t;
        });
        static_for<VL>([&](auto I) {
            load_to_lds(vs[I], lds0 + 2 * KBYTES + buf * VBYTES + (wv * VL + I) * 1024);
            vs[I] += TOKEN_ROWS ? kPromptTileKeys * a.v_t : kPromptTileKeys;
        });
    };
    floatx16_a o[VT];
    static_for<VT>([&](auto I) {
#pragma unroll
        for (int j = 0; j < 16; j++) o[decltype(I)::value][j] = 0.0f;
    });
    float m = kNone, l = 0.0f;

    // LDS addresses of this lane's reads: row `col` of K, chunk 2 i + hi
    // A row per channel: 8 chunks at VT distances; the chunks' addresses are kept and the distances are offsets (32 or 64 sums do not fit, or
    // are formed again beside every product: 8192 tokens 635 us).
    uint32_t ka[KS], va[TOKEN_ROWS ? VT : 8];
    static_for<KS>([&](auto I) { ka[I] = lds0 + col * (DKP * 2) + ((2 * I + hi) ^ k_swz(col)) * 16; });
    static_for<TOKEN_ROWS ? VT : 8>([&](auto I) {
        constexpr int i = decltype(I)::value;
        if (TOKEN_ROWS) {           // 16 lanes read 4 tokens x 16 channels and get them transposed
            const int row = 4 * hi + ((lane & 15) >> 2), chunk = 4 * i + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
            va[i] = lds0 + 2 * KBYTES + row * (DVP * 2) + (chunk ^ v_swz(row)) * 16 + (lane & 1) * 8;
        } else {                    // chunk i of row `col`: rows 32 apart have the same swizzle
            va[i] = lds0 + 2 * KBYTES + hi * 8 + col * 128 + (i ^ v_swz(col)) * 16;
        }
    });
    auto step = [&](int it, auto BUF) {
        constexpr int buf = decltype(BUF)::value;
        if (it + 1 < it1) fetch(it + 1, IC<buf ^ 1>{});
        const int key0 = it * kPromptTileKeys;
        if (key0 <= wave_last && (!WINDOW || key0 + kPromptTileKeys - 1 > wave_first - a.window)) {        // uniform over the wavefront
            floatx16_a s[2];
            // (this lane: query qi, keys key0 + 32 u + 8 (j / 4) + 4 hi + j % 4)
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int j = 0; j < 16; j++) s[u][j] = 0.0f;
            constexpr int KD = KS < kAhead ? KS : kAhead;
            u32x4_a kf[KD][2];
            auto k_load = [&](auto I) {
                constexpr int i = decltype(I)::value;
                kf[i % KD][0] = *lds_ptr<lds_u32x4>(ka[i] + buf * KBYTES);
                kf[i % KD][1] = *lds_ptr<lds_u32x4>(ka[i] + buf * KBYTES + 32 * DKP * 2);
            };
            static_for<KD>(k_load);
            static_for<KS>([&](auto I) {
                constexpr int i = decltype(I)::value;
                s[0] = mma32<T>(kf[i % KD][0], q[i], s[0]);
                s[1] = mma32<T>(kf[i % KD][1], q[i], s[1]);
                if constexpr (i + KD < KS) k_load(IC<i + KD>{});
            });
            order<kDsRead, 2 * KD>();
            static_for<KS - KD>([&](auto) {
                order<kMatrix, 2>();
                order<kDsRead, 2>();
            });
            order<kMatrix, 2 * KD>();
            if (WINDOW) {                                           // from here on in units of the exponent, the bias taken off
                const float base = -slope2 * static_cast<float>(limit - key0 - 4 * hi);
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int j = 0; j < 16; j++)
                        s[u][j] = __builtin_fmaf(s[u][j], scale2, __builtin_fmaf(slope2, static_cast<float>(32 * u + 8 * (j >> 2) + (j & 3)), base));
            }
            if (key0 + kPromptTileKeys - 1 > past + qw || key0 < lo || (WINDOW && key0 <= wave_last - a.window)) {
                const int oldest = WINDOW && limit - a.window + 1 > lo ? limit - a.window + 1 : lo;
                const int last = limit - key0 - 4 * hi, first = oldest - key0 - 4 * hi;
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int j = 0; j < 16; j++) {
                        const int e = 32 * u + 8 * (j >> 2) + (j & 3);
                        s[u][j] = (e <= last && e >= first) ? s[u][j] : -INFINITY;
                    }
            }
            float mx = fmaxf(s[0][0], s[1][0]);
#pragma unroll
            for (int j = 1; j < 16; j++) mx = fmaxf(fmaxf(mx, s[0][j]), s[1][j]);
            mx = both_halves_max(mx) * (WINDOW ? 1.0f : scale2);
            if (__any(mx > m)) {
                const float mn = fmaxf(m, mx), al = exp2_hw(m - mn);
                l *= al;
                static_for<VT>([&](auto I) {
#pragma unroll
                    for (int j = 0; j < 16; j++) o[decltype(I)::value][j] *= al;
                });
                m = mn;
            }
            // right operands of the four 16-token steps, each made beside the products of the one before it
            u32x4_a p[2], vf[2][VT];
            float sum[2] = {0.0f, 0.0f};
            auto v_load = [&](auto J, auto I) {
                constexpr int j = decltype(J)::value, i = decltype(I)::value;
                u32x2_a w0, w1;
                if constexpr (TOKEN_ROWS) {
                    const uint32_t at = va[i] + buf * VBYTES + j * 16 * DVP * 2;
                    w0 = __builtin_bit_cast(u32x2_a, __builtin_amdgcn_ds_read_tr16_b64_v4i16(lds_ptr<lds_short4>(at)));
                    w1 = __builtin_bit_cast(u32x2_a, __builtin_amdgcn_ds_read_tr16_b64_v4i16(lds_ptr<lds_short4>(at + 8 * DVP * 2)));
                } else {
                    w0 = *lds_ptr<lds_u32x2>(va[2 * j] + 32 * i * 128 + buf * VBYTES);
                    w1 = *lds_ptr<lds_u32x2>(va[2 * j + 1] + 32 * i * 128 + buf * VBYTES);
                }
                vf[j & 1][i] = u32x4_a{w0.x, w0.y, w1.x, w1.y};
            };
            auto weights = [&](auto J, auto N) {                    // the Nth two of step J
                constexpr int u = decltype(J)::value >> 1, n = decltype(N)::value, j = 8 * (decltype(J)::value & 1) + 2 * n;
                auto weight = [&](float x) { return exp2_hw(WINDOW ? x - m : __builtin_fmaf(x, scale2, -m)); };
                const float e0 = weight(s[u][j]), e1 = weight(s[u][j + 1]);
                sum[0] += e0;
                sum[1] += e1;
                p[decltype(J)::value & 1][n] = pack_pair<T>(e0, e1);
            };
            static_for<VT>([&](auto I) { v_load(IC<0>{}, I); });
            static_for<4>([&](auto N) { weights(IC<0>{}, N); });
            __builtin_amdgcn_sched_barrier(0);
            static_for<4>([&](auto J) {
                constexpr int j = decltype(J)::value;
                static_for<VT>([&](auto I) {
                    constexpr int i = decltype(I)::value;
                    o[i] = mma32<T>(vf[j & 1][i], p[j & 1], o[i]);
                    if constexpr (j < 3) {
                        v_load(IC<j + 1>{}, I);
                        if constexpr (VT < 4) { weights(IC<j + 1>{}, IC<2 * i>{}); weights(IC<j + 1>{}, IC<2 * i + 1>{}); }
                        else if constexpr (i % (VT / 4) == 0) weights(IC<j + 1>{}, IC<i / (VT / 4)>{});
                    }
                    __builtin_amdgcn_sched_barrier(0);              // (left alone, the compiler makes all weights first)
                });
            });
            l += sum[0] + sum[1];
        }
        wait_lds_loads();
        __syncthreads();
    };
    if (it0 < it1) fetch(it0, IC<0>{});
    mask_queries();
    wait_lds_loads();
    __syncthreads();
    for (int it = it0; it < it1; it += 2) {
        step(it, IC<0>{});
        if (it + 1 < it1) step(it + 1, IC<1>{});
    }
    l += __shfl_xor(l, 32);
    if (!valid) return;
    float inv = l > 0.0f ? (WINDOW ? a.out_scale : 1.0f) / l : 0.0f;
    if (!WINDOW && a.sink) {
        const float sink2 = a.sink[h] * kLog2e, mf = fmaxf(m, sink2), al = exp2_hw(m - mf);
        inv = al / (l * al + exp2_hw(sink2 - mf));
    }
    const size_t row = static_cast<size_t>(b) * a.L + qi;
    uint16_t* out = static_cast<uint16_t*>(a.out) + row * a.out_row + static_cast<size_t>(h) * Dv;
    const uint16_t* gate = !WINDOW && a.gate ? static_cast<const uint16_t*>(a.gate) + row * a.gate_row + static_cast<size_t>(h) * Dv : nullptr;
    const bool quads = WINDOW || (Dv % 4 == 0 && a.out_row % 4 == 0 && (!gate || a.gate_row % 4 == 0));
    static_for<VT>([&](auto I) {
        constexpr int i = decltype(I)::value;
#pragma unroll
        for (int j4 = 0; j4 < 4; j4++) {
            const int ch = i * 32 + 8 * j4 + 4 * hi;
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = o[i][4 * j4 + j] * inv;
            if (quads && ch + 4 <= Dv) {
                if (gate) {
                    const uint2 gv = *reinterpret_cast<const uint2*>(gate + ch);
                    const uint32_t gw[2] = {gv.x, gv.y};
#pragma unroll
                    for (int j = 0; j < 4; j++) v[j] = v[j] / (1.0f + __expf(-lo2f<T>(static_cast<uint16_t>(gw[j >> 1] >> (16 * (j & 1))))));
                }
                *reinterpret_cast<uint2*>(out + ch) = make_uint2(pack_pair<T>(v[0], v[1]), pack_pair<T>(v[2], v[3]));
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (ch + j < Dv) out[ch + j] = f2lo<T>(gate ? v[j] / (1.0f + __expf(-lo2f<T>(gate[ch + j]))) : v[j]);
            }
        }
    });
}

template <typename T, int DKP, int DVP, bool TOKEN_ROWS, bool WINDOW = false>
static int launch_prompt_attn(const PromptAttnArgs& a, hipStream_t st) {
    constexpr size_t bytes = 2 * 2 * static_cast<size_t>(kPromptTileKeys) * (DKP + DVP);
    static_assert(bytes <= 160 * 1024, "LDS");
    if (bytes > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prompt_attn_kernel<T, DKP, DVP, TOKEN_ROWS, WINDOW>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
        if (e != hipSuccess) return static_cast<int>(e);
    }
    dim3 grid(a.H, (a.L + kPromptTileRows - 1) / kPromptTileRows, a.B), block(256);
    hipLaunchKernelGGL((prompt_attn_kernel<T, DKP, DVP, TOKEN_ROWS, WINDOW>), grid, block, bytes, st, a);
    return static_cast<int>(hipGetLastError());
}

}  // namespace pq
