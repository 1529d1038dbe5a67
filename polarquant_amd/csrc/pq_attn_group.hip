// Fused polar-key decode attention for calls too small to fill the device: eight wavefronts share one slice of a context, 128 tokens
// at a time (reference decode branch: models/modeling_llama_polar.py:66-99).
//
// The scorer / accumulator pairs (pq_attn_pair.hip) and the one-wavefront kernels (pq_attn.hip) keep every SIMD of a full device
// busy; a call of a few dozen groups leaves most of it idle and waits for one wavefront's chain of table, scores and values
// instead (13 to 17 us whatever the length, up to 8000 tokens).  Here that chain is cut eight ways:
//   table   64 pairs x 16 bins: a thread makes two bins of its pair
//   scores  a wavefront looks up a quarter of the pairs (16 codes, one 16-byte load) of half the tokens; the quarters are added through LDS
//   values  a wavefront takes 16 tokens: running maximum, weights and sums of its own, P.V on the matrix cores
// and the eight wavefronts' results are joined at the end as the merge joins slices.  Residual keys go 16 to a wavefront.
// Everything that is read is requested before anything is waited for.
//
// What is left is the start of a launch, one trip to memory and three barriers: 5.9 us for a window of residual keys alone, 8.6
// with a group (pairs: 9.3 and 11.3; the one-wavefront kernel with 4-bit values 13.2, here 8.7), 16-bit values, 2000 tokens, 8 KV heads.
// Which calls come here: launch_attn_partials.
// This file is compiled once per dtype (-DPQ_DTYPE=0 float16, 1 bfloat16).
#include "pq_attn_device.h"

#ifndef PQ_DTYPE
#error "compile with -DPQ_DTYPE=0 (float16) or 1 (bfloat16)"
#endif

namespace pq {

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wint-to-pointer-cast"

constexpr int kGroupWaves = 8;

// What a wavefront has requested of a group of quantized tokens.
template <bool V4, bool PK6> struct GroupLoads {
    uint32_t code[PK6 ? 3 : 4];             // 16 codes of this lane's token
    uint16_t meta[4];                       // rscale, rmn, tscale, tmn of pair `lane`
    uint4 v[V4 ? 1 : 4];                    // values: dims 8 n .. of tokens 4 g + i
    uint32_t v4[V4 ? 4 : 1], sz[V4 ? 4 : 1][2];     // 4-bit values: word n, scale and zero point of tokens 4 i + g
    uint32_t keep[4];                       // mask bytes of the same tokens
};

template <typename T, int REPP, bool V4, bool PK6>
__global__ __launch_bounds__(kWave * kGroupWaves, 4) void attn_group_kernel(PQ_ATTN_KERNEL_PARAMS, int tbits, uint16_t* __restrict__ direct_out) {
    // entries of the table as in pq_device.h, always 16 slots to a pair: slot bin ^ (pair & 15), heads 4 .. 7 in a second half
    using L = Lut<4, REPP>;
    __shared__ __attribute__((aligned(16))) char lut_mem[REPP * kHeadDim * kGroupWaves * 4];       // the table, then the wavefronts' results
    __shared__ __attribute__((aligned(16))) float part[4][REPP][kGroup];
    __shared__ float ml[kGroupWaves][REPP][2];
    static_assert(L::BYTES <= REPP * kHeadDim * kGroupWaves * 4, "the table fits");
    PQ_ATTN_KERNEL_PACK;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int g = lane >> 4, n = lane & 15, quarter = wv >> 1, half = wv & 1;
    const int kvh = blockIdx.x, b = blockIdx.y, split = blockIdx.z;
    const uint32_t lut = lds_addr(lut_mem);
    const SeqCounts sc = seq_counts<V4>(p, v4, b);

    int gps = (sc.nb + n_splits - 1) / n_splits;
    gps = gps < min_gps ? min_gps : gps;
    gps = gps < 1 ? 1 : gps;
    // the residual keys have a slice of their own behind the groups' if there is one, else they are the last group's slice's
    const int used = (sc.nb + gps - 1) / gps;
    const int resid_split = sc.nres == 0 ? -1 : used < n_splits ? used : used - 1;
    if (split >= (used > 0 ? used : 1) && split != resid_split) {
        if (tid < rep) {
            float* pw = ws + ((static_cast<size_t>(b) * N + static_cast<size_t>(kvh) * rep_stride + tid) * n_splits + split) * kPartialFloats;
            pw[0] = -INFINITY;
            pw[1] = 0.0f;
        }
        return;
    }
    const int g0 = split * gps < sc.nb ? split * gps : sc.nb, g1 = g0 + gps < sc.nb ? g0 + gps : sc.nb;
    const int nres = split == resid_split ? sc.nres : 0;

    const int bh = b * Nk + kvh;
    const uint16_t* qb = p.q + (static_cast<size_t>(b) * N + static_cast<size_t>(kvh) * rep_stride) * kHeadDim;
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(p.v + static_cast<size_t>(bh) * v_capacity * kHeadDim,
                                                static_cast<uint32_t>((V4 ? sc.nres : sc.n_tokens) * (kHeadDim * 2)));
    const uint32_t voff_v = static_cast<uint32_t>(g) * (4 * kHeadDim * 2) + static_cast<uint32_t>(n) * 16;
    const bool has_mask = p.mask != nullptr;
    const __amdgpu_buffer_rsrc_t rm = make_rsrc(has_mask ? p.mask + static_cast<size_t>(b) * p.mask_stride : nullptr,
                                                has_mask ? static_cast<uint32_t>(sc.n_tokens < p.mask_stride ? sc.n_tokens : p.mask_stride) : 0u);
    constexpr int kRowB = PK6 ? kPackedRowBytes : kPairs;
    const size_t plane = static_cast<size_t>(bh) * group_capacity;
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(p.codes + plane * (kGroup * kRowB), static_cast<uint32_t>(sc.nb) * (kGroup * kRowB));
    const size_t vplane = static_cast<size_t>(bh) * static_cast<size_t>(V4 ? v4.capacity : 0);
    const __amdgpu_buffer_rsrc_t rq = make_rsrc(V4 ? v4.codes + vplane * 16 : nullptr, V4 ? static_cast<uint32_t>(sc.nb) * (kGroup * 64) : 0u);
    const __amdgpu_buffer_rsrc_t rvs = make_rsrc(V4 ? v4.scale + vplane : nullptr, V4 ? static_cast<uint32_t>(sc.nb) * (kGroup * 2) : 0u);
    const __amdgpu_buffer_rsrc_t rvz = make_rsrc(V4 ? v4.zero + vplane : nullptr, V4 ? static_cast<uint32_t>(sc.nb) * (kGroup * 2) : 0u);

    // token `i` (0 .. 3) of this lane in a wavefront's 16: the order in which the products take them
    auto token_of = [&](int i) { return V4 ? 4 * i + g : 4 * g + i; };
    using Loads = GroupLoads<V4, PK6>;
    auto request = [&](Loads& ld, int grp) {
        const uint32_t tok0 = static_cast<uint32_t>(grp) * kGroup, mine = tok0 + 16 * wv;
        if constexpr (PK6) {
#pragma unroll
            for (int i = 0; i < 3; i++)
                ld.code[i] = static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b32(rc, (kWave * half + lane) * kRowB + 12 * quarter + 4 * i, static_cast<int>(tok0 * kRowB), kAuxStream));
        } else {
            const uint4 w = buf_load16(rc, (kWave * half + lane) * kRowB + 16 * quarter, tok0 * kRowB);
            ld.code[0] = w.x; ld.code[1] = w.y; ld.code[2] = w.z; ld.code[3] = w.w;
        }
        const size_t m = (plane + grp) * kPairs + lane;
        ld.meta[0] = p.rscale[m]; ld.meta[1] = p.rmn[m]; ld.meta[2] = p.tscale[m]; ld.meta[3] = p.tmn[m];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (V4) {
                ld.v4[i] = static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b32(rq, g * 64 + n * 4 + 256 * i, static_cast<int>(mine * 64), kAuxStream));
                ld.sz[i][0] = __builtin_amdgcn_raw_buffer_load_b16(rvs, token_of(i) * 2, static_cast<int>(mine * 2), 0);
                ld.sz[i][1] = __builtin_amdgcn_raw_buffer_load_b16(rvz, token_of(i) * 2, static_cast<int>(mine * 2), 0);
            } else {
                ld.v[i] = buf_load16(rv, voff_v + i * (kHeadDim * 2), mine * (kHeadDim * 2));
            }
            ld.keep[i] = __builtin_amdgcn_raw_buffer_load_b8(rm, token_of(i), static_cast<int>(mine), 0);       // (no mask: out of range, 0)
        }
    };

    float m = -INFINITY, l = 0.0f, zp = 0.0f;           // of head n, over this wavefront's tokens; l and zp: this lane's share
    floatx4 acc[8];                                      // acc[e][i]: head n, dim 8 (4 g + i) + e
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    // raises the maximum over tokens whose scores (log2 units) this lane holds four of, and returns their weights
    auto weigh = [&](const float (&t)[4], float (&w)[4]) {
        float mx = fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]));
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32)));
        const float al = mx == -INFINITY ? 1.0f : exp2_raw(m - mx), ms = mx == -INFINITY ? 0.0f : mx;
        m = mx;
        l *= al;
        zp *= al;
#pragma unroll
        for (int e = 0; e < 8; e++) acc[e] *= al;
#pragma unroll
        for (int i = 0; i < 4; i++) { w[i] = exp2_raw(t[i] - ms); l += w[i]; }
    };
    // adds weights x rows of values in the model's dtype
    auto add_rows = [&](const uint4 (&v)[4], const float (&w)[4]) {
        const uint2 pb = make_uint2(static_cast<uint32_t>(f2lo<T>(w[0])) | (static_cast<uint32_t>(f2lo<T>(w[1])) << 16),
                                    static_cast<uint32_t>(f2lo<T>(w[2])) | (static_cast<uint32_t>(f2lo<T>(w[3])) << 16));
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
            auto word = [&](const uint4& x) { return (e >> 1) == 0 ? x.x : (e >> 1) == 1 ? x.y : (e >> 1) == 2 ? x.z : x.w; };
            acc[e] = mfma16<T>(make_uint2(__builtin_amdgcn_perm(word(v[1]), word(v[0]), sel), __builtin_amdgcn_perm(word(v[3]), word(v[2]), sel)), pb, acc[e]);
        }
    };
    const bool head = n < rep;

    uint4 rkeys[4], rvals[4], qv[4];
    uint32_t rkeep[4];
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(p.k_resid ? p.k_resid + static_cast<size_t>(bh) * resid_capacity * kHeadDim : nullptr,
                                                static_cast<uint32_t>(nres) * (kHeadDim * 2));
    auto request_resid = [&](int r) {
        const uint32_t key = static_cast<uint32_t>(r) * kGroup + 16 * wv, row = static_cast<uint32_t>(sc.nb) * kGroup + key;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            rkeys[i] = buf_load16(rk, n * (kHeadDim * 2) + g * 16 + 64 * i, key * (kHeadDim * 2));
            rvals[i] = buf_load16(rv, voff_v + i * (kHeadDim * 2), (V4 ? key : row) * (kHeadDim * 2));
            rkeep[i] = __builtin_amdgcn_raw_buffer_load_b8(rm, 4 * g + i, static_cast<int>(row), 0);
        }
    };
    Loads ld;
    if (g0 < g1) request(ld, g0);
    uint16_t qraw[REPP][2];
#pragma unroll
    for (int j = 0; j < REPP; j++) {
        const uint16_t* qrow = qb + (j < rep ? j : 0) * kHeadDim + lane;
        qraw[j][0] = qrow[0];
        qraw[j][1] = qrow[kPairs];
    }

    const uint32_t tmask = ((1u << tbits) - 1u) * 0x01010101u, rmask = (0xFFu >> tbits) * 0x01010101u;
    for (int grp = g0; grp < g1; grp++) {
        float cdv;
        {
            const float ts = lo2f<T>(ld.meta[2]), tm = lo2f<T>(ld.meta[3]), rs = lo2f<T>(ld.meta[0]), rmp = __builtin_fmaf(rs, 0.5f, lo2f<T>(ld.meta[1]));
            float a;
            if (rs != 0.0f) { a = rs; cdv = rmp / rs; }
            else            { a = rmp * 0x1p-40f; cdv = 0x1p40f; }   // (rho + 2^40) * 2^-40 == 1 exactly
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int bin = 2 * wv + u;
                if (bin < (1 << tbits)) {                            // uniform
                    float s, c, e[REPP];
                    sincos_bin(__builtin_fmaf(ts, static_cast<float>(bin) + 0.5f, tm), &s, &c);
#pragma unroll
                    for (int j = 0; j < REPP; j++) e[j] = j < rep ? __builtin_fmaf(lo2f<T>(qraw[j][0]) * a, c, (lo2f<T>(qraw[j][1]) * a) * s) : 0.0f;
                    const uint32_t at = lut + lane * L::PB + ((bin ^ (lane & 15)) << L::SH);
                    lds_store_w<L::W0>(at, e);
                    if constexpr (L::W1 > 0) lds_store_w<L::W1>(at + L::HB, e + 4);
                }
            }
        }
        float cds[16];                                     // of this wavefront's quarter of the pairs, the same in all lanes
#pragma unroll
        for (int d = 0; d < 16; d++) cds[d] = readlane_f(cdv, 16 * quarter + d);
        __syncthreads();
        {
            uint32_t cw[4];
            if constexpr (PK6) {
                // 16 codes of 6 bits, word c: codes 4 c .. 4 c + 3
                const uint32_t x[4] = {ld.code[0], __builtin_amdgcn_alignbit(ld.code[1], ld.code[0], 24), __builtin_amdgcn_alignbit(ld.code[2], ld.code[1], 16), ld.code[2] >> 8};
#pragma unroll
                for (int c = 0; c < 4; c++) cw[c] = (x[c] & 0x3Fu) | ((x[c] << 2) & 0x3F00u) | ((x[c] << 4) & 0x3F0000u) | ((x[c] << 6) & 0x3F000000u);
            } else {
#pragma unroll
                for (int c = 0; c < 4; c++) cw[c] = ld.code[c];
            }
            float s[REPP];
#pragma unroll
            for (int j = 0; j < REPP; j++) s[j] = 0.0f;
            const uint32_t base = lut + quarter * 16 * L::PB;
            static_for<16>([&](auto D) {
                constexpr int d = decltype(D)::value, c = d >> 2, i = d & 3;
                const uint32_t theta = ((cw[c] & tmask) >> (8 * i)) & 0xFFu, rho = (((cw[c] >> tbits) & rmask) >> (8 * i)) & 0xFFu;
                float e[L::WORDS];
                const uint32_t at = base + d * L::PB + ((theta ^ d) << L::SH);
                lds_load_w<L::W0>(at, e);
                if constexpr (L::W1 > 0) lds_load_w<L::W1>(at + L::HB, e + 4);
                const float r = static_cast<float>(rho) + cds[d];
#pragma unroll
                for (int j = 0; j < REPP; j++) s[j] = __builtin_fmaf(e[j], r, s[j]);
                keep_spare_word<REPP>(e);
                if constexpr ((d & 3) == 3) __builtin_amdgcn_sched_barrier(0);     // (four codes' entries in registers at a time)
            });
#pragma unroll
            for (int j = 0; j < REPP; j++) part[quarter][j][kWave * half + lane] = s[j];
        }
        __syncthreads();
        float t[4], w[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int tok = 16 * wv + token_of(i), row = head ? n : 0;
            const float s = (part[0][row][tok] + part[1][row][tok]) + (part[2][row][tok] + part[3][row][tok]);
            t[i] = head && (!has_mask || ld.keep[i] != 0) ? s * scale_log2 : -INFINITY;
        }
        weigh(t, w);
        if constexpr (V4) {
            // weights times the row's scale in half precision, nibbles as subnormals, the zero point's term with the same rounded
            // weights: see softmax_pv_tile_v4
            uint16_t wh[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float scale = lo2f<T>(static_cast<uint16_t>(ld.sz[i][0])), zero = lo2f<T>(static_cast<uint16_t>(ld.sz[i][1]));
                const float scp = scale == 0.0f ? 1.0f : scale;
                wh[i] = f2lo<F16>(w[i] * scp);
                zp = __builtin_fmaf(lo2f<F16>(wh[i]), zero * __builtin_amdgcn_rcpf(scp), zp);
            }
            const uint2 pb = make_uint2(static_cast<uint32_t>(wh[0]) | (static_cast<uint32_t>(wh[1]) << 16), static_cast<uint32_t>(wh[2]) | (static_cast<uint32_t>(wh[3]) << 16));
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const uint32_t by = static_cast<uint32_t>(e >> 1), sel = 0x0c000c00u | ((4u + by) << 16) | by, mask4 = (e & 1) ? 0xf0f0f0f0u : 0x0f0f0f0fu;
                acc[e] = mfma16<F16>(make_uint2(__builtin_amdgcn_perm(ld.v4[1] & mask4, ld.v4[0] & mask4, sel), __builtin_amdgcn_perm(ld.v4[3] & mask4, ld.v4[2] & mask4, sel)), pb, acc[e]);
            }
        } else {
            add_rows(ld.v, w);
        }
        if (grp + 1 < g1) request(ld, grp + 1);
    }
    if constexpr (V4) {                                    // accumulators to real units
        zp += __shfl_xor(zp, 16);
        zp += __shfl_xor(zp, 32);
#pragma unroll
        for (int e = 0; e < 8; e++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[e][i] = __builtin_fmaf(acc[e][i], (e & 1) ? kV4PostOdd : kV4PostEven, zp);
        zp = 0.0f;
    }
    if (nres > 0) {
#pragma unroll
        for (int kb = 0; kb < 4; kb++) qv[kb] = *reinterpret_cast<const uint4*>(qb + (head ? n : 0) * kHeadDim + 32 * kb + 8 * g);
        request_resid(0);
    }
    for (int r = 0; r * kGroup < nres; r++) {
        floatx4 d = {0.0f, 0.0f, 0.0f, 0.0f};              // scores of keys 4 g + i for head n
#pragma unroll
        for (int kb = 0; kb < 4; kb++) {
            d = mfma16<T>(make_uint2(rkeys[kb].x, rkeys[kb].y), make_uint2(qv[kb].x, qv[kb].y), d);
            d = mfma16<T>(make_uint2(rkeys[kb].z, rkeys[kb].w), make_uint2(qv[kb].z, qv[kb].w), d);
        }
        float t[4], w[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const bool keep = head && r * kGroup + 16 * wv + 4 * g + i < nres && (!has_mask || rkeep[i] != 0);
            t[i] = keep ? lo2f<T>(f2lo<T>(d[i])) * scale_log2 : -INFINITY;       // the reference multiplies q.K^T in the model dtype (:79)
        }
        weigh(t, w);
        add_rows(rvals, w);
        if ((r + 1) * kGroup < nres) request_resid(r + 1);
    }

    // ---- the wavefronts' results, as the merge joins slices
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (head) {
        if (g == 0) { ml[wv][n][0] = m; ml[wv][n][1] = l; }
        float* a = reinterpret_cast<float*>(lut_mem) + (wv * REPP + n) * kHeadDim + 32 * g;         // (nobody reads the table any more)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            *reinterpret_cast<float4*>(a + 8 * i) = make_float4(acc[0][i], acc[1][i], acc[2][i], acc[3][i]);
            *reinterpret_cast<float4*>(a + 8 * i + 4) = make_float4(acc[4][i], acc[5][i], acc[6][i], acc[7][i]);
        }
    }
    __syncthreads();
    for (int at = tid; at < rep * kHeadDim; at += kWave * kGroupWaves) {
        const int j = at / kHeadDim, dim = at % kHeadDim;
        float mx = ml[0][j][0], num = 0.0f, den = 0.0f;
#pragma unroll
        for (int k = 1; k < kGroupWaves; k++) mx = fmaxf(mx, ml[k][j][0]);
#pragma unroll
        for (int k = 0; k < kGroupWaves; k++) {
            const float mk = ml[k][j][0], lk = ml[k][j][1];
            // a wavefront without tokens contributes nothing; scores that are all NaN leave no maximum but a sum that is NaN
            const float wk = mk == -INFINITY ? (lk == lk ? 0.0f : lk) : exp2_raw(mk - mx);
            if (wk != 0.0f) {
                den = __builtin_fmaf(wk, lk, den);
                num = __builtin_fmaf(wk, reinterpret_cast<const float*>(lut_mem)[(k * REPP + j) * kHeadDim + dim], num);
            }
        }
        const size_t row = static_cast<size_t>(b) * N + static_cast<size_t>(kvh) * rep_stride + j;
        if (direct_out) {                                  // the only slice of its plane: what the merge would make of it
            direct_out[row * kHeadDim + dim] = f2lo<T>(den > 0.0f ? num / den : (den == den ? 0.0f : den));
        } else {
            float* pw = ws + (row * n_splits + split) * kPartialFloats;
            if (dim == 0) { pw[0] = den == den ? mx : den; pw[1] = den; }       // (the merge passes over a slice without a maximum)
            pw[4 + dim] = num;
        }
    }
}

#pragma clang diagnostic pop

#if PQ_DTYPE == 0
int launch_attn_group_f16(const AttnArgs& a, hipStream_t st) {
    using T = F16;
#else
int launch_attn_group_bf16(const AttnArgs& a, hipStream_t st) {
    using T = BF16;
#endif
    const int rep = a.N / a.Nk;
    const dim3 grid(a.Nk, a.B, a.n_splits), block(kWave * kGroupWaves);
    const float scale_log2 = a.sm_scale * kLog2e;
    const V4Args v4{static_cast<const uint32_t*>(a.v4_codes), static_cast<const uint16_t*>(a.v4_scale),
                    static_cast<const uint16_t*>(a.v4_zero), a.v4_capacity};
#define PQ_LAUNCH_G(REPP, V4, PK6)                                                                                   \
    hipLaunchKernelGGL((attn_group_kernel<T, REPP, V4, PK6>), grid, block, 0, st, (const uint16_t*)a.q, a.codes,     \
                       (const uint16_t*)a.rscale, (const uint16_t*)a.rmn, (const uint16_t*)a.tscale,                 \
                       (const uint16_t*)a.tmn, a.group_capacity, a.n_groups, a.n_groups_per_seq,                     \
                       (const uint16_t*)a.k_resid, a.resid_capacity, a.n_resid, a.n_resid_per_seq,                   \
                       (const uint16_t*)a.v, a.v_capacity, a.mask, a.mask_stride, scale_log2, a.B, a.N, a.Nk, rep,   \
                       a.n_splits, a.min_groups_per_split, a.workspace, v4, rep, a.tbits, static_cast<uint16_t*>(a.out))
#define PQ_LAUNCH_GR(REPP)                                                                                           \
    do {                                                                                                             \
        if (a.v4_codes && a.packed6) PQ_LAUNCH_G(REPP, true, true);                                                  \
        else if (a.v4_codes) PQ_LAUNCH_G(REPP, true, false);                                                         \
        else if (a.packed6) PQ_LAUNCH_G(REPP, false, true);                                                          \
        else PQ_LAUNCH_G(REPP, false, false);                                                                        \
    } while (0)
    switch (rep_pad(rep)) {
        case 1: PQ_LAUNCH_GR(1); break;
        case 2: PQ_LAUNCH_GR(2); break;
        case 4: PQ_LAUNCH_GR(4); break;
        default: PQ_LAUNCH_GR(8); break;
    }
#undef PQ_LAUNCH_GR
#undef PQ_LAUNCH_G
    return static_cast<int>(hipGetLastError());
}

}  // namespace pq
