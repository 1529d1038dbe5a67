// Linear layers of the decode step: y[M, N] = x[M, K] . W[N, K]^T (+ bias) with M <= 16 rows
// (one new token per sequence), the q/k/v, o and MLP projections around the attention call
// (models/modeling_llama_polar.py:47-52, :131 and the decoder layer's MLP, :456-486).
//
// At M <= 16 the product is a stream of the weight matrix through HBM, 2*M flops per weight
// byte: the kernels are laid out for the stream, not for the matrix cores.  Two of them:
// small_m_linear_kernel (any M <= 16, described here) and small_m8_linear_kernel (M <= 8, further
// down: whole-line loads, half the x operand traffic).  A workgroup owns
// 16 output columns (16 rows of W) and splits K over its KSPLIT wavefronts; each wavefront
// keeps two stages of kStage 16-byte loads per lane in flight (ping-pong) and feeds them to
// v_mfma_f32_16x16x32 with the W rows as the A operand and x (rows >= M unused) as the B operand:
// lane l holds W[n0 + l % 16][k + 8 * (l / 16) .. + 8) and x[l % 16][same k], so a 16-byte
// load per lane is one MFMA operand and a wavefront load covers 16 rows x 64 contiguous
// bytes.  The KSPLIT partial 16x16 tiles are added in a fixed order through LDS, so results
// do not depend on scheduling.  x (at most 16 x K) is re-read by every workgroup from L2.
//
// GATED: two weight matrices share the x operand and the epilogue applies
// silu(gate) * up with the eager modules' roundings (gate, up and silu(gate) each rounded
// to the activation dtype), which saves the [M, 2 * N] round trip and one launch.
//
// EPI 0 is the kernel as described (bias, or the gated form); EPI 1 + e is the same stream for one of `heads` independent
// products per launch (blockIdx.y == head, operands `x_head` / N * K / `y_head` elements apart) with epilogue e of
// pq_steps_internal.h: plain, square of relu, times sigmoid(gate), unrounded float32 output, that scaled and soft-capped, or plain rows and
// behind them pairs of a gate's and another row whose results become gelu(gate) * other (small_m8_linear_kernel only; 8 rows, 18720 plain
// rows and 14336 pairs of 4096, in a chain: 65.1 -> 63.3 us, which was a launch of its own that moved 0.9 MB), or added to a residual
// stream with the first half of the norm behind it (ResidualOut; small_m8_linear_kernel only).
#pragma once
#include "pq_device.h"
#include "pq_linear_rules.h"
#include "pq_steps_internal.h"

namespace pq {

typedef float floatx4_l __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_l __attribute__((ext_vector_type(4)));
typedef _Float16 half8_l __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_l __attribute__((ext_vector_type(8)));

template <typename T> __device__ __forceinline__ floatx4_l mfma32(u32x4_l a, u32x4_l b, floatx4_l c);
template <> __device__ __forceinline__ floatx4_l mfma32<F16>(u32x4_l a, u32x4_l b, floatx4_l c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_l, a), __builtin_bit_cast(half8_l, b), c, 0, 0, 0);
}
template <> __device__ __forceinline__ floatx4_l mfma32<BF16>(u32x4_l a, u32x4_l b, floatx4_l c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_l, a), __builtin_bit_cast(bf16x8_l, b), c, 0, 0, 0);
}

template <typename T>
__device__ __forceinline__ float rnd_l(float f) { return lo2f<T>(f2lo<T>(f)); }

// a * u in the dtype.  Half: rounded once, by the instruction that gelu_mul_kernel's product compiles to (through float32 one result in ten
// thousand is the other neighbour of a tie).
template <typename T> __device__ __forceinline__ uint16_t times_rounded(float a, uint16_t u) { return f2lo<T>(a * lo2f<T>(u)); }
template <> __device__ __forceinline__ uint16_t times_rounded<F16>(float a, uint16_t u) {
    uint32_t r;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "=v"(r) : "v"(a), "v"(static_cast<uint32_t>(u)));
    return static_cast<uint16_t>(r);
}

// A norm cut in two between the products around it (pq_linear_residual; pq_gated_normed, pq_qkv_rope_append_normed).  norm(x) W^T is r (x w) W^T with one number
// r = rsqrt(mean x^2 + eps) a row: the product before stores x w, rounded once, and the sum of x^2 over every 16 columns; the product behind
// multiplies its sums by r, which it makes of those.  Every workgroup reads the sums, like x itself.  The norm had a launch of its own, of
// which nothing was work.  8 rows of 4096, products and norms in a chain of captured calls (us): o projection, norm, gate and up of 14336 50.3
// -> 49.0, down, norm, q, k and v 39.7 -> 37.2; each by itself norm 3.2, o 9.0 -> 9.5, gate and up 38.9 -> 39.9, down 22.8 -> 23.3, q, k and
// v 14.8 -> 15.0.  A step with two norms of the first kind and one of the second 289.3 -> 284.3.  Widths 256 to 8192, 1 to 8 rows: 1.00 to 1.21
// times as fast; from 6 rows on 28672 -> 8192 -> q, k, v takes as long either way.
struct NormedRows {
    const float* part;          // [M, n]: sums of squares of a row's 16 n elements
    int n;
    float eps;
};
struct ResidualOut {
    uint16_t* x;                // [M, N]: the residual stream; the product is added to it
    const uint16_t* norm_w;     // [N]
    uint16_t* xw;               // [M, N]
    float* part;                // [M, N / 16]
};
// The rows' r, by all threads of a workgroup, 8 KSPLIT to a row: requested behind the first weights and made while the next are on their way
// (behind the last ones they hold registers through the loop, and the fewer workgroups a unit has then cost as much).
constexpr int kNormedLoads = 2;
template <int KSPLIT>
struct RowScale {
    static constexpr int kThreads = 8 * KSPLIT;
    float4 v[kNormedLoads];
    __device__ __forceinline__ void load(const NormedRows& nr, int M) {
        const int row = threadIdx.x / kThreads, j = threadIdx.x % kThreads;
        const float* p = nr.part + static_cast<size_t>(row < M ? row : 0) * nr.n;
#pragma unroll
        for (int i = 0; i < kNormedLoads; i++) {
            const int at = (i * kThreads + j) * 4;
            v[i] = *reinterpret_cast<const float4*>(p + (at < nr.n ? at : 0));
        }
    }
    __device__ __forceinline__ void store(const NormedRows& nr, float* r) const {
        const int j = threadIdx.x % kThreads;
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < kNormedLoads; i++) s += (i * kThreads + j) * 4 < nr.n ? (v[i].x + v[i].y) + (v[i].z + v[i].w) : 0.0f;
#pragma unroll
        for (int o = kThreads / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (j == 0) r[threadIdx.x / kThreads] = rsqrtf(s / static_cast<float>(16 * nr.n) + nr.eps);
    }
};

struct HeadEpi {
    int64_t x_head, w_head, y_head;
    const uint16_t* gate;
    int64_t gate_row;
    float scale, cap;
    int32_t* advance;
    // kEpiGeluPairs: workgroups from this one on take as many rows of the gate as of those `pair_rows` further, and store at z
    int pair_from, pair_rows;
    uint16_t* z;
    int64_t z_row;
    NormedRows normed;           // of x (NORMED)
    ResidualOut res;             // kEpiResidual
};

// of logits: a counter that nothing in this launch reads is raised by its first thread
template <int EPI>
__device__ __forceinline__ void advance_once(const HeadEpi& he) {
    if constexpr (EPI == 1 + kEpiLogits)
        if (he.advance && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *he.advance += 1;
}

// stores outputs y[r][n .. n + 3] (n: column inside the head) through epilogue EPI - 1
template <typename T, int EPI>
__device__ __forceinline__ void store_head(const float (&s)[4], uint16_t* y, int64_t y_stride, int r, int n, int N, const HeadEpi& he) {
    const size_t o = static_cast<size_t>(r) * y_stride + blockIdx.y * he.y_head + n;
    if constexpr (EPI == 1 + kEpiF32 || EPI == 1 + kEpiLogits) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = s[i];
            if constexpr (EPI == 1 + kEpiLogits) {
                v[i] *= he.scale;
                if (he.cap > 0.0f) v[i] = he.cap * tanhf(v[i] / he.cap);
            }
        }
        *reinterpret_cast<float4*>(reinterpret_cast<float*>(y) + o) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
        uint16_t out[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float v = s[i];
            if constexpr (EPI == 1 + kEpiReluSq) {
                v = fmaxf(v, 0.0f);
                v = v * v;
            }
            if constexpr (EPI == 1 + kEpiSigmoidGate)
                v = v / (1.0f + __expf(-lo2f<T>(he.gate[static_cast<size_t>(r) * he.gate_row + static_cast<size_t>(blockIdx.y) * N + n + i])));
            out[i] = f2lo<T>(v);
        }
        *reinterpret_cast<uint2*>(y + o) = make_uint2(static_cast<uint32_t>(out[0]) | (static_cast<uint32_t>(out[1]) << 16),
                                                      static_cast<uint32_t>(out[2]) | (static_cast<uint32_t>(out[3]) << 16));
    }
}

template <bool GATED, int kStage>
struct StageT {
    u32x4_l w[kStage], x[kStage], u[GATED ? kStage : 1];
};

template <typename T, int KSPLIT, bool GATED, int kStage, int EPI = 0>
__global__ __launch_bounds__(kWave * KSPLIT) void small_m_linear_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* __restrict__ w, const uint16_t* __restrict__ w_up,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ y, int64_t y_stride, int M, int K, HeadEpi he) {
    advance_once<EPI>(he);
    if constexpr (EPI != 0) {
        x += blockIdx.y * he.x_head;
        w += blockIdx.y * he.w_head;
    }
    __shared__ float part[KSPLIT][GATED ? 2 : 1][4][kWave];
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16;
    const int klen = K / KSPLIT, steps = klen / 32;
    const int m = r < M ? r : 0;                           // tile columns >= M repeat row 0 and are never stored
    const size_t koff = static_cast<size_t>(wv) * klen + 8 * g;
    const uint16_t* wp = w + static_cast<size_t>(n0 + r) * K + koff;
    const uint16_t* up = GATED ? w_up + static_cast<size_t>(n0 + r) * K + koff : nullptr;
    const uint16_t* xp = x + static_cast<size_t>(m) * x_stride + koff;

    floatx4_l acc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, acu[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
    // No branch may sit between a stage's loads and the MFMAs of the other stage: at a join the
    // compiler has to wait for every outstanding load, which would serialize the two stages.  So
    // whole stages run in a branch-free ping-pong loop, and only the tail is predicated.
    auto load = [&](StageT<GATED, kStage>& st, int s0) {
        static_for<kStage>([&](auto U) {
            constexpr int u = decltype(U)::value;
            st.w[u] = *reinterpret_cast<const u32x4_l*>(wp + (s0 + u) * 32);
            if constexpr (GATED) st.u[u] = *reinterpret_cast<const u32x4_l*>(up + (s0 + u) * 32);
            st.x[u] = *reinterpret_cast<const u32x4_l*>(xp + (s0 + u) * 32);
        });
    };
    auto compute = [&](const StageT<GATED, kStage>& st) {
        static_for<kStage>([&](auto U) {
            constexpr int u = decltype(U)::value;
            acc[u & 1] = mfma32<T>(st.w[u], st.x[u], acc[u & 1]);
            if constexpr (GATED) acu[u & 1] = mfma32<T>(st.u[u], st.x[u], acu[u & 1]);
        });
    };
    const int full = steps / kStage;          // whole stages
    if (full > 0) {
        StageT<GATED, kStage> sa, sb;
        load(sa, 0);
        int st = 0;
        while (st + 2 < full) {
            load(sb, (st + 1) * kStage);
            compute(sa);
            load(sa, (st + 2) * kStage);
            compute(sb);
            st += 2;
        }
        if (full - st == 2) {
            load(sb, (st + 1) * kStage);
            compute(sa);
            compute(sb);
        } else {
            compute(sa);
        }
    }
    for (int s1 = full * kStage; s1 < steps; s1++) {      // fewer than kStage steps left
        const u32x4_l wv1 = *reinterpret_cast<const u32x4_l*>(wp + s1 * 32);
        const u32x4_l xv1 = *reinterpret_cast<const u32x4_l*>(xp + s1 * 32);
        acc[0] = mfma32<T>(wv1, xv1, acc[0]);
        if constexpr (GATED) acu[0] = mfma32<T>(*reinterpret_cast<const u32x4_l*>(up + s1 * 32), xv1, acu[0]);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        part[wv][0][i][lane] = acc[0][i] + acc[1][i];
        if constexpr (GATED) part[wv][1][i][lane] = acu[0][i] + acu[1][i];
    }
    __syncthreads();
    if (wv != 0 || r >= M) return;
    // the MFMA result layout: lane (r, g) holds tile rows 4g + i (i < 4) of tile column r = outputs y[r][n0 + 4g + i]
    if constexpr (EPI != 0) {
        float s4[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s4[i] = part[0][0][i][lane];
#pragma unroll
            for (int k = 1; k < KSPLIT; k++) s4[i] += part[k][0][i][lane];
        }
        store_head<T, EPI>(s4, y, y_stride, r, n0 + 4 * g, static_cast<int>(gridDim.x) * 16, he);
        return;
    }
    uint16_t out[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float s = part[0][0][i][lane];
#pragma unroll
        for (int k = 1; k < KSPLIT; k++) s += part[k][0][i][lane];
        if constexpr (GATED) {
            float t = part[0][1][i][lane];
#pragma unroll
            for (int k = 1; k < KSPLIT; k++) t += part[k][1][i][lane];
            const float gv = rnd_l<T>(s), uv = rnd_l<T>(t);
            const float a = rnd_l<T>(gv / (1.0f + __expf(-gv)));
            out[i] = f2lo<T>(a * uv);
        } else {
            if (bias) s += lo2f<T>(bias[n0 + 4 * g + i]);
            out[i] = f2lo<T>(s);
        }
    }
    *reinterpret_cast<uint2*>(y + static_cast<size_t>(r) * y_stride + n0 + 4 * g) =
        make_uint2(static_cast<uint32_t>(out[0]) | (static_cast<uint32_t>(out[1]) << 16),
                   static_cast<uint32_t>(out[2]) | (static_cast<uint32_t>(out[3]) << 16));
}

// M <= 8: each 16 x 16 MFMA tile is used as two 8 x 8 tiles on its diagonal.  Tile rows 0-7 are 8 rows
// of W over the first 32 of a 64-wide k-step, tile rows 8-15 the SAME 8 rows over the second 32; tile
// columns 0-7 are the rows of x over the first 32, columns 8-15 over the second 32.  Then
// y[m][n] = C[n][m] + C[n + 8][m + 8] and the off-diagonal quarters are ignored.  No lane loads a
// duplicate row of x, a wavefront load of W covers 8 rows x 128 contiguous bytes (whole cache lines,
// which is what lets the weight stream carry the non-temporal hint: with half lines the hint drops a
// line before its second half is asked for), and the workgroup's 8 NT rows of W are NT such tiles that
// share one x operand.  (Which NT: pq_linear_rules.h.)
template <bool GATED, int NT, int kStage>
struct Stage8T {
    u32x4_l w[NT][kStage], x[kStage], u[GATED ? NT : 1][GATED ? kStage : 1];
};

template <typename T, int KSPLIT, bool GATED, int kStage, int EPI = 0, int NT = 2, bool NORMED = false>
__global__ __launch_bounds__(kWave * KSPLIT) void small_m8_linear_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* __restrict__ w, const uint16_t* __restrict__ w_up,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ y, int64_t y_stride, int M, int K, HeadEpi he) {
    advance_once<EPI>(he);
    if constexpr (EPI != 0) {
        x += blockIdx.y * he.x_head;
        w += blockIdx.y * he.w_head;
    }
    __shared__ float part[KSPLIT][(GATED ? 2 : 1) * NT][4][kWave];
    __shared__ float row_scale[NORMED ? 8 : 1];
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    const int r = lane & 15, g = lane >> 4;
    const int row = r & 7, chunk = (r >> 3) * 4 + g;       // W row inside an 8-row tile == x row; 16-byte piece of the step
    constexpr bool kGelu = EPI == 1 + kEpiGeluPairs, kResidual = EPI == 1 + kEpiResidual;
    const bool pairs = kGelu && static_cast<int>(blockIdx.x) >= he.pair_from;
    // (a workgroup of pairs: the first half of its tiles are rows of the gate, the second those they meet)
    const int n0 = pairs ? (he.pair_from + static_cast<int>(blockIdx.x)) * 4 * NT : blockIdx.x * 8 * NT;
    const size_t apart = pairs ? static_cast<size_t>(he.pair_rows - 4 * NT) * K : 0;
    const int klen = K / KSPLIT, steps = klen / 64;
    const int m = row < M ? row : 0;                       // tile columns >= M repeat row 0 and are never stored
    const size_t koff = static_cast<size_t>(wv) * klen + 8 * chunk;
    const uint16_t* wp = w + static_cast<size_t>(n0 + row) * K + koff;
    const uint16_t* up = GATED ? w_up + static_cast<size_t>(n0 + row) * K + koff : nullptr;
    const uint16_t* xp = x + static_cast<size_t>(m) * x_stride + koff;
    const size_t tile = static_cast<size_t>(8) * K;

    // kResidual: the first wavefront stores, a lane the four columns 4 (g & 1) of tile (r / 8) + 2 (g / 2) of its row, and has requested
    // what they are added to and multiplied by
    const int width = static_cast<int>(gridDim.x) * 8 * NT, mine = (r >> 3) + 2 * (g >> 1), rn = n0 + 8 * (mine < NT ? mine : 0) + 4 * (g & 1);
    uint2 x_old = {0, 0}, norm_w = {0, 0};
    if constexpr (kResidual) {
        x_old = *reinterpret_cast<const uint2*>(he.res.x + static_cast<size_t>(m) * width + rn);
        norm_w = *reinterpret_cast<const uint2*>(he.res.norm_w + rn);
    }

    RowScale<KSPLIT> scale;
    floatx4_l acc[NT], acu[GATED ? NT : 1];
    static_for<NT>([&](auto I) {
        acc[I] = floatx4_l{0, 0, 0, 0};
        if constexpr (GATED) acu[I] = floatx4_l{0, 0, 0, 0};
    });
    auto ldw = [](const uint16_t* p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4_l*>(p)); };
    auto load = [&](Stage8T<GATED, NT, kStage>& st, int s0) {      // branch-free, see small_m_linear_kernel
        static_for<kStage>([&](auto U) {
            constexpr int u = decltype(U)::value;
            static_for<NT>([&](auto I) { st.w[I][u] = ldw((kGelu && I >= NT / 2 ? wp + apart : wp) + I * tile + (s0 + u) * 64); });
            if constexpr (GATED) static_for<NT>([&](auto I) { st.u[I][u] = ldw(up + I * tile + (s0 + u) * 64); });
            st.x[u] = *reinterpret_cast<const u32x4_l*>(xp + (s0 + u) * 64);
        });
    };
    auto compute = [&](const Stage8T<GATED, NT, kStage>& st) {
        static_for<kStage>([&](auto U) {
            constexpr int u = decltype(U)::value;
            static_for<NT>([&](auto I) {
                acc[I] = mfma32<T>(st.w[I][u], st.x[u], acc[I]);
                if constexpr (GATED) acu[I] = mfma32<T>(st.u[I][u], st.x[u], acu[I]);
            });
        });
    };
    const int full = steps / kStage;
    if (full > 0) {
        Stage8T<GATED, NT, kStage> sa, sb;
        load(sa, 0);
        if constexpr (NORMED) scale.load(he.normed, M);
        int st = 0;
        if constexpr (NORMED) {
            if (full > 2) {                        // (the loop's first trip, with the rows' factors in it)
                load(sb, kStage);
                __builtin_amdgcn_sched_barrier(0);
                compute(sa);
                load(sa, 2 * kStage);
                __builtin_amdgcn_sched_barrier(0);
                scale.store(he.normed, row_scale);
                __builtin_amdgcn_sched_barrier(0);
                compute(sb);
                st = 2;
            } else {
                scale.store(he.normed, row_scale);
            }
        }
        while (st + 2 < full) {
            load(sb, (st + 1) * kStage);
            compute(sa);
            load(sa, (st + 2) * kStage);
            compute(sb);
            st += 2;
        }
        if (full - st == 2) {
            load(sb, (st + 1) * kStage);
            compute(sa);
            compute(sb);
        } else {
            compute(sa);
        }
    }
    for (int s1 = full * kStage; s1 < steps; s1++) {
        const u32x4_l xv1 = *reinterpret_cast<const u32x4_l*>(xp + s1 * 64);
        static_for<NT>([&](auto I) {
            acc[I] = mfma32<T>(ldw((kGelu && I >= NT / 2 ? wp + apart : wp) + I * tile + s1 * 64), xv1, acc[I]);
            if constexpr (GATED) acu[I] = mfma32<T>(ldw(up + I * tile + s1 * 64), xv1, acu[I]);
        });
    }
    static_for<NT>([&](auto I) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            part[wv][I][i][lane] = acc[I][i];
            if constexpr (GATED) part[wv][NT + I][i][lane] = acu[I][i];
        }
    });
    __syncthreads();
    if constexpr (kResidual) {
        static_assert(NT <= 4, "a lane for every four columns");
        if (wv != 0) return;
        const int at = row + 16 * (g & 1), tile_ = mine < NT ? mine : 0;
        uint16_t xs[4], us[4];
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < KSPLIT; k++) s += part[k][tile_][i][at] + part[k][tile_][i][at + 40];
            const uint32_t xw = i < 2 ? x_old.x : x_old.y, ww = i < 2 ? norm_w.x : norm_w.y;
            if (bias) s += lo2f<T>(bias[rn + i]);
            xs[i] = f2lo<T>(lo2f<T>(static_cast<uint16_t>(i & 1 ? xw >> 16 : xw)) + rnd_l<T>(s));
            const float xv = lo2f<T>(xs[i]);
            us[i] = f2lo<T>(xv * lo2f<T>(static_cast<uint16_t>(i & 1 ? ww >> 16 : ww)));
            ss = __builtin_fmaf(xv, xv, ss);
        }
        ss += __shfl_xor(ss, 16);                            // the row's other four columns of the tile, then the other tile of 16 columns
        ss += __shfl_xor(ss, 8);
        if (row >= M || mine >= NT) return;
        const size_t o = static_cast<size_t>(row) * width + rn;
        *reinterpret_cast<uint2*>(he.res.x + o) = make_uint2(xs[0] | (static_cast<uint32_t>(xs[1]) << 16), xs[2] | (static_cast<uint32_t>(xs[3]) << 16));
        *reinterpret_cast<uint2*>(he.res.xw + o) = make_uint2(us[0] | (static_cast<uint32_t>(us[1]) << 16), us[2] | (static_cast<uint32_t>(us[3]) << 16));
        if (r < 8 && (g & 1) == 0) he.res.part[static_cast<size_t>(row) * (width / 16) + rn / 16] = ss;
        return;
    }
    // lane (r < 8, g < 2) owns outputs y[r][n0 + 8h + 4g + i] (h: which 8-row tile), each the sum of the tile's
    // entry (row 4g + i, column r) and its diagonal partner (row + 8, column + 8), which lane + 40 holds
    if (r >= 8 || r >= M || g >= 2) return;
    for (int h = wv; h < NT; h += KSPLIT) {
        if constexpr (kGelu) {
            if (pairs) {
                if (h >= NT / 2) continue;
                uint16_t out[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float s = 0.0f, t = 0.0f;
#pragma unroll
                    for (int k = 0; k < KSPLIT; k++) {
                        s += part[k][h][i][lane] + part[k][h][i][lane + 40];
                        t += part[k][h + NT / 2][i][lane] + part[k][h + NT / 2][i][lane + 40];
                    }
                    out[i] = times_rounded<T>(gelu_tanh(rnd_l<T>(s)), f2lo<T>(t));     // (both rounded as a product of its own leaves them)
                }
                const int c = (static_cast<int>(blockIdx.x) - he.pair_from) * 4 * NT + 8 * h + 4 * g;
                *reinterpret_cast<uint2*>(he.z + static_cast<size_t>(r) * he.z_row + c) =
                    make_uint2(static_cast<uint32_t>(out[0]) | (static_cast<uint32_t>(out[1]) << 16), static_cast<uint32_t>(out[2]) | (static_cast<uint32_t>(out[3]) << 16));
                continue;
            }
        }
        if constexpr (EPI != 0) {
            float s4[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                s4[i] = 0.0f;
#pragma unroll
                for (int k = 0; k < KSPLIT; k++) s4[i] += part[k][h][i][lane] + part[k][h][i][lane + 40];
            }
            store_head<T, EPI>(s4, y, y_stride, r, n0 + 8 * h + 4 * g, static_cast<int>(gridDim.x) * 8 * NT, he);
            continue;
        }
        uint16_t out[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float s = 0.0f, t = 0.0f;
#pragma unroll
            for (int k = 0; k < KSPLIT; k++) {
                s += part[k][h][i][lane] + part[k][h][i][lane + 40];
                if constexpr (GATED) t += part[k][NT + h][i][lane] + part[k][NT + h][i][lane + 40];
            }
            if constexpr (NORMED) { s *= row_scale[r]; t *= row_scale[r]; }
            if constexpr (GATED) {
                const float gv = rnd_l<T>(s), uv = rnd_l<T>(t);
                const float a = rnd_l<T>(gv / (1.0f + __expf(-gv)));
                out[i] = f2lo<T>(a * uv);
            } else {
                if (bias) s += lo2f<T>(bias[n0 + 8 * h + 4 * g + i]);
                out[i] = f2lo<T>(s);
            }
        }
        *reinterpret_cast<uint2*>(y + static_cast<size_t>(r) * y_stride + n0 + 8 * h + 4 * g) =
            make_uint2(static_cast<uint32_t>(out[0]) | (static_cast<uint32_t>(out[1]) << 16),
                       static_cast<uint32_t>(out[2]) | (static_cast<uint32_t>(out[3]) << 16));
    }
}

}  // namespace pq
