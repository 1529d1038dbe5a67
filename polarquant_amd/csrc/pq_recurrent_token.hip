// One token a sequence through a mixer with a matrix-valued state, from its columns of the input product to its columns of the output
// product's operand: what delta_prep_kernel or memory_gates_kernel, scan_kernel and head_norm_gate_kernel (pq_recurrent.hip) do for any
// number of tokens, the same operations in the same order; for the delta rule also the two low-rank products before them, whose sums are
// taken in another order (8 elements a lane, then 16 lanes) and rounded to the dtype like theirs.
//
// A workgroup per (head, sequence): the norm of what is read out runs over a head, so its state is not cut up.  What bounds it is the
// stream of the state in and out; everything else is a few hundred elements that each of the separate launches fetched, wrote and waited
// for.  So the state is requested first, and the rest is made while it is on its way: 16 lanes hold a column (a row of dim floats in
// memory), 8 rows each in quads, the other operands go through LDS.
// In a chain of captured calls, bfloat16, against the separate launches (us): delta rule, 32 heads of 128 x 128, ranks 128, 1 / 8 / 64
// sequences 6.4 / 9.4 / 54.4 against 13.3 / 18.7 / 68.0; matrix memory, 16 heads of 128 x 256, 5.2 / 7.2 / 43.3 against 7.5 / 12.0 / 47.2.
// (8 sequences: 34 MB of state in and out, 6.7 us at 5 TB/s.)  Very many heads times sequences go through the separate launches: recurrent_ops.py.
#include "pq_recurrent_device.h"
#include "pq_recurrent_internal.h"

namespace pq {

constexpr int kTokenRows = 8;                        // of a column, a lane's: dim up to 128

// the state's column at p, 16 lanes' quads
__device__ __forceinline__ void load_column(const float* p, int part, int dim, float (&s)[kTokenRows]) {
#pragma unroll
    for (int c = 0; c < kTokenRows / 4; c++) {
        const int r = c * 64 + part * 4;
        const float4 w = *reinterpret_cast<const float4*>(p + (r < dim ? r : 0));
        s[4 * c] = r < dim ? w.x : 0.0f; s[4 * c + 1] = r < dim ? w.y : 0.0f; s[4 * c + 2] = r < dim ? w.z : 0.0f; s[4 * c + 3] = r < dim ? w.w : 0.0f;
    }
}
__device__ __forceinline__ void store_column(float* p, int part, int dim, const float (&s)[kTokenRows]) {
#pragma unroll
    for (int c = 0; c < kTokenRows / 4; c++) {
        const int r = c * 64 + part * 4;
        if (r < dim) *reinterpret_cast<float4*>(p + r) = make_float4(s[4 * c], s[4 * c + 1], s[4 * c + 2], s[4 * c + 3]);
    }
}
// this lane's rows of a vector in LDS (zero past dim)
__device__ __forceinline__ void rows_of(const float* v, int part, float (&o)[kTokenRows]) {
#pragma unroll
    for (int c = 0; c < kTokenRows / 4; c++) {
        const float4 w = *reinterpret_cast<const float4*>(v + c * 64 + part * 4);
        o[4 * c] = w.x; o[4 * c + 1] = w.y; o[4 * c + 2] = w.z; o[4 * c + 3] = w.w;
    }
}

// head_norm_gate_kernel's row, by one wavefront, four channels a lane: o [vdim] in LDS
template <typename T>
__device__ __forceinline__ void token_read_out(const float* o, float den, int lane, int vdim, const float (&gate)[4], const float (&w)[4],
                                               float out_scale, float eps, void* out) {
    const int c = 4 * lane;
    float x[4], ss = 0.0f;
    const float div = 1.0f / den;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        x[j] = c < vdim ? o[c + j] : 0.0f;
        const float y = x[j] * div;
        ss = __builtin_fmaf(y, y, ss);
    }
    ss = row16_sum(ss);
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    const float r = div * out_scale / sqrtf(ss / static_cast<float>(vdim) + eps);
#pragma unroll
    for (int j = 0; j < 4; j++) x[j] = x[j] * r * w[j] * sigmoid(gate[j]);
    if (c < vdim) stv<T, 4>(out, c, x);
}

// ---- gated delta rule ----------------------------------------------------------------------------------------------------
// 512 threads, four columns to 16 lanes (vdim up to 128).  The low-rank products are spread over all of them, 16 lanes to a row of the
// weights; wavefronts 0 to 2 make the convolved q, k and v of the head, two channels a lane, and shift their rows of the state.
constexpr int kDeltaColumns = 4, kDeltaThreads = 512, kDeltaTaps = 4;

template <typename T>
__global__ __launch_bounds__(kDeltaThreads) void delta_token_kernel(DeltaTokenArgs a) {
    __shared__ __attribute__((aligned(16))) float sq[128], sk[128], sv[128], sg[128], so[128], sgate[128], scalars[3];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, part = lane & 15, grp = tid >> 4, h = blockIdx.x, b = blockIdx.y;
    const int H = a.H, dim = a.dim, vdim = a.vdim, taps = a.taps;
    constexpr int kGroups = kDeltaThreads / 16;
    float* state = a.state + (static_cast<size_t>(b) * H + h) * vdim * dim;
    float S[kDeltaColumns][kTokenRows];
#pragma unroll
    for (int j = 0; j < kDeltaColumns; j++) {
        const int col = grp + kGroups * j;
        load_column(state + static_cast<size_t>(col < vdim ? col : 0) * dim, part, dim, S[j]);
    }
    // the decays' and the gate's products: rows grp + 32 j of the head, 8 of the rank's elements a lane
    uint4 wa[4], wg[4], xa = make_uint4(0, 0, 0, 0), xg = xa;
    const int piece = 8 * part;
    if (piece < a.a_rank) xa = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.xa) + b * a.p_row + piece);
    if (piece < a.g_rank) xg = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.xg) + b * a.p_row + piece);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int r = grp + kGroups * j;
        wa[j] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.wa) + static_cast<size_t>(h * dim + (r < dim ? r : 0)) * a.a_rank + (piece < a.a_rank ? piece : 0));
        wg[j] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.wg) + static_cast<size_t>(h * vdim + (r < vdim ? r : 0)) * a.g_rank + (piece < a.g_rank ? piece : 0));
    }
    const bool real = !a.start || a.start[b] - (a.pos_dev ? *a.pos_dev : a.pos) <= 0;            // (padding otherwise)
    if (wv < 3) {
        const int width = wv == 2 ? vdim : dim, c = 2 * lane, all = 2 * H * dim + H * vdim, at = wv * H * dim + h * width;
        const bool own = c < width;
        const int ch = own ? c : 0;
        const uint16_t* x = static_cast<const uint16_t*>(wv == 0 ? a.q : wv == 1 ? a.k : a.v) + b * a.p_row + static_cast<size_t>(h) * width + ch;
        const uint16_t* w = static_cast<const uint16_t*>(wv == 0 ? a.w_q : wv == 1 ? a.w_k : a.w_v) + (static_cast<size_t>(h) * width + ch) * taps;
        float* conv = taps > 1 ? a.conv + static_cast<size_t>(b) * (taps - 1) * all + at + ch : nullptr;
        const int shift = kDeltaTaps - taps;                 // a shorter filter: zero taps in front
        float cw[kDeltaTaps][2], hist[kDeltaTaps][2];
#pragma unroll
        for (int j = 0; j < kDeltaTaps; j++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int tap = j - shift;
                cw[j][i] = tap >= 0 ? lo2f<T>(w[i * taps + tap]) : 0.0f;
                hist[j][i] = j == kDeltaTaps - 1 ? (real ? lo2f<T>(x[i]) : 0.0f) : tap >= 0 ? conv[static_cast<size_t>(tap) * all + i] : 0.0f;
            }
        float y[2], ss = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < kDeltaTaps; j++) s = __builtin_fmaf(cw[j][i], hist[j][i], s);
            y[i] = lo2f<T>(f2lo<T>(s * sigmoid(s)));          // (what the other launches pass on is rounded)
            ss = own ? __builtin_fmaf(y[i], y[i], ss) : ss;
        }
        float* dst = wv == 0 ? sq : wv == 1 ? sk : sv;
        dst[c] = own ? y[0] : 0.0f;
        dst[c + 1] = own ? y[1] : 0.0f;
        if (wv < 2) {
            ss = wave_sum(ss);
            if (lane == 0) scalars[wv] = (wv == 0 ? 1.0f / sqrtf(static_cast<float>(dim)) : 1.0f) / sqrtf(ss + 1e-6f);
        }
#pragma unroll
        for (int j = 1; j < kDeltaTaps; j++)
            if (j - shift - 1 >= 0 && own) *reinterpret_cast<float2*>(conv + static_cast<size_t>(j - shift - 1) * all) = make_float2(hist[j][0], hist[j][1]);
    } else if (wv == 3 && lane == 0) {
        scalars[2] = sigmoid(lo2f<T>(static_cast<const uint16_t*>(a.b)[b * a.p_row + h]));
    }
    {
        auto dot = [](const uint4& w, const uint4& x) {
            const uint32_t ww[4] = {w.x, w.y, w.z, w.w}, xx[4] = {x.x, x.y, x.z, x.w};
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                s = __builtin_fmaf(lo2f<T>(static_cast<uint16_t>(ww[i])), lo2f<T>(static_cast<uint16_t>(xx[i])), s);
                s = __builtin_fmaf(lo2f<T>(static_cast<uint16_t>(ww[i] >> 16)), lo2f<T>(static_cast<uint16_t>(xx[i] >> 16)), s);
            }
            return row16_sum(s);
        };
        float da[4], dg[4];
#pragma unroll
        for (int j = 0; j < 4; j++) { da[j] = dot(wa[j], xa); dg[j] = dot(wg[j], xg); }
        // lane j of the 16 finishes row grp + 32 j
        if (part < 4) {
            const float pa = part == 0 ? da[0] : part == 1 ? da[1] : part == 2 ? da[2] : da[3], pg = part == 0 ? dg[0] : part == 1 ? dg[1] : part == 2 ? dg[2] : dg[3];
            const int r = grp + kGroups * part;
            const float rate = -expf(lo2f<T>(static_cast<const uint16_t*>(a.A_log)[h]));
            const float bias = lo2f<T>(static_cast<const uint16_t*>(a.dt_bias)[static_cast<size_t>(h) * dim + (r < dim ? r : 0)]);
            sg[r] = exp_fast(rate * softplus(lo2f<T>(f2lo<T>(pa)) + bias));
            sgate[r] = lo2f<T>(f2lo<T>(pg));
        }
    }
    __syncthreads();
    float q[kTokenRows], k[kTokenRows], g[kTokenRows], e2 = 0.0f;
    rows_of(sq, part, q);
    rows_of(sk, part, k);
    rows_of(sg, part, g);
    const float q_inv = scalars[0], k_inv = scalars[1], beta = scalars[2];
#pragma unroll
    for (int i = 0; i < kTokenRows; i++) {
        k[i] *= k_inv;
        q[i] *= q_inv;
        e2 = __builtin_fmaf(k[i], q[i], e2);
    }
    e2 = row16_sum(e2);
#pragma unroll
    for (int j = 0; j < kDeltaColumns; j++) {
        const int col = grp + kGroups * j;
        float e0 = 0.0f, e1 = 0.0f;
#pragma unroll
        for (int i = 0; i < kTokenRows; i++) {
            S[j][i] *= g[i];
            e0 = __builtin_fmaf(S[j][i], k[i], e0);
            e1 = __builtin_fmaf(S[j][i], q[i], e1);
        }
        e0 = row16_sum(e0);
        e1 = row16_sum(e1);
        const float u = beta * (sv[col] - e0);
#pragma unroll
        for (int i = 0; i < kTokenRows; i++) S[j][i] = __builtin_fmaf(k[i], u, S[j][i]);
        if (real && col < vdim) store_column(state + static_cast<size_t>(col) * dim, part, dim, S[j]);
        if (part == 0) so[col] = real ? __builtin_fmaf(e2, u, e1) : 0.0f;
    }
    __syncthreads();
    if (wv == 0) {
        const int c = 4 * lane < vdim ? 4 * lane : 0;
        float gate[4], w[4];
#pragma unroll
        for (int j = 0; j < 4; j++) gate[j] = sgate[c + j];
        ldv<T, 4>(a.norm, c, w);
        token_read_out<T>(so, 1.0f, lane, vdim, gate, w, a.out_scale, a.eps, static_cast<uint16_t*>(a.out) + b * a.out_row + static_cast<size_t>(h) * vdim);
    }
}

int launch_delta_token(const DeltaTokenArgs& a, int dtype, hipStream_t st) {
    dim3 grid(static_cast<unsigned>(a.H), static_cast<unsigned>(a.B)), block(kDeltaThreads);
    if (dtype == 0) hipLaunchKernelGGL(delta_token_kernel<F16>, grid, block, 0, st, a);
    else hipLaunchKernelGGL(delta_token_kernel<BF16>, grid, block, 0, st, a);
    return static_cast<int>(hipGetLastError());
}

// ---- matrix memory -------------------------------------------------------------------------------------------------------
// 1024 threads, four columns to 16 lanes (vdim up to 256), the normalizer's column by the first 16 lanes behind them.  One lane makes the
// gates while the state is on its way.
constexpr int kMemoryColumns = 4, kMemoryThreads = 1024;

template <typename T>
__global__ __launch_bounds__(kMemoryThreads) void memory_token_kernel(MemoryTokenArgs a) {
    __shared__ __attribute__((aligned(16))) float so[256], scalars[3];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, part = lane & 15, grp = tid >> 4, h = blockIdx.x, b = blockIdx.y;
    const int H = a.H, dim = a.dim, vdim = a.vdim, columns = vdim + 1;
    constexpr int kGroups = kMemoryThreads / 16;
    float* state = a.state + (static_cast<size_t>(b) * H + h) * columns * dim;
    float S[kMemoryColumns][kTokenRows], N[kTokenRows], v[kMemoryColumns];
    const int64_t row = b * a.p_row;
    const uint16_t* vp = static_cast<const uint16_t*>(a.v) + row + static_cast<size_t>(h) * vdim;
#pragma unroll
    for (int j = 0; j < kMemoryColumns; j++) {
        const int col = grp + kGroups * j;
        load_column(state + static_cast<size_t>(col < vdim ? col : 0) * dim, part, dim, S[j]);
        v[j] = lo2f<T>(vp[col < vdim ? col : 0]);
    }
    if (wv == 0) load_column(state + static_cast<size_t>(vdim) * dim, part, dim, N);
    float q[kTokenRows], k[kTokenRows], gate[4], w[4];
#pragma unroll
    for (int c = 0; c < kTokenRows / 4; c++) {
        const int r = c * 64 + part * 4, at = r < dim ? r : 0;
        float q4[4], k4[4];
        ldv<T, 4>(a.q, static_cast<size_t>(row) + static_cast<size_t>(h) * dim + at, q4);
        ldv<T, 4>(a.k, static_cast<size_t>(row) + static_cast<size_t>(h) * dim + at, k4);
#pragma unroll
        for (int i = 0; i < 4; i++) { q[4 * c + i] = r < dim ? q4[i] : 0.0f; k[4 * c + i] = r < dim ? k4[i] : 0.0f; }
    }
    const bool real = !a.start || a.start[b] - (a.pos_dev ? *a.pos_dev : a.pos) <= 0;
    const int copies = (vdim + 16) / 16;
    float* mp = a.m + (static_cast<size_t>(b) * H + h) * copies;
    if (wv == 0) {
        const int c = 4 * lane < vdim ? 4 * lane : 0;
        ldv<T, 4>(a.gate, static_cast<size_t>(row) + static_cast<size_t>(h) * vdim + c, gate);
        ldv<T, 4>(a.norm, static_cast<size_t>(h) * a.w_head + c, w);
        float log_i, log_f;
        capped_gates(lo2f<T>(static_cast<const uint16_t*>(a.i)[row + h]) + lo2f<T>(static_cast<const uint16_t*>(a.b_i)[h]),
                     lo2f<T>(static_cast<const uint16_t*>(a.f)[row + h]) + lo2f<T>(static_cast<const uint16_t*>(a.b_f)[h]), a.cap, &log_i, &log_f);
        const float m = mp[0], mn = fmaxf(log_f + m, log_i);
        if (lane == 0) {
            scalars[0] = exp_fast(log_f + m - mn);
            scalars[1] = exp_fast(log_i - mn);
        }
        __builtin_amdgcn_wave_barrier();
        for (int i = lane; i < copies; i += 64)          // (read above by every lane)
            if (real) mp[i] = mn;
        if (lane == 0) scalars[2] = exp_fast(-mn);
    }
    __syncthreads();
    const float fa = scalars[0], ib = scalars[1];
    auto step = [&](float (&s)[kTokenRows], float in) {
        float e = 0.0f;
#pragma unroll
        for (int i = 0; i < kTokenRows; i++) {
            s[i] = __builtin_fmaf(k[i], in, fa * s[i]);
            e = __builtin_fmaf(s[i], q[i], e);
        }
        return row16_sum(e) * a.q_scale;
    };
#pragma unroll
    for (int j = 0; j < kMemoryColumns; j++) {
        const int col = grp + kGroups * j;
        const float e = step(S[j], ib * v[j]);
        if (real && col < vdim) store_column(state + static_cast<size_t>(col) * dim, part, dim, S[j]);
        if (part == 0) so[col] = real ? e : 0.0f;
    }
    float den = 1.0f;
    if (wv == 0) {
        const float e = step(N, ib);
        if (real && grp == 0) store_column(state + static_cast<size_t>(vdim) * dim, part, dim, N);
        den = real ? fmaxf(fabsf(e), scalars[2]) + 1e-6f : 1.0f;
    }
    __syncthreads();
    if (wv == 0)
        token_read_out<T>(so, den, lane, vdim, gate, w, a.out_scale, a.eps, static_cast<uint16_t*>(a.out) + b * a.out_row + static_cast<size_t>(h) * vdim);
}

int launch_memory_token(const MemoryTokenArgs& a, int dtype, hipStream_t st) {
    dim3 grid(static_cast<unsigned>(a.H), static_cast<unsigned>(a.B)), block(kMemoryThreads);
    if (dtype == 0) hipLaunchKernelGGL(memory_token_kernel<F16>, grid, block, 0, st, a);
    else hipLaunchKernelGGL(memory_token_kernel<BF16>, grid, block, 0, st, a);
    return static_cast<int>(hipGetLastError());
}

}  // namespace pq
