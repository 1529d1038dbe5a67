// RMS norms of the query latent and of the key/value latent, the latter written to its cache row.  fp32 arithmetic on
// whatever the operands' dtype is; results are rounded to it once.
#include "pq_elem.h"
#include "pq_latent_internal.h"

namespace pq {

// ---- norms of the two latents ---------------------------------------------------------------------------------------
// A wavefront per token when there are many (WIDE false), a workgroup per token otherwise.
template <typename T, int V, bool WIDE>
__global__ __launch_bounds__(256) void latent_norm_kernel(LatentNormArgs a) {
    __shared__ float part[2][4];
    const int wv = threadIdx.x >> 6, n_tok = a.B * a.L;
    const int first = (WIDE ? static_cast<int>(threadIdx.x) : static_cast<int>(threadIdx.x & 63)) * V, step = (WIDE ? 256 : 64) * V;
    int tok = WIDE ? static_cast<int>(blockIdx.x) : static_cast<int>(blockIdx.x) * 4 + wv;
    if (!WIDE && tok >= n_tok) return;
    const int b = tok / a.L, t = tok - b * a.L;
    const int Q = a.q_rank, R = a.w_kv ? a.kv_rank : 0;
    const elem_t<T>* p = static_cast<const elem_t<T>*>(a.p) + static_cast<size_t>(tok) * a.row_stride;
    float sq = 0.0f, sc = 0.0f, v[V];
    for (int i = first; i < Q + R; i += step) {
        ldv<T, V>(p, i, v);
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < V; j++) s = __builtin_fmaf(v[j], v[j], s);
        sq += i < Q ? s : 0.0f;
        sc += i < Q ? 0.0f : s;
    }
    sq = wave_sum(sq);
    sc = wave_sum(sc);
    if (WIDE) {
        if ((threadIdx.x & 63) == 0) { part[0][wv] = sq; part[1][wv] = sc; }
        __syncthreads();
        sq = part[0][0] + part[0][1] + part[0][2] + part[0][3];
        sc = part[1][0] + part[1][1] + part[1][2] + part[1][3];
    }
    const float rq = rsqrtf(sq / static_cast<float>(Q) + a.eps), rc = R ? rsqrtf(sc / static_cast<float>(R) + a.eps) : 0.0f;
    int64_t pos = (a.pos_dev ? *a.pos_dev : a.pos) + t;
    pos = pos < 0 ? 0 : (pos >= a.capacity ? a.capacity - 1 : pos);          // (never past the cache)
    elem_t<T>* qo = static_cast<elem_t<T>*>(a.q_out) + static_cast<size_t>(tok) * Q;
    elem_t<T>* co = static_cast<elem_t<T>*>(a.cache) + (static_cast<size_t>(b) * a.capacity + pos) * R;
    for (int i = first; i < Q + R; i += step) {
        const bool is_q = i < Q;
        float w[V];
        ldv<T, V>(p, i, v);
        ldv<T, V>(is_q ? a.w_q : a.w_kv, is_q ? i : i - Q, w);
        const float r = is_q ? rq : rc;
#pragma unroll
        for (int j = 0; j < V; j++) v[j] = w[j] * (v[j] * r);
        stv<T, V>(is_q ? qo : co, is_q ? i : i - Q, v);
    }
}

// Few tokens, NP pieces of 4 a thread: the row and the weights are requested at once and read once.  The same bits.  8 tokens of
// ranks 1536 and 512 2.6 -> 2.4 us in a chain of launches.
template <typename T, int NP>
__global__ __launch_bounds__(256) void latent_norm_row_kernel(LatentNormArgs a) {
    __shared__ float part[2][4];
    const int tok = blockIdx.x, wv = threadIdx.x >> 6, b = tok / a.L, t = tok - b * a.L;
    const int Q = a.q_rank, R = a.w_kv ? a.kv_rank : 0;
    const elem_t<T>* row = static_cast<const elem_t<T>*>(a.p) + static_cast<size_t>(tok) * a.row_stride;
    float v[NP][4], w[NP][4], sq = 0.0f, sc = 0.0f;
    auto at = [&](int p) { const int i = p * 1024 + static_cast<int>(threadIdx.x) * 4; return i < Q + R ? i : 0; };
    auto own = [&](int p) { return p * 1024 + static_cast<int>(threadIdx.x) * 4 < Q + R; };
#pragma unroll
    for (int p = 0; p < NP; p++) {
        ldv<T, 4>(row, at(p), v[p]);
        const bool is_q = at(p) < Q;
        ldv<T, 4>(is_q ? a.w_q : a.w_kv, is_q ? at(p) : at(p) - Q, w[p]);
    }
    int64_t pos = (a.pos_dev ? *a.pos_dev : a.pos) + t;
    pos = pos < 0 ? 0 : (pos >= a.capacity ? a.capacity - 1 : pos);          // (never past the cache)
#pragma unroll
    for (int p = 0; p < NP; p++) {
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) s = __builtin_fmaf(v[p][j], v[p][j], s);
        s = own(p) ? s : 0.0f;
        sq += at(p) < Q ? s : 0.0f;
        sc += at(p) < Q ? 0.0f : s;
    }
    sq = wave_sum(sq);
    sc = wave_sum(sc);
    if ((threadIdx.x & 63) == 0) { part[0][wv] = sq; part[1][wv] = sc; }
    __syncthreads();
    sq = part[0][0] + part[0][1] + part[0][2] + part[0][3];
    sc = part[1][0] + part[1][1] + part[1][2] + part[1][3];
    const float rq = rsqrtf(sq / static_cast<float>(Q) + a.eps), rc = R ? rsqrtf(sc / static_cast<float>(R) + a.eps) : 0.0f;
    elem_t<T>* qo = static_cast<elem_t<T>*>(a.q_out) + static_cast<size_t>(tok) * Q;
    elem_t<T>* co = static_cast<elem_t<T>*>(a.cache) + (static_cast<size_t>(b) * a.capacity + pos) * R;
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const bool is_q = at(p) < Q;
#pragma unroll
        for (int j = 0; j < 4; j++) v[p][j] = w[p][j] * (v[p][j] * (is_q ? rq : rc));
        if (own(p)) stv<T, 4>(is_q ? qo : co, is_q ? at(p) : at(p) - Q, v[p]);
    }
}

int launch_latent_norm(const LatentNormArgs& a, int dtype, hipStream_t st) {
    const bool v4 = a.q_rank % 4 == 0 && (!a.w_kv || a.kv_rank % 4 == 0) && a.row_stride % 4 == 0;
    const int n_tok = a.B * a.L;
    const bool wide = n_tok < 1024;
    const int pieces = (a.q_rank + (a.w_kv ? a.kv_rank : 0) + 1023) / 1024;
    if (v4 && wide && dtype != 2 && pieces <= 4) {
#define PQ_LR(T, N) hipLaunchKernelGGL((latent_norm_row_kernel<T, N>), dim3(n_tok), dim3(256), 0, st, a)
#define PQ_LRT(T) do { if (pieces == 1) PQ_LR(T, 1); else if (pieces == 2) PQ_LR(T, 2); else PQ_LR(T, 4); } while (0)
        if (dtype == 0) PQ_LRT(F16); else PQ_LRT(BF16);
#undef PQ_LRT
#undef PQ_LR
        return static_cast<int>(hipGetLastError());
    }
    dim3 grid(static_cast<unsigned>(wide ? n_tok : (n_tok + 3) / 4)), block(256);
#define PQ_LN1(T, V) do { if (wide) hipLaunchKernelGGL((latent_norm_kernel<T, V, true>), grid, block, 0, st, a); \
                          else hipLaunchKernelGGL((latent_norm_kernel<T, V, false>), grid, block, 0, st, a); } while (0)
#define PQ_LN(T) do { if (v4) PQ_LN1(T, 4); else PQ_LN1(T, 1); } while (0)
    if (dtype == 0) PQ_LN(F16); else if (dtype == 1) PQ_LN(BF16); else PQ_LN(F32);
#undef PQ_LN
#undef PQ_LN1
    return static_cast<int>(hipGetLastError());
}

}  // namespace pq
