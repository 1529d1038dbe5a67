// Causal attention of a prompt with half-precision keys and values, as the polar-key models' projections leave them: a row per
// token, any (batch, token, head) strides, KV heads shared by groups of query heads.  The kernel is pq_prompt_attn.h's.
#include "pq_prompt_attn.h"
#include "pq_internal.h"

namespace pq {

int launch_prompt_attn(const void* q, const void* k, const void* v, const int64_t* s, void* out, int B, int L, int N, int Nk,
                       float scale, int dtype, hipStream_t st) {
    PromptAttnArgs a{};
    a.q = q; a.q_b = s[0]; a.q_h = s[1]; a.q_t = s[2];
    a.k = k; a.k_b = s[3]; a.k_h = s[4]; a.k_t = s[5];
    a.v = v; a.v_b = s[6]; a.v_h = s[7]; a.v_t = s[8];
    a.out = out; a.out_row = static_cast<int64_t>(N) * kHeadDim;
    a.B = B; a.L = a.Lk = L; a.H = N; a.G = Nk; a.D = a.Dv = kHeadDim; a.scale = scale;
    return dtype == 0 ? launch_prompt_attn<F16, 128, 128, true>(a, st) : launch_prompt_attn<BF16, 128, 128, true>(a, st);
}

}  // namespace pq
