// Device code shared by the recurrent mixers' kernels.
#pragma once
#include "pq_elem.h"

namespace pq {

// (one instruction each, exact to about a unit in the last place)
__device__ __forceinline__ float exp_fast(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }
__device__ __forceinline__ float sigmoid(float z) { return __builtin_amdgcn_rcpf(1.0f + exp_fast(-z)); }
// max(z, 0) + log(1 + e), e = e^-|z|: for small e by its series, 1 + e would lose it
__device__ __forceinline__ float softplus(float z) {
    const float e = exp_fast(-fabsf(z));
    const float series = e * __builtin_fmaf(e, __builtin_fmaf(e, __builtin_fmaf(e, -0.25f, 0.33333334f), -0.5f), 1.0f);
    return fmaxf(z, 0.0f) + (e < 0.01f ? series : __builtin_amdgcn_logf(1.0f + e) * 0.6931471805599453f);
}

// the gates of a matrix memory as logarithms, capped before they are
__device__ __forceinline__ void capped_gates(float i, float f, float cap, float* log_i, float* log_f) {
    *log_i = cap * tanhf(i / cap);
    *log_f = -softplus(-(cap * tanhf(f / cap)));
}

// sum over 16 lanes, in each of them
__device__ __forceinline__ float row16_sum(float v) {
    v += __uint_as_float(row_rotate<8>(__float_as_uint(v)));
    v += __uint_as_float(row_rotate<4>(__float_as_uint(v)));
    v += __uint_as_float(row_rotate<2>(__float_as_uint(v)));
    v += __uint_as_float(row_rotate<1>(__float_as_uint(v)));
    return v;
}

}  // namespace pq
