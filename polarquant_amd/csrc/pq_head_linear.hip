// Launcher of the per-head products at <= 16 rows (kernels: pq_linear_device.h).
#include "pq_linear_device.h"

namespace pq {

// The same two kernels for `heads` products per launch; K of a head is short (a head's dimension, a latent's rank), so
// fewer wavefronts split it: each keeps at least two k-steps.
int launch_head_linear_mfma(const HeadLinearArgs& a, int dtype, hipStream_t st) {
    const bool m8 = a.M <= 8 && (a.K % 64) == 0;
    const int kstep = m8 ? 64 : 32;
    int ks = (m8 && a.K >= 8192) ? 8 : 4;
    while (ks > 1 && ((a.K % (kstep * ks)) != 0 || a.K / (kstep * ks) < 2)) ks >>= 1;
    const int nt = m8 && a.heads == 1 ? small_m8_row_tiles(a.M, a.N, ks, 1) : 2;      // (several heads: their K is short, nothing is gained)
    dim3 grid(a.N / (8 * nt), a.heads), block(kWave * ks);
    const HeadEpi he{a.x_head, static_cast<int64_t>(a.N) * a.K, a.y_head, static_cast<const uint16_t*>(a.gate), a.gate_row, a.scale, a.cap, a.advance, 0, 0, nullptr, 0};
#define PQ_H(KERNEL)                                                                                                 \
    hipLaunchKernelGGL((KERNEL), grid, block, 0, st, (const uint16_t*)a.x, a.x_row,                                  \
                       (const uint16_t*)a.w, nullptr, nullptr, (uint16_t*)a.y, a.y_row, a.M, a.K, he)
#define PQ_HN(T, E, NT)                                                                                              \
    do {                                                                                                             \
        if (ks == 8) PQ_H((small_m8_linear_kernel<T, 8, false, NT == 2 ? 2 : 1, 1 + E, NT>));                        \
        else if (ks == 4) PQ_H((small_m8_linear_kernel<T, 4, false, 1, 1 + E, NT>));                                 \
        else if (ks == 2) PQ_H((small_m8_linear_kernel<T, 2, false, 1, 1 + E, NT>));                                 \
        else PQ_H((small_m8_linear_kernel<T, 1, false, 1, 1 + E, NT>));                                              \
    } while (0)
#define PQ_H16(T, E)                                                                                                 \
    do {                                                                                                             \
        if (ks == 4) PQ_H((small_m_linear_kernel<T, 4, false, 4, 1 + E>));                                           \
        else if (ks == 2) PQ_H((small_m_linear_kernel<T, 2, false, 4, 1 + E>));                                      \
        else PQ_H((small_m_linear_kernel<T, 1, false, 4, 1 + E>));                                                   \
    } while (0)
#define PQ_HE(T, E)                                                                                                  \
    do {                                                                                                             \
        if (!m8) PQ_H16(T, E);                                                                                       \
        else if (nt == 8) PQ_HN(T, E, 8);                                                                            \
        else if (nt == 4) PQ_HN(T, E, 4);                                                                            \
        else PQ_HN(T, E, 2);                                                                                         \
    } while (0)
#define PQ_HT(T)                                                                                                     \
    do {                                                                                                             \
        if (a.epilogue == kEpiReluSq) PQ_HE(T, kEpiReluSq);                                                          \
        else if (a.epilogue == kEpiSigmoidGate) PQ_HE(T, kEpiSigmoidGate);                                           \
        else if (a.epilogue == kEpiF32) PQ_HE(T, kEpiF32);                                                           \
        else if (a.epilogue == kEpiLogits) PQ_HE(T, kEpiLogits);                                                     \
        else PQ_HE(T, kEpiPlain);                                                                                    \
    } while (0)
    if (dtype == 0) PQ_HT(F16); else PQ_HT(BF16);
#undef PQ_HT
#undef PQ_HE
#undef PQ_H16
#undef PQ_HN
#undef PQ_H
    return static_cast<int>(hipGetLastError());
}

// The rows of a workgroup and the split of K as above: a workgroup of pairs streams as many bytes as one of plain rows.
int launch_linear_gelu(const LinearGeluArgs& a, int dtype, hipStream_t st) {
    int ks = a.K >= 8192 ? 8 : 4;
    while (ks > 1 && ((a.K % (64 * ks)) != 0 || a.K / (64 * ks) < 2)) ks >>= 1;
    const int nt = linear_gelu_row_tiles(a.M, a.plain, a.ff, ks);
    dim3 grid(a.plain / (8 * nt) + a.ff / (4 * nt)), block(kWave * ks);
    const HeadEpi he{0, 0, 0, nullptr, 0, 1.0f, 0.0f, nullptr, a.plain / (8 * nt), a.ff, static_cast<uint16_t*>(a.z), a.z_row};
#define PQ_G(T, KS, NT)                                                                                              \
    hipLaunchKernelGGL((small_m8_linear_kernel<T, KS, false, KS == 8 && NT == 2 ? 2 : 1, 1 + kEpiGeluPairs, NT>), grid, block, 0, st,   \
                       (const uint16_t*)a.x, a.x_row, (const uint16_t*)a.w, nullptr, nullptr, (uint16_t*)a.y, a.y_row, a.M, a.K, he)
#define PQ_GN(T, NT)                                                                                                 \
    do { if (ks == 8) PQ_G(T, 8, NT); else if (ks == 4) PQ_G(T, 4, NT); else if (ks == 2) PQ_G(T, 2, NT); else PQ_G(T, 1, NT); } while (0)
#define PQ_GT(T) do { if (nt == 8) PQ_GN(T, 8); else if (nt == 4) PQ_GN(T, 4); else PQ_GN(T, 2); } while (0)
    if (dtype == 0) PQ_GT(F16); else PQ_GT(BF16);
#undef PQ_GT
#undef PQ_GN
#undef PQ_G
    return static_cast<int>(hipGetLastError());
}

}  // namespace pq
