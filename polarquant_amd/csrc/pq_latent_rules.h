// How latent decode attention is laid out over the units (plain C++: host code only).
#pragma once
#include <stdint.h>

namespace pq {

struct LatentDecodeLayout {
    int teams, slices;       // of wavefronts in a workgroup; of the context
};

// What one or two teams a workgroup take of `slices` slices, as the plan has them: two workgroups of one team on every unit.  `groups`: row tiles
// of all sequences; rank: padded to 64, 128, 256 or 512.
//
// Two teams halve a slice's chain of tiles and the partials in memory, but a workgroup of them is what a unit holds (LDS; at rank 64 several
// fit).  They pay where the call has few workgroups, and in full rows of them; a second, nearly empty round of workgroups costs more than
// everything they give.  Both launches in us, one team with the plan's slices / two teams with as many slices as fit, 32 heads:
//   rank 512   2000 keys: 64 sequences 56.7 / 52.3, 100 93.7 / 78.7, 129 122.8 / 116.5, 256 176.4 / 170.8, but 257 223 / 237, 300 236 / 249;
//              100 keys: 257 87 / 96
//   rank 256   3000 keys: 20 sequences 23.2 / 22.1, 64 40.9 / 40.8, but 86 58.4 / 62.3, 129 78 / 101, 192 102 / 111, 257 137 / 195
//   rank 128   500 keys: 20 sequences 12.9 / 12.3, but 3000 keys: 40 26.0 / 26.0, 86 42.1 / 43.8, 129 57.6 / 58.7, 300 110 / 126
//   rank 64    (as many slices as the plan) 4000 keys, 8 heads: 64 sequences 18.2 / 15.2, 129 28.0 / 23.2, 300 53.6 / 39.2, 1024 121 / 113
//   64 sequences of 500 keys, 5 slices of the plan / 4: rank 128 18.7 / 16.6, rank 64 (5 / 4 slices of two teams) 12.6 / 11.8
inline LatentDecodeLayout latent_decode_layout(int rank, int64_t groups, int slices) {
    constexpr int64_t kUnits = 256;
    const int64_t fit = kUnits / groups;
    if (slices <= fit) return {2, slices};
    if (4 * fit >= 3 * slices || (rank > 256 && fit >= 1) || (rank > 128 && fit >= 4)) return {2, static_cast<int>(fit)};
    return {rank <= 64 ? 2 : 1, slices};
}

}  // namespace pq
