// How many rows of W a workgroup of small_m8_linear_kernel takes (plain C++: host code only).
#pragma once

namespace pq {

// NT tiles of 8 rows.  What a compute unit can have on its way from memory is about its share of the HBM rate, so the units' rows set the
// time: those of the fullest unit if all started together, their mean if work spread evenly; measured, halfway between.  On top comes
// x, which every workgroup reads from L2: of 8 rows 0.42 of a tile's time (without the x loads 28672 x 4096 takes 37.4 us, the plain
// stream's time), of fewer as much less, and that is all that more tiles save.  Eight tiles, or four with K split eight ways, leave few
// workgroups to a unit, which costs 4 or 5 % by itself.
// Measured in a chain of calls, K = 4096, NT 2 / 4 / 8 in us, 8 rows: N 6144 13.5 / 12.3 / 23.9; 10240 20.7 / 22.6 / 24.9; 21504 37.6 /
// 34.9 / 38.6; 43136 65.6 / 62.3 / 59.1; 32768 50.3 / 45.8 / 44.8.  Of one row NT 2 / 8: 28672 38.7 / 41.4; 32768 43.3 / 45.0; 43136
// 57.6 / 60.5; 28672 x 8192 76.9 / 85.4; NT 2 / 4: 6144 11.7 / 11.6, 21504 33.9 / 33.2, 8192 x 8192 25.7 / 26.7.  (x kept in registers by
// persistent workgroups, 8 rows: 41 / 59 us at N 28672 / 43136, and 10.2 instead of 8.8 at 4096.)
inline int small_m8_row_tiles(int rows, int N, int ksplit, int matrices) {
    constexpr int kUnits = 256;
    const double x = 0.42 * rows / 8.0;
    int best = 2;
    double least = 0.0;
    for (int nt = 2; nt * matrices <= 8; nt *= 2) {
        if (N % (8 * nt)) break;
        const int groups = N / (8 * nt);
        // too few wavefronts to keep loads on the way: 3 per unit with four tiles' loads each, 7 with eight
        if (nt > 2 && groups * ksplit < (nt * matrices == 8 ? 7 : 3) * kUnits) break;
        const double unit = 0.5 * ((groups + kUnits - 1) / kUnits + static_cast<double>(groups) / kUnits);
        const double cost = unit * nt * (1.0 + x / (nt * matrices)) * (nt == 8 ? 1.04 : 1.0) * (nt > 2 && ksplit == 8 ? 1.05 : 1.0);
        if (nt == 2 || cost < least) { best = nt; least = cost; }
    }
    return best;
}

// The same of a product whose last 2 ff rows of W go to workgroups of pairs (launch_linear_gelu): whole workgroups of either kind, two tiles at least.
inline int linear_gelu_row_tiles(int rows, int plain, int ff, int ksplit) {
    const int N = plain + 2 * ff;
    int nt = N % 16 ? 2 : small_m8_row_tiles(rows, N, ksplit, 1);
    while (nt > 2 && (plain % (8 * nt) || ff % (4 * nt))) nt >>= 1;
    return nt;
}

// Depths that the products around a norm take (launch_linear_residual: `behind` false; the products behind it: true).  K is split four ways,
// from 8192 on eight, into whole steps of 64; and behind the norm a row's sums, one of 16 elements, have to be two 16-byte loads to a
// thread at most (8 KSPLIT threads a row): up to 4096, and 8192.  (More loads a thread, for the widths between, were not tried.)
inline bool normed_depth(int K, bool behind) {
    const int ks = K >= 8192 ? 8 : 4;
    return K >= 256 && K % (64 * ks) == 0 && (!behind || K / 16 <= 2 * 4 * 8 * ks);
}

}  // namespace pq
