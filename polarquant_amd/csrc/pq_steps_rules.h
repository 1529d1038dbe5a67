// How many tokens a strip of norm_conv_kernel takes (plain C++: host code only).
#pragma once
#include <stdint.h>

namespace pq {

// Strips as long as the device stays full with them: every strip recomputes taps - 1 norms, and its tokens follow each other (2.2 us a
// token).  Full is one workgroup per unit, two where a thread has one piece and few taps are recomputed.  8192 tokens of 4096, taps 4,
// strips of 32 / 16 / 8: 103 / 108 / 126 us; 2048 tokens 77 / 46 / 31; 512 tokens, down to strips of 4: 71 / 41 / 26 / 18.  6000 tokens
// of 2048 (a piece a thread), strips of 32 / 16: taps 5 62 / 71, taps 8 64 / 75, taps 12 91 / 122.
// With more than 8 taps and several pieces a thread the kernel spills: a token takes twice the time once more than some 128 (4 and more
// pieces: 32) workgroups do so side by side, no more beyond that.  Strips are not halved across that line: 9 taps, 3000 tokens of 4096,
// strips of 32 / 16: 268 / 300; 700 of 8192 1333 / 1510; but 1500 of 4096 260 / 158, 1500 of 8192 2858 / 1572.
inline int norm_conv_strip(int64_t tokens, int taps, int pieces_per_thread) {
    constexpr int64_t kUnits = 256;
    const int64_t full = pieces_per_thread == 1 && taps <= 4 ? 2 * kUnits : kUnits;
    const int64_t knee = taps <= 8 || pieces_per_thread == 1 ? 0 : pieces_per_thread == 2 ? 128 : 32;
    int strip = 32;
    while (strip > 4 && strip / 2 >= taps && tokens / (strip / 2) <= full && !(tokens / strip <= knee && tokens / (strip / 2) > knee)) strip /= 2;
    return strip;
}

}  // namespace pq
