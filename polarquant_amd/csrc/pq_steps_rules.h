// How many tokens a strip of norm_conv_kernel takes (plain C++: host code only).
#pragma once
#include <stdint.h>

namespace pq {

// Strips as long as the device stays full with them: every strip recomputes taps - 1 norms, and its tokens follow each other (2.2 us a
// token).  Full is one workgroup per unit, two where a thread has one piece and few taps are recomputed.  8192 tokens of 4096, taps 4,
// strips of 32 / 16 / 8: 103 / 108 / 126 us; 2048 tokens 77 / 46 / 31; 512 tokens, down to strips of 4: 71 / 41 / 26 / 18.  6000 tokens
// of 2048 (a piece a thread), strips of 32 / 16: taps 5 62 / 71, taps 8 64 / 75, taps 12 91 / 122.
inline int norm_conv_strip(int64_t tokens, int taps, int pieces_per_thread) {
    constexpr int64_t kUnits = 256;
    const int64_t full = pieces_per_thread == 1 && taps <= 4 ? 2 * kUnits : kUnits;
    int strip = 32;
    while (strip > 4 && strip / 2 >= taps && tokens / (strip / 2) <= full) strip /= 2;
    return strip;
}

}  // namespace pq
