// Which form of a kernel a context launches, by how many particle block parts it has (parts), of how many
// particles (n), and by what zmpm_autotune found (tuned; a size of 0 or a flag below 0: not tuned).  Every
// form gives the same bits.  Host code only.
#pragma once

#include <cstdint>

namespace zmpm {

// (Update with 64 and 256 threads, 2,197 parts of 126 particles: 19.7 and 22.5 us, of 157: 23.3 and 23.6, of
// 220: 27.5 and 27.8; 4,913 of 107: 30.6 and 34.7, of 133: 35.2 and 36.4, of 167: 42.6 and 38.6; 19,683 of
// 143: 127 and 162, of 179: 161 and 180, of 250: 242 and 227.  FLIP transfers, move and update together, 2,197
// of 126: 56 and 60; 4,913 of 133: 100 and 110, of 167: 117 and 119; 19,683 of 143: 376 and 445.)
inline bool many_small_parts(int64_t parts, int64_t n) { return parts >= 1536 && n <= 128 * parts; }

// Threads per workgroup (one part each) of the G2P kernels.  Few parts leave wave slots empty, so a part gets
// as many threads as pay; many fill the chip with one wave each, which waits at no barrier.
// Move, 180 parts of 363 particles: 12.4 us with 64 threads, 8.4 with 256, 8.2 with 512; 1,180 of
// 340: 15.1, 10.8, 16.9; 1,800 of 340: 16.5, 17.7, 24.2; 9,990 of 420: 46, 67, 114; 77,514 of 60:
// 165, 319, -.  Update, the same: 22.1, 12.4, 10.8; 27.8, 19.0, 21.7; 27.8, 25.5, 30.4; 127, 119,
// 153; 340, 506, -; about 400 parts: 24.9, 14.1, 13.0; 740: 26.5, 16.4, 18.4.
// FLIP transfers (the particles are all interpolated, twice the registers), move and update, 366
// parts: 27 and 34 with 64, 16 and 16 with 256, 15 and 19 with 512; 1,750: 37 and 44, 28 and 44, 34
// and 54; 5,800: 87 and 159, 68 and 144, 95 and 170.
inline int g2p_move_threads(int64_t parts, int64_t n, bool flip, int tuned) {
    if (tuned) return tuned;
    return (flip ? many_small_parts(parts, n) : parts >= 1536) ? 64 : 256;
}
inline int g2p_update_threads(int64_t parts, int64_t n, bool flip, int tuned) {
    if (tuned) return tuned;
    if (many_small_parts(parts, n)) return 64;
    return !flip && parts <= 512 ? 512 : 256;
}

// One-wave P2G for blocks of <= 64 particles, a launch of its own, where the chip is full of blocks and nearly
// all are that small.  P2G with and without, 17,576 blocks of 30, 36, 44 and 48 particles on average (Poisson):
// 77 and 80, 79 and 82, 86 and 84, 89 and 86 us; 39,304 of 36 and 48: 166 and 183, 181 and 194; 64,000 of 48:
// 288 and 319; 68,921 of 59: 424 and 360; 90 % of 10 and 10 % of 300, 17,576 and 64,000 blocks: 91 and 89, 298
// and 317; 4,913 of 10 and 33: 31 and 28, 32 and 30.
inline bool p2g_one_wave(int64_t parts, int64_t n, int tuned) {
    if (tuned >= 0) return tuned != 0;
    return parts >= 16384 && n <= (parts >= 32768 ? 48 : 36) * parts;
}

}  // namespace zmpm
