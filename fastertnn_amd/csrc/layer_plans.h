// How layers are cut into launches: rules on sizes alone (the host side of the kernels; plain C++).
#pragma once
#include <stdint.h>

#include <algorithm>

#include "pair_walk.h"

namespace ftnn {

inline bool ranges_meet(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + (uintptr_t)b_bytes && y < x + (uintptr_t)a_bytes;
}

// The grid of k_dense_rows: blocks of 32 rows along x and, past 2^23 of them, z (a grid dimension holds fewer than 2^32 threads), groups
// of four words along y.  Workgroups enough: each makes all the words of its rows, the input then comes through one L2 only (32 x 16 x 64 x 64,
// 5 x 5, BNN: 26.5 -> 24.4 us as a layer).
constexpr uint32_t kDenseBlocksX = 1u << 23;
struct DenseGrid {
    uint32_t x, y, z;
};
inline DenseGrid dense_rows_grid(int64_t M /* rows, below 2^31 */, int groups) {
    const int64_t blocks = (M + 31) / 32;
    DenseGrid g;
    g.x = (uint32_t)std::min<int64_t>(blocks, kDenseBlocksX);
    g.y = M >= 65536 ? 1u : (uint32_t)std::min(groups, 65535);
    g.z = (uint32_t)((blocks + kDenseBlocksX - 1) / kDenseBlocksX);
    return g;
}

// Dense rows straight from the fp32 input (k_dense_rows), or from its bit planes in two launches (k_dense_rows_planes).  The first reads a tap as
// `loads` values of 4 bytes, again for every window that holds it; the second quantises each pixel once and reads a tap as 8 or 16 bytes, for
// a launch more.  us of either side in a graph, but for what both have, fitted to 1050 layers of 1 to 32 channels, windows of 3 x 1 to 17 x 17 and 16 to
// 1200000 pixels; 0.6 is taken off the launch, so that a tie keeps the planes.  The choice is 0.3 % from the better form in the mean (the planes
// alone 13 %, the input alone 12 %), and 13 of the 1050 are 3 to 23 % slower than from the planes.  Layers, us, from the planes / the input:
// 22 x 9 x 209 x 209 -> 10, 3 x 3, BNN 79.8 / 66.1; 52 x 11 x 45 x 45 -> 25, 9 x 1, TNN 24.3 / 18.4; 61 x 19 x 186 x 186 -> 12, 9 x 9 stride 2, BNN 152 / 493;
// 26 x 17 x 70 x 70 -> 6, 11 x 11 stride 2, TNN 24.4 / 53.2.  Eight taps at most of 23 channels and more are one trip of a workgroup, which then
// waits longer than it works: 25 x 30 x 29 x 151 -> 39, 5 x 1, TNN 19.6 / 24.6, but on 6762 pixels, 7 x 1, 10.5 / 9.6.  Inputs of 4 GiB and
// more go by the planes: offsets within the input are 32 bits wide.
inline int dense_loads(int C) { return C <= 8 ? 8 : C <= 12 ? 12 : C <= 16 ? 16 : C <= 24 ? 24 : 32; }
inline bool dense_rows_from_input(bool ternary, int64_t pixels /* of the input */, int C, int64_t M, int taps, int W_stride) {
    if (pixels * C >= (1LL << 30) || (C > 22 && taps <= 8 && M > 20000)) return false;
    const double in = 1e-6 * (double)pixels, read = 1e-6 * (double)M * taps;   // pixels and taps, in millions
    if (C <= 8) return read * (W_stride > 1 ? 2.60 : 1.02) < 2.6 + 23.3 * in;
    return read * dense_loads(C) * (W_stride > 1 ? 0.473 : 0.223) < 0.9 + 15.5 * in + read * (ternary ? 1.49 : 1.94);
}

// Few kernels leave the tiles of k_rows mostly empty, so that such a layer's dense rows stay on the vector ALU: up to 15 on one group of words
// (256 x 16 x 16 x 16 -> 8 BTN 10.9 us on the vector ALU / 12.5), up to eight on some more (7 x 14 x 94 x 94 -> 8, 5 x 5, TBN 17.4 / 19.9; 57024 pixels -> 3,
// 28 words, TBN 32.6 / 37.6), but 212064 -> 3, 32 words, BTN 118 / 70 and 10000 -> 10, 60 words, TNN 24.6 / 19.3.  Of 400 layers of 1 to 24 kernels 4 are 6 to
// 9 % slower than on the vector ALU (15 by the first line alone).
inline bool few_kernels(int64_t M, int KN, int Kw) { return (KN < 16 && Kw == 4) || (KN <= 8 && Kw <= 44 && M <= 100000); }

}  // namespace ftnn
