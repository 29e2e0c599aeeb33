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

}  // namespace ftnn
