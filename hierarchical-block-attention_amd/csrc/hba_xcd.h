// Workgroup -> work mapping over the 8 XCDs, shared by the attention kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hba {

// Workgroup -> (batch*KV head combo, query tile).  Workgroup i runs on XCD
// i % 8; xmap 1 (8 % Cn == 0) and 2 (Cn % 8 == 0) give each XCD one combo's
// keys at a time, so the blocks it gathers share that XCD's L2.  Tiles go
// deepest first: a tile's union of routed blocks grows with its candidate
// count, and starting the longest workgroups first leaves the short ones to
// fill the end.
__device__ __forceinline__ void xcd_map(int i, int Cn, int ntiles, int xmap, int &combo, int &tile) {
    if (xmap == 1) {
        combo = (i & 7) % Cn;
        tile = (i >> 3) * (8 / Cn) + (i & 7) / Cn;
    } else if (xmap == 2) {
        combo = (i / (8 * ntiles)) * 8 + (i & 7);
        tile = (i >> 3) % ntiles;
    } else {
        combo = i / ntiles;
        tile = i % ntiles;
    }
    if (tile < ntiles) tile = ntiles - 1 - tile;   // padding workgroups (xmap 1) keep tile >= ntiles
}

// The mapping for Cn combos of ntiles tiles, and its grid size.
inline int xcd_pick(int64_t Cn, int64_t ntiles, int64_t &grid) {
    const int xmap = (8 % Cn == 0) ? 1 : (Cn % 8 == 0 ? 2 : 0);
    grid = (xmap == 1) ? 8 * ((ntiles + 8 / Cn - 1) / (8 / Cn)) : Cn * ntiles;
    return xmap;
}

}  // namespace hba
