// gemm_tiles.h -- tile order of the prefill kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace oilhip {

// Tile order: token blocks in groups of four; inside a group weight-row blocks ascending, the group's token blocks
// innermost.  A run of consecutive tiles therefore covers few token blocks and neighbouring weight rows.
__host__ __device__ inline void frag_tile_of(uint32_t T, uint32_t MT, uint32_t NT, uint32_t& mt, uint32_t& nt) {
    const uint32_t per = 4u * NT, lastg = (MT - 1u) / 4u;
    uint32_t mg = T / per;
    if (mg > lastg) mg = lastg;
    const uint32_t rem = T - mg * per, left = MT - 4u * mg, gm = left < 4u ? left : 4u;
    nt = rem / gm;
    mt = 4u * mg + rem % gm;
}

// Workgroups are dealt to the eight XCDs in turn; XCD x takes the x-th run of n / 8 consecutive items.
__device__ inline uint32_t xcd_chunk(uint32_t b, uint32_t n) {
    const uint32_t x = b & 7u, q = b >> 3, c = n >> 3, r = n & 7u;
    return (x < r ? x * (c + 1u) : r * (c + 1u) + (x - r) * c) + q;
}

}  // namespace oilhip
