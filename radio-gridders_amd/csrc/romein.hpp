// romein.hpp -- software-pipelined record loop of the W-towers band kernel, and the tap
// reads' buffer resource, which the W-projection tiles use too.
//
// Records are consumed in batches of U: `fetch(j, batch)` reads records
// [j, j + U) from LDS, computes each lane's footprint cell and issues the U
// kernel-tap loads; `update(batch)` applies them in stream order.  Two
// batches alternate so the loads of batch i + 1 are in flight while batch i
// is applied.  AHEAD: the loads ahead are issued without a condition (past the
// end the last batch again).  Where they may or may not have been issued the
// compiler's wait for batch i counts for the second case and drains batch i + 1 too:
// worth it where few wavefronts hide the latency (two a SIMD, band pass of row pairs: 1891
// -> 1860 us), not where the rest are enough (four: 2072 -> 2136 us).
#pragma once

#include "binning.hpp"

namespace rg {

// Kernel taps are read through a buffer resource: offsets beyond the table read zeros
// (TAP_NONE for a lane whose row the footprint misses, unpadded table).
constexpr uint32_t TAP_NONE = 0x80000000u;
// word 3 of a raw (unswizzled, stride 0) buffer resource on gfx9
constexpr int BUF_RSRC_W3 = 0x00020000;

template <int U, bool AHEAD, typename B, typename Fetch, typename Update>
__device__ inline void pipelined_records(uint32_t n, Fetch &&fetch, Update &&update)
{
    B a, b;
    if (n == 0)
        return;
    auto prefetch = [&](uint32_t j, B &bt) {
        if (AHEAD)
            fetch(min(j, n - U), bt);
        else if (j < n)
            fetch(j, bt);
    };
    fetch(0u, a);
    for (uint32_t j = 0; j < n; j += 2 * U) {
        prefetch(j + U, b);
        update(a);
        if (j + U >= n)
            break;
        prefetch(j + 2 * U, a);
        update(b);
    }
}

} // namespace rg
