// binning.hip -- scan kernels of the device-side counting sort.
#include <algorithm>

#include "scan.hpp"

namespace rg {

// Exclusive block scan of uint2 values (x and y scanned independently).
// Returns the exclusive prefix of the calling thread and the block total.
template <int NT>
__device__ inline uint2 block_exclusive_scan(uint2 v, uint2 &total, uint2 *lds /* NT */)
{
    lds[threadIdx.x] = v;
    __syncthreads();
    // Hillis-Steele inclusive scan in LDS (NT <= 1024)
    for (int off = 1; off < NT; off <<= 1) {
        uint2 add = make_uint2(0, 0);
        if ((int)threadIdx.x >= off)
            add = lds[threadIdx.x - off];
        __syncthreads();
        uint2 cur = lds[threadIdx.x];
        cur.x += add.x;
        cur.y += add.y;
        lds[threadIdx.x] = cur;
        __syncthreads();
    }
    uint2 inc = lds[threadIdx.x];
    total = lds[NT - 1];
    __syncthreads();
    return make_uint2(inc.x - v.x, inc.y - v.y);
}

// Phase 2 (more than SCAN_DIRECT blocks): block totals to exclusive prefixes, one block.
__global__ __launch_bounds__(1024) void k_scan_blocks(uint2 *block_sums, int nblocks)
{
    __shared__ uint2 lds[1024];
    const int per = (nblocks + 1023) / 1024;
    const int b0 = threadIdx.x * per;
    uint2 acc = make_uint2(0, 0);
    for (int j = 0; j < per; ++j) {
        if (b0 + j < nblocks) {
            const uint2 v = block_sums[b0 + j];
            acc.x += v.x;
            acc.y += v.y;
        }
    }
    uint2 total;
    uint2 run = block_exclusive_scan<1024>(acc, total, lds);
    for (int j = 0; j < per; ++j) {
        if (b0 + j < nblocks) {
            const uint2 v = block_sums[b0 + j];
            block_sums[b0 + j] = run;
            run.x += v.x;
            run.y += v.y;
        }
    }
}

int launch_scan_blocks(uint2 *bsums, int64_t nb, hipStream_t s)
{
    hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(1024), 0, s, bsums, (int)nb);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

// Keys per scan thread: one while the key space is small (more workgroups, the
// latency of their loads is all there is: 4225 keys in 16 replicas 17 -> 4 us
// a phase), four from 64 K keys.
int scan_per_thread(int64_t nkeys) { return nkeys >= 65536 ? 4 : 1; }

int64_t scan_blocks(int64_t nkeys)
{
    const int64_t tile = SCAN_BLOCK * scan_per_thread(nkeys);
    return (nkeys + tile - 1) / tile;
}

size_t scan_sums_bytes(int64_t nkeys)
{
    return sizeof(uint2) * (size_t)(std::max<int64_t>(scan_blocks(nkeys), 65536 / SCAN_BLOCK) + 1);
}

int scan_keys(const uint32_t *count, Replicas rp, int64_t nkeys, uint32_t per_item, uint2 *bsums,
              uint32_t *vis_start, uint32_t *item_start, uint32_t *cursor, Item *items,
              unsigned long long *stats, hipStream_t s, uint32_t *group_start, int group_keys)
{
    auto run = [&](auto nrep) {
        CountSource<decltype(nrep)::value> src;
        src.count = count;
        src.stride = rp.stride;
        src.vis_start = vis_start;
        src.cursor = cursor;
        src.group_start = group_start;
        src.group_keys = group_keys;
        return scan_source(src, nkeys, per_item, bsums, item_start, items, stats, s);
    };
    switch (rp.mask + 1) {
    case 1: return run(std::integral_constant<int, 1>{});
    case 2: return run(std::integral_constant<int, 2>{});
    case 4: return run(std::integral_constant<int, 4>{});
    case 8: return run(std::integral_constant<int, 8>{});
    default: return run(std::integral_constant<int, 16>{});
    }
}

int bin_plan(int64_t n, int64_t nkeys, uint32_t per_item, int64_t max_counters, size_t rec_bytes,
             BinPlan &pl)
{
    // record indices are 32-bit
    if (n >= (int64_t)0x7fffffff)
        return fail(RG_ERR_PARAM, "visibility stream too long for one call (%lld)", (long long)n);
    if (nkeys <= 0 || nkeys >= (int64_t)0x7fffffff)
        return fail(RG_ERR_PARAM, "invalid key space %lld", (long long)nkeys);
    if (per_item == 0)
        return fail(RG_ERR_PARAM, "work items need at least one record");
    const int64_t nblocks_scan = scan_blocks(nkeys);
    if (nblocks_scan > 1024 * 256)
        return fail(RG_ERR_PARAM, "key space too large (%lld)", (long long)nkeys);
    pl.max_items = nkeys + n / per_item + 1;
    // counter replicas: up to 16, at most max_counters counters in all
    // (replicas spread the atomics of hot keys; a stream without hot keys
    // is better served by fewer counters that stay in cache)
    pl.rp.stride = bin_stride(nkeys);
    uint32_t nrep = 16;
    while (nrep > 1 && (int64_t)nrep * pl.rp.stride > max_counters)
        nrep >>= 1;
    pl.rp.mask = nrep - 1;
    const int64_t n1 = n > 0 ? n : 1;
    pl.bytes[BIN_COUNT] = sizeof(uint32_t) * nrep * pl.rp.stride;
    pl.bytes[BIN_VIS_START] = sizeof(uint32_t) * (nkeys + 1);
    pl.bytes[BIN_ITEM_START] = sizeof(uint32_t) * (nkeys + 1);
    pl.bytes[BIN_CURSOR] = sizeof(uint32_t) * nrep * pl.rp.stride;
    pl.bytes[BIN_ITEMS] = sizeof(Item) * pl.max_items;
    pl.bytes[BIN_RECS] = rec_bytes * n1;
    pl.bytes[BIN_BSUMS] = sizeof(uint2) * (nblocks_scan + 1);
    pl.bytes[BIN_KRP] = sizeof(uint4) * n1;
    return RG_OK;
}

} // namespace rg
