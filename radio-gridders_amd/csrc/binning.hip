// binning.hip -- scan kernels of the device-side counting sort.
#include <algorithm>

#include "binning.hpp"

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

__device__ inline uint32_t items_of(uint32_t c, uint32_t per_item)
{
    return (c + per_item - 1) / per_item;
}

// Exclusive scan over the SCAN_BLOCK threads of (x, y) pairs: wavefront scans
// by shuffles, then the wavefronts' totals through LDS (two barriers).
__device__ inline uint2 scan_block(uint2 v, uint2 &total, uint2 *wtot /* SCAN_BLOCK / 64 */)
{
    const int lane = __lane_id(), wv = threadIdx.x / 64;
    uint2 inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t x = (uint32_t)__shfl_up((int)inc.x, o);
        const uint32_t y = (uint32_t)__shfl_up((int)inc.y, o);
        if (lane >= o) {
            inc.x += x;
            inc.y += y;
        }
    }
    __syncthreads(); // wtot of an earlier call has been read
    if (lane == 63)
        wtot[wv] = inc;
    __syncthreads();
    uint2 before = make_uint2(0, 0);
    total = make_uint2(0, 0);
#pragma unroll
    for (int k = 0; k < SCAN_BLOCK / 64; ++k) {
        const uint2 t = wtot[k];
        if (k < wv) {
            before.x += t.x;
            before.y += t.y;
        }
        total.x += t.x;
        total.y += t.y;
    }
    return make_uint2(before.x + inc.x - v.x, before.y + inc.y - v.y);
}

// Counts of keys k0 .. k0 + PER - 1 (0 past the last key) in every replica:
// all loads issued together, a run of four keys as one 16-byte load (k0 is a
// multiple of PER and the replicas lie a multiple of 64 counters apart).
template <int NREP, int PER>
__device__ inline void load_counts(const uint32_t *count, int64_t stride, int64_t nkeys, int64_t k0,
                                   uint32_t c[NREP][PER])
{
#pragma unroll
    for (int r = 0; r < NREP; ++r)
#pragma unroll
        for (int j = 0; j < PER; ++j)
            c[r][j] = 0;
    if (PER == 4 && k0 + PER <= nkeys) {
#pragma unroll
        for (int r = 0; r < NREP; ++r) {
            const uint4 v = *reinterpret_cast<const uint4 *>(count + r * stride + k0);
            c[r][0] = v.x;
            c[r][1 % PER] = v.y;
            c[r][2 % PER] = v.z;
            c[r][3 % PER] = v.w;
        }
    } else {
#pragma unroll
        for (int r = 0; r < NREP; ++r)
#pragma unroll
            for (int j = 0; j < PER; ++j)
                if (k0 + j < nkeys)
                    c[r][j] = count[r * stride + k0 + j];
    }
}

// Phase 1: block b's totals of (count, items).
template <int NREP, int PER>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_reduce(const uint32_t *count, int64_t stride,
                                                            int64_t nkeys, uint32_t per_item,
                                                            uint2 *block_sums)
{
    __shared__ uint2 wtot[SCAN_BLOCK / 64];
    const int64_t k0 = ((int64_t)blockIdx.x * SCAN_BLOCK + threadIdx.x) * PER;
    uint32_t c[NREP][PER];
    load_counts<NREP, PER>(count, stride, nkeys, k0, c);
    uint2 acc = make_uint2(0, 0);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        uint32_t t = 0;
#pragma unroll
        for (int r = 0; r < NREP; ++r)
            t += c[r][j];
        acc.x += t;
        acc.y += items_of(t, per_item);
    }
    uint2 total;
    scan_block(acc, total, wtot);
    if (threadIdx.x == 0)
        block_sums[blockIdx.x] = total;
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

// Phase 3: per-key starts, work items and the scatter cursors of every
// replica.  `direct`: block_sums holds block totals, of which the block adds
// up those before it itself (one launch less, and nothing waits for a single
// workgroup); otherwise their exclusive prefixes.  A key of more than two
// items (hot tiles have thousands of records) has them written by its whole
// wavefront.
template <int NREP, int PER>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_down(
    const uint32_t *count, int64_t stride, int64_t nkeys, uint32_t per_item,
    const uint2 *block_sums, int direct, uint32_t *vis_start, uint32_t *item_start,
    uint32_t *cursor, Item *items, unsigned long long *stats)
{
    __shared__ uint2 wtot[SCAN_BLOCK / 64];
    const int64_t k0 = ((int64_t)blockIdx.x * SCAN_BLOCK + threadIdx.x) * PER;
    uint32_t c[NREP][PER];
    load_counts<NREP, PER>(count, stride, nkeys, k0, c);
    uint2 before = make_uint2(0, 0);
    if (direct) {
        uint2 p = make_uint2(0, 0);
        for (int b = threadIdx.x; b < (int)blockIdx.x; b += SCAN_BLOCK) {
            const uint2 v = block_sums[b];
            p.x += v.x;
            p.y += v.y;
        }
        scan_block(p, before, wtot);
    } else {
        before = block_sums[blockIdx.x];
    }
    uint32_t tot[PER];
    uint2 acc = make_uint2(0, 0);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        tot[j] = 0;
#pragma unroll
        for (int r = 0; r < NREP; ++r)
            tot[j] += c[r][j];
        acc.x += tot[j];
        acc.y += items_of(tot[j], per_item);
    }
    uint2 total;
    uint2 run = scan_block(acc, total, wtot);
    run.x += before.x;
    run.y += before.y;
    uint32_t vs[PER], is[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        vs[j] = run.x;
        is[j] = run.y;
        run.x += tot[j];
        run.y += items_of(tot[j], per_item);
        // counts to the replicas' cursors
        uint32_t cur = vs[j];
#pragma unroll
        for (int r = 0; r < NREP; ++r) {
            const uint32_t t = c[r][j];
            c[r][j] = cur;
            cur += t;
        }
    }
    if (PER == 4 && k0 + PER <= nkeys) {
        *reinterpret_cast<uint4 *>(vis_start + k0) =
            make_uint4(vs[0], vs[1 % PER], vs[2 % PER], vs[3 % PER]);
        *reinterpret_cast<uint4 *>(item_start + k0) =
            make_uint4(is[0], is[1 % PER], is[2 % PER], is[3 % PER]);
        if (cursor)
#pragma unroll
            for (int r = 0; r < NREP; ++r)
                *reinterpret_cast<uint4 *>(cursor + r * stride + k0) =
                    make_uint4(c[r][0], c[r][1 % PER], c[r][2 % PER], c[r][3 % PER]);
    } else {
#pragma unroll
        for (int j = 0; j < PER; ++j)
            if (k0 + j < nkeys) {
                vis_start[k0 + j] = vs[j];
                item_start[k0 + j] = is[j];
                if (cursor)
#pragma unroll
                    for (int r = 0; r < NREP; ++r)
                        cursor[r * stride + k0 + j] = c[r][j];
            }
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const uint32_t ni = items_of(tot[j], per_item);
        auto put = [&](uint32_t key, uint32_t start, uint32_t cnt, uint32_t i0, uint32_t q) {
            Item it;
            it.key = key;
            it.start = start + q * per_item;
            it.count = min(per_item, cnt - q * per_item);
            items[i0 + q] = it;
        };
        if (ni <= 2)
            for (uint32_t q = 0; q < ni; ++q)
                put((uint32_t)(k0 + j), vs[j], tot[j], is[j], q);
        for (unsigned long long m = __ballot(ni > 2); m; m &= m - 1) {
            const int src = __ffsll((long long)m) - 1;
            const uint32_t key = (uint32_t)(k0 + j) + (uint32_t)(src - __lane_id()) * PER;
            const uint32_t st = (uint32_t)__shfl((int)vs[j], src);
            const uint32_t cn = (uint32_t)__shfl((int)tot[j], src);
            const uint32_t i0 = (uint32_t)__shfl((int)is[j], src);
            for (uint32_t q = __lane_id(); q < items_of(cn, per_item); q += 64)
                put(key, st, cn, i0, q);
        }
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        vis_start[nkeys] = before.x + total.x;
        item_start[nkeys] = before.y + total.y;
        stats[CNT_RECORDS] = before.x + total.x;
        stats[CNT_ITEMS] = before.y + total.y;
    }
}

// Keys per scan thread: one while the key space is small (more workgroups, the
// latency of their loads is all there is: 4225 keys in 16 replicas 17 -> 4 us
// a phase), four from 64 K keys.
static int scan_per_thread(int64_t nkeys) { return nkeys >= 65536 ? 4 : 1; }

int64_t scan_blocks(int64_t nkeys)
{
    const int64_t tile = SCAN_BLOCK * scan_per_thread(nkeys);
    return (nkeys + tile - 1) / tile;
}

size_t scan_sums_bytes(int64_t nkeys)
{
    return sizeof(uint2) * (size_t)(std::max<int64_t>(scan_blocks(nkeys), 65536 / SCAN_BLOCK) + 1);
}

template <int NREP, int PER>
static int scan_t(const uint32_t *count, int64_t stride, int64_t nkeys, uint32_t per_item,
                  uint2 *bsums, uint32_t *vis_start, uint32_t *item_start, uint32_t *cursor,
                  Item *items, unsigned long long *stats, hipStream_t s)
{
    const int64_t nb = scan_blocks(nkeys);
    // every block reads the totals before it while that stays below 16 MB in all
    const int direct = nb <= SCAN_DIRECT;
    if (nb > 1)
        hipLaunchKernelGGL((k_scan_reduce<NREP, PER>), dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s,
                           count, stride, nkeys, per_item, bsums);
    if (!direct)
        hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(1024), 0, s, bsums, (int)nb);
    hipLaunchKernelGGL((k_scan_down<NREP, PER>), dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, count,
                       stride, nkeys, per_item, (const uint2 *)bsums, direct, vis_start, item_start,
                       cursor, items, stats);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

int scan_keys(const uint32_t *count, Replicas rp, int64_t nkeys, uint32_t per_item, uint2 *bsums,
              uint32_t *vis_start, uint32_t *item_start, uint32_t *cursor, Item *items,
              unsigned long long *stats, hipStream_t s)
{
    auto run = [&](auto nrep) {
        constexpr int NREP = decltype(nrep)::value;
        return scan_per_thread(nkeys) == 4
                   ? scan_t<NREP, 4>(count, rp.stride, nkeys, per_item, bsums, vis_start,
                                     item_start, cursor, items, stats, s)
                   : scan_t<NREP, 1>(count, rp.stride, nkeys, per_item, bsums, vis_start,
                                     item_start, cursor, items, stats, s);
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
    pl.rp.stride = (nkeys + 1 + 63) / 64 * 64;
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

int items_from_lengths(rg_context *ctx, const uint32_t *len, int64_t nkeys, uint32_t per_item,
                       uint32_t *prefix, uint32_t *item_start, Item *items, hipStream_t s)
{
    const int64_t nblocks_scan = nkeys > 0 ? scan_blocks(nkeys) : 0;
    if (nkeys <= 0 || nblocks_scan > 1024 * 256)
        return fail(RG_ERR_PARAM, "invalid key space %lld", (long long)nkeys);
    RG_TRY(ensure_counters(ctx));
    RG_TRY(ctx->scratch[6].ensure(scan_sums_bytes(nkeys)));
    Replicas one;
    one.mask = 0;
    one.stride = nkeys + 1;
    // one replica: its cursors would be the prefix again
    return scan_keys(len, one, nkeys, per_item, ctx->scratch[6].as<uint2>(), prefix, item_start,
                     nullptr, items, ctx->counters.as<unsigned long long>(), s);
}

} // namespace rg
