// scan.hpp -- exclusive scan of per-key record counts into record starts, work
// items and what a source derives from them (device code and launches).
//
// A source gives the counts of PER consecutive keys (in NREP parts that are
// summed), and takes each key's first record and each part's start back:
//   load(nkeys, k0, c)               c[r][j] = part r of key k0 + j, 0 past the last key
//   store(nkeys, k0, start, c, tot)  start[j] first record of the key, c[r][j] start of
//                                    part r, tot[j] its records (whole wavefronts call)
//   finish(nkeys, total, stats)      once, by one thread
// and may choose the records per work item of a key of c records, and see each
// item put:
//   item_size(c, per_item)
//   item_put(index, size, per_item)
#pragma once

#include "binning.hpp"

namespace rg {

__device__ inline uint32_t items_of(uint32_t c, uint32_t per_item)
{
    return (c + per_item - 1) / per_item;
}

struct FixedItems {
    __device__ static uint32_t item_size(uint32_t, uint32_t per_item) { return per_item; }
    __device__ static void item_put(uint32_t, uint32_t, uint32_t) {}
};

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
                                   uint32_t (&c)[NREP][PER])
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

// v[j] to dst[k0 + j], keys past the last left out
template <int PER>
__device__ inline void store_keys(uint32_t *dst, int64_t nkeys, int64_t k0,
                                  const uint32_t (&v)[PER])
{
    if (PER == 4 && k0 + PER <= nkeys) {
        *reinterpret_cast<uint4 *>(dst + k0) =
            make_uint4(v[0], v[1 % PER], v[2 % PER], v[3 % PER]);
    } else {
#pragma unroll
        for (int j = 0; j < PER; ++j)
            if (k0 + j < nkeys)
                dst[k0 + j] = v[j];
    }
}

template <int NREPS, typename Items = FixedItems> struct CountSource : Items {
    static constexpr int NREP = NREPS;
    const uint32_t *count; // NREP replicas, stride apart
    int64_t stride;
    uint32_t *vis_start, *cursor; // cursor: as count, or NULL
    uint32_t *group_start;        // first record of every group_keys keys, or NULL
    int group_keys;

    template <int PER>
    __device__ void load(int64_t nkeys, int64_t k0, uint32_t (&c)[NREP][PER]) const
    {
        load_counts<NREP, PER>(count, stride, nkeys, k0, c);
    }
    template <int PER>
    __device__ void store(int64_t nkeys, int64_t k0, const uint32_t (&vs)[PER],
                          const uint32_t (&c)[NREP][PER], const uint32_t (&)[PER]) const
    {
        store_keys<PER>(vis_start, nkeys, k0, vs);
        if (group_start)
#pragma unroll
            for (int j = 0; j < PER; ++j)
                if (k0 + j < nkeys && ((k0 + j) & (group_keys - 1)) == 0)
                    group_start[(k0 + j) / group_keys] = vs[j];
        if (cursor)
#pragma unroll
            for (int r = 0; r < NREP; ++r)
                store_keys<PER>(cursor + r * stride, nkeys, k0, c[r]);
    }
    __device__ void finish(int64_t nkeys, uint32_t total, unsigned long long *) const
    {
        vis_start[nkeys] = total;
        if (group_start)
            group_start[nkeys / group_keys] = total;
    }
};

// Phase 1: block b's totals of (count, items).
template <typename Src, int PER>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_reduce(Src src, int64_t nkeys,
                                                            uint32_t per_item, uint2 *block_sums)
{
    constexpr int NREP = Src::NREP;
    __shared__ uint2 wtot[SCAN_BLOCK / 64];
    const int64_t k0 = ((int64_t)blockIdx.x * SCAN_BLOCK + threadIdx.x) * PER;
    uint32_t c[NREP][PER];
    src.load(nkeys, k0, c);
    uint2 acc = make_uint2(0, 0);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        uint32_t t = 0;
#pragma unroll
        for (int r = 0; r < NREP; ++r)
            t += c[r][j];
        acc.x += t;
        acc.y += items_of(t, src.item_size(t, per_item));
    }
    uint2 total;
    scan_block(acc, total, wtot);
    if (threadIdx.x == 0)
        block_sums[blockIdx.x] = total;
}

// Phase 3: per-key starts, work items and the source's own results.  `direct`: block_sums holds block totals, of which the block adds
// up those before it itself (one launch less, and nothing waits for a single
// workgroup); otherwise their exclusive prefixes.  A key of more than two
// items (hot tiles have thousands of records) has them written by its whole
// wavefront.
template <typename Src, int PER>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_down(
    Src src, int64_t nkeys, uint32_t per_item, const uint2 *block_sums, int direct,
    uint32_t *item_start, Item *items, unsigned long long *stats)
{
    constexpr int NREP = Src::NREP;
    __shared__ uint2 wtot[SCAN_BLOCK / 64];
    const int64_t k0 = ((int64_t)blockIdx.x * SCAN_BLOCK + threadIdx.x) * PER;
    uint32_t c[NREP][PER];
    src.load(nkeys, k0, c);
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
        acc.y += items_of(tot[j], src.item_size(tot[j], per_item));
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
        run.y += items_of(tot[j], src.item_size(tot[j], per_item));
        // counts to the replicas' cursors
        uint32_t cur = vs[j];
#pragma unroll
        for (int r = 0; r < NREP; ++r) {
            const uint32_t t = c[r][j];
            c[r][j] = cur;
            cur += t;
        }
    }
    store_keys<PER>(item_start, nkeys, k0, is);
    src.store(nkeys, k0, vs, c, tot);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const uint32_t ni = items_of(tot[j], src.item_size(tot[j], per_item));
        auto put = [&](uint32_t key, uint32_t start, uint32_t cnt, uint32_t i0, uint32_t q) {
            const uint32_t size = src.item_size(cnt, per_item);
            Item it;
            it.key = key;
            it.start = start + q * size;
            it.count = min(size, cnt - q * size);
            items[i0 + q] = it;
            src.item_put(i0 + q, size, per_item);
        };
        if (ni <= 2)
            for (uint32_t q = 0; q < ni; ++q)
                put((uint32_t)(k0 + j), vs[j], tot[j], is[j], q);
        for (unsigned long long m = __ballot(ni > 2); m; m &= m - 1) {
            const int from = __ffsll((long long)m) - 1;
            const uint32_t key = (uint32_t)(k0 + j) + (uint32_t)(from - __lane_id()) * PER;
            const uint32_t st = (uint32_t)__shfl((int)vs[j], from);
            const uint32_t cn = (uint32_t)__shfl((int)tot[j], from);
            const uint32_t i0 = (uint32_t)__shfl((int)is[j], from);
            const uint32_t nq = items_of(cn, src.item_size(cn, per_item));
            for (uint32_t q = __lane_id(); q < nq; q += 64)
                put(key, st, cn, i0, q);
        }
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        src.finish(nkeys, before.x + total.x, stats);
        item_start[nkeys] = before.y + total.y;
        stats[CNT_RECORDS] = before.x + total.x;
        stats[CNT_ITEMS] = before.y + total.y;
    }
}

// The scan of a source's counts: reduce (none for one block), totals of many
// blocks, down.
template <typename Src, int PER>
static int scan_source_per(const Src &src, int64_t nkeys, uint32_t per_item, uint2 *bsums,
                           uint32_t *item_start, Item *items, unsigned long long *stats,
                           hipStream_t s)
{
    const int64_t nb = scan_blocks(nkeys);
    // every block reads the totals before it while that stays below 16 MB in all
    const int direct = nb <= SCAN_DIRECT;
    if (nb > 1)
        hipLaunchKernelGGL((k_scan_reduce<Src, PER>), dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s,
                           src, nkeys, per_item, bsums);
    if (!direct)
        RG_TRY(launch_scan_blocks(bsums, nb, s));
    hipLaunchKernelGGL((k_scan_down<Src, PER>), dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, src,
                       nkeys, per_item, (const uint2 *)bsums, direct, item_start, items, stats);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

template <typename Src>
static int scan_source(const Src &src, int64_t nkeys, uint32_t per_item, uint2 *bsums,
                       uint32_t *item_start, Item *items, unsigned long long *stats, hipStream_t s)
{
    return scan_per_thread(nkeys) == 4
               ? scan_source_per<Src, 4>(src, nkeys, per_item, bsums, item_start, items, stats, s)
               : scan_source_per<Src, 1>(src, nkeys, per_item, bsums, item_start, items, stats, s);
}

} // namespace rg
