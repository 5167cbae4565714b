// binning_impl.hpp -- definitions of the sort in binning.hpp (included once
// per translation unit that instantiates bin_visibilities).
#pragma once

#include <algorithm>

#include "binning.hpp"

namespace rg {

template <typename Keyer, typename T>
int bin_run(const Keyer &kf, int64_t n, int64_t nkeys, uint32_t per_item, const BinPlan &pl,
            const BinBufs &b, ZeroList &zero, rg_context *timer_ctx, hipStream_t s, BinResult &out)
{
    const Replicas rp = pl.rp;
    out.vis_start = b.vis_start;
    out.item_start = b.item_start;
    out.items = b.items;
    out.recs = b.recs;
    out.max_items = pl.max_items;
    const bool small = bin_small(n, nkeys);
    RG_TRY(zero.launch(s));
    KernelTimer kt(timer_ctx, RG_TIMER_BINNING, s);
    if (small) {
        hipLaunchKernelGGL((k_bin_small<Keyer, T>), dim3(1), dim3(1024), 0, s, kf, (int)n,
                           (int)nkeys, per_item, b.vis_start, b.item_start, b.items,
                           (Rec<T> *)b.recs, out.group_start, out.group_keys, b.stats);
        RG_HIP(hipGetLastError());
        return RG_OK;
    }

    const int64_t nb = (n + BIN_CHUNK - 1) / BIN_CHUNK;
    if (nb > 0)
        hipLaunchKernelGGL((k_bin_count<Keyer>), dim3((unsigned)nb), dim3(BIN_TB), 0, s, kf, n,
                           b.count, rp, b.krp, b.stats);
    RG_HIP(hipGetLastError());
    RG_TRY(scan_keys(b.count, rp, nkeys, per_item, b.bsums, b.vis_start, b.item_start, b.cursor,
                     b.items, b.stats, s, out.group_start, out.group_keys));
    if (nb > 0)
        hipLaunchKernelGGL((k_bin_scatter<Keyer, T>), dim3((unsigned)nb), dim3(BIN_TB), 0, s, kf, n,
                           (const uint32_t *)b.cursor, rp, (const uint4 *)b.krp,
                           (Rec<T> *)b.recs);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

// context scratch slots of the sort (rg_internal.hpp)
static const int bin_slot[BIN__N] = {0, 1, 2, 3, 4, 5, 6, 15};
inline void *bin_buffer(rg_context *ctx, BinArray k) { return ctx->scratch[bin_slot[k]].p; }

template <typename T>
int bin_prepare(rg_context *ctx, int64_t n, int64_t nkeys, int64_t key_room, uint32_t per_item,
                int64_t max_counters, ZeroList &zero, BinPlan &pl, int64_t min_items)
{
    RG_TRY(bin_plan(n, nkeys, per_item, max_counters, sizeof(Rec<T>), pl));
    RG_TRY(ensure_counters(ctx));
    // items and scan sums: room for every call of up to this many visibilities
    // and keys, whatever item size it picks (scratch that a captured graph holds
    // cannot grow; a shorter stream, below 12 512^2, has at most 48 K items, K up to 256);
    // counters likewise: fewer keys, or another gridder's, may take more replicas
    auto counters = [](int64_t keys, int64_t most) {
        const int64_t stride = bin_stride(keys);
        return sizeof(uint32_t) * (size_t)std::max(stride, std::min(16 * stride, most));
    };
    const size_t count_bytes = pl.bytes[BIN_COUNT];
    for (int k : {BIN_COUNT, BIN_CURSOR})
        pl.bytes[k] =
            std::max(counters(nkeys, max_counters), counters(key_room, BIN_MAX_COUNTERS));
    key_room = std::max(key_room, nkeys);
    const int64_t items = std::max(
        min_items, key_room + std::max<int64_t>({n / per_item, 12288, n / 512}) + 1);
    for (int k : {BIN_VIS_START, BIN_ITEM_START})
        pl.bytes[k] = sizeof(uint32_t) * (size_t)(key_room + 1);
    pl.bytes[BIN_ITEMS] = sizeof(Item) * (size_t)items;
    pl.bytes[BIN_BSUMS] = scan_sums_bytes(key_room);
    DevBuf *buf[BIN__N];
    for (int k = 0; k < BIN__N; ++k)
        buf[k] = &ctx->scratch[bin_slot[k]];
    RG_TRY(ensure_together(buf, pl.bytes, BIN__N, (size_t)16 << 20));
    if (!bin_small(n, nkeys))
        RG_TRY(zero.add(ctx->scratch[bin_slot[BIN_COUNT]].p, count_bytes));
    return RG_OK;
}

template <typename Keyer, typename T>
int bin_visibilities(rg_context *ctx, const Keyer &kf, int64_t n, int64_t nkeys, int64_t key_room,
                     uint32_t per_item, ZeroList &zero, hipStream_t s, BinResult &out,
                     int64_t max_counters, const BinPlan *ready)
{
    BinPlan pl;
    if (ready)
        pl = *ready;
    else
        RG_TRY(bin_prepare<T>(ctx, n, nkeys, key_room, per_item, max_counters, zero, pl));
    const int *slot = bin_slot;
    BinBufs b;
    b.count = ctx->scratch[slot[BIN_COUNT]].as<uint32_t>();
    b.vis_start = ctx->scratch[slot[BIN_VIS_START]].as<uint32_t>();
    b.item_start = ctx->scratch[slot[BIN_ITEM_START]].as<uint32_t>();
    b.cursor = ctx->scratch[slot[BIN_CURSOR]].as<uint32_t>();
    b.items = ctx->scratch[slot[BIN_ITEMS]].as<Item>();
    b.recs = ctx->scratch[slot[BIN_RECS]].p;
    b.bsums = ctx->scratch[slot[BIN_BSUMS]].as<uint2>();
    b.krp = ctx->scratch[slot[BIN_KRP]].as<uint4>();
    b.stats = ctx->counters.as<unsigned long long>();
    return bin_run<Keyer, T>(kf, n, nkeys, per_item, pl, b, zero, ctx, s, out);
}

} // namespace rg
