// binning.hpp -- device-side counting sort of visibilities into work items.
//
// A "keyer" maps visibility i to (key, packed tile position, kernel-tap
// index).  Keys are dense in [0, nkeys).  The sort is:
//   count   : wave-aggregated atomics on count[rep][key]; each visibility
//             keeps the counter value it got (its rank inside the replica's
//             share of the key) with its key, position and tap index
//   scan    : exclusive scan of (count, ceil(count / K)), where count[key] is
//             the sum over the replicas, then the start of every replica's
//             share of every key and one work item per K records of a key
//   scatter : record i written at start[rep][key] + rank (no atomics)
// Chunk c of BIN_CHUNK visibilities uses counter replica rep = c mod NREP.
// Device-scope atomics on one address serialise, and a few keys (the
// short-baseline tiles at the uv centre) take thousands of wavefront updates,
// so the counters of a key are spread over NREP separate arrays; replica
// rep's records of a key follow those of replicas 0..rep-1.
// Consecutive visibilities of a wavefront that share a key keep their stream
// order, so baseline-track runs stay contiguous inside a key (the locality
// the W-projection Romein accumulation relies on).
#pragma once

#include <algorithm>

#include "rg_internal.hpp"

namespace rg {

constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_DIRECT = 2048; // scan blocks that add up the totals before them themselves

struct Item {
    uint32_t key;
    uint32_t start; // first record
    uint32_t count; // records
};

template <typename T> struct Vec2;
template <> struct Vec2<float> { using type = float2; };
template <> struct Vec2<double> { using type = double2; };

template <typename T> struct Rec {
    uint32_t pos;  // tile-local footprint top-left: lx | ly << 16
    uint32_t kidx; // sub-kernel (plane * R + yf) * R + xf; W-projection: its byte offset
    typename Vec2<T>::type vis;
};

// VIS_OVERFLOW: outside a capacity the call was sized for (counted as dropped
// and as an overrun of the call)
enum VisStatus { VIS_OK = 0, VIS_DROPPED = 1, VIS_BAD_PLANE = 2, VIS_OVERFLOW = 3 };

// A run is a maximal stretch of consecutive active lanes with the same key;
// its first lane (the head) adds the run length to the key's counter with one
// atomic.  All runs of the wavefront issue their atomics in one instruction
// and the results are gathered once, so a wavefront costs one atomic round
// trip whatever its keys (visibility streams are baseline-track ordered, so
// neighbouring lanes often share keys).  Where the runs are short, lanes of one key wherever
// they stand are gathered first, a few keys at a time: a crowded tile's records that alternate
// between plane groups or tiles would otherwise meet on a few counters one by one (3 M records
// of 4 tiles and 2 groups in random order: a call of 1104 us with runs alone, 527 us so; from the first
// key of a single lane on the rest stays as it is, so that streams of many keys pay for one look).
// wave_agg_issue returns the atomic's old value (meaningful on head lanes), the lane's head and
// its place among the head's; wave_agg_rank turns them into the lane's rank.  Splitting the
// two lets a thread keep several atomics in flight.  Must be called by the whole wavefront in
// uniform control flow.
struct AggPlace {
    int head, off;
};
constexpr int AGG_RUNS = 16; // runs of a wavefront that are short
constexpr int AGG_SAME = 2;  // lanes of one key worth gathering

__device__ inline uint32_t wave_agg_issue(uint32_t *counters, uint32_t key, bool active,
                                          AggPlace &place)
{
    const int lane = __lane_id();
    const unsigned long long below = (1ull << lane) - 1ull;
    const uint32_t prev = (uint32_t)__shfl_up((int)key, 1);
    unsigned long long act = __ballot(active);
    auto run_heads = [&]() {
        return __ballot(((act >> lane) & 1ull) &&
                        (lane == 0 || !((act >> (lane - 1)) & 1ull) || prev != key));
    };
    unsigned long long heads = run_heads();
    unsigned long long mine = 0; // gathered: the lanes of this lane's key
    if (__popcll(heads) > AGG_RUNS) {
        for (unsigned long long left = act; left;) {
            const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)key, __ffsll((long long)left) - 1);
            const unsigned long long same = __ballot(key == k) & left;
            if (__popcll(same) < AGG_SAME)
                break;
            if (key == k)
                mine = same;
            left &= ~same;
            act &= ~same;
        }
        mine = active ? mine : 0;
        heads = run_heads();
    }
    uint32_t base = 0;
    const bool leader = mine && !(mine & below);
    if (leader || ((heads >> lane) & 1ull)) {
        const unsigned long long ends = heads | ~act; // a run stops at the next head or idle lane
        const unsigned long long nxt = lane == 63 ? 0ull : (ends >> (lane + 1));
        const uint32_t len = leader ? (uint32_t)__popcll(mine)
                             : nxt  ? (uint32_t)__ffsll((long long)nxt)
                                    : (uint32_t)(64 - lane);
        base = atomicAdd(&counters[key], len);
    }
    const unsigned long long hm = heads & (below | 1ull << lane);
    place.head = mine ? __ffsll((long long)mine) - 1 : hm ? 63 - __clzll((long long)hm) : 0;
    place.off = mine ? __popcll(mine & below) : lane - place.head;
    return base;
}

__device__ inline uint32_t wave_agg_rank(uint32_t base, const AggPlace &place)
{
    return (uint32_t)__shfl((int)base, place.head) + (uint32_t)place.off;
}

// Both steps; the rank only when `want` (uniform) is set.
__device__ inline uint32_t wave_agg_add(uint32_t *counters, uint32_t key, bool active, bool want)
{
    AggPlace place;
    const uint32_t base = wave_agg_issue(counters, key, active, place);
    return want ? wave_agg_rank(base, place) : 0u;
}

// counters of a sort in all, at most (unless its keys are more)
constexpr int64_t BIN_MAX_COUNTERS = (int64_t)1 << 22;

// Counter replicas: NREP arrays of `stride` entries (stride >= nkeys + 1).
struct Replicas {
    uint32_t mask;   // NREP - 1, NREP a power of two
    int64_t stride;
};

// Per visibility after the count pass: key (KEY_NONE if not gridded), rank,
// packed position, tap index.
constexpr uint32_t KEY_NONE = 0xffffffffu;

// Count and scatter workgroups take BIN_CHUNK consecutive visibilities,
// BIN_VPT per thread (visibility chunk + q BIN_TB + thread, so the lanes of a
// wavefront hold consecutive visibilities); chunk c uses counter replica
// c mod NREP.
constexpr int BIN_TB = 256;
constexpr int BIN_VPT = 4;
constexpr int BIN_CHUNK = BIN_TB * BIN_VPT;

template <typename Keyer>
__global__ __launch_bounds__(BIN_TB) void k_bin_count(Keyer kf, int64_t n, uint32_t *count,
                                                      Replicas rp, uint4 *krp,
                                                      unsigned long long *stats)
{
    const int64_t i0 = (int64_t)blockIdx.x * BIN_CHUNK + threadIdx.x;
    uint32_t *cnt = count + (blockIdx.x & rp.mask) * rp.stride;
    uint32_t key[BIN_VPT], pos[BIN_VPT], kidx[BIN_VPT], base[BIN_VPT];
    int st[BIN_VPT];
    AggPlace place[BIN_VPT];
#pragma unroll
    for (int q = 0; q < BIN_VPT; ++q) {
        const int64_t i = i0 + q * BIN_TB;
        key[q] = pos[q] = kidx[q] = 0;
        st[q] = i < n ? kf.classify(i, key[q], pos[q], kidx[q]) : VIS_DROPPED;
    }
    // every atomic in flight before the first result is used
#pragma unroll
    for (int q = 0; q < BIN_VPT; ++q)
        base[q] = wave_agg_issue(cnt, key[q], i0 + q * BIN_TB < n && st[q] == VIS_OK, place[q]);
    uint32_t dropped = 0, badp = 0, over = 0;
#pragma unroll
    for (int q = 0; q < BIN_VPT; ++q) {
        const int64_t i = i0 + q * BIN_TB;
        const bool in = i < n, ok = in && st[q] == VIS_OK;
        const uint32_t rank = wave_agg_rank(base[q], place[q]);
        if (in)
            krp[i] = make_uint4(ok ? key[q] : KEY_NONE, rank, pos[q], kidx[q]);
        // per-wave status counts
        dropped += (uint32_t)__popcll(__ballot(in && (st[q] == VIS_DROPPED || st[q] == VIS_OVERFLOW)));
        badp += (uint32_t)__popcll(__ballot(in && st[q] == VIS_BAD_PLANE));
        over += (uint32_t)__popcll(__ballot(in && st[q] == VIS_OVERFLOW));
    }
    if (__lane_id() == 0) {
        if (dropped)
            atomicAdd(&stats[CNT_DROPPED], (unsigned long long)dropped);
        if (badp)
            atomicAdd(&stats[CNT_BAD_PLANE], (unsigned long long)badp);
        if (over)
            atomicAdd(&stats[CNT_OVERFLOW], (unsigned long long)over);
    }
}

// Same grid and chunks as k_bin_count.
template <typename Keyer, typename T>
__global__ __launch_bounds__(BIN_TB) void k_bin_scatter(Keyer kf, int64_t n,
                                                        const uint32_t *start, Replicas rp,
                                                        const uint4 *__restrict__ krp,
                                                        Rec<T> *recs)
{
    const int64_t i0 = (int64_t)blockIdx.x * BIN_CHUNK + threadIdx.x;
    const uint32_t *st = start + (blockIdx.x & rp.mask) * rp.stride;
    uint4 e[BIN_VPT];
    typename Vec2<T>::type v[BIN_VPT];
#pragma unroll
    for (int q = 0; q < BIN_VPT; ++q) {
        const int64_t i = i0 + q * BIN_TB;
        e[q] = make_uint4(KEY_NONE, 0, 0, 0);
        if (i < n) {
            e[q] = krp[i];
            v[q] = kf.template vis_value<T>(i);
        }
    }
#pragma unroll
    for (int q = 0; q < BIN_VPT; ++q) {
        if (e[q].x == KEY_NONE)
            continue;
        Rec<T> r;
        r.pos = e[q].z;
        r.kidx = e[q].w;
        r.vis = v[q];
        recs[st[e[q].x] + e[q].y] = r;
    }
}

// ---- short streams -------------------------------------------------------------------
// Up to BIN_SMALL visibilities over at most BIN_SMALL_KEYS keys are sorted by
// one workgroup with its counters in LDS: one launch instead of a clear, a
// count, two scans and a scatter, whose latencies are all there is to a short
// call (448 visibilities, 25 keys: 31 us -> one launch of about 8 us).
constexpr int BIN_SMALL_VPT = 4;
constexpr int BIN_SMALL_KPT = 8;
constexpr int BIN_SMALL = 1024 * BIN_SMALL_VPT;
constexpr int BIN_SMALL_KEYS = 1024 * BIN_SMALL_KPT;
inline bool bin_small(int64_t n, int64_t nkeys)
{
    return n <= BIN_SMALL && nkeys <= BIN_SMALL_KEYS;
}

template <typename Keyer, typename T>
__global__ __launch_bounds__(1024) void k_bin_small(Keyer kf, int n, int nkeys, uint32_t per_item,
                                                    uint32_t *vis_start, uint32_t *item_start,
                                                    Item *items, Rec<T> *recs,
                                                    uint32_t *group_start, int group_keys,
                                                    unsigned long long *stats)
{
    __shared__ uint32_t cnt[BIN_SMALL_KEYS];
    __shared__ uint2 wtot[16];
    __shared__ uint32_t s_stat[3];
    for (int k = threadIdx.x; k < nkeys; k += 1024)
        cnt[k] = 0;
    if (threadIdx.x < 3)
        s_stat[threadIdx.x] = 0;
    __syncthreads();
    uint32_t key[BIN_SMALL_VPT], rank[BIN_SMALL_VPT];
    Rec<T> rec[BIN_SMALL_VPT];
#pragma unroll
    for (int q = 0; q < BIN_SMALL_VPT; ++q) {
        const int i = q * 1024 + (int)threadIdx.x;
        key[q] = KEY_NONE;
        if (i < n) {
            uint32_t k = 0, pos = 0, kidx = 0;
            const int st = kf.classify(i, k, pos, kidx);
            if (st == VIS_OK) {
                key[q] = k;
                rank[q] = atomicAdd(&cnt[k], 1u);
                rec[q].pos = pos;
                rec[q].kidx = kidx;
                rec[q].vis = kf.template vis_value<T>(i);
            } else {
                atomicAdd(&s_stat[st == VIS_BAD_PLANE ? 1 : 0], 1u);
                if (st == VIS_OVERFLOW)
                    atomicAdd(&s_stat[2], 1u);
            }
        }
    }
    __syncthreads();
    // exclusive scan of (records, items) over the keys, BIN_SMALL_KPT per thread
    const int k0 = (int)threadIdx.x * BIN_SMALL_KPT;
    const int lane = __lane_id(), wv = threadIdx.x / 64;
    uint2 acc = make_uint2(0, 0);
    uint32_t c[BIN_SMALL_KPT];
#pragma unroll
    for (int j = 0; j < BIN_SMALL_KPT; ++j) {
        c[j] = k0 + j < nkeys ? cnt[k0 + j] : 0u;
        acc.x += c[j];
        acc.y += (c[j] + per_item - 1) / per_item;
    }
    uint2 inc = acc;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t x = (uint32_t)__shfl_up((int)inc.x, o);
        const uint32_t y = (uint32_t)__shfl_up((int)inc.y, o);
        if (lane >= o) {
            inc.x += x;
            inc.y += y;
        }
    }
    if (lane == 63)
        wtot[wv] = inc;
    __syncthreads();
    uint2 run = make_uint2(inc.x - acc.x, inc.y - acc.y), total = make_uint2(0, 0);
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        const uint2 t = wtot[w];
        if (w < wv) {
            run.x += t.x;
            run.y += t.y;
        }
        total.x += t.x;
        total.y += t.y;
    }
#pragma unroll
    for (int j = 0; j < BIN_SMALL_KPT; ++j) {
        const int k = k0 + j;
        if (k < nkeys) {
            cnt[k] = run.x;
            if (group_start && (k & (group_keys - 1)) == 0)
                group_start[k / group_keys] = run.x;
            vis_start[k] = run.x;
            item_start[k] = run.y;
            for (uint32_t b = 0; b < c[j]; b += per_item) {
                Item it;
                it.key = (uint32_t)k;
                it.start = run.x + b;
                it.count = min(per_item, c[j] - b);
                items[run.y++] = it;
            }
            run.x += c[j];
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < BIN_SMALL_VPT; ++q)
        if (key[q] != KEY_NONE)
            recs[cnt[key[q]] + rank[q]] = rec[q];
    if (threadIdx.x == 0) {
        vis_start[nkeys] = total.x;
        if (group_start)
            group_start[nkeys / group_keys] = total.x;
        item_start[nkeys] = total.y;
        stats[CNT_RECORDS] = total.x;
        stats[CNT_ITEMS] = total.y;
        stats[CNT_DROPPED] = s_stat[0];
        stats[CNT_BAD_PLANE] = s_stat[1];
        stats[CNT_OVERFLOW] += s_stat[2];
    }
}

// Starts, items and (cursor not NULL) the replicas' scatter cursors of the
// counted keys; totals to the call counters.  bsums holds scan_blocks(nkeys) + 1
// entries.
int scan_per_thread(int64_t nkeys);
int64_t scan_blocks(int64_t nkeys);
int launch_scan_blocks(uint2 *bsums, int64_t nb, hipStream_t s);
// Space for the scan blocks' sums of any call with up to nkeys keys (their
// number drops where a thread takes more keys): scratch that a captured graph
// holds then serves every smaller call.
size_t scan_sums_bytes(int64_t nkeys);
int scan_keys(const uint32_t *count, Replicas rp, int64_t nkeys, uint32_t per_item, uint2 *bsums,
              uint32_t *vis_start, uint32_t *item_start, uint32_t *cursor, Item *items,
              unsigned long long *stats, hipStream_t s, uint32_t *group_start = nullptr,
              int group_keys = 0);

// Host driver for count + scan + items + scatter.
struct BinResult {
    uint32_t *vis_start;  // [nkeys + 1] (last entry written by the scan)
    uint32_t *item_start; // [nkeys + 1]
    Item *items;          // [max_items]
    void *recs;           // Rec<T>[n]
    int64_t max_items;
    // optional, set by the caller: [nkeys / group_keys + 1] first record of every
    // group of group_keys (a power of two) consecutive keys
    uint32_t *group_start = nullptr;
    int group_keys = 0;
};

// Device arrays of one sort and their sizes (bin_plan).
enum BinArray {
    BIN_COUNT = 0,      // per-replica key counters
    BIN_VIS_START = 1,  // first record of every key
    BIN_ITEM_START = 2, // first work item of every key
    BIN_CURSOR = 3,     // per-replica scatter starts
    BIN_ITEMS = 4,      // work items
    BIN_RECS = 5,       // sorted records
    BIN_BSUMS = 6,      // scan block totals
    BIN_KRP = 7,        // per visibility: key, rank, position, tap index
    BIN__N = 8
};

struct BinPlan {
    Replicas rp;
    int64_t max_items;
    size_t bytes[BIN__N];
};

struct BinBufs {
    uint32_t *count, *vis_start, *item_start, *cursor;
    Item *items;
    void *recs;
    uint2 *bsums;
    uint4 *krp;
    unsigned long long *stats; // CNT__N call counters
};

// counters of one replica
inline int64_t bin_stride(int64_t nkeys) { return (nkeys + 1 + 63) / 64 * 64; }
// Validates the sort's sizes and fills the plan (no device work).
int bin_plan(int64_t n, int64_t nkeys, uint32_t per_item, int64_t max_counters, size_t rec_bytes,
             BinPlan &pl);
// The sort into caller-provided arrays of the plan's sizes; timer_ctx (may be
// NULL) receives the RG_TIMER_BINNING events.  The areas of `zero` are cleared before the
// sort; the sort's counters (unless bin_small) are among them, or clear already.
template <typename Keyer, typename T>
int bin_run(const Keyer &kf, int64_t n, int64_t nkeys, uint32_t per_item, const BinPlan &pl,
            const BinBufs &b, ZeroList &zero, rg_context *timer_ctx, hipStream_t s, BinResult &out);
// Plan and scratch (the context's slots 0-6 and 15, with room for key_room keys) of a
// sort, and what it needs cleared added to `zero`: for a caller that clears more in the same
// launch, or needs room for min_items items.
template <typename T>
int bin_prepare(rg_context *ctx, int64_t n, int64_t nkeys, int64_t key_room, uint32_t per_item,
                int64_t max_counters, ZeroList &zero, BinPlan &pl, int64_t min_items = 0);
// Keys of a W-projection of n_chan N^2 grids by the narrowest tiles, in one plane group: every
// gridding call makes room for them, so that a context whose scratch a captured graph
// of any gridder holds takes a W-projection of its grids.
inline int64_t wproj_key_room(int N, int n_chan)
{
    const int64_t nt = (N + 16 + 15) / 16;
    return nt * nt * n_chan;
}
// bin_run into the context's scratch; ready: the plan of a bin_prepare whose
// areas have been cleared (NULL: none).
template <typename Keyer, typename T>
int bin_visibilities(rg_context *ctx, const Keyer &kf, int64_t n, int64_t nkeys, int64_t key_room,
                     uint32_t per_item, ZeroList &zero, hipStream_t s, BinResult &out,
                     int64_t max_counters, const BinPlan *ready = nullptr);

} // namespace rg
