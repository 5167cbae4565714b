// wproj.hip -- Romein W-projection gridders.
//
// Plain path: the reference's launch structure (scatter_grid_kernel_flat,
// grid_cuda.cu:253-280, launched <<<512, 256>>> by wproj_CUDA_flat,
// grid_cuda.cu:893): contiguous bins of the flat stream, each thread owns one
// footprint position, FP64 coordinates per thread, FP64 atomics when the
// thread's grid point changes.
//
// Batched path: visibilities are counting-sorted by the grid tile of their
// footprint and the group of its W-plane (binning.hpp), coordinates computed once per
// visibility during the sort (FP64, same formulas), then accumulated per tile in LDS by the
// Romein kernel of tiles.hpp.
#include <algorithm>
#include <mutex>

#include "binning_impl.hpp"
#include "tiles.hpp"

namespace rg {

// ---- zero fill (graph-capturable, no memset nodes) ---------------------------

__global__ __launch_bounds__(256) void k_zero(ZeroList z) { z.clear(blockIdx.x, gridDim.x); }

int ZeroList::add(void *q, size_t nbytes)
{
    if (nbytes == 0)
        return RG_OK;
    if (((uintptr_t)q & 15) != 0)
        return fail(RG_ERR_PARAM, "zero_fill: pointer not 16-byte aligned");
    if (n == MAX)
        return fail(RG_ERR_PARAM, "zero_fill: too many areas");
    p[n] = q;
    bytes[n++] = nbytes;
    return RG_OK;
}

int ZeroList::launch(hipStream_t s)
{
    if (const unsigned nb = blocks())
        hipLaunchKernelGGL(k_zero, dim3(nb), dim3(256), 0, s, *this);
    RG_HIP(hipGetLastError());
    n = 0;
    return RG_OK;
}

int zero_fill(void *p, size_t bytes, hipStream_t s)
{
    ZeroList z;
    RG_TRY(z.add(p, bytes));
    return z.launch(s);
}

// ---- plain FP64 Romein (reference launch structure) ---------------------------

__device__ inline void grid_add_f64(double2 *grid, int N, int gu, int gv, double re, double im)
{
    // scatter_grid_add bounds check (grid_cuda.cu:29-31)
    if (gu < 0 || gu >= N || gv < 0 || gv >= N)
        return;
    double *g = reinterpret_cast<double *>(grid + (size_t)gv * N + gu);
    atomicAdd(g, re);
    atomicAdd(g + 1, im);
}

__global__ __launch_bounds__(256) void k_wproj_plain(const double *__restrict__ u,
                                                     const double *__restrict__ v,
                                                     const double *__restrict__ w,
                                                     const double2 *__restrict__ vis, int64_t nvis,
                                                     int nbins, const double2 *__restrict__ kern,
                                                     int P, int R, int S, double w_min,
                                                     double w_step, double2 *__restrict__ grid,
                                                     int N, double theta,
                                                     unsigned long long *stats)
{
    // bin_flat_visibilities (radio.cuh:504-590): equal bins, remainder to the last.
    const int64_t per = nvis / nbins;
    const int64_t i0 = per * blockIdx.x;
    const int64_t i1 = (blockIdx.x == (unsigned)nbins - 1) ? nvis : i0 + per;
    const int SS = S * S;
    for (int pos = threadIdx.x; pos < SS; pos += blockDim.x) {
        const int myU = pos % S, myV = pos / S;
        int cu = INT_MIN, cv = INT_MIN;
        double sr = 0.0, si = 0.0;
        for (int64_t i = i0; i < i1; ++i) {
            int gx, gy, xf, yf;
            frac_coord(N, S, R, theta, u[i], v[i], 0.0, 0.0, gx, gy, xf, yf);
            const int p = w_plane(w[i], w_min, w_step);
            if (p < 0 || p >= P) {
                if (pos == 0)
                    atomicAdd(&stats[CNT_BAD_PLANE], 1ull);
                continue;
            }
            int conv_u = (myU - gx) % S;
            int conv_v = (myV - gy) % S;
            if (conv_u < 0)
                conv_u += S;
            if (conv_v < 0)
                conv_v += S;
            const int gu = gx + conv_u, gv = gy + conv_v;
            if (gu != cu || gv != cv) {
                if (cu != INT_MIN)
                    grid_add_f64(grid, N, cu, cv, sr, si);
                sr = 0.0;
                si = 0.0;
                cu = gu;
                cv = gv;
            }
            const double2 k =
                kern[((size_t)(p * R + yf) * R + xf) * SS + (size_t)conv_v * S + conv_u];
            const double2 vv = vis[i];
            // sum += conj(k) * vis
            sr += k.x * vv.x + k.y * vv.y;
            si += k.x * vv.y - k.y * vv.x;
        }
        if (cu != INT_MIN)
            grid_add_f64(grid, N, cu, cv, sr, si);
    }
}

int wproj_plain(rg_context *ctx, const rg_grid_params *p, const rg_flat_vis *vis,
                const rg_wkern *wk, void *grid, hipStream_t s)
{
    if (vis->vis_type != RG_C128 || wk->type != RG_C128)
        return fail(RG_ERR_PARAM, "plain mode is FP64: visibilities and kernels must be RG_C128");
    const int N = p->grid_size;
    RG_TRY(zero_fill(grid, sizeof(double2) * (size_t)N * N, s));
    const int nbins = 512; // grid_cuda.cu:881-893
    KernelTimer kt(ctx, RG_TIMER_WPROJ_PLAIN, s);
    if (vis->n > 0)
        hipLaunchKernelGGL(k_wproj_plain, dim3(nbins), dim3(256), 0, s, vis->u, vis->v, vis->w,
                           (const double2 *)vis->vis, vis->n, nbins, (const double2 *)wk->data,
                           wk->plane_count, wk->oversampling, wk->size, wk->w_min, wk->w_step,
                           (double2 *)grid, N, p->theta,
                           ctx->counters.as<unsigned long long>());
    RG_HIP(hipGetLastError());
    return RG_OK;
}

// Workgroups of the tile kernel: enough that each takes one item of all but the
// longest calls; they loop beyond that.  (17.8 M visibilities of 256 channels, 1024^2: 65536
// of them 5.09 ms, twice and eight times as many 5.04; a call with few items pays for idle
// ones from 500 k on, 8.4 M visibilities 1104 -> 1123 us.)
constexpr int64_t TILE_GRID = 131072;

// ---- batched tiled Romein -------------------------------------------------------

struct WprojKeyer {
    const double *u, *v, *w;
    const void *vis;
    int vis_type;
    int N, S, R, P;
    double theta, w_min, w_step;
    int tw, ntx, ntiles;     // columns of positions of a tile; tiles per row and grid
    const uint32_t *group_planes; // device: W-planes per plane group; NULL: one group
    int min_planes;          // of the finest groups, which the keys have room for
    int zb;                  // bytes per kernel tap
    const int64_t *chan_off;
    int nchan;

    __device__ int chan_of(int64_t i) const
    {
        int lo = 0, hi = nchan - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (chan_off[mid] <= i)
                lo = mid;
            else
                hi = mid - 1;
        }
        return lo;
    }

    // tile of visibility i (at ui, vi) over all grids, its position there; false: off the grid
    __device__ bool place(int64_t i, double ui, double vi, uint32_t &tile, uint32_t &pos, int &xf,
                          int &yf) const
    {
        int gx, gy;
        frac_coord(N, S, R, theta, ui, vi, 0.0, 0.0, gx, gy, xf, yf);
        if (gx <= -S || gx >= N || gy <= -S || gy >= N)
            return false;
        const int tx = (gx + S) / tw, ty = (gy + S) / TILE_POS;
        const int c = nchan > 1 ? chan_of(i) : 0;
        tile = (uint32_t)(c * ntiles + ty * ntx + tx);
        pos = (uint32_t)(gx + S - tx * tw) | (uint32_t)(gy + S - ty * TILE_POS) << 16;
        return true;
    }

    __device__ int classify(int64_t i, uint32_t &key, uint32_t &pos, uint32_t &kidx) const
    {
        int xf, yf;
        uint32_t tile;
        if (!place(i, u[i], v[i], tile, pos, xf, yf))
            return VIS_DROPPED;
        const int p = w_plane(w[i], w_min, w_step);
        if (p < 0 || p >= P)
            return VIS_BAD_PLANE;
        key = tile;
        if (group_planes)
            key += (uint32_t)p / max(*group_planes, (uint32_t)min_planes) *
                   (uint32_t)(nchan * ntiles);
        // byte offset of the sub-kernel
        kidx = (uint32_t)((p * R + yf) * R + xf) * (uint32_t)(S * S * zb);
        return VIS_OK;
    }

    template <typename T> __device__ typename Vec2<T>::type vis_value(int64_t i) const
    {
        typename Vec2<T>::type r;
        if (vis_type == RG_C128) {
            const double2 d = reinterpret_cast<const double2 *>(vis)[i];
            r.x = (T)d.x;
            r.y = (T)d.y;
        } else {
            const float2 f = reinterpret_cast<const float2 *>(vis)[i];
            r.x = (T)f.x;
            r.y = (T)f.y;
        }
        return r;
    }
};

// The keys [key0, key0 + count) of a grid whose keys are too many to sort at once.
struct StripKeyer : WprojKeyer {
    uint32_t key0, count;

    __device__ int classify(int64_t i, uint32_t &key, uint32_t &pos, uint32_t &kidx) const
    {
        const int r = WprojKeyer::classify(i, key, pos, kidx);
        if (r != VIS_OK)
            return r;
        key -= key0;
        return key < count ? VIS_OK : VIS_DROPPED;
    }
};

// Plane groups.  Sub-kernels are read fastest while the planes in use at a time fit an
// XCD's L2, so items are ordered by groups of W-planes; but every item adds the cells its
// records touch to the grid, so a tile whose few records fall into many groups costs more
// than it saves.  How many records share a tile depends on the stream: tracks crowd the
// centre (520 k visibilities on 4225 tiles: 123 a tile, 4020 on a record's own), even
// coverage does not.  A sample of the stream tells, while the call's memory is
// cleared: pairs of samples on one tile, D records on a record's tile.  As many groups as
// leave a key 80 of them, an even number (the planes around w = 0, which tracks
// crowd, lie at a group's end then), at most max_groups, of which each has min_planes planes.
// Calls, us, in one group / the finest groups / these: 8.4 M tracks, 2048^2, FP32 1694 / 1110 / 1123; 520 k,
// 1024^2, FP64 248 / 213 / 217; even coverage of 1024^2, 320 planes, FP32, 66 a tile 134 / 354 / 141, 260
// 407 / 530 / 374, 520 753 / 648 / 529; of 4096^2, 70 a tile 1641 / 5340 / 1660.
struct PlaneGroups {
    uint32_t *planes;      // device: the choice, planes per group
    uint32_t *done;        // device: 0 between launches
    uint32_t *bin;         // device: [samples]
    int min_planes;        // of the finest groups
    int max_groups;
    int samples;           // 0: one group
};
constexpr int SAMPLE_THREADS = 256, SAMPLE_BINS = 8192;
constexpr double GROUP_RECORDS = 80.0;

__device__ inline uint32_t sample_bin(uint32_t tile)
{
    tile = (tile ^ tile >> 16) * 0x9e3779b1u;
    tile = (tile ^ tile >> 13) * 0x85ebca77u;
    return (tile ^ tile >> 16) % SAMPLE_BINS;
}

constexpr uint32_t NO_BIN = 0xffffffffu;

// The first samples / SAMPLE_THREADS workgroups look at a sample a thread (one workgroup's
// misses alone would take 30 us for 4096) and the last of them to finish chooses the plane groups; the
// other workgroups clear the areas of z.
__global__ __launch_bounds__(SAMPLE_THREADS) void k_clear_and_sample(ZeroList z, WprojKeyer kf,
                                                                     int64_t n, PlaneGroups pg)
{
    const unsigned nsb = (unsigned)pg.samples / SAMPLE_THREADS;
    if (blockIdx.x >= nsb) {
        z.clear(blockIdx.x - nsb, gridDim.x - nsb);
        return;
    }
    __shared__ __align__(16) uint32_t bins[SAMPLE_BINS];
    __shared__ double wsum[SAMPLE_THREADS / 64];
    __shared__ uint32_t s_last;
    {
        const int k = (int)(blockIdx.x * SAMPLE_THREADS + threadIdx.x);
        const int64_t i = (int64_t)(k * ((double)n / pg.samples));
        uint32_t tile, pos;
        int xf, yf;
        const uint32_t bin =
            kf.place(i, kf.u[i], kf.v[i], tile, pos, xf, yf) ? sample_bin(tile) : NO_BIN;
        // device-scope exchange; its result is awaited before the workgroup is counted
        const uint32_t old = __hip_atomic_exchange(&pg.bin[k], bin, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" : : "v"(old) : "memory");
    }
    __syncthreads();
    if (threadIdx.x == 0)
        s_last = __hip_atomic_fetch_add(pg.done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                 nsb - 1;
    for (int k = threadIdx.x; k < SAMPLE_BINS / 4; k += SAMPLE_THREADS)
        reinterpret_cast<uint4 *>(bins)[k] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    if (!s_last)
        return;
#pragma unroll 4
    for (int k = threadIdx.x; k < pg.samples; k += SAMPLE_THREADS) {
        const uint32_t bin =
            __hip_atomic_load(&pg.bin[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (bin < SAMPLE_BINS)
            atomicAdd(&bins[bin], 1u);
    }
    __syncthreads();
    double pairs = 0.0;
    for (int k = threadIdx.x; k < SAMPLE_BINS; k += SAMPLE_THREADS)
        pairs += (double)bins[k] * ((double)bins[k] - 1.0);
    for (int o = 32; o > 0; o >>= 1)
        pairs += __shfl_xor(pairs, o);
    if (__lane_id() == 0)
        wsum[threadIdx.x / 64] = pairs;
    __syncthreads();
    if (threadIdx.x == 0) {
        pairs = 0.0;
        for (int k = 0; k < SAMPLE_THREADS / 64; ++k)
            pairs += wsum[k];
        // less the pairs that only share a bin
        const double m = pg.samples;
        const double d = (double)n * (pairs / (m * (m - 1.0)) - 1.0 / SAMPLE_BINS);
        const int g = d < 2 * GROUP_RECORDS ? 1 : (int)fmin(d / GROUP_RECORDS, 65536.0) / 2 * 2;
        *pg.planes = (uint32_t)(g >= pg.max_groups ? pg.min_planes : max((kf.P + g - 1) / g, 1));
        *pg.done = 0;
    }
}

// Tile geometry and sort parameters of batched W-projection.
struct WprojShape {
    int tw, ntx, ntiles;
    int min_planes;   // W-planes per plane group at least
    int max_groups;   // plane groups at most
    int64_t nkeys;    // max_groups x grids x tiles
    uint32_t key0 = 0; // tile of the sort's key 0 (strips)
    uint32_t per_item;
    // FP32 grids: records of a key whose items add up in FP64 first (0: no key),
    // slots for such keys of this stream, and for any shorter one too
    uint32_t hot_min;
    int64_t hot_slots, hot_room;
    // records per work item of a call without such slots, whose items are added up in FP32:
    // with 512 a dense tile's sum would be rounded four times as often
    static constexpr uint32_t COLD_ITEM = 2048;

    size_t hot_bytes(int S, int64_t slots) const
    {
        return slots * sizeof(double) * (size_t)tile_slot(S, tw);
    }
    void wide(int N, int S)
    {
        tw = 2 * TILE_POS;
        ntx = (N + S + tw - 1) / tw;
        ntiles = ntx * ((N + S + TILE_POS - 1) / TILE_POS);
    }
    // no room for the slots
    void cold()
    {
        hot_min = 0;
        hot_slots = hot_room = 0;
        per_item = std::max(per_item, COLD_ITEM);
    }
    void one_group(int planes, int n_chan)
    {
        min_planes = std::max(planes, 1);
        max_groups = 1;
        nkeys = (int64_t)ntiles * n_chan;
    }
    // The choice of plane groups, with words: the word of the planes per group and, 64 bytes
    // on, the one of finished workgroups; room: space for 16 bytes a record, in use later.  1024 samples up
    // to 256 k records, 4096 from 1 M (D is then known to 4e-6 n).
    PlaneGroups groups(char *words, void *room, int64_t nvis) const
    {
        PlaneGroups pg{};
        if (max_groups > 1 && nvis >= SAMPLE_THREADS) {
            pg.planes = reinterpret_cast<uint32_t *>(words);
            pg.done = reinterpret_cast<uint32_t *>(words + 64);
            pg.bin = static_cast<uint32_t *>(room);
            pg.min_planes = min_planes;
            pg.max_groups = max_groups;
            pg.samples = (int)std::min<int64_t>(nvis, std::clamp<int64_t>(nvis / 256, 1024, 4096)) /
                         SAMPLE_THREADS * SAMPLE_THREADS;
        }
        return pg;
    }
};

// The call's clears (emptying the list) and the choice of plane groups.
static int clear_and_sample(ZeroList &zero, const WprojKeyer &kf, int64_t n, const PlaneGroups &pg,
                            hipStream_t s)
{
    const unsigned nb = zero.blocks();
    hipLaunchKernelGGL(k_clear_and_sample, dim3((unsigned)pg.samples / SAMPLE_THREADS + nb), dim3(SAMPLE_THREADS), 0, s, zero, kf, n, pg);
    RG_HIP(hipGetLastError());
    zero.n = 0;
    return RG_OK;
}

struct HotSlots {
    double *sums;
    uint32_t *key;
};

template <typename T, int S, int TW, bool COMP, typename GT>
static int launch_tiles(const BinResult &br, rg_context *timer_ctx,
                        const unsigned long long *stats, const rg_wkern *wk, void *grid, int N,
                        int n_chan, const WprojShape &sh, const HotSlots &hot, hipStream_t s)
{
    TileSink sink;
    sink.hot_min = sizeof(GT) == 4 ? sh.hot_min : 0;
    sink.key0 = sh.key0;
    sink.key_start = br.vis_start;
    sink.hot = hot.sums;
    sink.hot_key = hot.key;
    sink.base = grid;
    sink.gsize = N;
    sink.ntx = sh.ntx;
    sink.tw = TW;
    sink.ntiles = sh.ntiles;
    sink.groups = n_chan;
    KernelTimer kt(timer_ctx, RG_TIMER_WPROJ_TILES, s);
    const uint64_t kbytes = (uint64_t)wk->plane_count * wk->oversampling * wk->oversampling * S *
                            S * sizeof(typename Vec2<T>::type);
    if (kbytes > 0x7fffffffull)
        return fail(RG_ERR_UNSUPPORTED, "batched W-projection kernel tables above 2 GiB");
    if (br.max_items > 0) {
        const int64_t nb = std::min<int64_t>(br.max_items, TILE_GRID);
        hipLaunchKernelGGL((k_tiles<T, S, TW, COMP, GT>), dim3((unsigned)nb), dim3(64), 0, s,
                           (const Rec<T> *)br.recs, (const Item *)br.items, stats,
                           (const typename Vec2<T>::type *)wk->data, (uint32_t)kbytes, sink);
        if (sink.hot_min)
            hipLaunchKernelGGL((k_hot_tiles<S, TW>), dim3((unsigned)sh.hot_slots), dim3(256), 0, s,
                               sink);
    }
    RG_HIP(hipGetLastError());
    return RG_OK;
}

template <typename T, int S, int TW>
static int dispatch_comp_grid(const BinResult &br, rg_context *timer_ctx,
                              const unsigned long long *stats, const rg_wkern *wk, void *grid,
                              int grid_type, bool comp, int N, int n_chan, const WprojShape &sh,
                              const HotSlots &hot, hipStream_t s)
{
    auto run = [&](auto c, auto g) {
        return launch_tiles<T, S, TW, decltype(c)::value, decltype(g)>(
            br, timer_ctx, stats, wk, grid, N, n_chan, sh, hot, s);
    };
    if constexpr (std::is_same<T, double>::value) {
        if (grid_type != RG_C128)
            return fail(RG_ERR_PARAM, "FP64 kernels need an RG_C128 grid");
        return run(std::false_type{}, double{});
    } else {
        if (grid_type == RG_C128)
            return comp ? run(std::true_type{}, double{}) : run(std::false_type{}, double{});
        return comp ? run(std::true_type{}, float{}) : run(std::false_type{}, float{});
    }
}

template <typename T>
static int dispatch_tiles(const BinResult &br, rg_context *timer_ctx,
                          const unsigned long long *stats, const rg_wkern *wk, void *grid,
                          int grid_type, bool comp, int N, int n_chan, const WprojShape &sh,
                          const HotSlots &hot, hipStream_t s)
{
    auto run = [&](auto sz) {
        if (sh.tw == 32)
            return dispatch_comp_grid<T, decltype(sz)::value, 32>(
                br, timer_ctx, stats, wk, grid, grid_type, comp, N, n_chan, sh, hot, s);
        return dispatch_comp_grid<T, decltype(sz)::value, 16>(br, timer_ctx, stats, wk, grid, grid_type,
                                                          comp, N, n_chan, sh, hot, s);
    };
    using std::integral_constant;
    return wk->size == 16 ? run(integral_constant<int, 16>{}) : run(integral_constant<int, 8>{});
}

// Records per work item when the caller leaves it open.  A wavefront walks its
// item's records one after another, and every item adds its tile to the grid, so both the
// records of an item and the items grow with the stream: the largest power of two from 8 to
// 512 with 12 K^2 <= records.  Tile kernel or call, us, at half / this / twice the size:
// 448 records FP64 5.2 / 6.7 / 8.1 (the call is shortest at 8); 16 k FP64 on 2000^2 60 / 54 / 57; 150 k FP32 69 / 65
// / -; 520 k FP64 225 / 204 / 237; 8.4 M FP32 1032 / 1042 / 1161.
static uint32_t default_item(int64_t nvis)
{
    uint32_t k = 8;
    while (k < TILE_SORT && 12 * (int64_t)(2 * k) * (2 * k) <= nvis)
        k *= 2;
    return k;
}

static int wproj_shape(const rg_grid_params *p, int64_t nvis, int n_chan, const rg_wkern *wk,
                       WprojShape &sh)
{
    const int S = wk->size;
    // both values of the parameter run the same tiles
    const int tile = p->tile > 0 ? p->tile : 32;
    if (tile != 32 && tile != 48)
        return fail(RG_ERR_UNSUPPORTED, "batched tile must be 32 or 48 (got %d)", tile);
    if (S != 8 && S != 16)
        return fail(RG_ERR_UNSUPPORTED, "batched W-projection supports kernel sizes 8 and 16 (got %d)", S);
    sh.tw = TILE_POS;
    const int nty = (p->grid_size + S + TILE_POS - 1) / TILE_POS;
    sh.ntx = nty;
    sh.ntiles = nty * nty;
    // The finest plane groups hold 2^18 taps (2 MB in FP32, 4 MB in FP64), of up to 64 groups.
    // Streams of fewer than 64 records a tile take at most four groups and, on grids beyond 64 MB, whose
    // cells are no longer added to in L2, tiles twice as wide (S = 8: only these streams; 16 channels of 1024^2, even
    // coverage, 9 / 30 / 150 records a tile, S = 16: 428 / 775 / 3354 us, wide 375 / 751 / 3148).
    const int64_t plane_taps = (int64_t)wk->oversampling * wk->oversampling * S * S;
    const int64_t planes = std::max<int64_t>(wk->plane_count, 1);
    int64_t group = std::max<int64_t>({1, ((int64_t)1 << 18) / std::max<int64_t>(plane_taps, 1),
                                       (planes + 63) / 64});
    int64_t one = (int64_t)sh.ntiles * n_chan;
    const bool dense = nvis >= 64 * one, sparse = nvis < 8 * one;
    const bool large = (int64_t)p->grid_size * p->grid_size * n_chan *
                           (wk->type == RG_C128 ? 16 : 8) > (int64_t)64 << 20;
    if (large && !sparse && (S == 16 || !dense)) {
        sh.wide(p->grid_size, S);
        one = (int64_t)sh.ntiles * n_chan;
    }
    sh.one_group(wk->plane_count, n_chan);
    if (!dense)
        group = std::max(group, (planes + 3) / 4);
    const int64_t all = (planes + group - 1) / group;
    // Sub-kernels of 512 bytes (S = 8, FP32) are read fast enough from a table of up to 48 MB
    // anyhow (15 MB, 8.4 M tracks, 2048^2: one group 529 us, grouped 540; 20 MB, 32 channels of
    // 1024^2, 154 a tile 1477 / 1669; 61 MB, 2048^2: 678 / 618).
    const int64_t sub_bytes = (int64_t)S * S * (wk->type == RG_C128 ? 16 : 8);
    const bool ungrouped =
        sub_bytes <= 512 && planes * wk->oversampling * wk->oversampling * sub_bytes <= (48 << 20);
    if (!sparse && !ungrouped && all > 1 && (dense || 2 * one * all <= BIN_MAX_COUNTERS)) {
        sh.min_planes = (int)group;
        sh.max_groups = (int)all;
        sh.nkeys = one * all;
    }
    // a key of eight default items or more (the shortest streams have too few items for
    // it to matter)
    const int64_t k = default_item(nvis);
    sh.hot_min = nvis >= 1024 ? (uint32_t)(8 * k) : 0;
    sh.hot_slots = sh.hot_min ? nvis / sh.hot_min + 1 : 0;
    // of the shorter streams the longest with items of k / 2, 12 k^2 - 1 records, takes most
    sh.hot_room = std::max<int64_t>(sh.hot_slots, sh.hot_min && k > 8 ? 3 * k : 0);
    // (items beyond what a wavefront sorts, 1024 to 4096 in parameters that were tuned for
    // workgroups, leave the choice open too: a call of 150 k FP32 records takes 97 us, with 512
    // of them an item 109; of 1 M 226, 259)
    sh.per_item = p->vis_per_item > 0 && p->vis_per_item <= TILE_SORT ? (uint32_t)p->vis_per_item
                                                                      : default_item(nvis);
    return RG_OK;
}

static WprojKeyer wproj_keyer(const rg_grid_params *p, const rg_flat_vis *vis, const rg_wkern *wk,
                              const WprojShape &sh, const int64_t *d_off, int n_chan, int zb,
                              const PlaneGroups &pg)
{
    WprojKeyer kf;
    kf.u = vis->u;
    kf.v = vis->v;
    kf.w = vis->w;
    kf.vis = vis->vis;
    kf.vis_type = vis->vis_type;
    kf.N = p->grid_size;
    kf.S = wk->size;
    kf.R = wk->oversampling;
    kf.P = wk->plane_count;
    kf.theta = p->theta;
    kf.w_min = wk->w_min;
    kf.w_step = wk->w_step;
    kf.tw = sh.tw;
    kf.ntx = sh.ntx;
    kf.ntiles = sh.ntiles;
    kf.group_planes = pg.samples ? pg.planes : nullptr;
    kf.min_planes = pg.min_planes;
    kf.zb = zb;
    kf.chan_off = d_off;
    kf.nchan = n_chan;
    return kf;
}

template <typename T>
static int wproj_batched_t(rg_context *ctx, const rg_grid_params *p, const rg_flat_vis *vis,
                           const int64_t *d_off, int n_chan, const rg_wkern *wk, void *grid,
                           int grid_type, hipStream_t s)
{
    const int N = p->grid_size;
    WprojShape sh;
    RG_TRY(wproj_shape(p, vis->n, n_chan, wk, sh));

    // the call's counters, the grids and the sort's counters in one launch
    const size_t gbytes = (size_t)(grid_type == RG_C128 ? 16 : 8) * N * N * n_chan;
    ZeroList zero;
    RG_TRY(zero.add(ctx->counters.p, sizeof(unsigned long long) * CNT__N));
    RG_TRY(zero.add(grid, gbytes));
    // a context's first call: the grids are cleared while the host allocates
    if (!ctx->scratch[5].p)
        RG_TRY(zero.launch(s));
    HotSlots hot{};
    if (grid_type == RG_C64 && sh.hot_min) {
        const size_t kb = (sizeof(uint32_t) * (size_t)sh.hot_room + 255) / 256 * 256;
        DevBuf &buf = ctx->scratch[20];
        // (scratch that a captured graph holds, of another kind of call perhaps, may not do)
        if (buf.ensure(kb + sh.hot_bytes(wk->size, sh.hot_room)) == RG_OK) {
            hot.key = buf.as<uint32_t>();
            hot.sums = reinterpret_cast<double *>(buf.as<char>() + kb);
            RG_TRY(zero.add(hot.key, kb));
            RG_TRY(zero.add(hot.sums, sh.hot_bytes(wk->size, sh.hot_slots)));
        } else {
            sh.cold();
        }
    }
    const int64_t room = wproj_key_room(N, n_chan);
    BinPlan pl;
    int rc = bin_prepare<T>(ctx, vis->n, sh.nkeys, room, sh.per_item, BIN_MAX_COUNTERS, zero, pl);
    if (rc != RG_OK && sh.nkeys != (int64_t)sh.ntiles * n_chan) {
        // no room for the plane groups (a captured graph holds the scratch): without them
        sh.one_group(wk->plane_count, n_chan);
        rc = bin_prepare<T>(ctx, vis->n, sh.nkeys, room, sh.per_item, BIN_MAX_COUNTERS, zero, pl);
    }
    if (rc != RG_OK)
        return rc;

    if (sh.max_groups > 1) {
        uint32_t *done; // the word after COUNTER_PLANES'
        RG_TRY(range_done_counter(ctx, &done, s));
    }
    const PlaneGroups pg = sh.groups(ctx->counters.as<char>() + COUNTER_PLANES,
                                     bin_buffer(ctx, BIN_KRP), vis->n);
    const WprojKeyer kf = wproj_keyer(p, vis, wk, sh, d_off, n_chan,
                                      (int)sizeof(typename Vec2<T>::type), pg);
    if (pg.samples)
        RG_TRY(clear_and_sample(zero, kf, vis->n, pg, s));
    BinResult br;
    RG_TRY((bin_visibilities<WprojKeyer, T>(ctx, kf, vis->n, sh.nkeys, room, sh.per_item,
                                            zero, s, br, BIN_MAX_COUNTERS, &pl)));
    return dispatch_tiles<T>(br, ctx, ctx->counters.as<unsigned long long>(), wk, grid, grid_type,
                             p->compensated != 0, N, n_chan, sh, hot, s);
}

int wproj_batched(rg_context *ctx, const rg_grid_params *p, const rg_flat_vis *vis,
                  const int64_t *d_off, int n_chan, const rg_wkern *wk, void *grid,
                  int grid_type, hipStream_t s)
{
    if (wk->type == RG_C64)
        return wproj_batched_t<float>(ctx, p, vis, d_off, n_chan, wk, grid, grid_type, s);
    return wproj_batched_t<double>(ctx, p, vis, d_off, n_chan, wk, grid, grid_type, s);
}

// ---- allocation-free batched W-projection ------------------------------------------------
// One file-scope device array serves every call on a device: the sort's
// counters, key starts, work items, records and per-visibility keys, and the
// call counters.  Host code never passes the array's name to a kernel: its
// device address on the current device comes from hipGetSymbolAddress, looked
// up once per device and kept.  Calls on one device share the array, so calls
// that overlap in time on one device (several streams or host threads) race.
// (A device array is set up with the library's first kernel, which takes 27 ms with
// 64 MiB and 78 ms with 192 MiB.)
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[NOALLOC_MAX_DEVICES];

static int noalloc_scratch(void **out)
{
    int dev = 0;
    RG_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES)
        return fail(RG_ERR_UNSUPPORTED, "device %d beyond the %d devices of the static scratch",
                    dev, NOALLOC_MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        RG_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (!ptr)
            return fail(RG_ERR_HIP, "no device address for the static scratch on device %d", dev);
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return RG_OK;
}

size_t noalloc_scratch_bytes() { return NOALLOC_SCRATCH_BYTES; }

template <typename T>
static int wproj_noalloc_t(const rg_grid_params *p, const rg_flat_vis *vis, const rg_wkern *wk,
                           void *grid, int grid_type, int accumulate, hipStream_t s)
{
    const int N = p->grid_size;
    WprojShape sh;
    RG_TRY(wproj_shape(p, vis->n, 1, wk, sh));
    auto aligned = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t head = aligned(COUNTER_BYTES); // call counters first
    // The limit on the stream is that of a sort by tiles of the parameter's 32 or 48
    // cells with separate cursors, items of 2048 records and scan blocks of 1024 keys:
    // about 2.0 M visibilities with FP32 kernels, 1.4 M with FP64 at 2048^2.
    BinPlan pl;
    const uint32_t limit_item = p->vis_per_item > 0 ? (uint32_t)p->vis_per_item : 2048u;
    const int64_t lt = p->tile > 0 ? p->tile : 32, ln = (N + wk->size + lt - 1) / lt, lk = ln * ln;
    RG_TRY(bin_plan(vis->n, lk, limit_item, BIN_MAX_COUNTERS, sizeof(Rec<T>), pl));
    size_t want = head;
    for (int k = 0; k < BIN__N; ++k)
        want += aligned(k == BIN_BSUMS ? sizeof(uint2) * (size_t)((lk + 1023) / 1024 + 1)
                                       : pl.bytes[k]);
    if (want > NOALLOC_SCRATCH_BYTES)
        return fail(RG_ERR_PARAM,
                    "rg_grid_noalloc: %lld visibilities on a %d^2 grid need %zu bytes of scratch; "
                    "the static scratch holds %zu: split the stream over calls with accumulate = 1",
                    (long long)vis->n, N, want, NOALLOC_SCRATCH_BYTES);
    if (grid_type != RG_C64) {
        sh.hot_min = 0;
        sh.hot_slots = 0;
    }
    // Carve the arrays from the static scratch, 256-byte aligned.  The scatter
    // cursors take the place of the counters they are made from.
    size_t off[BIN__N], hot_at = 0, hot_keys = 0;
    auto carve = [&](int64_t max_counters) {
        RG_TRY(bin_plan(vis->n, sh.nkeys, sh.per_item, max_counters, sizeof(Rec<T>), pl));
        size_t at = head;
        for (int k = 0; k < BIN__N; ++k) {
            if (k == BIN_CURSOR) {
                off[k] = off[BIN_COUNT];
            } else {
                off[k] = at;
                at += aligned(pl.bytes[k]);
            }
        }
        hot_at = at;
        hot_keys = aligned(sizeof(uint32_t) * (size_t)sh.hot_slots);
        at += hot_keys + aligned(sh.hot_bytes(wk->size, sh.hot_slots));
        return at <= NOALLOC_SCRATCH_BYTES ? RG_OK : RG_ERR_NOMEM;
    };
    // as many counters a key as there is room for
    auto carve_any = [&](int64_t least) {
        int rc = RG_ERR_NOMEM;
        for (int64_t c = 16; c >= least && rc == RG_ERR_NOMEM; c /= 2)
            rc = carve(std::min(BIN_MAX_COUNTERS, c * bin_stride(sh.nkeys)));
        return rc;
    };
    // The longest streams' records take almost all of the array.  Such a call does without the
    // plane groups; a stream whose FP64 sums of items find no room then (the last tenth below
    // the limit) is gridded in two halves (2.1 M, FP32, tracks on 1024^2: 501 us, without the sums
    // and with the items of 2048 records that keep the error 622); without such sums
    // wider tiles have half the keys; and a very large grid is sorted by one strip of
    // tile rows after another.
    int rc = carve_any(2);
    if (rc == RG_ERR_NOMEM && sh.max_groups > 1) {
        sh.one_group(wk->plane_count, 1);
        rc = carve_any(2);
    }
    if (rc == RG_ERR_NOMEM && sh.hot_min && vis->n >= (1 << 16) &&
        pl.bytes[BIN_VIS_START] <= NOALLOC_SCRATCH_BYTES / 16) {
        rg_flat_vis half = *vis;
        half.n = vis->n / 128 * 64;
        RG_TRY(wproj_noalloc_t<T>(p, &half, wk, grid, grid_type, accumulate, s));
        const size_t vsz = vis->vis_type == RG_C128 ? 16 : 8;
        half.u += half.n;
        half.v += half.n;
        half.w += half.n;
        half.vis = (const char *)half.vis + vsz * (size_t)half.n;
        half.n = vis->n - half.n;
        return wproj_noalloc_t<T>(p, &half, wk, grid, grid_type, 1, s);
    }
    if (rc == RG_ERR_NOMEM) {
        sh.wide(N, wk->size);
        sh.one_group(wk->plane_count, 1);
        rc = carve_any(1);
    }
    if (rc == RG_ERR_NOMEM) {
        if (grid_type == RG_C64)
            sh.cold();
        sh.per_item = std::max(sh.per_item, limit_item);
        rc = carve_any(1);
    }
    const int64_t tiles = sh.nkeys;
    for (int64_t rows = tiles / sh.ntx; rc == RG_ERR_NOMEM && rows > 1;) {
        rows = (rows + 1) / 2;
        sh.nkeys = rows * sh.ntx;
        rc = carve(1);
    }
    if (rc == RG_ERR_NOMEM)
        return fail(RG_ERR_PARAM, "rg_grid_noalloc: no room for a row of tiles");
    RG_TRY(rc);
    void *base = nullptr;
    RG_TRY(noalloc_scratch(&base));
    char *b0 = static_cast<char *>(base);
    BinBufs b;
    b.stats = reinterpret_cast<unsigned long long *>(b0);
    b.count = reinterpret_cast<uint32_t *>(b0 + off[BIN_COUNT]);
    b.vis_start = reinterpret_cast<uint32_t *>(b0 + off[BIN_VIS_START]);
    b.item_start = reinterpret_cast<uint32_t *>(b0 + off[BIN_ITEM_START]);
    b.cursor = reinterpret_cast<uint32_t *>(b0 + off[BIN_CURSOR]);
    b.items = reinterpret_cast<Item *>(b0 + off[BIN_ITEMS]);
    b.recs = b0 + off[BIN_RECS];
    b.bsums = reinterpret_cast<uint2 *>(b0 + off[BIN_BSUMS]);
    b.krp = reinterpret_cast<uint4 *>(b0 + off[BIN_KRP]);
    // the previous call's counters are still there: start from zero
    ZeroList zero;
    RG_TRY(zero.add(b.stats, sizeof(unsigned long long) * CNT__N));
    HotSlots hot{};
    if (sh.hot_min) {
        hot.key = reinterpret_cast<uint32_t *>(b0 + hot_at);
        hot.sums = reinterpret_cast<double *>(b0 + hot_at + hot_keys);
        RG_TRY(zero.add(hot.key, hot_keys + sh.hot_bytes(wk->size, sh.hot_slots)));
    }
    if (!accumulate)
        RG_TRY(zero.add(grid, (size_t)(grid_type == RG_C128 ? 16 : 8) * N * N));
    if (vis->n == 0)
        return zero.launch(s);
    const PlaneGroups pg = sh.groups(b0 + COUNTER_PLANES, b.krp, vis->n);
    const WprojKeyer kf =
        wproj_keyer(p, vis, wk, sh, nullptr, 1, (int)sizeof(typename Vec2<T>::type), pg);
    auto tiles_of = [&](const BinResult &br) {
        return dispatch_tiles<T>(br, nullptr, b.stats, wk, grid, grid_type, p->compensated != 0, N, 1,
                                 sh, hot, s);
    };
    if (sh.nkeys < tiles) {
        for (int64_t k = 0; k < tiles; k += sh.nkeys) {
            sh.key0 = (uint32_t)k;
            StripKeyer sk;
            static_cast<WprojKeyer &>(sk) = kf;
            sk.key0 = sh.key0;
            sk.count = (uint32_t)sh.nkeys;
            if (k > 0)
                RG_TRY(zero.add(b.stats, sizeof(unsigned long long) * CNT__N));
            RG_TRY(zero.add(b.count, pl.bytes[BIN_COUNT]));
            BinResult br;
            RG_TRY((bin_run<StripKeyer, T>(sk, vis->n, sh.nkeys, sh.per_item, pl, b, zero, nullptr,
                                           s, br)));
            RG_TRY(tiles_of(br));
        }
        return RG_OK;
    }
    if (!bin_small(vis->n, sh.nkeys))
        RG_TRY(zero.add(b.count, pl.bytes[BIN_COUNT]));
    if (pg.samples)
        RG_TRY(clear_and_sample(zero, kf, vis->n, pg, s));
    BinResult br;
    RG_TRY((bin_run<WprojKeyer, T>(kf, vis->n, sh.nkeys, sh.per_item, pl, b, zero, nullptr,
                                   s, br)));
    return tiles_of(br);
}

int wproj_noalloc(const rg_grid_params *p, const rg_flat_vis *vis, const rg_wkern *wk, void *grid,
                  int grid_type, int accumulate, hipStream_t s)
{
    if (wk->type == RG_C64)
        return wproj_noalloc_t<float>(p, vis, wk, grid, grid_type, accumulate, s);
    return wproj_noalloc_t<double>(p, vis, wk, grid, grid_type, accumulate, s);
}

} // namespace rg

