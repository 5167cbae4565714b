// tiles.hpp -- tiled Romein accumulation kernel of batched W-projection
// (device code).
//
// One wavefront takes one work item: up to K sorted records of one key.  A key
// is (plane group, group, tile): the group selects the target array (a channel grid), the tile a
// TW x 16 block of footprint top-left positions, whose footprints cover
// (S + TW - 1) x (S + 15) cells held in LDS, and the plane group a range of
// W-planes (items of a group follow one another, so the sub-kernels in use at a time
// stay in an XCD's L2).
//
// The wavefront holds the sums of a whole footprint in registers, S S / 64
// taps a lane, for as long as consecutive records have the same position,
// and adds them into LDS when the position changes (a wavefront's LDS region is
// its own: plain read-modify-write).  Records are therefore ordered by position
// first: SORT at a time, by counts in LDS.  A record costs a lane its 4 FMAs a tap,
// three lane reads (first tap as the loads' scalar offset, value) and one or
// two 16-byte tap loads whose addresses are fixed per lane.  At the end the region is
// added to the target with global atomics (neighbouring tiles and items of the
// same tile overlap), a row at a time as consecutive numbers.
//
// Bound by the tap reads: the vector cache's data return is 94 % busy (2 KB a record in FP32,
// 18 TB/s, of which 4.4 come from beyond L2), VALU issue 59 % (31 instructions a record, 16
// of them the FMAs).  With a workgroup of S S threads
// per item, a tap a lane (every lane of four wavefronts found its own cell and tap
// address for every record: about 64 instructions) and records of all planes mixed
// (a 60 MB table read past L2), tiles took, now, us: 8.4 M visibilities FP32 1571 -> 950;
// 520 k FP64 273 -> 168; 448 FP64 7.3 -> 6.6.
#pragma once

#include "binning.hpp"
#include "romein.hpp"

namespace rg {

template <typename T> __device__ inline void two_sum_into(T &hi, T &lo, T b)
{
#pragma clang fp contract(off)
    const T s = hi + b;
    const T bp = s - hi;
    const T e = (hi - (s - bp)) + (b - bp);
    hi = s;
    lo += e;
}

constexpr int TILE_POS = 16; // rows of footprint positions of a tile; columns: 16 or 32

struct TileSink {
    void *base; // target arrays, group g at base + g * gsize^2 complex elements
    int gsize;  // edge of a target array
    int ntx;    // tiles per row
    int tw;     // columns of positions of a tile
    int ntiles; // tiles per group
    int groups; // target arrays
    uint32_t key0; // tile of key 0
    // FP32 arrays: keys of at least hot_min records (0: none) add their items up in FP64
    // slots of tile_slot() numbers, which k_hot_tiles then adds to the arrays
    uint32_t hot_min;
    const uint32_t *key_start; // first record of every key
    double *hot;
    uint32_t *hot_key; // key + 1 of every slot in use
};

// Numbers of a tile and its halo.
constexpr int tile_slot(int S, int TW) { return 2 * (TILE_POS + S - 1) * (TW + S - 1); }

// Tile of a key: its array and the cell of its corner.
struct TilePlace {
    uint32_t group;
    int ox, oy;
    __device__ TilePlace(const TileSink &sink, uint32_t key, int S)
    {
        const uint32_t gt = (key + sink.key0) % (uint32_t)(sink.ntiles * sink.groups);
        group = gt / (uint32_t)sink.ntiles;
        const int tile = (int)(gt - group * (uint32_t)sink.ntiles);
        ox = tile % sink.ntx * sink.tw - S;
        oy = tile / sink.ntx * TILE_POS - S;
    }
};

__device__ inline float lane_value(float v, int lane)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ inline double lane_value(double v, int lane)
{
    const uint2 b = __builtin_bit_cast(uint2, v);
    uint2 r;
    r.x = (uint32_t)__builtin_amdgcn_readlane((int)b.x, lane);
    r.y = (uint32_t)__builtin_amdgcn_readlane((int)b.y, lane);
    return __builtin_bit_cast(double, r);
}

// Complex values per lane and load of a sub-kernel read by one wavefront.
template <typename T, int S> struct TapSpan {
    static constexpr int Z = 2 * (int)sizeof(T);
    static constexpr int BYTES = S * S * Z;
    static constexpr int LOAD = BYTES / 64 < 16 ? BYTES / 64 : 16; // bytes per lane and load
    static constexpr int NL = BYTES / (64 * LOAD);                 // loads
    static constexpr int E = LOAD / Z;                             // taps per load
};

template <typename T, int E> struct TapLoad;
template <> struct TapLoad<float, 1> {
    float2 t[1];
    __device__ void load(__amdgpu_buffer_rsrc_t r, int voff, int soff)
    {
        t[0] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
    }
};
template <> struct TapLoad<float, 2> {
    float2 t[2];
    __device__ void load(__amdgpu_buffer_rsrc_t r, int voff, int soff)
    {
        const float4 v =
            __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
        t[0] = make_float2(v.x, v.y);
        t[1] = make_float2(v.z, v.w);
    }
};
template <> struct TapLoad<double, 1> {
    double2 t[1];
    __device__ void load(__amdgpu_buffer_rsrc_t r, int voff, int soff)
    {
        t[0] = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
    }
};

constexpr int TILE_SORT = 512;    // records ordered by position at a time
constexpr int TILE_UNSORTED = 16; // up to this many are taken as they come

template <typename T, int S, int TW, bool COMP, typename GT>
__global__ __launch_bounds__(64, TW > 16 ? 2 : sizeof(T) == 4 && !COMP ? 4 : 3) void k_tiles(
    const Rec<T> *__restrict__ recs, const Item *__restrict__ items,
    const unsigned long long *__restrict__ stats, const typename Vec2<T>::type *__restrict__ kern,
    uint32_t kern_bytes, TileSink sink)
{
    using T2 = typename Vec2<T>::type;
    using Span = TapSpan<T, S>;
    constexpr int TH = TILE_POS;
    constexpr int RW = TW + S - 1, RH = TH + S - 1;
    // odd row stride: the rows a wavefront adds to start in different LDS banks
    constexpr int RS = RW | 1;
    constexpr int CELLS = RH * RS;
    constexpr int LC = COMP ? CELLS : 1;
    constexpr int BINS = TW * TH;
    constexpr int BPL = BINS / 64; // bins per lane
    static_assert(BINS % 64 == 0 && TILE_SORT % 64 == 0, "whole wavefronts");
    __shared__ T2 s_cell[CELLS]; // (re, im) of every cell of the tile and its halo
    __shared__ T2 s_lo[LC];      // COMP: the two-sum low parts
    __shared__ uint32_t s_bin[BINS];
    __shared__ uint16_t s_order[TILE_SORT];

    const int lane = threadIdx.x;
    const __amdgpu_buffer_rsrc_t ktab =
        __builtin_amdgcn_make_buffer_rsrc((void *)kern, 0, (int)kern_bytes, BUF_RSRC_W3);
    // the lane's first cell of load 0, from the footprint's corner
    const int lbase = lane * Span::E / S * RS + lane * Span::E % S;

    const uint32_t nitems = (uint32_t)stats[CNT_ITEMS];
    // the grid is no larger than the item list: the first item is read beside its length
    Item item = items[blockIdx.x];
    for (uint32_t it = blockIdx.x; it < nitems; it += gridDim.x) {
        if (it != blockIdx.x)
            item = items[it];
        double *slot = nullptr; // of a hot key
        if (sizeof(GT) == 4 && sink.hot_min) {
            const uint32_t k0 = sink.key_start[item.key];
            if (sink.key_start[item.key + 1] - k0 >= sink.hot_min) {
                // hot keys start at least hot_min records apart
                const uint32_t h = k0 / sink.hot_min;
                slot = sink.hot + (size_t)h * tile_slot(S, TW);
                if (item.start == k0 && lane == 0)
                    sink.hot_key[h] = item.key + 1;
            }
        }
#pragma unroll 2
        for (int c = lane; c < CELLS; c += 64) {
            s_cell[c].x = T(0);
            s_cell[c].y = T(0);
            if (COMP) {
                s_lo[c].x = T(0);
                s_lo[c].y = T(0);
            }
        }
        T2 sum[Span::NL][Span::E];
        int cur = -1; // corner cell of the footprint the sums belong to
        auto clear = [&]() {
#pragma unroll
            for (int l = 0; l < Span::NL; ++l)
#pragma unroll
                for (int e = 0; e < Span::E; ++e)
                    sum[l][e].x = sum[l][e].y = T(0);
        };
        auto flush = [&]() {
            const int c0 = cur + lbase;
#pragma unroll
            for (int l = 0; l < Span::NL; ++l)
#pragma unroll
                for (int e = 0; e < Span::E; ++e) {
                    const int c = c0 + l * (64 * Span::E / S) * RS + e;
                    if (COMP) {
                        two_sum_into(s_cell[c].x, s_lo[c].x, sum[l][e].x);
                        two_sum_into(s_cell[c].y, s_lo[c].y, sum[l][e].y);
                    } else {
                        s_cell[c].x += sum[l][e].x;
                        s_cell[c].y += sum[l][e].y;
                    }
                }
        };
        clear();
        for (uint32_t b = 0; b < item.count; b += TILE_SORT) {
            const int n = (int)min((uint32_t)TILE_SORT, item.count - b);
            const Rec<T> *r0 = recs + item.start + b;
            // order the n records by position
            const bool ordered = n > TILE_UNSORTED;
            if (ordered) {
                __syncthreads();
#pragma unroll
                for (int k = 0; k < BPL; ++k)
                    s_bin[lane + 64 * k] = 0;
                __syncthreads();
                auto bin = [&](int i) {
                    const uint32_t p = r0[i].pos;
                    return (p >> 16) * TW + (p & 0xffffu);
                };
#pragma unroll 2
                for (int i = lane; i < n; i += 64)
                    atomicAdd(&s_bin[bin(i)], 1u);
                __syncthreads();
                uint32_t c[BPL], tot = 0;
#pragma unroll
                for (int k = 0; k < BPL; ++k) {
                    c[k] = s_bin[lane * BPL + k];
                    tot += c[k];
                }
                uint32_t inc = tot;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const uint32_t x = (uint32_t)__shfl_up((int)inc, o);
                    if (lane >= o)
                        inc += x;
                }
                uint32_t run = inc - tot;
#pragma unroll
                for (int k = 0; k < BPL; ++k) {
                    s_bin[lane * BPL + k] = run;
                    run += c[k];
                }
                __syncthreads();
#pragma unroll 2
                for (int i = lane; i < n; i += 64)
                    s_order[atomicAdd(&s_bin[bin(i)], 1u)] = (uint16_t)i;
                __syncthreads();
            }

            auto record = [&](int k) {
                Rec<T> r;
                r.pos = 0;
                r.kidx = 0;
                r.vis.x = T(0);
                r.vis.y = T(0);
                if (k + lane < n)
                    r = r0[ordered ? (int)s_order[k + lane] : k + lane];
                return r;
            };
            // FP64 taps take twice the registers
            constexpr int U = Span::NL * Span::LOAD > 32 ? 2 : 4;
            struct Batch {
                TapLoad<T, Span::E> t[U][Span::NL];
            };
            auto fetch = [&](uint32_t kidx, int j, Batch &bt) {
#pragma unroll
                for (int q = 0; q < U; ++q) {
                    const int off = __builtin_amdgcn_readlane((int)kidx, j + q);
#pragma unroll
                    for (int l = 0; l < Span::NL; ++l)
                        bt.t[q][l].load(ktab, lane * Span::LOAD + l * 64 * Span::LOAD, off);
                }
            };
            // Taps are fetched U records ahead without a condition, so that the wait
            // for a batch leaves the next one in flight; across a chunk's end from the
            // next chunk's records (records past the last read the first sub-kernel).
            Rec<T> next = record(0);
            Batch ba, bb;
            fetch(next.kidx, 0, ba);
            for (int k = 0; k < n; k += 64) {
                const Rec<T> r = next;
                next = record(k + 64);
                const int m = min(64, n - k);
                const int cell = (int)((r.pos >> 16) * RS + (r.pos & 0xffffu));
                int prev = __shfl_up(cell, 1);
                if (lane == 0)
                    prev = cur;
                const unsigned long long change = __ballot(cell != prev);
                auto update = [&](int j, const Batch &bt) {
#pragma unroll
                    for (int q = 0; q < U; ++q) {
                        const int i = j + q;
                        if (i >= m)
                            break;
                        if ((change >> i) & 1ull) {
                            if (cur >= 0) {
                                flush();
                                clear();
                            }
                            cur = __builtin_amdgcn_readlane(cell, i);
                        }
                        const T vr = lane_value(r.vis.x, i), vi = lane_value(r.vis.y, i);
#pragma unroll
                        for (int l = 0; l < Span::NL; ++l)
#pragma unroll
                            for (int e = 0; e < Span::E; ++e) {
                                // conj(tap) * value
                                const T2 t = bt.t[q][l].t[e];
                                T2 &s = sum[l][e];
                                s.x = fma(t.x, vr, s.x);
                                s.x = fma(t.y, vi, s.x);
                                s.y = fma(t.x, vi, s.y);
                                s.y = fma(-t.y, vr, s.y);
                            }
                    }
                };
                for (int j = 0; j < m; j += 2 * U) {
                    fetch(r.kidx, j + U, bb);
                    update(j, ba);
                    fetch(j + 2 * U < 64 ? r.kidx : next.kidx, (j + 2 * U) & 63, ba);
                    update(j + U, bb);
                }
            }
        }
        flush();
        __syncthreads();

        const TilePlace at(sink, item.key, S);
        const int ox = at.ox, oy = at.oy;
        const int G = sink.gsize;
        GT *g = reinterpret_cast<GT *>(sink.base) + (size_t)at.group * G * G * 2;
        // a row's cells as 2 RW consecutive numbers: whole 64-byte pieces of the grid's row
        // in one instruction; FB rows' LDS reads in flight
        constexpr int FB = 8;
        const T *cf = reinterpret_cast<const T *>(s_cell), *lf = reinterpret_cast<const T *>(s_lo);
        for (int f = lane; f < 2 * RW; f += 64) {
            if (!slot && (unsigned)(ox + f / 2) >= (unsigned)G)
                continue;
            GT *gf = g + 2 * ((int64_t)oy * G + ox) + f;
            for (int r0 = 0; r0 < RH; r0 += FB) {
                GT v[FB];
#pragma unroll
                for (int q = 0; q < FB; ++q) {
                    const int ry = min(r0 + q, RH - 1);
                    v[q] = (GT)cf[ry * 2 * RS + f];
                    if (COMP)
                        v[q] += (GT)lf[ry * 2 * RS + f];
                }
#pragma unroll
                for (int q = 0; q < FB; ++q) {
                    if (r0 + q >= RH || v[q] == GT(0))
                        continue;
                    if (slot)
                        atomicAdd(slot + (r0 + q) * 2 * RW + f, (double)v[q]);
                    else if ((unsigned)(oy + r0 + q) < (unsigned)G)
                        atomicAdd(gf + 2 * (int64_t)(r0 + q) * G, v[q]);
                }
            }
        }
        __syncthreads();
    }
}

// Adds the hot keys' FP64 sums to their arrays: one workgroup per slot.  A dense tile has
// hundreds of items, and adding each to an FP32 array directly rounds at the size of the whole sum every
// time: 400 k visibilities on 462^2 3.7e-7 from the exact grid (items of 2048 records 1.5e-7).
template <int S, int TW>
__global__ __launch_bounds__(256) void k_hot_tiles(TileSink sink)
{
    const uint32_t key = sink.hot_key[blockIdx.x];
    if (key == 0)
        return;
    constexpr int RW = TW + S - 1;
    const TilePlace at(sink, key - 1, S);
    const int G = sink.gsize;
    float *g = reinterpret_cast<float *>(sink.base) + (size_t)at.group * G * G * 2;
    const double *slot = sink.hot + (size_t)blockIdx.x * tile_slot(S, TW);
    for (int e = threadIdx.x; e < tile_slot(S, TW); e += 256) {
        const int ry = e / (2 * RW), f = e - ry * 2 * RW;
        const float v = (float)slot[e];
        if ((unsigned)(at.oy + ry) < (unsigned)G && (unsigned)(at.ox + f / 2) < (unsigned)G && v != 0.0f)
            atomicAdd(g + 2 * ((int64_t)(at.oy + ry) * G + at.ox) + f, v);
    }
}

} // namespace rg
