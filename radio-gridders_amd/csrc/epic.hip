// epic.hip -- EPIC E-field gridding (epic_romein / scatter_grid_kernel,
// src/epic/epic_grid.cu:54-218), batches of antenna E-fields each gridded
// with a small illumination pattern onto its own g x g grid.
//
// A workgroup owns a band of rows of one batch's grid in LDS: it lists the antennas whose
// footprints meet the band, adds their taps there and writes the rows to HBM once, coalesced: no
// global atomics, one pass of output traffic, nothing cleared in HBM.  Grids of any size are
// cut into bands; few grids of very many antennas are cleared and added to with global
// atomics instead.
#include <algorithm>

#include "rg_internal.hpp"

namespace rg {

constexpr int EPIC_THREADS = 256;
constexpr int EPIC_LDS = 32 * 1024;

// c += val: compare-and-swap of the 64-bit pair, tried again by the lanes that lost the cell to
// another; those that lose twice, where many taps fall on a cell at a time, use float
// atomics.  ds_add_f32 takes four to five cycles a lane, whatever the cells: 1000 grids of 256 antennas, 2 x 2
// taps, 18.0 us with it alone, 8.6 us (the launch's own time) with these.  Compare-and-swap alone
// takes a round per lane that meets on a cell: all antennas on one, 528 us (call), 24 so.
__device__ inline void lds_add(float2 *c, float2 val)
{
    auto *p = reinterpret_cast<unsigned long long *>(c);
    unsigned long long seen = *p;
#pragma unroll
    for (int round = 0; round < 2; ++round) {
        float2 v = __builtin_bit_cast(float2, seen);
        v.x += val.x;
        v.y += val.y;
        const unsigned long long got = atomicCAS(p, seen, __builtin_bit_cast(unsigned long long, v));
        if (got == seen)
            return;
        seen = got;
    }
    atomicAdd(&c->x, val.x);
    atomicAdd(&c->y, val.y);
}

// SUPP: the support, or 0 to take it at run time (magic: 2^32 / supp^2, rounded up).  One thread
// per antenna and tap, the taps of an antenna next to each other: a wavefront's lanes fall on one
// cell only where antennas stand on each other or overlap.  Workgroups of a band of all grids
// follow one another: where the array's dense core lies in one band, its workgroups are spread over
// all CUs (band after band of each grid instead: 200 grids of 512 antennas within 4 x 4 cells, 4 x 4 taps,
// 27 -> 154 us a call).
template <int SUPP>
__global__ __launch_bounds__(EPIC_THREADS) void k_epic_band(
    const float2 *__restrict__ f, const int32_t *__restrict__ x, const int32_t *__restrict__ y,
    int n_ant, const float2 *__restrict__ illum, int supp_rt, uint32_t magic, int g, int rows,
    int nbatch, float2 *__restrict__ grids)
{
    extern __shared__ __align__(16) float2 sg[];
    struct Ant {
        int x, y;
        float2 v;
    };
    __shared__ Ant s_ant[EPIC_THREADS];
    __shared__ int s_cnt[2];
    const int supp = SUPP ? SUPP : supp_rt, taps = supp * supp;
    const unsigned band = blockIdx.x / (unsigned)nbatch, b = blockIdx.x - band * (unsigned)nbatch;
    const int r0 = (int)band * rows, r1 = min(g, r0 + rows);
    const int cells = (r1 - r0) * g;
    const size_t a0 = (size_t)b * n_ant;
    const int tid = threadIdx.x;
    // the next antenna's loads are in flight while the band is cleared, or added to
    Ant next;
    auto load = [&](int a) {
        if (a < n_ant) {
            next.x = x[a0 + a];
            next.y = y[a0 + a];
            next.v = f[a0 + a];
        }
    };
    load(tid);
    for (int e = tid; e < (cells + 1) / 2; e += EPIC_THREADS)
        reinterpret_cast<float4 *>(sg)[e] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (tid < 2)
        s_cnt[tid] = 0;
    for (int base = 0, half = 0; base < n_ant; base += EPIC_THREADS, half ^= 1) {
        __syncthreads(); // the list before has been read, its successor's length is 0
        // antennas whose footprints meet the band
        const bool in = base + tid < n_ant && (int64_t)next.y + supp > r0 && next.y < r1 &&
                        (int64_t)next.x + supp > 0 && next.x < g;
        const unsigned long long m = __ballot(in);
        int at = 0;
        if (m && __lane_id() == __ffsll((long long)m) - 1)
            at = atomicAdd(&s_cnt[half], __popcll(m));
        at = __shfl(at, m ? __ffsll((long long)m) - 1 : 0);
        if (in)
            s_ant[at + __popcll(m & ((1ull << __lane_id()) - 1ull))] = next;
        load(base + EPIC_THREADS + tid);
        __syncthreads();
        if (tid == 0)
            s_cnt[half ^ 1] = 0;
        const int work = s_cnt[half] * taps;
        for (int e = tid; e < work; e += EPIC_THREADS) {
            // e < 256 supp^2 <= 2^20, where the product with magic is exact
            const int a = SUPP ? e / (SUPP * SUPP) : (int)__umulhi((uint32_t)e, magic);
            const int t = e - a * taps, ty = t / supp, tx = t - ty * supp;
            const Ant q = s_ant[a];
            const float2 k = illum[t];
            const int X = q.x + tx, Y = q.y + ty;
            // scatter_grid_add's bounds check; conj(k) v (epic_grid.cu:121-123)
            if (X >= 0 && X < g && Y >= r0 && Y < r1)
                lds_add(sg + (Y - r0) * g + X,
                        make_float2(k.x * q.v.x + k.y * q.v.y, k.x * q.v.y - k.y * q.v.x));
        }
    }
    __syncthreads();
    float2 *out = grids + (size_t)b * g * g + (size_t)r0 * g;
    if ((reinterpret_cast<uintptr_t>(out) & 15) == 0 && cells % 2 == 0) {
        for (int e = tid; e < cells / 2; e += EPIC_THREADS)
            reinterpret_cast<float4 *>(out)[e] = reinterpret_cast<const float4 *>(sg)[e];
    } else {
        for (int e = tid; e < cells; e += EPIC_THREADS)
            out[e] = sg[e];
    }
}

__global__ __launch_bounds__(256) void k_epic_atomic(const float2 *__restrict__ f,
                                                     const int32_t *__restrict__ x,
                                                     const int32_t *__restrict__ y, int n_ant,
                                                     const float2 *__restrict__ illum, int supp,
                                                     int g, float2 *grids)
{
    const int b = blockIdx.x;
    const int gg = g * g;
    float2 *out = grids + (size_t)b * gg;
    const int taps = supp * supp;
    const int work = n_ant * taps;
    for (int e = blockIdx.y * blockDim.x + threadIdx.x; e < work; e += gridDim.y * blockDim.x) {
        const int a = e / taps, t = e - a * taps;
        const size_t i = (size_t)b * n_ant + a;
        const int X = x[i] + t % supp, Y = y[i] + t / supp;
        if (X < 0 || X >= g || Y < 0 || Y >= g)
            continue;
        const float2 k = illum[t], v = f[i];
        float *c = reinterpret_cast<float *>(out) + 2 * (Y * g + X);
        atomicAdd(c, k.x * v.x + k.y * v.y);
        atomicAdd(c + 1, k.x * v.y - k.y * v.x);
    }
}

int epic_grid(const void *f, const int32_t *x, const int32_t *y, int n_ant, int nbatch,
              const void *illum, int supp, int g, void *grids, hipStream_t s)
{
    // grids beyond 64 KiB need 16-byte alignment (they may be cleared in place)
    if ((size_t)g * g * sizeof(float2) > 64 * 1024 && ((uintptr_t)grids & 15) != 0)
        return fail(RG_ERR_PARAM, "EPIC grids above 64 KiB must be 16-byte aligned");
    // Bands of up to 32 KiB (four workgroups per CU), and shorter ones while there
    // are fewer than 1024 of them.
    int rows = std::max(1, std::min(g, EPIC_LDS / (8 * g)));
    auto bands = [&](int r) { return (int64_t)((g + r - 1) / r); };
    while (rows > 8 && nbatch * bands(rows) < 1024)
        rows = (rows + 1) / 2;
    const int64_t nbands = bands(rows);
    // A band's workgroup takes 2.2 ns for each antenna it looks at and 0.9 ns a tap, and 768 of them
    // run at a time; global atomics take 0.05 ns a tap in all, beside clearing the grids and
    // a second launch.  So bands, unless few grids of many antennas leave the chip idle: us,
    // bands and atomics, 1 grid of 20 000 antennas, 64^2, 2 x 2 taps 114 / 21 (with one band); 2 of 100 000,
    // 512^2 236 / 52; 200 of 20 000, 64^2 126 / 840; 1000 of 1000, 16^2 18 / 171.
    const double taps = (double)supp * supp, ant = n_ant;
    const double t_bands = std::max(1.0, (double)nbatch * nbands / 768) * ant * (2.2 + 0.9 * taps / nbands);
    const double t_atomics = 1e4 + nbatch * (ant * taps * 0.05 + (double)g * g * 8 / 4000);
    if (t_bands <= t_atomics && nbands * nbatch <= 0x7fffffff) {
        const uint32_t magic = (uint32_t)((((uint64_t)1 << 32) + supp * supp - 1) / (supp * supp));
        auto run = [&](auto k) {
            hipLaunchKernelGGL(k, dim3((unsigned)(nbands * nbatch)), dim3(EPIC_THREADS),
                               ((size_t)rows * g * sizeof(float2) + 15) / 16 * 16, s,
                               (const float2 *)f, x, y, n_ant, (const float2 *)illum, supp, magic, g,
                               rows, nbatch, (float2 *)grids);
        };
        if (supp == 1)
            run(k_epic_band<1>);
        else if (supp == 2)
            run(k_epic_band<2>);
        else
            run(k_epic_band<0>);
        RG_HIP(hipGetLastError());
        return RG_OK;
    }
    RG_TRY(zero_fill(grids, sizeof(float2) * (size_t)nbatch * g * g, s));
    const int64_t per = ((int64_t)n_ant * supp * supp + 255) / 256;
    const unsigned share = (unsigned)std::max<int64_t>(1, std::min<int64_t>(per, 1024));
    hipLaunchKernelGGL(k_epic_atomic, dim3((unsigned)nbatch, share), dim3(256), 0, s,
                       (const float2 *)f, x, y, n_ant, (const float2 *)illum, supp, g,
                       (float2 *)grids);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

} // namespace rg
