// epic.hip -- EPIC E-field gridding: scatter_grid_kernel / epic_romein
// (src/epic/epic_grid.cu:54-218), batches of antenna E-fields each gridded
// with a small illumination pattern onto its own g x g grid.
//
// A workgroup owns a band of rows of one batch's grid in LDS: it adds the taps
// of every antenna that fall on its rows there (one thread per antenna, LDS
// float atomics) and writes the rows to HBM once, coalesced: no global atomics,
// one pass of output traffic, nothing cleared in HBM.  Grids of any size are
// cut into bands; a grid of so many bands that every workgroup's look at all antennas would cost
// more than the output (many antennas on a large grid) is cleared and added
// to with global atomics instead.
#include <algorithm>

#include "rg_internal.hpp"

namespace rg {

constexpr int EPIC_THREADS = 256;
constexpr int EPIC_LDS = 32 * 1024;

// c[j] += val[j] for the active j of N distinct cells, among the lanes of the
// workgroup: compare-and-swap of the 64-bit pair, the N of them in flight
// together, retried by the lanes that lost a cell to another (at least one of
// the lanes that meet on a cell succeeds in every round).  ds_add_f32 takes
// four to five cycles a lane here: 1000 grids of 256 antennas, 2 x 2 taps, 18.0 us
// with it, 8.4 us (the launch's own time) with these.
template <int N>
__device__ inline void lds_add(float2 *const (&c)[N], const float2 (&val)[N], uint32_t active)
{
    unsigned long long seen[N];
#pragma unroll
    for (int j = 0; j < N; ++j)
        if ((active >> j) & 1u)
            seen[j] = *reinterpret_cast<unsigned long long *>(c[j]);
    while (active) {
        unsigned long long got[N];
#pragma unroll
        for (int j = 0; j < N; ++j)
            if ((active >> j) & 1u) {
                float2 v = __builtin_bit_cast(float2, seen[j]);
                v.x += val[j].x;
                v.y += val[j].y;
                got[j] = atomicCAS(reinterpret_cast<unsigned long long *>(c[j]), seen[j],
                                   __builtin_bit_cast(unsigned long long, v));
            }
#pragma unroll
        for (int j = 0; j < N; ++j)
            if ((active >> j) & 1u) {
                if (got[j] == seen[j])
                    active &= ~(1u << j);
                seen[j] = got[j];
            }
    }
}

// SUPP: the support, or 0 to take it at run time.  N taps of a footprint row at
// a time (the whole 2 x 2).  One thread per antenna: the lanes take the same
// taps at the same time, so two of them meet on a cell only when their antennas
// stand on one.  BYROW: one thread per antenna and footprint row, for large
// footprints on grids of several bands, where most of an antenna's rows miss
// the band (300 antennas, 8 x 8 taps, 256^2: 27 -> 14.5 us), while there is at most a
// tap per cell (beyond, the lanes meet on cells: 512 antennas, 64^2: 48 -> 68 us).
template <int SUPP, int N, bool BYROW>
__global__ __launch_bounds__(EPIC_THREADS) void k_epic_band(
    const float2 *__restrict__ f, const int32_t *__restrict__ x, const int32_t *__restrict__ y,
    int n_ant, const float2 *__restrict__ illum, int supp_rt, int g, int rows, int nbands,
    float2 *__restrict__ grids)
{
    extern __shared__ __align__(16) float2 sg[];
    const int supp = SUPP ? SUPP : supp_rt;
    const unsigned b = blockIdx.x / (unsigned)nbands;
    const int r0 = (int)(blockIdx.x - b * (unsigned)nbands) * rows, r1 = min(g, r0 + rows);
    const int cells = (r1 - r0) * g;
    const size_t a0 = (size_t)b * n_ant;
    const int work = BYROW ? n_ant * supp : n_ant;
    // the first antenna's loads are in flight while the band is cleared
    int w = threadIdx.x, X0 = 0, Y0 = 0, row0 = 0;
    float2 v = make_float2(0.f, 0.f);
    auto load = [&]() {
        if (w < work) {
            const int a = BYROW ? w / supp : w;
            row0 = BYROW ? w - a * supp : 0;
            X0 = x[a0 + a];
            Y0 = y[a0 + a];
            v = f[a0 + a];
        }
    };
    load();
    for (int e = threadIdx.x; e < (cells + 1) / 2; e += EPIC_THREADS)
        reinterpret_cast<float4 *>(sg)[e] = make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();
    constexpr int NR = SUPP == 2 ? 2 : 1; // footprint rows at a time
    static_assert(SUPP != 2 || N == 4, "the whole 2 x 2");
    for (; w < work; w += EPIC_THREADS, load()) {
        const int row1 = BYROW ? row0 + 1 : supp;
        for (int ty0 = row0; ty0 < row1; ty0 += NR) {
            // rows off the grid lie outside every band
            if (NR == 1 && ((int64_t)Y0 + ty0 < r0 || (int64_t)Y0 + ty0 >= r1))
                continue;
#pragma unroll 1
            for (int t0 = 0; t0 < supp; t0 += N / NR) {
                float2 *c[N];
                float2 val[N];
                uint32_t active = 0;
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    const int tx = t0 + j / NR, ty = ty0 + j % NR;
                    const int64_t X = (int64_t)X0 + tx, Y = (int64_t)Y0 + ty;
                    // scatter_grid_add's bounds check
                    const bool in = tx < supp && X >= 0 && X < g && Y >= r0 && Y < r1;
                    const float2 k = illum[ty * supp + min(tx, supp - 1)];
                    c[j] = sg + (in ? (int)(Y - r0) * g + (int)X : 0);
                    // conj(k) v (epic_grid.cu:121-123)
                    val[j] = make_float2(k.x * v.x + k.y * v.y, k.x * v.y - k.y * v.x);
                    active |= (in ? 1u : 0u) << j;
                }
                lds_add<N>(c, val, active);
            }
        }
    }
    __syncthreads();
    float2 *out = grids + (size_t)b * g * g + (size_t)r0 * g;
    if ((reinterpret_cast<uintptr_t>(out) & 15) == 0 && cells % 2 == 0) {
        for (int e = threadIdx.x; e < cells / 2; e += EPIC_THREADS)
            reinterpret_cast<float4 *>(out)[e] = reinterpret_cast<const float4 *>(sg)[e];
    } else {
        for (int e = threadIdx.x; e < cells; e += EPIC_THREADS)
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
    // Bands of up to 32 KiB (five workgroups per CU), and shorter ones while there
    // are fewer than 1024 of them.  Every workgroup looks at all antennas of its batch,
    // which stays below the cost of writing the grid while bands x antennas <= 4 g^2.
    int rows = std::max(1, std::min(g, EPIC_LDS / (8 * g)));
    while (rows > 8 && (int64_t)nbatch * ((g + rows - 1) / rows) < 1024)
        rows = (rows + 1) / 2;
    const int64_t nbands = (g + rows - 1) / rows;
    if (nbands * n_ant <= (int64_t)4 * g * g && nbands * nbatch <= 0x7fffffff) {
        auto run = [&](auto k) {
            hipLaunchKernelGGL(k, dim3((unsigned)(nbands * nbatch)), dim3(EPIC_THREADS),
                               ((size_t)rows * g * sizeof(float2) + 15) / 16 * 16, s,
                               (const float2 *)f, x, y, n_ant, (const float2 *)illum, supp, g,
                               rows, (int)nbands, (float2 *)grids);
        };
        if (supp == 1)
            run(k_epic_band<1, 1, false>);
        else if (supp == 2)
            run(k_epic_band<2, 4, false>);
        else if (supp == 3)
            run(k_epic_band<3, 3, false>);
        else if (nbands > 1 && (int64_t)n_ant * supp * supp <= (int64_t)g * g)
            run(k_epic_band<0, 4, true>);
        else
            run(k_epic_band<0, 1, false>);
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
