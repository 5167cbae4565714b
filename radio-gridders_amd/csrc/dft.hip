// dft.hip -- direct DFT (the accuracy oracle of the reference, dft_cuda.cu)
// and point-source prediction of synthetic visibilities.
#include <algorithm>

#include "binning.hpp"

namespace rg {

constexpr int DFT_THREADS = 256;

// Pixel p of the call: from the list, or of the full image (row-major).
template <bool LIST>
__device__ inline void dft_pixel(const int32_t *px, const int32_t *py, int64_t p, int N,
                                 double lambda, double &l, double &m, double &nn)
{
    int x, y;
    if (LIST) {
        x = px[p];
        y = py[p];
    } else {
        y = (int)(p / N);
        x = (int)(p - (int64_t)y * N);
    }
    l = ((double)(y - N / 2) / lambda) * 1.0;
    m = ((double)(x - N / 2) / lambda) * 1.0;
    nn = 1 - sqrt(1 - l * l - m * m);
}

// FP32-rotation mode.  One thread per pixel; visibilities are staged through
// LDS in chunks of DFT_THREADS.  The phase l u + m v + (1 - n) w stays FP64, is
// reduced mod 1, the rotation is FP32 and each chunk is summed in FP32 into an
// FP64 sum (calculate_dft_sum_flat, dft_cuda.cu:15-39, at the pixel map of
// image_dft_flat, dft_cuda.cu:98-112).  With few pixels the visibility stream
// is also split over gridDim.y ranges: range r writes its partial sums to
// out + r * npix and k_dft_sum adds the ranges in order (the same summation
// order on every run).
template <bool LIST, typename VT>
__global__ __launch_bounds__(DFT_THREADS) void k_dft_mixed(
    const double *__restrict__ u, const double *__restrict__ v, const double *__restrict__ w,
    const VT *__restrict__ vis, int64_t nvis, const int32_t *__restrict__ px,
    const int32_t *__restrict__ py, int64_t npix, int N, double lambda, double2 *out)
{
    const int64_t per = (nvis + gridDim.y - 1) / gridDim.y;
    const int64_t v0 = per * blockIdx.y, v1 = min(nvis, v0 + per);
    out += (int64_t)blockIdx.y * npix;
    __shared__ double su[DFT_THREADS], sv[DFT_THREADS], sw[DFT_THREADS];
    __shared__ double2 svis[DFT_THREADS];
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    double l, m, nn;
    dft_pixel<LIST>(px, py, min(p, npix - 1), N, lambda, l, m, nn);
    double re = 0.0, im = 0.0;
    for (int64_t base = v0; base < v1; base += DFT_THREADS) {
        const int nloc = (int)min((int64_t)DFT_THREADS, v1 - base);
        __syncthreads();
        if ((int)threadIdx.x < nloc) {
            const int64_t i = base + threadIdx.x;
            su[threadIdx.x] = u[i];
            sv[threadIdx.x] = v[i];
            sw[threadIdx.x] = w[i];
            svis[threadIdx.x] = make_double2((double)vis[i].x, (double)vis[i].y);
        }
        __syncthreads();
        float fre = 0.f, fim = 0.f;
        for (int j = 0; j < nloc; ++j) {
            const double ph = l * su[j] + m * sv[j] + nn * sw[j];
            const float f = (float)(ph - rint(ph)); // revolutions in [-1/2, 1/2]
            float s, c;
            sincospif(2.0f * f, &s, &c);
            const float vr = (float)svis[j].x, vi = (float)svis[j].y;
            fre += vr * c + vi * s;
            fim += -vr * s + vi * c;
        }
        re += fre;
        im += fim;
    }
    if (p < npix)
        out[p] = make_double2(re, im);
}

// sin and cos of pi t, t given in half turns.  t = q + r with q the nearest
// integer and r exact; both series are Chebyshev fits in r^2 over |r| <= 1/2
// with 9 terms (errors 7e-19 and 4e-18; 3.1e-17 and 9.8e-17 with the
// coefficients rounded to FP64), and q mod 2 is the common sign: adding 1.5 * 2^52
// leaves q in the low mantissa bits for |t| < 2^51.  (From there on t has no digits
// left below half a turn: any sign will do, but r has to stay the remainder.)  Against
// libm's sincos of the angle in radians (argument reduction with pi, branches, about 75
// instructions) this is 25 instructions without a branch.
__device__ inline void half_turn_sincos(double t, double &s, double &c)
{
    const double qm = t + 6755399441055744.0; // 1.5 * 2^52
    const double r = t - rint(t);
    const double z = r * r;
    double ps = 7.697826768224191e-07, pc = 4.149564353942586e-06;
    ps = fma(ps, z, -2.1903497074626018e-05);
    pc = fma(pc, z, -0.00010456655338748738);
    ps = fma(ps, z, 0.0004662998161898394);
    pc = fma(pc, z, 0.0019295562724817132);
    ps = fma(ps, z, -0.007370430505916944);
    pc = fma(pc, z, -0.025806888737002202);
    ps = fma(ps, z, 0.0821458865731029);
    pc = fma(pc, z, 0.23533063012953284);
    ps = fma(ps, z, -0.5992645293189447);
    pc = fma(pc, z, -1.335262768843447);
    ps = fma(ps, z, 2.5501640398773007);
    pc = fma(pc, z, 4.058712126416497);
    ps = fma(ps, z, -5.167712780049969);
    pc = fma(pc, z, -4.934802200544676);
    ps = fma(ps, z, 3.141592653589793);
    pc = fma(pc, z, 1.0);
    ps *= r;
    const int sign = (int)((unsigned)__double2loint(qm) << 31);
    s = __hiloint2double(__double2hiint(ps) ^ sign, __double2loint(ps));
    c = __hiloint2double(__double2hiint(pc) ^ sign, __double2loint(pc));
}

// FP64 mode (calculate_dft_sum_flat, dft_cuda.cu:15-39, at the pixel map of
// image_dft_flat, dft_cuda.cu:98-112).  A wavefront owns PT tiles of 16 pixels
// and walks its range of the stream 16 visibilities at a time.  The phases of
// a 16 x 16 tile are a product with inner dimension 3, (l, m, 1 - n) times
// (u, v, w), and come from one v_mfma_f64_16x16x4 on the matrix pipe; the
// vector pipe is left with the sine, the cosine and the sum.  Lane (k, j) =
// (lane / 16, lane % 16) holds component k of pixel j (A, kept in registers) and
// of visibility j (B, one load), and gets the phases of pixels k + 4 i, i < 4,
// with visibility j, so it sums its own visibilities for those four pixels and
// the 16 lanes of a row are added once at the end.  Visibilities past the
// range enter as zeros (phase 0, value 0).
// Bound by the FP64 rate: 28 vector instructions (25 of them FP64) and a
// quarter of an MFMA per pixel and visibility.  65 536 pixels x 262 144
// visibilities: 41.2 ms with libm's sincos and one thread per pixel, 16.3 ms
// now (1.05e12 rotations/s, 26e12 FP64 lane instructions/s of the 39e12 the
// vector pipe issues at its peak clock).
typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int DFT_WAVES = DFT_THREADS / 64;

template <bool LIST, typename VT, int PT>
__global__ __launch_bounds__(DFT_THREADS) void k_dft_fp64(
    const double *__restrict__ u, const double *__restrict__ v, const double *__restrict__ w,
    const VT *__restrict__ vis, int64_t nvis, int64_t per, const int32_t *__restrict__ px,
    const int32_t *__restrict__ py, int64_t npix, int N, double lambda,
    double2 *__restrict__ out)
{
    const int lane = threadIdx.x % 64, k = lane / 16, j = lane % 16;
    const int64_t p0 =
        ((int64_t)blockIdx.x * DFT_WAVES + threadIdx.x / 64) * (16 * PT);
    const int64_t v0 = per * blockIdx.y, v1 = min(nvis, v0 + per);
    if (p0 >= npix)
        return;
    double a[PT];
    double re[PT][4], im[PT][4];
#pragma unroll
    for (int t = 0; t < PT; ++t) {
        double c[4] = {0.0, 0.0, 0.0, 0.0};
        const int64_t p = p0 + 16 * t + j;
        if (p < npix)
            dft_pixel<LIST>(px, py, p, N, lambda, c[0], c[1], c[2]);
        // phases in half turns
        a[t] = 2.0 * (k == 0 ? c[0] : k == 1 ? c[1] : k == 2 ? c[2] : 0.0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            re[t][i] = im[t][i] = 0.0;
    }
    const double *comp = k == 0 ? u : k == 1 ? v : w;
    // visibility v of the next step: loaded one step ahead
    auto load = [&](int64_t i, double &b, double &vr, double &vi) {
        b = vr = vi = 0.0;
        if (i < v1) {
            const VT e = vis[i];
            vr = (double)e.x;
            vi = (double)e.y;
            if (k < 3)
                b = comp[i];
        }
    };
    double b, vr, vi;
    load(v0 + j, b, vr, vi);
    for (int64_t base = v0; base < v1; base += 16) {
        double bn, vrn, vin;
        load(base + 16 + j, bn, vrn, vin);
#pragma unroll
        for (int t = 0; t < PT; ++t) {
            const v4d ph = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b, v4d{0.0, 0.0, 0.0, 0.0},
                                                                0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                double s, c;
                half_turn_sincos(ph[i], s, c);
                re[t][i] = fma(vr, c, fma(vi, s, re[t][i]));
                im[t][i] = fma(vi, c, fma(-vr, s, im[t][i]));
            }
        }
        b = bn;
        vr = vrn;
        vi = vin;
    }
    out += (int64_t)blockIdx.y * npix;
#pragma unroll
    for (int t = 0; t < PT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            double x = re[t][i], y = im[t][i];
            for (int o = 8; o > 0; o >>= 1) {
                x += __shfl_xor(x, o);
                y += __shfl_xor(y, o);
            }
            const int64_t p = p0 + 16 * t + k + 4 * i;
            if (j == 0 && p < npix)
                out[p] = make_double2(x, y);
        }
}

// out[p] = sum over ranges r of part[r][p], r in order
__global__ __launch_bounds__(256) void k_dft_sum(const double2 *__restrict__ part, int nr,
                                                 int64_t npix, double2 *out)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npix)
        return;
    double2 a = part[p];
    for (int r = 1; r < nr; ++r) {
        const double2 b = part[(int64_t)r * npix + p];
        a.x += b.x;
        a.y += b.y;
    }
    out[p] = a;
}

// Ranges the partial sums of which the context's scratch can take: as many as wanted,
// but a call that is being captured allocates nothing and none takes the scratch away
// from a captured one, so these make do with the ranges that fit it (one needs none).
static int dft_fit(rg_context *ctx, int64_t &nr, int64_t npix, bool &capturing, hipStream_t s)
{
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    RG_HIP(hipStreamIsCapturing(s, &cap));
    capturing = cap != hipStreamCaptureStatusNone;
    if (capturing || ctx->frozen || ctx->dft_captured)
        nr = std::max<int64_t>(
            1, std::min<int64_t>(nr, (int64_t)(ctx->scratch[14].bytes / sizeof(double2)) / npix));
    return RG_OK;
}

// partial sums of nr ranges (fitted) in scratch when there are several
static int dft_ranges(rg_context *ctx, int64_t nr, int64_t npix, bool capturing, double2 *out,
                      double2 **dst)
{
    *dst = out;
    if (nr > 1) {
        RG_TRY(ctx->scratch[14].ensure(sizeof(double2) * (size_t)(nr * npix)));
        *dst = ctx->scratch[14].as<double2>();
        ctx->dft_captured = ctx->dft_captured || capturing;
    }
    return RG_OK;
}

static int dft_add_ranges(int64_t nr, int64_t npix, const double2 *part, double2 *out,
                          hipStream_t s)
{
    if (nr > 1) {
        hipLaunchKernelGGL(k_dft_sum, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, s, part,
                           (int)nr, npix, out);
        RG_HIP(hipGetLastError());
    }
    return RG_OK;
}

// Ranges of at least 64 K visibilities, at most 256, enough for about 4096
// workgroups of 256 pixels: one range (no scratch) below 131 072 visibilities.
static int64_t long_ranges(int64_t nvis, int64_t npix)
{
    const int64_t blocks = (npix + DFT_THREADS - 1) / DFT_THREADS;
    const int64_t nr = std::min<int64_t>(256, (4096 + blocks - 1) / blocks);
    return std::max<int64_t>(1, std::min<int64_t>(nr, nvis / 65536));
}

template <bool LIST, typename VT>
static int launch_mixed(rg_context *ctx, const rg_flat_vis *vis, const int32_t *px,
                        const int32_t *py, int64_t npix, int N, double lambda, double2 *out,
                        hipStream_t s)
{
    const int64_t blocks = (npix + DFT_THREADS - 1) / DFT_THREADS;
    int64_t nr = long_ranges(vis->n, npix);
    bool capturing;
    RG_TRY(dft_fit(ctx, nr, npix, capturing, s));
    double2 *dst;
    RG_TRY(dft_ranges(ctx, nr, npix, capturing, out, &dst));
    hipLaunchKernelGGL((k_dft_mixed<LIST, VT>), dim3((unsigned)blocks, (unsigned)nr),
                       dim3(DFT_THREADS), 0, s, vis->u, vis->v, vis->w, (const VT *)vis->vis,
                       vis->n, px, py, npix, N, lambda, dst);
    RG_HIP(hipGetLastError());
    return dft_add_ranges(nr, npix, dst, out, s);
}

template <bool LIST, typename VT, int PT>
static int launch_fp64(rg_context *ctx, const rg_flat_vis *vis, const int32_t *px,
                       const int32_t *py, int64_t npix, int N, double lambda, double2 *out,
                       hipStream_t s)
{
    const int64_t per_block = (int64_t)DFT_WAVES * 16 * PT;
    const int64_t blocks = (npix + per_block - 1) / per_block;
    // visibility ranges: about 4096 workgroups in all (16 per CU, two rounds of
    // the 8 that fit), at least 256 visibilities each (the epilogue and the
    // partial sums stay below a few percent), at most 1024
    int64_t nr = std::min<int64_t>(1024, (4096 + blocks - 1) / blocks);
    nr = std::max<int64_t>(1, std::min<int64_t>(nr, vis->n / 256));
    bool capturing;
    RG_TRY(dft_fit(ctx, nr, npix, capturing, s));
    const int64_t per = ((vis->n + nr - 1) / nr + 15) / 16 * 16;
    nr = std::max<int64_t>(1, (vis->n + per - 1) / std::max<int64_t>(per, 1));
    double2 *dst;
    RG_TRY(dft_ranges(ctx, nr, npix, capturing, out, &dst));
    hipLaunchKernelGGL((k_dft_fp64<LIST, VT, PT>), dim3((unsigned)blocks, (unsigned)nr),
                       dim3(DFT_THREADS), 0, s, vis->u, vis->v, vis->w, (const VT *)vis->vis,
                       vis->n, per, px, py, npix, N, lambda, dst);
    RG_HIP(hipGetLastError());
    return dft_add_ranges(nr, npix, dst, out, s);
}

template <bool LIST, typename VT>
static int launch_dft(rg_context *ctx, const rg_flat_vis *vis, const int32_t *px,
                      const int32_t *py, int64_t npix, int N, double lambda, double2 *out, int mode,
                      hipStream_t s)
{
    if (npix == 0)
        return RG_OK;
    if (mode == RG_DFT_MIXED)
        return launch_mixed<LIST, VT>(ctx, vis, px, py, npix, N, lambda, out, s);
    // four pixel tiles per wavefront share a step's loads (65 536 pixels: 17.4 ms
    // with one, 16.6 with two, 16.2 with four); one while there are few pixels,
    // where the tiles past the last pixel would be idle work
    if (npix <= 4096)
        return launch_fp64<LIST, VT, 1>(ctx, vis, px, py, npix, N, lambda, out, s);
    return launch_fp64<LIST, VT, 4>(ctx, vis, px, py, npix, N, lambda, out, s);
}

int dft_run(rg_context *ctx, const rg_flat_vis *vis, const int32_t *px, const int32_t *py,
            int64_t npix, int N, double lambda, void *out, int mode, hipStream_t s)
{
    double2 *o = (double2 *)out;
    const bool c128 = vis->vis_type == RG_C128;
    if (px)
        return c128 ? launch_dft<true, double2>(ctx, vis, px, py, npix, N, lambda, o, mode, s)
                    : launch_dft<true, float2>(ctx, vis, px, py, npix, N, lambda, o, mode, s);
    return c128 ? launch_dft<false, double2>(ctx, vis, px, py, npix, N, lambda, o, mode, s)
                : launch_dft<false, float2>(ctx, vis, px, py, npix, N, lambda, o, mode, s);
}

// ---- point-source prediction ----------------------------------------------------

template <typename VT>
__global__ __launch_bounds__(256) void k_predict(const double *__restrict__ u,
                                                 const double *__restrict__ v,
                                                 const double *__restrict__ w, int64_t n,
                                                 const double *__restrict__ l,
                                                 const double *__restrict__ m,
                                                 const double *__restrict__ flux, int nsrc,
                                                 VT *out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const double ui = u[i], vi = v[i], wi = w[i];
    double re = 0.0, im = 0.0;
    for (int k = 0; k < nsrc; ++k) {
        const double nk = sqrt(1.0 - l[k] * l[k] - m[k] * m[k]);
        const double ph = ui * l[k] + vi * m[k] + wi * (nk - 1.0);
        const double f = ph - rint(ph);
        double s, c;
        sincospi(2.0 * f, &s, &c);
        // exp(-2 pi i ph)
        re += flux[k] * c;
        im -= flux[k] * s;
    }
    out[i].x = re;
    out[i].y = im;
}

int predict_run(const double *u, const double *v, const double *w, int64_t n, const double *l,
                const double *m, const double *flux, int nsrc, void *out, int type, hipStream_t s)
{
    const int64_t blocks = (n + 255) / 256;
    if (blocks == 0)
        return RG_OK;
    if (type == RG_C128)
        hipLaunchKernelGGL(k_predict<double2>, dim3((unsigned)blocks), dim3(256), 0, s, u, v, w, n,
                           l, m, flux, nsrc, (double2 *)out);
    else
        hipLaunchKernelGGL(k_predict<float2>, dim3((unsigned)blocks), dim3(256), 0, s, u, v, w, n, l,
                           m, flux, nsrc, (float2 *)out);
    RG_HIP(hipGetLastError());
    return RG_OK;
}

} // namespace rg
