"""Direct DFT on the GPU against the oracle; prediction against numpy."""
import math

import numpy as np
import pytest
import torch

import pyoracle as orc
import rgamd
import synth
from gpu_util import dev, rel_max, small_obs, stage

pytestmark = pytest.mark.gpu


def test_dft_fp64_and_mixed(ctx):
    obs, vis = small_obs(n_st=10, n_dumps=20)
    N, lam = obs.grid_size, obs.lam
    rng = np.random.default_rng(4)
    px = rng.integers(0, N, 500).astype(np.int32)
    py = rng.integers(0, N, 500).astype(np.int32)
    ref = orc.dft(px, py, N, lam, obs.u, obs.v, obs.w, vis)
    _, fv = stage(obs.u, obs.v, obs.w, vis)
    dpx, dpy = dev(px), dev(py)
    out = torch.empty(500, dtype=torch.complex128, device="cuda")
    ctx.dft(fv, dpx, dpy, N, lam, out, rgamd.RG_DFT_FP64)
    torch.cuda.synchronize()
    assert rel_max(out.cpu().numpy(), ref) < 1e-11
    ctx.dft(fv, dpx, dpy, N, lam, out, rgamd.RG_DFT_MIXED)
    torch.cuda.synchronize()
    assert rel_max(out.cpu().numpy(), ref) < 1e-5


def test_dft_image_layout_and_contract(ctx):
    obs, vis = small_obs(n_st=6, n_dumps=8, lam=320.0)
    N, lam = obs.grid_size, obs.lam
    _, fv = stage(obs.u, obs.v, obs.w, vis)
    img = torch.empty(N * N, dtype=torch.complex128, device="cuda")
    ctx.dft_image(fv, N, lam, img, N * N // 64, 64)
    torch.cuda.synchronize()
    ys, xs = np.divmod(np.arange(N * N), N)
    ref = orc.dft(xs, ys, N, lam, obs.u, obs.v, obs.w, vis)
    assert rel_max(img.cpu().numpy(), ref) < 1e-11
    with pytest.raises(rgamd.RGError) as e:
        ctx.dft_image(fv, N, lam, img, N * N // 64 - 1, 64)
    assert e.value.code == rgamd.RG_ERR_PARAM


def test_predict_matches_numpy():
    obs = synth.config_small(n_st=8, n_dumps=10, n_src=7)
    ref = synth.predict_numpy(obs.u, obs.v, obs.w, obs.l, obs.m, obs.flux)
    for dt, tol in ((torch.complex128, 1e-12), (torch.complex64, 1e-6)):
        out = torch.empty(obs.n_vis, dtype=dt, device="cuda")
        rgamd.predict_points(dev(obs.u), dev(obs.v), dev(obs.w), dev(obs.l), dev(obs.m),
                             dev(obs.flux), out)
        torch.cuda.synchronize()
        assert rel_max(out.cpu().numpy(), ref) < tol


def test_dft_split_over_visibility_ranges(ctx):
    """Few pixels and many visibilities: the stream is split over several
    ranges whose partial sums are added in order; same result as the oracle,
    and identical on a second run."""
    rng = np.random.default_rng(8)
    n = 300_000
    u, v = rng.uniform(-5000, 5000, n), rng.uniform(-5000, 5000, n)
    w = rng.uniform(-300, 300, n)
    vis = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    N, lam = 2048, 20480.0
    px = rng.integers(0, N, 40).astype(np.int32)
    py = rng.integers(0, N, 40).astype(np.int32)
    ref = orc.dft(px, py, N, lam, u, v, w, vis)
    for vdt, mode, tol in ((torch.complex128, rgamd.RG_DFT_FP64, 1e-11),
                           (torch.complex64, rgamd.RG_DFT_MIXED, 2e-5)):
        _, fv = stage(u, v, w, vis, vdt)
        out = torch.empty(40, dtype=torch.complex128, device="cuda")
        ctx.dft(fv, dev(px), dev(py), N, lam, out, mode)
        torch.cuda.synchronize()
        a = out.cpu().numpy()
        ctx.dft(fv, dev(px), dev(py), N, lam, out, mode)
        torch.cuda.synchronize()
        assert np.array_equal(a, out.cpu().numpy())
        assert rel_max(a, ref) < tol, mode


@pytest.mark.parametrize("npix,nvis", [(1, 1), (15, 16), (17, 15), (63, 17), (65, 255), (129, 513),
                                       (4096, 40), (4097, 33), (4351, 16), (130, 5000)])
@pytest.mark.parametrize("vdt", [torch.complex128, torch.complex64])
def test_dft_tile_remainders(ctx, npix, nvis, vdt):
    """One (up to 4096 pixels) and four 16-pixel tiles per wavefront, visibility steps of 16 and ranges of 256 with
    remainders.  Each term's phase (below 400 turns, three rounded products)
    is off by at most 2 pi * 400 * 3 * 2^-53 = 8e-13 of its visibility."""
    rng = np.random.default_rng(npix * 7 + nvis)
    u, v = rng.uniform(-3000, 3000, nvis), rng.uniform(-3000, 3000, nvis)
    w = rng.uniform(-300, 300, nvis)
    vis = rng.standard_normal(nvis) + 1j * rng.standard_normal(nvis)
    N, lam = 2048, 20480.0
    px = rng.integers(0, N, npix).astype(np.int32)
    py = rng.integers(0, N, npix).astype(np.int32)
    _, fv = stage(u, v, w, vis, vdt)
    ref = orc.dft(px, py, N, lam, u, v, w, vis.astype(np.complex64).astype(np.complex128)
                  if vdt == torch.complex64 else vis)
    out = torch.empty(npix, dtype=torch.complex128, device="cuda")
    ctx.dft(fv, dev(px), dev(py), N, lam, out)
    torch.cuda.synchronize()
    assert np.abs(out.cpu().numpy() - ref).max() < 1e-12 * np.abs(vis).sum()


@pytest.mark.parametrize("mode,tol", [(rgamd.RG_DFT_FP64, 1e-11), (rgamd.RG_DFT_MIXED, 2e-5)])
@pytest.mark.parametrize("warm", [0, 40, 400])
def test_dft_capture_keeps_its_partial_sums(mode, tol, warm):
    """A captured DFT takes no more partial sums than the scratch of the calls before it holds
    (none, some, all of what it would like), and later calls on the context, which would like more
    of it, leave it in place: they are right, and so is every replay after them."""
    rng = np.random.default_rng(5)
    N, lam = 2048, 20480.0
    c = rgamd.Context(0)

    def stream(n, npix):
        u, v = rng.uniform(-5000, 5000, (2, n))
        w = rng.uniform(-300, 300, n)
        vis = rng.standard_normal(n) + 1j * rng.standard_normal(n)
        px, py = rng.integers(0, N, (2, npix)).astype(np.int32)
        keep, fv = stage(u, v, w, vis)
        return (keep, fv, dev(px), dev(py), torch.empty(npix, dtype=torch.complex128, device="cuda"),
                orc.dft(px, py, N, lam, u, v, w, vis))

    a, b = stream(140_000, 400), stream(200_000, 500)
    if warm:
        c.dft(a[1], a[2][:warm].clone(), a[3][:warm].clone(), N, lam, a[4][:warm].clone(), mode)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c.dft(a[1], a[2], a[3], N, lam, a[4], mode,
              stream=torch.cuda.current_stream().cuda_stream)
    for rep in range(3):
        c.dft(b[1], b[2], b[3], N, lam, b[4], mode)
        a[4].zero_()
        torch.cuda.synchronize()
        assert rel_max(b[4].cpu().numpy(), b[5]) < tol
        graph.replay()
        torch.cuda.synchronize()
        assert rel_max(a[4].cpu().numpy(), a[5]) < tol, rep
    del graph
    c.thaw()
    c.dft(b[1], b[2], b[3], N, lam, b[4], mode)
    torch.cuda.synchronize()
    assert rel_max(b[4].cpu().numpy(), b[5]) < tol
    c.close()


@pytest.mark.parametrize("vdt", [torch.complex128, torch.complex64])
@pytest.mark.parametrize("npix", [300, 5000])
def test_dft_flagged_samples_far_away(ctx, vdt, npix):
    """Samples at coordinates far outside any array, whose phases have no digits left below a turn,
    add nothing if their value is 0 and at most its modulus otherwise.  The bound of the tile test
    on the rest."""
    rng = np.random.default_rng(npix)
    n, N, lam = 2000, 2048, 20480.0
    u, v = rng.uniform(-3000, 3000, (2, n))
    w = rng.uniform(-300, 300, n)
    vis = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64).astype(complex)
    px, py = rng.integers(0, N, (2, npix)).astype(np.int32)
    far = rng.permutation(n)[:400]
    vis[far] = 0
    ref = orc.dft(px, py, N, lam, u, v, w, vis)
    bound = 1e-12 * np.abs(vis).sum()
    u[far[:300]] = 10.0 ** rng.uniform(14, 24, 300)
    v[far[100:]] = -10.0 ** rng.uniform(14, 24, 300)
    w[far[300:]], u[far[:3]] = 1e22, 1e300
    for value in (0.0, 1.0):
        vis[far] = value
        _, fv = stage(u, v, w, vis, vdt)
        out = torch.empty(npix, dtype=torch.complex128, device="cuda")
        ctx.dft(fv, dev(px), dev(py), N, lam, out)
        torch.cuda.synchronize()
        assert (np.abs(out.cpu().numpy() - ref) <= bound + value * 400 * (1 + 1e-12)).all()
