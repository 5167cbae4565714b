"""The visibility sort at the edges of its forms: the one-workgroup sort of
short streams, scan blocks of one and four keys per thread, the two- and
three-launch scans, hot keys with many work items."""
import numpy as np
import pytest
import torch

import pyoracle as orc
import rgamd
from gpu_util import dev, kern, rel_max, stage

pytestmark = pytest.mark.gpu

THETA, S, R = 0.1, 8, 4


@pytest.fixture(scope="module")
def table():
    return rgamd.make_wkernels(11, R, S, THETA, -5.0, 1.0)


def stream(n, half, wmax, seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-half, half, n), rng.uniform(-half, half, n), rng.uniform(-wmax, wmax, n),
            rng.standard_normal(n) + 1j * rng.standard_normal(n))


@pytest.mark.parametrize("n", [0, 1, 31, 33, 1025, 4095, 4096, 4097, 23_000])
@pytest.mark.parametrize("per_item", [0, 5])
def test_wprojection_hot_tile(ctx, table, n, per_item):
    """Visibilities of a few tiles, some outside the table's planes: FP64 sums
    of at most 23 000 terms of order 0.1 against the oracle's."""
    N = 128
    u, v, w, vis = stream(n, 60.0, 6.0, n + 1)
    ref, _, bad = orc.grid_wprojection(N, THETA, u, v, w, vis, table, -5.0, 1.0)
    _, fv = stage(u, v, w, vis)
    _, wk = kern(table, -5.0, 1.0)
    g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    p = rgamd.params(N, THETA, vis_per_item=per_item)
    ctx.grid(p, fv, wk, g)
    st = ctx.stats()
    assert st.n_bad_plane == bad and st.n_gridded == n - bad and st.n_dropped == 0
    assert st.n_records == n - bad
    assert np.abs(g.cpu().numpy() - ref).max() <= 1e-12 * max(np.abs(ref).max(), 1e-300)
    g2 = torch.zeros_like(g)
    rgamd.grid_noalloc(p, fv, wk, g2)
    torch.cuda.synchronize()
    assert rel_max(g2.cpu().numpy(), ref) <= 1e-12 or n == 0


@pytest.mark.parametrize("nchan", [3, 60, 70])
def test_channels_across_scan_forms(ctx, table, nchan):
    """1089 keys per channel: below and above the 65 536 keys at which a scan
    thread takes four."""
    N = 1024
    counts = np.random.default_rng(nchan).integers(0, 300, nchan)
    counts[1] = 0
    counts[2] = 5000
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    u, v, w, vis = stream(off[-1], 4500.0, 5.0, 9)
    (du, dv, dw, dvis), fv = stage(u, v, w, vis)
    _, wk = kern(table, -5.0, 1.0)
    p = rgamd.params(N, THETA)
    g = torch.empty((nchan, N, N), dtype=torch.complex128, device="cuda")
    ctx.grid_channels(p, fv, off, wk, g)
    assert ctx.stats().n_gridded == off[-1]
    one = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    for c in (0, 1, 2, nchan - 1):
        a, b = off[c], off[c + 1]
        fc = rgamd.flat_vis(du[a:b].clone(), dv[a:b].clone(), dw[a:b].clone(), dvis[a:b].clone())
        ctx.grid(rgamd.params(N, THETA, mode=rgamd.RG_MODE_PLAIN), fc, wk, one)
        torch.cuda.synchronize()
        scale = max(float(one.abs().max()), 1e-300)
        assert float((g[c] - one).abs().max()) <= 1e-12 * scale


def test_wtowers_with_millions_of_keys(ctx, table):
    """2500 floors of 121 towers: over 2048 scan blocks, whose totals a launch
    of their own scans."""
    N = 512
    u, v, w, vis = stream(300, 2400.0, 12_000.0, 5)
    _, fv = stage(u, v, w, vis)
    _, wk = kern(table, -5.0, 1.0)
    kw = dict(subgrid=64, margin=16, winc=10.0)
    ref = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    g = torch.empty_like(ref)
    ctx.grid(rgamd.params(N, THETA, mode=rgamd.RG_MODE_PLAIN, **kw), fv, wk, ref)
    for _ in range(2):  # the measuring call, then one by its plan
        ctx.grid(rgamd.params(N, THETA, **kw), fv, wk, g)
        torch.cuda.synchronize()
        assert float((g - ref).abs().max()) <= 1e-11 * float(ref.abs().max())


def test_short_call_on_a_frozen_context(table):
    """Scratch held by a captured graph serves shorter calls, which pick other
    item sizes."""
    c = rgamd.Context(0)
    N = 128
    _, wk = kern(table, -5.0, 1.0)
    keep = [stage(*stream(n, 60.0, 4.0, n)) for n in (60_000, 30_000, 4096, 10)]
    g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    p = rgamd.params(N, THETA)
    c.grid(p, keep[0][1], wk, g)
    s = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=s):
        c.grid(p, keep[0][1], wk, g)
    want = torch.empty_like(g)
    for _, fv in keep:
        c.grid(p, fv, wk, g)
        ctx2 = rgamd.Context(0)
        ctx2.grid(rgamd.params(N, THETA, mode=rgamd.RG_MODE_PLAIN), fv, wk, want)
        torch.cuda.synchronize()
        assert float((g - want).abs().max()) <= 1e-12 * float(want.abs().max())
        ctx2.close()
    c.grid(p, keep[0][1], wk, want)
    for _ in range(3):
        g.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert float((g - want).abs().max()) <= 1e-12 * float(want.abs().max())
    del graph
    c.close()


@pytest.mark.parametrize("first,sizes", [
    (("c64", 60_000), (49_151, 12_287, 1_025, 60_000)), (("c64", 200_000), (196_607, 190_000)),
    (("c128", 60_000), (60_000, 49_151, 1_025)), (("towers", 60_000), (60_000, 49_151, 1_025))])
def test_single_precision_calls_on_a_frozen_context(table, first, sizes):
    """FP32 calls with an FP32 grid on a context whose scratch a captured graph holds: of a longer
    call of that kind, of one with an FP64 grid and of a W-towers one, neither of which has sums
    of dense tiles; at the lengths where the item size halves.  A cell is a sum of at most n products of four
    roundings each."""
    N, kind, n0 = 128, *first
    c, plain = rgamd.Context(0), rgamd.Context(0)
    _, wk = kern(table, -5.0, 1.0, torch.complex64)
    t64 = table.astype(np.complex64).astype(np.complex128)
    _, wk64 = kern(t64, -5.0, 1.0)
    _, wkabs = kern(np.abs(t64) + 0j, -5.0, 1.0)
    u, v, w, vis = stream(n0, 60.0, 4.0, 3)
    vis = vis.astype(np.complex64)
    g32 = torch.empty((N, N), dtype=torch.complex64, device="cuda")
    g128 = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    p = rgamd.params(N, THETA)
    keep, fv = stage(u, v, w, vis, torch.complex64)
    call = {"c64": (p, fv, wk, g32), "c128": (p, fv, wk, g128),
            "towers": (rgamd.params(N, THETA, subgrid=64, margin=16, winc=10.0), fv, wk, g128)}[kind]
    for _ in range(2):
        c.grid(*call)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c.grid(*call)
    want = call[3].clone()
    for n in sizes:
        k, f = stage(u[:n], v[:n], w[:n], vis[:n], torch.complex64)
        got = torch.empty_like(g32)
        c.grid(p, f, wk, got)
        _, f64 = stage(u[:n], v[:n], w[:n], vis[:n].astype(np.complex128))
        _, fabs = stage(u[:n], v[:n], w[:n], np.abs(vis[:n].astype(np.complex128)) + 0j)
        ref, mag = torch.empty_like(g128), torch.empty_like(g128)
        pp = rgamd.params(N, THETA, mode=rgamd.RG_MODE_PLAIN)
        plain.grid(pp, f64, wk64, ref)
        plain.grid(pp, fabs, wkabs, mag)
        torch.cuda.synchronize()
        assert ((got.to(torch.complex128) - ref).abs() <= (n + 4) * 2.0 ** -24 * mag.real).all(), n
    for _ in range(3):
        call[3].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert float((call[3] - want).abs().max()) <= 1e-5 * float(want.abs().max())
    del graph
    c.close()
    plain.close()


@pytest.mark.parametrize("captured", ["towers", "two channels"])
def test_more_keys_than_the_captured_call(table, captured):
    """On a context whose scratch a captured graph holds, W-projections of the same stream with more keys:
    after a W-towers call of few towers and one floor (2880 keys), after two sparse channels, whose
    tiles are wide (1024^2 grids, 4225 keys, and 1216^2, of about as many cells as the two channels have)."""
    N, n = 1024, 70_000
    c, plain = rgamd.Context(0), rgamd.Context(0)
    _, wk = kern(table, -5.0, 1.0)
    u, v, w, vis = stream(n, 4500.0, 4.0, 8)
    _, fv = stage(u, v, w, vis)
    off = np.array([0, n // 3, n], dtype=np.int64)
    if captured == "towers":
        p = rgamd.params(N, THETA, subgrid=512, margin=16, winc=10.0)
        g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
        call = lambda: c.grid(p, fv, wk, g)  # noqa: E731
    else:
        p = rgamd.params(N, THETA)
        g = torch.empty((2, N, N), dtype=torch.complex128, device="cuda")
        call = lambda: c.grid_channels(p, fv, off, wk, g)  # noqa: E731
    for _ in range(2):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    want = g.clone()
    for size in (N, 1216) if captured != "towers" else (N,):
        got = torch.empty((size, size), dtype=torch.complex128, device="cuda")
        ref = torch.empty_like(got)
        c.grid(rgamd.params(size, THETA), fv, wk, got)
        plain.grid(rgamd.params(size, THETA, mode=rgamd.RG_MODE_PLAIN), fv, wk, ref)
        torch.cuda.synchronize()
        assert float((got - ref).abs().max()) <= 1e-12 * float(ref.abs().max())
    for _ in range(3):
        g.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert float((g - want).abs().max()) <= 1e-12 * float(want.abs().max())
    del graph
    c.close()
    plain.close()


@pytest.mark.parametrize("tiles", [1, 2, 5, 30, 64])
@pytest.mark.parametrize("n", [5000, 70_001])
def test_few_keys_in_any_order(ctx, tiles, n):
    """Records that alternate between a few keys (tiles, and plane groups from 64 a tile on), some
    dropped, so that the lanes of a key stand apart in their wavefront: keys with one lane, two and many.
    FP64 against the plain form, W-projection and W-towers."""
    N, s, planes, r = 256, 8, 140, 8
    rng = np.random.default_rng(tiles)
    pick = rng.choice(tiles, n, p=1.0 / np.arange(1, tiles + 1) / (1.0 / np.arange(1, tiles + 1)).sum())
    place = rng.uniform(-110, 110, (2, tiles))
    u, v = (place[:, pick] + rng.uniform(0, 4, (2, n))) / THETA
    u[rng.integers(0, n, n // 50)] = 1e6
    w = rng.uniform(-0.4, planes - 0.6, n)
    vis = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    t = rng.standard_normal((planes, r, r, s, s)) + 1j * rng.standard_normal((planes, r, r, s, s))
    _, fv = stage(u, v, w, vis)
    _, wk = kern(t, 0.0, 1.0)
    g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    ref = torch.empty_like(g)
    for kw in ({}, dict(subgrid=64, margin=16, winc=200.0)):
        ctx.grid(rgamd.params(N, THETA, mode=rgamd.RG_MODE_PLAIN, **kw), fv, wk, ref)
        for _ in range(2):
            ctx.grid(rgamd.params(N, THETA, **kw), fv, wk, g)
            assert float((g - ref).abs().max()) <= 1e-11 * float(ref.abs().max())


def spread(n, N, planes, seed, even):
    """n visibilities over the grid and past its edges: evenly, or crowded as tracks are (the
    density falling by e every twentieth of the grid)."""
    rng = np.random.default_rng(seed)
    half = N / THETA / 2
    if even:
        u, v = rng.uniform(-1.02 * half, 1.02 * half, (2, n))
    else:
        r, t = rng.exponential(half / 10, n), rng.uniform(0, 2 * np.pi, n)
        u, v = r * np.cos(t), r * np.sin(t)
    return (u, v, rng.uniform(-0.5, planes - 0.4, n),
            rng.standard_normal(n) + 1j * rng.standard_normal(n))


@pytest.mark.parametrize("N,s,per", [(256, 16, 63.9), (256, 16, 64.1), (256, 16, 400), (256, 8, 400),
                                     (2100, 16, 7.9), (2100, 16, 8.1), (2100, 8, 20), (2100, 16, 64.1),
                                     (2100, 8, 64.1)])
def test_plane_groups_by_sample(N, s, per):
    """Streams of even coverage and crowded ones around 8 and 64 records a tile, grids below and
    above 64 MB: the number of plane groups comes from a sample of the stream, in the call, so that a
    captured call serves either.  FP64 sums against the plain form's: at most n products a cell."""
    planes, r = 300, 8
    one = ((N + s + 15) // 16) ** 2
    n = int(per * one)
    table = torch.randn((planes, r, r, s, s), dtype=torch.complex128, device="cuda")
    wk = rgamd.wkern_desc(table, 0.0, 1.0)
    c, plain = rgamd.Context(0), rgamd.Context(0)
    p, pp = rgamd.params(N, THETA), rgamd.params(N, THETA, mode=rgamd.RG_MODE_PLAIN)
    g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    ref = torch.empty_like(g)
    streams = [stage(*spread(n, N, planes, 5, even)) for even in (True, False)]
    (du, dv, dw, dvis), fv = stage(*spread(n, N, planes, 6, True))
    for keep, f in streams:
        plain.grid(pp, f, wk, ref)
        c.grid(p, f, wk, g)
        assert float((g - ref).abs().max()) <= 1e-12 * float(ref.abs().max())
        if n <= 700_000:
            rgamd.grid_noalloc(p, f, wk, g)
            assert float((g - ref).abs().max()) <= 1e-12 * float(ref.abs().max())
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        c.grid(p, fv, wk, g)
    for keep, f in streams * 2:
        for dst, src in zip((du, dv, dw, dvis), keep):
            dst.copy_(src)
        plain.grid(pp, f, wk, ref)
        g.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert float((g - ref).abs().max()) <= 1e-12 * float(ref.abs().max())
    del graph
    c.close()
    plain.close()


def crowd(n, N, s, planes, seed):
    """n visibilities: half in one 16 x 16 tile of positions (several a position), half over
    the grid and its edges; planes of the whole table."""
    rng = np.random.default_rng(seed)
    half = N / THETA / 2
    k = n // 2
    u = np.concatenate([rng.uniform(-60.0, 60.0, k), rng.uniform(-1.1 * half, 1.1 * half, n - k)])
    v = np.concatenate([rng.uniform(-60.0, 60.0, k), rng.uniform(-1.1 * half, 1.1 * half, n - k)])
    w = rng.uniform(-0.5, planes - 0.6, n)
    order = rng.permutation(n)
    return (u[order], v[order], w[order], rng.standard_normal(n) + 1j * rng.standard_normal(n))


@pytest.mark.parametrize("s,planes", [(16, 35), (8, 140)])
@pytest.mark.parametrize("n,per_item", [(15, 16), (16, 16), (17, 17), (65, 512), (129, 512),
                                        (1599, 0), (1600, 0), (1601, 513), (6000, 512)])
@pytest.mark.parametrize("dt,gdt,comp", [(torch.complex128, torch.complex128, 0),
                                         (torch.complex64, torch.complex64, 0),
                                         (torch.complex64, torch.complex128, 1)])
def test_wprojection_item_edges(ctx, s, planes, n, per_item, dt, gdt, comp):
    """Items up to and above the 16 records that are taken unordered, one and more chunks of 64,
    whole items of 512; streams below and above 64 records a tile (25 tiles at S = 16, 25 at
    S = 8), where planes come in groups (16 and 64 planes, the last one partial).  Every cell is
    a sum of at most n products, and a product takes four roundings: an error of
    (n + 4) eps sum |k| |v|, with the sum gridded from the absolute values."""
    N, r = 64, 8
    rng = np.random.default_rng(s)
    table = (rng.standard_normal((planes, r, r, s, s)) +
             1j * rng.standard_normal((planes, r, r, s, s)))
    u, v, w, vis = crowd(n, N, s, planes, n)
    np_dt = np.complex64 if dt == torch.complex64 else np.complex128
    table, vis = table.astype(np_dt).astype(np.complex128), vis.astype(np_dt).astype(np.complex128)
    ref, _, bad = orc.grid_wprojection(N, THETA, u, v, w, vis, table, 0.0, 1.0)
    mag, _, _ = orc.grid_wprojection(N, THETA, u, v, w, np.abs(vis) + 0j, np.abs(table) + 0j, 0.0,
                                     1.0)
    _, fv = stage(u, v, w, vis, dt)
    _, wk = kern(table, 0.0, 1.0, dt)
    g = torch.empty((N, N), dtype=gdt, device="cuda")
    ctx.grid(rgamd.params(N, THETA, vis_per_item=per_item, compensated=comp), fv, wk, g)
    st = ctx.stats()
    assert st.n_bad_plane == bad
    eps = 2.0 ** -24 if dt == torch.complex64 else 2.0 ** -53
    # the oracle's own sums, too, in FP64
    bound = (n + 4) * (eps + 2.0 ** -53) * mag.real
    err = np.abs(g.cpu().numpy().astype(np.complex128) - ref)
    assert (err <= bound).all(), float((err / np.maximum(bound, 1e-300)).max())


@pytest.mark.parametrize("planes", [35, 140])
@pytest.mark.parametrize("n", [599, 600, 601, 4799, 4800, 9000])
@pytest.mark.parametrize("dt,gdt,comp", [(torch.complex128, torch.complex128, 0),
                                         (torch.complex64, torch.complex64, 0),
                                         (torch.complex64, torch.complex128, 1)])
def test_channels_wide_tiles(ctx, planes, n, dt, gdt, comp):
    """Three channels around 8 and 64 records a tile (3 x 25 tiles), between which tiles are twice
    as wide, with one group of planes (35) and with groups of 64 (140).  The bound of the item test."""
    N, r, s = 64, 8, 16
    rng = np.random.default_rng(planes)
    table = (rng.standard_normal((planes, r, r, s, s)) +
             1j * rng.standard_normal((planes, r, r, s, s)))
    u, v, w, vis = crowd(n, N, s, planes, n)
    np_dt = np.complex64 if dt == torch.complex64 else np.complex128
    table, vis = table.astype(np_dt).astype(np.complex128), vis.astype(np_dt).astype(np.complex128)
    off = np.array([0, n // 5, n // 5, n], dtype=np.int64)  # the second channel is empty
    _, fv = stage(u, v, w, vis, dt)
    _, wk = kern(table, 0.0, 1.0, dt)
    g = torch.empty((3, N, N), dtype=gdt, device="cuda")
    ctx.grid_channels(rgamd.params(N, THETA, compensated=comp), fv, off, wk, g)
    eps = (2.0 ** -24 if dt == torch.complex64 else 2.0 ** -53) + 2.0 ** -53
    for c in range(3):
        sl = slice(off[c], off[c + 1])
        got = g[c].cpu().numpy().astype(np.complex128)
        if off[c] == off[c + 1]:
            assert not got.any()
            continue
        ref, _, _ = orc.grid_wprojection(N, THETA, u[sl], v[sl], w[sl], vis[sl], table, 0.0, 1.0)
        mag, _, _ = orc.grid_wprojection(N, THETA, u[sl], v[sl], w[sl], np.abs(vis[sl]) + 0j,
                                         np.abs(table) + 0j, 0.0, 1.0)
        assert (np.abs(got - ref) <= (n + 4) * eps * mag.real).all(), c


@pytest.mark.parametrize("per_item", [513, 1024, 2048, 4096])
def test_large_items_are_the_stream_s_choice(ctx, per_item):
    """Items of more records than a wavefront sorts are chosen by the stream's length, as 0 is:
    the same number of items; 512 is taken as it stands."""
    rng = np.random.default_rng(4)
    n, N = 30000, 512
    u, v = (rng.random((2, n)) - 0.5) * 40 / THETA
    _, fv = stage(u, v, np.zeros(n), np.ones(n, complex))
    _, wk = kern(np.ones((1, 2, 2, 8, 8), complex), 0.0, 1.0)
    g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    items = []
    for k in (0, per_item, 512):
        ctx.grid(rgamd.params(N, THETA, vis_per_item=k), fv, wk, g)
        items.append(ctx.stats().n_items)
    # 12 32^2 <= n < 12 64^2
    assert items[0] == items[1] >= n // 32 > 4 * items[2]


@pytest.mark.parametrize("nchan", [15, 16])
def test_channels_by_scan_threads_of_one_and_four_keys(ctx, table, nchan):
    """4225 tiles of 16 x 16 cells per channel (65^2): 63 375 keys, the last number of channels at
    which a scan thread takes one of them, and 67 600, where it takes four.  FP64 sums of at most
    5000 terms against the plain form's."""
    N = 1024
    counts = np.random.default_rng(nchan).integers(0, 300, nchan)
    counts[1], counts[2] = 0, 5000
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    u, v, w, vis = stream(off[-1], 4500.0, 5.0, 9)
    (du, dv, dw, dvis), fv = stage(u, v, w, vis)
    _, wk = kern(table, -5.0, 1.0)
    g = torch.empty((nchan, N, N), dtype=torch.complex128, device="cuda")
    ctx.grid_channels(rgamd.params(N, THETA), fv, off, wk, g)
    assert ctx.stats().n_gridded == off[-1]
    one = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    for c in range(nchan):
        a, b = off[c], off[c + 1]
        fc = rgamd.flat_vis(du[a:b].clone(), dv[a:b].clone(), dw[a:b].clone(), dvis[a:b].clone())
        ctx.grid(rgamd.params(N, THETA, mode=rgamd.RG_MODE_PLAIN), fc, wk, one)
        torch.cuda.synchronize()
        assert float((g[c] - one).abs().max()) <= 1e-12 * max(float(one.abs().max()), 1e-300)


@pytest.mark.parametrize("planes", [1536, 1537])
def test_plane_groups_by_the_size_of_the_table(ctx, planes):
    """FP32 sub-kernels of 8 x 8 taps: one plane group up to tables of 48 MB (1536 planes), as many as
    the stream asks for beyond.  Small whole numbers: FP32 sums are exact in any order, and equal
    to the plain form's."""
    N, n, r, s = 128, 200_000, 8, 8
    gen = torch.Generator(device="cuda").manual_seed(planes)
    small = lambda *sh: torch.randint(-2, 3, (*sh, 2), generator=gen, device="cuda",  # noqa: E731
                                      dtype=torch.int32).double()
    table = torch.view_as_complex(small(planes, r, r, s, s))
    u, v, _, _ = spread(n, N, planes, 3, True)
    w = np.random.default_rng(2).integers(0, planes, n).astype(float)
    vis = torch.view_as_complex(small(n)).cpu().numpy()
    got = torch.empty((N, N), dtype=torch.complex64, device="cuda")
    want = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    keep, f = stage(u, v, w, vis)
    ctx.grid(rgamd.params(N, THETA, mode=rgamd.RG_MODE_PLAIN), f, rgamd.wkern_desc(table, 0.0, 1.0),
             want)
    torch.cuda.synchronize()
    assert float(want.abs().max()) > 0
    t32 = table.to(torch.complex64)
    keep32, f32 = stage(u, v, w, vis, torch.complex64)
    wk = rgamd.wkern_desc(t32, 0.0, 1.0)
    for call in (ctx.grid, rgamd.grid_noalloc):
        got.fill_(1)
        call(rgamd.params(N, THETA), f32, wk, got)
        torch.cuda.synchronize()
        assert bool((torch.view_as_real(got.to(torch.complex128)) == torch.view_as_real(want)).all())
