"""W-stacking predict on the GPU against the oracle restatement (reduced
grid, FP64 to 1e-10) and, at the reference test's full geometry (theta 0.1,
lambda 20480: 4096^2 x 8 planes), against the direct sum over the quantised
sky within the method's error."""
import os
import re
import subprocess

import numpy as np
import pytest
import torch

import pyoracle as orc
import rgamd
from gpu_util import dev

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not rgamd.lib().rg_hdf5_available(), reason="libhdf5 not loadable")]

SZE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "sze")


@pytest.fixture(scope="module")
def kernels():
    uv = rgamd.load_sep_kern(os.path.join(SZE, "sepkern_uv_transpose.hdf5"), True)
    w = rgamd.load_sep_kern(os.path.join(SZE, "sepkern_w_transpose.hdf5"), True)
    lm = rgamd.load_sep_kern(os.path.join(SZE, "sepkern_lm.hdf5"), False)
    n = rgamd.load_sep_kern(os.path.join(SZE, "sepkern_n.hdf5"), False)
    d = {k: dev(x.data) for k, x in dict(uv=uv, w=w, lm=lm, n=n).items()}
    desc = {k: rgamd.sep_kern_desc(d[k], x.size, x.oversampling)
            for k, x in dict(uv=uv, w=w, lm=lm, n=n).items()}
    return dict(host=dict(uv=uv, w=w, lm=lm, n=n), dev=d, desc=desc)


def card(theta):
    p = np.array([0.95, 0.95, -0.95, -0.95, 0.95, -0.95, -0.95, 0.95, 0.0, 0.5, 0.0, -0.5, 0.5, 0.0,
                  -0.5, 0.0]) * (theta / 2)
    return p[0::2].copy(), p[1::2].copy()


def uvw(rng, theta, lam, dw, nv):
    return (rng.uniform(-theta * lam / 2, theta * lam / 2, nv),
            rng.uniform(-theta * lam / 2, theta * lam / 2, nv), rng.uniform(-dw, dw, nv))


def params(k, theta, lam):
    h = k["host"]
    return rgamd.wstack_params(theta, lam, h["uv"].du, h["w"].dw, h["lm"].x0, h["uv"].size,
                               h["w"].size)


@pytest.mark.parametrize("lam,sky", [(640.0, "card"), (2560.0, "random"), (1280.0, "many")])
def test_predict_matches_oracle(ctx, kernels, lam, sky):
    """Skies of up to 64 sources transform their source rows only and sum
    the columns directly; larger ones (here 100 sources) run the 2-D FFT."""
    theta = 0.1
    h, d = kernels["host"], kernels["desc"]
    rng = np.random.default_rng(21)
    if sky == "card":
        l, m = card(theta)
        flux = None
    else:
        ns = 40 if sky == "random" else 100
        l = rng.uniform(-0.45 * theta, 0.45 * theta, ns)
        m = rng.uniform(-0.45 * theta, 0.45 * theta, ns)
        flux = rng.uniform(0.1, 1.0, ns)
    u, v, w = uvw(rng, theta, lam, h["w"].dw, 20000)
    stack, skipped = orc.wstack_build(theta, lam, l, m, flux, h["uv"].du, h["w"].dw, h["w"].size,
                                      h["lm"].x0, h["lm"].data, h["n"].data)
    g = int(np.floor(theta * lam))
    ref, nd = orc.wstack_degrid(stack, g, u, v, w, h["uv"].du, h["w"].dw, h["uv"].data,
                                h["uv"].size, h["uv"].oversampling, h["w"].data, h["w"].size,
                                h["w"].oversampling)
    assert skipped == 0 and nd == 0
    p = params(kernels, theta, lam)
    out = torch.empty(len(u), dtype=torch.complex128, device="cuda")
    og, wp, sk = ctx.wstack_build(p, dev(l), dev(m), None if flux is None else dev(flux), d["lm"],
                                  d["n"])
    assert (og, wp, sk) == (stack.shape[1], stack.shape[0], 0)
    gs = ctx.wstack_stack(og, wp)
    assert np.abs(gs - stack).max() < 1e-11 * np.abs(stack).max()
    ctx.wstack_degrid(p, dev(u), dev(v), dev(w), d["uv"], d["w"], out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.abs(got - ref).max() < 1e-10 * np.abs(ref).max()
    st = ctx.stats()
    assert st.n_vis == len(u) and st.n_dropped == 0 and st.n_gridded == len(u)


def test_reference_geometry_matches_the_quantised_sum(ctx, kernels):
    """test/test_wstack.cpp:56-141 at its own geometry (4096^2 x 8 planes),
    1 M random visibilities; checked against the direct sum on 20 000 of
    them (the method's error is about 5e-4 per unit source)."""
    theta, lam = 0.1, 20480.0
    h, d = kernels["host"], kernels["desc"]
    l, m = card(theta)
    rng = np.random.default_rng(22)
    nv = 1_000_000
    u, v, w = uvw(rng, theta, lam, h["w"].dw, nv)
    out = torch.empty(nv, dtype=torch.complex128, device="cuda")
    p = params(kernels, theta, lam)
    ctx.wstack_predict(p, dev(l), dev(m), None, dev(u), dev(v), dev(w), d["uv"], d["w"], d["lm"],
                       d["n"], out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    sel = rng.choice(nv, 20000, replace=False)
    ref = orc.predict_quantized(l, m, None, theta, lam, u[sel], v[sel], w[sel])
    err = np.abs(got[sel] - ref)
    assert err.max() < 1e-3 * len(l), err.max()
    assert err.mean() < 4e-4 * len(l), err.mean()
    assert ctx.stats().n_dropped == 0


def test_outside_visibilities_and_points_are_counted(ctx, kernels):
    theta, lam = 0.1, 640.0
    d = kernels["desc"]
    p = params(kernels, theta, lam)
    l = np.array([0.0, 0.2, 0.01])
    m = np.array([0.0, 0.0, np.nan])
    og, wp, sk = ctx.wstack_build(p, dev(l), dev(m), None, d["lm"], d["n"])
    assert sk == 2
    u = np.array([0.0, 1e6, 0.0, np.nan, 1.0])
    v = np.zeros(5)
    w = np.array([0.0, 0.0, 1e4, 0.0, -3.0])
    out = torch.full((5,), 7.0, dtype=torch.complex128, device="cuda")
    ctx.wstack_degrid(p, dev(u), dev(v), dev(w), d["uv"], d["w"], out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert got[0] != 0 and got[4] != 0 and np.all(got[1:4] == 0)
    st = ctx.stats()
    assert st.n_dropped == 3 and st.n_gridded == 2


def test_invalid_parameters_are_rejected(ctx, kernels):
    d = kernels["desc"]
    p = params(kernels, 0.1, 640.0)
    p.aa_support_uv = 7
    e = torch.zeros(1, dtype=torch.float64, device="cuda")
    with pytest.raises(rgamd.RGError):
        ctx.wstack_build(p, e, e, None, d["lm"], d["n"])
    p = params(kernels, 0.1, 600.0)  # og = 120 is no power of two
    with pytest.raises(rgamd.RGError):
        ctx.wstack_build(p, e, e, None, d["lm"], d["n"])


def test_cli_reports_the_aggregate_error():
    """wstack.out (src/wstack/wstack.cpp) in predict mode with the reference's
    kernel files: random visibilities (seeded) and a fixed (pu, pv, pw)."""
    exe = os.path.join(os.path.dirname(SZE), "..", "..", "radio-gridders_amd", "wstack.out")
    base = [exe, "-theta=0.1", "-lambda=20480", "-mode=0", "-cuda=1",
            f"-sepkern_uv={SZE}/sepkern_uv_transpose.hdf5", f"-sepkern_w={SZE}/sepkern_w_transpose.hdf5",
            f"-sepkern_lm={SZE}/sepkern_lm.hdf5", f"-sepkern_n={SZE}/sepkern_n.hdf5"]
    r = subprocess.run(base + ["-npts=200000", "-random_points=1", "-seed=4"], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    per = float(re.search(r"Aggregate Error / Npts: (\S+)", r.stdout).group(1))
    assert 0 < per < 8 * 4e-4, r.stdout
    r = subprocess.run(base + ["-npts=16", "-pu=100.3", "-pv=-250.7", "-pw=12.5"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    per = float(re.search(r"Aggregate Error / Npts: (\S+)", r.stdout).group(1))
    assert per < 8 * 1e-3, r.stdout


def test_other_supports_match_oracle(ctx, kernels):
    """Supports other than the reference's 8 x 4 (here 4 x 2 and 16 x 4, with
    synthetic positive kernel tables) run the generic degridding kernel."""
    theta, lam = 0.1, 1280.0
    h, d = kernels["host"], kernels["desc"]
    rng = np.random.default_rng(31)
    l, m = card(theta)
    for auv, aw in ((4, 2), (16, 4)):
        ov = 64
        cuv = rng.uniform(0.1, 1.0, auv * ov)
        cw = rng.uniform(0.1, 1.0, aw * ov)
        u, v, w = uvw(rng, theta, lam, h["w"].dw, 5000)
        stack, _ = orc.wstack_build(theta, lam, l, m, None, h["uv"].du, h["w"].dw, aw, h["lm"].x0,
                                    h["lm"].data, h["n"].data)
        g = int(np.floor(theta * lam))
        ref, nd = orc.wstack_degrid(stack, g, u, v, w, h["uv"].du, h["w"].dw, cuv, auv, ov, cw,
                                    aw, ov)
        p = rgamd.wstack_params(theta, lam, h["uv"].du, h["w"].dw, h["lm"].x0, auv, aw)
        ctx.wstack_build(p, dev(l), dev(m), None, d["lm"], d["n"])
        duv, dw_ = dev(cuv), dev(cw)
        out = torch.empty(len(u), dtype=torch.complex128, device="cuda")
        ctx.wstack_degrid(p, dev(u), dev(v), dev(w), rgamd.sep_kern_desc(duv, auv, ov),
                          rgamd.sep_kern_desc(dw_, aw, ov), out)
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.abs(got - ref).max() < 1e-10 * np.abs(ref).max(), (auv, aw)
        assert ctx.stats().n_dropped == nd


@pytest.mark.parametrize("layout", ["sparse", "concentrated"])
def test_sort_handles_sparse_and_concentrated_streams(ctx, kernels, layout):
    """The degridding sort at a 1024^2 stack (24 576 (tile, plane) keys):
    a few visibilities spread over the whole stack (chunks of the bucketed
    records span more keys than the LDS window and rank with device atomics),
    and one (u, v, w) repeated 50 000 times (every chunk reserves its share of
    the same key)."""
    theta, lam = 0.1, 5120.0
    h, d = kernels["host"], kernels["desc"]
    rng = np.random.default_rng(41)
    l, m = card(theta)
    g = int(np.floor(theta * lam))
    reach = (g - h["uv"].size // 2 - 1) * h["uv"].du
    if layout == "sparse":
        nv = 6000
        u = rng.uniform(-reach, reach, nv)
        v = rng.uniform(-reach, reach, nv)
        w = rng.uniform(-h["w"].dw, h["w"].dw, nv)
    else:
        nv = 50000
        u, v, w = np.full(nv, 123.4), np.full(nv, -77.7), np.full(nv, 12.5)
    stack, skipped = orc.wstack_build(theta, lam, l, m, None, h["uv"].du, h["w"].dw, h["w"].size,
                                      h["lm"].x0, h["lm"].data, h["n"].data)
    sel = slice(None) if layout == "sparse" else slice(0, 1)
    ref, nd = orc.wstack_degrid(stack, g, u[sel], v[sel], w[sel], h["uv"].du, h["w"].dw,
                                h["uv"].data, h["uv"].size, h["uv"].oversampling, h["w"].data,
                                h["w"].size, h["w"].oversampling)
    assert skipped == 0 and nd == 0
    p = params(kernels, theta, lam)
    ctx.wstack_build(p, dev(l), dev(m), None, d["lm"], d["n"])
    out = torch.empty(nv, dtype=torch.complex128, device="cuda")
    ctx.wstack_degrid(p, dev(u), dev(v), dev(w), d["uv"], d["w"], out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    if layout == "concentrated":
        ref = np.full(nv, ref[0])
    assert np.abs(got - ref).max() < 1e-10 * np.abs(ref).max()
    st = ctx.stats()
    assert st.n_vis == nv and st.n_dropped == 0 and st.n_gridded == nv


def test_empty_and_all_dropped_streams(ctx, kernels):
    """No visibilities, and visibilities that all leave the stack: the sort
    sees no records (empty buckets, no work items) and every output is 0."""
    theta, lam = 0.1, 640.0
    d = kernels["desc"]
    p = params(kernels, theta, lam)
    l, m = card(theta)
    ctx.wstack_build(p, dev(l), dev(m), None, d["lm"], d["n"])
    e = torch.zeros(0, dtype=torch.float64, device="cuda")
    out0 = torch.zeros(0, dtype=torch.complex128, device="cuda")
    ctx.wstack_degrid(p, e, e, e, d["uv"], d["w"], out0)
    torch.cuda.synchronize()
    assert ctx.stats().n_vis == 0 and ctx.stats().n_gridded == 0
    nv = 3000
    u = np.full(nv, 1e7)
    out = torch.full((nv,), 5.0, dtype=torch.complex128, device="cuda")
    ctx.wstack_degrid(p, dev(u), dev(np.zeros(nv)), dev(np.zeros(nv)), d["uv"], d["w"], out)
    torch.cuda.synchronize()
    assert torch.all(out == 0)
    st = ctx.stats()
    assert st.n_vis == nv and st.n_dropped == nv and st.n_gridded == 0


@pytest.mark.parametrize("lam", [5120.0, 10240.0])
def test_dense_sky_with_long_rows(ctx, kernels, lam):
    """More sources than the sparse form takes, on planes of 1024 and 2048: the
    row pass of long lines skips the rows without a source."""
    theta = 0.1
    h, d = kernels["host"], kernels["desc"]
    rng = np.random.default_rng(31)
    ns = 90
    l = rng.uniform(-0.45 * theta, 0.45 * theta, ns)
    m = rng.uniform(-0.1 * theta, 0.1 * theta, ns)
    flux = rng.uniform(0.1, 1.0, ns)
    stack, _ = orc.wstack_build(theta, lam, l, m, flux, h["uv"].du, h["w"].dw, h["w"].size,
                                h["lm"].x0, h["lm"].data, h["n"].data)
    og, wp, _ = ctx.wstack_build(params(kernels, theta, lam), dev(l), dev(m), dev(flux), d["lm"],
                                 d["n"])
    assert (og, wp) == (stack.shape[1], stack.shape[0])
    assert np.abs(ctx.wstack_stack(og, wp) - stack).max() < 1e-11 * np.abs(stack).max()


@pytest.mark.parametrize("per_tile", [1536, 1537, 3071, 3072, 3073, 4609, 8193, 16385])
def test_dense_keys_at_their_edges(ctx, kernels, per_tile):
    """Visibilities of one (16 x 16-cell tile, plane) key around the sizes where
    it becomes dense and where it is split into work items: spread over the
    tile's cells, with a full batch and a batch of one in two of them, next to a
    key of a few visibilities, a key of one cell only and visibilities that leave
    the stack (0), in random order.  Results are sums of 256 products of at most
    |stack| sum |taps| each, so FP64 agrees far below 1e-10."""
    theta, lam = 0.1, 640.0
    h, d = kernels["host"], kernels["desc"]
    rng = np.random.default_rng(per_tile)
    du, dw = h["uv"].du, h["w"].dw
    l, m = card(theta)
    g = int(np.floor(theta * lam))
    def at(cell):  # a coordinate whose centre tap is `cell` of the stack
        return (cell - g - rng.uniform(0.01, 0.99, len(cell))) * du

    base = 64  # a tile's first cell
    cu, cv = rng.integers(base, base + 16, (2, per_tile))
    cu[:33], cv[:33] = base + 3, base + 5  # two full batches and more
    dense = at(cu), at(cv)
    cu, cv = base + 16 + rng.integers(0, 16, 40), np.full(40, base + 2)
    sparse = at(cu), at(cv)
    one = at(np.full(4500, base + 7)), at(np.full(4500, base + 24))
    gone = np.full(19, 1e7), np.zeros(19)
    u, v = (np.concatenate([a[k] for a in (dense, sparse, one, gone)]) for k in (0, 1))
    w = -rng.uniform(0.01, 0.99, len(u)) * dw
    order = rng.permutation(len(u))
    u, v, w = u[order], v[order], w[order]
    stack, _ = orc.wstack_build(theta, lam, l, m, None, du, dw, h["w"].size, h["lm"].x0,
                                h["lm"].data, h["n"].data)
    ref, nd = orc.wstack_degrid(stack, g, u, v, w, du, dw, h["uv"].data, h["uv"].size,
                                h["uv"].oversampling, h["w"].data, h["w"].size,
                                h["w"].oversampling)
    assert nd == 19
    p = params(kernels, theta, lam)
    ctx.wstack_build(p, dev(l), dev(m), None, d["lm"], d["n"])
    out = torch.full((len(u),), 5.0, dtype=torch.complex128, device="cuda")
    ctx.wstack_degrid(p, dev(u), dev(v), dev(w), d["uv"], d["w"], out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.abs(got - ref).max() < 1e-10 * np.abs(ref).max()
    assert np.all(got[order >= len(order) - 19] == 0)
    st = ctx.stats()
    assert st.n_dropped == 19 and st.n_gridded == len(u) - 19


def test_shorter_prediction_on_a_frozen_context(kernels):
    """A prediction sized the scratch, a captured gridding call holds it: shorter predictions, one of
    which the sort cuts into more workgroups (1 090 000 into 355, 1 040 000 into 508)."""
    theta, lam = 0.1, 640.0
    h, d = kernels["host"], kernels["desc"]
    rng = np.random.default_rng(3)
    c = rgamd.Context(0)
    p = params(kernels, theta, lam)
    l, m = card(theta)
    c.wstack_build(p, dev(l), dev(m), None, d["lm"], d["n"])
    n = 1_090_000
    u, v, w = (dev(a) for a in uvw(rng, theta, lam, h["w"].dw, n))
    out = torch.empty(n, dtype=torch.complex128, device="cuda")
    c.wstack_degrid(p, u, v, w, d["uv"], d["w"], out)
    want = out.clone()
    k = torch.randn((1, 4, 4, 8, 8), dtype=torch.complex128, device="cuda")
    g = torch.empty((128, 128), dtype=torch.complex128, device="cuda")
    fv = rgamd.flat_vis(u[:5000], v[:5000], w[:5000], want[:5000])
    for _ in range(2):
        c.grid(rgamd.params(128, theta), fv, rgamd.wkern_desc(k, 0.0, 1e9), g)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c.grid(rgamd.params(128, theta), fv, rgamd.wkern_desc(k, 0.0, 1e9), g)
    for n1 in (1_040_000, n, 3000):
        out.zero_()
        c.wstack_degrid(p, u[:n1], v[:n1], w[:n1], d["uv"], d["w"], out[:n1])
        torch.cuda.synchronize()
        assert float((out[:n1] - want[:n1]).abs().max()) <= 1e-12 * float(want.abs().max()), n1
    del graph
    c.close()


# visibilities beside a test's own, on another plane, so that the stream is long enough for
# kernels of dense keys (2^20)
LONG = 1 << 20


def with_filler(rng, theta, lam, dw, u, v, w):
    k = LONG - len(u)
    fu, fv, _ = uvw(rng, theta, lam, dw, k)
    return (np.concatenate([u, fu]), np.concatenate([v, fv]),
            np.concatenate([w, rng.uniform(0.01, 0.99, k) * dw]))


@pytest.mark.parametrize("copies,long", [(3073, False), (6145, False), (3071, True), (3072, True),
                                         (4097, True), (20_481, True)])
def test_every_part_of_a_dense_key_is_predicted_once(ctx, kernels, copies, long):
    """Copies of one visibility: one kernel takes every part of its key.  The weights along u are
    scaled by 1e180, those along v and w by 1e-180: the sparse keys' kernel multiplies by v and w
    first, which underflows to 0, the dense ones' by u and w, which does not, so that a part
    that both have computed shows the last one's 0."""
    theta, lam = 0.1, 640.0
    h, d = kernels["host"], kernels["desc"]
    rng = np.random.default_rng(11)
    l = rng.uniform(-0.45 * theta, 0.45 * theta, 40)
    m = rng.uniform(-0.45 * theta, 0.45 * theta, 40)
    p = params(kernels, theta, lam)
    ctx.wstack_build(p, dev(l), dev(m), None, d["lm"], d["n"])
    uv, kw = kernels["dev"]["uv"].clone().reshape(-1), kernels["dev"]["w"] * 1e-180
    half = h["uv"].size * (h["uv"].oversampling // 2)
    uv[:half] *= 1e180
    uv[half:] *= 1e-180
    du = h["uv"].du
    u, v, w = (np.full(copies, x) for x in (2.75 * du, 2.25 * du, -0.3 * h["w"].dw))
    if long:
        u, v, w = with_filler(rng, theta, lam, h["w"].dw, u, v, w)
    out = torch.empty(len(u), dtype=torch.complex128, device="cuda")
    ctx.wstack_degrid(p, dev(u), dev(v), dev(w),
                      rgamd.sep_kern_desc(uv, h["uv"].size, h["uv"].oversampling),
                      rgamd.sep_kern_desc(kw, h["w"].size, h["w"].oversampling), out)
    torch.cuda.synchronize()
    out = out[:copies]
    assert bool(out[0]) == (long and copies >= 3072)
    assert float((out - out[0]).abs().max()) <= 1e-13 * float(out[0].abs())


@pytest.mark.parametrize("per_tile", [3071, 3072, 4095, 4097, 8191, 8193, 20_481])
def test_dense_keys_of_a_long_stream(ctx, kernels, per_tile):
    """One (16 x 16-cell tile, plane) key around the sizes where it becomes dense and where it is
    split into parts (4096 records, a 256th of the stream), with two full batches and one visibility more in one
    of its cells, and a key of one cell only; the rest of the stream on the next plane, about
    3 k to 16 k a key.  Sums of 256 products of at most |stack| sum |taps| each."""
    theta, lam = 0.1, 640.0
    h, d = kernels["host"], kernels["desc"]
    rng = np.random.default_rng(per_tile)
    du, dw = h["uv"].du, h["w"].dw
    l, m = card(theta)
    g = int(np.floor(theta * lam))

    def at(cell):  # a coordinate whose centre tap is `cell` of the stack
        return (cell - g - rng.uniform(0.01, 0.99, len(cell))) * du

    cu, cv = 64 + rng.integers(0, 16, (2, per_tile))
    cu[:33], cv[:33] = 67, 69
    u = np.concatenate([at(cu), at(np.full(4500, 71))])
    v = np.concatenate([at(cv), at(np.full(4500, 88))])
    w = -rng.uniform(0.01, 0.99, len(u)) * dw
    u, v, w = with_filler(rng, theta, lam, dw, u, v, w)
    order = rng.permutation(len(u))
    u, v, w = u[order], v[order], w[order]
    stack, _ = orc.wstack_build(theta, lam, l, m, None, du, dw, h["w"].size, h["lm"].x0,
                                h["lm"].data, h["n"].data)
    ref, _ = orc.wstack_degrid(stack, g, u, v, w, du, dw, h["uv"].data, h["uv"].size,
                               h["uv"].oversampling, h["w"].data, h["w"].size,
                               h["w"].oversampling)
    p = params(kernels, theta, lam)
    ctx.wstack_build(p, dev(l), dev(m), None, d["lm"], d["n"])
    out = torch.full((len(u),), 5.0, dtype=torch.complex128, device="cuda")
    ctx.wstack_degrid(p, dev(u), dev(v), dev(w), d["uv"], d["w"], out)
    torch.cuda.synchronize()
    assert np.abs(out.cpu().numpy() - ref).max() < 1e-10 * np.abs(ref).max()
    assert ctx.stats().n_dropped == 0
