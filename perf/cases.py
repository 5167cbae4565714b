"""Timing cases of the gridding engine: what a user's program has it do,
through the Python binding of librg, from a few hundred visibilities to tens
of millions.

Observations are Earth-rotation tracks of a random station layout (dec -30
deg, 4 h, 150 MHz; radii Exp(0.6 R) cut at R, R = 0.244 lambda metres, so that
every baseline fits the 10 km of a 20 480-wavelength field), 10 to 50 point
sources, W-kernels of support S and oversampling R sampled from a prolate
taper.  All inputs follow from the seed; the sizes are those of the
repository's benchmark workloads and tests.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "radio-gridders_amd"))

import rgamd  # noqa: E402

WAVELENGTH = 299792458.0 / 150e6
LAT, DEC = math.radians(-26.7), math.radians(-30.0)
W_STEP = 10.0  # W-projection plane spacing
WINC = 10.0    # W-towers floor spacing; its kernel planes are 1 wavelength apart


def listed():
    return [
        # one short snapshot on a test-sized grid: launches and latency are all there is
        dict(name="wproj_8st_fp64", kind="wproj", st=8, dumps=16, theta=0.1, n=128, s=16, r=8,
             fp=64, tile=0),
        # the whole CPU-convention image of a 27-station observation (uniform weights, FP64
        # gridding, hermitian completion, transform, taper): what grid.out -cpu_image computes
        dict(name="cpu_image_27st", kind="cpu_image", st=27, dumps=256, theta=0.1, n=2048, s=16,
             r=8, fp=64, tile=0),
        # an ordinary FP64 W-projection call
        dict(name="wproj_128st_fp64", kind="wproj", st=128, dumps=64, theta=0.1, n=1024, s=16, r=8,
             fp=64, tile=0),
        # the 512-station stream through W-projection in single precision (tuned tile)
        dict(name="wproj_512st_fp32", kind="wproj", st=512, dumps=64, theta=0.1, n=2048, s=16, r=8,
             fp=32, tile=48),
        # many channels with uneven counts in one call
        dict(name="channels_64", kind="channels", st=256, dumps=64, chan=64, median=40000,
             theta=0.05, n=1024, s=16, r=8, fp=32, tile=0),
        # a small array through W-towers, support-8 kernels
        dict(name="wtowers_27st_fp32", kind="wtowers", st=27, dumps=64, theta=0.1, n=1024, s=8, r=8,
             fp=32, sub=128, margin=16),
        # W-towers in double precision, the accuracy choice
        dict(name="wtowers_128st_fp64", kind="wtowers", st=128, dumps=64, theta=0.1, n=1024, s=16,
             r=8, fp=64, sub=256, margin=16),
        # the headline workload: 512 stations, 2048^2 grid, subgrid 512
        dict(name="wtowers_512st_fp32", kind="wtowers", st=512, dumps=64, theta=0.1, n=2048, s=16,
             r=8, fp=32, sub=512, margin=16),
        # the direct DFT that checks an image: 65 536 sampled pixels of the 2048^2 field
        dict(name="dft_65536px", kind="dft", nvis=262144, px=65536, image=False, theta=0.1, n=2048),
        # the final transform of a large grid
        dict(name="to_image_4096", kind="to_image", n=4096, fp=64, width=0.2),
        # W-stacking predict at the reference test's workload
        dict(name="wstack_40M", kind="wstack", nvis=40_000_000, src=8, lam=20480.0, theta=0.1),
        # EPIC imaging at the reference's workload
        dict(name="epic_1000x256", kind="epic", nb=1000, ant=256, g=64, supp=2),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["wproj", "wproj", "wproj", "cpu_image", "channels", "wtowers", "wtowers",
                       "wtowers", "dft", "dft", "to_image", "wstack", "epic", "epic"])
    c = dict(kind=kind)
    if kind in ("wproj", "cpu_image"):
        c.update(st=_logint(rng, 8, 300), dumps=_logint(rng, 7, 128),
                 theta=rng.choice([0.05, 0.1]),
                 n=2 * _logint(rng, 50, 1024) if kind == "wproj" else rng.choice([256, 512, 1024,
                                                                                  2048]),
                 s=rng.choice([8, 16, 16]), r=rng.choice([4, 8, 8]),
                 fp=64 if kind == "cpu_image" else rng.choice([32, 32, 64]),
                 tile=rng.choice([0, 32, 48]))
    elif kind == "channels":
        c.update(st=_logint(rng, 16, 200), dumps=_logint(rng, 9, 64), chan=_logint(rng, 2, 96),
                 median=_logint(rng, 300, 30000), theta=0.05, n=rng.choice([256, 500, 1024]),
                 s=rng.choice([8, 16]), r=8, fp=rng.choice([32, 64]), tile=0)
    elif kind == "wtowers":
        sub = rng.choice([64, 128, 256, 512])
        c.update(st=_logint(rng, 8, 256), dumps=_logint(rng, 7, 64), theta=0.1,
                 n=sub * rng.choice([1, 2, 3, 4, 4] if sub > 128 else [2, 3, 4, 8]),
                 s=rng.choice([8, 16]), r=8, fp=rng.choice([32, 32, 64]), sub=sub,
                 margin=rng.choice([16, 16, 24, 32]))
    elif kind == "dft":
        image = rng.random() < 0.4
        n = rng.choice([64, 100, 128, 256]) if image else rng.choice([512, 1024, 2048])
        px = n * n if image else _logint(rng, 100, 65536)
        c.update(nvis=_logint(rng, 500, min(2_000_000, 16_000_000_000 // px)), px=px, image=image,
                 theta=rng.choice([0.05, 0.1]), n=n)
    elif kind == "to_image":
        c.update(n=rng.choice([64, 128, 256, 512, 1024, 2048, 4096]), fp=rng.choice([32, 64]),
                 width=round(rng.uniform(0.05, 0.4), 3))
    elif kind == "wstack":
        c.update(nvis=_logint(rng, 10_000, 20_000_000), src=_logint(rng, 1, 300),
                 lam=rng.choice([640.0, 2560.0, 5120.0, 10240.0, 20480.0]), theta=0.1)
    else:
        g = rng.choice([32, 64, 90, 128, 200, 256])
        c.update(nb=_logint(rng, 4, min(2000, 8_000_000 // (g * g))), ant=_logint(rng, 16, 512),
                 g=g, supp=rng.choice([1, 2, 3, 4, 8]))
    return c


# ---- inputs -----------------------------------------------------------------------------------

def _tracks(c, rng, dev):
    """u, v, w in wavelengths, baseline -> time order."""
    lam = c["n"] / c["theta"]
    rmax = 0.244 * lam * WAVELENGTH / 2.0
    rad = -0.6 * rmax * np.log(1.0 - rng.random(c["st"]) * (1.0 - math.exp(-1 / 0.6)))
    ang = rng.uniform(0.0, 2 * math.pi, c["st"])
    pos = torch.from_numpy(np.stack([rad * np.cos(ang), rad * np.sin(ang)], 1)).to(dev)
    i, j = torch.triu_indices(c["st"], c["st"], 1, device=dev)
    e, nn = (pos[j] - pos[i]).T[:, :, None]
    x, z = -math.sin(LAT) * nn, math.cos(LAT) * nn
    ha = torch.linspace(-math.pi / 6, math.pi / 6, c["dumps"], dtype=torch.float64, device=dev)
    sh, ch, sd, cd = torch.sin(ha), torch.cos(ha), math.sin(DEC), math.cos(DEC)
    u = sh * x + ch * e
    v = -sd * ch * x + sd * sh * e + cd * z
    w = cd * ch * x - cd * sh * e + sd * z
    return [(t / WAVELENGTH).reshape(-1).contiguous() for t in (u, v, w)]


def _w_range(c):
    """Largest |w| of the tracks (0.46 of the longest baseline, at 200 MHz for channels)."""
    return 0.46 * 0.244 * c["n"] / c["theta"] * (1.34 if c["kind"] == "channels" else 1.0)


def _predict(u, v, w, rng, nsrc, theta):
    vis = torch.zeros(u.numel(), dtype=torch.complex128, device=u.device)
    for l, m, f in zip(rng.uniform(-theta / 2, theta / 2, nsrc), rng.uniform(-theta / 2, theta / 2,
                                                                             nsrc),
                       rng.uniform(0.1, 1.0, nsrc)):
        ph = u * l + v * m + w * (math.sqrt(1 - l * l - m * m) - 1)
        ph -= torch.round(ph)
        vis += torch.polar(torch.full_like(ph, f), -2 * math.pi * ph)
    return vis


def _table(c, w_min, w_step, planes, dev):
    """W-kernel table [P][R][R][S][S], complex128."""
    s, r, m, theta = c["s"], c["r"], 128, c["theta"]
    xs = (np.arange(m) + 0.5 - 0.5 * m) / m
    taper = torch.from_numpy(rgamd.pswf_eval(math.pi * s / 4, 2 * xs)).to(dev)
    d = (np.arange(s) - s // 2)[None, :] - np.arange(r)[:, None] / r
    ph = torch.from_numpy(2 * math.pi * d.reshape(-1, 1) * xs[None, :]).to(dev)
    e = torch.polar(torch.ones_like(ph), ph)  # [R S][M]
    l2 = torch.from_numpy((theta * xs) ** 2).to(dev)
    nn = torch.sqrt(1 - l2[:, None] - l2[None, :]) - 1
    amp = taper[:, None] * taper[None, :] / (m * m)
    out = torch.empty((planes, r, r, s, s), dtype=torch.complex128, device=dev)
    for p in range(planes):
        ph = nn * (-2 * math.pi * (w_min + p * w_step))
        k = torch.mm(torch.mm(e, torch.polar(torch.ones_like(ph), ph) * amp), e.T.contiguous())
        out[p] = k.reshape(r, s, r, s).permute(0, 2, 1, 3)
    return out


_tables = {}


def _kernels(c, dev="cuda"):
    """(table, w_min, w_step): it depends on the geometry alone, so programs keep it."""
    if c["kind"] == "wtowers":
        w_min, step, planes = -WINC / 2, 1.0, int(WINC) + 1
    else:
        half = math.ceil(_w_range(c) / W_STEP) + 1
        w_min, step, planes = -half * W_STEP, W_STEP, 2 * half + 1
    key = (c["s"], c["r"], c["theta"], w_min, step, planes)
    if key not in _tables:
        _tables.clear()  # one geometry at a time
        _tables[key] = _table(c, w_min, step, planes, dev)
    return _tables[key], w_min, step


def _inputs(c, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def rand(n):
        return torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)

    kind = c["kind"]
    d = {}
    if kind in ("wproj", "cpu_image", "wtowers", "channels"):
        u, v, w = _tracks(c, rng, "cuda")
        if kind == "channels":
            # channel c keeps round(LogNormal(ln median, 1)) of the samples, in track order
            freq = np.linspace(100e6, 200e6, c["chan"]) / 150e6
            cnt = np.rint(rng.lognormal(math.log(c["median"]), 1.0, c["chan"])).astype(np.int64)
            cnt = np.minimum(cnt, u.numel())
            # the same total for every seed
            total = _channel_total(c)
            cnt = np.minimum(np.maximum((cnt * (total / cnt.sum())).astype(np.int64), 1), u.numel())
            us, vs, ws = [], [], []
            for f, k in zip(freq, cnt):
                pick = torch.randperm(u.numel(), device="cuda", generator=gen)[:int(k)].sort()[0]
                us.append(u[pick] * f)
                vs.append(v[pick] * f)
                ws.append(w[pick] * f)
            u, v, w = torch.cat(us), torch.cat(vs), torch.cat(ws)
            d["off"] = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
        d["u"], d["v"], d["w"] = u, v, w
        d["vis"] = _predict(u, v, w, rng, 50 if c["st"] > 256 else 10, c["theta"])
        if c["fp"] == 32:
            d["vis"] = d["vis"].to(torch.complex64)
    elif kind == "dft":
        lam = c["n"] / c["theta"]
        # tracks, then a random sample of them in stream order
        st = max(8, int(math.sqrt(2 * c["nvis"] / 16)) + 2)
        u, v, w = _tracks(dict(c, st=st, dumps=16), rng, "cuda")
        pick = torch.randperm(u.numel(), device="cuda", generator=gen)[:c["nvis"]].sort()[0]
        d["u"], d["v"], d["w"] = u[pick], v[pick], w[pick]
        d["vis"] = _predict(d["u"], d["v"], d["w"], rng, 10, c["theta"])
        d["lam"] = lam
        if not c["image"]:
            px = torch.randperm(c["n"] * c["n"], device="cuda", generator=gen)[:c["px"]]
            d["px"] = (px % c["n"]).to(torch.int32)
            d["py"] = (px // c["n"]).to(torch.int32)
    elif kind == "to_image":
        g = torch.randn((c["n"], c["n"]), dtype=torch.complex128, device="cuda", generator=gen)
        r = torch.arange(c["n"], device="cuda", dtype=torch.float64) - c["n"] / 2
        g *= torch.exp(-(r[:, None] ** 2 + r[None, :] ** 2) / (c["width"] * c["n"]) ** 2)
        d["grid"] = g.to(torch.complex64) if c["fp"] == 32 else g
    elif kind == "wstack":
        th, lam = c["theta"], c["lam"]
        d["u"] = (rand(c["nvis"]) - 0.5) * (th * lam)
        d["v"] = (rand(c["nvis"]) - 0.5) * (th * lam)
        d["w"] = (rand(c["nvis"]) * 2 - 1) * WS_DW
        d["l"] = torch.from_numpy(rng.uniform(-0.45 * th, 0.45 * th, c["src"])).cuda()
        d["m"] = torch.from_numpy(rng.uniform(-0.45 * th, 0.45 * th, c["src"])).cuda()
        d["flux"] = torch.from_numpy(rng.uniform(0.1, 1.0, c["src"])).cuda()
    else:
        nb, na, g, s = c["nb"], c["ant"], c["g"], c["supp"]
        d["f"] = 5 * torch.randn((nb, na), dtype=torch.complex64, device="cuda", generator=gen)
        # antennas stand still: one layout for every timestamp
        x = torch.randint(s, g - s + 1, (na,), device="cuda", generator=gen, dtype=torch.int32)
        y = torch.randint(s, g - s + 1, (na,), device="cuda", generator=gen, dtype=torch.int32)
        d["x"] = x.repeat(nb, 1).contiguous()
        d["y"] = y.repeat(nb, 1).contiguous()
        d["illum"] = torch.randn((s, s), dtype=torch.complex64, device="cuda", generator=gen)
    return d


def _channel_total(c):
    """Visibilities of a channels case (the mean of LogNormal(ln median, 1) per channel)."""
    return int(c["chan"] * min(c["median"] * math.exp(0.5), c["st"] * (c["st"] - 1) / 2 *
                               c["dumps"] * 0.5))


# separable kernels of W-stacking in the layout of the reference's files: 8 x 4
# supports, 4096 rows of taps, corrections of 10 001 samples
WS_UV, WS_W, WS_OV, WS_CORR = 8, 4, 4096, 10001
WS_DU, WS_DW, WS_X0 = 5.0, 49.93742167907413, 0.25


def _sep_kernels():
    def conv(size):
        t = (np.arange(size) - size // 2)[None, :] + np.arange(WS_OV)[:, None] / WS_OV
        k = np.i0(2.3 * size * np.sqrt(np.maximum(0.0, 1 - (2 * t / size) ** 2)))
        return (k / k.sum(1).mean()).reshape(-1)

    t = np.linspace(-1, 1, WS_CORR)
    corr = np.maximum(np.cos(0.5 * math.pi * t * 0.9) ** 2, 0.01)
    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in
            (conv(WS_UV), conv(WS_W), corr, 0.2 + 0.8 * corr)]


def _taper(c):
    """Image-plane taper at the pixel positions (kept away from its zeros at the edge)."""
    x = (np.arange(c["n"]) - c["n"] / 2) / (c["n"] / 2)
    return torch.from_numpy(np.maximum(np.cos(0.45 * math.pi * x), 1e-2)).cuda()


def _params(c):
    p = dict(tile=c.get("tile", 0))
    if c["kind"] == "wtowers":
        p.update(subgrid=c["sub"], margin=c["margin"], winc=WINC)
    return rgamd.params(c["n"], c["theta"], rgamd.RG_MODE_BATCHED, **p)


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    kind = c["kind"]
    st = dict(d, case=c, kind=kind, ctx=rgamd.Context(0))
    if kind in ("wproj", "cpu_image", "wtowers", "channels"):
        table, w_min, step = _kernels(c)
        table = table.to(torch.complex64) if c["fp"] == 32 else table.clone()
        st["wk"] = rgamd.wkern_desc(table, w_min, step)
        st["p"] = _params(c)
        n = c["n"]
        gt = torch.complex64 if c["fp"] == 32 and kind != "wtowers" else torch.complex128
        shape = (c["chan"], n, n) if kind == "channels" else (n, n)
        st["grid"] = torch.empty(shape, dtype=gt, device="cuda")
        if kind == "cpu_image":
            st["raw"] = st["vis"].clone()
            st["taper"] = _taper(c)
        st["fv"] = rgamd.flat_vis(st["u"], st["v"], st["w"], st["vis"])
    elif kind == "dft":
        st["fv"] = rgamd.flat_vis(st["u"], st["v"], st["w"], st["vis"])
        st["out"] = torch.empty(c["px"], dtype=torch.complex128, device="cuda")
    elif kind == "to_image":
        st["out"] = torch.empty_like(st["grid"])
    elif kind == "wstack":
        kuv, kw, klm, kn = st["kern"] = _sep_kernels()
        st["d_uv"] = rgamd.sep_kern_desc(kuv, WS_UV, WS_OV)
        st["d_w"] = rgamd.sep_kern_desc(kw, WS_W, WS_OV)
        st["d_lm"] = rgamd.sep_kern_desc(klm, WS_CORR, 1)
        st["d_n"] = rgamd.sep_kern_desc(kn, WS_CORR, 1)
        st["p"] = rgamd.wstack_params(c["theta"], c["lam"], WS_DU, WS_DW, WS_X0, WS_UV, WS_W)
        st["out"] = torch.empty(c["nvis"], dtype=torch.complex128, device="cuda")
    else:
        st["grids"] = torch.empty((c["nb"], c["g"], c["g"]), dtype=torch.complex64, device="cuda")
    return st


def run(state):
    st, ctx, kind = state, state["ctx"], state["kind"]
    if kind in ("wproj", "wtowers"):
        ctx.grid(st["p"], st["fv"], st["wk"], st["grid"])
        return st["grid"]
    if kind == "channels":
        ctx.grid_channels(st["p"], st["fv"], st["off"], st["wk"], st["grid"])
        return st["grid"]
    if kind == "cpu_image":
        c = st["case"]
        st["vis"].copy_(st["raw"])
        ctx.weight(st["u"], st["v"], st["vis"], c["n"], c["theta"])
        ctx.grid(st["p"], st["fv"], st["wk"], st["grid"])
        rgamd.make_hermitian(st["grid"])
        rgamd.fft_shift(st["grid"])
        ctx.fft2d(st["grid"], -1)
        rgamd.fft_shift(st["grid"])
        rgamd.gcf_correct(st["grid"], st["taper"])
        return {"image": st["grid"], "weighted": st["vis"]}
    if kind == "dft":
        c = st["case"]
        if c["image"]:
            ctx.dft_image(st["fv"], c["n"], st["lam"], st["out"], c["n"], c["n"])
        else:
            ctx.dft(st["fv"], st["px"], st["py"], c["n"], st["lam"], st["out"])
        return st["out"]
    if kind == "to_image":
        st["out"].copy_(st["grid"])  # the grid is kept, the image replaces its copy
        ctx.grid_to_image(st["out"])
        return st["out"]
    if kind == "wstack":
        ctx.wstack_predict(st["p"], st["l"], st["m"], st["flux"], st["u"], st["v"], st["w"],
                           st["d_uv"], st["d_w"], st["d_lm"], st["d_n"], st["out"])
        return st["out"]
    ctx.epic_grid(st["f"], st["x"], st["y"], st["illum"], st["grids"])
    return st["grids"]


# ---- what a pass cannot do without --------------------------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    if kind in ("wproj", "cpu_image", "wtowers", "channels"):
        nv = (_channel_total(c) if kind == "channels" else
              c["st"] * (c["st"] - 1) // 2 * c["dumps"])
        z = c["fp"] // 4  # bytes of a complex value
        planes = (int(WINC) + 1 if kind == "wtowers" else
                  2 * (math.ceil(_w_range(c) / W_STEP) + 1) + 1)
        taps = c["s"] ** 2
        table = planes * c["r"] ** 2 * taps * z
        ng = c["n"] ** 2 * c.get("chan", 1)
        gz = 16 if kind in ("wtowers", "cpu_image") or c["fp"] == 64 else 8
        b = nv * (24 + z) + min(table, nv * taps * z) + ng * gz
        f = 8.0 * taps * nv
        if kind == "cpu_image":
            b += nv * z + c["n"] * 8
            f += 5.0 * ng * math.log2(ng)
        if kind == "wtowers":
            # one inverse FFT and screen per occupied (tower, floor), one forward FFT per tower
            n2, towers, tasks = c["sub"] ** 2, *_towers(c)
            f += tasks * (5.0 * n2 * math.log2(n2) + 8 * n2) + towers * 5.0 * n2 * math.log2(n2)
        return dict(bytes=b, flops=f)
    if kind == "dft":
        # phase (3 multiply-adds), reduction, sine and cosine (about 30), complex multiply-add
        return dict(bytes=c["nvis"] * 40 + c["px"] * (16 if c["image"] else 24),
                    flops=44.0 * c["nvis"] * c["px"])
    if kind == "to_image":
        n2, z = c["n"] ** 2, c["fp"] // 4
        return dict(bytes=2 * n2 * z, flops=5.0 * n2 * math.log2(n2))
    if kind == "wstack":
        g, og, wp = _ws_geometry(c)
        return dict(bytes=c["nvis"] * 40 + 16.0 * og * og * wp,
                    flops=c["nvis"] * 4.0 * WS_UV * WS_UV * WS_W +
                    wp * 5.0 * og * og * math.log2(og * og))
    return dict(bytes=c["nb"] * (c["ant"] * 16 + 8 * c["g"] ** 2) + 8 * c["supp"] ** 2,
                flops=8.0 * c["nb"] * c["ant"] * c["supp"] ** 2)


def _towers(c):
    """(occupied towers, occupied (tower, floor) pairs) of one layout, counted on the host."""
    u, v, w = [t.numpy() for t in _tracks(c, np.random.default_rng(0), "cpu")]
    chunk = c["sub"] - c["margin"]
    cc = c["n"] // chunk + 1
    cx = ((np.floor(u * c["theta"] + 0.5) + c["n"] // 2) / chunk).astype(np.int64)
    cy = ((np.floor(v * c["theta"] + 0.5) + c["n"] // 2) / chunk).astype(np.int64)
    t = cy * cc + cx
    wp = np.floor(w / WINC + 0.5).astype(np.int64)
    used = np.zeros((cc * cc, int(wp.max() - wp.min()) + 1), bool)
    used[t, wp - wp.min()] = True
    return int(used.any(1).sum()), int(used.sum())


# ---- 64-bit values --------------------------------------------------------------------------------
# Indices on the host in numpy (each operation rounded as written), values in
# torch complex128.

def _frac(n, s, r, theta, u, du):
    x = theta * (u - du)
    fl = np.floor(x + .5 / r)
    f = np.clip(np.floor((x - fl) * r + .5), 0, r - 1).astype(np.int64)
    return fl.astype(np.int64) + n // 2 - s // 2, f


def _scatter(out, base_rows, gx, gy, n, kidx, table, vis):
    """out (flat, rows of n cells, arrays starting at base_rows rows) += conj(kernel) vis over
    every footprint; visibilities in stretches to bound the temporaries."""
    s = table.shape[-1]
    k = table.reshape(-1, s * s)
    o = torch.view_as_real(out)
    for a in range(0, vis.numel(), 1 << 22):
        sl = slice(a, a + (1 << 22))
        g0, g1, br, kk = gx[sl], gy[sl], base_rows[sl], kidx[sl]
        val = vis[sl]
        for t in range(s * s):
            x, y = g0 + t % s, g1 + t // s
            ok = (x >= 0) & (x < n) & (y >= 0) & (y < n)
            cell = torch.where(ok, (br + y) * n + x, 0)
            add = torch.where(ok, k[kk, t].conj() * val, 0)
            o.index_add_(0, cell, torch.view_as_real(add))


def _exact_grids(c, d, table, w_min, step, vis):
    n, s, r = c["n"], c["s"], c["r"]
    u, v, w = [d[x].cpu().numpy() for x in "uvw"]
    gx, xf = _frac(n, s, r, c["theta"], u, 0.0)
    gy, yf = _frac(n, s, r, c["theta"], v, 0.0)
    p = np.floor((w - w_min) / step + .5).astype(np.int64)
    ok = (p >= 0) & (p < table.shape[0])
    chan = c.get("chan", 1)
    row = np.zeros(len(u), np.int64)
    if chan > 1:
        row = np.repeat(np.arange(chan) * n, np.diff(d["off"]))
    out = torch.zeros(chan * n * n, dtype=torch.complex128, device="cuda")
    dev = [torch.from_numpy(a[ok]).cuda() for a in (row, gx, gy, (p * r + yf) * r + xf)]
    _scatter(out, dev[0], dev[1], dev[2], n, dev[3], table, vis[torch.from_numpy(ok).cuda()])
    return out.reshape((chan, n, n) if chan > 1 else (n, n))


def _exact_towers(c, d, table, w_min, step):
    n, s, r, big, theta = c["sub"], c["s"], c["r"], c["n"], c["theta"]
    chunk = n - c["margin"]
    cc = big // chunk + 1
    u, v, w = [d[x].cpu().numpy() for x in "uvw"]
    cx = ((np.floor(u * theta + 0.5) + big // 2) / chunk).astype(np.int64)
    cy = ((np.floor(v * theta + 0.5) + big // 2) / chunk).astype(np.int64)
    wp = np.floor(w / WINC + 0.5).astype(np.int64)
    gx, xf = _frac(n, s, r, theta, u, (chunk * cx - big // 2 + chunk // 2) / theta)
    gy, yf = _frac(n, s, r, theta, v, (chunk * cy - big // 2 + chunk // 2) / theta)
    p = np.floor((w - wp * WINC - w_min) / step + .5).astype(np.int64)
    ok = (p >= 0) & (p < table.shape[0])
    task, inv = np.unique(((cy * cc + cx) * 100000 + wp + 50000)[ok], return_inverse=True)
    order = np.argsort(inv, kind="stable")
    start = np.concatenate([[0], np.cumsum(np.bincount(inv, minlength=len(task)))])
    cols = [torch.from_numpy(a[ok][order]).cuda() for a in (gx, gy, (p * r + yf) * r + xf)]
    inv = torch.from_numpy(inv[order]).cuda()
    vis = d["vis"].to(torch.complex128)[torch.from_numpy(np.nonzero(ok)[0][order]).cuda()]
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    lm = theta * torch.where(k < n // 2, k, k - n) / n
    base = 1 - torch.sqrt(1 - lm[:, None] ** 2 - lm[None, :] ** 2)
    imgs = {}
    q = max(1, (1 << 27) // (n * n))
    for t0 in range(0, len(task), q):
        t1 = min(len(task), t0 + q)
        a, b = int(start[t0]), int(start[t1])
        sub = torch.zeros((t1 - t0) * n * n, dtype=torch.complex128, device="cuda")
        _scatter(sub, (inv[a:b] - t0) * n, cols[0][a:b], cols[1][a:b], n, cols[2][a:b], table,
                 vis[a:b])
        sub = sub.reshape(-1, n, n)
        for i in range(t0, t1):
            tower, fl = int(task[i]) // 100000, int(task[i]) % 100000 - 50000
            ph = base * (-fl * WINC)
            ph -= torch.round(ph)
            img = torch.fft.ifft2(sub[i - t0]) * torch.polar(torch.ones_like(ph),
                                                             2 * math.pi * ph)
            imgs[tower] = imgs[tower] + img if tower in imgs else img
    out = torch.zeros((big, big), dtype=torch.complex128, device="cuda")
    for tower, img in imgs.items():
        # ifft2 divides by n^2, as the fold does
        uv = torch.fft.fft2(img)
        x0 = chunk * (tower % cc) - c["margin"] // 2
        y0 = chunk * (tower // cc) - c["margin"] // 2
        ya, yb, xa, xb = max(y0, 0), min(y0 + n, big), max(x0, 0), min(x0 + n, big)
        if ya < yb and xa < xb:
            out[ya:yb, xa:xb] += uv[ya - y0:yb - y0, xa - x0:xb - x0]
    return out


def _shift(a):
    return torch.roll(a, (a.shape[0] // 2, a.shape[1] // 2), (0, 1))


def _exact_cpu_image(c, d, table, w_min, step):
    n, theta = c["n"], c["theta"]
    u, v = d["u"].cpu().numpy(), d["v"].cpu().numpy()
    x, y = [np.floor(theta * a + .5).astype(np.int64) + n // 2 for a in (u, v)]
    inside = (x >= 0) & (x < n) & (y >= 0) & (y < n)
    cell = np.where(inside, y * n + x, 0)
    cnt = np.bincount(cell[inside], minlength=n * n)
    wt = np.where(inside, cnt[cell], 1)
    vis = d["vis"] / torch.from_numpy(wt).cuda()
    g = _exact_grids(c, d, table, w_min, step, vis).reshape(-1)
    lo = n + 1 if n % 2 == 0 else 0
    mid = (n + 1) * (n // 2)
    k = torch.arange(mid - lo, device="cuda")
    a, b = g[lo + k].clone(), g[n * n - 1 - k].clone()
    g[lo + k] = a + b.conj()
    g[n * n - 1 - k] = b + a.conj()
    g[mid] += g[mid].conj()
    img = _shift(torch.fft.fft2(_shift(g.reshape(n, n))))
    t = _taper(c)
    return {"image": img / (t[:, None] * t[None, :]), "weighted": vis}


def _exact_dft(c, d):
    n, lam = c["n"], d["lam"]
    if c["image"]:
        i = np.arange(n * n)
        px, py = i % n, i // n
    else:
        px, py = d["px"].cpu().numpy(), d["py"].cpu().numpy()
    l, m = (py - n // 2) / lam, (px - n // 2) / lam
    nn = 1 - np.sqrt(1 - l * l - m * m)
    l, m, nn = [torch.from_numpy(a).cuda()[:, None] for a in (l, m, nn)]
    vis = d["vis"].to(torch.complex128)
    out = torch.zeros(len(px), dtype=torch.complex128, device="cuda")
    q = max(1, (1 << 26) // len(px))
    for a in range(0, vis.numel(), q):
        sl = slice(a, a + q)
        ph = l * d["u"][None, sl] + m * d["v"][None, sl] + nn * d["w"][None, sl]
        ph -= torch.round(ph)
        e = torch.polar(torch.ones_like(ph), ph * (-2 * math.pi))
        out += (e * vis[None, sl]).sum(1)
    return out


def _ws_geometry(c):
    g = int(math.floor(c["theta"] * c["lam"]))
    og = int(round(0.5 / WS_X0) * g)
    wp = int(math.ceil(math.sin(c["theta"] / 2) * math.sqrt(2.0 * g * g) / WS_DW)) + WS_W + 1
    return g, og, wp


def _exact_wstack(c, d):
    g, og, wp = _ws_geometry(c)
    th, lam = c["theta"], c["lam"]
    kuv, kw, klm, kn = [a.cpu().numpy() for a in _sep_kernels()]
    l, m, flux = [d[x].cpu().numpy() for x in ("l", "m", "flux")]
    lc = np.floor((l / th + 0.5) * g).astype(np.int64)
    mc = np.floor((m / th + 0.5) * g).astype(np.int64)
    lq, mq = lc / lam - th / 2, mc / lam - th / 2
    nq = np.sqrt(1.0 - lq * lq - mq * mq) - 1.0
    step = 1.0 / WS_CORR
    iu = np.floor(WS_DU * lq / step).astype(np.int64) + WS_CORR // 2
    iv = np.floor(WS_DU * mq / step).astype(np.int64) + WS_CORR // 2
    iw = np.floor(WS_DW * nq / step).astype(np.int64) + WS_CORR // 2
    val = flux / (klm[iu] * klm[iv] * kn[iw])
    lp, mp = th * (lc - g // 2) / g, th * (mc - g // 2) / g
    ph = WS_DW * (1.0 - np.sqrt(1.0 - lp * lp - mp * mp))
    xs, ys = (og - g) // 2 + lc, (og - g) // 2 + mc
    stack = torch.zeros((wp, og, og), dtype=torch.complex128, device="cuda")
    for k in range(wp):
        plane = np.zeros((og, og), np.complex128)
        np.add.at(plane, (ys, xs), val * np.exp(2j * math.pi * (k - wp // 2) * ph))
        stack[k] = _shift(torch.fft.fft2(_shift(torch.from_numpy(plane).cuda())))
    out = torch.empty(c["nvis"], dtype=torch.complex128, device="cuda")
    kuv_d = torch.from_numpy(kuv.reshape(WS_OV, WS_UV)).cuda()
    kw_d = torch.from_numpy(kw.reshape(WS_OV, WS_W)).cuda()
    flat = stack.reshape(-1)
    for a in range(0, c["nvis"], 1 << 22):
        sl = slice(a, a + (1 << 22))
        cells, ovs = [], []
        for x, dx, ov in (("u", WS_DU, WS_OV), ("v", WS_DU, WS_OV), ("w", WS_DW, WS_OV)):
            t = d[x][sl].cpu().numpy()
            cl = np.ceil(t / dx)
            ovs.append(torch.from_numpy(np.minimum(np.floor(np.abs(t - cl * dx) / dx * ov), ov - 1)
                                        .astype(np.int64)).cuda())
            cells.append(torch.from_numpy(cl.astype(np.int64)).cuda())
        us, vs, ws = cells[0] + g, cells[1] + g, cells[2] + wp // 2
        acc = torch.zeros(us.numel(), dtype=torch.complex128, device="cuda")
        for iw in range(WS_W):
            gw = kw_d[ovs[2], iw]
            for jv in range(WS_UV):
                gv = gw * kuv_d[ovs[1], jv]
                row = ((ws - WS_W // 2 + iw) * og + vs - WS_UV // 2 + jv) * og + us - WS_UV // 2
                for ju in range(WS_UV):
                    acc += flat[row + ju] * (gv * kuv_d[ovs[0], ju])
        out[sl] = acc
    return out


def _exact_epic(c, d):
    nb, g, s = c["nb"], c["g"], c["supp"]
    out = torch.zeros(nb * g * g, dtype=torch.complex128, device="cuda")
    o = torch.view_as_real(out)
    b = torch.arange(nb, device="cuda")[:, None]
    f, k = d["f"].to(torch.complex128), d["illum"].to(torch.complex128)
    for ty in range(s):
        for tx in range(s):
            x, y = d["x"].long() + tx, d["y"].long() + ty
            ok = (x >= 0) & (x < g) & (y >= 0) & (y < g)
            cell = torch.where(ok, (b * g + y) * g + x, 0).reshape(-1)
            add = torch.where(ok, k[ty, tx].conj() * f, 0).reshape(-1)
            o.index_add_(0, cell, torch.view_as_real(add))
    return out.reshape(nb, g, g)


def exact(case, seed):
    c, d = case, _inputs(case, seed)
    kind = c["kind"]
    if kind in ("wproj", "channels", "cpu_image", "wtowers"):
        table, w_min, step = _kernels(c)
        if c["fp"] == 32:  # the table the call is given
            table = table.to(torch.complex64).to(torch.complex128)
        if kind == "cpu_image":
            return _exact_cpu_image(c, d, table, w_min, step)
        if kind == "wtowers":
            return _exact_towers(c, d, table, w_min, step)
        return _exact_grids(c, d, table, w_min, step, d["vis"].to(torch.complex128))
    if kind == "dft":
        return _exact_dft(c, d)
    if kind == "to_image":
        return _shift(torch.fft.ifft2(_shift(d["grid"].to(torch.complex128)), norm="forward"))
    if kind == "wstack":
        return _exact_wstack(c, d)
    return _exact_epic(c, d)
