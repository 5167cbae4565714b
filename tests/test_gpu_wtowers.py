"""W-towers on the GPU (plain and batched) against the oracle."""
import numpy as np
import pytest
import torch

import pyoracle as orc
import rgamd
import synth
from gpu_util import kern, rel_max, rel_rms, small_obs, stage

pytestmark = pytest.mark.gpu

SUB, MARGIN, WINC = 64, 16, 10.0


@pytest.fixture(scope="module")
def case():
    obs, vis = small_obs(n_st=14, n_dumps=32, arm_m=700.0, lam=2560.0)  # N = 256
    w_step = 1.0
    table = rgamd.make_wkernels(11, 8, 16, obs.theta, -5.0, w_step)
    ref, fl, bad = orc.grid_wtowers(obs.grid_size, obs.theta, obs.u, obs.v, obs.w, vis, table,
                                    -5.0, w_step, SUB, MARGIN, WINC, nthreads=8)
    assert bad == 0 and fl == 8 * 256 * obs.n_vis
    return obs, vis, table, ref


def run(ctx, obs, vis, table, mode, dt=torch.complex128, **kw):
    _, fv = stage(obs.u, obs.v, obs.w, vis, dt)
    kt, wk = kern(table, -5.0, 1.0, dt)
    N = obs.grid_size
    g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    ctx.grid(rgamd.params(N, obs.theta, mode=mode, subgrid=SUB, margin=MARGIN, winc=WINC, **kw),
             fv, wk, g)
    st = ctx.stats()
    torch.cuda.synchronize()
    return g.cpu().numpy(), st


def test_plain_fp64_matches_oracle(ctx, case):
    obs, vis, table, ref = case
    g, st = run(ctx, obs, vis, table, rgamd.RG_MODE_PLAIN)
    assert rel_max(g, ref) < 1e-11
    assert st.n_tasks > 1 and st.n_towers >= 1


@pytest.mark.parametrize("floor_batch,band,radix", [(1, 8, 0), (5, 8, 0), (128, 8, 0), (5, 4, 0),
                                                   (5, 8, 4), (0, 4, 4)])
def test_batched_fp64_matches_oracle(ctx, case, floor_batch, band, radix):
    """radix 4: the column pass's FFT in radix-4 stages (4, 4, 4 at n = 64)."""
    obs, vis, table, ref = case
    g, st = run(ctx, obs, vis, table, rgamd.RG_MODE_BATCHED, floor_batch=floor_batch,
                vis_per_item=50, tile=band, fft_radix=radix)
    assert rel_max(g, ref) < 1e-11
    assert st.n_gridded == obs.n_vis and st.n_dropped == 0


@pytest.mark.parametrize("band,per_item,comp", [(8, 0, 0), (8, 37, 0), (16, 0, 0), (16, 37, 0),
                                               (4, 0, 0), (4, 37, 0), (8, 37, 1), (16, 0, 1),
                                               (4, 37, 1)])
def test_batched_fp32_within_tolerance(ctx, case, band, per_item, comp):
    """FP32 bands of 8 / 16 / 4 rows; per_item 37 splits most band keys over
    several work items (spilled parts summed by the combine pass); comp: two-sum
    compensated register sums."""
    obs, vis, table, ref = case
    g, st = run(ctx, obs, vis, table, rgamd.RG_MODE_BATCHED, dt=torch.complex64, tile=band,
                vis_per_item=per_item, compensated=comp)
    img, img_ref = orc.grid_to_image(g), orc.grid_to_image(ref)
    assert rel_max(img, img_ref) < 1e-5 and rel_rms(img, img_ref) < 1e-5
    assert st.n_gridded == obs.n_vis


def test_task_count_matches_binning(ctx, case):
    obs, vis, table, ref = case
    _, st = run(ctx, obs, vis, table, rgamd.RG_MODE_BATCHED)
    N, chunk = obs.grid_size, SUB - MARGIN
    tasks = {(orc.tower_index(obs.u[i], obs.theta, N, chunk),
              orc.tower_index(obs.v[i], obs.theta, N, chunk),
              orc.floor_index(obs.w[i], WINC)) for i in range(obs.n_vis)}
    assert st.n_tasks == len(tasks)
    assert st.n_towers == len({(a, b) for a, b, _ in tasks})


def test_fp64_required_for_plain(ctx, case):
    obs, vis, table, ref = case
    with pytest.raises(rgamd.RGError) as e:
        run(ctx, obs, vis, table, rgamd.RG_MODE_PLAIN, dt=torch.complex64)
    assert e.value.code == rgamd.RG_ERR_PARAM


def test_stress_shape_matches_oracle(ctx):
    """The stress-workload shape at reduced size: 4096^2 grid (theta 0.2),
    subgrid 256, margin 16, winc 10, phase centre at zenith angle 60 deg
    (|w| up to thousands of wavelengths, hundreds of floors), three channels."""
    obs = synth.config_c5(n_st=20, n_chan=3, n_dumps=24)
    vis = synth.predict_numpy(obs.u, obs.v, obs.w, obs.l, obs.m, obs.flux)
    sub, margin, winc = 256, 16, 10.0
    table = rgamd.make_wkernels(11, 8, 16, obs.theta, -5.0, 1.0)
    ref, fl, bad = orc.grid_wtowers(obs.grid_size, obs.theta, obs.u, obs.v, obs.w, vis, table,
                                    -5.0, 1.0, sub, margin, winc, nthreads=8)
    assert bad == 0 and obs.grid_size == 4096
    N = obs.grid_size
    for dt, tol in ((torch.complex128, 1e-11), (torch.complex64, 1e-5)):
        _, fv = stage(obs.u, obs.v, obs.w, vis, dt)
        kt, wk = kern(table, -5.0, 1.0, dt)
        g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
        ctx.grid(rgamd.params(N, obs.theta, mode=rgamd.RG_MODE_BATCHED, subgrid=sub,
                              margin=margin, winc=winc), fv, wk, g)
        st = ctx.stats()
        torch.cuda.synchronize()
        got = g.cpu().numpy()
        assert rel_max(got, ref) < tol, dt
        assert st.n_gridded == obs.n_vis and st.n_tasks > 50
        del g


@pytest.mark.parametrize("sub,margin,S", [(128, 16, 8), (128, 8, 8), (256, 16, 16)])
@pytest.mark.parametrize("radix", [8, 4])
def test_other_shapes_match_oracle(ctx, sub, margin, S, radix):
    """Kernel support 8 and subgrids 128 / 256 through the batched path, the
    column pass's FFT in radix-8 stages (8, 8, 2 / 8, 8, 4) or radix-4 stages
    (4, 4, 4, 2 / 4, 4, 4, 4)."""
    obs, vis = small_obs(n_st=14, n_dumps=24, arm_m=900.0, lam=5120.0)  # N = 512
    table = rgamd.make_wkernels(11, 4, S, obs.theta, -5.0, 1.0)
    ref, _, bad = orc.grid_wtowers(obs.grid_size, obs.theta, obs.u, obs.v, obs.w, vis, table,
                                   -5.0, 1.0, sub, margin, WINC, nthreads=8)
    assert bad == 0
    N = obs.grid_size
    for dt, tol in ((torch.complex128, 1e-11), (torch.complex64, 1e-5)):
        _, fv = stage(obs.u, obs.v, obs.w, vis, dt)
        kt, wk = kern(table, -5.0, 1.0, dt)
        g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
        ctx.grid(rgamd.params(N, obs.theta, mode=rgamd.RG_MODE_BATCHED, subgrid=sub,
                              margin=margin, winc=WINC, vis_per_item=97, fft_radix=radix),
                 fv, wk, g)
        st = ctx.stats()
        torch.cuda.synchronize()
        assert rel_max(g.cpu().numpy(), ref) < tol, (dt, sub, S)
        assert st.n_gridded == obs.n_vis


@pytest.mark.parametrize("sub", [64, 128, 256, 512])
@pytest.mark.parametrize("n,spread", [(1, 1.0), (9, 20.0), (129, 30.0), (257, 200.0), (600, 3.0)])
def test_batched_fp32_row_pairs(ctx, sub, n, spread):
    """Support-16 tables in 8-row bands, where a lane takes two rows: single records, batches of
    8 and one more, stages of 256 records, one column and many (the wavefronts' runs meet in
    one footprint), every subgrid size.  FP32 against the oracle in FP64, the image to the 1e-5 of
    the other FP32 tests."""
    N, theta = sub, 0.1
    rng = np.random.default_rng(sub + n)
    u = 40.0 + rng.uniform(-spread, spread, n)
    v = -30.0 + rng.uniform(-spread, spread, n)
    w = rng.uniform(-14.0, 14.0, n)
    vis = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    table = rgamd.make_wkernels(11, 4, 16, theta, -5.0, 1.0)
    ref, _, bad = orc.grid_wtowers(N, theta, u, v, w, vis, table, -5.0, 1.0, sub, MARGIN, WINC)
    assert bad == 0
    _, fv = stage(u, v, w, vis, torch.complex64)
    _, wk = kern(table, -5.0, 1.0, torch.complex64)
    g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    ctx.grid(rgamd.params(N, theta, subgrid=sub, margin=MARGIN, winc=WINC), fv, wk, g)
    assert ctx.stats().n_gridded == n
    img, img_ref = orc.grid_to_image(g.cpu().numpy()), orc.grid_to_image(ref)
    assert rel_max(img, img_ref) < 1e-5 and rel_rms(img, img_ref) < 1e-5


@pytest.fixture(scope="module")
def outside():
    """2^22 visibilities outside every tower: with them a stream is long enough for two band rows a
    lane."""
    n = 1 << 22
    return [torch.full((n,), 1e9, dtype=torch.float64, device="cuda") for _ in range(3)] + [
        torch.ones(n, dtype=torch.complex64, device="cuda")]


@pytest.mark.parametrize("sub", [64, 128, 256, 512])
@pytest.mark.parametrize("n,spread,planes", [(1, 1.0, 11), (9, 20.0, 11), (129, 30.0, 11), (257, 200.0, 11),
                                             (600, 3.0, 11), (600, 30.0, 121)])
def test_long_streams_by_row_pairs(ctx, outside, sub, n, spread, planes):
    """The streams and the bound of the test above, in calls long enough for row pairs; a table too
    large for pairs (121 planes at R = 4: 12 MB)."""
    N, theta = sub, 0.1
    rng = np.random.default_rng(sub + n)
    u = 40.0 + rng.uniform(-spread, spread, n)
    v = -30.0 + rng.uniform(-spread, spread, n)
    w = rng.uniform(-14.0, 14.0, n)
    vis = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    step = 10.0 / (planes - 1)
    table = rgamd.make_wkernels(planes, 4, 16, theta, -5.0, step)
    ref, _, bad = orc.grid_wtowers(N, theta, u, v, w, vis, table, -5.0, step, sub, MARGIN, WINC)
    assert bad == 0
    few, _ = stage(u, v, w, vis, torch.complex64)
    keep = [torch.cat([o[:(1 << 21) + 7], f, o[(1 << 21) + 7:]]) for f, o in zip(few, outside)]
    _, wk = kern(table, -5.0, step, torch.complex64)
    g = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    ctx.grid(rgamd.params(N, theta, subgrid=sub, margin=MARGIN, winc=WINC), rgamd.flat_vis(*keep),
             wk, g)
    assert ctx.stats().n_gridded == n
    img, img_ref = orc.grid_to_image(g.cpu().numpy()), orc.grid_to_image(ref)
    assert rel_max(img, img_ref) < 1e-5 and rel_rms(img, img_ref) < 1e-5


def test_row_pairs_and_single_rows_agree(ctx):
    """A dense stream of 2^22 visibilities (row pairs) and of one less (a row a lane), both in FP32,
    against FP64: the same products and sums, so neither is further off by more than a half."""
    N, theta, sub, n = 1024, 0.1, 256, 1 << 22
    rng = np.random.default_rng(2)
    u, v = rng.uniform(-4000, 4000, (2, n))
    w = rng.uniform(-24.0, 24.0, n)
    vis = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    vis[-1] = 0
    vis = vis.astype(np.complex64)
    table = rgamd.make_wkernels(11, 8, 16, theta, -5.0, 1.0).astype(np.complex64)
    p = rgamd.params(N, theta, subgrid=sub, margin=MARGIN, winc=WINC)
    keep, f64 = stage(u, v, w, vis.astype(np.complex128))
    _, k64 = kern(table.astype(np.complex128), -5.0, 1.0)
    ref = torch.empty((N, N), dtype=torch.complex128, device="cuda")
    ctx.grid(p, f64, k64, ref)
    _, k32 = kern(table, -5.0, 1.0, torch.complex64)
    v32 = keep[3].to(torch.complex64)
    err = []
    for m in (n, n - 1):
        g = torch.empty_like(ref)
        ctx.grid(p, rgamd.flat_vis(keep[0][:m], keep[1][:m], keep[2][:m], v32[:m]), k32, g)
        err.append(float((g - ref).norm() / ref.norm()))
    assert err[0] <= 1.5 * err[1] and err[1] <= 1.5 * err[0] and max(err) < 1e-5, err
