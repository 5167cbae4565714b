"""EPIC E-field gridding on the GPU (src/epic/epic_grid.cu) against the
oracle: the reference's workload shape (1000 timestamps x 256 antennas,
64^2 grids, 2x2 top hat), a complex illumination with antennas on the grid
edges, and a grid too large for LDS (global-atomic path)."""
import numpy as np
import pytest
import torch

import pyoracle as orc
import rgamd
from gpu_util import dev

pytestmark = pytest.mark.gpu


def run(ctx, f, x, y, il, g):
    nb = f.shape[0]
    grids = torch.full((nb, g, g), 3.0, dtype=torch.complex64, device="cuda")
    ctx.epic_grid(dev(f.astype(np.complex64)), dev(x.astype(np.int32)),
                  dev(y.astype(np.int32)), dev(il.astype(np.complex64)), grids)
    torch.cuda.synchronize()
    return grids.cpu().numpy()


def fields(rng, nb, na):
    return (rng.normal(0, 5, (nb, na)) + 1j * rng.normal(0, 5, (nb, na))).astype(np.complex64)


def test_reference_workload_matches_oracle(ctx):
    g, S, nb, na = 64, 2, 1000, 256
    rng = np.random.default_rng(1)
    f = fields(rng, nb, na)
    x = rng.integers(S, g - S + 1, nb * na)  # loc_distribution(ILLUM_X, GRID_SIZE - ILLUM_X)
    y = rng.integers(S, g - S + 1, nb * na)
    il = np.ones((S, S), np.complex64)
    got = run(ctx, f, x, y, il, g)
    ref = orc.epic_grid(f.astype(np.complex128), x, y, il, g)
    assert np.abs(got - ref).max() < 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("g,S", [(40, 3), (128, 4)])
def test_complex_illumination_and_edges_match_oracle(ctx, g, S):
    rng = np.random.default_rng(g)
    nb, na = 7, 300
    f = fields(rng, nb, na)
    x = rng.integers(-S, g + 1, nb * na)  # some footprints hang over every edge
    y = rng.integers(-S, g + 1, nb * na)
    il = (rng.standard_normal((S, S)) + 1j * rng.standard_normal((S, S))).astype(np.complex64)
    got = run(ctx, f, x, y, il, g)
    ref = orc.epic_grid(f.astype(np.complex128), x, y, il.astype(np.complex128), g)
    assert np.abs(got - ref).max() < 1e-5 * np.abs(ref).max()


def test_invalid_arguments_are_rejected(ctx):
    f = torch.zeros((2, 3), dtype=torch.complex64, device="cuda")
    xy = torch.zeros(6, dtype=torch.int32, device="cuda")
    il = torch.zeros((0, 0), dtype=torch.complex64, device="cuda")
    grids = torch.zeros((2, 8, 8), dtype=torch.complex64, device="cuda")
    with pytest.raises(rgamd.RGError):
        ctx.epic_grid(f, xy, xy, il, grids)  # support 0


@pytest.mark.parametrize("g,S,nb,na,spread", [
    (5, 1, 3, 40, 7), (33, 2, 2, 257, 40), (64, 2, 1, 300, 1), (64, 8, 3, 512, 70),
    (91, 3, 2, 300, 95), (200, 5, 2, 64, 210), (256, 8, 1, 300, 3), (400, 16, 1, 20, 420),
    (128, 4, 2, 5000, 130)])
def test_bands_footprints_and_collisions(ctx, g, S, nb, na, spread):
    """Every kernel form: supports 1, 2, 3 and run-time ones, one and several
    bands, odd grids, antennas that all stand on a few cells, and the global
    atomics taken with many antennas.  FP32 sums of at most na S^2 terms a
    cell: each is off by at most terms 2^-23 of the sum of their moduli."""
    rng = np.random.default_rng(g + S)
    f = fields(rng, nb, na)
    x = rng.integers(-S, spread - S + 1, nb * na)
    y = rng.integers(-S, spread - S + 1, nb * na)
    il = (rng.standard_normal((S, S)) + 1j * rng.standard_normal((S, S))).astype(np.complex64)
    got = run(ctx, f, x, y, il, g)
    ref = orc.epic_grid(f.astype(np.complex128), x, y, il.astype(np.complex128), g)
    mod = orc.epic_grid(np.abs(f).astype(np.complex128), x, y, np.abs(il).astype(np.complex128), g)
    hits = orc.epic_grid(np.ones_like(f, np.complex128), x, y, np.ones((S, S), np.complex128), g)
    assert (np.abs(got - ref) <= (hits.real + 4) * 2.0 ** -23 * mod.real + 1e-30).all()


@pytest.mark.parametrize("na", [1, 255, 256, 257, 513])
@pytest.mark.parametrize("g,S,nb,spread", [(64, 2, 5, 2), (64, 4, 3, 20), (100, 7, 2, 100),
                                           (70, 64, 1, 30), (300, 2, 2, 310)])
def test_lists_of_antennas_on_shared_cells(ctx, g, S, nb, na, spread):
    """Antennas around the 256 that a workgroup lists at a time, within 4 x 4 cells, close together
    and spread over the grid, footprints up to the largest.  The bound of the test above."""
    rng = np.random.default_rng(na + S)
    f = fields(rng, nb, na)
    x, y = rng.integers(-S, spread - S + 1, (2, nb * na)) + min(S, g // 4)
    il = (rng.standard_normal((S, S)) + 1j * rng.standard_normal((S, S))).astype(np.complex64)
    got = run(ctx, f, x, y, il, g)
    ref = orc.epic_grid(f.astype(np.complex128), x, y, il.astype(np.complex128), g)
    mod = orc.epic_grid(np.abs(f).astype(np.complex128), x, y, np.abs(il).astype(np.complex128), g)
    hits = orc.epic_grid(np.ones_like(f, np.complex128), x, y, np.ones((S, S), np.complex128), g)
    assert (np.abs(got - ref) <= (hits.real + 4) * 2.0 ** -23 * mod.real + 1e-30).all()


@pytest.mark.parametrize("g,S,nb,na", [(64, 2, 1, 60_000), (91, 3, 1, 40_001), (256, 1, 2, 90_000),
                                       (64, 2, 40, 6000), (8, 1, 2, 100)])
def test_many_antennas_by_bands_and_by_atomics(ctx, g, S, nb, na):
    """One or two grids of very many antennas (global atomics) and more of them (bands, many lists
    each).  The bound of the tests above."""
    rng = np.random.default_rng(na)
    f = fields(rng, nb, na)
    x, y = rng.integers(-S, g + 1, (2, nb * na))
    il = (rng.standard_normal((S, S)) + 1j * rng.standard_normal((S, S))).astype(np.complex64)
    got = run(ctx, f, x, y, il, g)
    ref = orc.epic_grid(f.astype(np.complex128), x, y, il.astype(np.complex128), g)
    mod = orc.epic_grid(np.abs(f).astype(np.complex128), x, y, np.abs(il).astype(np.complex128), g)
    hits = orc.epic_grid(np.ones_like(f, np.complex128), x, y, np.ones((S, S), np.complex128), g)
    assert (np.abs(got - ref) <= (hits.real + 4) * 2.0 ** -23 * mod.real + 1e-30).all()
