"""GPU parity of pitremove where its tiles and bands meet, bit for bit.

A tile is 64 x 32 cells, held by four waves of 8 rows; a visit starts from
the bands of 8 rows next to a changed edge.  These rasters send the only
change of a tile through one edge, one corner or one band, and cover sizes on
either side of every boundary.
"""
import numpy as np
import pytest

from oracle import pyoracle
from tests.test_gpu_fill import ND, gpu_fill

pytestmark = pytest.mark.gpu


def check(z, nodata=ND, pad=0):
    ref, _, ok = pyoracle.pit_remove(z, nodata)
    assert ok
    got, _ = gpu_fill(z, nodata, pad)
    assert np.array_equal(got, ref), np.argwhere(got != ref)[:5].tolist()


@pytest.mark.parametrize("rows,cols", [(1, 1), (2, 70), (3, 3), (8, 64), (9, 65), (31, 63), (32, 64), (33, 65),
                                       (34, 66), (40, 129), (63, 127), (65, 193), (97, 66), (129, 200)])
def test_sizes_around_tiles_and_bands(rows, cols):
    rng = np.random.default_rng(1000 * rows + cols)
    z = (rng.random((rows, cols)) * 20 + np.add.outer(np.arange(rows), np.arange(cols)) * 0.3).astype(np.float32)
    z[rng.random((rows, cols)) < 0.01] = ND
    check(z, pad=cols % 5)


@pytest.mark.parametrize("row,col", [(31, 63), (32, 64), (31, 64), (32, 63), (39, 63), (40, 64), (47, 100), (63, 128)])
def test_one_outlet_floods_the_rest(row, col):
    # a wall of frozen cells inside the border; one NoData cell inside opens
    # the basin, so every change starts at that cell and crosses the edges
    # and corners around it
    rng = np.random.default_rng(row * 100 + col)
    z = (rng.random((100, 200)) * 5).astype(np.float32)
    z[1:3], z[-3:], z[:, 1:3], z[:, -3:] = 10001.0, 10001.0, 10001.0, 10001.0
    z[row, col] = ND
    check(z)


@pytest.mark.parametrize("horizontal", [True, False])
def test_one_cell_corridor_through_every_band(horizontal):
    # a corridor one cell wide between frozen walls, folded through the raster
    z = np.full((75, 140), 10000.0, dtype=np.float32)
    for i, r in enumerate(range(4, 70, 4)):
        z[r, 4:135] = 50.0 - 0.1 * i
        z[r:r + 5, 134 if i % 2 == 0 else 4] = 50.0
    z[0:5, 4] = 1.0
    check(z if horizontal else np.ascontiguousarray(z.T))


@pytest.mark.parametrize("nodata", [20000.0, np.inf, -np.inf, -3.4028234663852886e38])
def test_nodata_outside_the_usual_range(nodata):
    rng = np.random.default_rng(7)
    z = (rng.random((70, 130)) * 40).astype(np.float32)
    z[20, 64], z[33, 65] = 9999.9995, 12000.0
    if np.isfinite(nodata):
        z[40:43, 60:70] = nodata
    check(z, nodata)


@pytest.mark.parametrize("rows,cols", [(1050, 32001), (16401, 2011)])
def test_two_waves_a_tile(rows, cols):
    # rasters of 16,384 tiles and more; too large for the oracle's sweeps, so
    # the settled equations, which have one solution, are checked at every cell
    import torch
    from pargo_amd import hydro, synth
    z = torch.from_numpy(synth.workload_dem("slope_d8", rows, cols)).cuda()
    w, _ = hydro.pit_remove(z, ND)
    d = z.double()
    out = (d - ND).abs() <= 1e-6
    out[0], out[-1], out[:, 0], out[:, -1] = True, True, True, True
    assert bool((w[out] == ND).all())
    v = torch.where(out, torch.full_like(w, -np.inf), w)  # NoData opens its neighbours
    n = torch.full_like(v[1:-1, 1:-1], np.inf)
    for i in range(3):
        for j in range(3):
            if (i, j) != (1, 1):
                n = torch.minimum(n, v[i:rows - 2 + i, j:cols - 2 + j])
    want = torch.clamp(torch.maximum(d[1:-1, 1:-1], n + 0.0005), max=10000.0)
    live = ~out[1:-1, 1:-1]
    assert bool((w[1:-1, 1:-1][live] == want[live]).all())
