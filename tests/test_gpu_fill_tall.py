"""pitremove with two waves of 16 rows a tile (rasters of 16,384 tiles and
more) where its bands and tiles meet, bit for bit against the oracle.

The directed rasters are stacked until there are enough tiles, their first and
last rows NoData as the border would be: every copy has to come out as the one
raster does, whatever row of a tile it begins on.
"""
import numpy as np
import pytest

from oracle import pyoracle
from tests.test_gpu_fill import ND, gpu_fill

pytestmark = pytest.mark.gpu

TILES = 16384


def check(z, nodata=ND, pad=0):
    import torch
    from pargo_amd import hydro
    z[0], z[-1] = nodata, nodata
    ref, _, ok = pyoracle.pit_remove(z, nodata)
    assert ok
    rows, cols = z.shape
    copies = -(-(TILES // -(-cols // 64) * 32) // rows)
    dem = torch.zeros((copies * rows, cols + pad), dtype=torch.float32, device="cuda")
    dem[:, :cols] = torch.from_numpy(z).cuda().repeat(copies, 1)
    w, _ = hydro.pit_remove(dem[:, :cols], nodata)
    got = w.reshape(copies, rows, cols)
    bad = torch.nonzero(got != torch.from_numpy(ref).cuda()[None])
    assert len(bad) == 0, (len(bad), bad[:5].tolist())


@pytest.mark.parametrize("rows,cols", [(3, 3), (8, 64), (9, 65), (15, 63), (16, 64), (17, 65), (31, 63), (32, 64),
                                       (33, 65), (34, 66), (40, 129), (63, 127), (65, 193), (97, 66), (129, 200)])
def test_sizes_around_tiles_and_bands(rows, cols):
    rng = np.random.default_rng(1000 * rows + cols + 1)
    z = (rng.random((rows, cols)) * 20 + np.add.outer(np.arange(rows), np.arange(cols)) * 0.3).astype(np.float32)
    z[rng.random((rows, cols)) < 0.01] = ND
    check(z, pad=cols % 5)


@pytest.mark.parametrize("row,col", [(31, 63), (32, 64), (31, 64), (32, 63), (15, 63), (16, 64), (47, 100), (48, 63),
                                     (63, 128)])
def test_one_outlet_floods_the_rest(row, col):
    rng = np.random.default_rng(row * 100 + col)
    z = (rng.random((100, 200)) * 5).astype(np.float32)
    z[1:3], z[-3:], z[:, 1:3], z[:, -3:] = 10001.0, 10001.0, 10001.0, 10001.0
    z[row, col] = ND
    check(z)


@pytest.mark.parametrize("horizontal", [True, False])
def test_one_cell_corridor_through_every_band(horizontal):
    z = np.full((75, 140), 10000.0, dtype=np.float32)
    for i, r in enumerate(range(4, 70, 4)):
        z[r, 4:135] = 50.0 - 0.1 * i
        z[r:r + 5, 134 if i % 2 == 0 else 4] = 50.0
    z[0:5, 4] = 1.0
    check(z if horizontal else np.ascontiguousarray(z.T))


@pytest.mark.parametrize("nodata", [20000.0, np.inf, -np.inf, -3.4028234663852886e38])
def test_nodata_outside_the_usual_range(nodata):
    # a raster of 5 columns, small enough for the oracle with all its tiles
    rng = np.random.default_rng(7)
    z = (rng.random((TILES * 32, 5)) * 40).astype(np.float32)
    z[20::97, 2], z[33::101, 3] = 9999.9995, 12000.0
    if np.isfinite(nodata):
        z[40::211, 1:3] = nodata
    ref, _, ok = pyoracle.pit_remove(z, nodata)
    assert ok
    got, _ = gpu_fill(z, nodata)
    assert np.array_equal(got, ref), np.argwhere(got != ref)[:5].tolist()
