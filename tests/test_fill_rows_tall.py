"""The CPU restatement of pitremove's evaluation (test_fill_rows.py) with the
bands of 16 rows that large rasters take."""
import numpy as np
import pytest

from oracle import pyoracle
from tests.test_fill_rows import settle


@pytest.mark.parametrize("seed", range(8))
def test_bands_of_16_rows_reach_the_oracles_values(seed):
    rng = np.random.default_rng(940 + seed)
    rows, cols = int(rng.integers(30, 75)), int(rng.integers(60, 140))
    nodata = [-9999.0, 20000.0, np.inf, -np.inf, -9999.0, -9999.0, -3.4028234663852886e38, -9999.0][seed]
    dem = np.round(rng.random((rows, cols)) * 20, 2).astype(np.float32).astype(np.float64)
    if seed % 2 == 0:
        dem += np.add.outer(np.arange(rows), np.arange(cols)) * 0.25
    dem[rng.random(dem.shape) < 0.03] = 12000.0
    if np.isfinite(nodata):
        dem[rng.random(dem.shape) < 0.02] = nodata
    ref, _, ok = pyoracle.pit_remove(dem, nodata)
    assert ok
    got = settle(dem, nodata, 32, 64, 16)
    assert np.array_equal(got, ref), np.argwhere(got != ref)[:5].tolist()
