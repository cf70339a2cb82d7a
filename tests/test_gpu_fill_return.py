"""pitremove is done with the caller's rasters when it returns, also when it
refuses the DEM: nothing is written into the output any more, and after a
refusal the stream holds no work.  A DEM is refused exactly when it holds NaN
or when NoData lies within 1e-6 of a value a cell can take, on the device as
on the host.
"""
import ctypes

import numpy as np
import pytest

from oracle import pyoracle
from pargo_amd import _lib, synth
from pargo_amd.focal import grid_of
from tests.test_gpu_fill import ND, gpu_fill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("what,code", [("nan", _lib.PARGO_E_INVALID), ("nodata inside", _lib.PARGO_E_UNSUPPORTED),
                                       ("accepted", _lib.PARGO_OK)])
@pytest.mark.parametrize("side", [70, 3000])
def test_nothing_is_written_after_the_return(what, code, side):
    import torch
    z = synth.workload_dem("slope_d8", side, side + 13)
    if what == "nan":
        z[side // 2, side // 3] = np.nan
    dem = torch.from_numpy(z).cuda()
    # NoData above every elevation, inside the range that ends at 10000
    g = grid_of(dem, 1.0, 9000.0 if what == "nodata inside" else ND)
    out = torch.zeros(dem.shape, dtype=torch.float64, device="cuda")
    stream, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    L, ctx, passes = _lib.lib(), _lib.default_context(0), ctypes.c_int(-1)
    with torch.cuda.stream(stream):
        ctx.bind_stream()
        stream.synchronize()
        rc = L.pargo_pit_remove(ctx.h, ctypes.byref(g), _lib._ptr(dem), _lib._ptr(out), ctypes.byref(passes))
        idle = stream.query()
    with torch.cuda.stream(other):  # both rasters are the caller's again
        dem.fill_(-1.0)
        out.fill_(7.0)
    torch.cuda.synchronize()
    assert rc == code and (idle or code == _lib.PARGO_OK)
    assert bool((out == 7.0).all())


@pytest.mark.parametrize("nodata,refused", [(50.0 - 2e-6, False), (50.0, False), (50.0 + 2e-6, True), (9000.0, True),
                                            (10000.0, True), (10000.0 + 5e-7, True), (10000.0 + 2e-6, False)])
def test_refused_exactly_inside_the_range(nodata, refused):
    rng = np.random.default_rng(61)
    z = (50 + np.round(rng.random((40, 150)) * 30, 2)).astype(np.float32)
    z[20, 100] = 50.0  # the lowest cell (NoData itself where nodata is 50)
    if refused:
        with pytest.raises(_lib.PargoError) as e:
            gpu_fill(z, nodata)
        assert e.value.code == _lib.PARGO_E_UNSUPPORTED
        return
    ref, _, ok = pyoracle.pit_remove(z, nodata)
    assert ok
    got, _ = gpu_fill(z, nodata)
    assert np.array_equal(got, ref), np.argwhere(got != ref)[:5].tolist()


def test_no_valid_cell_is_accepted_whatever_nodata():
    z = np.full((40, 70), 500.0, np.float32)
    got, _ = gpu_fill(z, 500.0)
    assert (got == 500.0).all()


def test_the_passes_reported_are_those_that_had_tiles():
    z = (100 + np.add.outer(np.arange(30), np.arange(60)) * 0.5).astype(np.float32)
    _, passes = gpu_fill(z)
    assert passes == 1  # one tile, and none beside it to schedule
    # a basin over two tiles with its outlet in the left one: what the right
    # tile settles to waits for the left one, so the first pass is not the last
    z = np.full((32, 128), 10001.0, np.float32)
    z[3:-3, 3:-3] = 50.0
    z[10, 5] = ND
    ref, _, ok = pyoracle.pit_remove(z, ND)
    assert ok
    got, passes = gpu_fill(z)
    assert np.array_equal(got, ref) and 2 <= passes < 8, passes
