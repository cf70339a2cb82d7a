"""Windows with Inf, NaN or |z| >= 2^40, redone exactly: by the waves that met
them in a raster of up to 16,384 wave-rows (rows times 256-column strips), from
the queue in a larger one, from the static queue in pargo_slope_d8_noalloc.
"""
import ctypes

import numpy as np
import pytest

from oracle import pyoracle
from pargo_amd import _lib, focal, synth
from tests.test_gpu_launch_faults import failing_context

pytestmark = pytest.mark.gpu

ND = -9999.0
ROWS, COLS = 2049, 2050  # 2049 x 9 wave-rows


def raster():
    z = synth.workload_dem("slope_d8", ROWS, COLS, seed=71)
    rng = np.random.default_rng(72)
    cells = [(1, 1), (1, COLS - 2), (ROWS - 2, 1), (ROWS - 2, COLS - 2), (0, 700), (900, 0), (1024, 255), (1024, 256)]
    cells += [(int(rng.integers(3, ROWS - 3)), int(rng.integers(3, COLS - 3))) for _ in range(40)]
    values = [3.0e12, np.inf, -np.inf, np.nan, -2.5e13, 3.0e38, 2.0 ** 40]
    for i, (r, c) in enumerate(cells):
        z[r, c] = values[i % len(values)]
    return z, cells


def bits(t):
    import torch
    return t.view(torch.int32) if t.dtype == torch.float32 else t


@pytest.mark.parametrize("method,dirtype", [("FD", 256), ("FD", 8), ("TFDW", 8)])
def test_queue_and_wave_give_the_same_bits(method, dirtype):
    import torch
    z, cells = raster()
    dem = torch.from_numpy(z).cuda()
    s, c, m = focal.slope_d8(dem, 30.0, ND, method, "tan", dirtype, want_mask=True)
    assert torch.equal(bits(focal.slope(dem, 30.0, ND, method)), bits(s))
    for r, col in cells:
        r0, c0 = max(0, r - 4), max(0, col - 4)
        r1, c1 = min(ROWS, r + 5), min(COLS, col + 5)
        crop = dem[r0:r1, c0:c1].contiguous()
        cs, cc, _ = focal.slope_d8(crop, 30.0, ND, method, "tan", dirtype, want_mask=True)
        a, b = slice(1, r1 - r0 - 1), slice(1, c1 - c0 - 1)
        assert torch.equal(bits(s)[r0:r1, c0:c1][a, b], bits(cs)[a, b]), (r, col)
        assert torch.equal(c[r0:r1, c0:c1][a, b], cc[a, b]), (r, col)
    # the exact pass matters: without it (its launch failed) windows differ
    p = torch.zeros_like(s)
    q = torch.zeros_like(c)
    L, ctx = _lib.lib(), failing_context(1)
    ctx.bind_stream()
    g = focal.grid_of(dem, 30.0, ND)
    rc = L.pargo_slope_d8(ctx.h, ctypes.byref(g), _lib._ptr(dem), focal.get_slope_algorithm(method), 0, dirtype,
                          _lib._ptr(p), _lib._ptr(q), None)
    torch.cuda.synchronize()
    ctx.close()
    assert rc == _lib.PARGO_E_DEVICE
    differs = (bits(p) != bits(s)) | (q != c)
    near = torch.zeros_like(differs)
    for r, col in cells:
        near[max(0, r - 1):r + 2, max(0, col - 1):col + 2] = True
    assert bool(differs.any()) and not bool((differs & ~near).any())


def test_codes_match_the_oracle():
    import torch
    z, _ = raster()
    _, c, m = focal.slope_d8(torch.from_numpy(z).cuda(), 30.0, ND, want_mask=True)
    ref = pyoracle.d8(z, ND, 256)
    nd = ref == ND
    assert np.array_equal(focal.unpack_mask(m, COLS).cpu().numpy(), nd)
    got = np.where(nd, 0, c.cpu().numpy().astype(np.int64))
    assert np.array_equal(got, np.where((ref == -1) | nd, 0, ref).astype(np.int64))


def test_noalloc_queue_gives_the_same_bits():
    import torch
    z, _ = raster()
    dem = torch.from_numpy(z).cuda()
    ref = focal.slope_d8(dem, 30.0, ND, want_mask=True)
    L, ctx = _lib.lib(), failing_context(2)  # a context without a queue of its own
    ctx.bind_stream()
    g = focal.grid_of(dem, 30.0, ND)
    # twice, the second time on what an interrupted call left in the counters
    for interrupted in (False, True):
        out = [torch.zeros_like(t) for t in ref]
        args = (ctx.h, ctypes.byref(g), _lib._ptr(dem), 0, 0, 256) + tuple(_lib._ptr(t) for t in out)
        if interrupted:
            assert L.pargo_slope_d8_noalloc(*args) == _lib.PARGO_E_DEVICE
        ctx.check(L.pargo_slope_d8_noalloc(*args))
        torch.cuda.synchronize()
        for a, b in zip(out, ref):
            assert torch.equal(bits(a), bits(b))
    ctx.close()
