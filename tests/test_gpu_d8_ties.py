"""dirType-8 codes where steepest directions tie (small whole elevations, so
that most cells have several), bit for bit against the oracle: every column
remainder of the vector and the per-element path, with and without slope and
mask, and through a batch.
"""
import numpy as np
import pytest

from oracle import pyoracle
from pargo_amd import batch, focal

pytestmark = pytest.mark.gpu

ND = -9999.0


def lattice(rows, cols):
    rng = np.random.default_rng(rows * 1000 + cols)
    z = rng.integers(0, 4, size=(rows, cols)).astype(np.float32)
    z[rng.random((rows, cols)) < 0.01] = ND
    return z


def expect(z, dirtype):
    ref = pyoracle.d8(z, ND, dirtype)
    nd, flat = ref == ND, 255 if dirtype == 8 else 0
    return np.where(nd | (ref == -1), flat, ref).astype(np.uint8), nd


@pytest.mark.parametrize("cols", [3, 66, 255, 256, 257, 258, 259, 513, 1030])
@pytest.mark.parametrize("dirtype", [8, 256])
def test_tied_codes(cols, dirtype):
    import torch
    z = lattice(61, cols)
    code, nd = expect(z, dirtype)
    t = torch.from_numpy(z).cuda()
    for want_slope in (True, False):
        for want_mask in (True, False):
            for method in ("FD", "SD"):
                _, c, m = focal.slope_d8(t, 30.0, ND, method, "tan", dirtype, want_slope=want_slope, want_mask=want_mask)
                assert np.array_equal(c.cpu().numpy(), code)
                if want_mask:
                    assert np.array_equal(focal.unpack_mask(m, cols).cpu().numpy(), nd)


@pytest.mark.parametrize("dirtype", [8, 256])
@pytest.mark.parametrize("mode", [batch.PER_TILE, batch.PERSISTENT, batch.GRAPH])
def test_tied_codes_in_a_batch(dirtype, mode):
    import torch
    zs = [lattice(r, c) for r, c in ((40, 300), (97, 129), (3, 3), (130, 517))]
    b = batch.Batch([torch.from_numpy(z).cuda() for z in zs], 30.0, ND, want_slope=mode != batch.PERSISTENT, dirtype=dirtype)
    for _ in range(3):
        _, codes = b.run(mode)
    for z, c in zip(zs, codes):
        assert np.array_equal(c.cpu().numpy(), expect(z, dirtype)[0])
