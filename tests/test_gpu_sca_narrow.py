"""Contributing area of rasters of one column of tiles (up to 32 cells) or one
row (up to 16): bit for bit against the oracle on either side of the sizes
where their memory layout begins, and the working memory they take.
"""
import numpy as np
import pytest

from oracle import pyoracle
from pargo_amd import _lib, hydro
from tests.test_gpu_sca import ND
from tests.test_gpu_sca_tiles import CODE, along, check, snake

pytestmark = pytest.mark.gpu

SIZES = [(200, c) for c in (1, 2, 3, 4, 17, 31, 32, 33)] + [(r, 400) for r in (1, 2, 3, 4, 8, 15, 16, 17)] + \
    [(3, 3), (5, 64), (10, 33), (16, 64), (16, 65), (33, 32), (32, 32), (65, 9), (64, 3), (3, 128), (4, 129)]


@pytest.mark.parametrize("rows,cols", SIZES)
def test_random_codes(rows, cols):
    rng = np.random.default_rng(101 * rows + cols)
    # long chains along the raster, some against the sweep, some turning back
    along_it = [7, 7, 7, 6, 8, 7, 1] if rows > cols else [5, 5, 5, 2, 8, 5, 3]
    for extra in ([0, 1, 2, 3, 5, 6, 7, 8, -1, ND], []):
        d8 = rng.choice(along_it * 2 + extra, size=(rows, cols)).astype(float)
        check(d8, cols % 3)


@pytest.mark.parametrize("rows,cols", [(300, 12), (300, 3), (12, 500), (3, 500)])
@pytest.mark.parametrize("flip", [False, True])
def test_one_path_through_every_cell(rows, cols, flip):
    if rows > cols:
        cells = snake(1, rows - 1, 1, cols - 1)
    else:
        cells = [(c, r) for r, c in snake(1, cols - 1, 1, rows - 1)]
    check(along(cells[::-1] if flip else cells, (rows, cols)))


@pytest.mark.parametrize("at", [(31, 5), (63, 8), (40, 3)])
def test_cycles_across_an_edge(at):
    r, c = at
    rng = np.random.default_rng(r)
    d8 = rng.choice([6.0, 7.0, 8.0], size=(150, 14))
    for a, b in zip([(0, 0), (0, 1), (1, 1), (1, 0)], [(0, 1), (1, 1), (1, 0), (0, 0)]):
        d8[r + a[0], c + a[1]] = CODE[(b[0] - a[0], b[1] - a[1])]
    check(d8)
    turned = np.full((14, 150), -1.0)  # the same raster on its side
    for (dr, dc), k in CODE.items():
        turned[(d8 == k).T] = CODE[(dc, dr)]
    check(turned)


@pytest.mark.parametrize("rows,cols", [(400_000, 1), (200_000, 3), (60_000, 32), (1, 400_000), (16, 60_000)])
def test_working_memory_by_the_cell(rows, cols):
    import torch
    rng = np.random.default_rng(rows % 97)
    d8 = rng.choice([5.0, 6.0, 7.0, 8.0, 2.0], size=(rows, cols))
    ctx = _lib.Context(0)
    flow = hydro.d8_classify(torch.from_numpy(d8).cuda(), ND, ctx=ctx)
    hydro.sca_d8(torch.zeros((40, 40), dtype=torch.uint8, device="cuda"), ND, ctx=ctx)  # kernels loaded
    torch.cuda.synchronize()
    out = hydro.sca_d8(flow, ND, ctx=ctx)  # torch's own memory is reserved from here on
    del out
    ctx.close()
    ctx = _lib.Context(0)
    before = torch.cuda.mem_get_info()[0]
    got = hydro.sca_d8(flow, ND, ctx=ctx)
    torch.cuda.synchronize()
    used = before - torch.cuda.mem_get_info()[0]
    assert used <= 3 * rows * cols + (4 << 20), used
    ref, _ = pyoracle.sca_d8(d8, ND, False)
    assert np.array_equal(got.cpu().numpy(), ref)
    ctx.close()
