"""GPU parity of the contributing area where its 64 x 32 tiles meet, bit for
bit: sizes on either side of tile edges, one path through every cell of a
tile and on through its neighbours, cycles of codes inside a tile and across
an edge, and areas that must not cross an edge (not done in the one-sweep
order, or a border cell draining inward).
"""
import numpy as np
import pytest

from oracle import pyoracle
from tests.test_gpu_sca import ND, OFF, gpu_from_double

pytestmark = pytest.mark.gpu

CODE = {(dr, dc): k for k, (dr, dc) in enumerate(OFF)}


def check(d8, pad=0):
    for mode in ("reference", "converge"):
        ref, _ = pyoracle.sca_d8(d8, ND, mode == "converge")
        got = gpu_from_double(d8, ND, mode, pitch_pad=pad)
        assert np.array_equal(got, ref), (mode, np.argwhere(got != ref)[:5].tolist())


def along(cells, shape, fill=-1.0):
    """A raster whose cells drain along a list of neighbouring cells."""
    d8 = np.full(shape, fill)
    for (r, c), (r1, c1) in zip(cells, cells[1:]):
        d8[r, c] = CODE[(r1 - r, c1 - c)]
    return d8


def snake(r0, r1, c0, c1):
    return [(r, c) for i, r in enumerate(range(r0, r1)) for c in (range(c0, c1) if i % 2 == 0 else range(c1 - 1, c0 - 1, -1))]


@pytest.mark.parametrize("rows,cols", [(1, 1), (2, 3), (3, 3), (31, 63), (32, 64), (33, 65), (34, 66), (64, 128),
                                       (65, 129), (66, 130), (97, 203), (130, 76), (35, 300)])
def test_random_codes_around_tile_sizes(rows, cols):
    rng = np.random.default_rng(31 * rows + cols)
    # mostly southward and eastward codes, so that long chains cross tiles
    d8 = rng.choice([0, 1, 2, 3, 5, 6, 7, 8, 5, 7, 8, 7, -1, ND], size=(rows, cols)).astype(float)
    check(d8, cols % 3)


@pytest.mark.parametrize("flip", [False, True])
def test_one_path_through_every_cell(flip):
    cells = snake(1, 99, 1, 199)
    check(along(cells[::-1] if flip else cells, (100, 200)))


@pytest.mark.parametrize("at", [(31, 63), (32, 64), (40, 63), (63, 127), (20, 20)])
def test_cycles_and_what_drains_into_them(at):
    r, c = at
    rng = np.random.default_rng(r * 7 + c)
    d8 = rng.choice([5.0, 6.0, 7.0, 8.0], size=(100, 200))
    for a, b in zip([(0, 0), (0, 1), (1, 1), (1, 0)], [(0, 1), (1, 1), (1, 0), (0, 0)]):
        d8[r + a[0], c + a[1]] = CODE[(b[0] - a[0], b[1] - a[1])]
    check(d8)


def test_not_done_across_edges():
    # chains that run against the sweep order (north and west) between ones
    # that run with it, and border cells draining inward
    rng = np.random.default_rng(3)
    d8 = np.where(rng.random((140, 210)) < 0.15, rng.choice([0.0, 1.0, 2.0, 3.0], size=(140, 210)),
                  rng.choice([5.0, 6.0, 7.0, 8.0], size=(140, 210)))
    d8[0], d8[:, 0], d8[-1], d8[:, -1] = 7.0, 5.0, 1.0, 3.0
    d8[rng.random(d8.shape) < 0.02] = ND
    check(d8)


def test_last_cell_in_the_corner_of_a_tile():
    # the last work cell NoData, in the first row and column of its tile
    rng = np.random.default_rng(9)
    for rows, cols in ((34, 66), (33, 65), (98, 130)):
        d8 = rng.choice([5.0, 7.0, 8.0], size=(rows, cols))
        d8[rows - 2, cols - 2] = ND
        d8[rows - 3, cols - 3], d8[rows - 3, cols - 2], d8[rows - 2, cols - 3] = 8.0, 7.0, 5.0
        check(d8)
