"""pitremove's evaluation, restated on the CPU with small tiles: cells beside
NoData opened at the start, NoData read as +infinity, the update
min(W, max(dem, min over the three rows' h) + gap)) with the cell itself in
the minimum, rows evaluated only when a bit says so, and tiles scheduled with
flags that name the edge, band or corner that changed.  Every variant has to
reach the oracle's values.
"""
import numpy as np
import pytest

from oracle import pyoracle

GAP = 0.0005
INF = np.inf


def opened(dem, nodata):
    """W before the first pass, with NoData as +infinity, and the live cells."""
    rows, cols = dem.shape
    nd = ~(np.abs(dem - nodata) > 1e-6) if np.isfinite(nodata) else np.zeros(dem.shape, bool)
    nd[0], nd[-1], nd[:, 0], nd[:, -1] = True, True, True, True
    near = np.zeros_like(nd)
    for dr in (-1, 0, 1):
        for dc in (-1, 0, 1):
            near[max(0, dr):rows + min(0, dr), max(0, dc):cols + min(0, dc)] |= \
                nd[max(0, -dr):rows + min(0, -dr), max(0, -dc):cols + min(0, -dc)]
    w = np.where(nd, INF, 10000.0)
    if nodata != INF:
        w = np.where(~nd & near, np.minimum(dem, 10000.0), w)
    return w, ~nd, near


def settle(dem, nodata, th, tw, band):
    rows, cols = dem.shape
    w, live, near = opened(dem, nodata)
    floor = np.where(live, dem, INF)
    ty, tx = -(-rows // th), -(-cols // tw)
    flags = {}
    for r, c in np.argwhere(near):
        for y in range(max(0, r - 1) // th, min(rows - 1, r + 1) // th + 1):
            for x in range(max(0, c - 1) // tw, min(cols - 1, c + 1) // tw + 1):
                flags.setdefault((y, x), set()).add("all")
    while flags:
        todo, flags = flags, {}
        for (y, x), why in todo.items():
            r0, c0, r1, c1 = y * th, x * tw, min(rows, y * th + th), min(cols, x * tw + tw)
            pad = np.pad(w, 1, constant_values=INF)
            halo = pad[r0:r1 + 2, c0:c1 + 2]  # the tile and its halo; the tile's part is updated
            h = lambda i: np.minimum(np.minimum(halo[i, :-2], halo[i, 1:-1]), halo[i, 2:])
            n = r1 - r0
            dirty = set(range(n)) if "all" in why else set()
            for f in why:
                if f[0] in "LR":
                    dirty |= set(range(int(f[1:]) * band, min(n, int(f[1:]) * band + band)))
                elif f[0] == "T":
                    dirty.add(0)
                elif f[0] == "B":
                    dirty.add(n - 1)
            changed = np.zeros((n, c1 - c0), bool)
            while dirty:
                i = dirty.pop()
                t = np.maximum(floor[r0 + i, c0:c1], np.minimum(np.minimum(h(i), h(i + 1)), h(i + 2)) + GAP)
                low = t < halo[i + 1, 1:-1]
                if low.any():
                    halo[i + 1, 1:-1] = np.minimum(halo[i + 1, 1:-1], t)
                    changed[i] |= low
                    dirty |= {q for q in (i - 1, i, i + 1) if 0 <= q < n}
            w[r0:r1, c0:c1] = halo[1:-1, 1:-1]

            def flag(dy, dx, name):
                if 0 <= y + dy < ty and 0 <= x + dx < tx:
                    flags.setdefault((y + dy, x + dx), set()).add(name)
            if changed[0].any():
                flag(-1, 0, "B")
            if changed[-1].any():
                flag(1, 0, "T")
            for col, dx, name in ((0, -1, "R"), (-1, 1, "L")):
                for i in np.flatnonzero(changed[:, col]):
                    for q in (i - 1, i, i + 1):
                        if 0 <= q < n:
                            flag(0, dx, "%s%d" % (name, q // band))
                if changed[0, col]:
                    flag(-1, dx, "Bcorner")
                if changed[-1, col]:
                    flag(1, dx, "Tcorner")
    return np.where(live, w, nodata)


@pytest.mark.parametrize("seed", range(8))
@pytest.mark.parametrize("th,tw,band", [(4, 6, 2), (8, 5, 4), (3, 3, 1), (32, 64, 8)])
def test_rows_and_flags_reach_the_oracles_values(seed, th, tw, band):
    rng = np.random.default_rng(900 + seed)
    rows, cols = int(rng.integers(3, 40)), int(rng.integers(3, 45))
    nodata = [-9999.0, 20000.0, np.inf, -np.inf, -9999.0, -9999.0, -3.4028234663852886e38, -9999.0][seed]
    dem = np.round(rng.random((rows, cols)) * 20, 2).astype(np.float32).astype(np.float64)
    if seed % 2 == 0:
        dem += np.add.outer(np.arange(rows), np.arange(cols)) * 0.25
    dem[rng.random(dem.shape) < 0.03] = 12000.0
    if np.isfinite(nodata):
        dem[rng.random(dem.shape) < 0.02] = nodata
    ref, _, ok = pyoracle.pit_remove(dem, nodata)
    assert ok
    got = settle(dem, nodata, th, tw, band)
    assert np.array_equal(got, ref), np.argwhere(got != ref)[:5].tolist()
