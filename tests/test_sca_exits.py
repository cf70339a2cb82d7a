"""scad8 by tiles, restated on the CPU with small tiles: every tile solved with
its outside inflows taken as done arrivals of area 0, the exits' sums, counts
and flags joined by a walk over the exits, and every tile solved again with
what arrives.  The result must be the oracle's on random codes of every class,
both modes, tiles down to a single cell.
"""
import numpy as np
import pytest

from oracle import pyoracle

ND = -9999.0
OFF = [(-1, -1), (-1, 0), (-1, 1), (0, -1), (0, 0), (0, 1), (1, -1), (1, 0), (1, 1)]


def cells(d8, converge):
    """Per cell: has an area, sources, pending inflows, poisoned, target."""
    rows, cols = d8.shape
    flows = lambda r, c, k: k != 4 and d8[r, c] == k
    inside = lambda r, c: 1 <= r <= rows - 2 and 1 <= c <= cols - 2
    nodata = np.abs(d8 - ND) < 1e-6

    def inflows(r, c):
        found = []
        for k, (dr, dc) in enumerate(OFF):
            u = (r + dr, c + dc)
            if k != 4 and 0 <= u[0] < rows and 0 <= u[1] < cols and flows(*u, 8 - k) and d8[r, c] + (8 - k) != 8:
                found.append((k, u))
        return found

    into = {(r, c): inflows(r, c) if not nodata[r, c] else [] for r in range(rows) for c in range(cols)}
    out = {}
    for r in range(1, rows - 1):
        for c in range(1, cols - 1):
            if nodata[r, c]:
                continue
            nsrc, pend, bad = 0, [], False
            for k, u in into[r, c]:
                if inside(*u) and not nodata[u] and not into[u]:
                    nsrc += 1
                elif inside(*u) and not nodata[u] and (converge or k < 4):
                    pend.append(u)
                else:
                    bad = True
            out[r, c] = dict(area=1 + nsrc, pend=pend, bad=bad)
    target = {u: t for t, s in out.items() for u in s["pend"]}
    return out, target


def settle(members, target, outside, arrived):
    """Areas and done flags of the cells of one tile; `outside` gives what has
    arrived from other tiles per cell: (awaited still, area, not done)."""
    left = {c: sum(u in members for u in s["pend"]) + outside(c)[0] for c, s in members.items()}
    area = {c: s["area"] + outside(c)[1] for c, s in members.items()}
    bad = {c: s["bad"] or outside(c)[2] for c, s in members.items()}
    todo = [c for c in members if left[c] == 0]
    complete = set(todo)
    while todo:
        c = todo.pop()
        t = target.get(c)
        if t in members:
            left[t] -= 1
            if bad[c]:
                bad[t] = True
            else:
                area[t] += area[c]
                arrived[t] = arrived.get(t, 0) + arrived.get(c, 0)
            if left[t] == 0:
                complete.add(t)
                todo.append(t)
    return area, bad, complete


def by_tiles(d8, converge, th, tw):
    info, target = cells(d8, converge)
    tile = lambda c: (c[0] // th, c[1] // tw)
    tiles = {}
    for c in info:
        tiles.setdefault(tile(c), {})[c] = info[c]
    ext = {c: [u for u in s["pend"] if tile(u) != tile(c)] for c, s in info.items()}
    exits, leads = {}, {}
    for members in tiles.values():
        arrived = {c: len(ext[c]) for c in members}  # outside inflows upstream, along done cells
        area, bad, complete = settle(members, target, lambda c: (0, 0, False), arrived)
        for c in members:
            if target.get(c) is not None and target[c] not in members and c in complete:
                exits[c] = dict(area=area[c], left=0 if bad[c] else arrived[c], bad=bad[c])
        for c in members:
            if ext[c]:
                at, steps = c, 0
                while target.get(at) in members and steps < len(members):
                    at, steps = target[at], steps + 1
                leads[c] = at if at in exits else None
    follow = {}
    for e in exits:
        x = leads[target[e]]
        follow[e] = x if x is not None and exits[x]["left"] else None
    todo = [e for e, x in exits.items() if x["left"] == 0]
    while todo:
        e = todo.pop()
        x = follow[e]
        if x is not None:
            exits[x]["area"] += 0 if exits[e]["bad"] else exits[e]["area"]
            exits[x]["bad"] |= exits[e]["bad"]
            exits[x]["left"] -= 1
            if exits[x]["left"] == 0:
                todo.append(x)
    result = np.full(d8.shape, ND)
    done = {}
    for members in tiles.values():
        def outside(c):
            come = [exits[u] for u in ext[c] if u in exits and exits[u]["left"] == 0]
            return (len(ext[c]) - len(come), sum(x["area"] for x in come if not x["bad"]), any(x["bad"] for x in come))

        area, bad, complete = settle(members, target, outside, {})
        for c in members:
            result[c] = area[c]
            done[c] = c in complete and not bad[c]
    rows, cols = d8.shape
    last = (rows - 2, cols - 2)
    if not converge and rows >= 3 and cols >= 3 and last not in info:
        v = result[last]
        for k, (dr, dc) in enumerate(OFF):
            u = (last[0] + dr, last[1] + dc)
            if k != 4 and d8[u] == 8 - k and done.get(u):
                v += result[u]
        result[last] = v
    return result


@pytest.mark.parametrize("seed", range(10))
@pytest.mark.parametrize("converge", [False, True])
def test_tiles_give_the_oracles_areas(seed, converge):
    rng = np.random.default_rng(600 + seed)
    rows, cols = int(rng.integers(3, 26)), int(rng.integers(3, 30))
    weights = [0.05, 0.06, 0.05, 0.06, 0.02, 0.22, 0.16, 0.18, 0.16, 0.02, 0.02] if seed % 2 else [1 / 11] * 11
    d8 = rng.choice([0.0, 1, 2, 3, 4, 5, 6, 7, 8, -1, ND], size=(rows, cols), p=weights)
    ref, _ = pyoracle.sca_d8(d8, ND, converge)
    for th, tw in ((4, 5), (1, 1), (2, 7), (32, 64)):
        got = by_tiles(d8, converge, th, tw)
        assert np.array_equal(got, ref), ((th, tw), np.argwhere(got != ref)[:5].tolist())
