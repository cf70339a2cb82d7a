"""The measured cases: what programs that use pargo_amd have it do.

A case is a dict of plain values; "op" says which entry point it calls and
the other keys are that call's sizes and options.  prepare(case, seed) makes
what a program holds before the call, run(state) is one pass through the
public entry points, work(case) the bytes and operations the pass cannot do
without, and exact(case, seed) the same outputs in 64 bits by plain torch.

Rasters follow the repository's own recipe (fractal DEM, 2 % plateaus, 1 %
NoData discs, pargo_amd.synth) and IDW samples its sample recipe (half
uniform, half clustered); only the seeds and sizes differ.
"""
import math

import torch

from pargo_amd import autograd, batch, focal, hydro, idw, synth

CELL = 30.0
NODATA = -9999.0
DEV = "cuda"


def listed():
    return [
        # One map tile as a tile server or a test asks for it: launch-bound.
        {"name": "tile_256", "op": "focal", "rows": 256, "cols": 256, "method": "FD", "unit": "tan", "slope": True,
         "dirtype": 256, "mask": False},
        # The slope program's own small raster (the 1024 x 1024 workload).
        {"name": "slope_1k", "op": "focal", "rows": 1024, "cols": 1024, "method": "FD", "unit": "tan", "slope": True,
         "dirtype": 0, "mask": False},
        # The headline benchmark: slope and D8 of a whole sheet in one pass.
        {"name": "slope_d8_16k", "op": "focal", "rows": 16384, "cols": 16384, "method": "FD", "unit": "tan",
         "slope": True, "dirtype": 256, "mask": False},
        # A ragged raster with the options the programs offer: another slope
        # method, degrees, the dirType-8 codes and NoData mask scad8 reads.
        {"name": "methods_ragged", "op": "focal", "rows": 7001, "cols": 5003, "method": "TFDW", "unit": "degrees",
         "slope": True, "dirtype": 8, "mask": True},
        # A differentiable slope layer in a fitting loop: forward and backward.
        {"name": "slope_grad_8k", "op": "slope_grad", "rows": 8192, "cols": 8192},
        # Interpolation of 20,000 stations onto a 4096 x 4096 grid.
        {"name": "idw_4k", "op": "idw", "rows": 4096, "cols": 4096, "samples": 20000, "k": 12, "power": 2,
         "buffer": 5000.0, "block": 5000.0},
        # Fitting station values through the interpolated grid: one step.
        {"name": "idw_grad_ragged", "op": "idw_grad", "rows": 1101, "cols": 1503, "samples": 2000, "k": 8, "power": 2,
         "buffer": 5000.0, "block": 5000.0},
        # Many uneven rasters at once (a mosaic's tiles) through the batch graph.
        {"name": "batch_32", "op": "batch", "tiles": 32, "side_min": 256, "side_max": 4096},
        # Contributing area of the headline sheet's D8 codes, the reference's sweep.
        {"name": "sca_16k", "op": "sca", "rows": 16384, "cols": 16384, "mode": "reference", "layer": False},
        # scad8 as its operator runs it: a float64 code layer read from a
        # file, classified, then the full flow accumulation.
        {"name": "sca_layer_ragged", "op": "sca", "rows": 5003, "cols": 7001, "mode": "converge", "layer": True},
        # Depression filling of the headline sheet.
        {"name": "pit_16k", "op": "pit", "rows": 16384, "cols": 16384},
        # The hydrology chain on a ragged catchment: fill, D8, accumulation.
        {"name": "chain_ragged", "op": "chain", "rows": 1501, "cols": 2003, "mode": "converge"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, lo, hi):
    """A raster of side lo .. hi (log-uniform) and aspect 1/2 .. 2."""
    side, aspect = _log_int(rng, lo, hi), math.exp(rng.uniform(-0.69, 0.69))
    return max(64, int(side * math.sqrt(aspect))), max(64, int(side / math.sqrt(aspect)))


def draw(rng):
    op = rng.choice(["focal", "focal", "focal", "slope_grad", "idw", "idw_grad", "batch", "sca", "sca", "pit", "chain"])
    if op == "focal":
        rows, cols = _shape(rng, 96, 12000)
        what = rng.choice(["both", "both", "slope", "d8"])
        return {"op": op, "rows": rows, "cols": cols,
                "method": rng.choice(["FD", "FD", "FFD", "MD", "SD", "SFD", "TFD", "TFDW"]),
                "unit": rng.choice(["tan", "tan", "degrees"]), "slope": what != "d8",
                "dirtype": 0 if what == "slope" else rng.choice([8, 256]), "mask": rng.random() < 0.5}
    if op == "slope_grad":
        rows, cols = _shape(rng, 256, 8192)
        return {"op": op, "rows": rows, "cols": cols}
    if op in ("idw", "idw_grad"):
        rows, cols = _shape(rng, 256, 4096)
        # 500 .. 2000 samples per 1000 x 1000 cells, the recipe's 1200 between
        n = max(50, int(rows * cols * 1e-6 * _log_int(rng, 500, 2000)))
        return {"op": op, "rows": rows, "cols": cols, "samples": n, "k": rng.randint(4, 16), "power": rng.choice([1, 2, 2, 3]),
                "buffer": float(rng.choice([3000, 5000, 8000])), "block": float(rng.choice([3000, 5000]))}
    if op == "batch":
        lo = _log_int(rng, 64, 512)
        return {"op": op, "tiles": _log_int(rng, 4, 32), "side_min": lo, "side_max": lo * rng.randint(2, 8)}
    if op == "sca":
        rows, cols = _shape(rng, 200, 12000)
        return {"op": op, "rows": rows, "cols": cols, "mode": rng.choice(["reference", "converge"]),
                "layer": rows * cols < 40_000_000 and rng.random() < 0.5}
    if op == "pit":
        rows, cols = _shape(rng, 200, 12000)
        return {"op": op, "rows": rows, "cols": cols}
    rows, cols = _shape(rng, 200, 3000)
    return {"op": op, "rows": rows, "cols": cols, "mode": rng.choice(["reference", "converge"])}


# ---- inputs ----------------------------------------------------------------

def _dem(rows, cols, seed):
    return torch.from_numpy(synth.workload_dem("slope_d8", rows, cols, synth.BASE_SEED + 7919 * seed)).to(DEV)


def _randn(shape, seed):
    return torch.randn(shape, dtype=torch.float32, device=DEV, generator=torch.Generator(DEV).manual_seed(seed))


def _samples(case, seed):
    return synth.samples(synth.BASE_SEED + 7919 * seed, case["samples"], width=case["cols"] * CELL,
                         height=case["rows"] * CELL, cellsize=CELL)


def _batch_dems(case, seed):
    # the workload's own shapes depend on the seed; here every seed has the
    # same ones, so that a case is one amount of work
    shapes = batch.tile_shapes(case["tiles"], 41, case["side_min"], case["side_max"])
    return [_dem(r, c, seed * 1000 + t) for t, (r, c) in enumerate(shapes)]


def prepare(case, seed):
    op = case["op"]
    s = {"case": case}
    if op in ("focal", "pit", "chain"):
        s["dem"] = _dem(case["rows"], case["cols"], seed)
    elif op == "slope_grad":
        s["dem"] = _dem(case["rows"], case["cols"], seed).requires_grad_(True)
        s["grad"] = _randn((case["rows"], case["cols"]), seed)
    elif op in ("idw", "idw_grad"):
        xs, ys, vals = _samples(case, seed)
        s["op"] = idw.IDWOperator(CELL, case["k"], case["power"], case["buffer"], case["block"]).read_samples(xs, ys, vals)
        if op == "idw_grad":
            s["values"] = torch.from_numpy(vals).to(DEV).requires_grad_(True)
            s["grad"] = _randn((s["op"].rows, s["op"].cols), seed)
    elif op == "batch":
        s["batch"] = batch.Batch(_batch_dems(case, seed), CELL, NODATA)
    elif op == "sca":
        code, mask = focal.d8(_dem(case["rows"], case["cols"], seed), CELL, NODATA, 8, want_mask=True)
        if case["layer"]:
            s["layer"] = focal.codes_to_reference(code, focal.unpack_mask(mask, case["cols"]), 8, NODATA)
        else:
            s["code"], s["mask"] = code, mask
    return s


def run(state):
    c = state["case"]
    op = c["op"]
    if op == "focal":
        return focal.slope_d8(state["dem"], CELL, NODATA, c["method"], c["unit"], c["dirtype"] or 256, c["slope"],
                              c["dirtype"] != 0, c["mask"])
    if op == "slope_grad":
        s = autograd.slope(state["dem"], CELL, NODATA)
        return (s.detach(), *torch.autograd.grad(s, state["dem"], state["grad"]))
    if op == "idw":
        return state["op"].run()
    if op == "idw_grad":
        out = autograd.idw(state["values"], state["op"])
        return (out.detach(), *torch.autograd.grad(out, state["values"], state["grad"]))
    if op == "batch":
        return state["batch"].run()
    if op == "sca":
        if c["layer"]:
            return hydro.SCAOperator(c["mode"]).d8_layer(state["layer"], NODATA).run()
        return hydro.sca_d8(state["code"], NODATA, state["mask"], c["mode"])
    if op == "pit":
        return hydro.pit_remove(state["dem"], NODATA)[0]
    # the chain: the filled DEM goes on as the float32 raster flowdird8 reads
    filled, _ = hydro.pit_remove(state["dem"], NODATA)
    code, mask = focal.d8(filled.float(), CELL, NODATA, 8, want_mask=True)
    return filled, code, mask, hydro.sca_d8(code, NODATA, mask, c["mode"])


# ---- what a pass cannot do without ----------------------------------------

def work(case):
    op = case["op"]
    if op == "batch":
        cells = sum(r * c for r, c in batch.tile_shapes(case["tiles"], 41, case["side_min"], case["side_max"]))
        return {"bytes": 9 * cells, "flops": 40 * cells}
    cells = case["rows"] * case["cols"]
    if op == "focal":
        per = 4 + (4 if case["slope"] else 0) + (1 if case["dirtype"] else 0) + (0.125 if case["mask"] else 0)
        return {"bytes": int(per * cells), "flops": cells * ((20 if case["slope"] else 0) + (20 if case["dirtype"] else 0))}
    if op == "slope_grad":  # forward: z in, s out; backward: z and ds in, dz out
        return {"bytes": 20 * cells, "flops": 60 * cells}
    if op in ("idw", "idw_grad"):
        # every cell needs its k nearest samples' distances and weights
        per = 10 * case["k"] * (2 if op == "idw_grad" else 1)
        return {"bytes": (4 if op == "idw" else 8) * cells + 24 * case["samples"], "flops": per * cells}
    if op == "sca":  # a code (1 B and a mask bit, or a double) in, a double out
        return {"bytes": int((16 if case["layer"] else 9.125) * cells), "flops": cells}
    if op == "pit":
        return {"bytes": 12 * cells, "flops": 9 * cells}
    return {"bytes": int((12 + 12 + 5.125 + 9.125) * cells), "flops": 30 * cells}


# ---- 64-bit results by plain torch ------------------------------------------

def _window(z):
    """The 3 x 3 window of every interior cell, row-major."""
    r, c = z.shape
    return [z[i:r - 2 + i, j:c - 2 + j] for i in range(3) for j in range(3)]


def _bands(rows, step=1024):
    for r0 in range(1, rows - 1, step):
        yield r0, min(r0 + step, rows - 1)


def _slope64(dem, method, unit):
    out = torch.full(dem.shape, NODATA, dtype=torch.float64, device=dem.device)
    q = math.sqrt(2.0)
    for r0, r1 in _bands(dem.shape[0]):
        d = _window(dem[r0 - 1:r1 + 1].double())
        if method == "MD":
            m = torch.zeros_like(d[4])
            for k in (0, 1, 2, 3, 5, 6, 7, 8):
                m = torch.maximum(m, d[4] - d[k])
            s = m / (CELL * q)
        else:
            if method == "FFD":
                dx, dy, k = d[8] - d[6] + d[2] - d[0], d[0] - d[6] + d[2] - d[8], 4.0
            elif method == "SD":
                dx, dy, k = d[4] - d[3], d[4] - d[7], 1.0
            elif method == "SFD":
                dx, dy, k = d[5] - d[3], d[1] - d[7], 2.0
            elif method == "TFD":  # d[6] twice, as the operator defines it
                dx, dy, k = d[8] + d[5] + d[2] - d[0] - d[3] - d[6], d[2] + d[1] + d[0] - d[6] - d[7] - d[6], 6.0
            else:
                w, k = (q, 4.0 + math.sqrt(8.0)) if method == "TFDW" else (2.0, 8.0)
                dx = d[8] + w * d[5] + d[2] - d[6] - w * d[3] - d[0]
                dy = d[2] + w * d[1] + d[0] - d[6] - w * d[7] - d[8]
            s = torch.sqrt(dx * dx + dy * dy) / (k * CELL)
        if unit == "degrees":
            s = torch.rad2deg(torch.atan(s))
        nd = torch.zeros_like(d[4], dtype=torch.bool)
        for v in d:
            nd |= (v - NODATA).abs() < 1e-7
        out[r0:r1, 1:-1] = torch.where(nd, NODATA, s)
    return out


def _slope_grad64(dem, grad):
    """(slope, dL/dz) of the Horn slope; cells without a slope or with none
    of its gradient defined contribute 0."""
    z = dem.double()
    d = _window(z)
    dx = (d[8] + 2 * d[5] + d[2] - d[6] - 2 * d[3] - d[0]) / (8 * CELL)
    dy = (d[2] + 2 * d[1] + d[0] - d[6] - 2 * d[7] - d[8]) / (8 * CELL)
    nd = torch.zeros_like(d[4], dtype=torch.bool)
    for v in d:
        nd |= (v - NODATA).abs() < 1e-7
    del d
    s = torch.sqrt(dx * dx + dy * dy)
    f = torch.where(nd | (s == 0), 0.0, grad[1:-1, 1:-1].double() / (s * 8 * CELL))
    dx, dy = f * dx, f * dy
    out = torch.zeros_like(z)
    r, c = z.shape
    wx, wy = (-1, 0, 1, -2, 0, 2, -1, 0, 1), (1, 2, 1, 0, 0, 0, -1, -2, -1)
    for k in range(9):
        if k != 4:
            out[k // 3:r - 2 + k // 3, k % 3:c - 2 + k % 3] += wx[k] * dx + wy[k] * dy
    slope = torch.full_like(z, NODATA)
    slope[1:-1, 1:-1] = torch.where(nd, NODATA, s)
    return slope, out


def _d8_64(dem):
    """dirType-8 codes (255: flat) and the NoData set, on the 64-bit drops."""
    code = torch.full(dem.shape, 255, dtype=torch.uint8, device=dem.device)
    nodata = torch.ones(dem.shape, dtype=torch.bool, device=dem.device)
    for r0, r1 in _bands(dem.shape[0]):
        d = _window(dem[r0 - 1:r1 + 1].double())
        nd = torch.zeros_like(d[4], dtype=torch.bool)
        for v in d:
            nd |= (v - NODATA).abs() < 1e-6
        drop = [(d[4] - v) / math.sqrt(2.0) if k in (0, 2, 6, 8) else d[4] - v for k, v in enumerate(d)]
        top = torch.zeros_like(d[4])
        for v in drop:
            top = torch.maximum(top, v)
        tied = torch.stack([(v - top).abs() < 1e-6 for v in drop])
        rank = tied.cumsum(0)
        half = rank[-1] // 2 + 1  # the median tied window index
        pick = (tied & (rank == half)).to(torch.uint8).argmax(0).to(torch.uint8)
        code[r0:r1, 1:-1] = torch.where(top < 1e-6, 255, pick).to(torch.uint8)
        nodata[r0:r1, 1:-1] = nd
    return code, nodata


def _sca64(code, nodata, mode):
    """Contributing area by waves of completed cells."""
    rows, cols = code.shape
    n = rows * cols
    c, valid = code.flatten(), ~nodata.flatten()
    off = torch.tensor([(k // 3 - 1) * cols + k % 3 - 1 for k in range(9)], device=DEV)
    u = torch.nonzero(valid & (c < 9) & (c != 4)).flatten()
    t = u + off[c[u].long()]
    keep = valid[t] & (c[t].int() + c[u].int() != 8)
    u, t = u[keep], t[keep]
    fed = torch.zeros(n, dtype=torch.bool, device=DEV)
    fed[t] = True
    source = ~fed[u]
    early = c[u] > 4  # the cell precedes its target in row-major order
    area = valid.long()
    area.index_add_(0, t[source], torch.ones_like(t[source]))
    waits = ~source & (early if mode == "reference" else torch.ones_like(early))
    bad = torch.zeros(n, dtype=torch.bool, device=DEV)
    bad[t[~source & ~waits]] = True
    pending = torch.zeros(n, dtype=torch.int32, device=DEV)
    pending.index_add_(0, t[waits], torch.ones_like(t[waits], dtype=torch.int32))
    target = torch.full((n,), -1, dtype=torch.int64, device=DEV)
    target[u[waits]] = t[waits]
    del u, t, keep, source, early, waits
    front = torch.nonzero((target >= 0) & (pending == 0)).flatten()
    first = torch.empty(n, dtype=torch.int64, device=DEV)
    while front.numel():
        to = target[front]
        ok = ~bad[front]
        area.index_add_(0, to, area[front] * ok)
        bad[to[~ok]] = True
        pending.index_add_(0, to, torch.full_like(to, -1, dtype=torch.int32))
        to = to[pending[to] == 0]
        at = torch.arange(to.numel(), device=DEV)
        first[to] = at
        to = to[first[to] == at]  # each completed cell once
        front = to[target[to] >= 0]
    out = torch.where(valid, area.double(), NODATA).reshape(rows, cols)
    r, q = rows - 2, cols - 2
    if mode == "reference" and bool(nodata[r, q]):
        # the sweep's last work cell adds its finished inflows to NoData
        v = NODATA
        for k in (0, 1, 2, 3, 5, 6, 7, 8):
            i, j = r + k // 3 - 1, q + k % 3 - 1
            if not bool(nodata[i, j]) and int(code[i, j]) == 8 - k and not bool(bad[i * cols + j]) \
                    and int(pending[i * cols + j]) == 0:
                v += float(area[i * cols + j])
        out[r, q] = v
    return out


def _pit64(dem):
    """Filled DEM: the settled state of the operator's update."""
    z = dem.double()
    nd = (z - NODATA).abs() <= 1e-6
    nd[0], nd[-1], nd[:, 0], nd[:, -1] = True, True, True, True
    w = torch.full_like(z, 10000.0)
    w[nd] = -math.inf  # a NoData neighbour gives a cell its own elevation
    floor, live = z[1:-1, 1:-1], ~nd[1:-1, 1:-1]
    while True:
        before = w.clone()
        for _ in range(64):
            m = torch.minimum(torch.minimum(w[:, :-2], w[:, 1:-1]), w[:, 2:])
            m = torch.minimum(torch.minimum(m[:-2], m[1:-1]), m[2:]) + 0.0005
            w[1:-1, 1:-1] = torch.where(live, torch.minimum(w[1:-1, 1:-1], torch.maximum(floor, m)), w[1:-1, 1:-1])
        if torch.equal(before, w):
            return torch.where(nd, NODATA, w)


def _idw64(case, seed, grad=None):
    """The grid and, with grad, dL/d(values): for each block of cells the
    rings of sample blocks around it, each cell stopping by its own distance."""
    xs, ys, vals = (torch.from_numpy(a).to(DEV) for a in _samples(case, seed))
    k, power, buf, size = case["k"], case["power"], case["buffer"], case["block"]
    x0, y0 = float(xs.min()) - CELL / 2, float(ys.min()) - CELL / 2
    cols, rows = int((float(xs.max()) - x0) / CELL), int((float(ys.max()) - y0) / CELL)
    cols += float(xs.max()) - x0 != cols * CELL
    rows += float(ys.max()) - y0 != rows * CELL
    y1 = y0 + CELL * rows
    sr, sc = ((y1 - ys) / size).long(), ((xs - x0) / size).long()
    cx = (torch.arange(cols, device=DEV, dtype=torch.float64) + 0.5) * CELL + x0
    cy = y1 - (torch.arange(rows, device=DEV, dtype=torch.float64) + 0.5) * CELL
    br, bc = ((y1 - cy) / size).long(), ((cx - x0) / size).long()
    out = torch.zeros((rows, cols), dtype=torch.float64, device=DEV)
    gv = torch.zeros_like(vals)
    most = int(max(br.max(), bc.max(), sr.max(), sc.max())) + 1
    for b in range(int(br.max()) + 1):
        for a in range(int(bc.max()) + 1):
            rr, cc = torch.nonzero(br == b).flatten(), torch.nonzero(bc == a).flatten()
            if not rr.numel() or not cc.numel():
                continue
            y, x = (v.flatten() for v in torch.meshgrid(cy[rr], cx[cc], indexing="ij"))
            edge = torch.minimum(torch.minimum((x - (a * size + x0)).abs(), (x - ((a + 1) * size + x0)).abs()),
                                 torch.minimum((y - (y1 - b * size)).abs(), (y - (y1 - (b + 1) * size)).abs()))
            dist = torch.full((x.numel(), k), math.inf, dtype=torch.float64, device=DEV)
            who = torch.zeros((x.numel(), k), dtype=torch.int64, device=DEV)
            ring_of = torch.maximum((sr - b).abs(), (sc - a).abs())
            live, seen = torch.ones_like(x, dtype=torch.bool), 0
            for ring in range(most + 1):
                reach = (ring - 1) * size + edge
                if buf > 0:
                    live = live & (reach < buf)
                if not bool(live.any()):
                    break
                s = torch.nonzero(ring_of == ring).flatten()
                seen += s.numel()
                if s.numel():
                    at = torch.nonzero(live).flatten()
                    for part in at.split(max(1, 50_000_000 // s.numel())):
                        d = torch.sqrt((xs[s][None] - x[part, None]) ** 2 + (ys[s][None] - y[part, None]) ** 2)
                        d = torch.where(d == 0, 1e-7, d)
                        best, i = d.topk(min(k, s.numel()), 1, largest=False)
                        both, ids = torch.cat([dist[part], best], 1), torch.cat([who[part], s[i]], 1)
                        dist[part], j = both.topk(k, 1, largest=False)
                        who[part] = ids.gather(1, j)
                if seen >= k:
                    live = live & (reach < dist[:, -1])
            w = torch.where(dist.isfinite(), dist, 1.0) ** -power * dist.isfinite()
            w = w / torch.where(w.sum(1) > 0, w.sum(1), 1.0)[:, None]
            cells = rr[:, None] * cols + cc[None]
            out.view(-1)[cells.flatten()] = (w * vals[who]).sum(1)
            if grad is not None:
                g = grad.view(-1)[cells.flatten()].double()
                gv.index_add_(0, who.flatten(), (w * g[:, None]).flatten())
    return (out, gv) if grad is not None else out


def exact(case, seed):
    op = case["op"]
    if op == "focal":
        if not case["slope"]:
            return None  # codes and mask words alone
        return _slope64(_dem(case["rows"], case["cols"], seed), case["method"], case["unit"]), None, None
    if op == "slope_grad":
        return _slope_grad64(_dem(case["rows"], case["cols"], seed), _randn((case["rows"], case["cols"]), seed))
    if op == "idw":
        return _idw64(case, seed)
    if op == "idw_grad":
        xs, ys, _ = _samples(case, seed)
        rows, cols, _, _ = idw.grid(xs, ys, CELL)
        return _idw64(case, seed, _randn((rows, cols), seed))
    if op == "batch":
        dems = _batch_dems(case, seed)
        return [_slope64(d, "FD", "tan") for d in dems], [None] * len(dems)
    if op == "sca":
        return _sca64(*_d8_64(_dem(case["rows"], case["cols"], seed)), case["mode"])
    if case["rows"] * case["cols"] > 10_000_000:
        return None  # thousands of whole-grid sweeps
    filled = _pit64(_dem(case["rows"], case["cols"], seed))
    if op == "pit":
        return filled
    code, nodata = _d8_64(filled.float())
    return filled, None, None, _sca64(code, nodata, case["mode"])
