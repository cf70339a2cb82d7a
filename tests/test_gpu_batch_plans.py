"""Batch plans one after the other on a context: the plan's device copy is
shared and uploaded in stream order, the first run of a plan is launched as it
is, later ones replay its graph, and a caller's capture takes the launches.
"""
import pytest

from pargo_amd import _lib, batch, focal
from tests.test_gpu_batch import make_tiles

pytestmark = pytest.mark.gpu


def expected(dems):
    return [focal.slope_d8(d, 30.0, -9999.0) for d in dems]


def check(b, ref):
    import torch
    for s, c, (rs, rc, _) in zip(b.slopes, b.codes, ref):
        assert torch.equal(s, rs) and torch.equal(c, rc)


def clear(b):
    for s, c in zip(b.slopes, b.codes):
        s.zero_()
        c.zero_()


def test_plans_in_turn_without_waiting():
    import torch
    ctx = _lib.Context(0)
    sets = [make_tiles(n, 40 + n, 20, 500) for n in (3, 17, 40)]
    refs = [expected(d) for d in sets]
    bs = [batch.Batch(d, ctx=ctx) for d in sets]
    for _ in range(3):
        for b in bs:
            clear(b)
        for b in bs + bs[::-1]:  # no synchronisation in between
            b.run(batch.GRAPH)
        torch.cuda.synchronize()
        for b, r in zip(bs, refs):
            check(b, r)
    ctx.close()


@pytest.mark.parametrize("runs", [1, 2])
def test_run_inside_a_callers_capture(runs):
    import torch
    ctx = _lib.Context(0)
    dems = make_tiles(12, 77, 20, 400)
    ref = expected(dems)
    b = batch.Batch(dems, ctx=ctx)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for _ in range(runs):
            b.run(batch.GRAPH)
        stream.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            b.run(batch.GRAPH)
        for _ in range(3):
            clear(b)
            g.replay()
            stream.synchronize()
            check(b, ref)
            expected(dems[:2])  # other work in between
            stream.synchronize()
    ctx.close()
