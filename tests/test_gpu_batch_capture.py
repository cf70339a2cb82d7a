"""A batch in a caller's graph: the plan it captured stays as it was while the
context runs other batches, smaller, larger or in another order, and a batch
that cannot be captured leaves the caller's capture and the plan alone.
"""
import pytest

from pargo_amd import _lib, batch
from tests.test_gpu_batch import make_tiles
from tests.test_gpu_batch_plans import check, clear, expected

pytestmark = pytest.mark.gpu


def tiles(n, seed, lo, hi):
    dems = make_tiles(n, seed, lo, hi)
    for d in dems[::3]:
        d[7, 9], d[11, 3] = -2e13, 3e13  # strips for the exact pass
    return dems


def capture(b, stream, mode):
    import torch
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        b.run(mode)
    return g


@pytest.mark.parametrize("mode", [batch.PERSISTENT, batch.GRAPH, batch.PER_TILE])
def test_replays_between_other_plans(mode):
    import torch
    ctx = _lib.Context(0)
    sets = [tiles(12, 81, 20, 400), tiles(3, 82, 30, 60), tiles(60, 83, 20, 300)]
    refs = [expected(d) for d in sets]
    a, small, large = [batch.Batch(d, ctx=ctx) for d in sets]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        a.run(mode)
        graphs = [(capture(a, stream, mode), a, refs[0])]
        for other, ref in ((small, refs[1]), (large, refs[2]), (small, refs[1])):
            for _ in range(2):
                other.run(batch.GRAPH)
            for g, b, r in graphs:
                for x in (a, other):
                    clear(x)
                g.replay()
                other.run(mode)
                stream.synchronize()
                check(b, r)
                check(other, ref)
        # a second plan captured, and the first one captured once more
        graphs.append((capture(small, stream, mode), small, refs[1]))
        a.run(mode)
        graphs.append((capture(a, stream, mode), a, refs[0]))
        large.run(mode)
        for _ in range(3):
            for g, b, r in graphs:
                clear(b)
                g.replay()
                stream.synchronize()
                check(b, r)
    ctx.close()


def test_a_first_run_is_refused_and_the_capture_goes_on():
    import torch
    ctx = _lib.Context(0)
    sets = [tiles(9, 84, 20, 300), tiles(20, 85, 20, 300)]
    refs = [expected(d) for d in sets]
    a, b = [batch.Batch(d, ctx=ctx) for d in sets]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(3):
            a.run(batch.GRAPH)  # the plan holds a graph of its own by now
        stream.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            with pytest.raises(_lib.PargoError, match="cannot be captured"):
                b.run(batch.GRAPH)
            a.run(batch.GRAPH)
        b.run(batch.GRAPH)
        for _ in range(3):
            clear(a)
            g.replay()
            stream.synchronize()
            check(a, refs[0])
            check(b, refs[1])
    ctx.close()
