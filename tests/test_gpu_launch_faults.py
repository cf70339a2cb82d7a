"""A launch that fails between a kernel that fills a device queue and the pass
that empties it: the call reports it, and the next call on the context does
not see what the queues were left holding (work items skipped, strips of other
rasters).  PARGO_FAIL_LAUNCH makes the chosen launch fail before it is made.
"""
import os

import pytest

from pargo_amd import _lib, batch, focal
from tests.test_gpu_batch_capture import tiles
from tests.test_gpu_batch_plans import check, clear, expected

pytestmark = pytest.mark.gpu

_gen = [0]


class failing_launch:
    """The n-th launch of a queue-emptying pass inside the block fails."""

    def __init__(self, n=1):
        self.n = n

    def __enter__(self):
        _gen[0] += 1
        os.environ["PARGO_FAIL_LAUNCH"] = "%d:%d" % (self.n, _gen[0])

    def __exit__(self, *exc):
        os.environ.pop("PARGO_FAIL_LAUNCH", None)


@pytest.mark.parametrize("mode", [batch.PERSISTENT, batch.GRAPH, batch.PER_TILE])
@pytest.mark.parametrize("runs_before", [0, 1, 2])
def test_batch_after_a_failed_fixup_launch(mode, runs_before):
    import torch
    ctx = _lib.Context(0)
    # enough wave-rows that the waves take items from the queue
    dems = tiles(64, 91, 300, 800)
    ref = expected(dems)
    b = batch.Batch(dems, ctx=ctx)
    for _ in range(runs_before):
        b.run(mode)
    with failing_launch(7 if mode == batch.PER_TILE else 1):
        if mode == batch.GRAPH and runs_before == 2:
            b.run(mode)  # a replay makes no launch of its own
        else:
            with pytest.raises(_lib.PargoError, match="injected at fixup pass"):
                b.run(mode)
    for _ in range(3):
        clear(b)
        b.run(mode)
        torch.cuda.synchronize()
        check(b, ref)
    ctx.close()


def test_rasters_and_batches_share_the_queue():
    # a batch whose strips for the exact pass stay in the queue, then a single
    # raster that uses it, and the other way round
    import torch
    ctx = _lib.Context(0)
    dems = tiles(64, 92, 300, 800)
    big = torch.from_numpy(batch.tile_dem(3, 2049, 2050)).cuda()
    big[1000, 1000], big[5, 2040] = 3e13, -2e13
    refs, (rs, rc, _) = expected(dems), focal.slope_d8(big, 30.0, -9999.0)
    b = batch.Batch(dems, ctx=ctx)
    for _ in range(2):
        with failing_launch(), pytest.raises(_lib.PargoError, match="injected at fixup pass"):
            b.run(batch.PERSISTENT)
        s, c, _ = focal.slope_d8(big, 30.0, -9999.0, ctx=ctx)
        torch.cuda.synchronize()
        assert torch.equal(s, rs) and torch.equal(c, rc)
        b.run(batch.GRAPH)
        with failing_launch(), pytest.raises(_lib.PargoError, match="injected at fixup pass"):
            focal.slope_d8(big, 30.0, -9999.0, ctx=ctx)
        clear(b)
        b.run(batch.GRAPH)
        torch.cuda.synchronize()
        check(b, refs)
    ctx.close()
