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


def failing_context(n):
    """A context whose n-th launch of a queue-emptying pass fails."""
    os.environ["PARGO_FAIL_LAUNCH"] = str(n)
    try:
        return _lib.Context(0)
    finally:
        del os.environ["PARGO_FAIL_LAUNCH"]


@pytest.mark.parametrize("mode,runs_before", [(batch.PERSISTENT, 0), (batch.PERSISTENT, 2), (batch.GRAPH, 0),
                                              (batch.GRAPH, 1), (batch.PER_TILE, 0), (batch.PER_TILE, 1)])
def test_batch_after_a_failed_fixup_launch(mode, runs_before):
    import torch
    # enough wave-rows that the waves take items from the queue
    dems = tiles(64, 91, 300, 800)
    ref = expected(dems)
    # (the second run in graph mode captures the launches)
    ctx = failing_context(64 * runs_before + 7 if mode == batch.PER_TILE else runs_before + 1)
    b = batch.Batch(dems, ctx=ctx)
    for _ in range(runs_before):
        b.run(mode)
    with pytest.raises(_lib.PargoError, match="launch failure"):
        b.run(mode)
    for _ in range(3):
        clear(b)
        b.run(mode)
        torch.cuda.synchronize()
        check(b, ref)
    ctx.close()


@pytest.mark.parametrize("fails", ["batch", "raster"])
def test_rasters_and_batches_share_the_queue(fails):
    # a batch whose strips for the exact pass stay in the queue, then a single
    # raster that uses it, and the other way round
    import torch
    dems = tiles(64, 92, 300, 800)
    big = torch.from_numpy(batch.tile_dem(3, 2049, 2050)).cuda()
    big[1000, 1000], big[5, 2040] = 3e13, -2e13
    refs, (rs, rc, _) = expected(dems), focal.slope_d8(big, 30.0, -9999.0)
    ctx = failing_context(1 if fails == "batch" else 2)
    b = batch.Batch(dems, ctx=ctx)
    if fails == "batch":
        with pytest.raises(_lib.PargoError, match="launch failure"):
            b.run(batch.PERSISTENT)
    else:
        b.run(batch.PERSISTENT)
        with pytest.raises(_lib.PargoError, match="launch failure"):
            focal.slope_d8(big, 30.0, -9999.0, ctx=ctx)
        clear(b)
        b.run(batch.GRAPH)  # the plan of before
        torch.cuda.synchronize()
        check(b, refs)
    s, c, _ = focal.slope_d8(big, 30.0, -9999.0, ctx=ctx)
    clear(b)
    b.run(batch.GRAPH)
    torch.cuda.synchronize()
    assert torch.equal(s, rs) and torch.equal(c, rc)
    check(b, refs)
    ctx.close()
