"""A contributing area in a caller's graph: the scratch it captured stays while
larger rasters make the context take more, and a call that would need more
scratch during a capture is refused and leaves the capture alone.
"""
import numpy as np
import pytest

from pargo_amd import _lib, hydro

pytestmark = pytest.mark.gpu

ND = -9999.0


def codes(rows, cols, seed):
    import torch
    rng = np.random.default_rng(seed)
    return torch.from_numpy(rng.choice([5, 6, 7, 8, 7, 2], size=(rows, cols)).astype(np.uint8)).cuda()


def test_replays_after_the_scratch_has_grown():
    import torch
    ctx = _lib.Context(0)
    small, large, larger = codes(90, 300, 1), codes(700, 900, 2), codes(1100, 1300, 3)
    refs = [hydro.sca_d8(f, ND, mode="converge").clone() for f in (small, large, larger)]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        hydro.sca_d8(small, ND, mode="converge", ctx=ctx)
        stream.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            out = hydro.sca_d8(small, ND, mode="converge", ctx=ctx)
            with pytest.raises(_lib.PargoError, match="cannot be captured"):
                hydro.sca_d8(large, ND, mode="converge", ctx=ctx)
            again = hydro.sca_d8(small, ND, mode="converge", ctx=ctx)
        for flow, ref in ((large, refs[1]), (larger, refs[2]), (small, refs[0])):
            for _ in range(2):
                got = hydro.sca_d8(flow, ND, mode="converge", ctx=ctx)
                out.zero_()
                again.zero_()
                g.replay()
                after = hydro.sca_d8(flow, ND, mode="converge", ctx=ctx)
                stream.synchronize()
                assert torch.equal(out, refs[0]) and torch.equal(again, refs[0])
                assert torch.equal(got, ref) and torch.equal(after, ref)
    ctx.close()
