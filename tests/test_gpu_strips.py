"""Strips of every length the row rules choose: rasters on either side of the
sizes where they change give the same bits as the same raster with its rows
walked in strips of 16, and the slope adjoint the same bits as the raster as
part of a taller one.
"""
import os

import numpy as np
import pytest

from pargo_amd import autograd, focal, synth

pytestmark = pytest.mark.gpu

ND = -9999.0


def dem(rows, cols):
    import torch
    z = synth.workload_dem("slope_d8", rows, cols)
    z[rows // 2, cols // 3] = 3e13  # a window for the exact pass
    return torch.from_numpy(z).cuda()


@pytest.mark.parametrize("rows,cols", [(3, 3), (17, 255), (257, 257), (1025, 1025), (1366, 769), (2049, 2048), (4097, 1025),
                                       (4400, 4097)])
@pytest.mark.parametrize("method,dirtype,mask", [("FD", 256, False), ("FD", 8, True), ("TFDW", 8, True)])
def test_strip_lengths_give_the_same_bits(rows, cols, method, dirtype, mask):
    import torch
    z = dem(rows, cols)
    got = focal.slope_d8(z, 30.0, ND, method, "tan", dirtype, want_mask=mask)
    os.environ["PARGO_FOCAL_ROWS"] = "16"
    try:
        ref = focal.slope_d8(z, 30.0, ND, method, "tan", dirtype, want_mask=mask)
    finally:
        del os.environ["PARGO_FOCAL_ROWS"]
    for a, b in zip(got, ref):
        assert (a is None and b is None) or torch.equal(a, b)


@pytest.mark.parametrize("rows,cols", [(3, 3), (64, 300), (1025, 1025), (1366, 769), (2049, 2047), (2050, 4097)])
def test_adjoint_strip_lengths_give_the_same_bits(rows, cols):
    # the raster on top of copies of itself takes longer strips; its rows
    # that do not see the copies' first two rows keep their bits
    import torch
    z = torch.from_numpy(synth.workload_dem("slope_d8", rows, cols)).cuda()
    g = torch.randn((rows, cols), device="cuda", generator=torch.Generator("cuda").manual_seed(rows))
    got = autograd.slope_adjoint(z, g, 30.0, ND)
    tall = autograd.slope_adjoint(z.repeat(9, 1), g.repeat(9, 1), 30.0, ND)
    keep = rows - 2
    assert torch.equal(got[:keep], tall[:keep])
