"""The FBP row filter at every transform length it has a kernel for: detector
widths on both sides of each power of two from 512 to 8192 points, widths that
need one and two column pairs per group and ragged last ones. Against the FP64
direct sum at the 1e-5-of-peak bar of the filter's other sizes."""
import numpy as np
import pytest
import torch

from newrecon_amd.fbp import filter_taps
from newrecon_amd.geometry import Geometry, arc_angles
from newrecon_amd.ostr import DBTSystem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbx,nby", [(256, 7), (257, 8), (512, 5), (513, 4), (1024, 3),
                                     (1025, 8), (2049, 6)])
def test_filter_lengths(dev, nbx, nby):
    from oracle import fbp as F
    g = Geometry.half_cone(16, 16, 4, 1.0, 1.0, 1.0, nbx, nby, 0.14, 0.14)
    ang = arc_angles(2, 7.5)
    taps = filter_taps(nbx, g.dbx, "hann").astype(np.float32)
    p = np.random.default_rng(nbx).random((2,) + g.view_shape).astype(np.float32)
    S = DBTSystem(g, ang, device=dev)
    q = S.fbp_filter(torch.from_numpy(p).to(dev), torch.from_numpy(taps).to(dev), 0, 2)
    ref = F.fbp_filter(g, ang, p, taps.astype(np.float64))
    assert np.abs(q.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("nbx,nby", [(100, 7), (300, 8), (1025, 6), (2049, 5)])
def test_row_major_output(dev, nbx, nby):
    """ostr_fbp_filter_rows holds ostr_fbp_filter's values, transposed."""
    g = Geometry.half_cone(16, 16, 4, 1.0, 1.0, 1.0, nbx, nby, 0.14, 0.14)
    S = DBTSystem(g, arc_angles(3, 7.5), device=dev)
    taps = torch.from_numpy(filter_taps(nbx, g.dbx, "ramp").astype(np.float32)).to(dev)
    p = torch.rand((2,) + g.view_shape, device=dev)
    rows = S.fbp_filter(p, taps, 1, 3, rows=True)
    assert torch.equal(rows, S.fbp_filter(p, taps, 1, 3).transpose(1, 2))
