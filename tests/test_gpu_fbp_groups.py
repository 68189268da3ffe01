"""The FBP row filter on both sides of the line between its kernels at 1024
points, 512 work-groups of two column pairs: a launch over two views against the
same views one by one (half the groups, the other kernel just past the line), bit
for bit, in both layouts, and against the FP64 direct sum at the filter's
1e-5-of-peak bar."""
import numpy as np
import pytest
import torch

from newrecon_amd.fbp import filter_taps
from newrecon_amd.geometry import Geometry, arc_angles
from newrecon_amd.ostr import DBTSystem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbx,nby", [(260, 1024), (260, 1025), (512, 1028), (512, 1029)])
@pytest.mark.parametrize("rows", [False, True])
def test_line_between_the_kernels(dev, nbx, nby, rows):
    from oracle import fbp as F
    g = Geometry.half_cone(16, 16, 4, 1.0, 1.0, 1.0, nbx, nby, 0.14, 0.14)
    ang = arc_angles(2, 7.5)
    taps = filter_taps(nbx, g.dbx, "hann").astype(np.float32)
    p = np.random.default_rng(nbx).random((2,) + g.view_shape).astype(np.float32)
    S = DBTSystem(g, ang, device=dev)
    pt, tt = torch.from_numpy(p).to(dev), torch.from_numpy(taps).to(dev)
    both = S.fbp_filter(pt, tt, 0, 2, rows=rows)
    each = [S.fbp_filter(pt[v:v + 1].clone(), tt, v, v + 1, rows=rows) for v in (0, 1)]
    assert torch.equal(both, torch.cat(each))
    ref = F.fbp_filter(g, ang, p, taps.astype(np.float64))
    got = both.transpose(1, 2) if rows else both
    assert np.abs(got.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
