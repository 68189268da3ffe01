"""The exact transpose at the edges of its candidate ranges and tile shapes.

Against the oracle's geometric transpose (voxel-driven clip, FP64), at the
1e-5-of-peak bar of the full-size comparison: volumes that take 1, 2 and 4 rows
per wave with ragged last tiles, voxels whose shadow holds more columns and
rows than are clipped at a time, a detector smaller than the shadow, and
16-bit sinograms. A non-finite bin reaches only the voxels its ray meets.
"""
import numpy as np
import pytest
import torch

from newrecon_amd.geometry import Geometry, arc_angles
from newrecon_amd.ostr import DBTSystem

pytestmark = pytest.mark.gpu

# nx, ny, nz, voxel, dz, nbx, nby, bin
CASES = {
    "1-row": (37, 21, 6, 0.5, 1.0, 60, 30, 0.56),
    "2-rows": (129, 67, 21, 0.5, 1.0, 150, 80, 0.56),
    "4-rows": (70, 131, 65, 0.5, 0.5, 90, 150, 0.56),
    "coarse-voxels": (19, 11, 7, 3.0, 4.0, 260, 150, 0.3),
    "small-detector": (100, 60, 10, 0.5, 1.0, 51, 33, 0.6),
}


def make(name, views=5):
    nx, ny, nz, v, dz, nbx, nby, b = CASES[name]
    g = Geometry.half_cone(nx, ny, nz, v, v, dz, nbx, nby, b, b)
    return g, arc_angles(views, 12.5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name", CASES)
def test_transpose_matches_the_clip_oracle(dev, oracle_lib, name, dtype):
    g, ang = make(name)
    rng = np.random.default_rng(3)
    prj = torch.from_numpy(rng.standard_normal((len(ang),) + g.view_shape).astype(np.float32))
    prj = prj.to(dtype)
    S = DBTSystem(g, ang, device=dev)
    ref = oracle_lib.bproj_clip(g, ang, prj.double().numpy(), 0, len(ang))
    got = S.bproj_matched(prj.to(dev), 0, len(ang)).cpu().numpy()
    err = np.abs(got - ref).max() / np.abs(ref).max()
    assert err <= 1e-5, err


@pytest.mark.parametrize("name", ["1-row", "4-rows", "coarse-voxels"])
def test_non_finite_bins_stay_on_their_rays(dev, name):
    g, ang = make(name, views=1)
    S = DBTSystem(g, ang, device=dev)
    one = S.sinogram(1)
    one[0, g.nbx // 2, g.nby // 2] = 1.0
    met = S.bproj_matched(one, 0, 1) > 0
    assert met.any()
    one[0, g.nbx // 2, g.nby // 2] = float("inf")
    got = S.bproj_matched(one, 0, 1)
    assert torch.equal(~torch.isfinite(got), met)
