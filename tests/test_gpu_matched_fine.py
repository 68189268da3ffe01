"""The exact transpose of voxels whose shadow holds more detector rows (and
columns) than a wave keeps in its lanes, at every number of voxel rows per wave
(1, 2 and 4 by the volume's size) with a ragged last tile. Against the oracle's
geometric transpose (voxel-driven clip, FP64) at the 1e-5-of-peak bar of the
full-size comparison."""
import numpy as np
import pytest
import torch

from newrecon_amd.geometry import Geometry, arc_angles
from newrecon_amd.ostr import DBTSystem

pytestmark = pytest.mark.gpu

# nx, ny, nz, dz: rows of 64 voxels in all 63, 4158, 10349; 5 bins to a voxel
CASES = {1: (9, 9, 7, 3.0), 2: (5, 66, 63, 0.5), 4: (5, 131, 79, 0.5)}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("rows", CASES)
def test_more_rows_than_lanes_hold(dev, oracle_lib, rows, dtype):
    nx, ny, nz, dz = CASES[rows]
    nbx, nby = int(nx * 6.5), int(ny * 5.5)
    g = Geometry.half_cone(nx, ny, nz, 1.0, 1.0, dz, nbx, nby, 0.2, 0.2)
    ang = arc_angles(3, 7.5)
    prj = torch.from_numpy(np.random.default_rng(3).standard_normal((3,) + g.view_shape)
                           .astype(np.float32)).to(dtype)
    ref = oracle_lib.bproj_clip(g, ang, prj.double().numpy(), 0, 3)
    got = DBTSystem(g, ang, device=dev).bproj_matched(prj.to(dev), 0, 3).cpu().numpy()
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
