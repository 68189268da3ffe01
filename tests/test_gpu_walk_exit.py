"""Rays almost parallel to a voxel plane that leave the volume through that
plane's far or near face, between the slices: the source a few micrometres
inside the face, the bin centres a few micrometres outside, so that in FP32 the
exit crossing and the exit parameter differ by many steps of the walk. The walk
follows the oracle's operations one for one: 1e-6 of the peak as in the
full-size comparison, equal zero pattern, exact segment count."""
import numpy as np
import pytest
import torch

from newrecon_amd.geometry import Geometry
from newrecon_amd.ostr import DBTSystem

pytestmark = pytest.mark.gpu

# voxels along the axis, voxel size, slices, slice thickness, depth of the source
# under the face
CASES = {
    "1400-thick": (1400, 0.1, 60, 1.0, 4e-3),
    "1400-thin": (1400, 0.1, 300, 0.1, 2e-3),
    "1400-close": (1400, 0.1, 60, 1.0, 3e-4),
    "256": (256, 0.1, 60, 1.0, 2e-3),
}


def make(name, axis, side):
    """The volume's far (side +1) or near (-1) face along `axis` at `depth` from
    the source at 0; bins from 0.98 to 1.12 of depth across it."""
    n, h, nz, dz, depth = CASES[name]
    p0 = -n * h + depth if side > 0 else -depth
    bins = 96
    pitch = 0.14 * depth / bins
    d0 = 0.98 * depth if side > 0 else -1.12 * depth
    across = dict(n=24, h=0.5, p0=-12.0, bins=40, pitch=0.6, d0=-12.0)
    along = dict(n=n, h=h, p0=p0, bins=bins, pitch=pitch, d0=d0)
    x, y = (along, across) if axis == "x" else (across, along)
    g = Geometry(nx=x["n"], ny=y["n"], nz=nz, dx=x["h"], dy=y["h"], dz=dz, x_p0=x["p0"],
                 y_p0=y["p0"], z_p0=0.0, nbx=x["bins"], nby=y["bins"], dbx=x["pitch"],
                 dby=y["pitch"], x_d0=x["d0"], y_d0=y["d0"], detector_r=0.0, source_r=660.0,
                 source_y=0.0)
    return g, np.zeros(1, np.float32)


@pytest.mark.parametrize("side", [1, -1])
@pytest.mark.parametrize("axis", ["x", "y"])
@pytest.mark.parametrize("name", CASES)
def test_walk_ends_at_the_face(dev, oracle_lib, name, axis, side):
    g, ang = make(name, axis, side)
    x = 1.0 + np.random.default_rng(5).random(g.vol_shape).astype(np.float32)
    S = DBTSystem(g, ang, device=dev)
    ref = oracle_lib.fproj(g, ang, x, 0, 1)
    xt = torch.from_numpy(x).to(dev)
    got = S.fproj(xt, 0, 1).cpu().numpy()
    assert np.count_nonzero(ref)
    assert np.abs(got.astype(np.float64) - ref).max() <= 1e-6 * np.abs(ref).max()
    assert np.array_equal(got == 0, ref == 0)
    rows = oracle_lib.gamma(g, ang, 0, 1, 1)
    assert np.abs(S.gamma(0, 1, "row_sum").cpu().numpy() - rows).max() <= 1e-6 * rows.max()
    prj, norm = S.fproj_sart(xt, 0, 1, cos_weight=True)
    assert np.array_equal(prj.cpu().numpy(), got)
    assert np.array_equal(norm.cpu().numpy(), S.gamma(0, 1, "row_sum").cpu().numpy())
    assert S.count_nnz(0, 1) == oracle_lib.count_nnz(g, ang, 0, 1)
