"""The Siddon walk's plain and flagged batches and the ray kernels' tile bands.

Geometries whose rays take no plain batch (a volume of a few voxels), end
inside the first turns, cross hundreds of planes of one axis (long in x at
steep angles, many thin slices), run parallel to a voxel plane (a bin centre
under the source) or hold many ties (bin and voxel grids aligned), on detectors
of less than one band, whole bands and a ragged last band, 1 to 5 views. The
walk follows the oracle's operations one for one: 1e-6 of the peak as in the
full-size comparison, equal zero pattern, exact segment count.
"""
import numpy as np
import pytest
import torch

from newrecon_amd.geometry import Geometry
from newrecon_amd.ostr import OSTR, DBTSystem

pytestmark = pytest.mark.gpu

# nx, ny, nz, voxel, dz, nbx, nby, bin, views, half span (degrees)
CASES = {
    "few-voxels": (3, 2, 1, 1.0, 1.0, 9, 3, 1.0, 1, 5.0),
    "long-in-x": (700, 30, 2, 0.1, 6.0, 130, 5, 0.7, 3, 55.0),
    "thin-slices": (6, 5, 300, 1.0, 0.1, 21, 17, 0.6, 5, 20.0),
    "aligned-grids": (64, 32, 16, 1.0, 1.0, 65, 33, 1.0, 3, 10.0),
    "one-band": (90, 4, 10, 0.5, 1.0, 150, 4, 0.56, 5, 7.5),
    "ragged-bands": (60, 70, 24, 0.5, 1.0, 70, 67, 0.56, 3, 7.5),
}


def make(name):
    nx, ny, nz, v, dz, nbx, nby, b, views, span = CASES[name]
    g = Geometry.half_cone(nx, ny, nz, v, v, dz, nbx, nby, b, b)
    ang = np.radians(np.linspace(-span, span, views) if views > 1 else [0.0]).astype(np.float32)
    x = np.random.default_rng(5).random(g.vol_shape).astype(np.float32)
    return g, ang, x


def rel_max(a, ref):
    return float(np.abs(np.asarray(a, np.float64) - ref).max() / max(np.abs(ref).max(), 1e-30))


@pytest.mark.parametrize("name", CASES)
def test_walk_matches_oracle(dev, oracle_lib, name):
    g, ang, x = make(name)
    n = len(ang)
    S = DBTSystem(g, ang, device=dev)
    ref = oracle_lib.fproj(g, ang, x, 0, n)
    got = S.fproj(torch.from_numpy(x).to(dev), 0, n).cpu().numpy()
    assert np.count_nonzero(ref) and rel_max(got, ref) <= 1e-6
    assert np.array_equal(got == 0, ref == 0)
    rows = oracle_lib.gamma(g, ang, 0, n, 1)
    assert rel_max(S.gamma(0, n, "row_sum").cpu().numpy(), rows) <= 1e-6
    prj, norm = S.fproj_sart(torch.from_numpy(x).to(dev), 0, n, cos_weight=True)
    assert np.array_equal(prj.cpu().numpy(), got)
    assert np.array_equal(norm.cpu().numpy(), S.gamma(0, n, "row_sum").cpu().numpy())
    assert S.count_nnz(0, n) == oracle_lib.count_nnz(g, ang, 0, n)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_walk_of_16_bit_images(dev, oracle_lib, dtype):
    g, ang, x = make("ragged-bands")
    xt = torch.from_numpy(x).to(dtype)
    S = DBTSystem(g, ang, device=dev)
    ref = oracle_lib.fproj(g, ang, xt.float().numpy(), 0, len(ang))
    assert rel_max(S.fproj(xt.to(dev), 0, len(ang)).cpu().numpy(), ref) <= 1e-6


@pytest.mark.parametrize("rows", [1, 2, 4, 8])
def test_batched_bands_equal_single_launches(dev, rows):
    """Every tile height of the batched forward on detectors of less than one
    band, ragged and whole bands, in one batch: bit-identical h."""
    from newrecon_amd.batch import DEFAULT_TILE, BatchOSTR
    from newrecon_amd.geometry import OSTRConfig
    recs = []
    for name in ("one-band", "ragged-bands", "aligned-grids"):
        g, ang, x = make(name)
        y = torch.full((len(ang),) + g.view_shape, 900.0, device=dev)
        recs.append(OSTR(g, ang, y, torch.full_like(y, 1e3), x0=0.02 * torch.from_numpy(x),
                         cfg=OSTRConfig(n_subsets=1), device=dev))
    bt = BatchOSTR(recs, tile=dict(DEFAULT_TILE, fwd_rows=rows))
    bt.fproj_h()
    for r in recs:
        want = r.sys.fproj_h(r.x, r.y, r.b, r.r, 0, r.vs, hsub=torch.empty_like(r.h))
        assert torch.equal(r.h, want)
