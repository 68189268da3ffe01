"""Volumes of one voxel in x whose rows, 2^28 and more, make more than 2^32
threads along one grid dimension. Every kernel's upper and middle slices against
a volume that holds these slices alone (all sizes are powers of two, so the
coordinates are the same floats): the same values, the priors inside its
slices."""
import numpy as np
import pytest
import torch

from newrecon_amd.geometry import Geometry
from newrecon_amd.ostr import DBTSystem

pytestmark = pytest.mark.gpu

N, D, SLAB = 1 << 14, 2.0 ** -7, 6


def system(z0, nz, dev):
    g = Geometry(nx=1, ny=N, nz=nz, dx=1.0, dy=D, dz=D, x_p0=-0.5, y_p0=-N * D, z_p0=z0 * D,
                 nbx=4, nby=64, dbx=1.0, dby=3.0, x_d0=-2.0, y_d0=-192.0, detector_r=0.0,
                 source_r=512.0, source_y=0.0)
    return DBTSystem(g, np.zeros(1, np.float32), device=dev)


@pytest.fixture(scope="module")
def slabs(dev):
    gen = torch.Generator(device=dev).manual_seed(1)
    h = 1e-3 * torch.rand((1, 64, 4), generator=gen, device=dev)
    x = torch.rand((N, N, 1), generator=gen, device=dev)
    # one slab on each side of the line between two rows of groups, and the last
    at = (0, N // 2 - 3, N - SLAB)
    return h, x, system(0, N, dev), [(z, system(z, SLAB, dev)) for z in at]


CALLS = {
    "sbp": lambda S, x, h: S.bproj_sbp_rows(h, 0, 1),
    "matched": lambda S, x, h: S.bproj_matched(h, 0, 1, rows=True),
    "sart": lambda S, x, h: S.sart_update_fused(x, torch.empty_like(x), h, 0, 1, 0.9),
    "sart-prior": lambda S, x, h: S.sart_update_fused(x, torch.empty_like(x), h, 0, 1, 0.9, -2e-3,
                                                      1e-3),
    "huber": lambda S, x, h: S.prior_sart(x, 1e-3),
    "update": lambda S, x, h: S.update_fused(x, torch.empty_like(x), torch.ones_like(x), h, 0, 1,
                                             1e3, 1.0, "q2", 5e-4),
    "update-matched": lambda S, x, h: S.update_fused_matched(x, torch.empty_like(x),
                                                             torch.ones_like(x), h, 0, 1, 1e3, 1.0,
                                                             "q2", 5e-4),
}


@pytest.mark.parametrize("call", CALLS)
def test_slices(slabs, call):
    h, x, S, parts = slabs
    got = CALLS[call](S, x, h)
    for z, part in parts:
        want = CALLS[call](part, x[z:z + SLAB].contiguous(), h)
        inner = slice(1, SLAB - 1)
        assert torch.count_nonzero(want[inner])
        assert torch.equal(got[z:z + SLAB][inner], want[inner])
