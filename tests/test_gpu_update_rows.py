"""The SBP kernels at the sizes where their rows per wave change (2, 4 and 8),
with ragged last tiles in x and y: the backprojection against the oracle and the
fused updates against the launcher-by-launcher sequence, at the bars of the
full-size comparisons (1e-5 of the oracle's peak; the fused OSTR update 1e-6 of
the unfused image's peak; the fused OS-SART update bit for bit)."""
import numpy as np
import pytest
import torch

from newrecon_amd.geometry import Geometry, arc_angles
from newrecon_amd.ostr import DBTSystem

pytestmark = pytest.mark.gpu

SIZES = {2: (67, 33, 9), 4: (131, 101, 57), 8: (641, 203, 93)}


@pytest.fixture(params=sorted(SIZES))
def case(request, dev):
    nx, ny, nz = SIZES[request.param]
    g = Geometry.half_cone(nx, ny, nz, 0.2, 0.2, 0.6, int(nx * 0.9) + 9, int(ny * 0.9) + 9, 0.25,
                           0.25)
    S = DBTSystem(g, arc_angles(2, 7.5), device=dev)
    gen = torch.Generator(device=dev).manual_seed(1)
    x = 0.05 * torch.rand(g.vol_shape, generator=gen, device=dev)
    h = torch.randn((2, g.nby, g.nbx), generator=gen, device=dev)
    return g, S, x, h


def test_backprojection(case, oracle_lib):
    g, S, x, h = case
    nat = h.transpose(1, 2).contiguous()
    got = S.bproj_sbp(nat, 0, 2).cpu().numpy()
    ref = oracle_lib.bproj_sbp(g, S.angles, nat.cpu().numpy(), 0, 2)
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("h_dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("prior", ["hyperbola", "lange", "q2"])
def test_fused_update(case, prior, h_dtype):
    g, S, x, h = case
    h = h.to(h_dtype)
    d = S.volume(fill=50.0)
    out = S.update_fused(x, torch.empty_like(x), d, h, 0, 2, 20.0, 3.0, prior, 5e-4)
    cap = S.bproj_sbp_rows(h, 0, 2)
    rdd, rd = S.prior(x, prior, 5e-4)
    want = S.update_est(x.clone(), cap, rd, d, rdd, 20.0, 3.0, guard=True)
    assert float((out - want).abs().max()) <= 1e-6 * float(want.abs().max())


@pytest.mark.parametrize("beta", [0.0, -2e-3])
def test_fused_sart_update(case, beta):
    g, S, x, h = case
    h = 1e-3 * h
    out = S.sart_update_fused(x, torch.empty_like(x), h, 0, 2, 0.9, beta, 1e-3)
    prior = S.prior_sart(x, 1e-3) if beta else None
    want = S.bproj_sart(h.transpose(1, 2).contiguous(), 0, 2, x.clone(), 0.9, prior, beta)
    assert torch.equal(out, want)


@pytest.mark.parametrize("nbx,nby,n", [(1, 1, 1), (33, 31, 2), (65, 127, 3), (700, 1300, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layout_transpose(dev, nbx, nby, n, dtype):
    """Both tile sizes of the layout transpose (the larger from 512 tiles of
    64x64 on), whole and ragged."""
    g = Geometry.half_cone(4, 4, 2, 1.0, 1.0, 1.0, nbx, nby, 1.0, 1.0)
    S = DBTSystem(g, arc_angles(n, 7.5) if n > 1 else [0.0], device=dev)
    p = torch.randn((n, nbx, nby), device=dev).to(dtype)
    assert torch.equal(S.to_rows(p), p.transpose(1, 2))
