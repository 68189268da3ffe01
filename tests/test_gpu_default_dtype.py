"""The initialisers under another default dtype of torch: their buffers are FP32
whatever it is, and the images the same bits."""
import numpy as np
import pytest
import torch

from newrecon_amd import fbp, recondbt
from newrecon_amd.geometry import Geometry, arc_angles

pytestmark = pytest.mark.gpu

CALLS = {
    "fbp": lambda g, a, y, x: fbp.fbp_dbt(g, a, y),
    "ml": lambda g, a, y, x: recondbt.ml_dbt(g, a, y, x, 2.0, 1, 1.0),
    "sart": lambda g, a, y, x: recondbt.sart_dbt(g, a, y, x, 1, 0.5),
}


@pytest.mark.parametrize("call", CALLS)
def test_same_image(dev, call):
    g = Geometry.half_cone(40, 30, 8, 1.0, 1.0, 2.0, 60, 40, 1.0, 1.0)
    ang = arc_angles(3, 7.5)
    rng = np.random.default_rng(2)
    y = torch.from_numpy(rng.random((3,) + g.view_shape).astype(np.float32)).to(dev)
    x = torch.from_numpy(rng.random(g.vol_shape).astype(np.float32)).to(dev)
    want = CALLS[call](g, ang, y, x)
    torch.set_default_dtype(torch.float64)
    try:
        got = CALLS[call](g, ang, y, x)
    finally:
        torch.set_default_dtype(torch.float32)
    assert got.dtype == torch.float32 and torch.equal(got, want)
