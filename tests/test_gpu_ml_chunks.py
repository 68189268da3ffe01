"""ml_dbt over views in several launches: chunks of one, two and all views of a
scan whose last chunk is ragged, scalar and per-bin blanks, against the FP64
restatement per iteration at its 1e-4 bar, and the sinogram memory the chunk
bounds (four buffers: three of torch's, one of the handle)."""
import numpy as np
import pytest
import torch

from newrecon_amd import recondbt
from newrecon_amd.geometry import Geometry, arc_angles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blank", ["scalar", "per-bin"])
@pytest.mark.parametrize("views", [1, 2, 5])
def test_chunks(dev, oracle_lib, monkeypatch, views, blank):
    from oracle import recondbt as R
    g = Geometry.half_cone(40, 30, 8, 1.0, 1.0, 2.0, 60, 40, 1.0, 1.0)
    ang = arc_angles(5, 7.5)
    rng = np.random.default_rng(4)
    x0 = (0.02 + 0.03 * rng.random(g.vol_shape)).astype(np.float32)
    i0 = 1e4 if blank == "scalar" else (1e4 + 100 * rng.random((5,) + g.view_shape)).astype(np.float32)
    y = rng.poisson(6e3, (5,) + g.view_shape).astype(np.float32)
    monkeypatch.setattr(recondbt, "CHUNK_BYTES", views * 4 * g.n_bin + 3)
    got = recondbt.ml_dbt(g, ang, y, x0, i0, 3, 1.0, saveiter=True, device=dev).cpu().numpy()
    ref = R.ml_dbt(g, ang, y, x0, i0, 3, 1.0, saveiter=True)
    for a, b in zip(got, ref):
        assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b)


def test_memory(dev, monkeypatch):
    g = Geometry.half_cone(40, 30, 8, 1.0, 1.0, 2.0, 1024, 1024, 0.05, 0.05)
    y = torch.full((9,) + g.view_shape, 900.0, device=dev)
    x0 = torch.full(g.vol_shape, 0.02, device=dev)
    monkeypatch.setattr(recondbt, "CHUNK_BYTES", 3 * 4 * g.n_bin)
    before = torch.cuda.memory_allocated(dev)
    torch.cuda.reset_peak_memory_stats(dev)
    recondbt.ml_dbt(g, arc_angles(9, 7.5), y, x0, 1e3, 1, 1.0, device=dev)
    held = torch.cuda.max_memory_allocated(dev) - before
    assert held <= 3 * recondbt.CHUNK_BYTES + 16 * 4 * g.n_vox + (1 << 20)
