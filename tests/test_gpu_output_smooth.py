"""The smoothed residual of the network (ostr_cnn_output_smooth) on slices that cut its
tiles raggedly, smaller than the filter, of several slices and of more slices than groups, for every radius: against
the FP64 filter with repeated edges. Two sums of 2r + 1 FP32 FMAs with taps that sum to
1 err by at most 2 (2r + 1) half-ulps of the largest value, and three more roundings
follow: (4 r + 5) * 2^-24 of the peak."""
import ctypes

import numpy as np
import pytest
import torch
from scipy.ndimage import convolve1d

from newrecon_amd.warmstart import _ptr, cnn_lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 4), (2, 3, 2), (1, 16, 64), (3, 17, 65), (2, 50, 131),
                                   (65540, 1, 2)])
@pytest.mark.parametrize("r", [0, 1, 3, 4])
@pytest.mark.parametrize("ocs,clamp", [(16, 0), (8, 1)])
def test_tiles_and_edges(dev, shape, r, ocs, clamp):
    gen = torch.Generator(device=dev).manual_seed(shape[1] * 10 + r)
    nz, ny, nx = shape
    out = torch.randn((*shape, ocs), device=dev, generator=gen).to(torch.bfloat16)
    img = torch.randn(shape, device=dev, generator=gen)
    pred = torch.full((*shape, 1), 7.0, device=dev)
    taps = np.exp(-0.5 * (np.arange(-r, r + 1) / 1.3) ** 2)
    taps = (taps / taps.sum()).astype(np.float32)
    assert cnn_lib().ostr_cnn_output_smooth(
        _ptr(out), ocs, _ptr(img), nz, ny, nx, 4.0, taps.ctypes.data_as(ctypes.c_void_p), r,
        clamp, _ptr(pred), None) == 0
    torch.cuda.synchronize()
    t = taps.astype(np.float64)
    s = out[..., 0].double().cpu().numpy()
    s = convolve1d(convolve1d(s, t, axis=2, mode="nearest"), t, axis=1, mode="nearest")
    want = img.double().cpu().numpy() + s / 4.0
    want = np.maximum(want, 0.0) if clamp else want
    peak = np.abs(s).max() + np.abs(want).max()
    assert np.abs(pred[..., 0].double().cpu().numpy() - want).max() <= (4 * r + 5) * 2**-24 * peak
