"""The network's convolution on volumes that cut its tiles raggedly in x, y and z
(one slice, chunks of one and several slices), for layers with the weights in
registers, in LDS and read per chunk, from a channel range of a wider buffer,
with and without bias, ReLU and a ReLU mask: against the FP64 convolution of the
same BF16 inputs, at the BF16 bar of the layer tests (1e-2 of the peak), and
bit-identical between a channel range and a dense buffer."""
import numpy as np
import pytest
import torch

from newrecon_amd.warmstart import _ptr, cnn_lib

pytestmark = pytest.mark.gpu


def bf16(t):
    return t.to(torch.bfloat16)


def conv(dev, cin, cout, x, w, bias, mask, relu, stride, offset):
    """ostr_cnn_conv3d of x [nz][ny][nx][cin] held at `offset` of `stride` channels."""
    L = cnn_lib()
    nz, ny, nx, _ = x.shape
    buf = torch.full((nz, ny, nx, stride), 3.0, dtype=torch.bfloat16, device=dev)
    buf[..., offset:offset + cin] = x
    wf = torch.zeros(cout * L.ostr_cnn_kpad(cin), dtype=torch.int16, device=dev)
    wd = torch.zeros(cin * L.ostr_cnn_kpad(cout), dtype=torch.int16, device=dev)
    assert L.ostr_cnn_pack(_ptr(w), cin, cout, _ptr(wf), _ptr(wd), None) == 0
    y = torch.full((nz, ny, nx, cout), 7.0, dtype=torch.bfloat16, device=dev)
    assert L.ostr_cnn_conv3d(cin, cout, _ptr(buf), stride, offset, _ptr(wf), _ptr(bias), _ptr(y),
                             cout, 0, _ptr(mask), cout, 0, int(relu), nz, ny, nx, None) == 0
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("cin,cout", [(8, 16), (16, 16), (16, 32), (32, 32), (32, 64), (96, 32),
                                      (16, 48), (64, 64), (64, 32), (32, 96)])
@pytest.mark.parametrize("shape", [(1, 5, 70), (3, 9, 33), (13, 17, 65)])
def test_ragged_tiles(dev, cin, cout, shape):
    gen = torch.Generator(device=dev).manual_seed(cin * cout + shape[0])
    x = bf16(torch.randn(shape + (cin,), generator=gen, device=dev))
    w = torch.randn((cout, 27, cin), generator=gen, device=dev) / (27 * cin) ** 0.5
    bias = torch.randn(cout, generator=gen, device=dev)
    mask = bf16(torch.randn(shape + (cout,), generator=gen, device=dev))
    pad = torch.nn.functional.pad(x.double(), (0, 0, 1, 1, 1, 1, 1, 1))
    wq = bf16(w).double()
    nz, ny, nx = shape
    ref = sum(pad[t // 9:t // 9 + nz, t // 3 % 3:t // 3 % 3 + ny, t % 3:t % 3 + nx] @ wq[:, t].T
              for t in range(27))
    for b, m, relu in ((bias, None, True), (None, mask, False), (bias, mask, False)):
        want = ref if b is None else ref + b.double()
        want = want.clamp(min=0) if relu else want
        want = want if m is None else torch.where(m > 0, want, torch.zeros_like(want))
        y = conv(dev, cin, cout, x, w, b, m, relu, cin, 0)
        assert float((y.double() - want).abs().max()) <= 1e-2 * float(want.abs().max())
        assert torch.equal(conv(dev, cin, cout, x, w, b, m, relu, cin + 16, 8), y)
