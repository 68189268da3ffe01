"""The network's weight and bias gradients of every layer shape on volumes smaller than
a tile, of one slice, and that cut the tiles raggedly in x, y and z, from channel ranges
of wider buffers whose other channels hold NaN. The inputs are small whole numbers, so
every FP32 sum is exact (below 2^24) and the result has to equal the FP64 one."""
import pytest
import torch

from newrecon_amd.warmstart import _ptr, cnn_lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin,cout", [(8, 16), (16, 16), (48, 16), (16, 32), (32, 32),
                                      (32, 64), (64, 64), (96, 32)])
@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 4, 32), (2, 5, 33), (3, 9, 65), (5, 17, 130)])
def test_equals_exact_sums(dev, cin, cout, shape):
    gen = torch.Generator().manual_seed(cin + cout + shape[2])
    nz, ny, nx = shape
    x = torch.randint(-2, 3, (*shape, cin), generator=gen).double()
    dy = torch.randint(-2, 3, (*shape, cout), generator=gen).double()
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    want = torch.stack([dy.reshape(-1, cout).T @ xp[z:z + nz, y:y + ny, c:c + nx].reshape(-1, cin)
                        for z in range(3) for y in range(3) for c in range(3)], 1)

    def view(t, extra, offset):
        buf = torch.full((*shape, t.shape[-1] + extra), float("nan"), dtype=torch.bfloat16)
        buf[..., offset:offset + t.shape[-1]] = t
        return buf.to(dev)

    xd, dd = view(x, 16, 8), view(dy, 8, 0)
    L = cnn_lib()
    nbytes = L.ostr_cnn_wgrad_workspace(cin, cout, nz, ny, nx, 64)
    work = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    dw = torch.full((cout, 27, cin), float("nan"), device=dev)
    db = torch.full((cout,), float("nan"), device=dev)
    assert L.ostr_cnn_wgrad(cin, cout, _ptr(xd), cin + 16, 8, _ptr(dd), cout + 8, 0, nz, ny, nx,
                            _ptr(dw), _ptr(db), _ptr(work), nbytes, 64, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(dw.double().cpu(), want)
    assert torch.equal(db.double().cpu(), dy.reshape(-1, cout).sum(0))
