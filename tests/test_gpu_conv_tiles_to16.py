"""test_gpu_conv_tiles' ragged volumes for the two remaining layer shapes: 48 and 32
input channels to 16."""
import pytest

from test_gpu_conv_tiles import test_ragged_tiles as ragged_tiles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin", [48, 32])
@pytest.mark.parametrize("shape", [(1, 5, 70), (3, 9, 33), (13, 17, 65)])
def test_to_16_channels(dev, cin, shape):
    ragged_tiles(dev, cin, 16, shape)
