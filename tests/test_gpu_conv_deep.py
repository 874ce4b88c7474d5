"""Convolutions of several hundred input channels, whose boxes are the few that LDS holds, against
numpy (tests/test_gpu_conv_tiles.py has the bound)."""
import pytest

import test_gpu_conv_tiles as tiles
from test_gpu_conv_tiles import nn  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


# columns of 48 and rows of 64 and 128: their largest splits do not fit LDS with these channels; the last two are the
# gathering kernel's by cost and a box's with little room
@pytest.mark.parametrize("shape,cin,cout", [((48, 3, 64), 448, 16), ((48, 5, 128), 320, 40), ((3, 32, 64), 384, 24),
                                            ((12, 12, 12), 1056, 72), ((6, 5, 7), 576, 64)])
def test_forward(nn, shape, cin, cout):  # noqa: F811
    tiles.test_forward(nn, shape, cin, cout)
