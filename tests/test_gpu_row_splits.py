"""The network's pooling, upsampling and branch-point passes where rows are cut (few long rows) and
where they share workgroups (many rows shorter than a wave), in whole groups of eight channels and
single ones: the checks of test_gpu_conv_rows.py, the same bits as numpy."""
import pytest

from test_gpu_conv_rows import test_row_passes as row_passes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,cl,cs,shift", [
    ((2, 6, 1380), 24, 3, 0), ((2, 2, 514), 64, 40, 0), ((4, 2, 300), 5, 8, 0), ((2, 4, 130), 8, 8, 1),
    ((134, 126, 2), 3, 5, 0), ((130, 132, 4), 8, 16, 0), ((66, 64, 6), 16, 24, 0), ((130, 260, 2), 24, 8, 1),
    ((66, 64, 64), 8, 8, 0), ((66, 64, 62), 1, 1, 0), ((182, 184, 2), 1, 1, 0)])
def test_splits(shape, cl, cs, shift):
    row_passes(shape, cl, cs, shift)
