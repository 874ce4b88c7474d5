"""The gathering convolution (channel counts whose boxes do not fit LDS): small grids against
numpy, and each of its forms, which share loads between voxel and channel tiles, against the form
of small grids on a slab of the same planes: their sums run in the same order, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import test_gpu_conv_tiles as tiles
from test_gpu_conv_tiles import nn  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

CIN = 1104  # no box of this many channels fits LDS


@pytest.mark.parametrize("shape,cout", [((3, 2, 5), 8), ((2, 5, 9), 40)])
def test_small_grids(nn, shape, cout):  # noqa: F811
    tiles.test_forward(nn, shape, CIN, cout)


# planes, output channels: one to eight and ten channel tiles; one and two with one voxel tile to a
# wave and with two (from 65536 voxels); 255 voxels to a plane, so that the last tiles are broken
@pytest.mark.parametrize("depth,cout", [(176, 10), (272, 10), (176, 24), (272, 24), (176, 40), (176, 64), (112, 80), (112, 96),
                                        (112, 112), (112, 128), (112, 150)])
def test_forms_on_repeating_planes(nn, depth, cout):  # noqa: F811
    print(f"[conv-gather] {depth} planes {CIN}->{cout}", flush=True)
    L, period, H, W = nn.lib(), 16, 17, 15
    rng = np.random.default_rng(cout)
    planes = nn.bf16_bits(rng.standard_normal((period, H, W, CIN), dtype=np.float32))
    wd, kp = tiles.weights(nn, rng.normal(0, 0.2, (cout, 27 * CIN)), CIN, cout)
    bd = nn.DevArray.from_numpy(rng.normal(0, 0.1, cout).astype(np.float32), "f32")

    def run(n):
        x, y = nn.DevArray((n, H, W, CIN), "bf16"), nn.DevArray((n, H, W, cout), "f32")
        for z in range(0, n, period):
            assert L.mfnn_copy(C.c_void_p(x.data_ptr() + z * planes[0].nbytes), planes.ctypes.data_as(C.c_void_p),
                               planes.nbytes, 0) == 0
        assert L.mfnn_conv3(nn.ptr(x), nn.ptr(wd), nn.ptr(bd), None, n, H, W, CIN, kp, cout, 0, None, nn.ptr(y), None) == 0
        return y.numpy()

    ref, got = run(3 * period), run(depth)
    assert ref.any() and np.all(np.isfinite(ref))
    assert np.array_equal(got[:period], ref[:period]) and np.array_equal(got[-period:], ref[-period:])
    for z in range(period, depth - period, period):
        assert np.array_equal(got[z:z + period], ref[period:2 * period]), z
