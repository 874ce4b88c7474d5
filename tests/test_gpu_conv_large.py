"""Convolutions on grids of many boxes: planes repeat along z, so that the output of a large grid
must repeat too, and be that of a slab of 48 planes, whose sums run in the same order, bit for
bit (the slab's sizes are those that the smaller tests compare with numpy)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PERIOD = 16


@pytest.mark.parametrize("side,cin,cout", [(256, 48, 16), (256, 16, 48), (320, 8, 32)])
def test_repeating_planes(side, cin, cout):
    from mflbm import nn
    print(f"[conv-large] {side}^3 {cin}->{cout}", flush=True)
    L = nn.lib()
    rng = np.random.default_rng(cin)
    planes = nn.bf16_bits(rng.standard_normal((PERIOD, side, side, cin), dtype=np.float32))
    w = np.zeros((nn.wrows(cout), nn.rup(27 * cin, 32)), np.float32)
    w[:cout, :27 * cin] = rng.normal(0, 0.2, (cout, 27 * cin))
    wd, bd = nn.DevArray.from_numpy(w, "bf16"), nn.DevArray.from_numpy(rng.normal(0, 0.1, cout).astype(np.float32), "f32")

    def run(depth):
        x, y = nn.DevArray((depth, side, side, cin), "bf16"), nn.DevArray((depth, side, side, cout), "bf16")
        for z in range(0, depth, PERIOD):
            assert L.mfnn_copy(C.c_void_p(x.data_ptr() + z * planes[0].nbytes), planes.ctypes.data_as(C.c_void_p),
                               planes.nbytes, 0) == 0
        assert L.mfnn_conv3(nn.ptr(x), nn.ptr(wd), nn.ptr(bd), None, depth, side, side, cin, w.shape[1], cout, 1, nn.ptr(y),
                            None, None) == 0
        assert L.mfnn_sync() == 0
        out = np.empty((depth, side, side, cout), np.uint16)
        assert L.mfnn_copy(out.ctypes.data_as(C.c_void_p), nn.ptr(y), out.nbytes, 1) == 0
        return out

    ref, got = run(3 * PERIOD), run(side)
    assert ref.any()
    assert np.array_equal(got[:PERIOD], ref[:PERIOD]) and np.array_equal(got[-PERIOD:], ref[-PERIOD:])
    for z in range(PERIOD, side - PERIOD, PERIOD):
        assert np.array_equal(got[z:z + PERIOD], ref[PERIOD:2 * PERIOD]), z
