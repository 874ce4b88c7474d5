"""Weight gradients of small whole numbers: every product and every partial sum is a whole number
below 2^24, exact in bfloat16 operands and float32 sums whatever their order, so the result must be
the exact one.  The shapes take every form of the two kernels: rows with one and two groups of
waves, whole and half slices of channels, chunks of several stages within a plane and across planes,
inputs above 16 MB (a chunk's workgroups on one XCD), and the gathering kernel with one and two
tiles to a wave."""
import numpy as np
import pytest

import nn_oracle as N

pytestmark = pytest.mark.gpu


def check(shape, cin, cout, chunk, accumulate=0):
    from mflbm import nn
    print(f"[wgrad-exact] {shape} {cin}->{cout} chunk {chunk}", flush=True)
    assert 4 * int(np.prod(shape)) < 2 ** 24
    rng = np.random.default_rng(cin * 1000 + cout + shape[2])
    x = rng.integers(-2, 3, shape + (cin,)).astype(np.float32)
    dz = rng.integers(-2, 3, shape + (cout,)).astype(np.float32)
    L, (D, H, W) = nn.lib(), shape
    kp, rows = nn.rup(27 * cin, 32), nn.rup(cout, 16)
    xd, zd = nn.DevArray.from_numpy(x, "bf16"), nn.DevArray.from_numpy(dz, "bf16")
    work = nn.DevArray.from_numpy(np.full(L.mfnn_wgrad_workspace(D, H, W, kp, cout, chunk), np.nan, np.float32), "f32")
    dw, db = nn.DevArray.from_numpy(np.ones((rows, kp), np.float32)), nn.DevArray.from_numpy(np.ones(cout, np.float32))
    assert L.mfnn_conv3_wgrad(nn.ptr(xd), nn.ptr(zd), D, H, W, cin, kp, cout, chunk, nn.ptr(work), nn.ptr(dw), nn.ptr(db),
                              accumulate, None) == 0
    dw_ref, db_ref = N.conv3_wgrad(x.astype(np.float64), dz.astype(np.float64))
    got = dw.numpy()
    assert np.abs(dw_ref).max() > 0
    assert np.array_equal(got[:cout, :27 * cin], dw_ref + accumulate)
    assert np.array_equal(db.numpy(), db_ref + accumulate)
    assert np.all(got[cout:] == accumulate) and np.all(got[:, 27 * cin:] == accumulate)


@pytest.mark.parametrize("shape,cin,cout,chunk", [
    ((40, 33, 30), 48, 32, 1024), ((40, 66, 70), 32, 16, 2048), ((40, 66, 70), 40, 8, 2048), ((6, 11, 150), 96, 64, 1024),
    ((33, 34, 35), 16, 48, 512), ((1, 1, 1), 8, 8, 96), ((9, 3, 2), 40, 48, 96)])
def test_stages(shape, cin, cout, chunk):
    check(shape, cin, cout, chunk)


@pytest.mark.parametrize("shape,cin,cout,chunk", [
    ((4, 5, 421), 48, 24, 96), ((4, 15, 421), 16, 16, 96), ((2, 3, 600), 24, 24, 512), ((3, 40, 430), 40, 72, 96)])
def test_wide_grids(shape, cin, cout, chunk):
    check(shape, cin, cout, chunk)


@pytest.mark.parametrize("shape,cin,cout", [((9, 10, 11), 16, 24), ((4, 5, 421), 48, 24)])
def test_accumulate(shape, cin, cout):
    check(shape, cin, cout, 512, accumulate=1)
