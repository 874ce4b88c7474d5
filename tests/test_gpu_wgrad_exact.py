"""Weight gradients of small whole numbers: every product and every partial sum is a whole number
below 2^24, exact in bfloat16 operands and float32 sums whatever their order, so the result must be
the exact one.  The shapes take every form of the two kernels: rows with one and two groups of
waves, whole and half slices of channels, chunks of several stages within a plane and across planes,
inputs above 16 MB (a chunk's workgroups on one XCD), and the gathering kernel with one and two
tiles to a wave, on both sides of each rule that chooses between them."""
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


# the last width of each rule and the first beyond it, for one slice, several, and a half slice; few
# waves and many of a half slice; few voxels with a short and a long chain of slices
@pytest.mark.parametrize("shape,cin,cout,chunk", [
    ((3, 5, 340), 16, 16, 96), ((3, 5, 341), 16, 16, 96), ((3, 4, 270), 32, 16, 96), ((3, 4, 271), 32, 16, 96),
    ((4, 6, 212), 24, 40, 96), ((4, 6, 213), 24, 40, 96), ((5, 40, 340), 32, 16, 2048), ((5, 40, 341), 32, 16, 2048),
    ((4, 75, 230), 24, 40, 512), ((4, 75, 231), 24, 40, 512), ((4, 40, 512), 8, 16, 2048), ((4, 40, 513), 8, 16, 2048),
    ((4, 5, 421), 48, 24, 96), ((4, 15, 421), 16, 16, 96), ((7, 8, 9), 24, 24, 512), ((17, 18, 19), 72, 72, 512),
    ((1, 2, 3), 192, 40, 512), ((1, 3, 5), 16, 32, 512), ((2, 3, 600), 24, 24, 512), ((3, 40, 430), 40, 72, 96)])
def test_both_sides_of_the_rules(shape, cin, cout, chunk):
    check(shape, cin, cout, chunk)


@pytest.mark.parametrize("shape,cin,cout", [((9, 10, 11), 16, 24), ((4, 5, 421), 48, 24)])
def test_accumulate(shape, cin, cout):
    check(shape, cin, cout, 512, accumulate=1)
