"""GPU checks of the convolution kernels at the sizes where their tiles can go wrong: boxes and
rows that no tile divides, one-voxel grids, channel counts that leave a half slice or a ragged
quad, grids too wide or too deep in channels for LDS, and values that must not spread.

Tolerances are derived: an fp32 sum of n products, in any order, is within n 2^-23 of the sum
of their magnitudes (Higham's gamma_n with a factor two in hand); bf16 stores add 2^-8 of the
value."""
import ctypes as C

import numpy as np
import pytest

import nn_oracle as N

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -23


@pytest.fixture(scope="module")
def nn():
    from mflbm import nn as mod
    mod.lib()
    return mod


def bf16_round(nn, a):
    return nn.bf16_values(nn.bf16_bits(np.asarray(a, np.float32))).astype(np.float64)


def operands(nn, shape, cin, cout, seed):
    rng = np.random.default_rng(seed)
    x = bf16_round(nn, rng.normal(size=shape + (cin,)))
    w = bf16_round(nn, rng.normal(0, 0.2, (cout, 27 * cin)))
    b = rng.normal(0, 0.1, cout).astype(np.float32).astype(np.float64)
    return rng, x, w, b


def weights(nn, w, cin, cout):
    full = np.zeros((nn.wrows(cout), nn.rup(27 * cin, 32)), np.float32)
    full[:cout, :27 * cin] = w
    return nn.DevArray.from_numpy(full, "bf16"), full.shape[1]


@pytest.mark.parametrize("shape,cin,cout", [
    ((1, 1, 1), 8, 8), ((6, 5, 7), 8, 16), ((17, 19, 21), 96, 32), ((5, 9, 33), 24, 40), ((2, 3, 70), 16, 10),
    ((3, 4, 9), 24, 3), ((2, 50, 2), 144, 17), ((7, 8, 9), 192, 64), ((3, 2, 5), 640, 8), ((33, 34, 35), 16, 48)])
def test_forward(nn, shape, cin, cout):
    """(3, 2, 5) with 640 channels gathers from memory; the others stage boxes"""
    print(f"[conv-tiles] forward {shape} {cin}->{cout}", flush=True)
    rng, x, w, b = operands(nn, shape, cin, cout, cin + cout)
    gate = bf16_round(nn, rng.normal(size=shape + (cout,)))
    D, H, W = shape
    xd, bd, gd = nn.DevArray.from_numpy(x, "bf16"), nn.DevArray.from_numpy(b, "f32"), nn.DevArray.from_numpy(gate, "bf16")
    wd, kp = weights(nn, w, cin, cout)
    yb, yf = nn.DevArray(shape + (cout,), "bf16"), nn.DevArray(shape + (cout,), "f32")
    ref, size = N.conv3(x, w, b), N.conv3(np.abs(x), np.abs(w), np.abs(b))
    tol = (27 * cin + 2) * EPS * size
    L = nn.lib()

    def run(relu, gated, out_b, out_f):
        rc = L.mfnn_conv3(nn.ptr(xd), nn.ptr(wd), nn.ptr(bd), nn.ptr(gd) if gated else None, D, H, W, cin, kp, cout, relu,
                          nn.ptr(out_b), nn.ptr(out_f), None)
        assert rc == 0

    run(0, False, None, yf)
    assert np.all(np.abs(yf.numpy() - ref) <= tol)
    run(1, False, yb, None)
    want = np.maximum(ref, 0.0)
    assert np.all(np.abs(yb.numpy() - want) <= tol + 2.0 ** -8 * want)
    run(0, True, yb, yf)
    want = ref * (gate > 0)
    assert np.all(np.abs(yf.numpy() - want) <= tol)
    assert np.all(np.abs(yb.numpy() - want) <= tol + 2.0 ** -8 * np.abs(want))


@pytest.mark.parametrize("shape,cin,cout", [
    ((1, 1, 1), 8, 8), ((6, 5, 7), 8, 16), ((17, 19, 21), 96, 32), ((5, 9, 33), 24, 40), ((3, 5, 300), 16, 16),
    ((2, 3, 600), 16, 16), ((9, 3, 2), 40, 48), ((1, 40, 16), 16, 24)])
@pytest.mark.parametrize("chunk", [96, 512])
def test_weight_gradient(nn, shape, cin, cout, chunk):
    """rows of 300 voxels load part of a stage when it is stored, rows of 600 take the gathering
    kernel; chunks of 96 voxels end inside rows and planes"""
    print(f"[conv-tiles] wgrad {shape} {cin}->{cout} chunk {chunk}", flush=True)
    rng, x, _, _ = operands(nn, shape, cin, cout, cin * cout)
    dz = bf16_round(nn, rng.normal(size=shape + (cout,)))
    D, H, W = shape
    L = nn.lib()
    kp, rows = nn.rup(27 * cin, 32), nn.rup(cout, 16)
    xd, zd = nn.DevArray.from_numpy(x, "bf16"), nn.DevArray.from_numpy(dz, "bf16")
    work = nn.DevArray.from_numpy(np.full(L.mfnn_wgrad_workspace(D, H, W, kp, cout, chunk), np.nan, np.float32), "f32")
    dw, db = nn.DevArray((rows, kp), "f32"), nn.DevArray((cout,), "f32")
    assert L.mfnn_conv3_wgrad(nn.ptr(xd), nn.ptr(zd), D, H, W, cin, kp, cout, chunk, nn.ptr(work), nn.ptr(dw), nn.ptr(db), 0,
                              None) == 0
    dw_ref, db_ref = N.conv3_wgrad(x, dz)
    dw_size, db_size = N.conv3_wgrad(np.abs(x), np.abs(dz))
    got = dw.numpy()
    n = D * H * W + 16
    assert np.all(np.abs(got[:cout, :27 * cin] - dw_ref) <= n * EPS * dw_size)
    assert np.all(np.abs(db.numpy() - db_ref) <= n * EPS * db_size)
    assert np.all(got[cout:] == 0) and np.all(got[:, 27 * cin:] == 0)


def test_unaligned_outputs(nn):
    """outputs and bias at addresses that allow no vector store"""
    shape, cin, cout = (4, 5, 18), 16, 16
    _, x, w, b = operands(nn, shape, cin, cout, 5)
    xd = nn.DevArray.from_numpy(x, "bf16")
    wd, kp = weights(nn, w, cin, cout)
    n = int(np.prod(shape)) * cout
    yb, yf, bd = nn.DevArray((n + 1,), "bf16", zero=True), nn.DevArray((n + 1,), "f32", zero=True), nn.DevArray((cout + 1,), "f32")
    bd.upload(np.concatenate([[0.0], b]))
    at = lambda d, nbytes: C.c_void_p(d.data_ptr() + nbytes)
    assert nn.lib().mfnn_conv3(nn.ptr(xd), nn.ptr(wd), at(bd, 4), None, *shape, cin, kp, cout, 0, at(yb, 2), at(yf, 4), None) == 0
    ref = N.conv3(x, w, b).ravel()
    tol = (27 * cin + 2) * EPS * N.conv3(np.abs(x), np.abs(w), np.abs(b)).ravel()
    assert np.all(np.abs(yf.numpy()[1:] - ref) <= tol) and yf.numpy()[0] == 0
    assert np.all(np.abs(yb.numpy()[1:] - ref) <= tol + 2.0 ** -8 * np.abs(ref)) and yb.numpy()[0] == 0


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_bad_values_stay_local(nn, bad):
    """an infinity or NaN of the input reaches the outputs of its neighbourhood and the weight
    gradients of its channel only (no padding, tail or neighbouring tile multiplies it)"""
    shape, cin, cout = (5, 6, 19), 8, 16
    rng, x, w, b = operands(nn, shape, cin, cout, 9)
    x[2, 3, 18, 5] = bad
    xd = nn.DevArray.from_numpy(x, "bf16")
    wd, kp = weights(nn, w, cin, cout)
    yf = nn.DevArray(shape + (cout,), "f32")
    L = nn.lib()
    assert L.mfnn_conv3(nn.ptr(xd), nn.ptr(wd), None, None, *shape, cin, kp, cout, 0, None, nn.ptr(yf), None) == 0
    near = np.zeros(shape, bool)
    near[1:4, 2:5, 17:19] = True
    assert np.all(np.isfinite(yf.numpy()).all(axis=3) == ~near)
    dz = bf16_round(nn, rng.normal(size=shape + (cout,)))
    zd = nn.DevArray.from_numpy(dz, "bf16")
    work = nn.DevArray((L.mfnn_wgrad_workspace(*shape, kp, cout, 96),), "f32")
    dw, db = nn.DevArray((16, kp), "f32"), nn.DevArray((cout,), "f32")
    assert L.mfnn_conv3_wgrad(nn.ptr(xd), nn.ptr(zd), *shape, cin, kp, cout, 96, nn.ptr(work), nn.ptr(dw), nn.ptr(db), 0, None) == 0
    finite = np.isfinite(dw.numpy()[:, :27 * cin].reshape(16, 27, cin)).all(axis=(0, 1))
    assert list(finite) == [c != 5 for c in range(cin)]
    assert np.all(np.isfinite(db.numpy()))


@pytest.mark.parametrize("shape,cin,cout,chunk", [
    ((40, 33, 30), 48, 32, 1024), ((40, 66, 70), 32, 16, 2048), ((40, 66, 70), 40, 8, 2048), ((6, 11, 150), 96, 64, 1024)])
def test_weight_gradient_many_stages(nn, shape, cin, cout, chunk):
    """chunks of several stages with one group of waves per workgroup (more than 512 workgroups),
    stages inside a plane and across two, and inputs above 16 MB, whose chunks go to one XCD"""
    test_weight_gradient(nn, shape, cin, cout, chunk)
