"""Entry points of the network's library that its own network passes by (it takes the joint passes):
channel copies, gradients met at a branch, weights laid out for the data gradient.  They move
bfloat16 values and add at most two, so the results must be the same bits as numpy's."""
import numpy as np
import pytest

from mflbm import nn

pytestmark = pytest.mark.gpu

f32 = np.float32


def rnd(a):
    return nn.bf16_values(nn.bf16_bits(np.asarray(a, f32)))


@pytest.mark.parametrize("nvox,C,ct,c0", [(1, 1, 1, 0), (37, 3, 8, 5), (300, 8, 24, 8), (129, 16, 16, 0)])
def test_channels(nvox, C, ct, c0):
    print(f"[nn-entry] channels {nvox} {C} of {ct}", flush=True)
    rng = np.random.default_rng(nvox)
    narrow, wide = rnd(rng.normal(size=(nvox, C))), rnd(rng.normal(size=(nvox, ct)))
    L = nn.lib()
    src, dst = nn.DevArray.from_numpy(narrow, "bf16"), nn.DevArray.from_numpy(wide, "bf16")
    assert L.mfnn_channels(nn.ptr(src), nvox, C, ct, c0, 1, nn.ptr(dst), None) == 0
    want = wide.copy()
    want[:, c0:c0 + C] = narrow
    assert np.array_equal(dst.numpy(), want)
    src, dst = nn.DevArray.from_numpy(wide, "bf16"), nn.DevArray((nvox, C), "bf16", zero=True)
    assert L.mfnn_channels(nn.ptr(src), nvox, C, ct, c0, 0, nn.ptr(dst), None) == 0
    assert np.array_equal(dst.numpy(), wide[:, c0:c0 + C])


@pytest.mark.parametrize("n", [1, 255, 257, 5000])
def test_add_gate(n):
    print(f"[nn-entry] add_gate {n}", flush=True)
    rng = np.random.default_rng(n)
    a, b, gate = (rnd(rng.normal(size=n)) for _ in range(3))
    gate[0] = 0.0
    L = nn.lib()
    ad, bd, gd = (nn.DevArray.from_numpy(v, "bf16") for v in (a, b, gate))
    for with_b in (True, False):
        for with_gate in (True, False):
            out = nn.DevArray((n,), "bf16", zero=True)
            assert L.mfnn_add_gate(nn.ptr(ad), nn.ptr(bd) if with_b else None, nn.ptr(gd) if with_gate else None, n,
                                   nn.ptr(out), None) == 0
            want = rnd(a + b) if with_b else a
            assert np.array_equal(out.numpy(), np.where(gate > 0, want, f32(0)) if with_gate else want)


@pytest.mark.parametrize("cin,cout", [(8, 16), (24, 40), (48, 16), (16, 8)])
def test_flip_weights(cin, cout):
    """alone, and with the weight gradient"""
    print(f"[nn-entry] flip {cin}->{cout}", flush=True)
    rng = np.random.default_rng(cin)
    kp, kp2, cinp = nn.rup(27 * cin, 32), nn.rup(27 * cout, 32), nn.rup(cin, 16)
    w = np.zeros((nn.wrows(cout), kp), f32)
    w[:cout, :27 * cin] = rnd(rng.normal(size=(cout, 27 * cin)))
    want = np.zeros((cinp, kp2), f32)
    for tap in range(27):
        want[:cin, tap * cout:(tap + 1) * cout] = w[:cout, (26 - tap) * cin:(27 - tap) * cin].T
    L = nn.lib()
    wd, wt = nn.DevArray.from_numpy(w, "bf16"), nn.DevArray.from_numpy(np.full((cinp, kp2), 7.0, f32), "bf16")
    assert L.mfnn_flip_weights(nn.ptr(wd), cin, kp, cout, kp2, cinp, nn.ptr(wt), None) == 0
    assert np.array_equal(wt.numpy(), want)
    shape, chunk = (3, 4, 5), 512
    x, dz = nn.DevArray(shape + (cin,), "bf16", zero=True), nn.DevArray(shape + (cout,), "bf16", zero=True)
    work = nn.DevArray((L.mfnn_wgrad_workspace(*shape, kp, cout, chunk),), "f32")
    dw, db = nn.DevArray((nn.rup(cout, 16), kp), "f32"), nn.DevArray((cout,), "f32")
    both = nn.DevArray.from_numpy(np.full((cinp, kp2), 7.0, f32), "bf16")
    assert L.mfnn_conv3_wgrad_flip(nn.ptr(x), nn.ptr(dz), *shape, cin, kp, cout, chunk, nn.ptr(work), nn.ptr(dw), nn.ptr(db), 0,
                                   nn.ptr(wd), kp2, cinp, nn.ptr(both), None) == 0
    assert np.array_equal(both.numpy(), want) and not dw.numpy().any() and not db.numpy().any()
