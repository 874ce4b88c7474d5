"""The network's pooling, upsampling and branch-point passes against numpy, at the forms where a
row pass can go wrong: channel counts in whole and broken groups of eight, pointers aligned for 16
bytes and not, rows shorter than a wave and longer than a workgroup, parts of wider tensors.
The passes move bfloat16 values and add at most eight of them in float32 in a fixed order, so the
results must be the same bits."""
import ctypes as C

import numpy as np
import pytest

from mflbm import nn

pytestmark = pytest.mark.gpu

f32 = np.float32


def rnd(a):
    return nn.bf16_values(nn.bf16_bits(np.asarray(a, f32)))


def values(rng, shape):
    a = np.asarray(rng.normal(size=shape), f32)
    flat = a.reshape(-1)
    flat[:4] = [0.0, -0.0, np.inf, -3.0e38]
    return rnd(a)


class Buf:
    """a bfloat16 tensor at an offset of `shift` elements in its allocation"""

    def __init__(self, a, shift):
        self.shift, self.shape = shift, a.shape
        full = np.zeros(a.size + shift, f32)
        full[shift:] = a.reshape(-1)
        self.t = nn.DevArray.from_numpy(full, "bf16")

    def ptr(self):
        return C.c_void_p(self.t.data_ptr() + 2 * self.shift)

    def numpy(self):
        nn.sync()
        return np.asarray(self.t.numpy(), f32)[self.shift:].reshape(self.shape)


def blocks(x):
    """the eight voxels of each 2x2x2 block in the order dz, dy, dx"""
    return [x[dz::2, dy::2, dx::2] for dz in (0, 1) for dy in (0, 1) for dx in (0, 1)]


def sum8(x):
    s = np.zeros(x[::2, ::2, ::2].shape, f32)
    for b in blocks(x):
        s = s + b
    return s


def up(x):
    return x.repeat(2, 0).repeat(2, 1).repeat(2, 2)


CASES = [((2, 2, 2), 8, 8, 0), ((4, 6, 10), 16, 24, 0), ((2, 4, 70), 40, 16, 0), ((6, 2, 4), 5, 8, 0), ((4, 4, 6), 8, 3, 0),
         ((2, 6, 34), 16, 8, 1), ((2, 2, 514), 8, 8, 0)]


@pytest.mark.parametrize("shape,cl,cs,shift", CASES)
def test_row_passes(shape, cl, cs, shift):
    print(f"[gpu-conv-rows] {shape} {cl}+{cs} shift {shift}", flush=True)
    rng = np.random.default_rng(cl + 100 * cs + shape[2])
    L, ct = nn.lib(), cl + cs
    coarse = tuple(n // 2 for n in shape)
    low, skip, wide = values(rng, coarse + (cl,)), values(rng, shape + (cs,)), values(rng, shape + (ct,))
    gate, pooled, fgate = values(rng, coarse + (cl,)), values(rng, coarse + (cs,)), values(rng, shape + (cs,))
    b = {k: Buf(v, shift) for k, v in dict(low=low, skip=skip, wide=wide, gate=gate, pooled=pooled, fgate=fgate).items()}
    out = {k: Buf(np.full(s, 7.0, f32), shift) for k, s in
           dict(cat=shape + (ct,), up=shape + (ct,), split=coarse + (cl,), plain=coarse + (cl,), merge=shape + (cs,),
                adj=shape + (cs,), pool=coarse + (cs,)).items()}
    with np.errstate(all="ignore"):
        assert L.mfnn_up2_cat(b["low"].ptr(), cl, b["skip"].ptr(), cs, *shape, ct, 0, out["cat"].ptr(), None) == 0
        assert np.array_equal(out["cat"].numpy(), np.concatenate([up(low), skip], 3))
        assert L.mfnn_up2(b["low"].ptr(), *shape, cl, ct, cs, out["up"].ptr(), 0, None) == 0
        assert np.array_equal(out["up"].numpy(), np.concatenate([np.full(shape + (cs,), 7.0, f32), up(low)], 3))
        s = rnd(sum8(wide[..., :cl]))
        assert L.mfnn_up2(b["wide"].ptr(), *shape, cl, ct, 0, out["plain"].ptr(), 1, None) == 0
        assert np.array_equal(out["plain"].numpy(), s)
        assert L.mfnn_up2_split(b["wide"].ptr(), *shape, cl, ct, 0, b["gate"].ptr(), out["split"].ptr(), None) == 0
        assert np.array_equal(out["split"].numpy(), np.where(gate > 0, s, f32(0)))
        adj = rnd(f32(0.125) * up(pooled))
        assert L.mfnn_pool2(b["pooled"].ptr(), *shape, cs, out["adj"].ptr(), 1, None) == 0
        assert np.array_equal(out["adj"].numpy(), adj)
        assert L.mfnn_pool2_merge(b["pooled"].ptr(), *shape, cs, b["wide"].ptr(), ct, cl, b["fgate"].ptr(),
                                  out["merge"].ptr(), None) == 0
        assert np.array_equal(out["merge"].numpy(), np.where(fgate > 0, rnd(wide[..., cl:] + adj), f32(0)), equal_nan=True)
        assert L.mfnn_pool2(b["skip"].ptr(), *shape, cs, out["pool"].ptr(), 0, None) == 0
        assert np.array_equal(out["pool"].numpy(), rnd(f32(0.125) * sum8(skip)), equal_nan=True)


def test_adam_many_matches_one_by_one():
    """more tensors than one launch holds, empty and odd sizes among them: the same bits as a call
    per tensor"""
    rng = np.random.default_rng(5)
    sizes = [1, 255, 256, 257, 0, 1000] * 9
    print(f"[gpu-conv-rows] adam {len(sizes)} tensors", flush=True)
    full = [[np.asarray(rng.normal(size=n + 1), f32) for n in sizes] for _ in range(4)]
    full[3] = [np.abs(m) for m in full[3]]
    a, b = [[[nn.DevArray.from_numpy(v) for v in part] for part in full] + [[nn.DevArray((n + 1,), "bf16", zero=True) for n in sizes]]
            for _ in range(2)]
    nn.adam_many([nn.AdamTensor(*(a[j][i].data_ptr() for j in range(4)), n, a[4][i].data_ptr() if i % 3 else None)
                  for i, n in enumerate(sizes)], 3, 1e-2)
    for i, n in enumerate(sizes):
        if n:
            assert nn.lib().mfnn_adam(*(nn.ptr(b[j][i]) for j in range(4)), n, 1e-2, 0.9, 0.999, 1e-8, 3,
                                      nn.ptr(b[4][i]) if i % 3 else None, None) == 0
    nn.sync()
    for j in (0, 2, 3, 4):
        for i in range(len(sizes)):
            assert np.array_equal(a[j][i].numpy(), b[j][i].numpy()), (j, i)
