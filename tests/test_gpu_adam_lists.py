"""Adam steps of tensors alone in their launch and in lists: the two kernels give the same bits, also
where a list of 49 leaves one tensor for a second launch."""
import numpy as np
import pytest

from mflbm import nn

pytestmark = pytest.mark.gpu


def step(parts, lists):
    """one step of copies of `parts` in launches of the given tensors; what it leaves"""
    dev = [[nn.DevArray.from_numpy(a) for a in p] + [nn.DevArray((p[0].size,), "bf16", zero=True)] for p in parts]
    for which in lists:
        nn.adam_many([nn.AdamTensor(*(t.data_ptr() for t in dev[k][:4]), parts[k][0].size, dev[k][4].data_ptr() if k % 3 else None)
                      for k in which], 2, 1e-2)
    nn.sync()
    return [[t.numpy() for t in d] for d in dev]


@pytest.mark.parametrize("count", [1, 2, 48, 49])
def test_alone_and_in_lists(count):
    print(f"[gpu-adam-lists] {count}", flush=True)
    rng = np.random.default_rng(count)
    parts = [[np.abs(rng.normal(size=1 + 97 * k)).astype(np.float32) if j == 3 else rng.normal(size=1 + 97 * k).astype(np.float32)
              for j in range(4)] for k in range(count)]
    together, alone = step(parts, [range(count)]), step(parts, [[k] for k in range(count)])
    assert not np.array_equal(together[0][0], parts[0][0])
    for a, b in zip(together, alone):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
