"""Arguments that the network's entry points refuse before they launch anything (no GPU needed:
a call that went on to its launch would report a launch error, -2)."""
from mflbm import nn


def test_adam_many_refuses_negative_sizes():
    """the blocks of one launch are split between the tensors in order, so that a negative size would
    give its neighbours' blocks to other tensors"""
    L = nn.lib()
    f = lambda *sizes: (nn.AdamTensor * len(sizes))(*[nn.AdamTensor(None, None, None, None, n, None) for n in sizes])
    hyper = (1e-2, 0.9, 0.999, 1e-8)
    assert L.mfnn_adam_many(f(1000, -1000), 2, *hyper, 1, None) == -1
    assert L.mfnn_adam_many(f(-1, 1000), 2, *hyper, 1, None) == -1
    assert L.mfnn_adam_many(f(-1), 1, *hyper, 1, None) == -1
    assert L.mfnn_adam_many(None, 1, *hyper, 1, None) == -1
    assert L.mfnn_adam_many(f(10), -1, *hyper, 1, None) == -1
    assert L.mfnn_adam_many(f(10), 1, *hyper, 0, None) == -1
    # nothing to do
    assert L.mfnn_adam_many(f(0, 0), 2, *hyper, 1, None) == 0
    assert L.mfnn_adam_many(None, 0, *hyper, 1, None) == 0
