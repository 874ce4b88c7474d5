"""Large reads into pinned memory: the same values as into ordinary memory."""
import ctypes as C

import numpy as np
import pytest
import torch

from helpers import small_drainage
from mflbm import gpu

pytestmark = pytest.mark.gpu


def test_read_into_pinned_memory():
    geo, p = small_drainage(n=(84, 84, 85), seed=3, radius=4.0, porosity=0.6, jper=1, buffer=2)
    s = gpu.Solver(p, geo, gpu.FP64)
    s.setup()
    size = gpu.load().mflbm_field_size(s.h, gpu.FIELDS["phi"])
    print(f"[gpu-copy-pinned] {size * 8 / 1e6:.2f} MB", flush=True)
    want = np.arange(size, dtype=np.float64)
    s.upload("phi", want.reshape(s.shape(gpu.HALO["phi"])))
    out = torch.empty(size, dtype=torch.float64, pin_memory=True)
    assert gpu.load().mflbm_download(s.h, gpu.FIELDS["phi"], C.c_void_p(out.data_ptr()), size * 8) == 0
    assert np.array_equal(out.numpy(), want)
    assert np.array_equal(s.download("phi").reshape(-1), want)
