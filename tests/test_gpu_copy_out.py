"""Large copies to the host (pinned slots, several threads) against the same field read in small
pieces: sizes in whole and broken chunks, several threads on one handle and on two."""
import threading

import numpy as np
import pytest

from helpers import small_drainage
from mflbm import gpu

pytestmark = pytest.mark.gpu


def solver(n, seed):
    geo, p = small_drainage(n=n, seed=seed, radius=4.0, porosity=0.6, jper=1, buffer=2)
    s = gpu.Solver(p, geo, gpu.FP64)
    s.setup()
    return s


# phi: 6.3 MB (just above the staged copy's least size), 6.0 (below), 13.1 and 36 (chunks of a share, of a slot)
@pytest.mark.parametrize("n", [(84, 84, 85), (82, 82, 85), (110, 110, 110), (157, 157, 157)])
def test_upload_comes_back(n):
    s = solver(n, 3)
    size = gpu.load().mflbm_field_size(s.h, gpu.FIELDS["phi"])
    print(f"[gpu-copy-out] {n} {size * 8 / 1e6:.2f} MB", flush=True)
    want = np.arange(size, dtype=np.float64).reshape(s.shape(gpu.HALO["phi"]))
    s.upload("phi", want)
    for _ in range(2):
        assert np.array_equal(s.download("phi"), want)


def test_threads_on_one_and_two_handles():
    print("[gpu-copy-out] threads", flush=True)
    a, b = solver((100, 100, 100), 4), solver((101, 99, 100), 5)
    want = [s.download("phi") for s in (a, b)]
    bad = []

    def read(k):
        for _ in range(4):
            if not np.array_equal((a, b)[k].download("phi"), want[k]):
                bad.append(k)

    threads = [threading.Thread(target=read, args=(k,)) for k in (0, 0, 1, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
