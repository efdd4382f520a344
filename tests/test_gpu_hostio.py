"""F2 between host and device at the sizes where the transfer changes its way
(the runtime's copy, the pinned ring, last chunks of any length), and from
several host threads at once, each with its own context."""
import threading

import numpy as np
import pytest

from conftest import gpu_available
from ramgpu.capi import RamGpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="no GPU")]

# (NS, NR, NT, NE, NPA): 0.3 MB; 8 MiB less and more a column; 33 and 75 MB
DIMS = [(2, 6, 7, 13, 35), (1, 16, 32, 32, 63), (1, 16, 32, 32, 64), (1, 16, 33, 32, 65), (3, 17, 31, 37, 71),
        (4, 23, 41, 35, 71)]


def _round_trips(dims, seed, n):
    rng = np.random.default_rng(seed)
    g = RamGpu(*dims)
    try:
        for _ in range(n):
            f = np.asfortranarray(rng.standard_normal(dims))
            g.put_f2(f)
            np.testing.assert_array_equal(g.get_f2(), f)
    finally:
        g.close()


@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "x".join(map(str, d)))
def test_f2_round_trip(dims):
    _round_trips(dims, sum(dims), 2)


def test_f2_round_trips_from_threads():
    errors = []

    def work(i):
        try:
            _round_trips(DIMS[2 + i], i, 4)
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]
