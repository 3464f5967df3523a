"""The bit-exact cutoff sweep's time per triplet with long neighbour lists."""
import time

import numpy as np
import pytest

import threebodymdalgorithms_amd as tb3

pytestmark = pytest.mark.gpu


def test_long_lists_keep_their_waves():
    """8000 particles at cutoff 3.8 (lists of 460, capacity 1024) against 32768 at
    cutoff 2 (67, 128), per triplet: 1.6 times the time with 5 waves per CU, 2.3
    times with lists so large that 3 fit."""
    rng = np.random.default_rng(0)
    per = []
    with tb3.Engine(0) as eng:
        for n, cutoff in ((32768, 2.0), (8000, 3.8)):
            box = (n / 2.0) ** (1.0 / 3.0)
            eng.set_particles(rng.uniform(0.0, box, (n, 3)))
            eng.configure("p3bca", cutoff=cutoff, domain_L=np.full(3, box), precision="exact")
            count = [eng.compute_forces() for _ in range(3)][0]
            times = []
            for _ in range(15):
                start = time.perf_counter()
                eng.compute_forces()
                times.append(time.perf_counter() - start)
            per.append(np.median(times) / count)
    assert per[1] < 1.95 * per[0], per
