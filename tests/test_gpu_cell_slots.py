"""tb3_set_cell_slots and single passes: a request made after a cell outgrew its
slots is followed."""
import numpy as np
import pytest
import torch

import threebodymdalgorithms_amd as tb3

pytestmark = pytest.mark.gpu


def test_slots_asked_for_after_a_full_cell(oracle):
    """8000 cells, 60 particles in one of them (32 slots by default): a sweep
    with 256 slots asked for allocates their 65.5 MB, and is right."""
    rng = np.random.default_rng(0)
    P = np.concatenate([rng.uniform(0.0, 30.2, (16000, 3)), rng.uniform(4.6, 5.9, (60, 3))])
    L = np.full(3, 30.2)
    co = oracle.energy(P, cutoff=1.5, L=L)[1]
    with tb3.Engine(0) as eng:
        eng.set_particles(P)
        eng.configure("p3bca", cutoff=1.5, domain_L=L, precision="fp64")
        for _ in range(2):
            assert eng.compute_forces() == co
        free = torch.cuda.mem_get_info()[0]
        eng.set_cell_slots(256)
        for _ in range(2):
            assert eng.compute_forces() == co
        assert free - torch.cuda.mem_get_info()[0] >= 8000 * 256 * 32 - (8 << 20)
