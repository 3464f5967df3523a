"""A device-pointer call that is refused leaves its outputs as they were."""
import numpy as np
import pytest
import torch

import threebodymdalgorithms_amd as tb3

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32", "exact"])
@pytest.mark.parametrize("grad", [False, True])
def test_refused_call_leaves_the_outputs(precision, grad):
    """More neighbours than a list holds (16384): found after the sweep's first
    tries, whose sums must not show.  The next call on the context is served."""
    n = 16600
    P = np.random.default_rng(3).uniform(5.0, 5.6, (n, 3))
    L = np.full(3, 12.0)
    with tb3.Engine(0) as eng:
        eng.configure("p3bca", cutoff=2.0, domain_L=L, precision=precision)
        x = torch.tensor(P, device="cuda")
        E = torch.full((), 7.0, dtype=torch.float64, device="cuda")
        G = torch.full_like(x, 7.0)
        torch.cuda.synchronize()

        def call(m):
            if grad:
                return eng.energy_grad_dev(m, x.data_ptr(), 1.0, E.data_ptr(), G.data_ptr(), want_count=True)
            return eng.energy_dev(m, x.data_ptr(), 1.0, E.data_ptr(), want_count=True)

        with pytest.raises(tb3.TB3Error, match="neighbours"):
            call(n)
        assert float(E) == 7.0 and bool((G == 7.0).all())
        assert call(40) == 40 * 39 * 38 // 6
        assert float(E) != 7.0 and bool((G[40:] == 7.0).all()) and bool((G[:40] != 7.0).all()) == grad
