"""Transfers through the pinned buffers of a context whose device is not the current one (needs two GPUs)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# creating a context makes its device current; positions and momenta of a context on another device still cross, in
# one part and in several
@pytest.mark.parametrize("N,L", [(500, 9.0), (200000, 62.0)])
def test_transfers_with_another_device_current(chmc, N, L):
    x = np.random.default_rng(1).uniform(0, 1, (N, 3)) * L
    with chmc.Engine(chmc.Chain(N=N, L=L, cutoff=2.5), device=0) as a:
        try:
            b = chmc.Engine(chmc.Chain(N=100, L=10.0), device=1)
        except chmc.ChmcError:
            pytest.skip("one GPU")
        with b:
            a.set_positions(x)
            a.set_momenta(-x)
            assert np.array_equal(a.positions(), x) and np.array_equal(a.momenta(), -x)
            y = x[:100] * (10.0 / L)
            b.set_positions(y)
            assert np.array_equal(b.positions(), y)
