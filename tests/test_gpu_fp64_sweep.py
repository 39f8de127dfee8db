"""The FP64 force sweep at the edges of its launch shapes: several workgroups of 8 waves a cell (with waves that get
several atoms, one or none, and workgroups that get none), one, and workgroups of 4 waves beyond 2048 cells."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RC = 2.5


# cells x workgroups: 1 x 39, 8 x 7, 27 x 4, 27 x 9, 512 x 1 or 2, 2048 x 1, 2197, and clustered atoms in mostly empty
# cells (the mean asks for one workgroup, cells hold hundreds)
@pytest.mark.parametrize("N,L,cluster", [
    (234, 4.9, False), (300, 5.2, False), (512, 8.6, False), (1500, 9.9, False), (5000, 20.2, False),
    (9000, 20.2, False), (3000, (40.2, 40.2, 20.2), False), (3000, 32.7, False), (1200, 30.0, True)])
def test_fp64_sweep_shapes(chmc, orc, N, L, cluster):
    box = np.broadcast_to(np.asarray(L, float), (3,)).copy()
    s = int(np.ceil(N ** (1 / 3) - 1e-9))
    i = np.arange(N)
    rng = np.random.default_rng(N)
    x = (np.stack((i % s, (i // s) % s, i // (s * s)), -1) + 0.5 + rng.uniform(-0.1, 0.1, (N, 3))) / s
    x = x * (0.35 if cluster else 1.0) * box
    p = rng.normal(size=(N, 3))
    f = orc.force_binning(x, box, RC)
    # every pair term within a few units of 2^-53, up to a few hundred terms an atom, in any order
    tol = 1e-12 * np.max(np.abs(f)) + 1e-13 * 48 * len(f) ** 0.5
    with chmc.Engine(chmc.Chain(N=N, L=tuple(box), cutoff=RC), fp64_forces=True) as e:
        e.set_positions(x)
        e.set_momenta(p)
        e.compute_force(fp64=True)
        assert np.max(np.abs(e.force() - f)) <= tol
        dt = 1e-3
        e.update_momenta(dt)
        assert np.max(np.abs(e.momenta() - (p - dt * f))) <= dt * tol + 1e-15 * np.max(np.abs(p)) + dt * 1e-15 * np.max(np.abs(f))
