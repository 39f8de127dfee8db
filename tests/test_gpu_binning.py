"""Binning at the edges of its paths (one workgroup up to 4096 atoms and cells, four launches beyond),
against the FP64 oracle's stable counting sort: bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RC = 2.5


def _check(e, orc, x, L, prev, chain=0):
    perm, cnt, off = e.bins(chain)
    po, co, oo = orc.binning(x, L, RC, perm=prev)
    assert np.array_equal(cnt, co) and np.array_equal(off, oo) and np.array_equal(perm, po)
    return perm


# one atom, one cell, the last sizes of one workgroup (4096 atoms, 4096 cells) and the first beyond in either
@pytest.mark.parametrize("N,L,order", [
    (1, 6.0, False), (7, 2.6, False), (1023, 11.0, False), (1025, (8.0, 13.0, 40.0), False), (4096, 40.0, False),
    (4096, 17.0, True), (4095, 17.0, False), (4097, 17.0, False), (3000, 43.0, False), (3000, 43.0, True)])
def test_binning_sizes(chmc, orc, N, L, order):
    box = np.broadcast_to(np.asarray(L, float), (3,)).copy()
    rng = np.random.default_rng(N)
    x = rng.uniform(0, 1, (N, 3)) * box
    with chmc.Engine(chmc.Chain(N=N, L=tuple(box), cutoff=RC), atom_id_order=order) as e:
        e.set_positions(x)
        e.bin()
        prev = _check(e, orc, x, box, None)
        # stable with respect to the previous permutation after a drift; all atoms in one corner at last
        e.set_momenta(rng.normal(size=(N, 3)) * 3.0)
        e.update_positions(0.7)
        e.bin()
        prev = _check(e, orc, e.positions(), box, None if order else prev)
        x = rng.uniform(0, 1, (N, 3)) * 2.4
        e.set_positions(x)
        e.bin()
        _check(e, orc, x, box, None if order else prev)


def test_binning_two_chains(chmc, orc):
    rng = np.random.default_rng(2)
    Ns, Ls = (700, 1300), (9.5, 12.5)
    with chmc.Engine([chmc.Chain(N=n, L=l, cutoff=RC) for n, l in zip(Ns, Ls)]) as e:
        xs = [rng.uniform(0, l, (n, 3)) for n, l in zip(Ns, Ls)]
        for k, x in enumerate(xs):
            e.set_positions(x, k)
        e.bin()
        for k, x in enumerate(xs):
            _check(e, orc, x, [Ls[k]] * 3, None, k)


# the cell path of both sizes runs the integrator with the same arithmetic: kick, drift and force of the
# per-call API against one integrate call (FP64 forces, bitwise)
@pytest.mark.parametrize("N", [500, 4913])
def test_cell_md_sequence(chmc, N):
    L = (N / 0.8) ** (1 / 3)
    rng = np.random.default_rng(N)
    out = []
    for whole in (True, False):
        with chmc.Engine(chmc.Chain(N=N, L=L, cutoff=RC, beta=0.7), fp64_forces=True) as e:
            e.init_lattice(3, 0.05)
            e.set_momenta(np.random.default_rng(1).normal(size=(N, 3)))
            if whole:
                e.integrate(chmc.LEAPFROG, 0.004, 3)
            else:
                e.update_momenta(0.002)
                for k in range(3):
                    e.update_positions(0.004)
                    e.update_momenta(0.002 if k == 2 else 0.004)
            out.append((e.positions(), e.momenta()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
