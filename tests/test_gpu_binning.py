"""Binning at the edges of its paths (one workgroup up to 3072 atoms and cells, four launches beyond),
against the FP64 oracle's stable counting sort: bitwise."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RC = 2.5


def _check(e, orc, x, L, prev, chain=0):
    perm, cnt, off = e.bins(chain)
    po, co, oo = orc.binning(x, L, RC, perm=prev)
    assert np.array_equal(cnt, co) and np.array_equal(off, oo) and np.array_equal(perm, po)
    return perm


# one atom, one cell, the last sizes of one workgroup (3072 atoms, 3072 cells; of 512 threads: 512 and 512) and the
# first beyond in either
@pytest.mark.parametrize("N,L,order", [
    (1, 6.0, False), (7, 2.6, False), (1023, 11.0, False), (1025, (8.0, 13.0, 40.0), False), (4096, 40.0, False),
    (4096, 17.0, True), (4095, 17.0, False), (4097, 17.0, False), (3000, 43.0, False), (3000, 43.0, True),
    (3072, (40.0, 40.0, 30.0), False), (3073, 17.0, True), (2000, (40.0, 40.0, 32.5), False),
    (512, 20.0, False), (513, 20.0, True), (300, (20.0, 20.0, 22.5), False)])
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


# FP64 sweep: both workgroup shapes (fewer than 512 cells, and more), cells denser than one LDS pass (768
# neighbour entries), atoms with more than 64 neighbours within rc, one- and two-cell boxes, an empty cell
@pytest.mark.parametrize("N,L", [(1, 6.0), (60, 2.6), (700, 5.1), (2500, 8.0), (6000, 20.0), (9000, 21.0), (400, (30.0, 6.0, 5.2)),
                                 (3000, 9.5)])
def test_fp64_sweep_sizes(chmc, orc, N, L):
    box = np.broadcast_to(np.asarray(L, float), (3,)).copy()
    rng = np.random.default_rng(N)
    s = int(np.ceil(N ** (1 / 3) - 1e-9))
    k = np.arange(N)
    x = ((np.stack((k % s, (k // s) % s, k // (s * s)), -1) + 0.5) / s + rng.uniform(-0.2, 0.2, (N, 3)) / s) * box
    x -= box * np.floor(x / box)
    sig = 0.8 * float(np.min(box / s))
    with chmc.Engine(chmc.Chain(N=N, L=tuple(box), cutoff=RC, sigma=sig, beta=0.8)) as e:
        e.set_positions(x)
        e.compute_force(fp64=True)
        f, fo = e.force(), orc.force_binning(x, box, RC, sigma=sig)
        # a few roundings per term of up to several hundred terms, against the largest force
        assert np.max(np.abs(f - fo)) <= 1e-12 * max(np.max(np.abs(fo)), 1e-300)
        V, W = e.compute_potential()[0], e.virial()[0]
        Vo, Wo = orc.potential_binning(x, box, RC, sigma=sig), orc.virial_binning(x, box, RC, sigma=sig)
        assert abs(V - Vo) <= 1e-12 * abs(Vo) and abs(W - Wo) <= 1e-12 * abs(Wo)
        nc, ni = e.pair_counts()
        assert (nc, ni) == orc.pair_counts(x, box, RC)
        # the kick of an FP64 force evaluation
        p = rng.normal(size=(N, 3))
        e.set_momenta(p)
        e.kick(0.01)
        assert np.allclose(e.momenta(), p - 0.01 * 0.8 * f, rtol=0, atol=1e-13 * max(1.0, np.max(np.abs(f))))


# evaluate_potential takes the bins as they are: positions that moved (also across the box) keep their old
# cells, and the pairs are those of the old stencil at the current positions
@pytest.mark.parametrize("N,step", [(2000, 0.05), (2000, 3.0), (20000, 0.3)])
def test_evaluate_potential_with_old_bins(chmc, orc, N, step):
    L = (N / 0.7) ** (1 / 3)
    with chmc.Engine(chmc.Chain(N=N, L=L, cutoff=RC)) as e:
        e.init_lattice(5, 0.1)
        e.bin()
        perm, cnt, off = e.bins()
        e.set_momenta(np.random.default_rng(N).normal(size=(N, 3)))
        e.update_positions(step)
        x = e.positions()
        V = e.evaluate_potential()[0]
        Vo = orc.potential_binning(x, [L] * 3, RC, bins=(perm, cnt, off))
        assert abs(V - Vo) <= 1e-11 * abs(Vo)
        Vn = orc.potential_binning(x, [L] * 3, RC)
        assert abs(e.compute_potential()[0] - Vn) <= 1e-11 * abs(Vn)


# An FP32 cell-path EULER or RUTH sequence ends with a drift that has been counted but not placed (contexts beyond
# one workgroup's binning).  Whatever moves the positions next, the following binning is the stable counting sort
# of the new positions from the last placement, the one of the last force evaluation.  RUTH's placements between
# are not reproduced here, so it runs in atom id order, which does not depend on them.
@pytest.mark.parametrize("N", [700, 4913])
@pytest.mark.parametrize("scheme,order", [("EULER", False), ("RUTH", True)])
@pytest.mark.parametrize("then", ["set", "update", "restore", "train", "bin"])
def test_binning_after_a_counted_drift(chmc, orc, N, scheme, order, then):
    L = (N / 0.7) ** (1 / 3)
    rng = np.random.default_rng(N)
    with chmc.Engine(chmc.Chain(N=N, L=L, cutoff=RC), cell_md=True, atom_id_order=order) as e:
        if then == "train":
            par = {k: rng.normal(size=shp) * 0.1 for k, shp in chmc.SURR_LAYOUT}
            par["scale"] = np.ones(32)
            e.surrogate_set_params(par)
            e.surrogate_reserve_configs(1)
            e.init_lattice(9, 0.1)
            e.surrogate_collect_config()
        e.init_lattice(5, 0.1)
        e.set_momenta(rng.normal(size=(N, 3)))
        e.save_positions()
        prev = None if order else orc.binning(e.positions(), [L] * 3, RC)[0]
        e.integrate(getattr(chmc, scheme), 0.02, 1)
        if then == "set":
            e.set_positions(rng.uniform(0, 1, (N, 3)) * L)
        elif then == "update":
            e.update_positions(0.9)
        elif then == "restore":
            e.restore_positions()
        elif then == "train":
            e.surrogate_train_fm(1, 0.1, 1e-6)
        if then != "train":                    # the training pass has binned already
            e.bin()
        prev = _check(e, orc, e.positions(), [L] * 3, prev)
        e.update_positions(0.3)
        e.bin()
        _check(e, orc, e.positions(), [L] * 3, None if order else prev)


# evaluate_potential after an EULER sequence, whose last drift follows the last force evaluation: the bins are
# those of that evaluation, in contexts of either size (a count of the drifted positions may be pending)
@pytest.mark.parametrize("N", [700, 4913])
def test_evaluate_potential_after_a_counted_drift(chmc, orc, N):
    L = (N / 0.7) ** (1 / 3)
    with chmc.Engine(chmc.Chain(N=N, L=L, cutoff=RC, sigma=0.3), cell_md=True) as e:
        e.init_lattice(5, 0.05)
        bins = orc.binning(e.positions(), [L] * 3, RC)
        e.set_momenta(np.random.default_rng(N).normal(size=(N, 3)))
        e.integrate(chmc.EULER, 0.2, 1)
        x = e.positions()
        V = e.evaluate_potential()[0]
        Vo = orc.potential_binning(x, [L] * 3, RC, sigma=0.3, bins=bins)
        Vn = orc.potential_binning(x, [L] * 3, RC, sigma=0.3)
        assert abs(Vo - Vn) > 1e-7 * abs(Vn)               # the two binnings differ here
        assert abs(V - Vo) <= 1e-11 * abs(Vo)
        assert abs(e.compute_potential()[0] - Vn) <= 1e-11 * abs(Vn)
        e.bin()
        _check(e, orc, x, [L] * 3, bins[0])


def _dense_case(name):
    """(positions, box, cut-off) of a system with cells of many atoms"""
    rng = np.random.default_rng(len(name))
    N, L, rc, ball = {
        "one_cell_160": (160, 5.0, 2.6, None), "one_cell_161": (161, 5.0, 2.6, None), "one_cell_512": (512, 5.0, 2.6, None),
        "eight_cells_512": (512, 5.1, 2.5, None), "one_cell_3072": (3072, 9.0, 5.0, None), "27_cells_3000": (3000, 16.0, 5.3, None),
        "3000_in_a_corner": (3000, 30.0, 2.5, 6.0), "160_of_700": (700, 30.0, 2.5, None), "161_of_700": (700, 30.0, 2.5, None),
        "one_cell_3073": (3073, 9.0, 5.0, None), "27_cells_4096": (4096, 16.0, 5.3, None), "27_cells_8000": (8000, 20.0, 6.6, None),
        "64_a_cell": (8000, 12.6, 2.5, None), "8_cells_20000": (20000, 29.0, 14.0, None),
        "droplet": (9000, 45.0, 2.5, 9.0), "corner": (9000, 45.0, 2.5, 4.0),
        "windows": (140000, 50.0, 10.0, None), "windows_corner": (70000, 80.0, 2.5, 4.0)}[name]
    x = rng.uniform(0, 1, (N, 3)) * L
    if name.endswith("_of_700"):   # so many in one cell of 1728, the others elsewhere
        x = 5.0 + x * (25.0 / L)
        k = rng.permutation(N)[:int(name[:3])]
        x[k] = rng.uniform(0, 2.4, (len(k), 3))
    if ball:                       # two thirds of the atoms close together, in random order of their ids
        k = rng.permutation(N)[:2 * N // 3]
        x[k] = rng.uniform(0, ball, (len(k), 3)) + 1.0
    return x, L, rc


# cells of many atoms: of the one-launch binning at the limit of its pairwise ranking (160 atoms a cell in contexts of
# more than 512 atoms or cells), with 8, 27 and few dense cells among many; of the four-launch one at its limit (64) with a workgroup a cell and with sixteen,
# pairwise (up to 362 keys in one window) and by bits in one window and in several
@pytest.mark.parametrize("name", ["one_cell_160", "one_cell_161", "one_cell_512", "eight_cells_512", "one_cell_3072",
                                  "27_cells_3000", "3000_in_a_corner", "160_of_700", "161_of_700", "one_cell_3073", "27_cells_4096", "27_cells_8000",
                                  "64_a_cell", "8_cells_20000", "droplet", "corner", "windows", "windows_corner"])
@pytest.mark.parametrize("order", [False, True])
def test_binning_dense_cells(chmc, orc, name, order):
    x, L, rc = _dense_case(name)
    N = len(x)
    prev = None
    with chmc.Engine(chmc.Chain(N=N, L=L, cutoff=rc), atom_id_order=order) as e:
        e.set_momenta(np.random.default_rng(3).normal(size=(N, 3)))
        for k in range(3):                       # from atom ids, then from the last order, after small and large moves
            if k == 0:
                e.set_positions(x)
            else:
                e.update_positions(0.1 if k == 1 else 2.0)
            e.bin()
            perm, cnt, off = e.bins()
            po, co, oo = orc.binning(e.positions(), [L] * 3, rc, perm=prev)
            assert np.array_equal(cnt, co) and np.array_equal(off, oo) and np.array_equal(perm, po), k
            prev = None if order else perm


# the time of a binning does not grow with the square of a cell's atoms: systems in eight cells or in one take 1.1
# (3000 atoms), 1.5 to 2.8 (20,000) and 2.2 to 7.1 times (100,000, one cell being one workgroup's work) as long as
# spread out; ranked pairwise they took 9, 200 and 2000 times as long and more
@pytest.mark.parametrize("N,L,times", [(3000, 30.0, 4), (20000, 60.0, 8), (100000, 110.0, 16)])
def test_binning_time_of_dense_cells(chmc, N, L, times):
    rng = np.random.default_rng(N)

    def best(x):
        with chmc.Engine(chmc.Chain(N=N, L=L, cutoff=RC)) as e:
            e.set_positions(x)
            e.bin()
            t = []
            for _ in range(30):
                t0 = time.perf_counter()
                e.bin()
                t.append(time.perf_counter() - t0)
            return min(t)

    spread = best(rng.uniform(0, L, (N, 3)))
    assert best(rng.uniform(0, 5.0, (N, 3))) <= times * spread
    assert best(rng.uniform(0, 2.4, (N, 3))) <= times * spread
