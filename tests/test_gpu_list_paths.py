"""The list rebuild at the edges of its paths: the scan of chains beyond 3072 list cells in parts of 8192 (chains
that begin, end and lie across a part), and the build workgroups of 16 waves (up to 512 cells in all) and of 4."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RC, SKIN = 2.5, 0.6


def _start(e, k, N, L, seed):
    s = int(np.ceil(N ** (1 / 3) - 1e-9))
    i = np.arange(N)
    rng = np.random.default_rng(seed)
    x = (np.stack((i % s, (i // s) % s, i // (s * s)), -1) + 0.5 + rng.uniform(-0.1, 0.1, (N, 3))) * (L / s)
    e.set_positions(x, k)
    e.set_momenta(rng.normal(size=(N, 3)), k)


# list cells: 12^3 = 1728, 20^3 = 8000, 24^3 = 13824, 13^3: the parts of 8192 begin inside the second, third
# and third chain
def test_batch_across_scan_parts_equals_single_chains(chmc):
    sizes = [(2000, 38.0), (5000, 62.5), (9000, 75.0), (3000, 40.5)]
    chains = [chmc.Chain(N=n, L=l, cutoff=RC) for n, l in sizes]
    with chmc.Engine(chains) as e:
        e.set_skin(SKIN)
        for k, (n, l) in enumerate(sizes):
            _start(e, k, n, l, 10 + k)
        e.integrate(chmc.LEAPFROG, 0.01, 12)
        e.integrate(chmc.LEAPFROG, 0.01, 12)
        got = [(e.positions(k), e.momenta(k)) for k in range(len(sizes))]
    for k, (n, l) in enumerate(sizes):
        with chmc.Engine(chains[k]) as e:
            e.set_skin(SKIN)
            _start(e, 0, n, l, 10 + k)
            e.integrate(chmc.LEAPFROG, 0.01, 12)
            e.integrate(chmc.LEAPFROG, 0.01, 12)
            assert np.array_equal(e.positions(), got[k][0]) and np.array_equal(e.momenta(), got[k][1]), k


# 1, 8, 512 (the last of 16 waves) and 729 list cells, and an anisotropic box; cells with more members than
# waves, and empty ones
@pytest.mark.parametrize("N,L", [(60, 5.0), (500, 8.9), (12000, 24.9), (12000, 28.0), (200, (25.0, 6.4, 7.0)), (40, 24.9)])
@pytest.mark.parametrize("bits", [32, 16])
def test_build_lists_every_pair(chmc, N, L, bits):
    box = tuple(np.broadcast_to(np.asarray(L, float), (3,)))
    s = int(np.ceil(N ** (1 / 3) - 1e-9))
    rng = np.random.default_rng(N)
    i = np.arange(N)
    x = (np.stack((i % s, (i // s) % s, i // (s * s)), -1) + 0.5 + rng.uniform(-0.15, 0.15, (N, 3))) / s * np.asarray(box)
    with chmc.Engine(chmc.Chain(N=N, L=box, cutoff=RC)) as e:
        e.set_list_entry_bits(bits)
        e.set_skin(SKIN)
        e.set_positions(x)
        _, nint, _ = e.list_stats()
        assert nint == e.pair_counts()[1]
        e.integrate(chmc.LEAPFROG, 0.0, 1)
        fl = e.force()
        e.compute_force(fp64=True)
        f = e.force()
        # FP32 coordinates relative to the cells (2^-22 of a cell side) and FP32 sums of up to ~100 terms
        scale = np.sqrt(np.mean(f ** 2)) + np.max(np.abs(f)) * 1e-2
        near = 4e-2 * (48 * RC ** -7)            # a pair within 1e-6 of rc may fall on either side
        assert np.max(np.abs(fl - f)) <= 2e-4 * scale + near


# rows below, at and past the first batch of every sweep shape (64 to 128 entries; about 125 rho entries a row),
# with the steps after it partly and wholly filled, and a last tile of 5 slots
@pytest.mark.parametrize("rho", [0.5, 0.72, 0.95, 1.1])
@pytest.mark.parametrize("bits", [32, 16])
def test_sweep_shapes_past_the_first_batch(chmc, rho, bits):
    N, dt = 997, 0.004
    L = (N / rho) ** (1 / 3)
    i = np.arange(N)
    rng = np.random.default_rng(7)
    x = (np.stack((i % 10, (i // 10) % 10, i // 100), -1) + 0.5 + rng.uniform(-0.15, 0.15, (N, 3))) / 10 * L
    p = rng.normal(size=(N, 3))
    with chmc.Engine(chmc.Chain(N=N, L=L, cutoff=RC)) as e:
        e.set_list_entry_bits(bits)
        e.set_skin(SKIN)
        first = None
        for lanes in (8, 4, 16, 810, 811, 812, 816):
            e.set_list_lanes(lanes)
            e.set_positions(x)
            e.set_momenta(p)
            e.integrate(chmc.LEAPFROG, 0.0, 1)
            fl = e.force()
            e.compute_force(fp64=True)
            f = e.force()
            # the bound of the lists' forces above
            bound = 2e-4 * (np.sqrt(np.mean(f ** 2)) + np.max(np.abs(f)) * 1e-2) + 4e-2 * (48 * RC ** -7)
            assert np.max(np.abs(fl - f)) <= bound, lanes
            e.integrate(chmc.LEAPFROG, dt, 3)
            end = e.momenta()
            # four kicks of dt with two forces each off by at most the bound (which also holds for the later
            # configurations: their forces are not larger by more than a factor of two)
            first = end if first is None else first
            assert np.max(np.abs(end - first)) <= 4 * dt * 2 * 2 * bound, lanes
