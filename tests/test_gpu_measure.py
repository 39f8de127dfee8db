"""The pair measurements (RDF histogram, open-boundary sum) at the edges of their kernels, against plain
numpy in FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rdf_counts(x, L, nb, size):
    """Ordered pair counts per bin: the minimum image of every dimension as min((d-L)^2, d^2, (d+L)^2),
    bin = (int)(r / size)."""
    L = np.broadcast_to(np.asarray(L, float), (3,))
    c = np.zeros(nb, np.uint64)
    for i in range(len(x) - 1):
        d = x[i + 1:] - x[i]
        q = np.minimum(np.minimum((d - L) ** 2, d * d), (d + L) ** 2)
        b = np.minimum(np.sqrt((q[:, 0] + q[:, 1]) + q[:, 2]) / size, 2.0 ** 30).astype(np.int64)
        c += 2 * np.bincount(b[b < nb], minlength=nb).astype(np.uint64)
    return c


def _lattice(N, L):
    s = int(np.ceil(N ** (1 / 3) - 1e-9))
    k = np.arange(N)
    return (np.stack((k % s, (k // s) % s, k // (s * s)), -1) + 0.5) * (np.asarray(L, float) / s)


# one atom, tiles of 256 i atoms and 32 j atoms with remainders, an anisotropic box, one bin, the most bins,
# bins so narrow or so wide that every pair is decided in FP64, and a lattice whose distances lie on bin edges
@pytest.mark.parametrize("N,L,nb,size,lattice", [
    (1, 6.0, 10, 0.3, False), (2, 6.0, 10, 0.6, False), (31, 6.0, 100, 0.05, False), (255, 7.0, 64, 0.06, False),
    (257, 7.0, 333, 0.02, False), (289, (5.0, 7.5, 11.0), 200, 0.04, False), (1025, 11.0, 1, 2.0, False),
    (1100, 11.0, 4000, 0.0025, False), (600, 9.0, 50, 1e-9, False), (600, 9.0, 50, 40.0, False),
    (512, 16.0, 64, 0.5, True), (512, 16.0, 16, 2.0, True), (700, (9.0, 9.0, 18.0), 90, 0.1, True)])
def test_rdf_counts_edges(chmc, N, L, nb, size, lattice):
    box = np.broadcast_to(np.asarray(L, float), (3,))
    x = _lattice(N, box) if lattice else np.random.default_rng(N + nb).uniform(0, 1, (N, 3)) * box
    with chmc.Engine(chmc.Chain(N=N, L=tuple(box), cutoff=2.5)) as e:
        e.set_positions(x)
        counts, _ = e.rdf(nb, size)
    assert np.array_equal(counts, _rdf_counts(x, box, nb, size))


def _open_sum(x, n, a, b):
    """(sum over pairs of a / r^n - b / r^6, sum of the terms' magnitudes)"""
    v = m = 0.0
    for i in range(len(x) - 1):
        r = np.sqrt(((x[i + 1:] - x[i]) ** 2).sum(1))
        p, q = a / r ** float(n), b / r ** 6.0
        v += (p - q).sum()
        m += (np.abs(p) + np.abs(q)).sum()
    return v, m


# 64-tiles with remainders up to their last size, the first size of the 256-tiles, and exponents even, odd,
# zero and negative.  Each term is within ~|n| roundings of the exact one and the sums add ~50 more, so the
# bound is 1e-13 of the terms' magnitudes
@pytest.mark.parametrize("N,n", [(2, 12), (3, 9), (63, 12), (64, 7), (65, 1), (130, 0), (200, -2), (257, 12), (1000, 8),
                                 (16384, 12), (16385, 12)])
def test_open_potential_edges(chmc, N, n):
    x = np.ascontiguousarray(_lattice(N, [1.1 * np.ceil(N ** (1 / 3) - 1e-9)] * 3)
                             + np.random.default_rng(N).uniform(-0.2, 0.2, (N, 3)))
    got = chmc.potential_energy_open(x, n=n, a=4.0, b=3.0)
    v, m = _open_sum(x, n, 4.0, 3.0)
    assert abs(got - v) <= 1e-13 * m, (got, v, m)


def test_open_potential_coincident_pair(chmc):
    x = np.zeros((5, 3))
    x[2:] = [[1, 0, 0], [0, 1.2, 0], [0, 0, 1.3]]
    assert np.isnan(chmc.potential_energy_open(x, a=4.0, b=4.0))      # inf - inf, as a / 0 - b / 0


# bins far below the fixed-point step of the coordinates (2^-32 L = 2e-9): pairs all over the counted range, the last
# bins among them, for which the FP32 quotient is off by several bins
@pytest.mark.parametrize("L,nb,size", [(9.0, 50, 1e-9), ((7.0, 9.0, 11.0), 50, 1e-9), (9.0, 400, 1e-10), (9.0, 3, 5e-11)])
def test_rdf_counts_bins_below_the_coordinate_step(chmc, L, nb, size):
    box = np.broadcast_to(np.asarray(L, float), (3,))
    rng = np.random.default_rng(nb)
    a = rng.uniform(0.1, 0.9, (400, 3)) * box
    u = rng.normal(size=(400, 3))
    u /= np.sqrt((u * u).sum(1))[:, None]
    x = np.concatenate((a, a + u * (rng.uniform(0, 1.2, 400) * nb * size)[:, None]))
    want = _rdf_counts(x, box, nb, size)
    assert want.sum() > 600 and want[-(nb // 20 + 1):].sum() > 0
    with chmc.Engine(chmc.Chain(N=800, L=tuple(box), cutoff=2.5)) as e:
        e.set_positions(x)
        counts, _ = e.rdf(nb, size)
    assert np.array_equal(counts, want)
