"""Tersoff sets of 5 to 21 neighbours within R2 (the unordered-pair kernel's
bond bounds of 8, 16 and 20, one neighbour on either side of each, and the
looped kernel above) against the FP64 oracle: a central atom with exactly k
neighbours among atoms with fewer, force and energy configurations, one and
two species, several lane blocks.  Fitness within 1e-5 relative of the
oracle, the bound of every FP32 population path; terms within 2e-5 of the
per-individual path's, the bound between the two paths."""
import numpy as np
import pytest

from conftest import print_case

pytestmark = pytest.mark.gpu

ONE = (np.array([2.9, 1.3, 2.2, 1.8, 0.5, 0.05, -0.8, 2.6, 3.2], np.float32),
       np.array([3.3, 1.5, 2.4, 2.2, 0.8, 0.4, -0.6, 2.7, 3.2], np.float32))
TWO = (np.concatenate([ONE[0][:4], ONE[0][:4], ONE[0][4:]]),
       np.concatenate([ONE[1][:4], ONE[1][:4], ONE[1][4:]]))


def _set(k, two, seed):
    """Five clusters of 1 + k, 1 + k/2, 4, 1 + k and 3 atoms: points spread over
    a sphere around a centre (and, with few, out of each other's reach)."""
    from gpuga_amd import synth
    from oracle import oracle as O
    rng = np.random.default_rng(seed)
    cells = []
    for n in (k, max(k // 2, 2), 3, k, 2):
        j = np.arange(n) + 0.5
        th, ph = np.arccos(1 - 2 * j / n), np.pi * (1 + 5 ** 0.5) * j
        p = 2.8 * np.stack([np.cos(ph) * np.sin(th), np.sin(ph) * np.sin(th), np.cos(th)], 1)
        p = np.concatenate([[[0, 0, 0]], p]) + rng.normal(0, 0.03, (n + 1, 3)) + 10.0
        cells.append((np.diag([20.0] * 3), p, (np.arange(n + 1) % 2 if two else
                                               np.zeros(n + 1)).astype(np.int32)))
    d = synth._assemble(cells, 0.4, rng)
    lo, hi = TWO if two else ONE
    d.update(potential_type=2 if two else 1, cutoff=3.2, weights=(0.3, 0.3, 0.4), pmin=lo, pmax=hi,
             truth=(0.5 * (lo + hi)).astype(np.float32))
    pot = {x: d[x] for x in ("potential_type", "cutoff", "weights", "pmin", "pmax")}
    return synth.label(d, O.Case(potential=pot, arrays=d).find_force), pot


@pytest.mark.parametrize("k,two", [(5, False), (8, True), (9, False), (16, True), (17, False),
                                   (20, True), (21, False)])
def test_neighbour_bounds_match_oracle(k, two):
    import gpuga_amd as G
    from oracle import oracle as O
    print_case("tersoff neighbours", k, two)
    d, pot = _set(k, two, k)
    genes = np.random.default_rng(k).random((70, len(d["pmin"])), dtype=np.float32)
    with G.Fitness(arrays=d) as fit:
        assert fit.max_neighbors == k
        f, terms = fit.compute(genes, terms=True)
        again, t2 = fit.compute(genes, terms=True)
        _, plain = fit.compute(genes, terms=True, plain=True)
    assert np.array_equal(f, again) and np.array_equal(terms, t2)
    ref, _ = O.Case(potential=pot, arrays=d).fitness(genes, threads=16)
    np.testing.assert_allclose(f, ref, rtol=1e-5)
    np.testing.assert_allclose(terms, plain, rtol=2e-5)


@pytest.mark.parametrize("k,two", [(3, False), (4, True), (5, False)])
def test_per_atom_outputs_of_few_neighbours(k, two):
    """find_force of the one-pass kernel (at most four neighbours) and of the
    two-kernel form above it, with atoms of 0 to k neighbours, the last atom of
    the set among those without; 2e-5 of the largest magnitude, the bound of
    every per-atom FP32 output."""
    import gpuga_amd as G
    from gpuga_amd import synth
    from oracle import oracle as O
    print_case("tersoff per-atom outputs", k, two)
    rng = np.random.default_rng(k)
    cells = []
    for n in (k, 1, 2, k, 0):  # a centre with n neighbours, and one atom out of reach
        th = np.arccos(np.linspace(0.9, -0.9, max(n, 1)))[:n]
        ph = 2.4 * np.arange(n)
        p = 2.4 * np.stack([np.cos(ph) * np.sin(th), np.sin(ph) * np.sin(th), np.cos(th)], 1)
        p = np.concatenate([[[0, 0, 0]], p + rng.normal(0, 0.03, p.shape), [[9, 9, 9]]]) + 5.0
        cells.append((np.diag([20.0] * 3), p, (np.arange(n + 2) % 2 if two else
                                               np.zeros(n + 2)).astype(np.int32)))
    d = synth._assemble(cells, 0.4, rng)
    lo, hi = TWO if two else ONE
    d.update(potential_type=2 if two else 1, cutoff=2.75, weights=(0.3, 0.3, 0.4), pmin=lo, pmax=hi,
             pe_ref=np.ones(5, np.float32), virial_ref=np.ones(30, np.float32),
             force_ref=np.ones(d["r"].size, np.float32))
    pot = {x: d[x] for x in ("potential_type", "cutoff", "weights", "pmin", "pmax")}
    params = (lo + (hi - lo) * rng.random(len(lo))).astype(np.float32)
    with G.Fitness(arrays=d) as fit:
        NN, _, _ = fit.neighbors()
        got = fit.find_force(params)
    assert NN.max() == k and NN[-1] == 0
    for a, b in zip(got, O.Case(potential=pot, arrays=d).find_force(params)):
        np.testing.assert_allclose(a, b, rtol=0, atol=2e-5 * np.abs(b).max())
