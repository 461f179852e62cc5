"""Pair potentials' population fitness by quadratic forms against the FP64
oracle and the other paths.

Tolerance against the oracle: 1e-5 relative for fitness and terms, the bound
of every FP32 population path (the forms are FP64; the geometry and, for NN2B,
the tabulated network are FP32)."""
import numpy as np
import pytest

from conftest import print_case

pytestmark = pytest.mark.gpu


def _oracle(d):
    from oracle import oracle as O
    keys = ("potential_type", "cutoff", "weights", "pmin", "pmax")
    pot = {k: d[k] for k in keys}
    pot["num_neurons"] = d.get("num_neurons", 0)
    return O.Case(potential=pot, arrays=d)


def _labelled(d):
    from gpuga_amd import synth
    return synth.label(d, _oracle(d).find_force)


def _ri(Nc=6, force=0.5, seed=5, rho=None):
    """Oxide cells, an odd number of force configurations; rho: the unlike
    pairs' lower bound of the Buckingham length (the rate that sets the
    elements)."""
    from gpuga_amd import synth
    d = synth.fluorite_ab2(Nc=Nc, force_fraction=force, seed=seed)
    if rho is not None:
        d["pmin"] = d["pmin"].copy()
        d["pmin"][5] = rho
    return _labelled(d)


def _dimers(Nc, ncf, n, seed, species=False, box=30.0):
    """Pairs from 1.3 to 8 A (inside, in and at the end of the taper)."""
    rng = np.random.default_rng(seed)
    r = np.zeros((3, 2 * Nc), np.float32)
    axis = rng.normal(size=(3, Nc))
    r[:, 1::2] = rng.uniform(1.3, 8.05, Nc) * axis / np.linalg.norm(axis, axis=0)
    V = n * (n + 4) + 1 + (n if species else 0)
    truth = rng.uniform(-1, 1, V).astype(np.float32)
    return _labelled(dict(
        potential_type=4 if species else 3, num_neurons=n, cutoff=8.0, weights=(0.5, 0.3, 0.2),
        Na=np.full(Nc, 2, np.int32), Nc_force=ncf, r=r.reshape(-1),
        type=rng.integers(0, 2, 2 * Nc).astype(np.int32),
        box=np.tile(np.diag([box] * 3).reshape(-1), Nc).astype(np.float32),
        pmin=np.full(V, -3, np.float32), pmax=np.full(V, 3, np.float32), truth=truth,
        pe_ref=np.zeros(Nc, np.float32), virial_ref=np.zeros(6 * Nc, np.float32),
        force_ref=np.zeros(6 * Nc, np.float32)))


def _genes(d, P, seed):
    return np.random.default_rng(seed).random((P, len(d["pmin"])), dtype=np.float32)


@pytest.mark.parametrize("P", [1, 15, 16, 17, 70])
@pytest.mark.parametrize("kind", ["ri", "ri_steep", "dimers", "species"])
def test_forms_match_oracle(kind, P):
    import gpuga_amd as G
    print_case("quadratic forms", kind, P)
    if kind == "ri":
        d = _ri()
    elif kind == "ri_steep":  # more elements
        d = _ri(rho=0.06)
    else:
        d = _dimers(61, 30, 7, 8, species=kind == "species")
    genes = _genes(d, P, P)
    with G.Fitness(arrays=d, nn2b_bf16=0) as fit:
        f, terms = fit.compute(genes, terms=True)
        again, t2 = fit.compute(genes, terms=True)
    assert np.array_equal(f, again) and np.array_equal(terms, t2)
    ref, rterms = _oracle(d).fitness(genes, threads=16)
    np.testing.assert_allclose(f, ref, rtol=1e-5)
    np.testing.assert_allclose(terms, rterms, rtol=1e-5)


def test_rows_in_several_chunks():
    """More configurations and force atoms than one chunk of the set-up."""
    import gpuga_amd as G
    print_case("quadratic forms, chunks")
    d = _dimers(2600, 1100, 6, 9)
    genes = _genes(d, 5, 3)
    with G.Fitness(arrays=d, nn2b_bf16=0) as fit:
        f, terms = fit.compute(genes, terms=True)
    ref, rterms = _oracle(d).fitness(genes, threads=16)
    np.testing.assert_allclose(f, ref, rtol=1e-5)
    np.testing.assert_allclose(terms, rterms, rtol=1e-5)


def test_genes_outside_the_bounds_take_the_pair_loop():
    """Genes outside [0, 1] (a shorter Buckingham length than the elements
    resolve) and a set whose bounds allow any length: the pair loop, whose
    fitness is the oracle's (its terms' accuracy is tested with that path); genes in range afterwards give the same bits as
    before."""
    import gpuga_amd as G
    print_case("quadratic forms, out of range")
    d = _ri()
    genes = _genes(d, 20, 4)
    wild = genes.copy()
    wild[3, 5], wild[7, 4] = -0.4, 1.3
    with G.Fitness(arrays=d) as fit:
        a, ta = fit.compute(genes, terms=True)
        w = fit.compute(wild)
        b, tb = fit.compute(genes, terms=True)
        rows = fit.trace(genes)  # the pair loop's timeline
        c, tc = fit.compute(genes, terms=True)
    assert len(rows) > 0
    for x, tx in ((b, tb), (c, tc)):
        assert np.array_equal(a, x) and np.array_equal(ta, tx)
    ref, _ = _oracle(d).fitness(wild, threads=16)
    np.testing.assert_allclose(w, ref, rtol=1e-5)
    d = _ri(rho=0.0)
    genes[:, 5] = 0.5 + 0.5 * genes[:, 5]
    with G.Fitness(arrays=d) as fit:
        f = fit.compute(genes)
    ref, _ = _oracle(d).fitness(genes, threads=16)
    np.testing.assert_allclose(f, ref, rtol=1e-5)


@pytest.mark.parametrize("kind,P", [("ri", 30), ("dimers", 30), ("large", 64)])
def test_device_generations_equal_the_host_loop(kind, P):
    """large: 64 x 1021 genes, which start from one pinned block but, with the
    history, do not return in one."""
    import gpuga_amd as G
    print_case("quadratic forms, device GA", kind)
    d = _ri() if kind == "ri" else _dimers(40, 20, 30 if kind == "large" else 6, 6)
    with G.Fitness(arrays=d, nn2b_bf16=0) as fit:
        host = G.GA(P, P // 2 + P // 2 % 2, fit.V, maximum_generation=40, seed=3)
        dev = G.GA(P, P // 2 + P // 2 % 2, fit.V, maximum_generation=40, seed=3)
        best = []
        for k in range(5):
            f = fit.compute(host.population)
            best.append(np.min(f))
            host.step(k, f)
        got, _ = fit.run_ga(dev, 0, 5)
    assert np.array_equal(host.population, dev.population)
    assert np.array_equal(np.array(best, np.float32), got)
