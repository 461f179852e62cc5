"""The population kernel's pair loops, for the calls that the quadratic forms
of a pair potential do not take: rigid-ion genes outside [0, 1], NN2B grids of
fewer than 256 or more than 2048 points."""
import ctypes

import numpy as np
import pytest

from conftest import print_case
from test_gpu_quadform import _dimers, _genes, _oracle, _ri

pytestmark = pytest.mark.gpu


def _wild(genes):
    """One rigid-ion gene outside [0, 1]: the whole call takes the pair loop."""
    g = genes.copy()
    g[0, 3] = -0.01
    return g


def test_launch_shape_is_tuned_when_the_pair_loop_is_first_needed(capfd):
    """Not by autotune() of a set with forms, whose tables may never be built,
    and once for the calls that take the loop."""
    import gpuga_amd as G
    print_case("pair loop, tuning")
    d = _ri(Nc=20)
    genes = _genes(d, 40, 1)

    def lines():
        ctypes.CDLL(None).fflush(None)
        return capfd.readouterr().out.count("autotune P=40")

    with G.Fitness(arrays=d, verbose=1) as fit:
        fit.autotune(40)
        fit.compute(genes)
        assert lines() == 0
        a = fit.compute(_wild(genes), terms=True)
        assert lines() > 1
        b = fit.compute(_wild(genes), terms=True)
        shape = fit.launch_shape(40)
        assert lines() == 0
        assert fit.autotune(40) == shape["chunk_cost"]
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def _case(kind, seed=60):
    """(set, potential, options) of a call that takes the pair loop."""
    import test_gpu_nn2b
    import test_gpu_ragged
    if kind == "ri":
        d = _ri(Nc=8, force=0.4, seed=seed)
    elif kind == "ri_ragged":
        d, _ = test_gpu_ragged._pair_ragged_set("ri", seed)
    elif kind == "nn2b_ragged":
        d, _ = test_gpu_ragged._pair_ragged_set("nn2b", seed)
    elif kind == "species":
        d, _ = test_gpu_nn2b._species_set(12, 10, seed)
    else:
        d = _dimers(300, 120, 12, seed)
    opts = {} if kind.startswith("ri") else dict(
        nn2b_bf16=int(kind == "bf16"), nn2b_grid=2048 if kind == "species" else 4096)
    return d, opts


def _loop_genes(kind, d, P, seed):
    g = _genes(d, P, seed)
    return _wild(g) if kind.startswith("ri") else g


def _takes_the_loop(fit, kind, d, opts, P):
    """After a call: the loop's tables are on the device."""
    if kind.startswith("ri"):
        pairs = int(np.sum(fit.neighbors()[0])) // 2
        return fit.device_bytes() - fit.before >= 16 * pairs
    codes = 3 if kind == "species" else 1
    return fit.device_bytes() >= 3 * 4 * 64 * ((P + 63) // 64) * codes * opts["nn2b_grid"]


@pytest.mark.parametrize("kind,P", [("ri", 70), ("ri", 3), ("ri_ragged", 70), ("ri_ragged", 5),
                                    ("dimers", 70), ("nn2b_ragged", 70), ("nn2b_ragged", 5),
                                    ("species", 70), ("bf16", 70)])
def test_pair_loop_matches_oracle(kind, P):
    """Fitness and terms: 1e-5 relative, 1e-4 with the split-BF16 layer; rigid
    ion's energy and virial terms 5e-5 and so its fitness: its FP32 pair terms
    nearly cancel (both of its FP32 paths show 2 to 3e-5)."""
    import gpuga_amd as G
    print_case("pair loop", kind, P)
    d, opts = _case(kind)
    genes = _loop_genes(kind, d, P, P)
    with G.Fitness(arrays=d, **opts) as fit:
        fit.before = fit.device_bytes()
        f, terms = fit.compute(genes, terms=True)
        again, t2 = fit.compute(genes, terms=True)
        assert _takes_the_loop(fit, kind, d, opts, P)
    assert np.array_equal(f, again) and np.array_equal(terms, t2)
    ref, rterms = _oracle(d).fitness(genes, threads=16)
    tol = np.full(3, 1e-4 if kind == "bf16" else 1e-5)
    if kind.startswith("ri"):
        tol[:2] = 5e-5
    assert np.all(np.abs(f - ref) <= tol.max() * ref)
    assert np.all(np.abs(terms - rterms) <= tol * rterms)


@pytest.mark.parametrize("kind", ["ri", "species", "dimers"])
def test_launch_shape_does_not_change_the_pair_loop(kind):
    """Queues and resident workgroups: the same bits.  Items of a few pairs,
    whose partials pass between waves many times: the same sums regrouped
    (1e-12), ten times the same bits."""
    import gpuga_amd as G
    print_case("pair loop, launch shape", kind)
    P = 130
    d, opts = _case(kind)
    genes = _loop_genes(kind, d, P, 5)

    def run(n=1, **shape):
        with G.Fitness(arrays=d, **opts, **shape) as fit:
            fit.before = fit.device_bytes()
            out = [fit.compute(genes, terms=True)[1] for _ in range(n)]
            assert _takes_the_loop(fit, kind, d, opts, P)
        assert all(np.array_equal(out[0], o) for o in out)
        return out[0]

    ref = run(chunk_cost=200)
    for shape in ({"queues": 16}, {"queues": 3}, {"blocks_per_cu": 1},
                  {"blocks_per_cu": 2, "queues": 64}):
        assert np.array_equal(run(chunk_cost=200, **shape), ref), shape
    np.testing.assert_allclose(run(10, chunk_cost=24), ref, rtol=1e-12)
    np.testing.assert_allclose(run(chunk_cost=10 ** 8), ref, rtol=1e-12)
