"""The three terms of the Tersoff population kernels against the FP64 oracle: as
near to it as the per-individual path, whose FP32 bond lengths and labels are
the same, and 1e-5 relative (1e-7 absolute for terms near zero)."""
import numpy as np
import pytest

import test_gpu_tersoff_moments as moments
import test_gpu_tersoff_shell as shell
from conftest import print_case

pytestmark = pytest.mark.gpu


def _crystal(cutoff, two):
    """Diamond cells whose taper ends past the second shell."""
    from gpuga_amd import synth
    from oracle import oracle as O
    d = synth.tersoff_si(Nc=10, reps=(3, 3, 3), seed=9)
    lo, hi = (a.copy() for a in (shell.TWO if two else shell.ONE))
    lo[-2], hi[-2] = cutoff - 1.0, cutoff - 0.6
    lo[-1] = hi[-1] = cutoff
    if two:
        d["type"] = np.tile(np.repeat(np.arange(2, dtype=np.int32), 4), len(d["type"]) // 8)
    d.update(potential_type=2 if two else 1, cutoff=cutoff, pmin=lo, pmax=hi,
             truth=(0.5 * (lo + hi)).astype(np.float32))
    pot = {x: d[x] for x in ("potential_type", "cutoff", "weights", "pmin", "pmax")}
    return synth.label(d, O.Case(potential=pot, arrays=d).find_force), pot


@pytest.mark.parametrize("kind,two,P", [
    ("strained", False, 70), ("strained", True, 20), ("alloy", True, 70), ("vacancy", False, 68),
    ("angle", False, 70), (8, False, 70), (16, True, 70), (20, False, 70), (3.6, False, 70),
    (3.9, True, 70), (4.0, False, 64)])
def test_terms_match_oracle(kind, two, P):
    """kind: a set of the moment records, neighbours of the clusters' centre, or
    a crystal's cut-off."""
    import gpuga_amd as G
    from oracle import oracle as O
    print_case("tersoff terms", kind, two, P)
    d, pot = (moments._set(kind, two) if isinstance(kind, str) else
              shell._set(kind, two, kind) if isinstance(kind, int) else _crystal(kind, two))
    genes = np.random.default_rng(P).random((P, len(d["pmin"])), dtype=np.float32)
    with G.Fitness(arrays=d) as fit:
        _, terms = fit.compute(genes, terms=True)
        _, plain = fit.compute(genes, terms=True, plain=True)
        assert isinstance(kind, str) or fit.max_neighbors > 4
    _, ref = O.Case(potential=pot, arrays=d).fitness(genes, threads=16)
    assert np.all(np.abs(terms - ref) <= 1e-5 * ref + 1e-7 + np.abs(plain - ref))
