"""Tersoff energy configurations whose atoms take their energy and virial from
moment records (four bonds of one kind inside every individual's R1) and those
that do not: bonds on both sides of R1, both kinds of bond at an atom, fewer
neighbours, and h next to the bond angles' cosine, where the records' sum of
squares is a small difference.  Full, packed and partial lane blocks, and
launches of one wave a SIMD.  Fitness within 1e-5 relative of the FP64 oracle,
the bound of every FP32 population path; terms within 2e-5 of the
per-individual path's (a term near zero: 1e-7, as for the ragged sets)."""
import numpy as np
import pytest

from conftest import print_case

pytestmark = pytest.mark.gpu


def _set(kind, two):
    from gpuga_amd import synth
    from oracle import oracle as O
    rng = np.random.default_rng(17)
    angle = kind == "angle"
    d = synth.tersoff_si(Nc=10, reps=(2, 2, 1), disp=0.03 if angle else 0.1,
                         strain=0.005 if angle else 0.03, force_fraction=0.2, seed=17)
    if angle:  # one sublattice along [111]: a bond's three angles are alike, not 109.5 degrees
        d["r"] = (d["r"].reshape(3, -1, 8) + 0.173 * (np.arange(8) >= 4)).astype(np.float32).reshape(-1)
    if kind == "vacancy":
        cells, at, N = [], 0, int(d["Na"].sum())
        r = d["r"].reshape(3, N)
        for c, na in enumerate(d["Na"]):
            keep = np.sort(rng.permutation(na)[: na - 1 - c % 3]) + at
            cells.append((d["box"].reshape(-1, 3, 3)[c], r[:, keep].T, np.zeros(len(keep), np.int32)))
            at += na
        e = synth._assemble(cells, 0.2, rng)
        d = {**d, **e}
    lo, hi = synth.TERSOFF_SI_MIN.copy(), synth.TERSOFF_SI_MAX.copy()
    if kind == "r1":
        lo[7], hi[7] = 2.3, 2.5
    if angle:
        lo[6], hi[6] = -0.225, -0.205
    if two:
        N = len(d["type"])
        d["type"] = ((rng.random(N) < 0.5).astype(np.int32) if kind == "alloy"
                     else np.tile(np.repeat(np.arange(2, dtype=np.int32), 4), N // 8))
        lo = np.concatenate([lo[:4], lo[:4] * 0.97, lo[4:]]).astype(np.float32)
        hi = np.concatenate([hi[:4], hi[:4] * 0.99, hi[4:]]).astype(np.float32)
    d.update(potential_type=2 if two else 1, pmin=lo, pmax=hi,
             truth=(0.4 * lo + 0.6 * hi).astype(np.float32))
    pot = {x: d[x] for x in ("potential_type", "cutoff", "weights", "pmin", "pmax")}
    return synth.label(d, O.Case(potential=pot, arrays=d).find_force), pot


@pytest.mark.parametrize("kind,two,P,opts", [
    ("strained", False, 70, {}), ("strained", False, 64, {"blocks_per_cu": 1}),
    ("strained", False, 5, {"pack_lanes": 0}), ("strained", True, 72, {}),
    ("strained", True, 3, {"pack_lanes": 0}), ("strained", True, 100, {}),
    ("alloy", True, 70, {}), ("alloy", True, 20, {}), ("r1", False, 70, {}), ("r1", True, 20, {}),
    ("vacancy", False, 68, {"chunk_cost": 10 ** 8}), ("vacancy", False, 20, {}),
    ("angle", False, 70, {}), ("angle", False, 20, {})])
def test_moment_records_match_oracle(kind, two, P, opts):
    import gpuga_amd as G
    from oracle import oracle as O
    print_case("tersoff moment records", kind, two, P, opts)
    d, pot = _set(kind, two)
    genes = np.random.default_rng(P).random((P, len(d["pmin"])), dtype=np.float32)
    with G.Fitness(arrays=d, **opts) as fit:
        f, terms = fit.compute(genes, terms=True)
        again, t2 = fit.compute(genes, terms=True)
        _, plain = fit.compute(genes, terms=True, plain=True)
    assert np.array_equal(f, again) and np.array_equal(terms, t2)
    ref, _ = O.Case(potential=pot, arrays=d).fitness(genes, threads=16)
    np.testing.assert_allclose(f, ref, rtol=1e-5)
    np.testing.assert_allclose(terms, plain, rtol=2e-5, atol=1e-7)
