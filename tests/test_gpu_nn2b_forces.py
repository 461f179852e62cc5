"""Per-atom outputs of the NN2B network kernel (MFMA hidden layer, eight atoms
a wave, bonds in tiles of 32) against the FP64 oracle, at the neuron counts
where its operands change shape (one and two blocks of 32 output neurons,
padding, a single neuron), with atom counts that leave the last wave part
full, atoms without neighbours, and pairs inside the taper (7-8 A).
Tolerance: 2e-5 of the largest magnitude, the bound of every per-atom FP32
output."""
import numpy as np
import pytest

from conftest import print_case

pytestmark = pytest.mark.gpu


def _set(n, species, seed):
    """Clusters of 2 to 37 atoms in 40 A boxes (pairs from 1.5 A; a dimer out
    of reach has no neighbours), two species."""
    rng = np.random.default_rng(seed)
    pos, Na = [], []
    for na in (2, 2, 5, 3, 37, 9):
        if len(Na) == 0:
            p = np.array([[0, 0, 0], [9.0, 0, 0]])
        else:  # on a 2.2 A grid, displaced, so no pair is too close
            grid = np.stack(np.meshgrid(*[np.arange(4)] * 3), -1).reshape(-1, 3)
            p = 2.2 * grid[rng.permutation(64)[:na]] + rng.uniform(-0.3, 0.3, (na, 3))
        pos.append(p + 10.0)
        Na.append(na)
    r = np.concatenate(pos).T.astype(np.float32)
    V = n * (n + 4) + 1 + (n if species else 0)
    return dict(potential_type=4 if species else 3, num_neurons=n, cutoff=8.0,
                weights=(0.9, 0.1, 0.0), Na=np.array(Na, np.int32), Nc_force=2,
                type=rng.integers(0, 2, r.shape[1]).astype(np.int32), r=r.reshape(-1),
                box=np.tile(np.diag([40.0] * 3).reshape(-1), len(Na)).astype(np.float32),
                pmin=np.full(V, -3, np.float32), pmax=np.full(V, 3, np.float32),
                pe_ref=np.ones(len(Na), np.float32), virial_ref=np.ones(6 * len(Na), np.float32),
                force_ref=np.ones(r.size, np.float32))


@pytest.mark.parametrize("n,species", [(1, 0), (10, 0), (16, 1), (17, 0), (32, 1), (33, 0),
                                       (64, 1)])
def test_per_atom_outputs_match_oracle(n, species):
    import gpuga_amd as G
    from oracle import oracle as O
    print_case("nn2b per-atom outputs", n, species)
    d = _set(n, species, 100 + n)
    pot = {k: d[k] for k in ("potential_type", "cutoff", "weights", "pmin", "pmax", "num_neurons")}
    case = O.Case(potential=pot, arrays=d)
    params = np.random.default_rng(n).uniform(-1.5, 1.5, len(d["pmin"])).astype(np.float32)
    with G.Fitness(arrays=d) as fit:
        NN, _, _ = fit.neighbors()
        got = fit.find_force(params)
    assert 0 in NN and fit.N % 8 != 0
    for a, b in zip(got, case.find_force(params)):
        np.testing.assert_allclose(a, b, rtol=0, atol=2e-5 * np.abs(b).max())
