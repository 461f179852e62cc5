"""Device memory of a resident training set and of a job's set-up."""
import numpy as np
import pytest

from conftest import print_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cutoff,slots", [(3.5, 8), (3.9, 16)])
def test_only_the_records_that_the_kernel_reads(cutoff, slots):
    """5 to 16 neighbours: the set keeps one cosine per pair of bonds, not the
    general records (1 + M + M^2 + M / 2 float4 an atom) too; these can still be
    looked at."""
    import gpuga_amd as G
    from gpuga_amd import synth
    print_case("memory, records", cutoff)
    d = synth.tersoff_si(Nc=12, reps=(3, 3, 3), seed=4)
    d["cutoff"] = cutoff
    d["pmax"] = d["pmax"].copy()
    d["pmax"][-1] = cutoff
    N = int(np.sum(d["Na"]))
    general = 16 * N * (1 + slots + slots * slots + slots // 2)
    with G.Fitness(arrays=d) as fit:
        kept = fit.device_bytes()
        bond, tri, rec = fit.geometry()
        assert fit.device_bytes() == kept
    assert rec.nbytes == general
    assert kept - bond.nbytes - tri.nbytes < general
