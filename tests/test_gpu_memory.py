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


def _used():
    """Bytes of device memory in use."""
    import ctypes

    import gpuga_amd as G
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert G.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return total.value - free.value


def _job(d, path, P):
    from gpuga_amd import synth
    synth.write_dir(d, str(path))
    (path / "ga.in").write_text(f"maximum_generation 2\npopulation_size {P}\nparent_number {P // 2}\n"
                                "mutation_rate 0.2\nseed 1\n")
    return str(path)


@pytest.mark.parametrize("kind", ["tersoff", "shell", "ri", "species"])
def test_the_estimate_covers_what_a_job_takes(tmp_path, kind):
    """Two jobs under a budget just below twice what one of them takes at its
    peak (set-up included, work items of one configuration, the fewest), as
    seen in the device's free memory while one is set up and evaluated: they must
    not run together.  (Allocations come in pages of 2 MiB, so a few of these are
    left out.)"""
    import threading

    import gpuga_amd as G
    from gpuga_amd import synth
    print_case("memory, estimate", kind)
    P = 64
    if kind in ("tersoff", "shell"):
        d = synth.tersoff_si(Nc=150, reps=(3, 3, 3), sizes="fixed", seed=4)
        if kind == "shell":
            d["cutoff"] = 4.0
            d["pmax"] = d["pmax"].copy()
            d["pmax"][-1] = 4.0
    elif kind == "ri":
        d = synth.fluorite_ab2(Nc=100, force_fraction=0.3, seed=5)
    else:
        d = synth.wurtzite_ab(Nc=700, n=10, force_fraction=0.2, seed=6, species=True)
    path = _job(d, tmp_path, P)
    G.Fitness(path).close()  # (the library's own allocations)
    base, peak, done = _used(), [0], threading.Event()

    def watch():
        while not done.is_set():
            peak[0] = max(peak[0], _used() - base)

    t = threading.Thread(target=watch)
    t.start()
    try:
        with G.Fitness(path, chunk_cost=10 ** 6) as fit:
            fit.compute(np.random.default_rng(0).random((P, fit.V), dtype=np.float32))
    finally:
        done.set()
        t.join()
    one = peak[0] - (30 << 20)
    print("one job takes", peak[0] / 2 ** 20, "MiB")
    assert one > 0
    s = G.Server(memory_budget_bytes=2.0 * one, max_active=4)
    ids = [s.submit(path) for _ in range(2)]
    most = finished = 0
    while finished < len(ids):
        active, _, finished = s.poll()
        most = max(most, active)
    assert most == 1
    assert all(s.job(i, 2000)["state"] == 2 for i in ids)
