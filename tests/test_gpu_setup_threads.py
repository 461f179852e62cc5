"""Sets of different potentials and form sizes set up at once on several threads,
as the server does: the same results as set up one after another."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from conftest import print_case
from test_gpu_quadform import _dimers, _genes, _ri

pytestmark = pytest.mark.gpu


def test_sets_built_on_several_threads():
    import gpuga_amd as G
    print_case("set-up on threads")
    jobs = [(_ri(Nc=4), {}), (_dimers(80, 30, 6, 1), dict(nn2b_grid=2048)),
            (_dimers(80, 30, 6, 2, species=True), dict(nn2b_grid=1024)),
            (_dimers(80, 30, 6, 3), dict(nn2b_grid=1536)), (_dimers(80, 30, 6, 4), dict(nn2b_grid=256))]

    def run(job):
        d, opts = job
        with G.Fitness(arrays=d, nn2b_bf16=0, chunk_cost=200, **opts) as fit:
            return fit.compute(_genes(d, 20, 1), terms=True)

    alone = [run(j) for j in jobs]
    with ThreadPoolExecutor(len(jobs)) as pool:
        for _ in range(3):
            for (f, t), (g, u) in zip(alone, pool.map(run, jobs)):
                assert np.array_equal(f, g) and np.array_equal(t, u)
