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
