"""Per-atom outputs of NN2B networks with small weights, whose activations are
near zero, where an absolute error of the tanh is a large relative one.

Tolerance of the energies against the FP64 oracle, root mean square over the
pairs: two units in the last place, 2^-22, of every term that is rounded (the
output layer's tanh, the products and biases that enter it, the first layer's
argument), in quadrature.  Forces and virials, whose bond vectors are FP32 too:
2e-6 of their root mean square."""
import numpy as np
import pytest

from conftest import print_case
from test_gpu_quadform import _dimers, _oracle

pytestmark = pytest.mark.gpu


def _rounded_terms(d, p, n):
    """Root sum square of the terms of U fc / 2 (an atom's energy), root mean
    square over the atoms."""
    r = np.asarray(d["r"], np.float64).reshape(3, -1, 2)
    dist = np.sqrt(((r[:, :, 1] - r[:, :, 0]) ** 2).sum(0))
    code = np.asarray(d["type"]).reshape(-1, 2).sum(1)
    w0, b0, w1 = p[:n], p[n:2 * n], p[2 * n:n * (n + 2)].reshape(n, n)
    b1, w2, ws = p[n * (n + 2):n * (n + 3)], p[n * (n + 3):n * (n + 4)], p[n * (n + 4) + 1:]
    shift = code[:, None] * ws if len(ws) else 0.0
    x = np.tanh(dist[:, None] * w0 + shift - b0)
    x2 = x ** 2 + (dist[:, None] * w0) ** 2 + np.square(shift) + b0 ** 2
    y = np.tanh(x @ w1.T - b1)
    terms = np.sqrt((y ** 2 + b1 ** 2 + x2 @ (w1 ** 2).T) @ w2 ** 2)
    fc = np.where(dist < 8, 0.5 * np.cos(np.pi * np.clip(dist - 7, 0, 1)) + 0.5, 0.0)
    return np.sqrt(np.mean((0.5 * fc * terms) ** 2))


@pytest.mark.parametrize("species", [False, True])
@pytest.mark.parametrize("n", [6, 20, 40])
@pytest.mark.parametrize("weight", [0.02, 0.05, 0.2, 1.0])
def test_energies_keep_their_digits(weight, n, species):
    import gpuga_amd as G
    print_case("small weights", weight, n, species)
    d = _dimers(500, 200, n, 50, species=species)
    rng = np.random.default_rng(51)
    p = (weight * rng.uniform(-1, 1, len(d["pmin"]))).astype(np.float32)
    p[n * (n + 4)] = 0.0  # (a constant would hide the network)
    with G.Fitness(arrays=d) as fit:
        f, w, e = fit.find_force(p)
    ref = _oracle(d).find_force(p)
    rms = [(np.sqrt(np.mean((a - b) ** 2)), np.sqrt(np.mean(b ** 2)))
           for a, b in zip((f, w, e), ref)]
    print("relative RMS error of force, virial, energy:", [a / b for a, b in rms])
    assert rms[0][0] < 2e-6 * rms[0][1] and rms[1][0] < 2e-6 * rms[1][1]
    assert rms[2][0] < 2.0 ** -22 * _rounded_terms(d, p.astype(np.float64), n)
