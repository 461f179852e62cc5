"""NN2B networks whose curve bends within a few hundredths of an angstrom: genes
at the ends of their range, genes beyond it (weights up to twice the bounds),
coarse grids.  The quadratic forms' elements do not resolve such a curve; the
call must be as accurate as the tabulation with cubic interpolation that
serves it then.

Tolerance against the FP64 oracle, for each individual and term: 1e-5 (1e-4
with the split-BF16 layer), the stated bounds of the population path, and the
error of the cubic interpolation itself, restated here in FP64."""
import numpy as np
import pytest

from conftest import print_case
from test_gpu_quadform import _dimers, _oracle

pytestmark = pytest.mark.gpu


def _network(w, n, d, code=0):
    """U, U', U'' at the distances d of pairs with this species code."""
    w0, b0, w1 = w[:n], w[n:2 * n], w[2 * n:n * (n + 2)].reshape(n, n)
    b1, w2, b2 = w[n * (n + 2):n * (n + 3)], w[n * (n + 3):n * (n + 4)], w[n * (n + 4)]
    b0 = b0 - (code * w[n * (n + 4) + 1:] if len(w) > n * (n + 4) + 1 else 0.0)
    x = np.tanh(d[:, None] * w0 - b0)
    s = 1 - x * x
    z, zd, zdd = x @ w1.T - b1, (s * w0) @ w1.T, (-2 * x * s * w0 ** 2) @ w1.T
    y = np.tanh(z)
    t = 1 - y * y
    return y @ w2 - b2, (t * zd) @ w2, (t * zdd - 2 * y * t * zd ** 2) @ w2


def _cubic(w, n, d, G, lo, hi, code):
    """U and U' by cubic Hermite interpolation on G points: lo to hi and a spare
    cell on either side."""
    h = (hi - lo) / (G - 3)
    first = lo - h
    i = np.minimum(((d - first) / h).astype(int), G - 2)
    q = (d - first) / h - i
    a, b, c, e = (2 * q - 3) * q * q + 1, ((q - 2) * q + 1) * q * h, (3 - 2 * q) * q * q, \
        (q - 1) * q * q * h
    U, D, S = _network(w, n, first + h * np.arange(G), code)
    return (a * U[i] + b * D[i] + c * U[i + 1] + e * D[i + 1],
            a * D[i] + b * S[i] + c * D[i + 1] + e * S[i + 1])


def _interpolation_error(d, w, n, G):
    """Relative error of the three terms (energy, virial, force) by the cubic
    interpolation, over cells of two atoms."""
    r = np.asarray(d["r"], np.float64).reshape(3, -1, 2)
    v = r[:, :, 1] - r[:, :, 0]
    dist = np.sqrt((v ** 2).sum(0))
    on = dist < d["cutoff"]
    phase = np.pi * np.clip(dist - 7, 0, 1)
    fc, fcp = 0.5 * np.cos(phase) + 0.5, -0.5 * np.pi * np.sin(phase)
    ncf = d["Nc_force"]
    fr = np.asarray(d["force_ref"], np.float64).reshape(3, -1, 2)[:, :ncf]
    wr = np.asarray(d["virial_ref"], np.float64).reshape(6, -1)[:, ncf:]
    er = np.asarray(d["pe_ref"], np.float64)[ncf:]

    def sums(U, D):
        full = np.zeros((2, len(dist)))
        full[:, on] = U, D
        U, G = full[0] * fc, full[1] * fc + full[0] * fc * fcp
        f = v / dist * G  # on the first atom; the second's is its negative
        w6 = np.stack([-v[a] * v[b] / dist * G for a, b in
                       ((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (2, 0))])
        return np.sqrt([((U[ncf:] - er) ** 2).sum(), ((w6[:, ncf:] - wr) ** 2).sum(),
                        ((f[:, :ncf] - fr[:, :, 0]) ** 2).sum()
                        + ((f[:, :ncf] + fr[:, :, 1]) ** 2).sum()])

    code = np.asarray(d["type"]).reshape(-1, 2).sum(1)[on] * (len(w) > n * (n + 4) + 1)
    at, lo, hi = dist[on], dist[on].min(), dist[on].max()
    values = np.zeros((2, 2, len(at)))
    for c in np.unique(code):
        m = code == c
        values[0][:, m] = _network(w, n, at[m], c)[:2]
        values[1][:, m] = _cubic(w, n, at[m], G, lo, hi, c)
    exact = sums(*values[0])
    return np.abs(sums(*values[1]) - exact) / exact


def _sharp_genes(V, P, kind, seed):
    rng = np.random.default_rng(seed)
    side = np.sign(rng.random((P, V)) - 0.5)
    if kind == "ends":  # weights of 0.3 to 1 of the bound
        return (0.5 + 0.5 * side * rng.uniform(0.3, 1, (P, V))).astype(np.float32)
    return (0.5 + side * rng.uniform(0, 1, (P, V))).astype(np.float32)  # up to twice the bound


@pytest.mark.parametrize("n,grid,kind,bf16,P,species", [
    (20, 1024, "ends", 0, 70, False), (32, 1024, "ends", 0, 70, False),
    (64, 1024, "ends", 0, 70, False), (32, 512, "ends", 0, 70, False),
    (20, 256, "ends", 0, 70, False), (10, 1024, "beyond", 0, 70, False),
    (32, 1024, "beyond", 0, 200, False), (20, 1024, "beyond", 1, 70, False),
    (32, 1024, "ends", 1, 130, False), (16, 1024, "beyond", 0, 40, True)])
def test_sharp_networks_match_oracle(n, grid, kind, bf16, P, species):
    """Populations in which the elements resolve some networks and not others,
    from one lane block to four; the same bits again."""
    import gpuga_amd as G
    print_case("sharp networks", n, grid, kind, bf16, P, species)
    d = _dimers(400, 150, n, 40 + n, species=species)
    genes = _sharp_genes(len(d["pmin"]), P, kind, n)
    with G.Fitness(arrays=d, nn2b_bf16=bf16, nn2b_grid=grid) as fit:
        f, terms = fit.compute(genes, terms=True)
        again, terms2 = fit.compute(genes, terms=True)
        weights = np.array([fit.denormalise(g) for g in genes], np.float64)
    assert np.array_equal(f, again) and np.array_equal(terms, terms2)
    ref, rterms = _oracle(d).fitness(genes, threads=16)
    tol = (1e-4 if bf16 else 1e-5) + np.array(
        [_interpolation_error(d, w, n, grid) for w in weights])
    err = np.abs(terms - rterms) / rterms
    print("largest error / tolerance by term:", (err / tol).max(0), "errors:", err.max(0))
    assert np.all(err <= tol)
    assert np.all(np.abs(f - ref) <= tol.max(1) * ref)


@pytest.mark.parametrize("P", [30, 150])
def test_device_generations_with_sharp_networks_equal_the_host_loop(P):
    """A run that starts without the pair loop's tables and meets individuals that
    need them, and one that has them."""
    import gpuga_amd as G
    print_case("sharp networks, device GA", P)
    d = _dimers(60, 25, 20, 12)

    def ga():
        return G.GA(P, P // 2 + P // 2 % 2, len(d["pmin"]), maximum_generation=40, seed=5)

    with G.Fitness(arrays=d, nn2b_bf16=0, nn2b_grid=256, chunk_cost=200) as fit:
        first, second, host = ga(), ga(), ga()
        before = fit.device_bytes()
        got, _ = fit.run_ga(first, 0, 6)
        tables = 3 * 256 * 64 * 4 * ((P + 63) // 64)  # of the tabulation
        assert fit.device_bytes() - before >= tables
        got2, _ = fit.run_ga(second, 0, 6)
        best = []
        for k in range(6):
            f = fit.compute(host.population)
            best.append(np.min(f))
            host.step(k, f)
    assert np.array_equal(host.population, first.population)
    assert np.array_equal(first.population, second.population)
    assert np.array_equal(np.array(best, np.float32), got) and np.array_equal(got, got2)


def test_a_gene_that_is_no_number_stays_in_its_individual():
    import gpuga_amd as G
    print_case("sharp networks, NaN")
    d = _dimers(60, 25, 10, 13)
    genes = np.random.default_rng(14).random((40, len(d["pmin"])), dtype=np.float32)
    bad = genes.copy()
    bad[[3, 31], [5, 40]] = np.nan
    with G.Fitness(arrays=d, nn2b_bf16=0) as fit:
        f = fit.compute(genes)
        b = fit.compute(bad)
    assert np.all(np.isnan(b[[3, 31]]))
    keep = np.setdiff1d(np.arange(40), [3, 31])
    assert np.array_equal(f[keep], b[keep])
