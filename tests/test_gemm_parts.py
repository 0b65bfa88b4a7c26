"""Products over a long k cut into parts, through the entry points that use them: the
explicit-column XTX at sample counts around the 64-row tiles and kept-SNP counts around the
parts' 128 and 16, and every eigenvector of orders around the batches of 64.

An FP64 product of k terms is off by at most k u of the sum of their magnitudes, with u =
2^-53; XTX's terms sum to at most sqrt(x_ii x_jj), bounded by the largest diagonal."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.fixture(scope="module")
def eng():
    import eig_amd
    e = eig_amd.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("N,M", [(63, 255), (64, 256), (65, 257), (130, 1025), (129, 4097), (200, 4200)])
def test_explicit_columns(eng, N, M):
    rng = np.random.default_rng(N + M)
    g = rng.binomial(2, rng.uniform(0.2, 0.8, M)[:, None], (M, N)).astype(np.int32)
    w = rng.uniform(0.5, 1.5, M)
    eng.load_packed(O.pack_genotypes(g), N)
    eng.select(np.arange(N, dtype=np.int32))
    eng.snpstats()
    scale, ynum, st, x = eng.xtx_normal(xtypes=np.zeros(N, np.int32), npop=1, weight=w)
    mean = g.mean(axis=1)
    p = 0.5 * mean
    z = ((g - mean[:, None]) / np.sqrt(p * (1 - p))[:, None] * w[:, None])[st["status"] == 0]
    ref = (z.T.astype(np.longdouble) @ z.astype(np.longdouble)).astype(float)
    ref *= (N - 1) / np.trace(ref)
    assert ynum == len(z)
    # both sides' entries and the scale: the products' error and a few roundings of the columns
    assert np.max(np.abs(x - ref)) <= 4 * (M + 16) * U * np.max(np.diag(ref))


@pytest.mark.parametrize("n", [127, 129, 193, 257, 400])
def test_all_vectors(eng, n):
    """A backward stable reduction's n u ||A||, the solves' and the back-transform's."""
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    a = 0.5 * (a + a.T)
    lam, v = eng.eigh(a, n)
    norm = np.max(np.abs(lam))
    assert np.max(np.abs(v @ v.T - np.eye(n))) <= 64 * n * U
    assert np.max(np.abs(v @ a - lam[:, None] * v)) <= 8 * n * U * norm
