"""Every eigenvector of matrices with eigenvalues repeated 40-fold (eig_eigh with nvec =
n): residuals within 8 n u ||A|| (a backward stable reduction's n u ||A||, the solves' and
the back-transform's, with a factor for each) and orthonormality within 64 n u."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    import eig_amd
    e = eig_amd.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("seed", range(4))
@pytest.mark.parametrize("n", [130, 321, 700])
def test_repeated(eng, n, seed):
    rng = np.random.default_rng(seed)
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    w = np.repeat(rng.uniform(1, 10, n // 40 + 1), 40)[:n]
    w[:3] = (50.0, 40.0, 30.0)
    a = (q * w) @ q.T
    a = 0.5 * (a + a.T)
    print(f"[gpu-case] eigh n={n} repeated seed {seed}", flush=True)
    lam, v = eng.eigh(a, n)
    u = 2.0 ** -53
    assert np.max(np.abs(v @ v.T - np.eye(n))) <= 64 * n * u
    assert np.max(np.abs(v @ a - lam[:, None] * v)) <= 8 * n * u * 50.0
