"""Eigenvectors past one batch of 64 (eig_eigh with nvec > 64): the edges of the batches
and of the 32-wide reflector panels, a spectrum whose clusters span batches, repeated
eigenvalues, and a matrix that is diagonal already.  Orthonormality and residuals within
n * 64 ulps of the norm (the solver's own bar: eigenvalues to a few ulps of the norm,
vectors orthogonalised twice)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    import eig_amd
    e = eig_amd.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("n,nvec,kind", [
    (65, 65, "random"), (66, 65, "random"), (97, 97, "diagonal"), (129, 128, "clustered"),
    (130, 129, "repeated"), (193, 193, "clustered"), (225, 70, "random"), (321, 321, "repeated")])
def test_many_eigenvectors(eng, n, nvec, kind):
    rng = np.random.default_rng(n + nvec)
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    if kind == "random":
        a = rng.standard_normal((n, n))
        a = a @ a.T
    elif kind == "diagonal":
        a = np.diag(rng.permutation(np.arange(n) // 3).astype(float))
    else:
        w = np.repeat(rng.uniform(1, 10, n // 40 + 1), 40)[:n] if kind == "repeated" else \
            1.0 + 1e-9 * np.arange(n)
        w[:3] = (50.0, 40.0, 30.0)
        a = (q * w) @ q.T
    a = 0.5 * (a + a.T)
    print(f"[gpu-case] eigh n={n} nvec={nvec} {kind}", flush=True)
    w, v = eng.eigh(a, nvec)
    norm = max(abs(w[0]), abs(w[-1]))
    tol = 64 * n * 2.0 ** -53
    assert np.max(np.abs(v @ v.T - np.eye(nvec))) <= tol
    assert np.max(np.abs(v @ a - w[:nvec, None] * v)) <= tol * norm
