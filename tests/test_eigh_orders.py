"""eig_eigh at the orders where the tridiagonalisation changes its launch shape (256, 512,
1,024, 2,048, and whole panels of 32 beyond), and with reflectors whose squared norms leave
[1e-280, 1e280], against LAPACK.  A Householder reduction is backward stable with an error of about
sqrt(n) u ||A||_F <= n u ||A||_2; two solvers and a factor of four make 8 n u ||A||_2 for
the eigenvalues and for the residuals of the vectors."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    import eig_amd
    e = eig_amd.Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("n,kind", [
    (1, "random"), (2, "random"), (3, "random"), (8, "random"), (9, "random"), (255, "random"),
    (256, "random"), (257, "random"), (511, "random"), (512, "scaled-up"), (513, "random"),
    (600, "diagonal"), (700, "tridiagonal"), (1023, "random"), (1024, "low-rank"),
    (1025, "tiny-offdiagonal"), (2047, "random"), (2048, "random"), (2049, "random"), (2080, "random"),
    (2081, "low-rank")])
def test_orders(eng, n, kind):
    rng = np.random.default_rng(n)
    if kind == "diagonal":
        a = np.diag(rng.permutation(n).astype(float) + 1)
    elif kind == "tridiagonal":
        e = rng.uniform(0.5, 1.5, n - 1)
        a = np.diag(np.arange(n) + 1.0) + np.diag(e, 1) + np.diag(e, -1)
    elif kind == "low-rank":
        f = rng.standard_normal((n, 5))
        a = f @ f.T
    else:
        g = rng.standard_normal((n, n))
        a = 0.5 * (g + g.T) * {"scaled-up": 1e140, "tiny-offdiagonal": 1e-150}.get(kind, 1.0)
        if kind == "tiny-offdiagonal":
            a += np.diag(rng.permutation(n).astype(float) + 1)
    nvec = min(n, 4)
    print(f"[gpu-case] eigh n={n} {kind}", flush=True)
    w, v = eng.eigh(a, nvec)
    ref = np.linalg.eigvalsh(a)[::-1]
    norm = np.max(np.abs(ref))
    tol = 8 * n * 2.0 ** -53
    assert np.max(np.abs(w - ref)) <= tol * norm
    assert np.max(np.abs(v @ v.T - np.eye(nvec))) <= 8 * tol
    assert np.max(np.abs((v @ a - w[:nvec, None] * v) / norm)) <= tol


@pytest.mark.parametrize("n", [2, 3, 31, 34, 127, 128, 129, 130, 161, 257, 385, 700])
def test_launches_alone(eng, n, monkeypatch):
    """the launches that longer columns take, at the edges of their 128-wide tiles"""
    monkeypatch.setenv("EIG_NO_MERGE", "1")
    test_orders(eng, n, "random")
