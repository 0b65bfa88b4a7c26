"""Eigenvalues by Sturm counts and vectors by inverse iteration at orders around their
pieces (16 rows a round of counts, 8 and 512 rows of a solve), on matrices whose leading
minors vanish at the counting points: repeated and zero diagonals, decoupled blocks,
against LAPACK.  A backward stable reduction and two solvers stay within 8 n u ||A||."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.fixture(scope="module")
def eng():
    import eig_amd
    e = eig_amd.Engine(0)
    yield e
    e.close()


def _matrix(kind, n):
    rng = np.random.default_rng(n)
    if kind == "identity":
        return np.eye(n)
    if kind == "blocks":  # decoupled pairs with eigenvalues 0 and 2
        a = np.eye(n)
        for i in range(0, n - 1, 2):
            a[i, i + 1] = a[i + 1, i] = 1.0
        return a
    if kind == "zero-diagonal":
        return np.diag(np.ones(n - 1), 1) + np.diag(np.ones(n - 1), -1)
    g = rng.standard_normal((n, n))
    return 0.5 * (g + g.T)


@pytest.mark.parametrize("n", [7, 8, 9, 15, 16, 17, 25, 33, 505, 514, 521, 1026])
def test_pieces(eng, n):
    _check(eng, "random", n)


@pytest.mark.parametrize("kind", ["identity", "blocks", "zero-diagonal"])
@pytest.mark.parametrize("n", [6, 130, 601])
def test_minors(eng, kind, n):
    _check(eng, kind, n)


def _check(eng, kind, n):
    a = _matrix(kind, n)
    nvec = min(n, 5)
    print(f"[gpu-case] eigh n={n} {kind}", flush=True)
    w, v = eng.eigh(a, nvec)
    ref = np.linalg.eigvalsh(a)[::-1]
    norm = np.max(np.abs(ref))
    tol = 8 * n * U
    assert np.max(np.abs(w - ref)) <= tol * norm
    assert np.max(np.abs(v @ v.T - np.eye(nvec))) <= 8 * tol
    assert np.max(np.abs((v @ a - w[:nvec, None] * v) / norm)) <= tol


@pytest.mark.parametrize("n", [2, 33, 34, 65, 512, 513, 545, 1025, 1599, 1600, 1601])
def test_back_transform(eng, n):
    """Panels of 32 reflectors, a thread's 512 rows, and the line between the two kernels."""
    _check(eng, "random", n)
