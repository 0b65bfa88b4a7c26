"""Eigensolves of matrices whose rank is used up long before their order: constant blocks and
their products leave a remainder of the same structure in every column of the reduction, so
that it shrinks by a rounding error each time.  The reduction's n reflections are orthogonal to
a few ulps each and every later step adds a few, so 20 n ulps bound the vectors' orthogonality
and, of the norm, their residual."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def matrices():
    b = np.random.default_rng(0).standard_normal((10, 10))
    b = b + b.T
    blocks = np.zeros((200, 200))
    blocks[:100, :100], blocks[100:, 100:] = 1, 2
    return {"ones64": np.ones((64, 64)), "ones150": np.ones((150, 150)), "ones257": np.ones((257, 257)),
            "ones1000": np.ones((1000, 1000)), "ones2113": np.ones((2113, 2113)), "blocks": blocks,
            "small": 1e-60 * blocks, "kron30": np.kron(b, np.ones((30, 30))),
            "kron100": np.kron(b @ b, np.ones((100, 100)))}


@pytest.mark.parametrize("name", list(matrices()))
def test_vectors_of_structured_matrices(name):
    import eig_amd
    a = np.ascontiguousarray(matrices()[name])
    n = len(a)
    w = np.linalg.eigvalsh(a)[::-1]
    norm = np.abs(w).max()
    tol = 20 * n * 2.0 ** -53
    eng = eig_amd.Engine(0)
    try:
        for nv in (10, 66 if n > 66 else n):
            print(f"[gpu-case] eigh {name} nvec={nv}", flush=True)
            ev, v = eng.eigh(a, nv)
            assert np.max(np.abs(ev - w)) <= tol * norm
            assert np.max(np.abs(a @ v.T - v.T * ev[:nv])) <= tol * norm
            assert np.max(np.abs(v @ v.T - np.eye(nv))) <= tol
    finally:
        eng.close()


def repeated(name):
    rng = np.random.default_rng(0)
    b = rng.standard_normal((10, 10))
    b = b + b.T
    if name.startswith("kron"):
        m = int(name[4:])
        return np.ascontiguousarray(np.kron(np.ones((m, m)), b))
    n = 520 if name == "split" else 300
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    lam = {"three": np.repeat([-4.0, 1.0, 4.0], [7, n - 19, 12]), "split": np.repeat([-3.0, 0.0, 0.5, 4.0], n // 4),
           "near": np.r_[1 + 2e-15 * rng.standard_normal(n - 60), rng.standard_normal(60)]}[name]
    a = q @ np.diag(lam) @ q.T
    return (a + a.T) / 2


@pytest.mark.parametrize("name", ["kron13", "kron30", "three", "split", "near"])
def test_eigenvalues_repeated_over_batches(name):
    """An eigenvalue that fills several batches of vectors.  A run of eigenvalues that takes one
    shift is at most 32 ulps of the tridiagonal's norm wide, which is at most three times the
    matrix'; with an ulp or two of every other step 100 ulps bound the residual."""
    import eig_amd
    a = repeated(name)
    n = len(a)
    norm = np.abs(np.linalg.eigvalsh(a)).max()
    eng = eig_amd.Engine(0)
    try:
        for nv in (10, 64, 65, n):
            print(f"[gpu-case] eigh repeated {name} nvec={nv}", flush=True)
            ev, v = eng.eigh(a, nv)
            assert np.max(np.abs(a @ v.T - v.T * ev[:nv])) <= 100 * 2.0 ** -52 * norm
            assert np.max(np.abs(v @ v.T - np.eye(nv))) <= 20 * n * 2.0 ** -53
    finally:
        eng.close()
