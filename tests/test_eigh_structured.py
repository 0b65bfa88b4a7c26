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
