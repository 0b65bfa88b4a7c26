"""The FP64 form's XTX as a matrix: what it is off in an entry must not add up over rows or
columns to an error of rank one, which the eigenvalues would see N times over.  A bracket's
rounding repeats for all samples of a genotype, most of all in panels of rare variants.

Tolerance, in the spectral norm: M products added in FP64 leave about sqrt(M) ulps of the
largest diagonal element, and the levels, the combination of the digits and the scaling 16
ulps (those of test_xtx_digits) of the largest eigenvalue.
"""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    import eig_amd
    e = eig_amd.Engine(0)
    yield e
    e.close()


def spectral(d):
    return float(np.abs(np.linalg.eigvalsh(d)).max())


@pytest.mark.parametrize("N,M,rare,miss,fancynorm", [
    (198, 2000, True, 0.0, 0), (300, 1025, True, 0.0, 0), (1500, 20000, True, 0.0, 0),
    (300, 1025, False, 0.0, 1), (300, 1025, False, 0.03, 1), (257, 900, True, 0.05, 0)])
def test_xtx_fp64_spectral_error(eng, N, M, rare, miss, fancynorm):
    rng = np.random.default_rng(N + M)
    p = rng.uniform(0.3 / N, 3.0 / N, M) if rare else rng.uniform(0.1, 0.5, M)
    g = rng.binomial(2, p[:, None], size=(M, N)).astype(np.int8)
    g[rng.random((M, N)) < miss] = -1
    print(f"[gpu-case] xtx spectral N={N} M={M} rare={rare} miss={miss} fancynorm={fancynorm}", flush=True)
    eng.load_packed(O.pack_genotypes(g.astype(np.int32)), N)
    eng.select(np.arange(N, dtype=np.int32))
    st = eng.snpstats(fancynorm=fancynorm)
    y, mat = eng.xtx(0)
    keep = st["status"] == 0
    g, mean, f = g[keep], st["mean"][keep], st["fancy"][keep]
    if miss == 0.0 and fancynorm == 0:  # integers but for the means: X = G'G - a_i - a_j + b
        assert np.all(f == 1.0)
        gg = g.astype(np.float64).T @ g.astype(np.float64)
        ml = mean.astype(np.longdouble)
        a = np.concatenate([(g[:, i:i + 100].astype(np.longdouble) * ml[:, None]).sum(axis=0)
                            for i in range(0, N, 100)])
        want = gg.astype(np.longdouble) - a[:, None] - a[None, :] + (ml * ml).sum()
    else:
        x = (g - mean[:, None].astype(np.longdouble)) * f[:, None].astype(np.longdouble)
        x[g < 0] = 0.0
        want = np.stack([(x * x[:, c:c + 1]).sum(axis=0) for c in range(N)])
    err = spectral((mat.astype(np.longdouble) * np.longdouble(y) - want).astype(np.float64))
    w64 = want.astype(np.float64)
    tol = 2.0 ** -53 * (math.sqrt(M) * np.diag(w64).max() + 16 * spectral(w64))
    print(f"error {err:.2e} of {tol:.2e}", flush=True)
    assert err <= tol
